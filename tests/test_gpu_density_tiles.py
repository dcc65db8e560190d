"""The density pipeline at the edges of its tiles and rules: numbers of ket
states around the plane tile (8 and 16), right tuples that fill it or do not fit,
coefficients gathered as stored and transposed first, and factors that are the stored
coefficients themselves (no creators, or no annihilators).

Tolerances: an element is a sum of products of two unit vectors' entries, so
it is at most 1 and its rounding a few hundred units of u = 2^-53 (sums of at
most 7e4 terms in pairs of partial sums); the adjoints are compared through the
sums they enter, with the absolute sums as the scale."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc
from qodeapplications_amd import density as D
from qodeapplications_amd import synthetic as syn
from qodeapplications_amd._lib import context, ptr

pytestmark = pytest.mark.gpu
U = 2.0 ** -53


def _blocks(op, n_orbs, n_elec, nI, nJ, seed=5):
    rng = np.random.default_rng(seed)
    nb = n_elec + op.count("c") - op.count("a")
    sk, sb = syn.random_states(n_orbs, n_elec, nJ, rng), syn.random_states(n_orbs, nb, nI, rng)
    return sb, sk, D.ChargeBlock.from_states(sb, n_orbs, 0), D.ChargeBlock.from_states(sk, n_orbs, 0)


@pytest.mark.parametrize("op", ["a", "aa", "c", "cc", "ca", "caa", "cca", "ccaa"])
@pytest.mark.parametrize("nI,nJ", [(1, 1), (3, 8), (2, 9), (5, 16), (4, 17), (1, 33)])
def test_planes_around_the_tile(op, nI, nJ):
    sb, sk, bra, ket = _blocks(op, 5, 4, nI, nJ)
    ref = orc.density(op, 5, 0, sb.coeffs, sk.coeffs, sk.configs)
    got = D.density(op, bra, ket).cpu().numpy()
    assert got.shape == ref.shape and np.abs(got - ref).max() < 400 * U


@pytest.mark.parametrize("op,n_orbs,n_elec", [("a", 13, 5), ("ca", 13, 5), ("caa", 13, 5), ("caaa", 13, 4), ("ccaaa", 6, 4),
                                              ("ccaa", 13, 4)])
def test_states_alone_and_together(op, n_orbs, n_elec):
    # one state a side: coefficients as stored; all: transposed first (n_elec = 5, > 1 MB)
    nI, nJ = 2, 10 if op != "ccaa" else 3
    sb, sk, bra, ket = _blocks(op, n_orbs, n_elec, nI, nJ)
    whole = D.density(op, bra, ket)
    for i, j in ((0, 0), (nI - 1, nJ - 1), (0, nJ - 1)):
        b1 = D.ChargeBlock(n_orbs, 0, sb.configs, sb.coeffs[i:i + 1])
        k1 = D.ChargeBlock(n_orbs, 0, sk.configs, sk.coeffs[j:j + 1])
        one = D.density(op, b1, k1)
        assert float((one[0, 0] - whole[i, j]).abs().max()) < 400 * U


@pytest.mark.parametrize("op", ["a", "aa", "c", "cc", "ca", "caa"])
@pytest.mark.parametrize("nI,nJ", [(1, 1), (3, 4), (17, 9)])
def test_adjoint_is_the_transpose_and_adds(op, nI, nJ):
    n, e = 7, 4
    _, _, bra, ket = _blocks(op, n, e, nI, nJ)
    rho = D.density(op, bra, ket)
    g = torch.Generator(device="cuda").manual_seed(1)
    Rb = torch.randn(rho.shape, dtype=torch.float64, device="cuda", generator=g)
    zb, zk = torch.ones_like(bra.coeffs), torch.ones_like(ket.coeffs)
    context(0).call("xr_density_adjoint", op.encode(), n, 0, e, nI, bra.n_configs, ptr(bra.coeffs), nJ,
                    ket.n_configs, ptr(ket.coeffs), ptr(Rb), ptr(zb), ptr(zk))
    want, scale = float((rho * Rb).sum()), float((rho * Rb).abs().sum()) + rho.numel() * U
    for z, zbar in ((bra.coeffs, zb), (ket.coeffs, zk)):
        # the dot products' own rounding goes with their absolute sum
        mag = float((z * (zbar - 1)).abs().sum())
        assert abs(float((z * (zbar - 1)).sum()) - want) < 400 * U * (scale + mag + float(z.abs().sum()))
