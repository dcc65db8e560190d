"""Out-of-memory paths and the store-or-recompute choice (forced from the
host, no GPU allocation actually fails):

  * with xr_set_memory_limit below what a density's scratch needs, the call
    fails with XR_ENOMEM (a clean error, the context stays usable) and runs
    again once the cap is lifted;
  * an XRSystem whose sigma budget is below every monomer sigma
    intermediate recomputes them in the adjoint, with the same energy and
    gradient as the one that stores them;
  * an FP64 product keeps its K split under a pin that admits it, and under a
    limit it is refused with its output untouched, or right;
  * an adjoint that is refused at any limit has added to none of its outputs."""
import numpy as np
import pytest
import torch

from qodeapplications_amd import density as D
from qodeapplications_amd import synthetic as syn
from qodeapplications_amd._lib import XR_ENOMEM, XRError, context, ptr
from qodeapplications_amd.gemm import mm

pytestmark = pytest.mark.gpu


def test_memory_limit_gives_enomem_and_recovers():
    rng = np.random.default_rng(1)
    st = syn.random_states(7, 4, 6, rng)
    sb = syn.random_states(7, 5, 5, rng)
    kb = D.ChargeBlock(7, 0, st.configs, st.coeffs)
    bb = D.ChargeBlock(7, 0, sb.configs, sb.coeffs)
    ctx = context(0)
    ctx.call("xr_trim")
    ctx.call("xr_set_memory_limit", 4096)
    try:
        with pytest.raises(XRError) as e:
            D.density("cca", bb, kb)
        assert e.value.code == XR_ENOMEM
    finally:
        ctx.call("xr_set_memory_limit", 0)
    ref = D.density("cca", bb, kb)
    again = D.density("cca", bb, kb)
    torch.cuda.synchronize()
    assert torch.equal(ref, again)


def test_sigma_recomputed_under_budget_matches_stored():
    from qodeapplications_amd.grad import energy_and_gradient
    from qodeapplications_amd.xr import XRSystem
    rng = np.random.default_rng(3)
    orbs = [3, 4]
    frags = [syn.make_fragment(n, [2, 3, 4], 3, 3, rng) for n in orbs]
    ints = syn.FragmentBlocked(orbs, syn.spatial_h(7, rng), syn.spatial_V(7, rng))
    keep = XRSystem(frags, ints, np.zeros((2, 2)))
    recompute = XRSystem(frags, ints, np.zeros((2, 2)), sigma_budget=0)
    E1, _, z1, i1 = energy_and_gradient(keep)
    assert any(F.E2W for F in keep.frags)
    E2, _, z2, i2 = energy_and_gradient(recompute)
    assert not any(F.E2W for F in recompute.frags)
    assert abs(E1 - E2) < 1e-12
    for m in range(2):
        for c in z1[m]:
            assert float((z1[m][c] - z2[m][c]).abs().max()) < 1e-10
    for k in i1:
        assert float((i1[k] - i2[k]).abs().max()) < 1e-10


def _product(M, N, K, beta=0.0):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    r = lambda a, b: torch.randn(a, b, dtype=torch.float64, device="cuda", generator=g)
    return r(M, K), r(K, N), r(M, N), beta


def test_pinned_product_runs_as_before_the_pin():
    # a product admitted under a pin because a larger one ran before it keeps
    # its K split (same bits), though the larger one staged nothing of its own
    A, B, C, _ = _product(64, 64, 400000)
    ctx = context(0)
    ctx.call("xr_trim")
    want = mm(A, B)
    ctx.call("xr_trim")
    a, b, c, beta = _product(2000, 2000, 320, 1.0)
    mm(a, b, out=c, beta=beta)
    ctx.call("xr_pin", 1)
    try:
        assert torch.equal(mm(A, B), want)
    finally:
        ctx.call("xr_pin", -1)


@pytest.mark.parametrize("M,N,K", [(300, 300, 20000), (64, 65, 100001)])
def test_product_under_a_limit_is_refused_or_right(M, N, K):
    A, B, C0, beta = _product(M, N, K, 0.5)
    ref = A @ B + beta * C0
    bound = (2 * (K + 2) + 4) * 2.0 ** -53 * (A.abs() @ B.abs() + beta * C0.abs())
    ctx = context(0)
    refused = 0
    limits = [4096] + [8 * M * N * s for s in (1, 2, 3, 5, 8, 13, 21, 34, 55, 89, 144, 233, 377, 610)]
    try:
        for limit in limits:
            ctx.call("xr_trim")
            ctx.call("xr_set_memory_limit", limit)
            C = C0.clone()
            try:
                mm(A, B, out=C, beta=beta)
            except XRError as e:
                assert e.code == XR_ENOMEM and torch.equal(C, C0)
                refused += 1
                continue
            assert bool(((C - ref).abs() <= bound).all()), limit
    finally:
        ctx.call("xr_set_memory_limit", 0)
    assert 0 < refused < len(limits)


@pytest.mark.parametrize("op", ["a", "aa", "c", "cc", "ca", "caa", "cca", "2e"])
def test_refused_adjoint_leaves_its_outputs(op):
    n, ne, nI, nJ = 6, 4, 7, 4
    nb = ne if op == "2e" else ne + op.count("c") - op.count("a")
    rng = np.random.default_rng(4)
    kb = D.ChargeBlock.from_states(syn.random_states(n, ne, nJ, rng), n, 0)
    bb = D.ChargeBlock.from_states(syn.random_states(n, nb, nI, rng), n, 0)
    dim = 2 * n
    rand = lambda *s: torch.as_tensor(rng.standard_normal(s), device="cuda")
    head = (n, 0, ne, nI, bb.n_configs, ptr(bb.coeffs), nJ, kb.n_configs, ptr(kb.coeffs))
    init = [rand(*bb.coeffs.shape), rand(*kb.coeffs.shape)]
    if op == "2e":
        V, Eb = rand(dim, dim, dim, dim), rand(nI, nJ)
        init.append(rand(dim, dim, dim, dim))
        call = lambda out: context(0).call("xr_monomer_2e_adjoint", *head, ptr(V), ptr(Eb), *[ptr(t) for t in out])
    else:
        Rb = rand(nI, nJ, *([dim] * len(op)))
        call = lambda out: context(0).call("xr_density_adjoint", op.encode(), *head, ptr(Rb), *[ptr(t) for t in out])
    want = [t.clone() for t in init]
    call(want)
    ctx = context(0)
    limit, refused = 2048, 0
    try:
        while True:
            ctx.call("xr_trim")
            ctx.call("xr_set_memory_limit", int(limit))
            out = [t.clone() for t in init]
            try:
                call(out)
                break
            except XRError as e:
                assert e.code == XR_ENOMEM
                assert all(torch.equal(a, b) for a, b in zip(out, init)), limit
                refused += 1
                limit *= 1.05
    finally:
        ctx.call("xr_set_memory_limit", 0)
    assert refused > 0
    # not the same bits: a limit may leave a product another split of K
    for a, b in zip(out, want):
        assert float((a - b).abs().max()) < 1e-12 * float(b.abs().max())
