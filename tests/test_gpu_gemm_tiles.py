"""The FP64 product kernels at the sizes where a tile can go wrong: one
short of, equal to and one past the fragment, tile and K-step sizes, rows
that are and are not 16-byte aligned, every transpose, beta, views of wider
buffers and K splits, against torch in FP64.

Tolerance, element by element: two FP64 sums of the same K products in
different orders differ by at most 2 (K + 2) u sum|a b| (u = 2^-53, the
standard bound of recursive summation for each side), plus the roundings of
alpha and beta."""
import pytest
import torch

from qodeapplications_amd._lib import context, ptr
from qodeapplications_amd.gemm import mm

pytestmark = pytest.mark.gpu


def _check(ta, tb, M, N, K, alpha=1.0, beta=0.0, pad=0, shift=0):
    g = torch.Generator(device="cuda").manual_seed(M * 7919 + N * 31 + K)
    r = lambda a, b: torch.randn(a, b + pad + shift, dtype=torch.float64, device="cuda",
                                 generator=g)[:, shift:shift + b]
    A = r(K, M) if ta else r(M, K)
    B = r(N, K) if tb else r(K, N)
    C0 = r(M, N)
    got = C0.clone() if not (pad or shift) else r(M, N).copy_(C0)
    # the columns around a view of a wider buffer must stay as they are
    base = got._base
    edges = None if base is None else [base[:, :shift].clone(), base[:, shift + N:].clone()]
    mm(A, B, transA=ta, transB=tb, alpha=alpha, out=got, beta=beta)
    if edges is not None:
        assert torch.equal(base[:, :shift], edges[0]) and torch.equal(base[:, shift + N:], edges[1])
    oa, ob = (A.T if ta else A).contiguous(), (B.T if tb else B).contiguous()
    ref = alpha * (oa @ ob) + beta * C0
    mag = abs(alpha) * (oa.abs() @ ob.abs()) + abs(beta) * C0.abs()
    bound = (2 * (K + 2) + 4) * 2.0 ** -53 * mag + 1e-300
    assert bool(((got - ref).abs() <= bound).all()), float(((got - ref).abs() / bound).max())


@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (1, 33, 7), (15, 17, 8), (16, 16, 9), (31, 32, 31), (33, 31, 33),
                                   (64, 65, 40), (127, 129, 257), (130, 66, 1), (96, 96, 3001), (45, 20, 20011),
                                   (64, 324, 64), (325, 325, 4003)])
def test_small_and_split_products(ta, tb, M, N, K):
    _check(ta, tb, M, N, K)
    _check(ta, tb, M, N, K, alpha=-0.5, beta=1.5, pad=3, shift=1)


# sizes large enough for each tile shape: 128 x 128, 128 x 64, 64 x 128 and
# 64 x 64, with K steps that end inside and at a step, and their odd neighbours
@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("M,N,K", [(2600, 10400, 96), (14950, 834, 98), (2050, 2046, 130), (1026, 17576, 26),
                                   (3070, 3074, 112), (1690, 2197, 303), (1691, 2198, 302), (2049, 2047, 17)])
def test_tile_edges(ta, tb, M, N, K):
    _check(ta, tb, M, N, K)
    _check(ta, tb, M, N, K, alpha=2.0, beta=1.0, pad=2)


@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 0), (0, 1), (1, 1)])
def test_unaligned_base(ta, tb):
    # even leading dimensions and extents, but rows that start 8 bytes off a 16-byte boundary
    _check(ta, tb, 700, 900, 330, pad=1, shift=1)


@pytest.mark.parametrize("n,K", [(1, 5), (65, 33), (129, 1000), (834, 4098), (835, 4097)])
@pytest.mark.parametrize("trans", [0, 1])
def test_syrk_tiles(n, K, trans):
    from qodeapplications_amd.gemm import syrk
    g = torch.Generator(device="cuda").manual_seed(n + K)
    A = torch.randn(*((K, n) if trans else (n, K)), dtype=torch.float64, device="cuda", generator=g)
    got = syrk(A, trans)
    X = A.T.contiguous() if trans else A
    bound = 2 * (K + 2) * 2.0 ** -53 * (X.abs() @ X.abs().T.contiguous())
    assert torch.equal(got, got.T)
    assert bool(((got - X @ X.T.contiguous()).abs() <= bound).all())


def test_grouped_mixed_alignment():
    # products whose rows are 16-byte aligned and products whose rows are not, in one call
    import numpy as np
    shapes = [(300, 200, 150), (301, 199, 151), (128, 64, 16), (129, 9, 33), (200, 20, 31)]
    g = torch.Generator(device="cuda").manual_seed(5)
    As = [torch.randn(m, k, dtype=torch.float64, device="cuda", generator=g) for m, n, k in shapes]
    Bs = [torch.randn(k, n, dtype=torch.float64, device="cuda", generator=g) for m, n, k in shapes]
    Cs = [torch.full((m, n), float("nan"), dtype=torch.float64, device="cuda") for m, n, k in shapes]
    i64 = lambda v: np.ascontiguousarray(np.asarray(v, dtype=np.int64))
    p64 = lambda ts: np.asarray([t.data_ptr() for t in ts], dtype=np.uint64)
    M, N, K = (i64([s[j] for s in shapes]) for j in range(3))
    a, b, c = p64(As), p64(Bs), p64(Cs)
    P = lambda x: x.ctypes.data
    context(0).call("xr_gemm_grouped", len(shapes), 0, 0, P(M), P(N), P(K), 1.0, P(a), P(K), P(b), P(N), P(c), P(N))
    for A, B, C in zip(As, Bs, Cs):
        bound = 2 * (A.shape[1] + 2) * 2.0 ** -53 * (A.abs() @ B.abs())
        assert bool(((C - A @ B).abs() <= bound).all())


def test_nan_and_inf_stay_in_their_rows():
    # padding must not carry a row's NaN or infinity into another row or column
    for M, N, K in ((70, 50, 37), (258, 260, 34), (259, 261, 35), (2050, 2050, 66)):
        for ta, tb in ((0, 0), (1, 1)):
            A = torch.ones(*((K, M) if ta else (M, K)), dtype=torch.float64, device="cuda")
            B = torch.ones(*((N, K) if tb else (K, N)), dtype=torch.float64, device="cuda")
            (A[:, M - 1] if ta else A[M - 1])[:] = float("nan")
            (B[0] if tb else B[:, 0])[:] = float("inf")
            C = mm(A, B, transA=ta, transB=tb)
            assert bool(torch.isnan(C[M - 1]).all()) and bool(torch.isinf(C[:M - 1, 0]).all())
            assert torch.equal(C[:M - 1, 1:], torch.full_like(C[:M - 1, 1:], float(K)))


@pytest.mark.parametrize("odd", [0, 1])
@pytest.mark.parametrize("rows", [65, 4096, 4160])
def test_grouped_on_either_side_of_the_one_launch_rule(rows, odd):
    # 64 x 64 tiles in all: 2 x 8, 64 x 8 = 512 (one launch) and 65 x 8 = 520 (apart by width)
    shapes = [(rows, 320 - odd, 130), (rows, 64 - odd, 129 + odd), (rows, 128 - odd, 65)]
    g = torch.Generator(device="cuda").manual_seed(rows + odd)
    r = lambda a, b: torch.randn(a, b, dtype=torch.float64, device="cuda", generator=g)
    As, Bs = [r(m, k) for m, w, k in shapes], [r(k, w) for m, w, k in shapes]
    Cs = [r(m, w) for m, w, k in shapes]
    n = len(shapes)
    import ctypes
    L = lambda v: (ctypes.c_int64 * n)(*v)
    P = lambda v: (ctypes.c_void_p * n)(*[t.data_ptr() for t in v])
    M, N, K = (L([s[i] for s in shapes]) for i in range(3))
    context(0).call("xr_gemm_grouped", n, 0, 0, M, N, K, 1.0, P(As), K, P(Bs), N, P(Cs), N)
    for A, B, C in zip(As, Bs, Cs):
        bound = 2 * (A.shape[1] + 2) * 2.0 ** -53 * (A.abs() @ B.abs())
        assert bool(((C - A @ B).abs() <= bound).all())
