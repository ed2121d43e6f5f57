"""GPU: kernels at the edges of their tiles and dispatch rules against plain
float64 torch or numpy.

Tolerances: a sum of K products of N(0, 1) entries in any order differs from
another order by less than K eps times the sum of the products' magnitudes.
"""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip('torch')
pytestmark = pytest.mark.gpu
EPS = 2.0 ** -52


@pytest.fixture(scope='module')
def lib():
    assert torch.cuda.is_available(), 'GPU tests need a HIP device'
    from scikit_tt_amd import _lib
    torch.cuda.set_device(0)
    return _lib.load()


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def _randn(gen, *shape, shift=0):
    """N(0, 1) entries; shift = 1 starts 8 bytes past a 16-byte boundary."""
    n = int(np.prod(shape))
    return torch.randn(n + shift, dtype=torch.float64, device='cuda', generator=gen)[shift:].view(*shape)


@pytest.mark.parametrize('n', [1, 4, 5, 8, 9, 16, 17, 32, 33])
@pytest.mark.parametrize('r1,m,r2,s1,p,s2,shift', [(1, 1, 1, 1, 1, 1, 0), (2, 3, 4, 5, 1, 6, 0), (2, 3, 4, 5, 1, 6, 1),
                                                   (3, 2, 7, 3, 2, 129, 0), (1, 5, 3, 300, 1, 2, 0)])
def test_core_product(lib, n, r1, m, r2, s1, p, s2, shift):
    gen = torch.Generator(device='cuda').manual_seed(n * 100 + s2)
    A, X = _randn(gen, r1, m, n, r2), _randn(gen, s1, n, p, s2, shift=shift)
    out = _randn(gen, r1 * s1, m, p, r2 * s2)
    assert lib.ttals_core_product(None, r1, m, n, r2, s1, p, s2, _ptr(A), _ptr(X), _ptr(out)) == 0

    def product(a, x):
        t = torch.tensordot(a, x, dims=([2], [1])).permute(0, 3, 1, 4, 2, 5)
        return t.reshape(r1 * s1, m, p, r2 * s2)

    torch.cuda.synchronize()
    bound = n * EPS * product(A.abs(), X.abs())
    assert bool(((out - product(A, X)).abs() <= bound).all())


# (m, c) of one panel: edges of the 16-column blocks, of the 16-row blocks, of the
# register forms (256, 512, 1024, 1536 rows) and of the rows one call holds (2304)
PANELS = [(1, 1), (5, 3), (16, 16), (17, 16), (16, 17), (20, 40), (33, 31), (255, 17), (257, 33), (512, 64), (513, 65),
          (1025, 20), (1537, 7), (2304, 18), (2305, 18), (5000, 40)]


@pytest.mark.parametrize('m,c', PANELS)
def test_panel_qr(lib, m, c):
    """Householder QR of one panel: the second core of a two-core train is the
    panel's transpose.  Norm (R only) and, where Q is formed, ortho_right:
    orthonormal rows and the same tensor, to c * m eps (Householder QR is
    backward stable: a modest multiple of it is the error bound)."""
    from scikit_tt_amd.tensor_train import TT
    gen = torch.Generator(device='cuda').manual_seed(m * 1000 + c)
    a, b = _randn(gen, 1, 3, 1, c), _randn(gen, c, m, 1, 1)
    full = a.view(3, c) @ b.view(c, m)
    tol = 4 * m * c * EPS
    assert abs(TT([a, b]).norm() - float(full.norm())) <= tol * float(full.norm())
    t = TT([a.clone(), b.clone()]).ortho_right()
    q = t.device_cores[1].reshape(t.ranks[1], m)
    assert t.ranks == [1, min(m, c), 1]
    assert float((q @ q.T - torch.eye(min(m, c), dtype=torch.float64, device='cuda')).abs().max()) <= tol
    assert float((t.device_cores[0].view(3, -1) @ q - full).norm()) <= tol * float(full.norm())
    # the reflectors' sign convention: R's first diagonal entry is -sign(pivot) |column|, or the pivot itself where
    # nothing lies below it (a one-row panel)
    ref = b.view(c, m)[0]
    first = -torch.sign(ref[0]) * ref / ref.norm() if m > 1 else torch.ones_like(ref)
    assert float((q[0] - first).norm()) <= tol


def test_panel_qr_of_zero_and_repeated_columns(lib):
    """Exactly reduced columns (H_j = I) and rank-deficient panels keep Q orthonormal and the tensor."""
    from scikit_tt_amd.tensor_train import TT
    gen = torch.Generator(device='cuda').manual_seed(1)
    b = _randn(gen, 24, 300, 1, 1)
    b[5] = 0.0
    b[17:] = b[:7]
    a = _randn(gen, 1, 2, 1, 24)
    full = a.view(2, 24) @ b.view(24, 300)
    t = TT([a.clone(), b.clone()]).ortho_right()
    q = t.device_cores[1].reshape(24, 300)
    tol = 4 * 24 * 300 * EPS
    assert float((q @ q.T - torch.eye(24, dtype=torch.float64, device='cuda')).abs().max()) <= tol
    assert float((t.device_cores[0].view(2, 24) @ q - full).norm()) <= tol * float(full.norm())


@pytest.mark.parametrize('m,c', [(1, 1), (2, 2), (1, 7), (3, 40), (16, 16), (33, 33), (64, 64), (100, 49), (97, 97),
                                 (98, 98), (97, 300), (120, 120)])
@pytest.mark.parametrize('rank', [None, 3])
def test_truncated_svd_sizes(lib, m, c, rank):
    """Singular values to m c eps s0 of LAPACK's, orthonormal factors, the
    matrix back: the sizes around the lanes-per-pair steps and the largest
    factor held in LDS (97), full rank and rank 3 (equal zero columns)."""
    from scikit_tt_amd.utils import truncated_svd
    gen = torch.Generator(device='cuda').manual_seed(m * 1000 + c)
    k = min(m, c)
    Y = _randn(gen, m, c)
    if rank is not None:
        Y = _randn(gen, m, rank) @ _randn(gen, rank, c)
    u, s, v = truncated_svd(Y)
    ref = np.linalg.svd(Y.cpu().numpy(), compute_uv=False)
    tol = 4 * m * c * EPS * ref[0]
    assert s.shape[0] == k and np.abs(s.cpu().numpy() - ref).max() <= tol
    assert float(((u * s) @ v - Y).abs().max()) <= tol
    live = min(k, rank or k)
    for f in (u[:, :live].T, v[:live]):
        assert float((f @ f.T - torch.eye(live, dtype=torch.float64, device='cuda')).abs().max()) <= 4 * m * c * EPS


@pytest.mark.parametrize('scale', [1e-200, 1e200])
def test_truncated_svd_scale(lib, scale):
    """Entries whose squares leave the range of a double."""
    from scikit_tt_amd.utils import truncated_svd
    gen = torch.Generator(device='cuda').manual_seed(5)
    Y = _randn(gen, 24, 24).triu()  # its QR needs no reflections: the SVD alone is at stake
    u, s, v = truncated_svd(Y * scale)
    ref = np.linalg.svd(Y.cpu().numpy(), compute_uv=False)
    assert np.abs(s.cpu().numpy() / scale - ref).max() <= 4 * 24 * 24 * EPS * ref[0]


def test_truncated_svd_not_finite(lib):
    """A NaN stays in the result; the kept rank stays in range."""
    from scikit_tt_amd.utils import truncated_svd
    Y = torch.ones((6, 5), dtype=torch.float64, device='cuda')
    Y[2, 3] = float('nan')
    u, s, v = truncated_svd(Y)
    assert s.shape[0] <= 5 and bool(torch.isnan(s).any())


# (a, P, n, Q, b): local sizes around the lane, wave and row-half edges of the register LU (1 .. 96 unknowns)
LOCAL = [(1, 1, 1, 1, 1), (1, 2, 3, 1, 1), (2, 3, 4, 2, 2), (1, 1, 31, 1, 1), (2, 2, 4, 2, 4), (3, 1, 11, 2, 1),
         (4, 3, 4, 3, 4), (5, 2, 13, 1, 1), (4, 2, 4, 2, 6), (5, 1, 19, 1, 1), (1, 2, 2, 4, 48)]


@pytest.mark.parametrize('kb', [61, 0])
@pytest.mark.parametrize('a,P,n,Q,b', LOCAL)
def test_local_lu(lib, a, P, n, Q, b, kb):
    """Dense local solve against LAPACK, in registers and (no arena) in global
    memory; the residual of LU with partial pivoting is below N^2 eps |M| |v|
    for these sizes and growth factors."""
    from scikit_tt_amd import _lib
    gen = torch.Generator(device='cuda').manual_seed(a * 100 + b)
    L, A, R = _randn(gen, a, P, a), _randn(gen, P, n, n, Q), _randn(gen, b, Q, b)
    N = a * n * b
    f, v = _randn(gen, N), _randn(gen, N)
    M = torch.tensordot(torch.tensordot(L, A, dims=([1], [0])), R, dims=([4], [1])).permute(1, 2, 5, 0, 3, 4).reshape(N, N)
    ctx = _lib.context(0)
    assert lib.ttals_set_arena_kb(ctx, kb) == 0
    try:
        its = ctypes.c_int()
        assert lib.ttals_local_solve(ctx, None, a, P, n, Q, b, _ptr(L), _ptr(A), _ptr(R), _ptr(f), _ptr(v), 1, 0, 1e-12,
                                     100, ctypes.byref(its)) == 0
    finally:
        assert lib.ttals_set_arena_kb(ctx, 61) == 0
    res = float((M @ v - f).norm())
    assert res <= 4 * N * N * EPS * float(M.norm()) * float(v.norm())


# (a, P, n, Q, b): a local problem in 61 KB, two in the CU's LDS alone, two in
# neither (all but the first on eight waves); uneven ranks, odd sizes
PIECES = [(8, 2, 10, 2, 8), (9, 2, 10, 2, 10), (8, 3, 17, 2, 8), (8, 2, 33, 2, 8), (5, 1, 40, 3, 12)]


@pytest.mark.parametrize('a,P,n,Q,b', PIECES)
def test_pieces_of_local_problems(lib, a, P, n, Q, b):
    """Matvec and left interface update against torch, the local solves by
    their residual (both iterations stop at 1e-11), the lowest eigenvalue
    against a dense eigensolver (residual 1e-11 of the norm bounds its error).
    Operator: twice the identity plus a symmetric part of norm below 1/2."""
    from scikit_tt_amd import _lib
    gen = torch.Generator(device='cuda').manual_seed(a * 1000 + n)

    def sym(x):
        x = x + x.transpose(0, -1)
        return x / (P * Q * 2.0 * torch.linalg.matrix_norm(x.permute(1, 0, 2), 2).max())

    L, R, A = _randn(gen, a, P, a), _randn(gen, b, Q, b), _randn(gen, P, n, n, Q)
    L = sym(L)
    R = sym(R)
    A = A + A.transpose(1, 2)
    A = A / torch.linalg.matrix_norm(A.permute(0, 3, 1, 2), 2).max()
    L[:, 0, :] = torch.eye(a, device='cuda', dtype=torch.float64)
    R[:, 0, :] = torch.eye(b, device='cuda', dtype=torch.float64)
    A[0, :, :, 0] = 2.0 * torch.eye(n, device='cuda', dtype=torch.float64)
    L, R, A = L.contiguous(), R.contiguous(), A.contiguous()
    N = a * n * b
    f, x = _randn(gen, N), _randn(gen, N)

    def chain(l, o, r, v):
        t = torch.tensordot(l, v.view(a, n, b), dims=([0], [0]))  # P a' n b
        t = torch.tensordot(t, o, dims=([0, 2], [0, 2]))          # a' b m Q
        return torch.tensordot(t, r, dims=([1, 3], [0, 1])).reshape(N)

    def left(l, o, v):
        t = torch.tensordot(l, v.view(a, n, b), dims=([0], [0]))
        t = torch.tensordot(t, o, dims=([0, 2], [0, 2]))
        return torch.tensordot(t, v.view(a, n, b), dims=([0, 2], [0, 1])).contiguous()  # b Q b'

    ctx = _lib.context(0)
    y = torch.empty(N, dtype=torch.float64, device='cuda')
    assert lib.ttals_micro_matvec(ctx, None, a, P, n, Q, b, _ptr(L), _ptr(A), _ptr(R), _ptr(x), _ptr(y)) == 0
    terms = (a + P * n + b * Q + 3) * EPS
    assert bool(((y - chain(L, A, R, x)).abs() <= 2 * terms * chain(L.abs(), A.abs(), R.abs(), x.abs())).all())
    out = torch.empty(b, Q, b, dtype=torch.float64, device='cuda')
    assert lib.ttals_stack_left_op(ctx, None, a, P, n, Q, b, _ptr(L), _ptr(A), _ptr(x), _ptr(out)) == 0
    bound = 2 * (a + P * n + a * n + 3) * EPS * left(L.abs(), A.abs(), x.abs())
    assert bool(((out - left(L, A, x)).abs() <= bound).all())
    for method in (2, 3):
        v, its = torch.zeros_like(f), ctypes.c_int()
        assert lib.ttals_local_solve(ctx, None, a, P, n, Q, b, _ptr(L), _ptr(A), _ptr(R), _ptr(f), _ptr(v), method, 1,
                                     1e-11, 400, ctypes.byref(its)) == 0
        assert float((chain(L, A, R, v) - f).norm()) <= 2e-11 * float(f.norm())
    lam, its = ctypes.c_double(), ctypes.c_int()
    v = f.clone()
    assert lib.ttals_local_eig(ctx, None, a, P, n, Q, b, _ptr(L), _ptr(A), _ptr(R), _ptr(v), 0, 0.0, 1e-11, 4000,
                               ctypes.byref(lam), ctypes.byref(its)) == 0
    M = torch.stack([chain(L, A, R, e) for e in torch.eye(N, dtype=torch.float64, device='cuda')])
    want = float(torch.linalg.eigvalsh(0.5 * (M + M.T))[0])
    assert abs(lam.value - want) <= 1e-10 * float(M.norm())


def test_one_schedule_result_does_not_depend_on_the_batch(lib):
    """Systems on both sides of the line between the two single-workgroup
    kernels (10240 unknowns): in one batch, in another order and alone, the
    same bits."""
    from scikit_tt_amd import tensor_train as tt, workloads as W
    from scikit_tt_amd.solvers import sle
    rng = np.random.default_rng(3)
    sizes = [(4, 16, 25), (4, 4, 4), (4, 16, 26), (5, 3, 7), (4, 41, 16)]  # N: 10000, 64, 10816, 147, 10496
    A = tt.from_host_batch([W.shifted_operator(rng, d, n) for d, n, r in sizes])
    b = tt.from_host_batch([W.random_tt(rng, [n] * d, 3) for d, n, r in sizes])
    x = tt.from_host_batch([W.random_tt(rng, [n] * d, [1] + [r] * (d - 1) + [1]) for d, n, r in sizes])
    together = sle.als_batch(A, x, b)
    back = sle.als_batch(A[::-1], x[::-1], b[::-1])
    for s in range(len(sizes)):
        alone = sle.als_batch(A[s:s + 1], x[s:s + 1], b[s:s + 1])[0]
        for t in (together[s], back[len(sizes) - 1 - s]):
            assert t.ranks == alone.ranks
            for c1, c2 in zip(t.device_cores, alone.device_cores):
                assert torch.equal(c1, c2)
        full = alone.matricize()
        want = A[s].dot(alone).matricize()
        assert np.linalg.norm(want - b[s].matricize()) <= 0.5 * np.linalg.norm(b[s].matricize())
        assert np.isfinite(full).all()
