"""GPU: the multi-workgroup (gang) engine against the fused one-workgroup
engine and the oracle, FP64 and mixed precision (FP32 Krylov iterations with
FP64 refinement of the local residual).

Both engines solve every local problem to the relative residual 1e-12 by
different Krylov paths (the gang engine uses Krylov also where the fused
engine factors small problems densely), so iterates agree to ~1e-9, not bit
for bit; ranks are identical.  The mixed path must agree with the FP64 path
to the same level, since it refines to the same local tolerance.
"""
import time

import numpy as np
import pytest

from oracle import tt_ops, sle_als
from scikit_tt_amd import workloads as W

torch = pytest.importorskip('torch')
pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def env():
    assert torch.cuda.is_available(), 'GPU tests need a HIP device'
    from scikit_tt_amd import _lib
    torch.cuda.set_device(0)
    _lib.load()


def _tt(cores):
    from scikit_tt_amd.tensor_train import TT
    return TT([np.asarray(c) for c in cores])


def _reldiff(x, y):
    return tt_ops.norm(tt_ops.sub(x, y)) / tt_ops.norm(y)


@pytest.mark.parametrize('gang', [1, 3, 0])
@pytest.mark.parametrize('precision', ['fp64', 'mixed'])
def test_gang_laplace_vs_oracle(env, gang, precision):
    """Symmetric operator (CG path), uneven gang splits of the rank rows."""
    import scikit_tt_amd.solvers.sle as sle
    print('case laplace d=6 n=5 r=5 gang=%d %s' % (gang, precision), flush=True)
    A, x0, b = W.laplace_small(seed=4, d=6, n=5, rank=5)
    (x,), (info,) = sle.als_gang([_tt(A)], [_tt(x0)], [_tt(b)], repeats=2, precision=precision, gang=gang,
                                 return_info=True)
    assert info.status == 0, info
    xr = sle_als.als(A, x0, b, repeats=2)
    assert x.ranks == tt_ops.ranks_of(xr)
    assert _reldiff(x.cores[:], xr) < 1e-8


@pytest.mark.parametrize('precision', ['fp64', 'mixed'])
def test_gang_nonsymmetric_batch_vs_fused(env, precision):
    """Non-symmetric operators (GMRES path), several gangs in one launch."""
    import scikit_tt_amd.solvers.sle as sle
    print('case shifted batch %s' % precision, flush=True)
    systems = [W.shifted_batch_instance(s, d_range=(4, 7), n_choices=(3, 4), r_range=(3, 9)) for s in range(4)]
    As = [_tt(A) for A, _, _ in systems]
    Xs = [_tt(x) for _, x, _ in systems]
    Bs = [_tt(b) for _, _, b in systems]
    gang_sols, infos = sle.als_gang(As, Xs, Bs, repeats=2, precision=precision, gang=2, return_info=True)
    fused = sle.als_batch(As, Xs, Bs, repeats=2)
    assert (infos.array['status'] == 0).all(), infos.array['status']
    for k in range(len(systems)):
        assert gang_sols[k].ranks == fused[k].ranks
        assert _reldiff(gang_sols[k].cores[:], fused[k].cores[:]) < 1e-8, k


def test_gang_full_size_laplace_mixed_vs_fp64(env):
    """The large Laplacian configuration (d=20, n=32, rank 32, rank-4 N(0,1)
    rhs): FP64 and mixed precision on one gang each, rel.res of both from the
    FP64 residual kernel, the mixed result's distance to the FP64 one."""
    import scikit_tt_amd.solvers.sle as sle
    from scikit_tt_amd.tensor_train import residual_norms
    A, x0, b = W.laplace_large()
    tA, tx, tb = _tt(A), _tt(x0), _tt(b)
    out = {}
    for prec in ('fp64', 'mixed'):
        print('case laplace_large %s' % prec, flush=True)
        torch.cuda.synchronize()
        t = time.perf_counter()
        (x,), (info,) = sle.als_gang([tA], [tx], [tb], repeats=2, precision=prec, return_info=True)
        torch.cuda.synchronize()
        dt = time.perf_counter() - t
        res, bn = residual_norms([tA], [x], [tb])
        out[prec] = (x, res[0] / bn[0], dt, info)
        print('  %s: 2 sweeps %.3f s, rel.res %.3e, krylov %d' % (prec, dt, res[0] / bn[0], info.krylov_iters),
              flush=True)
    assert out['fp64'][1] < 2e-9
    assert out['mixed'][1] < 1.1 * out['fp64'][1] + 1e-12
    d = _reldiff(out['mixed'][0].cores[:], out['fp64'][0].cores[:])
    print('  mixed vs fp64 iterate: %.3e' % d, flush=True)
    assert d < 1e-7


@pytest.mark.parametrize('gang', [2, 5])
def test_gang_rank_deficient_panels(env, gang):
    """A = alpha I (no perturbation) and a rank-2 right-hand side with a
    rank-6 start: the solution has rank 2, the new cores' panels are rank
    deficient (relative singular values ~1e-16), the Cholesky QR's pivots
    fail and the split Householder QR takes over (the reference's QR is
    Householder too).  The completion of such a basis is arbitrary, so the
    cores are not compared with the oracle's; both solve the system to
    rounding and agree as tensors, with the same ranks."""
    import scikit_tt_amd.solvers.sle as sle
    from scikit_tt_amd.tensor_train import residual_norms
    print('case rank-deficient panels gang=%d' % gang, flush=True)
    rng = np.random.default_rng(11)
    A = W.shifted_operator(rng, 6, 4, sigma=0.0)
    b = W.random_tt(rng, [4] * 6, 2)
    x0 = W.random_tt(rng, [4] * 6, 6)
    tA, tb = _tt(A), _tt(b)
    (x,), (info,) = sle.als_gang([tA], [_tt(x0)], [tb], repeats=2, gang=gang, return_info=True)
    assert info.status == 0, info
    xr = sle_als.als(A, x0, b, repeats=2)
    assert x.ranks == tt_ops.ranks_of(xr)
    res, bn = residual_norms([tA], [x], [tb])
    rr = tt_ops.norm(tt_ops.sub(tt_ops.dot(A, xr), b)) / tt_ops.norm(b)
    print('  rel.res gang %.2e oracle %.2e' % (res[0] / bn[0], rr), flush=True)
    assert res[0] / bn[0] < 1e-10 and rr < 1e-10
    assert _reldiff(x.cores[:], xr) < 1e-9


# both sides of the lines of the on-chip matvec: operator rank (3 and 4) times rows
# of a member 6 and 8, 9 and 12, members without rows, remainders of the unrolled
# loads, mode sizes whose pieces fit 136 KB in FP64, in FP32 alone and not at all
@pytest.mark.parametrize('precision', ['fp64', 'mixed'])
@pytest.mark.parametrize('d,n,r,gang', [(4, 5, 8, 4), (4, 5, 9, 4), (4, 6, 10, 2), (4, 7, 17, 17), (3, 36, 5, 5),
                                        (3, 54, 5, 5), (3, 66, 5, 5), (3, 3, 2, 5)])
def test_gang_few_rows_vs_one_workgroup(env, precision, d, n, r, gang):
    import scikit_tt_amd.solvers.sle as sle
    print('case d=%d n=%d r=%d gang=%d %s' % (d, n, r, gang, precision), flush=True)
    # -Laplacian + its norm: symmetric (CG), condition number below 2, so that local residuals of 1e-12 are local
    # errors of 2e-12 and the engines' solutions agree to the module's 1e-8; and a non-symmetric one (GMRES)
    lap = W.tt_sum(W.laplace_operator(d, n), W.identity_operator([n] * d, d * np.linalg.norm(W.laplace_1d(n), 2)))
    for op in (lap, W.shifted_operator(np.random.default_rng(n), d, n, alpha=10.0 * d)):
        A = _tt(op)
        rng = np.random.default_rng(n + r)
        b = _tt(W.random_tt(rng, [n] * d, 2, scale=1.0 / np.sqrt(n)))
        ranks = [1] + [min(r, n ** min(k, d - k)) for k in range(1, d)] + [1]
        x0 = _tt(W.right_orthonormal(W.random_tt(rng, [n] * d, ranks)))
        (x,), (info,) = sle.als_gang([A], [x0], [b], precision=precision, gang=gang, return_info=True)
        (y,) = sle.als_batch([A], [x0], [b])
        assert info.status == 0, info
        assert x.ranks == y.ranks
        assert _reldiff(x.cores[:], y.cores[:]) < 1e-8


# the split Householder QR: less than a block of 16 columns, a block and one more,
# two and one more, members without columns, 2304 rows (register blocks) and 2640
# (LDS blocks)
@pytest.mark.parametrize('d,n,r,gang', [(4, 6, 15, 2), (4, 6, 17, 3), (3, 40, 33, 5), (4, 5, 18, 32), (3, 72, 32, 2),
                                        (3, 80, 33, 2)])
def test_gang_rank_deficient_blocks(env, d, n, r, gang):
    """alpha I x = b with b of rank 2 held at rank r: every panel is rank
    deficient; the solution is b / alpha (bounds as above)."""
    import scikit_tt_amd.solvers.sle as sle
    print('case rank-deficient blocks d=%d n=%d r=%d gang=%d' % (d, n, r, gang), flush=True)
    rng = np.random.default_rng(r)
    A = W.shifted_operator(rng, d, n, sigma=0.0)
    b = W.random_tt(rng, [n] * d, 2, scale=1.0 / np.sqrt(n))
    ranks = [1] + [min(r, n ** min(k, d - k)) for k in range(1, d)] + [1]
    x0 = W.random_tt(rng, [n] * d, ranks, scale=1.0 / np.sqrt(n))
    (x,), (info,) = sle.als_gang([_tt(A)], [_tt(x0)], [_tt(b)], repeats=2, gang=gang, return_info=True)
    assert info.status == 0, info
    want = [c / float(d) if i == 0 else c for i, c in enumerate(b)]
    assert _reldiff(x.cores[:], want) < 1e-9
    for c in x.cores[1:]:  # right-orthonormal
        m = np.asarray(c).reshape(c.shape[0], -1)
        assert np.abs(m @ m.T - np.eye(c.shape[0])).max() < 1e-12
