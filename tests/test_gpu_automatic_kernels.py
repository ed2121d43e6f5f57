"""GPU: the kernels that a context chooses by itself, each test on a context on
which no arena was ever set (ttals_set_arena_kb keeps everything on the
four-wave kernels from then on).

That a case takes the eight-wave kernels shows in its bits: reductions over
512 threads round differently from those of a context pinned to the same
61 KB arena, while what stays on the four-wave kernels has the same bits."""
import ctypes

import numpy as np
import pytest

from tests import test_gpu_kernel_edges as edges

torch = pytest.importorskip('torch')
pytestmark = pytest.mark.gpu
EPS = edges.EPS


@pytest.fixture
def two(monkeypatch):
    """(library, automatic context, pinned context); the automatic one is the shared context of the test."""
    assert torch.cuda.is_available(), 'GPU tests need a HIP device'
    from scikit_tt_amd import _lib
    torch.cuda.set_device(0)
    lib = _lib.load()
    auto, pinned = _lib.new_context(0), _lib.new_context(0)
    assert lib.ttals_set_arena_kb(pinned, 61) == 0
    monkeypatch.setitem(_lib._ctx, 0, auto)
    yield lib, auto, pinned
    torch.cuda.synchronize()
    for ctx in (auto, pinned):
        lib.ttals_ctx_destroy(ctx)


_ptr = edges._ptr


def _solve(lib, ctx, dims, L, A, R, f, method, sym=0, tol=1e-11, maxit=400):
    v, its = torch.zeros_like(f), ctypes.c_int()
    rc = lib.ttals_local_solve(ctx, None, *dims, _ptr(L), _ptr(A), _ptr(R), _ptr(f), _ptr(v), method, sym, tol, maxit,
                               ctypes.byref(its))
    return rc, v


def _operands(dims, seed):
    """N(0, 1) operator pieces, the first ones near multiples of the identity."""
    a, P, n, Q, b = dims
    gen = torch.Generator(device='cuda').manual_seed(seed)

    def near(k, s, scale):
        x = 0.1 * edges._randn(gen, k, s, k)
        x[:, 0] += scale * torch.eye(k, dtype=torch.float64, device='cuda')
        return x

    A = 0.1 * edges._randn(gen, P, n, n, Q)
    A[0, :, :, 0] += 4.0 * torch.eye(n, dtype=torch.float64, device='cuda')
    return near(a, P, 1.0), A, near(b, Q, 1.0), edges._randn(gen, a * n * b)


@pytest.mark.parametrize('dims', edges.PIECES)
def test_pieces(two, dims):
    lib, auto, pinned = two
    edges.test_pieces_of_local_problems(lib, *dims)
    L, A, R, f = _operands(dims, sum(dims))
    (r0, v0), (r1, v1) = (_solve(lib, ctx, dims, L, A, R, f, 3) for ctx in (auto, pinned))
    assert r0 == r1 == 0
    fits_61_kb = dims == edges.PIECES[0]
    assert torch.equal(v0, v1) == fits_61_kb


# local problems off the 61 KB arena of one wave's, two waves' and eight waves' columns of the eight-wave register LU
# (32, 64, 96 unknowns), around its row half at 64 and with a partial last column block
@pytest.mark.parametrize('dims', [(1, 1, 1, 10, 30), (1, 2, 1, 9, 32), (3, 2, 1, 9, 11), (2, 8, 1, 9, 31),
                                  (2, 1, 1, 9, 32), (1, 1, 1, 2, 65), (1, 1, 1, 1, 95), (1, 1, 2, 4, 48),
                                  (2, 1, 1, 4, 48), (3, 1, 1, 9, 32), (1, 9, 1, 3, 83)])
def test_register_lu_of_eight_waves(two, dims):
    lib, auto, pinned = two
    a, P, n, Q, b = dims
    if a * P * a + P * n * n * Q + b * Q * b <= 61 * 128:  # pieces of 61 KB and more only
        Q = -(-(61 * 128) // (b * b)) + 1
        dims = (a, P, n, Q, b)
    N = a * n * b
    gen = torch.Generator(device='cuda').manual_seed(N)
    L, A, R = edges._randn(gen, a, P, a), edges._randn(gen, P, n, n, Q), edges._randn(gen, b, Q, b)
    f = edges._randn(gen, N)
    M = torch.tensordot(torch.tensordot(L, A, dims=([1], [0])), R, dims=([4], [1]))
    M = M.permute(1, 2, 5, 0, 3, 4).reshape(N, N)
    rc, v = _solve(lib, auto, dims, L, A, R, f, 1)
    assert rc == 0
    assert float((M @ v - f).norm()) <= 4 * N * N * EPS * float(M.norm()) * float(v.norm())
    # the same route with an iteration's reductions: other bits than with four waves
    ops = _operands(dims, N)
    (r0, v0), (r1, v1) = (_solve(lib, ctx, dims, *ops, 3) for ctx in (auto, pinned))
    assert r0 == r1 == 0 and not torch.equal(v0, v1)


@pytest.mark.parametrize('N', [95, 96])
def test_register_lu_pivots_in_the_upper_row_half(two, N):
    """M is R^T for one-entry L and A: the largest entries on the antidiagonal,
    so that the first pivots lie in the rows from 64 on, then in those below."""
    lib, auto, _ = two
    gen = torch.Generator(device='cuda').manual_seed(N)
    one = torch.ones(1, dtype=torch.float64, device='cuda')
    M = 0.1 * edges._randn(gen, N, N) + 10.0 * torch.eye(N, dtype=torch.float64, device='cuda').flip(0)
    f = edges._randn(gen, N)
    R = M.t().contiguous().view(N, 1, N)
    rc, v = _solve(lib, auto, (1, 1, 1, 1, N), one, one, R, f, 1)
    assert rc == 0
    # no growth (each pivot ten times its column): the backward error of one sweep over N rows
    assert float((M @ v - f).norm()) <= 4 * N * EPS * float(M.norm()) * float(v.norm())
    # a zero column in the upper half of the columns: singular, found at that step
    M[:, 70] = 0.0
    R = M.t().contiguous().view(N, 1, N)
    rc, v = _solve(lib, auto, (1, 1, 1, 1, N), one, one, R, f, 1)
    from scikit_tt_amd import _lib
    assert rc == _lib.S_SINGULAR


def test_one_schedule(two):
    """The bits of a batch do not depend on its order and company with systems
    on both kernels; the small ones have those of the four-wave kernel, the
    ones of 10240 unknowns and more do not."""
    lib, auto, pinned = two
    edges.test_one_schedule_result_does_not_depend_on_the_batch(lib)
    from scikit_tt_amd import _lib, tensor_train as tt, workloads as W
    from scikit_tt_amd.solvers import sle
    rng = np.random.default_rng(7)
    sizes = [(4, 16, 25), (4, 16, 26), (5, 3, 7), (3, 100, 11), (3, 92, 10)]  # N: 10000, 10816, 147, 12100, 9200
    A = tt.from_host_batch([W.shifted_operator(rng, d, n) for d, n, r in sizes])
    b = tt.from_host_batch([W.random_tt(rng, [n] * d, 3, scale=1.0 / np.sqrt(n)) for d, n, r in sizes])
    x = tt.from_host_batch([W.random_tt(rng, [n] * d, [1] + [r] * (d - 1) + [1], scale=1.0 / np.sqrt(n))
                            for d, n, r in sizes])
    here = sle.als_batch(A, x, b)
    _lib._ctx[0] = pinned
    there = sle.als_batch(A, x, b)
    _lib._ctx[0] = auto
    for s, (d, n, r) in enumerate(sizes):
        same = all(torch.equal(c, e) for c, e in zip(here[s].device_cores, there[s].device_cores))
        assert same == (n * r * r < 10240), (s, same)


def _time_us(lib, entry, ctx, args):
    best = float('inf')
    for _ in range(5):
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        for _ in range(20):
            assert getattr(lib, entry)(ctx, None, *args) == 0
        e1.record()
        e1.synchronize()
        best = min(best, e0.elapsed_time(e1) * 50.0)
    return best


@pytest.mark.parametrize('entry,dims', [('ttals_stack_left_rhs', (32, 4, 64, 1, 4)),
                                        ('ttals_stack_left_rhs', (16, 3, 16, 1, 48)),
                                        ('ttals_stack_left_op', (16, 2, 64, 1, 4)),
                                        ('ttals_stack_right_op', (3, 1, 64, 3, 16)),
                                        ('ttals_stack_right_rhs', (32, 4, 64, 1, 4)),
                                        ('ttals_micro_rhs', (16, 4, 64, 4, 2))])
def test_global_memory_pieces_are_no_slower(two, entry, dims):
    """The same result as on the four-wave kernel, and no slower (the first one:
    139 us with four waves, 181 us with eight while half of them worked on rows
    past the output's edge, 130 us since)."""
    lib, auto, pinned = two
    a, p, n, q, b = dims
    gen = torch.Generator(device='cuda').manual_seed(sum(dims))
    op = entry.endswith('_op')
    left = edges._randn(gen, *((a, p, a) if op else (p, a)))
    right = edges._randn(gen, *((b, q, b) if op else (q, b)))
    core = edges._randn(gen, p, n, n, q) if op else edges._randn(gen, p, n, q)
    x = edges._randn(gen, a, n, b)
    outs = [torch.full((a * n * b if 'micro' in entry else (b * q * b if 'left' in entry else a * p * a) if op else
                        (q * b if 'left' in entry else p * a),), float('nan'), dtype=torch.float64, device='cuda')
            for _ in range(2)]
    us = []
    for ctx, out in zip((auto, pinned), outs):
        first = [left, core, right, out] if 'micro' in entry else \
            [left if 'left' in entry else right, core, x, out]
        us.append(_time_us(lib, entry, ctx, (a, p, n, q, b, *map(_ptr, first))))
    print('  %.1f us, four waves %.1f us' % tuple(us), flush=True)
    # sums of K N(0, 1) products: K eps times the sum of the magnitudes, which exceeds the largest sum by less than
    # the number of its terms' square root
    bound = 4 * (a + p * n + a * n + n * q + n * b) * EPS * float(outs[1].abs().max()) * a * b * n * p * q
    assert float((outs[0] - outs[1]).abs().max()) <= bound
    assert us[0] <= 1.12 * us[1]
