"""GPU: the TT core product at its dispatch rule (by columns / by elements).

Tolerance: a sum of n products in any order differs from another order by
less than n eps times the sum of the products' magnitudes.
"""
import ctypes

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


def _randn(gen, *shape):
    return torch.randn(*shape, dtype=torch.float64, device='cuda', generator=gen)


def _call(lib, dims, A, X, out):
    assert lib.ttals_core_product(None, *dims, _ptr(A), _ptr(X), _ptr(out)) == 0


# (r1, m, n, r2, s1, p, s2): one column, a few, one row, both sides of the line at one n, n above 32, odd sizes
SHAPES = [(1, 1, 1, 1, 1, 1, 1), (48, 16, 16, 48, 1, 1, 1), (1, 1, 64, 200, 1, 1, 200), (7, 3, 5, 9, 1, 1, 2),
          (20, 64, 64, 20, 1, 1, 3), (3, 1, 29, 81, 10, 7, 1), (4, 16, 16, 4, 1, 1, 7), (4, 16, 16, 4, 19, 1, 19),
          (4, 16, 16, 4, 60, 1, 60), (300, 2, 2, 300, 1, 1, 1), (5, 3, 33, 2, 11, 2, 5), (1, 40, 70, 1, 1, 1, 1), (2, 1, 3, 1, 300, 2, 301)]


@pytest.mark.parametrize('dims', SHAPES)
def test_core_product_forms(lib, dims):
    r1, m, n, r2, s1, p, s2 = dims
    gen = torch.Generator(device='cuda').manual_seed(sum(dims))
    A, X, out = _randn(gen, r1, m, n, r2), _randn(gen, s1, n, p, s2), _randn(gen, r1 * s1, m, p, r2 * s2)
    _call(lib, dims, A, X, out)

    def product(a, x):
        return torch.tensordot(a, x, dims=([2], [1])).permute(0, 3, 1, 4, 2, 5).reshape(out.shape)

    bound = n * EPS * product(A.abs(), X.abs())
    assert bool(((out - product(A, X)).abs() <= bound).all())


def _time_us(lib, dims):
    r1, m, n, r2, s1, p, s2 = dims
    gen = torch.Generator(device='cuda').manual_seed(1)
    A, X = _randn(gen, r1, m, n, r2), _randn(gen, s1, n, p, s2)
    out = torch.empty(r1 * s1, m, p, r2 * s2, dtype=torch.float64, device='cuda')
    best = float('inf')
    for _ in range(5):
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        for _ in range(20):
            _call(lib, dims, A, X, out)
        e1.record()
        e1.synchronize()
        best = min(best, e0.elapsed_time(e1) * 50.0)
    return best


@pytest.mark.parametrize('few,many', [((128, 16, 16, 128, 1, 1, 1), (4, 16, 16, 4, 32, 1, 32)),
                                      ((1, 1, 64, 200, 1, 1, 200), (4, 16, 16, 4, 12, 1, 12))])
def test_few_columns_keep_the_chip_busy(lib, few, many):
    """An operator times a train of rank 1, and the first core of an inner
    product, take no more than four times as long as a product of as many
    elements with many columns (28 times where each column had one thread)."""
    a, b = _time_us(lib, few), _time_us(lib, many)
    print('  %.1f us and %.1f us' % (a, b), flush=True)
    assert a <= 4.0 * max(b, 5.0)


def test_more_columns_than_a_launch_has_threads(lib):
    """2^32 and more columns (34 GB each of X and out)."""
    s1 = s2 = 65537
    free, _ = torch.cuda.mem_get_info()
    if free < 80 << 30:
        pytest.skip('needs 80 GB of device memory')
    X = torch.empty(s1, 1, 1, s2, dtype=torch.float64, device='cuda')
    X.view(s1, s2).copy_(torch.arange(s2, dtype=torch.float64, device='cuda').expand(s1, s2))
    X.view(s1, s2)[:, 0] = torch.arange(s1, dtype=torch.float64, device='cuda')
    out = torch.empty(s1, 1, 1, s2, dtype=torch.float64, device='cuda')
    A = torch.full((1, 1, 1, 1), 2.0, dtype=torch.float64, device='cuda')
    _call(lib, (1, 1, 1, 1, s1, 1, s2), A, X, out)
    for lo in range(0, s1, 4096):
        assert bool((out[lo:lo + 4096] == 2.0 * X[lo:lo + 4096]).all())
    del X, out
    torch.cuda.empty_cache()
