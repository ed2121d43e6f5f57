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
