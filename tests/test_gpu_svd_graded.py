"""GPU: the Jacobi SVD on finite graded matrices, blocks of very different scale.

The blocks are decoupled by exact zeros and upper triangular (the QR before
the SVD leaves them as they are), so every block's singular values have the
error of that block alone: 4 m c eps of its largest one, the bound of the
other SVD tests, with the block's own LAPACK values as the reference.
"""
import numpy as np
import pytest

torch = pytest.importorskip('torch')
pytestmark = pytest.mark.gpu
EPS = 2.0 ** -52

CHAIN = np.array([[1.0, 1.0, 0.0], [0.0, 1.0, 1.0], [0.0, 0.0, 1.0]])  # equal column norms on the way
PAIR = np.array([[0.6, 0.8], [0.0, 1.0]])                              # two columns of one norm
UNEVEN = np.array([[1.0, 2.0], [0.0, 4.0]])


def _random(n, seed):
    return np.triu(np.random.default_rng(seed).standard_normal((n, n))) + 4.0 * np.eye(n)


CASES = [('chain', [(1.0, np.eye(1)), (s, CHAIN)]) for s in (1e-82, 1e-90, 1e-140)] + \
        [('pair', [(1.0, np.eye(1)), (s, PAIR)]) for s in (1e-85, 2.0 ** -300)] + \
        [('uneven', [(1.0, UNEVEN), (s, UNEVEN)]) for s in (1e-60, 1e-85, 1e-120)] + \
        [('random%d' % n, [(1.0, _random(n, 1)), (1e-85, _random(n + 1, 2)), (1e-130, _random(n, 3))])
         for n in (5, 13, 31)]


@pytest.fixture(scope='module', autouse=True)
def lib():
    assert torch.cuda.is_available(), 'GPU tests need a HIP device'
    from scikit_tt_amd import _lib
    torch.cuda.set_device(0)
    return _lib.load()


def _matrix(blocks):
    n = sum(len(b) for _, b in blocks)
    Y, at, spans = np.zeros((n, n)), 0, []
    for s, b in blocks:
        Y[at:at + len(b), at:at + len(b)] = s * b
        spans.append((at, at + len(b), s, np.linalg.svd(b, compute_uv=False)))
        at += len(b)
    return Y, spans


@pytest.mark.parametrize('name,blocks', CASES, ids=['%s-%.0e' % (n, b[-1][0]) for n, b in CASES])
def test_truncated_svd_of_graded_blocks(name, blocks):
    from scikit_tt_amd.utils import truncated_svd
    Y, spans = _matrix(blocks)
    n = len(Y)
    u, s, v = (t.cpu().numpy() for t in truncated_svd(torch.from_numpy(Y).cuda()))
    assert np.isfinite(u).all() and np.isfinite(s).all() and np.isfinite(v).all()
    back = (u * s) @ v
    for lo, hi, scale, ref in spans:
        tol = 4 * n * n * EPS * ref[0]
        assert np.abs(s[lo:hi] / scale - ref).max() <= tol
        assert np.abs(back[lo:hi, lo:hi] - Y[lo:hi, lo:hi]).max() <= tol * scale
    for f in (u.T, v):
        assert np.abs(f @ f.T - np.eye(n)).max() <= 4 * n * n * EPS
    # a relative threshold keeps what is above it: the first block
    u, s, v = (t.cpu().numpy() for t in truncated_svd(torch.from_numpy(Y).cuda(), threshold=1e-40, rel_truncation=True))
    lo, hi, scale, ref = spans[0]
    assert s.shape == (hi,) and np.abs(s - ref).max() <= 4 * n * n * EPS * ref[0]


@pytest.mark.parametrize('name,blocks', CASES[:5], ids=['%s-%.0e' % (n, b[-1][0]) for n, b in CASES[:5]])
def test_rounding_of_a_graded_core(name, blocks):
    """Rounding a two-core train whose second unfolding is graded keeps the dominant part."""
    from scikit_tt_amd.tensor_train import TT
    Y, spans = _matrix(blocks)
    n = len(Y)
    a = torch.eye(n, dtype=torch.float64, device='cuda').view(1, n, 1, n).contiguous()
    t = TT([a, torch.from_numpy(Y.T.copy()).cuda().view(n, n, 1, 1)]).ortho_right(threshold=1e-40)
    full = (t.device_cores[0].reshape(n, -1) @ t.device_cores[1].reshape(-1, n)).cpu().numpy()
    assert t.ranks == [1, spans[0][1], 1]
    assert np.isfinite(full).all() and np.abs(full - Y.T).max() <= 4 * n * n * EPS
