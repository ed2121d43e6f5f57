"""GPU: panels and factors at the lines below which the QR and the Jacobi SVD
take their forms for small sizes, held to the bounds of the other sizes."""
import pytest

from tests import test_gpu_kernel_edges as edges

torch = pytest.importorskip('torch')
pytestmark = pytest.mark.gpu
lib = edges.lib


# the register QR's boxes (32 x 32, 64 x 16), the column sweep's (256 x 1, 256 x 2 from 65 rows), both sides
@pytest.mark.parametrize('m,c', [(2, 1), (64, 1), (256, 1), (257, 1), (64, 2), (65, 2), (256, 2), (257, 2), (1, 5),
                                 (32, 32), (33, 32), (32, 33), (64, 16), (65, 16), (64, 17), (16, 40), (7, 3)])
def test_panels(lib, m, c):
    edges.test_panel_qr(lib, m, c)


# one wave up to 16 columns and rows
@pytest.mark.parametrize('m,c', [(1, 9), (2, 3), (4, 4), (7, 7), (8, 8), (9, 9), (15, 15), (16, 15), (16, 16), (17, 16),
                                 (16, 17), (17, 17), (300, 16), (300, 17)])
@pytest.mark.parametrize('rank', [None, 1])
def test_factors(lib, m, c, rank):
    edges.test_truncated_svd_sizes(lib, m, c, rank)


@pytest.mark.parametrize('scale', [1e-200, 1e200])
def test_scale(lib, scale):
    """Entries whose squares leave the range of a double, in the one-wave form."""
    import numpy as np
    from scikit_tt_amd.utils import truncated_svd
    gen = torch.Generator(device='cuda').manual_seed(6)
    Y = torch.randn(9, 9, dtype=torch.float64, device='cuda', generator=gen).triu()  # no reflections in its QR
    u, s, v = truncated_svd(Y * scale)
    ref = np.linalg.svd(Y.cpu().numpy(), compute_uv=False)
    assert np.abs(s.cpu().numpy() / scale - ref).max() <= 4 * 9 * 9 * edges.EPS * ref[0]
