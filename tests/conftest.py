import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)
GOLDEN = os.path.join(ROOT, 'tests', 'golden')


def pytest_configure(config):
    config.addinivalue_line('markers', 'gpu: needs a HIP device (MI355X)')
    config.addinivalue_line('markers', 'slow: long-running test')


def load_golden(name):
    """Golden fixture written by tests/golden/make_golden.py (plain arrays, no pickle)."""
    z = np.load(os.path.join(GOLDEN, name + '.npz'), allow_pickle=False)
    out = {k: z[k] for k in z.files}

    def tt(prefix):
        return [out['%s_%d' % (prefix, i)] for i in range(int(out[prefix + '_order']))]

    out['tt'] = tt
    return out


@pytest.fixture
def golden():
    return load_golden


@pytest.fixture(scope='module', autouse=True)
def contexts_of_the_module():
    """Every module gets shared engine contexts of its own: what a test sets on
    one (an arena of its choice switches the automatic choice of kernels off
    for good) ends with the module."""
    from scikit_tt_amd import _lib
    saved = dict(_lib._ctx)
    _lib._ctx.clear()
    yield
    if _lib._ctx:
        import torch
        torch.cuda.synchronize()
        for ctx in _lib._ctx.values():
            _lib.load().ttals_ctx_destroy(ctx)
    _lib._ctx.clear()
    _lib._ctx.update(saved)
