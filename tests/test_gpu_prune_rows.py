"""Final RobustPrune at the edges of its staged path: vector widths around a
wave and the LDS limit (204 coordinates), odd and unaligned ones, rows of 1 to
65 neighbours, ids past the set, duplicates, self-loops, equal distances.  Bar:
identical to the oracle."""
import numpy as np
import pytest
import torch

from gpu_helpers import require_gpu
from shear_amd import graph as G

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    return require_gpu()


def _table(rng, n, stride):
    t = rng.integers(0, n + 3, (n, stride)).astype(np.uint32)
    c = rng.integers(0, stride + 2, n).astype(np.uint32)
    t[::7, 0] = np.arange(0, n, 7)
    if stride > 2:
        t[::5, 1] = t[::5, 2]
    return t, c


def _check(gpu, orc, x, t, c, dev_x=None, **kw):
    out, cnt = G.robust_prune(torch.from_numpy(x).to(gpu) if dev_x is None else dev_x,
                              torch.from_numpy(t.view(np.int32)).to(gpu), torch.from_numpy(c.view(np.int32)).to(gpu), **kw)
    torch.cuda.synchronize()
    wt, wc = orc.robust_prune(x, t, c, **kw)
    assert np.array_equal(cnt.cpu().numpy().view(np.uint32), wc)
    assert np.array_equal(out.cpu().numpy().view(np.uint32), wt)


@pytest.mark.parametrize("dim", [1, 3, 4, 5, 31, 32, 63, 64, 65, 100, 127, 128, 129, 200, 204, 205, 208, 260])
@pytest.mark.parametrize("stride", [1, 40, 64, 65])
def test_widths(gpu, orc, dim, stride):
    rng = np.random.default_rng(dim * 100 + stride)
    x = rng.standard_normal((300, dim)).astype(np.float32)
    t, c = _table(rng, 300, stride)
    _check(gpu, orc, x, t, c, saturate=bool(dim % 2))


@pytest.mark.parametrize("kw", [dict(max_degree=5), dict(max_degree=100, saturate=True), dict(max_occlusion=1),
                                dict(max_occlusion=63, alpha=1.7), dict(alpha=0.5), dict(alpha=1.0, saturate=True)])
def test_options_with_equal_distances(gpu, orc, kw):
    rng = np.random.default_rng(3)
    x = rng.integers(0, 3, (400, 6)).astype(np.float32)
    t, c = _table(rng, 400, 64)
    _check(gpu, orc, x, t, c, **kw)


@pytest.mark.parametrize("dim", [64, 65])
def test_unaligned_vectors(gpu, orc, dim):
    rng = np.random.default_rng(4)
    x = rng.standard_normal((200, dim)).astype(np.float32)
    flat = torch.empty(200 * dim + 1, device=gpu)
    flat[1:] = torch.from_numpy(x.reshape(-1)).to(gpu)
    t, c = _table(rng, 200, 64)
    _check(gpu, orc, x, t, c, dev_x=flat[1:].view(200, dim))
