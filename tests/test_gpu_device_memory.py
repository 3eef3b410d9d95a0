"""The library's memory beside a torch cache that holds nearly all of the card,
and reservoirs that torch has no room for.  Nothing here touches the memory it
reserves."""
import numpy as np
import pytest
import torch

from gpu_helpers import require_gpu
from shear_amd import edges as E
from shear_amd import hashprune as H
from shear_amd import subtree as S
from shear_amd import tessa as T
from test_gpu_hashprune import _gpu_slots, _same

pytestmark = pytest.mark.gpu

GIB = 1 << 30


@pytest.fixture
def gpu():
    dev = require_gpu()
    torch.cuda.empty_cache()
    yield dev
    torch.cuda.empty_cache()


def _fill_cache(leave):
    """Torch's cache (unused blocks) takes all but `leave` bytes of what is free."""
    free = torch.cuda.mem_get_info()[0]
    block = torch.empty(free - leave, dtype=torch.uint8, device="cuda")
    del block
    assert torch.cuda.mem_get_info()[0] <= leave + GIB


def test_session_upload_beside_a_full_cache(gpu):
    rows, dim = 6 << 20, 1024
    sq8 = T.Sq8Matrix(torch.zeros((rows, dim), dtype=torch.int8, device=gpu), torch.ones(rows, device=gpu),
                      torch.zeros(rows, device=gpu), dim)
    gids = torch.arange(rows, dtype=torch.int32, device=gpu)
    sess = S.SubtreeSession(0)
    _fill_cache(2 * GIB)
    sess.upload_device(sq8, gids)  # 6 GiB
    assert sess.rows == rows


def test_large_reservoirs_are_not_torchs(gpu):
    points = H.MAX_CACHED_BYTES // 640 + 1  # one point over the bound
    _fill_cache(4 * GIB)
    with H.HashPruneReducer(points, 64) as hp:
        assert torch.cuda.memory_reserved() < GIB  # the cache went back for them, and holds none of them
        r = np.zeros(3, E.EDGE_RECORD_DTYPE)
        r["src"], r["dst"], r["hash"] = points - 1, [7, 8, 9], [1, 2, 3]
        r["dist"] = [0.5, 0.25, 0.75]
        hp.insert(r)
        t, c = hp.neighbors()
        assert int(c.sum()) == 3 and t[points - 1, :3].cpu().tolist() == [7, 8, 9]


def test_reservoirs_without_torchs_memory(gpu, orc, monkeypatch):
    # torch has none left (or may use no more of it): the library allocates them, as its own error says if it cannot
    rng = np.random.default_rng(3)
    r = np.zeros(4000, E.EDGE_RECORD_DTYPE)
    r["src"], r["dst"], r["hash"] = rng.integers(0, 90, 4000), rng.integers(0, 90, 4000), rng.integers(0, 500, 4000)
    r["dist"] = rng.random(4000)
    r = r[np.argsort(r["src"], kind="stable")]
    first = np.searchsorted(r["src"], np.arange(90))
    segs = np.stack([np.arange(90), first, np.zeros(90, np.int64), np.r_[first[1:], 4000] - first], 1).astype(np.uint32)
    rec = torch.from_numpy(r.view(np.uint8).view(np.int32).reshape(-1, 4).copy()).to(gpu)
    real = torch.empty

    def empty(*args, **kw):
        if kw.get("dtype") is torch.uint8:
            raise torch.cuda.OutOfMemoryError("no memory")
        return real(*args, **kw)

    monkeypatch.setattr(torch, "empty", empty)
    with H.HashPruneReducer(90, 20) as hp:
        hp.insert_segments(rec, torch.from_numpy(segs.view(np.int32)).to(gpu))
        _same(_gpu_slots(hp), orc.hashprune_reduce(90, 20, r), "reservoirs of the library's")
