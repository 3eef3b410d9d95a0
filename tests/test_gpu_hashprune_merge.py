"""The HashPrune merge at the edges of its batches (256 records of a source at
a time), its hash buckets and its border ties, against the oracle's record by
record reservoirs.  Bar: bit-identical slots."""
import numpy as np
import pytest
import torch

from gpu_helpers import require_gpu
from shear_amd import edges as E
from shear_amd import hashprune as H
from test_gpu_hashprune import _gpu_slots, _same

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    return require_gpu()


def _records(rng, counts, dists, targets, hashes):
    n = int(sum(counts))
    r = np.zeros(n, E.EDGE_RECORD_DTYPE)
    r["src"] = np.repeat(np.arange(len(counts)), counts)
    r["dst"] = rng.choice(targets, n)
    r["hash"] = rng.choice(hashes, n)
    r["dist"] = rng.choice(dists, n)
    return r


def _segments(r, rng, pieces):
    """One segment per source, or each source's run cut into `pieces` (some empty)."""
    segs = []
    for s in np.unique(r["src"]):
        at = np.nonzero(r["src"] == s)[0]
        a, b = int(at[0]), int(at[-1]) + 1
        cuts = np.sort(rng.integers(a, b + 1, pieces - 1))
        for i, j in zip(np.r_[a, cuts], np.r_[cuts, b]):
            segs.append((s, i, 0, j - i))
    return np.array(segs, np.uint32)[rng.permutation(len(segs))]


EDGE_COUNTS = [1, 63, 64, 65, 128, 191, 192, 193, 255, 256, 257, 511, 512, 513, 1025]
SPREAD = np.linspace(0.01, 3.0, 5000, dtype=np.float32)
# every class total_cmp orders, an all-ones NaN among them
ODD = np.array([0x00000000, 0x80000000, 0x00000001, 0x7F800000, 0xFF800000, 0x7FC00000, 0xFFFFFFFF, 0x7FFFFFFF,
                0x3F800000, 0xBF800000], np.uint32).view(np.float32)


@pytest.mark.parametrize("l_max", [1, 63, 64, 65, 128, 256])
@pytest.mark.parametrize("pieces", [1, 3, 64, 65, 130])
def test_batch_edges(gpu, orc, l_max, pieces):
    rng = np.random.default_rng(l_max * 1000 + pieces)
    # 16-bit hashes that share buckets (equal below bit 10) with few and many of each
    for hashes in (np.arange(0, 65536, 7), np.arange(0, 64) * 1024 + 5):
        r = _records(rng, EDGE_COUNTS, SPREAD, np.arange(4000), hashes.astype(np.uint16))
        with H.HashPruneReducer(len(EDGE_COUNTS), l_max) as hp:
            rec = torch.from_numpy(r.view(np.uint8).view(np.int32).reshape(-1, 4).copy()).to(gpu)
            segs = torch.from_numpy(_segments(r, rng, pieces).view(np.int32).copy()).to(gpu)
            hp.insert_segments(rec, segs[: len(segs) // 2])
            hp.insert_segments(rec, segs[len(segs) // 2:])
            _same(_gpu_slots(hp), orc.hashprune_reduce(len(EDGE_COUNTS), l_max, r), f"segments in {pieces} pieces")
            hp.clear()
            hp.insert(r)
            _same(_gpu_slots(hp), orc.hashprune_reduce(len(EDGE_COUNTS), l_max, r), "records")


@pytest.mark.parametrize("dists,targets", [
    (np.float32([0.5]), np.arange(6)),                           # ties settled by target, then by hash
    (np.float32([0.5]), np.array([0, 1, 0x7FFFFFFF, 0x80000000, 0xFFFFFFFE, 0xFFFFFFFF], np.uint32)),
    (np.float32([0.25, 0.5, 0.75]), np.arange(3000)),              # ties settled by target
    (ODD, np.array([0, 7, 0xFFFFFFFF], np.uint32)),                # keys of all ones among them
])
@pytest.mark.parametrize("l_max", [5, 64, 100])
def test_border_ties_and_odd_distances(gpu, orc, dists, targets, l_max):
    rng = np.random.default_rng(l_max)
    r = _records(rng, EDGE_COUNTS, dists, targets, np.arange(0, 3000, 3).astype(np.uint16))
    want = orc.hashprune_reduce(len(EDGE_COUNTS), l_max, r)
    with H.HashPruneReducer(len(EDGE_COUNTS), l_max) as hp:
        for part in np.array_split(r[rng.permutation(len(r))], 2):
            hp.insert(part)
        _same(_gpu_slots(hp), want, "records in two batches")


@pytest.mark.parametrize("l_max", [64, 100, 256])
def test_backfill_groups_across_batches(gpu, orc, l_max):
    # rows that fill in the first batch, in a later one, and never; few hashes, so that groups are deep
    rng = np.random.default_rng(l_max)
    r = np.concatenate([_records(rng, EDGE_COUNTS, SPREAD, np.arange(300), np.arange(m).astype(np.uint16))
                        for m in (20, l_max)])
    bf = H.PRODUCTION_BACKFILL
    t, hs, d, c, _ = orc.hashprune_rhalf_reduce(len(EDGE_COUNTS), l_max, r, mode=bf.mode, hash_quota=0,
                                                row_cap=bf.max_backfill_per_row,
                                                priority_alpha=bf.soft_tier_priority_alpha)
    with H.HashPruneReducer(len(EDGE_COUNTS), l_max, backfill=bf) as hp:
        for part in np.array_split(r[rng.permutation(len(r))], 3):
            hp.insert(part)
        gt, gh, gd, gc = _gpu_slots(hp)
    assert np.array_equal(gc, c)
    for p in range(len(c)):
        n = int(c[p])
        assert np.array_equal(gt[p, :n], t[p, :n]) and np.array_equal(gh[p, :n], hs[p, :n])
        assert np.array_equal(gd[p, :n].view(np.uint32), d[p, :n].view(np.uint32))
