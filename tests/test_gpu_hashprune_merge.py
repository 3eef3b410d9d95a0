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


FEW_COUNTS = [1, 2, 3, 0, 19, 20, 21, 22, 31, 32, 33, 34, 0, 63, 64, 65]
# no NaN (the order of a backup of NaN distance is no one's), every other class
PLAIN = np.array([0x00000000, 0x80000000, 0x00000001, 0x7F800000, 0x3F800000, 0x3F000000, 0x40000000, 0x41200000],
                 np.uint32).view(np.float32)


@pytest.mark.parametrize("mode,quota", [("rhalf-hash-slot-1", 1), ("rhalf-distance-first-q3", 2),
                                        ("rhalf-soft-tier-q3", 3), ("rhalf-hard-tier-q3", 3)])
@pytest.mark.parametrize("l_max", [2, 5, 63, 64, 65, 128, 130, 256])
def test_few_records_of_a_source_with_groups(gpu, orc, mode, quota, l_max):
    # batches of a few records per source go in one by one: into empty, underfull and full reservoirs, with hashes,
    # targets and distances that repeat, beside sources of more records in the same batch
    rng = np.random.default_rng(l_max * 10 + quota)
    for hashes, dists, targets in ((7, PLAIN, np.arange(9)), (l_max + 3, SPREAD, np.arange(40)),
                                   (3000, PLAIN, np.array([0, 1, 0x7FFFFFFF, 0x80000000, 0xFFFFFFFE], np.uint32))):
        parts = [_records(rng, list(rng.permutation(FEW_COUNTS)), dists, targets, np.arange(hashes).astype(np.uint16))
                 for _ in range(5)]
        cap = min(4, l_max // 2)
        alpha = 1.1 if mode == "rhalf-soft-tier-q3" else None
        bf = H.HashPruneBackfill(mode, quota, cap, alpha)
        t, hs, d, c, _ = orc.hashprune_rhalf_reduce(len(FEW_COUNTS), l_max, np.concatenate(parts), mode=mode,
                                                    hash_quota=quota, row_cap=cap, priority_alpha=alpha or 0.0)
        with H.HashPruneReducer(len(FEW_COUNTS), l_max, backfill=bf) as hp:
            for part in parts:
                hp.insert(part[rng.permutation(len(part))])
            gt, gh, gd, gc = _gpu_slots(hp)
        assert np.array_equal(gc, c)
        for p in range(len(c)):
            n = int(c[p])
            assert np.array_equal(gt[p, :n], t[p, :n]) and np.array_equal(gh[p, :n], hs[p, :n]), (hashes, p)
            assert np.array_equal(gd[p, :n].view(np.uint32), d[p, :n].view(np.uint32)), (hashes, p)


@pytest.mark.parametrize("backfill", [None, H.PRODUCTION_BACKFILL])
def test_sparse_batches(gpu, orc, backfill):
    # sources at the edges of the scan's blocks of 4,096 points, most points without a record
    rng = np.random.default_rng(2)
    n, l_max = 4096 * 5 + 17, 8
    src = np.array([0, 1, 4095, 4096, 4097, 8191, 12288, 20479, 20480, n - 1], np.uint32)
    r = _records(rng, [3, 40, 1, 21, 20, 300, 2, 1, 33, 32], SPREAD, np.arange(900), np.arange(60).astype(np.uint16))
    r["src"] = src[r["src"]]
    with H.HashPruneReducer(n, l_max, backfill=backfill) as hp:
        for part in np.array_split(r[rng.permutation(len(r))], 3):
            hp.insert(part)
        gt, gh, gd, gc = _gpu_slots(hp)
    if backfill is None:
        t, hs, d, c = orc.hashprune_reduce(n, l_max, r)[:4]
    else:
        t, hs, d, c, _ = orc.hashprune_rhalf_reduce(n, l_max, r, mode=backfill.mode, hash_quota=0,
                                                    row_cap=backfill.max_backfill_per_row,
                                                    priority_alpha=backfill.soft_tier_priority_alpha)
    assert np.array_equal(gc, c)
    for p in src:
        m = int(c[p])
        assert np.array_equal(gt[p, :m], t[p, :m]) and np.array_equal(gh[p, :m], hs[p, :m])
        assert np.array_equal(gd[p, :m].view(np.uint32), d[p, :m].view(np.uint32))


def test_a_small_batch_takes_its_own_time(gpu):
    # 1,000 records into 8 M reservoirs: the counts of all points are scanned, their reservoirs are not.  A wave for
    # every point took some twenty times what the same batch takes among 100,000 points.
    rng = np.random.default_rng(4)

    def ms(points):
        r = np.zeros(1000, E.EDGE_RECORD_DTYPE)
        r["src"], r["dst"], r["hash"] = rng.integers(0, points, 1000), rng.integers(0, points, 1000), rng.integers(0, 99, 1000)
        r["dist"] = rng.random(1000)
        rec = torch.from_numpy(r.view(np.uint8).view(np.int32).reshape(-1, 4).copy()).to(gpu)
        best = []
        with H.HashPruneReducer(points, 8, backfill=H.PRODUCTION_BACKFILL) as hp:
            for _ in range(6):
                a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                a.record()
                hp.insert(rec)
                b.record()
                b.synchronize()
                best.append(a.elapsed_time(b))
        return min(best)

    few, many = ms(100_000), ms(8_000_000)
    assert many < 5.0 * few, (many, few)
