"""Many small subtree roots in one run (tessa_session_partition_small_roots)
against the oracle's partition of each root and against one
tessa_session_run_subtree per root: the same leaves, rows and order."""
import numpy as np
import pytest
import torch

from gpu_helpers import require_gpu
from shear_amd import _native as N
from shear_amd import datagen
from shear_amd import pipeline as P
from shear_amd import subtree as S
from shear_amd import tessa as T

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    return require_gpu()


def _roots(gpu, sizes, dim, seed, sigma, comps):
    n = 3000
    x = datagen.gmm_numpy(n, dim, comps, sigma, seed)
    sq8 = T.quantize_sq_int8_matrix(torch.from_numpy(x).to(gpu))
    rng = np.random.default_rng(seed)
    rows = [np.sort(rng.permutation(n)[:m]).astype(np.int32) for m in sizes]
    offs = np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint64)
    return sq8, rows, offs


def _seed(n):
    return S.subtree_root_seed(42, 1, n, 5000, 64)


# sizes around the merge bound (64), bitmap words, ranking all keys or some, one leaf and many
SIZES = [2, 3, 5, 33, 63, 64, 65, 127, 128, 129, 200, 255, 256, 500, 1000, 1023, 1024, 2, 700]


@pytest.mark.parametrize("fanout,c_max,sizes,dim,sigma,comps", [
    (2, 1024, SIZES, 40, 0.3, 9),
    (1, 1024, SIZES, 16, 0.3, 9),
    (3, 2048, SIZES + [1365, 1364], 100, 0.02, 4),     # n * 3 at the small-node limit
    (4, 1024, SIZES, 768, 0.3, 2),
    (2, 2048, [2048, 2047, 1500, 1025], 24, 0.01, 3),  # tight clusters: many attempts
    (2, 1024, [900] * 300, 32, 0.3, 9),                # more roots than CUs
])
def test_leaves_equal_the_oracles_and_single_root_runs(gpu, orc, fanout, c_max, sizes, dim, sigma, comps):
    sq8, rows, offs = _roots(gpu, sizes, dim, len(sizes) + fanout, sigma, comps)
    params = S.PiPNNSubtreeParams(leaf_knn=8, c_max=c_max, fanout_second=fanout, max_leaders=128, max_depth=16)
    sess = S.SubtreeSession(0)
    row_t = torch.from_numpy(np.concatenate(rows)).to(gpu)
    seeds = np.array([_seed(m) for m in sizes], np.uint64)
    ro = sess.partition_roots(sq8, row_t, offs, seeds, params, depth=1, small=True)
    starts = ro.leaf_starts[: ro.leaf_count].cpu().numpy()
    lsz = ro.leaf_sizes[: ro.leaf_count].cpu().numpy()
    roots = ro.leaf_roots[: ro.leaf_count].cpu().numpy()
    got = ro.leaf_rows[: ro.leaf_rows_total].cpu().numpy()
    assert np.array_equal(starts, np.concatenate([[0], np.cumsum(lsz)[:-1]]))
    assert np.all(np.diff(roots) >= 0) and int(lsz.sum()) == ro.leaf_rows_total
    codes, scales, norms = (a.cpu().numpy() for a in (sq8.codes, sq8.scales, sq8.norms))
    for i in range(min(len(sizes), 24)):
        sub = T.Sq8Matrix(sq8.codes[torch.from_numpy(rows[i]).to(gpu).long()],
                          sq8.scales[torch.from_numpy(rows[i]).to(gpu).long()],
                          sq8.norms[torch.from_numpy(rows[i]).to(gpu).long()], sq8.dim)
        sess.upload_device(sub, torch.from_numpy(rows[i]).to(gpu))
        req = S.GpuSubtreePartitionRequest(point_ids=np.zeros(sizes[i], np.uint32), depth=1, parent_points=5000,
                                           min_recurse_size=64)
        one = sess.run(req, params, partition_only=True)
        want = [rows[i][one.leaf_row_ids[a:a + z].cpu().numpy()].tolist()
                for a, z in zip(one.leaf_starts[: one.leaf_count].tolist(), one.leaf_sizes[: one.leaf_count].tolist())]
        mine = [got[starts[j]:starts[j] + lsz[j]].tolist() for j in np.nonzero(roots == i)[0]]
        assert mine == want, f"root {i} of {sizes[i]} rows"
        r = rows[i]
        leaves, _ = orc.subtree_partition(codes[r], scales[r], norms[r], seed=_seed(sizes[i]), root_depth=1,
                                          max_depth=16, max_leaders=128, fanout_second=fanout, leaf_min=64,
                                          leaf_max=c_max, small_node_limit=4096)
        assert mine == [r[leaf].tolist() for leaf in leaves], f"root {i} of {sizes[i]} rows against the oracle"


def test_each_kind_of_root_is_refused_by_the_other_entry(gpu):
    sq8, rows, offs = _roots(gpu, [1500, 100], 16, 1, 0.3, 3)
    params = S.PiPNNSubtreeParams(leaf_knn=8, c_max=1024, fanout_second=2, max_leaders=128, max_depth=16)
    sess = S.SubtreeSession(0)
    row_t = torch.from_numpy(np.concatenate(rows)).to(gpu)
    seeds = np.array([1, 2], np.uint64)
    with pytest.raises(N.TessaError, match="root 0 of 1500 rows is a large root"):
        sess.partition_roots(sq8, row_t, offs, seeds, params, small=True)
    with pytest.raises(N.TessaError, match="root 1 of 100 rows is a small root"):
        sess.partition_roots(sq8, row_t, offs, seeds, params)
    bad = row_t.clone()
    bad[1550] = sq8.rows
    with pytest.raises(N.TessaError, match="outside the 3000 SQ8 rows"):
        sess.partition_roots(sq8, bad[1500:].contiguous(), np.array([0, 100], np.uint64), seeds[:1], params, small=True)


@pytest.mark.parametrize("n,comps,leaf_knn,fanout", [(4000, 20, 32, 2), (400, 200, 10, 2), (3000, 7, 32, 1)])
def test_build_equals_the_build_child_by_child(gpu, n, comps, leaf_knn, fanout):
    x = torch.from_numpy(datagen.gmm_numpy(n, 24, comps, 0.3, 3)).to(gpu)
    sk = torch.from_numpy(P.sketches_of(x.cpu().numpy(), P.sketch_planes(24, 12, 7))).to(gpu)
    lead = P.d0_leader_rows(n, min(n, 40), 5)
    images = []
    for many in (True, False):
        p = P.GraphBuildParams(leaf_knn=leaf_knn, fanout_second=fanout, multi_root=many)
        g = P.build_graph(x, sk, lead, p)
        images.append((g.image.cpu().numpy().tobytes(), g.start, g.stages["leaves"], g.stages["leaf_rows"],
                       g.stages["edge_records"], g.stages["terminal_depth_retries"]))
    assert images[0] == images[1]
