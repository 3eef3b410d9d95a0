"""Global D0 assignment with up to four of more than 128 leaders per row: the kernel that holds 64
rows per wave and ranks each leader tile during the next one's products, at the
edges of its row blocks (256), leader tiles (32) and code widths, against the
CPU oracle's restatement of the GPU-D0 kernels
(shear-core/src/algorithm/pipnn/compute_backend.rs:18016-18511); and, where
scales and norms are not finite, against the distances in f32 sorted on the host
(NaN behind every number, then by leader id) and the kernel of the longer lists.
Bar: identical fragments, offsets and grouped points."""
import numpy as np
import pytest
import torch

from gpu_helpers import require_gpu
from shear_amd import d0 as D
from shear_amd import tessa as T
from test_gpu_d0 import _run_case

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    return require_gpu()


@pytest.mark.parametrize("rows,dim,leaders,fanout", [
    (129, 16, 129, 1), (130, 16, 129, 2), (255, 128, 159, 2), (257, 129, 160, 2), (256, 256, 161, 4),
    (513, 257, 192, 3), (300, 512, 193, 2), (700, 513, 225, 4), (1025, 784, 130, 2), (321, 1024, 224, 3),
    (140, 768, 128, 2),  # the last count of the kernel with 32 rows per wave
])
def test_row_blocks_and_leader_tiles(gpu, orc, rows, dim, leaders, fanout):
    rng = np.random.default_rng(rows + dim)
    x = rng.standard_normal((rows, dim)).astype(np.float32)
    _run_case(gpu, orc, x, rng.permutation(rows)[:leaders].astype(np.int64), fanout)
    # every distance twice: the leader's id decides
    _run_case(gpu, orc, x, rng.permutation(rows)[:leaders].astype(np.int64), fanout, dup=True)


@pytest.mark.parametrize("fanout", [1, 2, 4])
def test_values_that_are_not_finite_rank_as_in_the_longer_lists(gpu, fanout):
    rng = np.random.default_rng(11)
    sq = T.quantize_sq_int8_matrix(torch.from_numpy(rng.standard_normal((600, 96)).astype(np.float32)).to(gpu))
    lead = T.Sq8Matrix(sq.codes[:170].clone(), sq.scales[:170].clone(), sq.norms[:170].clone(), sq.dim)
    odd = torch.tensor([float("nan"), float("inf"), -float("inf"), 0.0, 3.0e38], device=gpu)
    sq.scales[100:105], sq.norms[105:110] = odd, odd
    lead.scales[10:15], lead.norms[165:170] = odd, odd
    gids = torch.arange(600, device=gpu, dtype=torch.int32)
    lids = torch.arange(170, device=gpu, dtype=torch.int32).flip(0).contiguous()
    want = D.global_d0_assign(sq, gids, lead, lids, 8)[0]
    got = D.global_d0_assign(sq, gids, lead, lids, fanout)[0]
    assert torch.equal(got, want[:, :fanout])
    rc, rs, rn, lc, ls, ln = (a.cpu().numpy() for a in (sq.codes, sq.scales, sq.norms, lead.codes, lead.scales,
                                                        lead.norms))
    dot = (rc.astype(np.int32) @ lc.astype(np.int32).T).astype(np.float32)
    with np.errstate(all="ignore"):
        d = (rn[:, None] + ln[None, :]) - ((np.float32(2) * rs)[:, None] * ls[None, :]) * dot
    d = np.where(d <= 0, np.float32(0), d)
    assert np.isnan(d).any() and np.isinf(d).any()
    order = np.lexsort((np.broadcast_to(lids.cpu().numpy(), d.shape), np.nan_to_num(d, nan=0.0, posinf=np.inf),
                        np.isnan(d)), axis=1)
    g = got.cpu().numpy()
    number = ~np.isnan(np.take_along_axis(d, order[:, :fanout], 1))  # of several NaN the sign decides, not the host's
    assert np.array_equal(g[number], order[:, :fanout][number])
    assert np.isnan(np.take_along_axis(d, g.astype(np.int64), 1)[~number]).all()
