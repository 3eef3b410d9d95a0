"""The library's memory beside a torch cache that holds nearly all of the card.
Nothing here touches the memory it reserves."""
import pytest
import torch

from gpu_helpers import require_gpu
from shear_amd import subtree as S
from shear_amd import tessa as T

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
