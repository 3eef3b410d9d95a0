"""SQ8 quantizer at the edges of its row blocks: rows per block (4 to 32 by
width), words per lane (one to four in registers, more re-read), rows that lie
unaligned or at odd strides, wide padding, bad rows in any place.  Bar:
bit-identical to the oracle."""
import numpy as np
import pytest
import torch

from gpu_helpers import require_gpu
from shear_amd import tessa as T

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    return require_gpu()


def _rows(rng, rows, dim):
    x = (rng.standard_normal((rows, dim)) * rng.uniform(1e-3, 50, (rows, 1))).astype(np.float32)
    x[0] = 0.0
    x[rows // 2] = np.float32(1e-40)              # a subnormal scale
    x[-1] = np.round(x[-1] * 4) / 8               # quotients near half-integers
    return x


@pytest.mark.parametrize("dim", [1, 2, 3, 4, 15, 16, 17, 50, 63, 64, 65, 100, 255, 256, 257, 260, 272, 513, 768, 772,
                                 1000, 1024, 1028, 1030, 2000, 4001, 8192, 8193, 8196])
@pytest.mark.parametrize("rows", [1, 5, 70])
def test_widths(gpu, orc, dim, rows):
    x = _rows(np.random.default_rng(dim * 3 + rows), rows, dim)
    m = T.quantize_sq_int8_matrix(torch.from_numpy(x).to(gpu))
    codes, scales, norms = orc.quantize(x)
    assert np.array_equal(m.codes.cpu().numpy(), codes)
    assert np.array_equal(m.scales.cpu().numpy().view(np.uint32), scales.view(np.uint32))
    assert np.array_equal(m.norms.cpu().numpy().view(np.uint32), norms.view(np.uint32))


@pytest.mark.parametrize("dim", [37, 64, 768])
def test_unaligned_and_wide_padding(gpu, orc, dim):
    x = _rows(np.random.default_rng(dim), 45, dim)
    flat = torch.empty(45 * dim + 1, device=gpu)
    flat[1:] = torch.from_numpy(x.reshape(-1)).to(gpu)
    codes, scales, _ = orc.quantize(x)
    m = T.quantize_sq_int8_matrix(flat[1:].view(45, dim), k_align=320)
    got = m.codes.cpu().numpy()
    assert np.array_equal(got[:, :dim], codes[:, :dim]) and not got[:, dim:].any()
    assert np.array_equal(m.scales.cpu().numpy(), scales)


@pytest.mark.parametrize("dim", [37, 128, 9000])
@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
def test_bad_rows_are_reported(gpu, dim, value):
    x = np.ones((100, dim), np.float32)
    x[71, dim - 1] = value
    x[90, 0] = value
    with pytest.raises(ValueError, match="non-finite value in row 71"):
        T.quantize_sq_int8_matrix(torch.from_numpy(x).to(gpu))
