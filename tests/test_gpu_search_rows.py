"""Greedy search where its rows' reading changes: staged in LDS by pieces of 128
floats or 512 codes (128 to 2,048 aligned f32 columns, 257 to 2,048 SQ8 ones, up
to four queries per CU) or read by the lanes, rows of odd widths and unaligned sets, list lengths at
register edges, degrees around a wave, a slot's second query.  Bar: bit-identical
to the oracle."""
import numpy as np
import pytest
import torch

from gpu_helpers import require_gpu
from shear_amd import graph as G
from shear_amd import tessa as T

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    return require_gpu()


def _graph(rng, n, stride):
    t = rng.integers(0, n + 2, (n, stride)).astype(np.uint32)  # some ids past the set
    c = rng.integers(0, stride + 2, n).astype(np.uint32)        # some counts past the row
    return t, c


def _run(gpu, orc, x, q, t, c, L, K, data=None):
    f = G.greedy_search_sq8 if isinstance(data, T.Sq8Matrix) else G.greedy_search
    ids, d, cmps = f(torch.from_numpy(x).to(gpu) if data is None else data, torch.from_numpy(t.view(np.int32)).to(gpu),
                     torch.from_numpy(c.view(np.int32)).to(gpu), 3, torch.from_numpy(q).to(gpu), L, K)
    torch.cuda.synchronize()
    wi, wd, wc = orc.greedy_search(x, t, c, 3, q, L, K)
    assert np.array_equal(ids.cpu().numpy().view(np.uint32), wi)
    assert np.array_equal(d.cpu().numpy().view(np.uint32), np.asarray(wd).view(np.uint32))
    assert np.array_equal(cmps.cpu().numpy().view(np.uint32), wc)


@pytest.mark.parametrize("dim", [1, 4, 15, 16, 17, 63, 64, 124, 127, 128, 129, 132, 256, 260, 513, 644, 2048, 2052])
@pytest.mark.parametrize("L,stride,nq", [(16, 65, 5), (65, 130, 5)])
def test_row_widths(gpu, orc, dim, L, stride, nq):
    rng = np.random.default_rng(dim + L)
    x = rng.standard_normal((400, dim)).astype(np.float32)
    q = rng.standard_normal((nq, dim)).astype(np.float32)
    t, c = _graph(rng, 400, stride)
    _run(gpu, orc, x, q, t, c, L, 7)


@pytest.mark.parametrize("L", [1, 2, 63, 64, 65, 128, 129, 256])
@pytest.mark.parametrize("stride", [1, 63, 64, 200])
def test_list_lengths_and_degrees(gpu, orc, L, stride):
    rng = np.random.default_rng(L * 7 + stride)
    x = rng.integers(-3, 4, (900, 8)).astype(np.float32)  # many equal distances
    q = rng.integers(-3, 4, (9, 8)).astype(np.float32)
    t, c = _graph(rng, 900, stride)
    _run(gpu, orc, x, q, t, c, L, min(L, 20))


# above 1,024: every row is read by the lanes; above 4,096: a slot's wave clears its visited bits
# for a second query
@pytest.mark.parametrize("nq", [1024, 1025, 4100])
@pytest.mark.parametrize("kind,dim", [("f32", 132), ("f32", 129), ("sq8", 272), ("sq8", 400), ("f32", 516), ("sq8", 256)])
@pytest.mark.parametrize("L", [12, 100, 200])
def test_many_queries(gpu, orc, nq, kind, dim, L):
    rng = np.random.default_rng(nq + dim)
    x = rng.standard_normal((300, dim)).astype(np.float32)
    q = rng.standard_normal((nq, dim)).astype(np.float32)
    t, c = _graph(rng, 300, 20)
    data = None
    if kind == "sq8":
        data = T.quantize_sq_int8_matrix(torch.from_numpy(x).to(gpu))
        x = data.codes.cpu().numpy()[:, :dim].astype(np.float32) * data.scales.cpu().numpy()[:, None]
    _run(gpu, orc, x, q, t, c, L, 5, data=data)


@pytest.mark.parametrize("dim", [128, 640])
def test_unaligned_rows(gpu, orc, dim):
    rng = np.random.default_rng(8)
    x = rng.standard_normal((500, dim)).astype(np.float32)
    q = rng.standard_normal((6, dim)).astype(np.float32)
    t, c = _graph(rng, 500, 40)
    flat = torch.empty(500 * dim + 1, device=gpu)
    flat[1:] = torch.from_numpy(x.reshape(-1)).to(gpu)
    _run(gpu, orc, x, q, t, c, 30, 10, data=flat[1:].view(500, dim))


@pytest.mark.parametrize("dim,shift", [(16, 0), (100, 0), (256, 0), (257, 0), (272, 0), (512, 0), (528, 0), (1000, 0), (100, 4), (2049, 0), (2112, 0),
                                       (2127, 0), (4096, 0), (2100, 4)])
def test_sq8_rows(gpu, orc, dim, shift):
    rng = np.random.default_rng(dim)
    x = rng.standard_normal((400, dim)).astype(np.float32)
    q = rng.standard_normal((7, dim)).astype(np.float32)
    t, c = _graph(rng, 400, 66)
    m = T.quantize_sq_int8_matrix(torch.from_numpy(x).to(gpu))
    if shift:  # codes that do not start on 16 bytes
        flat = torch.empty(m.codes.numel() + shift, dtype=torch.int8, device=gpu)
        flat[shift:] = m.codes.view(-1)
        m = T.Sq8Matrix(flat[shift:].view(m.codes.shape), m.scales, m.norms, m.dim)
    deq = m.codes.cpu().numpy()[:, :dim].astype(np.float32) * m.scales.cpu().numpy()[:, None]
    _run(gpu, orc, deq, q, t, c, 24, 9, data=m)


def _ms(f, data, t, c, q):
    best = []
    for _ in range(4):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        f(data, t, c, 3, q, 32, 5)
        b.record()
        b.synchronize()
        best.append(a.elapsed_time(b))
    return min(best)


def _timed_set(gpu, n, dim, nq):
    rng = np.random.default_rng(1)
    x, q = (torch.from_numpy(rng.standard_normal((m, dim)).astype(np.float32)).to(gpu) for m in (n, nq))
    t = torch.from_numpy(rng.integers(0, n, (n, 48)).astype(np.int32)).to(gpu)
    return x, q, t, torch.full((n,), 48, dtype=torch.int32, device=gpu)


def test_wide_sq8_rows_are_read_in_wide_loads(gpu):
    # A quarter of the f32 rows' bytes and five instructions a code instead of three: no more than twice the f32
    # search's time at any width.  Read a byte at a time, they took four times as long.
    x, q, t, c = _timed_set(gpu, 4000, 2560, 500)
    a, b = _ms(G.greedy_search_sq8, T.quantize_sq_int8_matrix(x), t, c, q), _ms(G.greedy_search, x, t, c, q)
    assert a < 2.0 * b, (a, b)


def test_odd_widths_are_read_in_wide_loads(gpu):
    # 129 columns take little longer than 132.  Staged a float at a time they took four times as long (and 1.1-1.3
    # times what one float per lane and load had taken).
    a, b = (_ms(G.greedy_search, x, t, c, q) for x, q, t, c in (_timed_set(gpu, 20000, d, 64) for d in (129, 132)))
    assert a < 2.0 * b, (a, b)


def test_searches_on_several_streams(gpu, orc):
    # all searches of a GPU share its visited bits: one starts after another has ended, from two host threads too
    import threading

    rng = np.random.default_rng(12)
    x = rng.standard_normal((3000, 32)).astype(np.float32)
    t, c = _graph(rng, 3000, 32)
    qs = [rng.standard_normal((n, 32)).astype(np.float32) for n in (900, 5, 4500, 300)]
    want = [orc.greedy_search(x, t, c, 3, q, 24, 6) for q in qs]
    xd, td, cd = (torch.from_numpy(a).to(gpu) for a in (x, t.view(np.int32), c.view(np.int32)))
    qd = [torch.from_numpy(q).to(gpu) for q in qs]
    torch.cuda.synchronize()
    out = {}

    def work(who):
        streams = [torch.cuda.Stream(), torch.cuda.Stream()]
        for i in range(12):
            j = (i + who) % len(qd)
            out[who, i] = j, G.greedy_search(xd, td, cd, 3, qd[j], 24, 6, stream=streams[i % 2])
        for s in streams:
            s.synchronize()

    threads = [threading.Thread(target=work, args=(w,)) for w in range(2)]
    for h in threads:
        h.start()
    for h in threads:
        h.join()
    torch.cuda.synchronize()
    assert len(out) == 24
    for j, (ids, d, cmps) in out.values():
        wi, wd, wc = want[j]
        assert np.array_equal(ids.cpu().numpy().view(np.uint32), wi)
        assert np.array_equal(d.cpu().numpy().view(np.uint32), np.asarray(wd).view(np.uint32))
        assert np.array_equal(cmps.cpu().numpy().view(np.uint32), wc)
