"""Device memory that the library takes beside torch's cache: the bound a build
compares with what is free, and the second call after the driver has run out
(host code, no GPU work)."""
import ctypes as C
import types

import numpy as np
import pytest

from shear_amd import _native as N
from shear_amd import hashprune as H
from shear_amd import pipeline as P
from shear_amd import subtree as S


@pytest.mark.parametrize("rows", [1000, 200_000, 1_000_000, 10_000_000, 60_000_000])
@pytest.mark.parametrize("backfill", [None, H.PRODUCTION_BACKFILL])
@pytest.mark.parametrize("c_max,fanout", [(256, 1), (1024, 2), (2048, 4)])
def test_bound_covers_reservoirs_and_workspaces(rows, backfill, c_max, fanout):
    # all leaf rows in one batch, so the plan of a task of all rows holds what the library takes
    p = P.GraphBuildParams(fanout_second=fanout, c_max=c_max, hashprune_backfill=backfill, leaf_chunk_rows=1 << 40)
    sizes = np.full(100, rows * p.fanout_top // 100, np.int64)
    need = P.device_bytes_bound(rows, 768, sizes, p, False)
    state = C.c_uint64(0)
    pol = None if backfill is None else C.byref(backfill.native())
    N.check(N.load().tessa_hashprune_state_bytes(rows, p.l_max, pol, C.byref(state)), "state bytes")
    plan = S.plan_subtree(int(min(sizes.sum(), p.roots_rows_per_run)), p.leaf_knn, 128, fanout, None, c_max)
    image = rows * 4 * (p.l_max + 1)
    assert need >= state.value + plan.required_bytes + image
    # no reservoirs beside a host reducer; a child's own rows without many-root runs
    assert P.device_bytes_bound(rows, 768, sizes, p, True) >= plan.required_bytes + image
    p.multi_root = False
    one = S.plan_subtree(int(sizes.max()), p.leaf_knn, 128, fanout, None, c_max)
    assert P.device_bytes_bound(rows, 768, sizes, p, False) >= state.value + one.required_bytes + 2 * 780 * sizes.max()


def test_bound_stays_small_for_small_builds():
    # a build's memory, not the card's: a tenth of it is free on any card that builds run on
    p = P.GraphBuildParams(c_max=2048, hashprune_backfill=H.PRODUCTION_BACKFILL)
    assert P.device_bytes_bound(1_000_000, 768, np.full(1000, 2000, np.int64), p, False) < 28 << 30


def _status(code):
    st = N.TessaStatus()
    st.code = code
    return st


@pytest.mark.parametrize("codes,calls,emptied", [([0], 1, 0), ([5, 0], 2, 1), ([5, 5], 2, 1), ([2], 1, 0)])
def test_second_call_after_out_of_memory(monkeypatch, codes, calls, emptied):
    import torch

    done = types.SimpleNamespace(calls=0, emptied=0)

    def empty():
        done.emptied += 1

    monkeypatch.setattr(torch.cuda, "empty_cache", empty)

    def fn(a, b):  # as ctypes calls it: every result goes through errcheck
        assert (a, b) == (1, 2)
        st = _status(codes[done.calls])
        done.calls += 1
        return N._retry_without_cache(st, fn, (a, b))

    assert fn(1, 2).code == codes[-1]
    assert (done.calls, done.emptied) == (calls, emptied)


def test_allocating_entries_are_retried():
    lib = N.load()
    for name in N._ALLOCATING:
        assert getattr(lib, name).errcheck is N._retry_without_cache, name
