"""What is still queued on the leaf operator's stream when a many-root run ends
early (host code: streams, events and the session are stand-ins)."""
import types

import numpy as np
import pytest
import torch

from shear_amd import pipeline as P
from shear_amd import tessa as T


class _Stream:
    def __init__(self, name, log):
        self.name, self.log = name, log

    def wait_stream(self, other):
        self.log.append((self.name, "waits for", other.name))

    def wait_event(self, event):
        pass


class _Event:
    def __init__(self, enable_timing=False):
        pass

    def record(self, stream=None):
        pass

    def elapsed_time(self, other):
        return 0.0


@pytest.mark.parametrize("fails_in", ["emit", "consume", "second leaf_topk", None])
def test_caller_waits_for_queued_leaves(monkeypatch, fails_in):
    # four leaves of 8 rows in four batches: while one is emitted the next one's leaf operator is queued
    log, calls = [], []
    main, side = _Stream("main", log), _Stream("side", log)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: main)
    monkeypatch.setattr(torch.cuda, "Stream", lambda *a, **k: side)
    monkeypatch.setattr(torch.cuda, "Event", _Event)
    monkeypatch.setattr(torch.Tensor, "record_stream", lambda self, s: None)

    def leaf_topk(*a, **k):
        calls.append(1)
        if fails_in == "second leaf_topk" and len(calls) == 2:
            raise RuntimeError("no memory")

    monkeypatch.setattr(T, "leaf_topk", leaf_topk)
    monkeypatch.setattr(T, "raise_on_overflow", lambda *a: None)

    def emit(*a):
        if fails_in == "emit":
            raise RuntimeError("emission")
        return None, 0, None, 0

    def consume(*a):
        if fails_in == "consume":
            raise RuntimeError("merge")

    i32 = torch.int32
    ro = types.SimpleNamespace(partition_ms=0.0, leaf_count=4, leaf_rows=torch.arange(32, dtype=i32),
                               leaf_starts=torch.arange(4) * 8, leaf_sizes=torch.full((4,), 8, dtype=i32),
                               leaf_roots=torch.zeros(4, dtype=i32), leaf_depths=torch.ones(4, dtype=i32))
    sess = types.SimpleNamespace(partition_roots=lambda *a, **k: ro)
    sq8 = types.SimpleNamespace(codes=torch.zeros(32, 32, dtype=torch.int8))
    p = P.GraphBuildParams(leaf_knn=4, leaf_chunk_rows=8)
    st = {"part_ms": 0.0, "leaf_ms": 0.0, "records": 0, "leaves": 0, "leaf_rows": 0, "retries": 0, "runs": 0,
          "emit_s": 0.0, "reduce_s": 0.0}

    def run():
        P._run_root_group(sess, sq8, torch.arange(32, dtype=i32), torch.arange(32, dtype=i32),
                          np.array([0, 32], np.uint64), np.array([32], np.int64), [0], 32, p, p.subtree_params(), st,
                          emit, consume, None, False)

    if fails_in is None:
        run()
        assert st["leaves"] == 4
    else:
        with pytest.raises(RuntimeError):
            run()
        assert len(calls) == 2  # the second batch was queued when the first one failed
    assert log[-1] == ("main", "waits for", "side")
