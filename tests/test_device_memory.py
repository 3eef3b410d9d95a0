"""Device memory that the library takes beside torch's cache: the second call
after the driver has run out (host code, no GPU work)."""
import types

import pytest

from shear_amd import _native as N


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
