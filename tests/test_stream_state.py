"""What calls on one (device, stream) share, without a GPU: the library's entries are stubs."""

from __future__ import annotations

import ctypes
import threading
from types import SimpleNamespace

import pytest
import torch

from musa_aiter.ops import _hip

STREAM = 7
CPU = torch.device("cpu")


def _t(*shape, dtype=torch.int64):
    return torch.zeros(shape, dtype=dtype)


def _paged(call, **more):
    x = _t(64, dtype=torch.float32)
    return lambda: call(op="t", scatter=True, codec=0, cache_elt=4, lin_elt=4, lin_dtype=0, key_cache=x,
                        value_cache=x, num_blocks=2, num_heads=1, head_dim=4, block_size=8, **more)


def _callers():
    x, i = _t(64, dtype=torch.float32), _t(4)
    lin = dict(key_linear=x, value_linear=x, slots=i, num_layers=1, num_tokens=4, lin_token_stride=4,
               lin_layer_stride=16)
    rows = dict(op="t", device=CPU, src_planes=[1], dst_planes=[2], src_idx=i, dst_idx=i, src_rows=9, dst_rows=9,
                row_bytes=8, src_stride=8, dst_stride=8)
    return {
        "paged_tiles": _paged(_hip.paged_tiles, **lin),
        "paged_tiles_checked": _paged(_hip.paged_tiles_checked, **lin),
        "paged_dense_tiles": _paged(_hip.paged_dense_tiles, dense_k=x, dense_v=x, block_tables=i, seq_lens=i, batch=2,
                                    dense_len=2, max_blocks=2, dense_token_stride=4),
        "copy_rows": lambda: _hip.copy_rows(**rows, num_planes=1, num_tokens=4, num_rows_out=4, zero_invalid=False),
        "copy_rows_paged": lambda: _hip.copy_rows_paged(**rows),
        "copy_rows_paged_checked": lambda: _hip.copy_rows_paged_checked(**rows, low=-1),
        "copy_blocks": lambda: _hip.copy_blocks(op="t", src_k=x, src_v=x, dst_k=x, dst_v=x, block_mapping=_t(2, 2),
                                                num_layers=1, src_blocks=4, dst_blocks=4, block_bytes=16),
    }


@pytest.fixture
def state(monkeypatch):
    """Stubs of the GPU side; ``current`` holds each thread's stream handle, ``inside`` what an entry does."""
    state = SimpleNamespace(current=threading.local(), inside=lambda: None)

    def entry(*_args):
        state.inside()
        return 0

    def stream_ptr(_device):
        return ctypes.c_void_p(getattr(state.current, "stream", STREAM))

    monkeypatch.setattr(_hip, "fn", lambda _name: entry)
    monkeypatch.setattr(_hip, "stream_ptr", stream_ptr)
    monkeypatch.setattr(_hip, "_claim_sets", {})
    monkeypatch.setattr(_hip, "_check_sets", {})
    monkeypatch.setattr(_hip, "_CheckSet",
                        lambda _device: SimpleNamespace(report_ptr=0, values_ptr=0, guard_ptr=0, stamp=0,
                                                        lock=threading.Lock()))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    return state


def _epoch(stream=STREAM):
    return _hip._claim_sets[(0, stream)][1].epoch


_NAMES = ["paged_tiles", "paged_tiles_checked", "paged_dense_tiles", "copy_rows", "copy_rows_paged",
          "copy_rows_paged_checked", "copy_blocks"]


@pytest.mark.parametrize("first", _NAMES)
@pytest.mark.parametrize("second", _NAMES)
def test_claims_of_one_stream_are_used_one_call_at_a_time(state, first, second):
    # The library reads a call's epoch after the interpreter lock is released: until that call has returned,
    # no other thread's call on the stream may advance it.
    callers = _callers()
    callers[first]()  # the claim tags exist
    seen = []
    other = threading.Thread(target=callers[second])

    def inside():
        seen.append((threading.current_thread() is other, _epoch()))
        if threading.current_thread() is not other:
            other.start()
            other.join(0.1)
            assert other.is_alive() and _epoch() == seen[0][1]

    state.inside = inside
    callers[first]()
    other.join(10)
    assert not other.is_alive()
    assert seen == [(False, seen[0][1]), (True, seen[0][1] + 1)]


def test_claims_of_other_streams_do_not_wait(state):
    callers = _callers()
    done = []

    def elsewhere():
        state.current.stream = STREAM + 1
        callers["copy_rows"]()
        done.append(_epoch(STREAM + 1))

    other = threading.Thread(target=elsewhere)

    def inside():
        if threading.current_thread() is not other:
            other.start()
            other.join(10)
            assert done == [1]

    state.inside = inside
    callers["paged_tiles"]()
    assert done == [1] and _epoch() == 1


def test_check_sets_give_way_by_last_use(state):
    # A program with more streams than sets keeps the sets of those it uses, however early they were made, and
    # another device's sets are no reason to give one up.
    def used(device, stream):
        checks = _hip._check_set(device, stream)
        checks.stamp = next(_hip._stamps)  # as a call on the stream does
        return checks

    hot = used(CPU, 0)
    elsewhere = used(torch.device("cuda", 1), 0)
    second = used(CPU, 1)
    for stream in range(2, 3 * _hip._MAX_CHECK_SETS):
        used(CPU, stream)
        assert used(CPU, 0) is hot
    assert _hip._check_set(CPU, 1) is not second
    assert _hip._check_sets[(1, 0)] is elsewhere
    assert sum(k[0] == 0 for k in _hip._check_sets) == _hip._MAX_CHECK_SETS
