"""What checked calls share on a stream: verdict words, stamps and guard of one call say nothing about another."""

from __future__ import annotations

import threading
from types import SimpleNamespace

import pytest
import torch

import musa_aiter
from musa_aiter.ops import _hip

pytestmark = pytest.mark.gpu
DEV = "cuda"
NH, HD, BS = 2, 16, 16


def _paged(tokens, dtype=torch.bfloat16):
    nb = tokens // BS + 2
    slots = torch.randperm(nb * BS, device=DEV)[:tokens]
    caches = [torch.randn((nb, NH, HD, BS), device=DEV).to(dtype) for _ in range(2)]
    rows = [torch.randn((tokens, NH, HD), device=DEV).to(torch.bfloat16) for _ in range(2)]
    return nb, slots, caches, rows


def _refused_call(kind, tokens):
    """(an accepted call, the same call with one value to refuse, the error's text)."""
    if kind == "page":
        src, dst = (torch.randn((2, tokens + 2, 64), device=DEV) for _ in range(2))
        idx = torch.randperm(tokens + 2, device=DEV)[:tokens]
        bad = idx.clone()
        bad[0] = tokens + 2

        def move(i):
            musa_aiter.hicache_transfer_kv_all_layer(src, dst, src, dst.clone(), i, idx)

        return lambda: move(idx), lambda: move(bad), "page index is out of range"
    nb, slots, caches, rows = _paged(tokens)
    if kind == "scale":
        codes = [torch.zeros((nb, NH, HD, BS), dtype=torch.uint8, device=DEV) for _ in range(2)]
        good = torch.ones(NH, device=DEV)
        return (lambda: musa_aiter.kv_linear_to_paged_fp8(*rows, *codes, slots, good, good),
                lambda: musa_aiter.kv_linear_to_paged_fp8(*rows, *codes, slots, good, -good),
                "v_scale: FP8 scale must be positive and finite")
    bad = slots.clone()
    bad[0] = nb * BS
    if kind == "store":
        return (lambda: musa_aiter.kv_linear_to_paged(*rows, *caches, slots),
                lambda: musa_aiter.kv_linear_to_paged(*rows, *caches, bad), "out of bounds")
    return (lambda: musa_aiter.kv_paged_to_linear(*caches, slots),
            lambda: musa_aiter.kv_paged_to_linear(*caches, bad), "out of bounds")


# Calls of one verdict word (the moving kernel's own), and of several (a check kernel's, a gather's shares).
@pytest.mark.parametrize("tokens", [200, 1500, 5000])
@pytest.mark.parametrize("kind", ["store", "gather", "scale", "page"])
@pytest.mark.parametrize("which", ["shortest", "longest"])
def test_lengths_of_a_dense_call_are_no_verdict(which, kind, tokens):
    # A dense call's table check leaves sequence lengths in host memory; one that equals the next call's
    # "accepted" word (twice its stamp) must not be taken for that call's verdict.
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        accepted, refused, text = _refused_call(kind, tokens)
        accepted()  # the stream's state exists from here on
        checks = _hip._check_set(torch.device(DEV, torch.cuda.current_device()), stream.cuda_stream)
        word = 2 * (checks.stamp + 2)  # the dense call takes the next stamp
        lens = [word, word + 9] if which == "shortest" else [word - 1, word]
        cols = (max(lens) + BS - 1) // BS
        caches = [torch.zeros((cols, 1, 8, BS), dtype=torch.bfloat16, device=DEV) for _ in range(2)]
        # Both lengths in every workgroup of the table check (at most 64), so in every word it writes.
        lens = torch.tensor(lens, device=DEV).repeat_interleave(64)
        tables = torch.arange(cols, device=DEV).repeat(128, 1)
        musa_aiter.kv_load_and_reshape_flash(*caches, tables, lens)
        assert 2 * (checks.stamp + 1) == word
        with pytest.raises(ValueError, match=text):
            refused()
        accepted()
    torch.cuda.synchronize()


def test_calls_under_a_default_device():
    # torch.device / set_default_device redirects factory functions; the host words of a stream's first call
    # are host memory all the same.
    idx = torch.tensor([2, 0, 1], device=DEV)
    src, dst = torch.randn((2, 3, 64), device=DEV), torch.zeros((2, 3, 64), device=DEV)
    with torch.cuda.stream(torch.cuda.Stream()), torch.device(DEV), pytest.MonkeyPatch.context() as patch:
        patch.setattr(_hip, "_check_sets", {})
        musa_aiter.hicache_transfer_kv_all_layer(src, dst, src, dst.clone(), idx, idx)
        caches = [torch.ones((2, 1, 8, BS), dtype=torch.bfloat16) for _ in range(2)]
        k, _ = musa_aiter.kv_load_and_reshape_flash(*caches, torch.tensor([[0, 1]]), torch.tensor([20]))
        with pytest.raises(ValueError, match="invalid block id 2"):
            musa_aiter.kv_load_and_reshape_flash(*caches, torch.tensor([[0, 2]]), torch.tensor([20]))
    torch.cuda.synchronize()
    assert torch.equal(src, dst)
    assert k.shape == (1, 20, 1, 8) and bool((k == 1).all())


def test_index_max_of_a_short_vector_after_a_long_one():
    # The maxima of a long vector's 64 workgroups fill words in which a short vector's single stamp must not be
    # looked for: a maximum equal to the next stamp would be taken for that call's.
    long = torch.empty(64 * 4096, dtype=torch.int64, device=DEV)
    short = torch.tensor([12345678], device=DEV)
    assert _hip.index_max(short) == 12345678
    entry = _hip._index_max_bufs[torch.cuda.current_device()]
    for _ in range(2):
        long.fill_(entry[1] + 2)  # the stamp of the call after the long vector's
        assert _hip.index_max(long) == int(long[0])
        assert _hip.index_max(short) == 12345678


def test_first_checked_call_of_a_stream_leaves_another_threads_capture_alone():
    _, slots, caches, rows = _paged(200)
    musa_aiter.kv_linear_to_paged(*rows, *caches, slots)
    outs = [torch.empty_like(r) for r in rows]
    x = torch.zeros(8, device=DEV)
    stream, errors = torch.cuda.Stream(), []
    torch.cuda.synchronize()

    def work():
        try:
            with torch.cuda.stream(stream):
                musa_aiter.kv_paged_to_linear(*caches, slots, out_k=outs[0], out_v=outs[1])
        except Exception as e:  # reported by the main thread
            errors.append(repr(e))

    saved = dict(_hip._check_sets)
    _hip._check_sets.clear()
    graph = torch.cuda.CUDAGraph()
    try:
        with torch.cuda.graph(graph):  # in global mode: an allocation by another thread invalidates it
            x += 1
            thread = threading.Thread(target=work)
            thread.start()
            thread.join(30)
            x += 1
    finally:
        _hip._check_sets.update(saved)
    assert errors == [] and not thread.is_alive()
    for _ in range(2):
        graph.replay()
    torch.cuda.synchronize()
    assert x.tolist() == [4.0] * 8
    for r, o in zip(rows, outs):
        assert torch.equal(r, o)


@pytest.mark.parametrize("layers", [1, 2])
def test_failed_launches_name_the_operation(monkeypatch, layers):
    # The host module's status is reported under the name of the call, as the Python layer's own launches are.
    suffix = "_multi_layer" if layers > 1 else ""
    lead = (layers,) if layers > 1 else ()
    caches = [torch.zeros(lead + (4, NH, HD, BS), dtype=torch.bfloat16, device=DEV) for _ in range(2)]
    rows = [torch.zeros(lead + (5, NH, HD), dtype=torch.bfloat16, device=DEV) for _ in range(2)]
    codes = [torch.zeros(lead + (4, NH, HD, BS), dtype=torch.uint8, device=DEV) for _ in range(2)]
    slots, scale = torch.arange(5, device=DEV), torch.ones(NH, device=DEV)
    calls = {"kv_paged_to_linear": (*caches, slots), "kv_linear_to_paged": (*rows, *caches, slots),
             "kv_paged_fp8_to_linear": (*codes, slots, scale, scale),
             "kv_linear_to_paged_fp8": (*rows, *codes, slots, scale, scale)}
    for name, args in calls.items():
        getattr(musa_aiter, name + suffix)(*args)  # the stream's state exists from here on
    failed = SimpleNamespace(paged_call=lambda *_: (1, None, None), NOT_TAKEN=_hip.host().NOT_TAKEN)
    monkeypatch.setattr(_hip, "_host", failed)
    for name, args in calls.items():
        with pytest.raises(_hip.HipBackendError, match=f"^{name + suffix}: HIP launch failed with error 1 "):
            getattr(musa_aiter, name + suffix)(*args)


@pytest.mark.parametrize("tokens", [40, 700])  # the kernel's own duplicate table; claim tags
def test_threads_sharing_a_stream_lose_no_rows(tokens):
    # Scatters, refused scatters and block-table write-backs of several threads on one stream claim in one tag
    # array: every accepted row arrives.
    stream = torch.cuda.Stream()
    n, pages = 4, (tokens + BS - 1) // BS
    caches = [torch.zeros((n * pages + 1, NH, HD, BS), device=DEV) for _ in range(2)]
    rows = [torch.randn((n, tokens, NH, HD), device=DEV) for _ in range(2)]
    slots = [k * pages * BS + torch.randperm(pages * BS, device=DEV)[:tokens] for k in range(n)]
    dense = [torch.randn((1, BS, NH, HD), device=DEV) for _ in range(2)]
    table, length = torch.tensor([[n * pages]], device=DEV), torch.tensor([BS], device=DEV)
    torch.cuda.synchronize()
    errors = []

    def work(k):
        try:
            bad = slots[k].clone()
            bad[0] = (n * pages + 1) * BS
            for _ in range(50):
                with torch.cuda.stream(stream):
                    with pytest.raises(ValueError):
                        musa_aiter.kv_linear_to_paged(rows[0][k], rows[1][k], *caches, bad)
                    musa_aiter.kv_linear_to_paged(rows[0][k], rows[1][k], *caches, slots[k])
                    if k == 0:
                        musa_aiter.kv_reshape_and_cache_back_flash(*dense, *caches, table, length)
        except BaseException as e:  # reported by the main thread
            errors.append(repr(e))

    for _ in range(3):
        for c in caches:
            c.zero_()
        torch.cuda.synchronize()
        threads = [threading.Thread(target=work, args=(k,)) for k in range(n)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        torch.cuda.synchronize()
        assert errors == []
        for k in range(n):
            for want, got in zip(rows, musa_aiter.kv_paged_to_linear(*caches, slots[k])):
                assert torch.equal(want[k], got)
        for want, got in zip(dense, musa_aiter.kv_load_and_reshape_flash(*caches, table, length)):
            assert torch.equal(want, got)
