"""Slots and FP8 scales that a call must refuse are found on the device, before anything is written.

Calls of at most 256 tokens check them in the kernel that moves them, larger ones (and those whose kernel
cannot) in a kernel ahead of it on the stream.  Either way the error, the untouched caches and outputs
and the next call on the stream are what a check on the host ahead of the launch would give.
"""

from __future__ import annotations

import threading

import pytest
import torch

import musa_aiter

pytestmark = pytest.mark.gpu
DEV = "cuda"
NH, HD = 4, 64


def _setup(bs, tokens, layers, dtype=torch.bfloat16, seed=1):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    nb = tokens // bs + 4
    lead = (layers,) if layers > 1 else ()
    slots = torch.randperm(nb * bs, generator=gen, device=DEV)[:tokens]
    caches = [torch.randint(0, 255, lead + (nb, NH, HD, bs), generator=gen, device=DEV, dtype=torch.uint8)
              if dtype is torch.uint8 else torch.randn(lead + (nb, NH, HD, bs), generator=gen, device=DEV).to(dtype)
              for _ in range(2)]
    linear = [torch.randn(lead + (tokens, NH, HD), generator=gen, device=DEV).to(
        torch.bfloat16 if dtype is torch.uint8 else dtype) for _ in range(2)]
    return nb, slots, caches, linear


def _names(base, layers):
    return getattr(musa_aiter, base + ("_multi_layer" if layers > 1 else ""))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("bs", [5, 8, 16, 32, 64])
@pytest.mark.parametrize("tokens,layers", [(1, 1), (200, 1), (200, 20), (1500, 2), (70000, 1)])
def test_slot_past_the_cache_is_refused(dtype, bs, tokens, layers):
    nb, slots, caches, linear = _setup(bs, tokens, layers, dtype)
    before = [c.clone() for c in caches]
    outs = [torch.full_like(x, 7.0) for x in linear]
    gather, scatter = _names("kv_paged_to_linear", layers), _names("kv_linear_to_paged", layers)
    for at in {0, tokens // 2, tokens - 1}:
        bad = slots.clone()
        bad[at] = nb * bs
        with pytest.raises(ValueError, match=f"slot index {nb * bs} out of bounds"):
            scatter(*linear, *caches, bad)
        with pytest.raises(ValueError, match=f"slot index {nb * bs} out of bounds"):
            gather(*caches, bad, out_k=outs[0], out_v=outs[1])
    for c, b, o in zip(caches, before, outs):
        assert torch.equal(c, b)
        assert bool((o == 7.0).all())
    scatter(*linear, *caches, slots)
    for x, got in zip(linear, gather(*caches, slots)):
        assert torch.equal(x, got)


@pytest.mark.parametrize("bs", [5, 16, 32, 64])
@pytest.mark.parametrize("tokens,layers", [(1, 1), (200, 1), (200, 20), (1500, 2)])
@pytest.mark.parametrize("kind", ["scalar", "head", "layer"])
@pytest.mark.parametrize("value", [0.0, -1.0, float("nan"), float("inf")])
def test_unusable_scale_is_refused(bs, tokens, layers, kind, value):
    nb, slots, caches, linear = _setup(bs, tokens, layers, torch.uint8)
    shape = {"scalar": (), "head": (NH,), "layer": (layers, NH)}[kind if layers > 1 or kind != "layer" else "head"]
    good = torch.full(shape, 0.5, device=DEV)
    bad = good.clone()
    bad.view(-1)[-1] = value
    before = [c.clone() for c in caches]
    gather, scatter = _names("kv_paged_fp8_to_linear", layers), _names("kv_linear_to_paged_fp8", layers)
    outs = [torch.full_like(x, 7.0) for x in linear]
    for name, scales in (("k_scale", (bad, good)), ("v_scale", (good, bad)), ("k_scale", (bad, bad))):
        with pytest.raises(ValueError, match=f"{name}: FP8 scale must be positive and finite"):
            scatter(*linear, *caches, slots, *scales)
        with pytest.raises(ValueError, match=f"{name}: FP8 scale must be positive and finite"):
            gather(*caches, slots, *scales, out_k=outs[0], out_v=outs[1])
        # A slot past the cache is named first.
        worse = slots.clone()
        worse[-1] = nb * bs + 3
        with pytest.raises(ValueError, match=f"slot index {nb * bs + 3} out of bounds"):
            scatter(*linear, *caches, worse, *scales)
    # The value of a scale of the wrong shape is named before its shape.
    with pytest.raises(ValueError, match="k_scale: FP8 scale must be positive and finite"):
        scatter(*linear, *caches, slots, torch.full((NH + 1,), value, device=DEV), good)
    with pytest.raises(ValueError, match="v_scale: FP8 scale must be scalar"):
        scatter(*linear, *caches, slots, good, torch.full((NH + 1,), 0.5, device=DEV))
    for c, b, o in zip(caches, before, outs):
        assert torch.equal(c, b)
        assert bool((o == 7.0).all())
    scatter(*linear, *caches, slots, good, good)
    assert not torch.equal(caches[0], before[0])


def test_threads_on_streams_of_their_own():
    # Refused and accepted calls interleaved by four threads: each call's verdict is its own.
    errors = []

    def work(k):
        try:
            stream = torch.cuda.Stream()
            with torch.cuda.stream(stream):
                for tokens in (64, 3000):
                    nb, slots, caches, linear = _setup(16, tokens, 1, seed=k)
                    bad = slots.clone()
                    bad[k] = nb * 16
                    for _ in range(40):
                        try:
                            musa_aiter.kv_linear_to_paged(*linear, *caches, bad)
                            errors.append("accepted a slot past the cache")
                        except ValueError:
                            pass
                        musa_aiter.kv_linear_to_paged(*linear, *caches, slots)
                        got = musa_aiter.kv_paged_to_linear(*caches, slots)
                    stream.synchronize()
                    if not all(torch.equal(a, b) for a, b in zip(linear, got)):
                        errors.append("wrong rows")
        except Exception as e:  # reported by the main thread
            errors.append(repr(e))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert errors == []
