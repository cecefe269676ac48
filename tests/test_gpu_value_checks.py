"""Slots and FP8 scales that a call must refuse are found on the device, before anything is written.

Calls of at most 256 tokens check them in the kernel that moves them, 16- and 32-bit gathers into new rows in
extra workgroups of that kernel, the others in a kernel ahead of it on the stream.  Either way the error, the untouched caches and outputs
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


@pytest.mark.parametrize("index", [torch.int32, torch.int64])
@pytest.mark.parametrize("batch", [1, 3, 200])
def test_block_tables_are_checked_on_the_device(index, batch):
    bs, cols = 16, 5
    nb = batch * cols + 3
    gen = torch.Generator(device=DEV).manual_seed(batch)
    caches = [torch.randn((nb, NH, HD, bs), generator=gen, device=DEV).to(torch.bfloat16) for _ in range(2)]
    before = [c.clone() for c in caches]
    tables = torch.randperm(nb, generator=gen, device=DEV)[:batch * cols].view(batch, cols).to(index)
    lens = torch.full((batch,), 33, device=DEV, dtype=index)  # three blocks; the last sequence one token less
    lens[-1] = 32
    load, back = musa_aiter.kv_load_and_reshape_flash, musa_aiter.kv_reshape_and_cache_back_flash
    unused = tables.clone()
    unused[-1, 2] = -7      # past ceil(32 / 16): never read
    unused[0, 3:] = nb + 9  # past ceil(33 / 16)
    k, v = load(*caches, unused, lens)
    assert k.shape == (batch, int(lens.max()), NH, HD)
    assert back(k.neg(), v.neg(), *caches, unused, lens)
    assert not torch.equal(caches[0], before[0])
    assert back(k, v, *caches, tables, lens)
    for c, b in zip(caches, before):
        assert torch.equal(c, b)
    for at, value in ((0, nb), (1, -1)):
        bad = tables.clone()
        bad[-1, at] = value
        with pytest.raises(ValueError, match=f"invalid block id {value}"):
            load(*caches, bad, lens)
        with pytest.raises(ValueError, match=f"invalid block id {value}"):
            back(k.neg(), v.neg(), *caches, bad, lens)
    short = lens.clone()
    short[-1] = -2
    with pytest.raises(ValueError, match="seq_lens must be non-negative"):
        load(*caches, tables, short)
    with pytest.raises(ValueError, match="seq_lens exceeds dense sequence length"):
        back(k.neg(), v.neg(), *caches, tables, short)
    with pytest.raises(ValueError, match="smaller than seq_lens max"):
        load(*caches, tables, lens, max_seq_len=31)
    with pytest.raises(ValueError, match="enough columns"):
        load(*caches, tables, lens, max_seq_len=cols * bs + 1)
    wide = torch.zeros((batch, cols * bs + 1, NH, HD), device=DEV, dtype=torch.bfloat16)
    long = lens.clone()
    long[-1] = cols * bs + 1
    with pytest.raises(ValueError, match="enough columns"):
        back(wide, wide, *caches, tables, long)
    for c, b in zip(caches, before):
        assert torch.equal(c, b)


@pytest.mark.parametrize("row", [512, 1024, 1536])  # 2-byte elements: rows of 1, 2 and 3 KiB
@pytest.mark.parametrize("items,name", [(1, "per_layer"), (300, "all_layer"), (300, "all_layer_lf_pf"),
                                        (2500, "all_layer_lf_pf"), (2500, "per_layer_pf_lf")])
def test_hicache_page_indices_are_checked_on_the_device(row, items, name):
    layers, pages = 3, items + 9
    gen = torch.Generator(device=DEV).manual_seed(items + row)
    call = getattr(musa_aiter, f"hicache_transfer_kv_{name}")
    lf, pf = (layers, pages, row), (pages, layers, row)
    shapes = {"per_layer": (lf, lf), "all_layer": (lf, lf), "all_layer_lf_pf": (lf, pf), "per_layer_pf_lf": (pf, lf)}
    src, dst = ([torch.randn(shape, generator=gen, device=DEV).to(torch.bfloat16) for _ in range(2)]
                for shape in shapes[name])
    before = [d.clone() for d in dst]
    src_idx, dst_idx = (torch.randperm(pages, generator=gen, device=DEV)[:items] for _ in range(2))
    for at in (0, items - 1):
        for which in (0, 1):
            for value, text in ((pages, "out of range"), (-2, "must be -1 or non-negative")):
                idx = [src_idx.clone(), dst_idx.clone()]
                idx[which][at] = value
                with pytest.raises(ValueError, match=text):
                    call(src[0], dst[0], src[1], dst[1], *idx)
    for d, b in zip(dst, before):
        assert torch.equal(d, b)
    if items > 4:
        src_idx[3], dst_idx[2] = -1, -1       # skipped pairs
        dst_idx[1] = dst_idx[items - 1]       # the later pair wins
    call(src[0], dst[0], src[1], dst[1], src_idx, dst_idx)
    moved = [(int(s), int(d)) for s, d in zip(src_idx, dst_idx) if s >= 0 and d >= 0]
    from_to = dict((d, s) for s, d in moved)
    s_i = torch.tensor([from_to[d] for d in from_to], device=DEV)
    d_i = torch.tensor(list(from_to), device=DEV)
    only = slice(0, 1) if name.startswith("per_layer") else slice(None)
    for s, d, b in zip(src, dst, before):
        s_lf = s if shapes[name][0] is lf else s.transpose(0, 1)
        want = b.clone()
        want_lf = want if shapes[name][1] is lf else want.transpose(0, 1)
        want_lf[only, d_i] = s_lf[only, s_i]
        assert torch.equal(d, want)


@pytest.mark.parametrize("layers", [1, 3])
def test_native_argument_checks_agree_with_the_python_layer(layers, monkeypatch):
    """Every form of arguments gives one result and one error whether the host module takes the call or the
    Python layer does: other dtypes, strides, shapes, scale kinds and devices among them."""
    from musa_aiter.ops import _hip

    bs, tokens = 16, 40
    nb, slots, caches, linear = _setup(bs, tokens, layers)
    _, _, codes, _ = _setup(bs, tokens, layers, torch.uint8)
    head = torch.full((NH,), 0.5, device=DEV)
    strided = torch.stack(linear, -1)
    wide = [torch.cat([c, c], -1)[..., :bs] for c in caches]
    per_layer = torch.full((layers, NH), 0.5, device=DEV)
    empty = [x[..., :0, :, :] for x in linear]

    def store(k, v, kc, vc, s):
        got = [kc.clone(memory_format=torch.preserve_format), vc.clone(memory_format=torch.preserve_format)]
        _names("kv_linear_to_paged", layers)(k, v, *got, s)
        return got

    def quant(k, v, s, ks, vs, kc=codes[0], vc=codes[1], **kw):
        got = [kc.clone(), vc.clone()]
        _names("kv_linear_to_paged_fp8", layers)(k, v, *got, s, ks, vs, **kw)
        return [g.view(torch.uint8) for g in got]

    load = _names("kv_paged_to_linear", layers)
    dequant = _names("kv_paged_fp8_to_linear", layers)
    calls = [
        lambda: store(*linear, *caches, slots),
        lambda: store(*linear, *caches, slots.to(torch.int32)),
        lambda: store(*linear, *caches, slots.repeat_interleave(2)[::2]),
        lambda: store(*linear, *caches, slots.cpu()),
        lambda: store(*linear, *caches, slots[:-1]),
        lambda: store(*linear, *caches, slots.view(1, -1)),
        lambda: store(*linear, *caches, slots.float()),
        lambda: store(*(x.float() for x in linear), *caches, slots),
        lambda: store(linear[0], linear[1].float(), *caches, slots),
        lambda: store(strided[..., 0], strided[..., 1], *caches, slots),
        lambda: store(*linear, *wide, slots),
        lambda: store(*linear, caches[0], caches[1].half(), slots),
        lambda: store(*linear, caches[0], caches[1][..., :-1], slots),
        lambda: store(*(x[..., :-1] for x in linear), *caches, slots),
        lambda: store(*(x.double() for x in linear), *(c.double() for c in caches), slots),
        lambda: store(*empty, *caches, slots[:0]),
        lambda: load(*caches, slots),
        lambda: load(*wide, slots),
        lambda: load(*caches, slots[:0]),
        lambda: load(caches[0], caches[1].half(), slots),
        lambda: load(*(c.cpu() for c in caches), slots.cpu()),
        lambda: load(*caches, slots, fill_skipped="preserve"),
        lambda: load(*caches, torch.where(slots % 3 == 0, -1, slots)),
        lambda: quant(*linear, slots, head, head),
        lambda: quant(*linear, slots, 0.5, head),
        lambda: quant(*linear, slots, head[:1], 0.25),
        lambda: quant(*linear, slots, head.double(), head.cpu()),
        lambda: quant(*linear, slots, head.repeat(2)[::2], head),
        lambda: quant(*linear, slots, per_layer, head),
        lambda: quant(*linear, slots, per_layer, per_layer),
        lambda: quant(*linear, slots, head[:0], head),
        lambda: quant(*linear, slots, head, head, fp8_format="FP8_E5M2"),
        lambda: quant(*linear, slots, head, head, fp8_format="e5m2"),
        lambda: quant(*linear, slots, head, head, fp8_format="e3m4"),
        lambda: quant(*linear, slots, head, head, codes[0].view(torch.float8_e4m3fn), codes[1].view(torch.float8_e5m2)),
        lambda: quant(*linear, slots, head, head, codes[0].view(torch.int8), codes[1]),
        lambda: quant(*(x.double() for x in linear), slots, head, head),
        lambda: quant(linear[0], linear[1].float(), slots, head, head),
        lambda: quant(*empty, slots[:0], head, -head),
        lambda: dequant(*codes, slots, head, head),
        lambda: dequant(*codes, slots, per_layer, per_layer, out_dtype=torch.float32),
        lambda: dequant(*codes, slots, head, 0.5, out_dtype=torch.float64),
        lambda: dequant(*codes, slots, head, head, out_dtype=torch.float16, fp8_format="E4M3FN"),
        lambda: dequant(*codes, slots[:0], head, head),
        lambda: dequant(*codes, slots.to(torch.int16), head, head),
    ]

    def outcome(call):
        try:
            return [t.cpu() for t in call()]
        except Exception as e:
            return type(e), str(e)

    native = []
    real = _hip.paged_native
    monkeypatch.setattr(_hip, "paged_native", lambda *a, **k: (native.append(real(*a, **k)), native[-1])[1])
    outcome(calls[0]), outcome(calls[16])  # the stream's check and claim sets exist from here on
    first = []
    for call in calls:
        native.clear()
        first.append((outcome(call), bool(native) and native[-1] is not None))
    monkeypatch.setattr(_hip, "paged_native", lambda *a, **k: None)
    taken = 0
    for k, (call, (got, was_native)) in enumerate(zip(calls, first)):
        want = outcome(call)
        taken += was_native
        assert type(got) is type(want), (k, got, want)
        if isinstance(got, tuple):
            assert got == want, k
            assert not was_native, k
        else:
            assert all(a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride() and
                       torch.equal(a.view(torch.uint8), b.view(torch.uint8)) for a, b in zip(got, want)), k
    assert taken >= 8  # the plain forms do take the native path


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.uint8])
@pytest.mark.parametrize("bs", [5, 8, 16, 32, 64])
@pytest.mark.parametrize("tokens,layers", [(200, 20), (257, 1), (1500, 20), (16385, 2)])  # 16,385: a 65th share
def test_gather_into_new_rows_checks_itself_in_shares(dtype, bs, tokens, layers):
    # Without outputs of the caller's the launch that gathers (16- and 32-bit elements, aligned blocks) also
    # checks: the error, and the rows of the next call, are as before.  Bad slots at the edges of the waves'
    # shares of 256.
    nb, slots, caches, _ = _setup(bs, tokens, layers, dtype)
    fp8 = dtype is torch.uint8
    gather = _names("kv_paged_fp8_to_linear" if fp8 else "kv_paged_to_linear", layers)
    scales = [torch.full((NH,), s, device=DEV) for s in (0.5, 0.25)] if fp8 else []
    good = slots.clone()
    good[tokens // 3] = -1
    outs = [torch.full(((layers,) if layers > 1 else ()) + (tokens, NH, HD), 7.0, device=DEV,
                        dtype=torch.bfloat16 if fp8 else dtype) for _ in range(2)]
    kwargs = {"out_dtype": torch.bfloat16} if fp8 else {}
    want = gather(*caches, good, *scales, out_k=outs[0], out_v=outs[1], **kwargs)
    for at in sorted({0, 255, 256, 64 * 256 - 1, 64 * 256, tokens - 1}):
        if at >= tokens:
            continue
        bad = good.clone()
        bad[at] = nb * bs
        with pytest.raises(ValueError, match=f"slot index {nb * bs} out of bounds"):
            gather(*caches, bad, *scales, **kwargs)
    for k in range(2 * len(scales)):
        bad_scales = [s.clone() for s in scales]
        bad_scales[k // 2][-(k % 2)] = float("inf")
        with pytest.raises(ValueError, match="FP8 scale must be positive and finite"):
            gather(*caches, good, *bad_scales, **kwargs)
    for x, y in zip(gather(*caches, good, *scales, **kwargs), want):
        assert torch.equal(x.view(torch.int16 if x.element_size() == 2 else torch.int32),
                           y.view(torch.int16 if y.element_size() == 2 else torch.int32))
