"""GPU parity of caches whose block size is a multiple of 64, against the oracle.

Such blocks are copied in units of 64 columns by kernels of their own, with 64-token tiles and a
two-register slot window.  The mappings put runs across tile and unit edges, full units, partial
units, single tokens, skipped and repeated slots into one call; token counts sit on both sides of
the forms' limits (256 tokens: per-token gathers and in-kernel duplicate resolution).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import musa_aiter
from oracle import kv_oracle as ko
from tests.kvgen import bits, make_slots, random_payload
from tests.test_gpu_destination_order import tricky_slots

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _round_trip(dtype, layers, nh, hd, bs, slots, nb):
    gen = torch.Generator().manual_seed(len(slots) + bs)
    kc, vc = (random_payload((layers, nb, nh, hd, bs), dtype, gen) for _ in range(2))
    kl, vl = (random_payload((layers, len(slots), nh, hd), dtype, gen) for _ in range(2))
    s_d = torch.from_numpy(slots).to(DEV)
    ok, ov = musa_aiter.kv_paged_to_linear_multi_layer(kc.to(DEV), vc.to(DEV), s_d)
    assert np.array_equal(bits(ok), ko.paged_to_linear_multi_layer(bits(kc), slots))
    assert np.array_equal(bits(ov), ko.paged_to_linear_multi_layer(bits(vc), slots))
    kc_d, vc_d = kc.to(DEV), vc.to(DEV)
    musa_aiter.kv_linear_to_paged_multi_layer(kl.to(DEV), vl.to(DEV), kc_d, vc_d, s_d)
    want_k, want_v = bits(kc).copy(), bits(vc).copy()
    ko.linear_to_paged_multi_layer(bits(kl), want_k, slots)
    ko.linear_to_paged_multi_layer(bits(vl), want_v, slots)
    assert np.array_equal(bits(kc_d), want_k)
    assert np.array_equal(bits(vc_d), want_v)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("bs", [32, 64, 128, 192])
@pytest.mark.parametrize("nh, hd", [(4, 64), (3, 40)])
@pytest.mark.parametrize("layers,tokens,kind", [
    (1, 1, "sequences"),
    (1, 63, "decode"),
    (2, 256, "decode"),
    (1, 200, "duplicates"),
    (1, 257, "random"),
    (2, 700, "sequences"),
    (2, 900, "skips"),
    (1, 1500, "duplicates"),
    (3, 1500, "decode"),
])
def test_wide_blocks_match_oracle(dtype, bs, nh, hd, layers, tokens, kind):
    slots, nb = make_slots(kind, np.random.default_rng(tokens + bs), block_size=bs, tokens=tokens)
    _round_trip(dtype, layers, nh, hd, bs, slots, nb)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("bs", [32, 64, 128])
@pytest.mark.parametrize("layers", [3, 17])  # 17: past 32 planes, the XCD-contiguous order
def test_wide_blocks_in_destination_order(dtype, bs, layers):
    slots = tricky_slots(np.random.default_rng(bs), 12, bs)
    assert len(slots) * 4 >= 12 * bs
    _round_trip(dtype, layers, 2, 72, bs, slots, 12)


@pytest.mark.parametrize("bs", [32, 64, 128])
def test_wide_blocks_through_block_tables(bs):
    rng = np.random.default_rng(bs)
    nh, hd, nb, batch = 2, 64, 9, 3
    lengths = np.array([2 * bs, bs // 2 + 1, bs + 6])
    tables = rng.permutation(nb)[:batch * 2].reshape(batch, 2)
    gen = torch.Generator().manual_seed(3)
    kc, vc = (random_payload((nb, nh, hd, bs), torch.bfloat16, gen) for _ in range(2))
    dk, dv = (random_payload((batch, 2 * bs, nh, hd), torch.bfloat16, gen) for _ in range(2))
    t_d, l_d = torch.from_numpy(tables).to(DEV), torch.from_numpy(lengths).to(DEV)
    got = musa_aiter.kv_load_and_reshape_flash(kc.to(DEV), vc.to(DEV), t_d, l_d)
    pos = np.arange(2 * bs)
    slots = np.where(pos < lengths[:, None], tables[:, pos // bs] * bs + pos % bs, -1).reshape(-1)
    for out, cache in zip(got, (kc, vc)):
        assert np.array_equal(bits(out).reshape(-1, nh, hd), ko.paged_to_linear(bits(cache), slots))
    kc_d, vc_d = kc.to(DEV), vc.to(DEV)
    musa_aiter.kv_reshape_and_cache_back_flash(dk.to(DEV), dv.to(DEV), kc_d, vc_d, t_d, l_d)
    for cache, cache_d, dense in ((kc, kc_d, dk), (vc, vc_d, dv)):
        want = bits(cache).copy()
        ko.linear_to_paged(bits(dense).reshape(-1, nh, hd), want, slots)
        assert np.array_equal(bits(cache_d), want)


@pytest.mark.parametrize("fmt", ["e4m3", "e5m2"])
@pytest.mark.parametrize("lin", ["bfloat16", "float32"])
@pytest.mark.parametrize("bs", [64, 128])
@pytest.mark.parametrize("nh, hd", [(8, 128), (5, 72)])
@pytest.mark.parametrize("tokens,kind", [
    (1, "sequences"),
    (61, "decode"),
    (256, "decode"),
    (200, "duplicates"),
    (700, "decode"),
    (900, "skips"),
    (0, "tricky"),              # destination order
])
def test_wide_fp8_blocks_match_oracle(fmt, lin, bs, nh, hd, tokens, kind):
    rng = np.random.default_rng(tokens + bs)
    if kind == "tricky":
        nb = 12
        slots = tricky_slots(rng, nb, bs)
        assert len(slots) * 4 >= nb * bs
    else:
        slots, nb = make_slots(kind, rng, block_size=bs, tokens=tokens, spare_blocks=40)
    gen = torch.Generator().manual_seed(tokens)
    dtype = getattr(torch, lin)
    # Every eighth row far outside the fast quotient's range, so that tiles of both encoders appear.
    x = [(torch.randn((len(slots), nh, hd), generator=gen) * 3).to(dtype) for _ in range(2)]
    for t in x:
        t[3::8] *= 2.0 ** 70
    scales = [torch.rand(nh, generator=gen) * 0.02 + 0.001, torch.tensor(0.0071)]
    caches = [torch.randint(0, 256, (nb, nh, hd, bs), dtype=torch.uint8, generator=gen) for _ in range(2)]
    s_d = torch.from_numpy(slots).to(DEV)
    got = musa_aiter.kv_paged_fp8_to_linear(*(c.to(DEV) for c in caches), s_d, *(s.to(DEV) for s in scales),
                                            out_dtype=dtype, fp8_format=fmt)
    for out, cache, scale in zip(got, caches, scales):
        assert np.array_equal(bits(out), ko.paged_fp8_to_linear(cache.numpy(), slots, scale.numpy(), fmt, lin))
    caches_d = [c.to(DEV) for c in caches]
    musa_aiter.kv_linear_to_paged_fp8(*(t.to(DEV) for t in x), *caches_d, s_d, *(s.to(DEV) for s in scales),
                                      fp8_format=fmt)
    for t, cache, cache_d, scale in zip(x, caches, caches_d, scales):
        want = cache.numpy().copy()
        ko.linear_to_paged_fp8(t.to(torch.float32).numpy(), want, slots, scale.numpy(), fmt)
        assert np.array_equal(cache_d.cpu().numpy(), want)


def _fp8_round_trip(layers, nh, hd, bs, slots, nb):
    gen = torch.Generator().manual_seed(layers + len(slots))
    x = [(torch.randn((layers, len(slots), nh, hd), generator=gen) * 3).to(torch.bfloat16) for _ in range(2)]
    scales = [torch.rand((layers, nh), generator=gen) * 0.02 + 0.001 for _ in range(2)]
    caches = [torch.randint(0, 256, (layers, nb, nh, hd, bs), dtype=torch.uint8, generator=gen) for _ in range(2)]
    s_d, scales_d, caches_d = torch.from_numpy(slots).to(DEV), [s.to(DEV) for s in scales], [c.to(DEV) for c in caches]
    got = musa_aiter.kv_paged_fp8_to_linear_multi_layer(*caches_d, s_d, *scales_d, out_dtype=torch.bfloat16)
    musa_aiter.kv_linear_to_paged_fp8_multi_layer(*(t.to(DEV) for t in x), *caches_d, s_d, *scales_d)
    for out, t, cache, cache_d, scale in zip(got, x, caches, caches_d, scales):
        for layer in range(layers):
            assert np.array_equal(bits(out[layer]), ko.paged_fp8_to_linear(cache[layer].numpy(), slots,
                                                                           scale[layer].numpy(), "e4m3", "bfloat16"))
            want = cache[layer].numpy().copy()
            ko.linear_to_paged_fp8(t[layer].to(torch.float32).numpy(), want, slots, scale[layer].numpy(), "e4m3")
            assert np.array_equal(cache_d[layer].cpu().numpy(), want)


# By elements moved (tokens x rows x planes) a call on wide blocks takes the element kernel, the wide kernels'
# forms for small launches (one-wave workgroups or 16-token tiles for gathers, 8-token tiles for scatters) or
# their large ones.  About 540 tokens of every run shape: with 2,048 rows the forms change between one and three
# layers, 17 layers take the order of many planes; a cache of 12 blocks is scattered in destination order, one of
# 40 in token order.
@pytest.mark.parametrize("layers, nh, hd", [(1, 16, 128), (2, 16, 128), (3, 16, 128), (1, 17, 120), (2, 17, 120),
                                            (3, 17, 120), (1, 8, 128), (17, 8, 128)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.uint8])
@pytest.mark.parametrize("nb", [12, 40])
def test_wide_forms_by_elements_match_oracle(layers, nh, hd, dtype, nb):
    slots = tricky_slots(np.random.default_rng(layers), 12, 64)
    if dtype is torch.uint8:
        _fp8_round_trip(layers, nh, hd, 64, slots, nb)
    else:
        _round_trip(dtype, layers, nh, hd, 64, slots, nb)


# One layer of 1,024 rows: 128 tokens are 2**18 elements, the limits 128 to 2,048 tokens.
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.uint8])
@pytest.mark.parametrize("tokens", [128, 256, 384, 512, 640, 1024, 1536, 2048])
@pytest.mark.parametrize("below", [0, 1])
def test_wide_calls_at_the_limits_match_oracle(dtype, tokens, below):
    slots, nb = make_slots("skips", np.random.default_rng(tokens), block_size=64, tokens=tokens - below)
    if dtype is torch.uint8:
        _fp8_round_trip(1, 8, 128, 64, slots, nb)
    else:
        _round_trip(dtype, 1, 8, 128, 64, slots, nb)


def test_wide_fp8_blocks_with_more_row_chunks_than_a_grid_holds():
    # 32,769 heads of 128: 65,538 chunks of 64 rows, past the per-wave kernels' grid; the element kernel moves them.
    nh, hd, slots = 32769, 128, np.array([5, 40])
    gen = torch.Generator().manual_seed(1)
    x = [torch.randn((2, nh, hd), generator=gen) for _ in range(2)]
    scales = [torch.tensor(0.02), torch.tensor(0.03)]
    caches_d = [torch.zeros((1, nh, hd, 64), dtype=torch.uint8, device=DEV) for _ in range(2)]
    s_d, scales_d = torch.from_numpy(slots).to(DEV), [s.to(DEV) for s in scales]
    musa_aiter.kv_linear_to_paged_fp8(*(t.to(DEV) for t in x), *caches_d, s_d, *scales_d)
    got = musa_aiter.kv_paged_fp8_to_linear(*caches_d, s_d, *scales_d, out_dtype=torch.float32)
    for t, cache_d, out, scale in zip(x, caches_d, got, scales):
        # One-slot blocks: the same codes without the 62 columns that no token writes.
        want = np.zeros((2, nh, hd, 1), np.uint8)
        ko.linear_to_paged_fp8(t.numpy(), want, np.array([0, 1]), scale.numpy(), "e4m3")
        assert np.array_equal(cache_d[0, :, :, slots].permute(2, 0, 1).cpu().numpy(), want[..., 0])
        assert int((cache_d != 0).sum()) == int((want != 0).sum())
        assert np.array_equal(bits(out), ko.paged_fp8_to_linear(want, np.array([0, 1]), scale.numpy(), "e4m3", "float32"))


# The forms by elements over every layout that reaches them: rows of K and V apart, merged, and at a token stride
# of the caller's; dense tensors through block tables.  A token of 23 x 88 = 2,024 elements is no whole chunk; slots are
# skipped and repeated.  Every form only moves elements: results are equal bit for bit.
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("bs", [64, 192])
@pytest.mark.parametrize("tokens", [300, 700, 1500])  # 1.2, 2.8 and 6 Mi elements of K and V
@pytest.mark.parametrize("layout", ["merged", "strided", "dense"])
def test_wide_forms_in_every_layout(dtype, bs, tokens, layout):
    nh, hd, nb = 23, 88, tokens // bs + 5
    gen = torch.Generator(device=DEV).manual_seed(tokens)
    caches = [torch.randn((nb, nh, hd, bs), generator=gen, device=DEV).to(dtype) for _ in range(2)]

    def paged_rows(cache):
        return cache.permute(0, 3, 1, 2).reshape(nb * bs, nh, hd)

    if layout == "dense":
        batch, cols = 3, nb // 3
        tables = torch.randperm(nb, generator=gen, device=DEV)[:batch * cols].view(batch, cols)
        lens = torch.tensor([cols * bs - 7, bs // 2 + 1, cols * bs], device=DEV)
        pos = torch.arange(cols * bs, device=DEV)
        slots = torch.where(pos < lens[:, None], tables[:, pos // bs] * bs + pos % bs, -1).reshape(-1)
    else:
        runs = torch.arange(nb * bs, device=DEV).view(-1, 8)
        slots = runs[torch.randperm(len(runs), generator=gen, device=DEV)].reshape(-1)[:tokens].clone()
        slots[:64] = torch.arange(64, 128, device=DEV)           # a unit, in order
        slots[64::37] = -1
        slots[70] = slots[tokens - 3]                            # the later one wins
    moves = slots >= 0
    rows = [torch.randn((len(slots), nh, hd), generator=gen, device=DEV).to(dtype) for _ in range(2)]
    want = [torch.where(moves[:, None, None], paged_rows(c)[slots.clamp(min=0)], 0) for c in caches]
    stored = [paged_rows(c).clone() for c in caches]
    last = {int(s): t for t, s in enumerate(slots.tolist()) if s >= 0}
    at, by = (torch.tensor(x, device=DEV) for x in (list(last), list(last.values())))
    for s, r in zip(stored, rows):
        s[at] = r[by]
    if layout == "merged":
        got = musa_aiter.kv_paged_to_merged_linear(*caches, slots).unbind(1)
        musa_aiter.kv_merged_linear_to_paged(torch.stack(rows, 1), *caches, slots)
    elif layout == "strided":
        pads = [torch.full((tokens, nh + 2, hd), 5.0, dtype=dtype, device=DEV) for _ in range(2)]
        got = [p[:, :nh] for p in pads]
        musa_aiter.kv_paged_to_linear(*caches, slots, out_k=got[0], out_v=got[1])
        assert all(bool((p[:, nh:] == 5.0).all()) for p in pads)
        musa_aiter.kv_linear_to_paged(*(torch.cat([r, r[:, :2]], 1)[:, :nh] for r in rows), *caches, slots)
    else:
        got = [g.reshape(-1, nh, hd) for g in musa_aiter.kv_load_and_reshape_flash(*caches, tables, lens)]
        musa_aiter.kv_reshape_and_cache_back_flash(*(r.view(batch, -1, nh, hd) for r in rows), *caches, tables, lens)
    for g, w in zip(got, want):
        assert torch.equal(g, w)
    for c, s in zip(caches, stored):
        assert torch.equal(paged_rows(c), s)
