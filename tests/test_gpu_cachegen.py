"""GPU parity: CacheGen-style codec vs oracle/cachegen_oracle.py, bit-exact.

Restates the reference's tests (op_tests/test_kv_transfer.py:218-250) on ROCm and adds: every
input dtype and bin count against the oracle at ragged sizes (bins, codebook and CDF compared
bit for bit), the native-kernel rounding behind MUSA_AITER_NATIVE_KV_TRANSFER=1, known answers
that separate the two roundings and the two scale formulas, misaligned and non-contiguous
inputs, constant and NaN tensors, a 2**26-element tensor against the oracle plus size-free
properties, decode into every output element size with codebooks of 2..256 entries, the
out-of-range error, and both reference-named C entries called through ctypes.
"""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

import musa_aiter
from musa_aiter.ops import _hip
from oracle import cachegen_oracle as cg

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _np_input(x: torch.Tensor):
    if x.dtype == torch.bfloat16:
        return x.cpu().view(torch.int16).numpy().view(np.uint16), "bfloat16"
    return x.cpu().numpy(), str(x.dtype).split(".")[1]


def _bits(a) -> np.ndarray:
    return np.asarray(a, dtype=np.float32).view(np.uint32)


def _check_encode(x: torch.Tensor, num_bins: int, *, native: bool = False):
    enc, book, cdf = musa_aiter.kv_cachegen_encode(x, num_bins=num_bins)
    torch.cuda.synchronize()
    raw, name = _np_input(x)
    e_ref, b_ref, c_ref = cg.encode(raw, num_bins, native=native, dtype=name)
    assert enc.dtype == torch.uint8 and tuple(enc.shape) == tuple(x.shape)
    np.testing.assert_array_equal(enc.cpu().numpy(), e_ref)
    np.testing.assert_array_equal(_bits(book.cpu().numpy()), _bits(b_ref))
    np.testing.assert_array_equal(_bits(cdf.cpu().numpy()), _bits(c_ref))
    return enc, book, cdf


# ---- the reference's own tests ---------------------------------------------------------------

def test_reference_roundtrip_and_cdf():
    tensor = torch.linspace(-1.0, 1.0, steps=17, dtype=torch.float32, device=DEV).reshape(1, 17)
    encoded, codebook, cdf = musa_aiter.kv_cachegen_encode(tensor, num_bins=16)
    decoded = musa_aiter.kv_cachegen_decode(encoded, codebook, dtype=tensor.dtype)
    assert encoded.dtype == torch.uint8
    assert codebook.shape == (16,) and cdf.shape == (17,)
    assert cdf[0] == 0 and cdf[-1] == 1
    assert bool(torch.all(cdf[1:] >= cdf[:-1]))
    assert decoded.shape == tensor.shape
    assert torch.max(torch.abs(decoded - tensor)) <= (2.0 / 15.0)
    _check_encode(tensor, 16)


def test_reference_constant_tensor():
    tensor = torch.full((2, 3), 5.0, device=DEV)
    encoded, codebook, cdf = musa_aiter.kv_cachegen_encode(tensor, num_bins=8)
    decoded = musa_aiter.kv_cachegen_decode(encoded, codebook)
    assert encoded.max() == 0
    torch.testing.assert_close(decoded, tensor)
    assert cdf[0] == 0 and bool(torch.all(cdf[1:] == 1))
    _check_encode(tensor, 8)


def test_reference_rejects_invalid_inputs():
    with pytest.raises(ValueError):
        musa_aiter.kv_cachegen_encode(torch.arange(4, dtype=torch.int32, device=DEV))
    with pytest.raises(ValueError):
        musa_aiter.kv_cachegen_decode(torch.zeros(2, dtype=torch.int32, device=DEV), torch.zeros(4, device=DEV))
    with pytest.raises(ValueError, match="num_bins must be in"):
        musa_aiter.kv_cachegen_encode(torch.zeros(4, device=DEV), num_bins=257)
    with pytest.raises(ValueError, match="1-D with 2..256 bins"):
        musa_aiter.kv_cachegen_decode(torch.zeros(2, dtype=torch.uint8, device=DEV), torch.zeros(1, device=DEV))
    with pytest.raises(ValueError, match="same device"):
        musa_aiter.kv_cachegen_decode(torch.zeros(2, dtype=torch.uint8, device=DEV), torch.zeros(4))
    with pytest.raises(ValueError, match="floating dtype"):
        musa_aiter.kv_cachegen_decode(torch.zeros(2, dtype=torch.uint8, device=DEV),
                                      torch.zeros(4, dtype=torch.int32, device=DEV))


# ---- parity with the oracle -------------------------------------------------------------------

@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16, torch.float64])
@pytest.mark.parametrize("num_bins", [2, 3, 16, 255, 256])
def test_encode_matches_oracle(dtype, num_bins):
    g = torch.Generator().manual_seed(num_bins)
    for n in (1, 2, 3, 15, 17, 255, 4099, 100003, (1 << 20) + 7):
        x = (torch.randn(n, generator=g, dtype=torch.float64) * 3 + 0.5).to(dtype).to(DEV)
        _check_encode(x, num_bins)


@pytest.mark.parametrize("num_bins", [2, 16, 256])
def test_encode_native_rounding(monkeypatch, num_bins):
    monkeypatch.setenv("MUSA_AITER_NATIVE_KV_TRANSFER", "1")
    g = torch.Generator().manual_seed(7)
    for n in (5, 1000, 123457):
        x = (torch.randn(n, generator=g) * 2).to(DEV)
        _check_encode(x, num_bins, native=True)
        # ties: quarter steps over a range that makes the scale exact
        q = (torch.randint(0, 4 * (num_bins - 1) + 1, (n,), generator=g).float() / 4).to(DEV)
        q[0], q[-1] = 0.0, float(num_bins - 1)
        _check_encode(q, num_bins, native=True)
    # other dtypes keep the torch-path rounding, as in the reference
    _check_encode(torch.tensor([0.0, 0.5, 1.5, 2.5, 3.0], dtype=torch.float16, device=DEV), 4, native=True)


def test_known_answers_rounding_and_scale(monkeypatch):
    x = torch.tensor([0.0, 0.5, 1.5, 2.5, 3.0], device=DEV)
    assert musa_aiter.kv_cachegen_encode(x, num_bins=4)[0].tolist() == [0, 0, 2, 2, 3]
    x2 = torch.tensor([0.0, 0.51109046, 1.8889903], device=DEV)
    assert musa_aiter.kv_cachegen_encode(x2, num_bins=232)[0].tolist()[1] == 63
    monkeypatch.setenv("MUSA_AITER_NATIVE_KV_TRANSFER", "1")
    assert musa_aiter.kv_cachegen_encode(x, num_bins=4)[0].tolist() == [0, 1, 2, 3, 3]


def test_misaligned_and_strided_inputs():
    g = torch.Generator().manual_seed(3)
    base = torch.randn(4 * 4096 + 9, generator=g).to(DEV)
    for off in (1, 2, 3):
        _check_encode(base[off:off + 4096 * 4 + 5], 256)  # 4-byte aligned only: scalar path
    m = torch.randn(300, 77, generator=g).to(DEV)
    _check_encode(m.t(), 64)  # non-contiguous: encoded keeps the logical order
    h = torch.randn(2 * 999, generator=g).to(torch.float16).to(DEV)
    _check_encode(h[1:], 200)


def test_constant_and_special_tensors():
    _check_encode(torch.full((1000,), -0.0, device=DEV), 5)
    _check_encode(torch.full((3, 5), 2.0, dtype=torch.bfloat16, device=DEV), 256)
    _check_encode(torch.tensor([1.0, 1.0, 2.0], device=DEV), 2)
    # NaN anywhere: range and codebook are NaN, every bin is 0 (the reference's behaviour here depends on
    # the device; this is the defined behaviour of this implementation)
    x = torch.randn(5000).to(DEV)
    x[1234] = float("nan")
    enc, book, cdf = musa_aiter.kv_cachegen_encode(x, num_bins=16)
    assert int(enc.max()) == 0 and bool(torch.isnan(book).all())
    assert cdf.tolist() == [0.0] + [1.0] * 16


def test_float8_input_is_widened_first():
    x = (torch.randn(1000) * 4).to(torch.float8_e4m3fn)
    enc, book, cdf = musa_aiter.kv_cachegen_encode(x.to(DEV), num_bins=32)
    e_ref, b_ref, c_ref = cg.encode(x.float().numpy(), 32)
    np.testing.assert_array_equal(enc.cpu().numpy(), e_ref)
    np.testing.assert_array_equal(_bits(book.cpu().numpy()), _bits(b_ref))
    np.testing.assert_array_equal(_bits(cdf.cpu().numpy()), _bits(c_ref))


def test_encode_on_side_stream():
    x = torch.randn(1 << 18).to(DEV)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        enc, book, cdf = musa_aiter.kv_cachegen_encode(x, num_bins=128)
    s.synchronize()
    e_ref, b_ref, c_ref = cg.encode(x.cpu().numpy(), 128)
    np.testing.assert_array_equal(enc.cpu().numpy(), e_ref)
    np.testing.assert_array_equal(_bits(cdf.cpu().numpy()), _bits(c_ref))


def test_large_tensor_parity_and_properties():
    n = 1 << 26
    x = torch.randn(n, device=DEV) * 0.7 + 0.1
    enc, book, cdf = musa_aiter.kv_cachegen_encode(x, num_bins=256)
    torch.cuda.synchronize()
    e_ref, b_ref, c_ref = cg.encode(x.cpu().numpy(), 256)
    np.testing.assert_array_equal(enc.cpu().numpy(), e_ref)
    np.testing.assert_array_equal(_bits(book.cpu().numpy()), _bits(b_ref))
    np.testing.assert_array_equal(_bits(cdf.cpu().numpy()), _bits(c_ref))
    counts = torch.bincount(enc.long(), minlength=256)
    assert int(counts.sum()) == n and float(cdf[-1]) == 1.0
    dec = musa_aiter.kv_cachegen_decode(enc, book)
    lo, hi = float(x.min()), float(x.max())
    # half a bin, plus a few float32 ulps for the rounded codebook entries and scale
    bound = (hi - lo) / 255 / 2 + 8 * float(np.finfo(np.float32).eps) * max(abs(lo), abs(hi))
    assert float((dec - x).abs().max()) <= bound


# ---- decode -----------------------------------------------------------------------------------

@pytest.mark.parametrize("out_dtype", [None, torch.float16, torch.bfloat16, torch.float64, torch.int32,
                                       torch.complex64, torch.complex128, torch.bool, torch.int8])
@pytest.mark.parametrize("table_len", [2, 17, 255, 256])
def test_decode_matches_indexing(out_dtype, table_len):
    g = torch.Generator().manual_seed(table_len)
    book = torch.randn(table_len, generator=g) * 50
    for n in (1, 7, 16, 33, 4099, 300001):
        codes = torch.randint(0, table_len, (n,), generator=g, dtype=torch.uint8)
        out = musa_aiter.kv_cachegen_decode(codes.to(DEV), book.to(DEV), dtype=out_dtype)
        # the reference's expression, codebook[encoded.long()].to(dtype), with its cast on the device
        ref = book.to(DEV)[codes.to(DEV).long()]
        ref = (ref if out_dtype is None else ref.to(out_dtype)).cpu()
        assert out.dtype == ref.dtype and out.shape == ref.shape
        assert torch.equal(out.cpu(), ref)


def test_decode_codebook_dtypes_and_layouts():
    g = torch.Generator().manual_seed(5)
    codes = torch.randint(0, 100, (3, 5000), generator=g, dtype=torch.uint8)
    for book in (torch.randn(100, generator=g, dtype=torch.float64), torch.randn(100, generator=g).half(),
                 torch.randn(300, generator=g)[::3]):
        out = musa_aiter.kv_cachegen_decode(codes.to(DEV), book.to(DEV))
        assert torch.equal(out.cpu(), book[codes.long()])
    odd = codes.to(DEV).t()  # non-contiguous codes
    book = torch.randn(100, generator=g)
    assert torch.equal(musa_aiter.kv_cachegen_decode(odd, book.to(DEV)).cpu(), book[codes.t().long()])
    flat = torch.randint(0, 100, (4099,), generator=g, dtype=torch.uint8).to(DEV)
    for off in (1, 2, 3):  # misaligned codes: scalar path
        assert torch.equal(musa_aiter.kv_cachegen_decode(flat[off:], book.to(DEV)).cpu(), book[flat[off:].cpu().long()])


def test_decode_rejects_bins_past_codebook():
    book = torch.randn(16, device=DEV)
    codes = torch.randint(0, 16, (10000,), dtype=torch.uint8, device=DEV)
    musa_aiter.kv_cachegen_decode(codes, book)
    codes[7777] = 16
    with pytest.raises(ValueError, match="exceeds codebook size"):
        musa_aiter.kv_cachegen_decode(codes, book)
    codes[7777] = 255
    with pytest.raises(ValueError, match="exceeds codebook size"):
        musa_aiter.kv_cachegen_decode(codes[7000:], book)  # tail path


# ---- reference-named C entries ------------------------------------------------------------------

def test_reference_c_entries_through_ctypes():
    lib = _hip.library()
    enc_fn = lib.musa_aiter_kv_cachegen_encode_float
    enc_fn.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_float, ctypes.c_float, ctypes.c_longlong,
                       ctypes.c_longlong, ctypes.c_void_p]
    enc_fn.restype = ctypes.c_int
    dec_fn = lib.musa_aiter_kv_cachegen_decode_float
    dec_fn.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_longlong, ctypes.c_void_p]
    dec_fn.restype = ctypes.c_int
    g = torch.Generator().manual_seed(9)
    for n, nb in ((1, 16), (4101, 256), (100000, 7)):
        x = torch.randn(n, generator=g)
        xd = x.to(DEV)
        mn, mx = float(x.min()), float(x.max())
        scale = float((nb - 1) / (mx - mn)) if mx != mn else 0.0  # the reference's host arithmetic
        out = torch.empty(n, dtype=torch.uint8, device=DEV)
        assert enc_fn(xd.data_ptr(), out.data_ptr(), mn, scale, n, nb, None) == 0
        torch.cuda.synchronize()
        want = cg.native_bins(x.numpy(), np.float32(mn), np.float32(scale), nb)
        np.testing.assert_array_equal(out.cpu().numpy(), want)
        book = torch.randn(nb, generator=g)
        dec = torch.empty(n, device=DEV)
        assert dec_fn(out.data_ptr(), book.to(DEV).data_ptr(), dec.data_ptr(), n, None) == 0
        torch.cuda.synchronize()
        np.testing.assert_array_equal(_bits(dec.cpu().numpy()), _bits(book.numpy()[want.astype(np.int64)]))


@pytest.mark.parametrize("numel", [1, 1000, 70_001, 5_000_000])  # one range workgroup, a few, the most
@pytest.mark.parametrize("ws_bytes", [16384, 16384 + 2047, 40000, 75776 - 1])
def test_encode_in_a_smaller_workspace(numel, ws_bytes):
    # The entry takes any workspace from 16,384 bytes on, with fewer copies of the bin counters: the same codes,
    # codebook and CDF, and nothing written past its end.
    x = torch.randn(numel, device=DEV, dtype=torch.float32).to(torch.bfloat16)
    want = musa_aiter.kv_cachegen_encode(x, num_bins=200)
    guard = 4096
    workspace = torch.full((ws_bytes + guard,), 0xA5, dtype=torch.uint8, device=DEV)
    got = [torch.empty_like(t) for t in want]
    rc = _hip.fn("musa_aiter_hip_cachegen_encode")(
        x.data_ptr(), 2, numel, 200, 0, *(t.data_ptr() for t in got), workspace.data_ptr(), ws_bytes,
        torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    for g, w in zip(got, want):
        assert torch.equal(g, w)
    assert bool((workspace[ws_bytes:] == 0xA5).all())


def test_encode_refuses_a_workspace_that_is_too_small():
    x = torch.zeros(100, device=DEV)
    out = torch.empty(1024, dtype=torch.uint8, device=DEV)
    rc = _hip.fn("musa_aiter_hip_cachegen_encode")(
        x.data_ptr(), 0, 100, 16, 0, out.data_ptr(), out.data_ptr(), out.data_ptr(), out.data_ptr(), 16383,
        torch.cuda.current_stream().cuda_stream)
    assert rc == 1  # hipErrorInvalidValue, before any launch
