// Paged-A caches with wide blocks <-> token-major linear rows: 16-bit copies
// of block sizes that are multiples of 64, 32-bit ones of multiples of 32.
//
// A cache row of such a block is made of whole 128-byte lines, so the
// transpose needs no LDS: a unit is one line of columns (64 16-bit or 32
// 32-bit elements), a chunk as many rows, and lane (rg, cg) of a wave holds
// the tile of 16 / ELT rows x 16 / ELT columns at row group rg and column
// group cg (rg, cg < 8).  Its loads (one 16-byte piece per row) cover eight
// whole cache lines per wave instruction, the tile is transposed in
// registers, and its stores (one 16-byte piece per token) cover eight whole
// lines of eight linear rows; a scatter runs the same steps backwards.  Every
// wave is on its own (no barrier) and keeps 8 KiB of loads in flight.
//
// Slots.  A wave sees its tile's tokens in lanes 0 .. TT - 1 of a 64-token
// window and the 64 tokens after (and for gathers before) them in a second
// (third) register; a run (tokens of one unit in slot order) spans at most one
// unit, so every run that starts in the tile ends inside the window.
//
// Bound by HBM.  9,001 tokens of 16 layers with 64-token pages (1.18 GB, 8 x
// 128 bf16): gather 207-211 us (5.6-5.7 TB/s), scatter 224 us, against
// 1,217 us for the element kernel that served these block sizes before (its
// 2-byte loads, a cache row apart, touch a line per lane).  A workgroup-
// cooperative form with an LDS tile (512 threads, two 8 KiB chunks, as in
// kv_paged_tiles.hip) measured 258 us and 283 us.  Single tokens cost as many
// lines here as there; those of many layers whose blocks several tokens share
// run up to 1.6 times longer than with the element kernel, which finishes plane
// by plane and finds the shared lines in the memory-side cache (256 tokens of 16
// layers of 4,096 rows, 192 blocks: 534 against 326 us).
#include "kv_hip_common.h"
#include "kv_launch.h"
#include "kv_paged_args.h"

namespace kvhip {

namespace {

template <int ELT>
struct Wide {
  static constexpr int UC = 128 / ELT;  // columns of a unit, rows of a chunk
  static constexpr int P = 16 / ELT;    // rows and columns of a lane's tile
  static constexpr int kUnitShift = ELT == 2 ? 6 : 5;
  static_assert((1 << kUnitShift) == UC, "unit of one line");
};

// Byte offset of unit u's first row: unit u covers slots [UC * u, UC * (u + 1)).
template <int ELT>
__device__ __forceinline__ int64_t unit_offset(const TileArgs& a, int64_t unit) {
  const int64_t units = a.block_size / Wide<ELT>::UC;
  const int64_t blk = unit / units;
  return (blk * a.nrows * a.block_size + (unit - blk * units) * Wide<ELT>::UC) * ELT;
}

// Piece j of the transposed tile: element q of it is element j of d[q].
template <int ELT>
__device__ __forceinline__ u32x4 transposed(const u32x4 (&d)[Wide<ELT>::P], int j) {
  u32x4 o;
  if constexpr (ELT == 2) {
#pragma unroll
    for (int k = 0; k < 4; ++k) o[k] = pack16(elem16(d[2 * k], j), elem16(d[2 * k + 1], j));
  } else {
#pragma unroll
    for (int k = 0; k < 4; ++k) o[k] = d[k][j];
  }
  return o;
}

// This wave's chunk of one plane and its lane's place in it.
struct WaveChunk {
  uint8_t* cache;  // the plane's caches and linear rows at the chunk's first row
  uint8_t* lin;
  int rows;        // rows of the chunk (0: past the last row)
  uint32_t pitch;  // bytes between cache rows
  uint32_t stride; // bytes between tokens
  int rg, cg;
};

template <int ELT>
__device__ __forceinline__ WaveChunk wave_chunk(const TileArgs& a, uint32_t plane, int64_t chunk) {
  WaveChunk w;
  const int layer = static_cast<int>(plane >> 1);
  const int kv = static_cast<int>(plane & 1);
  const int64_t rb = chunk * Wide<ELT>::UC;
  const int64_t left = a.nrows - rb;
  w.rows = left <= 0 ? 0 : (left < Wide<ELT>::UC ? static_cast<int>(left) : Wide<ELT>::UC);
  w.pitch = static_cast<uint32_t>(a.block_size) * ELT;
  w.stride = static_cast<uint32_t>(a.lin_token_stride);
  w.cache = a.cache[kv] + static_cast<int64_t>(layer) * a.cache_layer_stride + rb * w.pitch;
  w.lin = a.lin[kv] + static_cast<int64_t>(layer) * a.lin_layer_stride + rb * ELT;
  w.rg = lane_id() >> 3;
  w.cg = lane_id() & 7;
  return w;
}

// The P bits of `cols` (a bit per unit column) that belong to column group cg.
template <int ELT>
__device__ __forceinline__ uint32_t group_bits(uint64_t cols, int cg) {
  constexpr int P = Wide<ELT>::P;
  return static_cast<uint32_t>(cols >> (cg * P)) & ((1u << P) - 1u);
}

// Unit columns `cols` -> linear rows; column c's token row sits at byte offset
// c * stride of `lin_col0` (the row column 0's token would have).
template <int ELT, int STP>
__device__ __forceinline__ void gather_unit(const WaveChunk& w, const uint8_t* unit, uint8_t* lin_col0,
                                            uint64_t cols) {
  constexpr int P = Wide<ELT>::P;
  const uint32_t bits = group_bits<ELT>(cols, w.cg);
  const bool row_in = w.rg * P < w.rows;
  const buf_t cbuf = make_buf(unit);
  const uint32_t coff = static_cast<uint32_t>(w.rg * P) * w.pitch + static_cast<uint32_t>(w.cg) * 16u;
  u32x4 d[P];
#pragma unroll
  for (int q = 0; q < P; ++q)
    d[q] = buf_ld16(cbuf, row_in && bits != 0 ? coff : kOffOob, static_cast<uint32_t>(q) * w.pitch);
  const buf_t lbuf = make_buf(lin_col0);
  const uint32_t loff = static_cast<uint32_t>(w.cg * P) * w.stride + static_cast<uint32_t>(w.rg) * 16u;
#pragma unroll
  for (int j = 0; j < P; ++j)
    buf_st16_p<STP>(lbuf, (row_in && ((bits >> j) & 1u) ? loff : kOffOob) + static_cast<uint32_t>(j) * w.stride,
                    transposed<ELT>(d, j));
}

// Stores a lane's transposed tile (piece q: row rg * P + q of the unit) into
// the columns of `cols`: whole pieces as vectors, others element by element.
template <int ELT, int STP>
__device__ __forceinline__ void store_unit(const WaveChunk& w, uint8_t* unit, uint64_t cols,
                                           const u32x4 (&d)[Wide<ELT>::P]) {
  constexpr int P = Wide<ELT>::P;
  constexpr uint32_t kAll = (1u << P) - 1u;
  const uint32_t bits = group_bits<ELT>(cols, w.cg);
  const bool row_in = w.rg * P < w.rows;
  const buf_t cbuf = make_buf(unit);
  const uint32_t coff = static_cast<uint32_t>(w.rg * P) * w.pitch + static_cast<uint32_t>(w.cg) * 16u;
  const uint32_t whole = row_in && bits == kAll ? coff : kOffOob;
#pragma unroll
  for (int q = 0; q < P; ++q)
    buf_st16_p<STP>(cbuf, whole + static_cast<uint32_t>(q) * w.pitch, transposed<ELT>(d, q));
  if (ballot(row_in && bits != 0 && bits != kAll) == 0) return;
#pragma unroll
  for (int j = 0; j < P; ++j) {
    const uint32_t off = row_in && bits != kAll && ((bits >> j) & 1u) ? coff + j * ELT : kOffOob;
#pragma unroll
    for (int q = 0; q < P; ++q) {
      const uint32_t v = piece_elem<ELT>(d[j], q);
      if constexpr (ELT == 2)
        __builtin_amdgcn_raw_buffer_store_b16(static_cast<uint16_t>(v), cbuf, off, static_cast<uint32_t>(q) * w.pitch,
                                              0);
      else
        __builtin_amdgcn_raw_buffer_store_b32(v, cbuf, off, static_cast<uint32_t>(q) * w.pitch, 0);
    }
  }
}

// Tokens moved one by one (a decode step's runs of one or a few tokens): one
// row per lane, a token's chunk of rows per instruction.  Lane i of `s` holds
// the slot of token t0 + i, bit i of `move` (i < TT) says that it moves.
template <int ELT, bool SCATTER, int TT>
__device__ __forceinline__ void wide_token_rows(const TileArgs& a, const WaveChunk& w, int64_t s, uint64_t move,
                                                int64_t t0) {
  constexpr int UC = Wide<ELT>::UC;
  const int lane = lane_id();
  const int64_t cbase = unit_offset<ELT>(a, s >> Wide<ELT>::kUnitShift) + (s & (UC - 1)) * ELT;
  const bool row_in = lane < w.rows;
  const uint32_t coff = row_in ? static_cast<uint32_t>(lane) * w.pitch : kOffOob;
  const uint32_t loff = row_in ? static_cast<uint32_t>(lane) * ELT : kOffOob;
  constexpr int kSrcPol = SCATTER ? kBufNT : 0, kDstPol = SCATTER ? 0 : kBufNT;
  auto desc = [&](int i, bool cache_side) {
    uint8_t* const base = cache_side ? w.cache + readlane64(cbase, i) : w.lin + (t0 + i) * a.lin_token_stride;
    return __builtin_amdgcn_make_buffer_rsrc(base, 0, ((move >> i) & 1ull) ? 0x7FFFFFFF : 0, 0x00020000);
  };
  constexpr int TB = TT < 16 ? TT : 16;  // tokens in flight
  static_assert(TT % TB == 0, "whole batches");
#pragma unroll 1
  for (int i0 = 0; i0 < TT; i0 += TB) {
    if (((move >> i0) & ((1ull << TB) - 1ull)) == 0) continue;
    uint32_t v[TB];
#pragma unroll
    for (int k = 0; k < TB; ++k) {
      const buf_t src = desc(i0 + k, !SCATTER);
      if constexpr (ELT == 2) v[k] = __builtin_amdgcn_raw_buffer_load_b16(src, SCATTER ? loff : coff, 0, kSrcPol);
      else v[k] = __builtin_amdgcn_raw_buffer_load_b32(src, SCATTER ? loff : coff, 0, kSrcPol);
    }
#pragma unroll
    for (int k = 0; k < TB; ++k) {
      const buf_t dst = desc(i0 + k, SCATTER);
      if constexpr (ELT == 2)
        __builtin_amdgcn_raw_buffer_store_b16(static_cast<uint16_t>(v[k]), dst, SCATTER ? coff : loff, 0, kDstPol);
      else
        __builtin_amdgcn_raw_buffer_store_b32(v[k], dst, SCATTER ? coff : loff, 0, kDstPol);
    }
  }
}

// Tiles whose runs average fewer than this many tokens move token by token.
constexpr int kWideShortRun = 6;
// (Gather tiles do below TileArgs::short_run, see wide_gather_short_run.)

__device__ __forceinline__ int64_t slot_or_none(const TileArgs& a, int64_t t) {
  return t >= 0 && t < a.num_tokens ? slot_at(a, t) : -1;
}

__device__ __forceinline__ uint64_t low_bits(int64_t n) { return n >= 64 ? ~0ull : (1ull << n) - 1ull; }

// True when the runs of a tile average fewer than short_run tokens: `v` marks
// its valid tokens, `c` those that continue the token before them.
__device__ __forceinline__ bool short_gather_tile(const TileArgs& a, uint64_t v, uint64_t c) {
  return __builtin_popcountll(v) < a.short_run * __builtin_popcountll(v & ~c);
}

// Gather.  Grid: x = tile * row_groups + group of WPB chunks (4, or 1 in small
// launches: wide_gather_few), y = plane.  A run
// is every token of the window whose slot lies in the head's unit at the
// head's distance from its token, so tokens skipped in between (slot < 0) do
// not cut it; its first token's tile moves it.  A tile of short runs instead
// moves its own tokens, no more, and the tile after it knows that from the
// same slots.
template <int ELT, bool XCD, int STP, int WPB = kWavesPerBlock>
__global__ __launch_bounds__(WPB * kWave) void paged_wide_gather_kernel(const TileArgs a) {
  using W = Wide<ELT>;
  constexpr int TT = W::UC;
  const int lane = lane_id();
  WgXyz wg = xcd_contiguous_wg<XCD>();
  const uint32_t ahead = static_cast<uint32_t>(a.check_groups);
  if (wg.x < ahead) {
    check_share<WPB * kWave>(a, wg.x, wg.y);
    return;
  }
  wg.x -= ahead;
  const uint32_t tile = wg.x / static_cast<uint32_t>(a.row_groups);
  const uint32_t group = wg.x - tile * static_cast<uint32_t>(a.row_groups);
  const int64_t t0 = static_cast<int64_t>(tile) * TT;
  const WaveChunk w = wave_chunk<ELT>(a, wg.y, static_cast<int64_t>(group) * WPB + wave_in_block());
  if (w.rows == 0) return;

  const int64_t s = slot_or_none(a, t0 + lane);
  const int64_t s_hi = slot_or_none(a, t0 + kWave + lane);
  const int64_t s_pre = slot_or_none(a, t0 - kWave + lane);
  if (refused_ahead(a.check)) return;
  const bool valid = s >= 0 && s < a.num_slots;
  const bool valid_pre = s_pre >= 0 && s_pre < a.num_slots;
  const uint64_t in_tile = low_bits(a.num_tokens - t0) & low_bits(TT);
  const uint64_t v_lo = ballot(valid);
  uint64_t pending = v_lo & in_tile;
  // Short runs, judged on a tile's own tokens alone; the tile before is the
  // last TT lanes of s_pre.
  const int64_t s_prev = from_prev_lane(s), s_pre_prev = from_prev_lane(s_pre);
  auto continues = [&](int64_t slot, int64_t before) { return slot == before + 1 && (slot & (W::UC - 1)) != 0; };
  const uint64_t c = ballot(valid && lane > 0 && continues(s, s_prev));
  const uint64_t c_pre = ballot(valid_pre && lane > kWave - TT && continues(s_pre, s_pre_prev));
  const bool pre_short = short_gather_tile(a, ballot(valid_pre) >> (kWave - TT), c_pre >> (kWave - TT));
  if (short_gather_tile(a, pending, c)) {
    wide_token_rows<ELT, false, TT>(a, w, s, pending, t0);
    pending = 0;
  }
  while (pending) {
    const int i = __builtin_ctzll(pending);
    const int64_t head = readlane64(s, i);
    const int64_t unit = head >> W::kUnitShift;
    const int64_t first = head - i;  // slot of lane 0, had the run begun there
    auto member = [&](int64_t slot, int at) { return (slot >> W::kUnitShift) == unit && slot - at == first; };
    const uint64_t lo = ballot(valid && member(s, lane));
    const uint64_t hi = ballot(member(s_hi, lane + kWave));
    const bool earlier = !pre_short && ballot(member(s_pre, lane - kWave)) != 0;  // the tile before moves the run
    pending &= ~lo;
    if (earlier) continue;
    const int c0 = static_cast<int>(head & (W::UC - 1));
    const uint64_t cols = ((lo >> i) | (i > 0 ? hi << (64 - i) : 0ull)) << c0;
    gather_unit<ELT, STP>(w, w.cache + unit_offset<ELT>(a, unit), w.lin + (t0 + i - c0) * a.lin_token_stride, cols);
  }

  if (a.fill_zeros) {
    const uint64_t skipped = ~v_lo & in_tile;
    if (skipped == 0) return;
    const buf_t lbuf = make_buf(w.lin + t0 * a.lin_token_stride);
    const u32x4 zero = {0u, 0u, 0u, 0u};
    // Eight tokens' lines per instruction: lane (token rg, piece cg).
#pragma unroll 1
    for (int i = w.rg; i < TT; i += 8) {
      const bool mine = ((skipped >> i) & 1ull) && w.cg * W::P < w.rows;
      buf_st16(lbuf, mine ? static_cast<uint32_t>(i) * w.stride + static_cast<uint32_t>(w.cg) * 16u : kOffOob, zero);
    }
  }
}

// A run of consecutive tokens loaded for a scatter: unit columns [c0, c0 + n).
template <int ELT>
__device__ __forceinline__ void load_run(const WaveChunk& w, const uint8_t* lin_col0, uint64_t cols,
                                         u32x4 (&d)[Wide<ELT>::P]) {
  constexpr int P = Wide<ELT>::P;
  const uint32_t bits = group_bits<ELT>(cols, w.cg);
  const bool row_in = w.rg * P < w.rows;
  const buf_t lbuf = make_buf(lin_col0);
  const uint32_t loff = static_cast<uint32_t>(w.cg * P) * w.stride + static_cast<uint32_t>(w.rg) * 16u;
#pragma unroll
  for (int j = 0; j < P; ++j)
    d[j] = buf_ld16(lbuf, row_in && ((bits >> j) & 1u) ? loff : kOffOob, static_cast<uint32_t>(j) * w.stride);
}

// Scatter in token order: the runs (consecutive tokens that write consecutive
// slots of one unit) that start in the tile.  Grid as the gather's.
template <int ELT, int TT>
__global__ __launch_bounds__(kBlockThreads) void paged_wide_scatter_kernel(const TileArgs a) {
  using W = Wide<ELT>;
  const int lane = lane_id();
  const uint32_t tile = blockIdx.x / static_cast<uint32_t>(a.row_groups);
  const uint32_t group = blockIdx.x - tile * static_cast<uint32_t>(a.row_groups);
  const int64_t t0 = static_cast<int64_t>(tile) * TT;
  const WaveChunk w = wave_chunk<ELT>(a, blockIdx.y, static_cast<int64_t>(group) * kWavesPerBlock + wave_in_block());
  const int64_t s = slot_or_none(a, t0 + lane);
  const int64_t s_hi = slot_or_none(a, t0 + kWave + lane);
  const int64_t s_before = slot_or_none(a, t0 - 1);
  if (a.scan_dupes && !scan_build<kBlockThreads>(scan_table(), a)) return;  // every wave, before any of them leaves
  if (refused_ahead(a.check)) return;
  if (w.rows == 0) return;
  auto writes = [&](int64_t slot, int64_t t) -> bool {
    bool valid = slot >= 0 && slot < a.num_slots;
    if (a.scan_dupes) {
      if (valid) valid = scan_is_last(scan_table(), slot, t);
    } else if (valid && a.owner != nullptr) {
      valid = a.owner[slot] == claim_tag(a.epoch, t);
    }
    return valid;
  };
  const bool valid = writes(s, t0 + lane);
  const bool valid_hi = writes(s_hi, t0 + kWave + lane);
  const uint64_t v_lo = ballot(valid), v_hi = ballot(valid_hi);
  // The token before lane 0 of each register: t0 - 1, and lane 63 of the first.
  const uint64_t pv_lo = (v_lo << 1) | (writes(s_before, t0 - 1) ? 1ull : 0ull);
  const uint64_t pv_hi = (v_hi << 1) | (v_lo >> 63);
  // The lane shuffles run in every lane: a lane switched off by a condition
  // would hand its neighbour nothing.
  const int64_t s_prev = from_prev_lane(s), s_hi_prev = from_prev_lane(s_hi);
  const int64_t last = readlane64(s, 63);
  const int64_t prev = lane == 0 ? s_before : s_prev;
  const int64_t prev_hi = lane == 0 ? last : s_hi_prev;
  auto continues = [&](int64_t slot, int64_t before) { return slot == before + 1 && (slot & (W::UC - 1)) != 0; };
  const uint64_t c_lo = ballot(valid && ((pv_lo >> lane) & 1ull) && continues(s, prev));
  const uint64_t c_hi = ballot(valid_hi && ((pv_hi >> lane) & 1ull) && continues(s_hi, prev_hi));
  const uint64_t in_tile = low_bits(a.num_tokens - t0) & low_bits(TT);
  uint64_t heads = v_lo & ~c_lo & in_tile;
  if (heads == 0) return;

  // Short runs move token by token, except a last one that goes on past the
  // tile.  Their lanes: what writes from the first head on (what lies before
  // it continues an earlier tile's run) up to that last run.
  uint64_t short_heads = heads, lanes = v_lo & in_tile & ~low_bits(__builtin_ctzll(heads));
  const bool goes_on = TT == 64 ? (c_hi & 1ull) : ((c_lo >> (TT & 63)) & 1ull);
  if (goes_on) {
    const uint64_t below_last = low_bits(63 - __builtin_clzll(heads));
    short_heads &= below_last;
    lanes &= below_last;
  }
  const int runs = __builtin_popcountll(short_heads);
  if (runs > 0 && __builtin_popcountll(lanes) < runs * kWideShortRun) {
    wide_token_rows<ELT, true, TT>(a, w, s, lanes, t0);
    heads &= ~short_heads;
  }
  while (heads) {
    const int i = __builtin_ctzll(heads);
    heads &= heads - 1;
    const int64_t head = readlane64(s, i);
    const int c0 = static_cast<int>(head & (W::UC - 1));
    const uint64_t cols = low_bits(run_length(c_lo, c_hi, i)) << c0;
    u32x4 d[W::P];
    load_run<ELT>(w, w.lin + (t0 + i - c0) * a.lin_token_stride, cols, d);
    store_unit<ELT, kBufNT>(w, w.cache + unit_offset<ELT>(a, head >> W::kUnitShift), cols, d);
  }
}

// Scatter in destination order (see paged_block_scatter_kernel in
// kv_paged_tiles.hip): x = unit * row_groups + group; the unit's claim tags
// name the token of each column, whatever their order, so a unit is loaded and
// written once.  The launcher keeps a plane's linear rows below 2 GiB.
template <int ELT, bool XCD, int STP>
__global__ __launch_bounds__(kBlockThreads) void paged_wide_unit_scatter_kernel(const TileArgs a) {
  using W = Wide<ELT>;
  const int lane = lane_id();
  const WgXyz wg = xcd_contiguous_wg<XCD>();
  const uint32_t unit = wg.x / static_cast<uint32_t>(a.row_groups);
  const uint32_t group = wg.x - unit * static_cast<uint32_t>(a.row_groups);
  const WaveChunk w = wave_chunk<ELT>(a, wg.y, static_cast<int64_t>(group) * kWavesPerBlock + wave_in_block());
  if (w.rows == 0) return;
  uint64_t tag = 0;
  if (lane < W::UC) tag = a.owner[static_cast<int64_t>(unit) * W::UC + lane];
  if (refused_ahead(a.check)) return;
  const bool valid = static_cast<uint32_t>(tag >> 32) == a.epoch && static_cast<uint32_t>(tag) != 0u;
  const uint64_t cols = ballot(valid);
  if (cols == 0) return;
  const uint32_t off = valid ? (static_cast<uint32_t>(tag) - 1u) * w.stride : kOffOob;
  const bool row_in = w.rg * W::P < w.rows;
  const buf_t lbuf = make_buf(w.lin);
  u32x4 d[W::P];
#pragma unroll
  for (int j = 0; j < W::P; ++j) {
    const uint32_t row = static_cast<uint32_t>(__shfl(static_cast<int>(off), w.cg * W::P + j));
    d[j] = buf_ld16(lbuf, row_in && row != kOffOob ? row + static_cast<uint32_t>(w.rg) * 16u : kOffOob);
  }
  store_unit<ELT, STP>(w, w.cache + unit_offset<ELT>(a, unit), cols, d);
}

// Planes from which each XCD takes a contiguous eighth of the grid.
constexpr int64_t kWideXcdPlanes = 32;

}  // namespace

template <int ELT, bool SCATTER>
hipError_t launch_wide(const TileArgs& a0, int64_t planes, bool lines, hipStream_t stream) {
  using W = Wide<ELT>;
  if (a0.check.report != nullptr && (SCATTER ? a0.scan_dupes == 0 : a0.check.words == 0)) return hipErrorNotSupported;
  TileArgs a = a0;
  const int64_t chunks = (a.nrows + W::UC - 1) / W::UC;
  const int64_t elems = a.num_tokens * a.nrows * planes;
  const int64_t unit_tiles = (a.num_tokens + W::UC - 1) / W::UC;
  const int64_t unit_groups = unit_tiles * ((chunks + kWavesPerBlock - 1) / kWavesPerBlock) * planes;
  const bool few = SCATTER ? wide_scatter_few(a.num_tokens, unit_groups) : wide_gather_few(ELT, elems);
  a.short_run = wide_gather_short_run(ELT, elems);
  const int wpb = few && !SCATTER ? 1 : kWavesPerBlock;
  const int64_t groups = (chunks + wpb - 1) / wpb;
  const int tt = SCATTER && few ? kWideFewScatterTile : W::UC;
  // Destination order under the narrow scatter's rule: the claim tags are this
  // call's inverse map and the tokens cover a quarter of the slots.
  const bool by_unit = SCATTER && a.owner != nullptr && a.owner_exclusive && a.num_tokens * 4 >= a.num_slots &&
                       (a.num_tokens + 1) * a.lin_token_stride < (int64_t{1} << 31);
  const int64_t tiles = by_unit ? a.num_slots / W::UC : (a.num_tokens + tt - 1) / tt;
  if (groups > 0x7FFFFFFF || tiles > 0x7FFFFFFF / groups) return hipErrorInvalidValue;
  a.row_groups = static_cast<int32_t>(groups);
  const int64_t extra = SCATTER ? 0 : (a.check.words + wpb - 1) / wpb;
  a.check_groups = static_cast<int32_t>(extra);
  if (tiles * groups > 0x7FFFFFFF - extra) return hipErrorInvalidValue;
  const dim3 grid(static_cast<uint32_t>(tiles * groups + extra), static_cast<uint32_t>(planes));
  const dim3 block(static_cast<uint32_t>(wpb * kWave));
  const bool xcd = planes >= kWideXcdPlanes && int64_t{grid.x} * planes <= int64_t{0xFFFFFFFF};
  if constexpr (SCATTER) {
    if (by_unit && xcd)
      hipLaunchKernelGGL((paged_wide_unit_scatter_kernel<ELT, true, kBufWT>), grid, block, 0, stream, a);
    else if (by_unit)
      hipLaunchKernelGGL((paged_wide_unit_scatter_kernel<ELT, false, kBufWT>), grid, block, 0, stream, a);
    else if (few)
      hipLaunchKernelGGL((paged_wide_scatter_kernel<ELT, kWideFewScatterTile>), grid, block, 0, stream, a);
    else
      hipLaunchKernelGGL((paged_wide_scatter_kernel<ELT, W::UC>), grid, block, 0, stream, a);
  } else if (few) {
    if (lines) hipLaunchKernelGGL((paged_wide_gather_kernel<ELT, false, kBufWT, 1>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((paged_wide_gather_kernel<ELT, false, kBufNT, 1>), grid, block, 0, stream, a);
  } else {
    if (xcd && lines)
      hipLaunchKernelGGL((paged_wide_gather_kernel<ELT, true, kBufWT>), grid, block, 0, stream, a);
    else if (xcd)
      hipLaunchKernelGGL((paged_wide_gather_kernel<ELT, true, kBufNT>), grid, block, 0, stream, a);
    else if (lines)
      hipLaunchKernelGGL((paged_wide_gather_kernel<ELT, false, kBufWT>), grid, block, 0, stream, a);
    else
      hipLaunchKernelGGL((paged_wide_gather_kernel<ELT, false, kBufNT>), grid, block, 0, stream, a);
  }
  return hipGetLastError();
}

template hipError_t launch_wide<2, false>(const TileArgs&, int64_t, bool, hipStream_t);
template hipError_t launch_wide<2, true>(const TileArgs&, int64_t, bool, hipStream_t);
template hipError_t launch_wide<4, false>(const TileArgs&, int64_t, bool, hipStream_t);
template hipError_t launch_wide<4, true>(const TileArgs&, int64_t, bool, hipStream_t);

}  // namespace kvhip
