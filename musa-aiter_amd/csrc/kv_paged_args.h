// Kernel arguments and element helpers shared by the paged-A tile kernels
// (kv_paged_tiles.hip: workgroup-cooperative kernel, generic element kernel;
// kv_paged_waves.hip: per-wave gather kernel).
#pragma once

#include "kv_hip_common.h"
#include "kv_launch.h"

namespace kvhip {

struct TileArgs {
  CallCheck check;             // report set: this kernel checks the call's slots and scales; guard set: one ahead did
  uint8_t* cache[2];
  uint8_t* lin[2];
  const int64_t* slots;
  const float* scale[2];
  const uint64_t* owner;
  int64_t num_tokens;
  int64_t num_slots;
  int64_t nrows;               // NH * HD
  int64_t head_dim;
  int64_t num_heads;
  int64_t cache_layer_stride;  // bytes
  int64_t lin_layer_stride;    // bytes
  int64_t lin_token_stride;    // bytes
  int32_t scale_mode;
  int32_t fill_zeros;
  uint32_t epoch;
  int32_t owner_exclusive;     // every tag of `epoch` in owner was claimed by this call
  int32_t block_size;          // used by the wide and generic kernels
  float inv_head_dim;          // 1 / head_dim, for small-integer division by head_dim
  BlockTableSlots bt;          // block_tables set: slots derived per dense token
  int32_t row_groups;          // tile kernel: row groups per block (grid x of a gather = tile * row_groups + group)
  int32_t check_groups;        // gather: workgroups at the front of each plane for check_share (0: none)
  int32_t scan_dupes;          // scatter: resolve repeated slots with a ScanTable instead of claim tags
  int32_t short_run;           // wide gather: tiles whose runs average fewer tokens move token by token
};

// Slot of token t: the slot vector's entry, or the block-table slot of the
// dense token t.
__device__ __forceinline__ int64_t slot_at(const TileArgs& a, int64_t t) {
  if (a.bt.block_tables != nullptr) return block_table_slot(a.bt, t);
  return a.slots[t];
}

constexpr int kTileTokens = 16;

// Cache columns of a per-wave kernel's BS-column unit: a block of 16 or 32
// columns, or with BS = 64 the 64 columns of a block whose size is any
// multiple of 64 (consecutive rows then lie block_size elements apart).  Slot
// s lies in unit s / BS either way.
template <int ELT, int BS>
__device__ __forceinline__ uint32_t unit_pitch(const TileArgs& a) {
  if constexpr (BS < 64) return BS * ELT;
  else return static_cast<uint32_t>(a.block_size) * ELT;
}

// Byte offset of row `row` of unit `unit` inside its plane.
template <int ELT, int BS>
__device__ __forceinline__ int64_t unit_row_offset(const TileArgs& a, int64_t unit, int64_t row) {
  if constexpr (BS < 64) {
    return (unit * a.nrows + row) * (BS * ELT);
  } else {
    const int64_t units = a.block_size / BS;
    const int64_t blk = unit / units;
    return ((blk * a.nrows + row) * a.block_size + (unit - blk * units) * BS) * ELT;
  }
}

// Length of the run starting at lane i, given the continuation bits of its
// 64-token window and of the 64 tokens after it (`hi`, 0 where a run cannot
// reach them).
__device__ __forceinline__ int run_length(uint64_t lo, uint64_t hi, int i) {
  const int n = i < 63 ? __builtin_ctzll(~(lo >> (i + 1))) : 0;  // the shift fills with zeros
  return i + 1 + n < 64 ? 1 + n : 1 + n + __builtin_ctzll(~hi);  // a unit ends before `hi` runs out
}

// Small scatters resolve repeated destinations without the claim pass (one
// launch and one dependent load fewer): every workgroup maps each slot of the
// call to the last token that writes it, in LDS -- open addressing over
// 2 x kScanTokens entries, a 64-bit compare-and-swap claiming an entry for the
// slot and an atomic max keeping the token -- and a token writes only if it is
// its slot's last token, the claim pass's rule (last writer wins).  The host
// keeps such calls at or below kScanTokens tokens, so at most half the
// entries are taken and every probe sequence ends.
constexpr int kScanEntries = 2 * kScanTokens;
constexpr unsigned long long kScanEmpty = ~0ull;

struct ScanTable {
  unsigned long long key[kScanEntries];
  int last[kScanEntries];
  int refused;  // some slot or scale of a checked call is not acceptable
};

// Entries of each scale array of the call.
__device__ __forceinline__ int64_t scale_count(const TileArgs& a) {
  if (a.scale[0] == nullptr) return 0;
  const int64_t layers = static_cast<int64_t>(gridDim.y) / 2;  // every paged kernel runs (.., plane, ..) grids
  return a.scale_mode == 0 ? 1 : a.scale_mode == 1 ? a.num_heads : layers * a.num_heads;
}

// This thread's share of the scales of a call checked by its own kernel.
template <int NT>
__device__ __forceinline__ bool scales_refused(const TileArgs& a) {
  bool bad = false;
  const int64_t n = scale_count(a);
  for (int64_t j = threadIdx.x; j < 2 * n; j += NT) bad |= scale_refused(a.scale[j >= n][j >= n ? j - n : j]);
  return bad;
}

// Workgroup 0's verdict on a checked call, for the polling host.
__device__ __forceinline__ void report_check(const CallCheck& c, bool refused) {
  if ((blockIdx.x | blockIdx.y | blockIdx.z | threadIdx.x) == 0)
    __hip_atomic_store(c.report, 2 * c.stamp + (refused ? 1 : 0), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// A gather whose output is thrown away when the call is refused runs unguarded
// (it skips the slots it cannot read anyway), so extra workgroups of its own
// launch, ahead of plane 0's tiles, check the slots, kCheckSlice at a time, and
// the call needs no check kernel ahead of it: one layer of 7,456 tokens (fp16,
// 16-token pages) 17.2 -> 14.0 us a call, 16 layers of 9,001 tokens (64-token
// pages) 213.8 -> 208.5.  (Behind plane 0's tiles they report so late that the
// host's next call waits: 15.5 us; the first waves checking on their way to
// their own tiles: 13.9 and 211.3 us.)  The word is all that a wave publishes,
// so its store is relaxed: a release at system scope would write back the L2,
// which holds the rows that other workgroups are storing.
// FP8 gathers keep the check kernel: theirs took as much longer as it had taken
// (6,007 tokens of 8 layers: 47.5 + 4.8 -> 51.6 us, the call 55 us both ways).
// `group`: index among the extra workgroups of the plane.
template <int NT>
__device__ __forceinline__ void check_share(const TileArgs& a, uint32_t group, uint32_t plane) {
  const int64_t word = static_cast<int64_t>(group) * (NT / kWave) + wave_in_block();
  if (word >= a.check.words || plane != 0) return;
  bool bad = false;
  for (int64_t base = word * kCheckSlice; base < a.num_tokens; base += a.check.words * kCheckSlice) {
    int64_t s[kCheckSlice / kWave];
#pragma unroll
    for (int k = 0; k < kCheckSlice / kWave; ++k) {
      const int64_t j = base + k * kWave + lane_id();
      s[k] = j < a.num_tokens ? a.slots[j] : -1;
    }
#pragma unroll
    for (int k = 0; k < kCheckSlice / kWave; ++k) bad |= s[k] >= a.num_slots;
  }
  const bool refused = ballot(bad) != 0;
  if (lane_id() == 0)
    __hip_atomic_store(a.check.report + word, 2 * a.check.stamp + (refused ? 1 : 0), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_SYSTEM);
}

// Checks a small call in the kernel that moves it (report set): every
// workgroup reads all slots and scales, so all of them decide alike.  Every
// thread of the workgroup calls it (it holds two barriers).  True: move nothing.
template <int NT>
__device__ bool check_in_kernel(const TileArgs& a) {
  __shared__ int refused;
  if (threadIdx.x == 0) refused = 0;
  __syncthreads();
  bool bad = scales_refused<NT>(a);
  for (int64_t j = threadIdx.x; j < a.num_tokens; j += NT) bad |= a.slots[j] >= a.num_slots;
  if (bad) refused = 1;
  __syncthreads();
  const bool r = refused != 0;
  report_check(a.check, r);
  return r;
}

// The workgroup's table (static LDS of the kernels that call it).
__device__ __forceinline__ ScanTable& scan_table() {
  __shared__ ScanTable tb;
  return tb;
}

__device__ __forceinline__ uint32_t scan_hash(int64_t s) {
  return static_cast<uint32_t>((static_cast<uint64_t>(s) * 0x9E3779B97F4A7C15ull) >> 40) & (kScanEntries - 1);
}

// Fills the table from the call's slots; every thread of the workgroup calls
// it (it holds two workgroup barriers).  A call checked by its own kernel is
// checked on the way; false: it is refused, move nothing.
template <int NT>
__device__ bool scan_build(ScanTable& tb, const TileArgs& a) {
  const int tid = static_cast<int>(threadIdx.x);
  const bool checked = a.check.report != nullptr;
  if (tid == 0) tb.refused = 0;
  for (int e = tid; e < kScanEntries; e += NT) {
    tb.key[e] = kScanEmpty;
    tb.last[e] = -1;
  }
  __syncthreads();
  bool bad = checked && scales_refused<NT>(a);
  for (int64_t j = tid; j < a.num_tokens; j += NT) {
    const int64_t s = slot_at(a, j);
    bad |= s >= a.num_slots;
    if (s < 0 || s >= a.num_slots) continue;
    uint32_t h = scan_hash(s);
    for (int probe = 0; probe < kScanEntries; ++probe) {
      const unsigned long long prev = atomicCAS(&tb.key[h], kScanEmpty, static_cast<unsigned long long>(s));
      if (prev == kScanEmpty || prev == static_cast<unsigned long long>(s)) {
        atomicMax(&tb.last[h], static_cast<int>(j));
        break;
      }
      h = (h + 1) & (kScanEntries - 1);
    }
  }
  if (checked && bad) tb.refused = 1;
  __syncthreads();
  if (!checked) return true;
  const bool refused = tb.refused != 0;
  report_check(a.check, refused);
  return !refused;
}

// True when token t is the last token of the call writing slot s (s valid).
__device__ __forceinline__ bool scan_is_last(const ScanTable& tb, int64_t s, int64_t t) {
  uint32_t h = scan_hash(s);
  for (int probe = 0; probe < kScanEntries; ++probe) {
    const unsigned long long k = tb.key[h];
    if (k == static_cast<unsigned long long>(s)) return tb.last[h] == static_cast<int>(t);
    if (k == kScanEmpty) return false;
    h = (h + 1) & (kScanEntries - 1);
  }
  return false;
}

// head = row / head_dim for rows below 2^24: a float reciprocal and one
// exact correction step.
__device__ __forceinline__ int head_of_row(const TileArgs& a, int row) {
  const int hd = static_cast<int>(a.head_dim);
  int head = static_cast<int>(static_cast<float>(row) * a.inv_head_dim);
  if (head * hd > row) --head;
  else if ((head + 1) * hd <= row) ++head;
  return head;
}

__device__ __forceinline__ float load_scale(const TileArgs& a, int kv, int layer, int64_t head) {
  const float* s = a.scale[kv];
  if (a.scale_mode == 0) return s[0];
  if (a.scale_mode == 1) return s[head];
  return s[static_cast<int64_t>(layer) * a.num_heads + head];
}

template <int ELT>
__device__ __forceinline__ void store_elem(uint8_t* p, uint32_t v) {
  if constexpr (ELT == 1) *p = static_cast<uint8_t>(v);
  else if constexpr (ELT == 2) *reinterpret_cast<uint16_t*>(p) = static_cast<uint16_t>(v);
  else *reinterpret_cast<uint32_t*>(p) = v;
}

template <int ELT>
__device__ __forceinline__ uint32_t load_elem(const uint8_t* p) {
  if constexpr (ELT == 1) return *p;
  else if constexpr (ELT == 2) return *reinterpret_cast<const uint16_t*>(p);
  else return *reinterpret_cast<const uint32_t*>(p);
}

// Element `idx` of a 16-byte piece holding ELT-byte elements.
template <int ELT>
__device__ __forceinline__ uint32_t piece_elem(const u32x4& v, int idx) {
  if constexpr (ELT == 1) return elem8(v, idx);
  else if constexpr (ELT == 2) return elem16(v, idx);
  else return v[idx];
}

// Per-wave LDS-staged gather (kv_paged_waves.hip), used for the FP8
// dequant-gather: its in-register 8x16 byte transposes need an eighth of the
// LDS instructions of the cooperative kernel's column reads.
template <int ELT_C, int ELT_L, int CODEC, int LDT, int BS>
hipError_t launch_wave_gather(const TileArgs& a, int64_t planes, hipStream_t stream);

// Per-wave linear -> paged FP8 quant-store (kv_paged_waves.hip): the
// converter packs four tokens of one cache row per dword, so the quantised
// tile leaves the lane already transposed.
template <int ELT_C, int ELT_L, int CODEC, int LDT, int BS>
hipError_t launch_wave_scatter(const TileArgs& a, int64_t planes, hipStream_t stream);

// Per-wave 16-bit linear -> paged scatter in destination order
// (kv_paged_waves.hip): needs this call's claim tags as the inverse map.
template <int BS>
hipError_t launch_wave_copy_scatter(const TileArgs& a, int64_t planes, hipStream_t stream);

// Paged-A copies whose cache rows are whole 128-byte lines (kv_paged_wide.hip).
// `lines`: every linear row covers whole 128-byte lines.
template <int ELT, bool SCATTER>
hipError_t launch_wide(const TileArgs& a, int64_t planes, bool lines, hipStream_t stream);

// Largest block size launch_wide takes: its 32-bit offsets span a workgroup's
// rows (at most 64) at a row pitch of block_size elements.
constexpr int64_t kWideMaxBlockSize = 65536;

// Rules of the wide blocks (64-column units; 32-bit copies 32-column ones).
// What a call costs depends on the elements it moves, tokens x rows x planes,
// hardly on how they split up: rows of 64 to 4,096 elements and 1 or 16 layers
// were timed with single tokens, runs of 4 and 16 and whole sequences of 200,
// caches read from HBM, device time of the C entry, claim pass included.  The
// pairs below are us with the element kernel -> the wide kernels, rows of
// 1,024 | of 64 elements, one layer.
//
// Calls of fewer elements stay with the element kernel, whose one element per
// thread spreads a few tokens over more waves:
//   16-bit gather, 768 Ki: single 29.9 -> 30.2 | 32.1 -> 33.8, runs of 4 11.4 ->
//     13.2 | 11.1 -> 13.7, of 16 9.0 -> 7.6 | 8.3 -> 8.0, sequences 7.7 -> 5.4 |
//     6.9 -> 5.7 (at 512 Ki single tokens and runs of 4 lose 4 us);
//   32-bit gather, 512 Ki: 21.3 -> 21.7 | 21.8 -> 22.6, 9.0 -> 8.7 | 8.3 -> 9.2,
//     7.5 -> 5.5 | 6.5 -> 5.8, 6.9 -> 5.2 | 5.9 -> 5.6;
//   FP8 gather, 1,250 Ki: 29.9 -> 31.7 | 32.0 -> 34.4, 13.0 -> 13.2 | 12.6 ->
//     14.2, 10.4 -> 7.6 | 10.2 -> 8.5, 9.3 -> 8.1 | 9.1 -> 8.6;
//   16- and 32-bit scatter, 256 Ki (16-bit): 16.0 -> 16.4 | 18.7 -> 19.9, 9.1 ->
//     9.1 | 10.1 -> 11.0, 7.1 -> 5.9 | 8.7 -> 7.3, 6.5 -> 5.3 | 8.5 -> 6.9;
//   FP8 scatter, 1 Mi: 36.4 -> 39.3 | 39.1 -> 41.7, 18.2 -> 19.4 | 18.6 -> 20.4,
//     13.6 -> 12.8 | 16.5 -> 14.2, 11.9 -> 11.9 | 14.8 -> 12.5.
// Scatters of at most 256 tokens x planes move in one launch with the wide
// kernels, which find repeated slots themselves, and in two with the element
// kernel: 128 tokens of a sequence 6.5 -> 5.3 us.  FP8 ones gain nothing by it
// (32 tokens in runs of 16, 5.8 -> 10.3 us: a partial piece is stored byte by
// byte), unless the kernel checks the call's values too and the host waits for
// one launch instead of two (a call of 48 single tokens 10.9 -> 10.6 us, of runs
// of 16 10.8 -> 11.7).
constexpr bool wide_scatter_wins(int cache_elt, int64_t tokens, int64_t planes, int64_t elems, bool checks) {
  return (tokens * planes <= 256 && (cache_elt != 1 || checks)) ||
         elems >= (cache_elt == 1 ? int64_t{1} << 20 : int64_t{1} << 18);
}
constexpr bool wide_gather_wins(int cache_elt, int64_t elems) {
  return elems >= (cache_elt == 1 ? int64_t{5} << 18 : cache_elt == 2 ? int64_t{3} << 18 : int64_t{1} << 19);
}

// Past these limits with fewer workgroups than CUs a wave's 64 (32) tokens are
// a long serial chain while CUs idle (16-bit gathers of 384 single tokens of
// 1,024 rows: 51.8 us, 30.2 in one-wave workgroups; FP8 gathers of 625: 57.0 us,
// 31.7 with 16-token tiles), so such calls take smaller pieces.  (The figures
// below are with the caches' lines still in the memory-side cache.)
constexpr int64_t kWideFewGroups = 256;  // CUs
// 16- and 32-bit gathers, one-wave workgroups: 1,536 tokens of 1,024 rows of
// 16 bits 9.5 us in runs of 16 and 24.8 in runs of 4, 10.4 and 27.4 with four
// waves; level past 4 Mi elements.  32-bit ones are level from 1 Mi.
constexpr bool wide_gather_few(int cache_elt, int64_t elems) {
  return elems < (cache_elt == 2 ? int64_t{1} << 22 : int64_t{1} << 20);
}
// ... and their tiles of runs shorter than this move token by token: runs of 4
// of 8,192 tokens of 64 rows of 16 bits take 12.3 us with 6, 20.2 with 3; from 2
// Mi elements (32-bit: 1 Mi) 3 is the faster one (1,536 tokens of 1,024 rows
// 24.8 us).
constexpr int wide_gather_short_run(int cache_elt, int64_t elems) {
  return elems < (cache_elt == 2 ? int64_t{1} << 21 : int64_t{1} << 20) ? 6 : 3;
}
// Scatters, 8-token tiles (`groups`: workgroups of 64- or 32-token tiles): 512
// tokens of 1,024 rows of 16 bits in runs of 4 14.4 us, 26.0 with 64-token
// tiles; 2,048 45 against 39 us.  Calls of few tokens always take them.
constexpr int kWideFewScatterTile = 8;
constexpr bool wide_scatter_few(int64_t tokens, int64_t groups) { return groups < kWideFewGroups || tokens <= 128; }
// FP8 scatters: 1,536 tokens of 1,024 rows in runs of 16 22.4 us with 8-token
// tiles and 26.2 with 64, whole sequences 14.8 and 12.7.
constexpr bool wide_quant_few(int64_t tokens, int64_t elems) {
  return elems < (int64_t{3} << 20) || tokens <= 128;
}

}  // namespace kvhip
