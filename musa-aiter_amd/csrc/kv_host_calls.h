/* Entries of libmusa_aiter_kv_hip.so that only this repository's Python host layer binds
 * (musa_aiter/ops/_hip.py packs their structs); the public ones are in include/musa_aiter_kv_hip.h. */
#ifndef MUSA_AITER_KV_HOST_CALLS_H_
#define MUSA_AITER_KV_HOST_CALLS_H_

#include <stdint.h>

#include "musa_aiter_kv_hip.h"

#ifdef __cplusplus
extern "C" {
#endif

/* Returned by the checked calls when an argument value is refused; nothing has moved. */
#define MUSA_AITER_HIP_REFUSED (-1)

/* musa_aiter_hip_paged_tiles (same fields) whose slots and scales are checked on the device: a slot
 * >= num_blocks * block_size or a scale that is not positive and finite refuses the call before
 * anything is written.  The verdict is read from `report`, `report_words` (>= 1) words of pinned
 * host memory, 0 at first, to which nothing but the verdicts of these entries is ever written; `guard`
 * is a device word (0 at first), `stamp` > 0 differs from every earlier call on the same report words
 * or guard, and calls sharing either are issued one after another on one stream.  The entry returns
 * when the verdict is there, which does not wait for the copy. */
typedef struct musa_aiter_hip_paged_tiles_call {
  int32_t scatter, codec, cache_elt, lin_elt, lin_dtype, scale_mode, fill_zeros, dedupe;
  int32_t discard;  /* a gather whose rows the caller throws away if it is refused: they may be written then */
  int32_t reserved;
  void *key_cache, *value_cache, *key_linear, *value_linear;
  const int64_t* slot_mapping;
  int64_t num_layers, num_tokens, num_blocks, num_heads, head_dim, block_size, lin_token_stride, lin_layer_stride;
  const float *k_scale, *v_scale;
  const musa_aiter_hip_claims* claims;
  int64_t* report;
  int64_t* guard;
  int64_t report_words, stamp;
} musa_aiter_hip_paged_tiles_call;
int musa_aiter_hip_paged_tiles_checked(const musa_aiter_hip_paged_tiles_call* call, void* stream);

/* musa_aiter_hip_copy_rows_paged (same fields) whose index entries are checked on the device as above:
 * one outside [low, src_rows) or [low, dst_rows) refuses the call (negative entries skip their row). */
typedef struct musa_aiter_hip_copy_rows_paged_call {
  const uint64_t *src_planes, *dst_planes;
  int64_t num_planes;
  const int64_t *src_idx, *dst_idx;
  int64_t num_tokens, src_rows, dst_rows, row_bytes, src_stride, dst_stride;
  int64_t src_page_rows, src_page_stride, dst_page_rows, dst_page_stride;
  int64_t low;
  const musa_aiter_hip_claims* claims;
  int64_t* report;
  int64_t* guard;
  int64_t report_words, stamp;
} musa_aiter_hip_copy_rows_paged_call;
int musa_aiter_hip_copy_rows_paged_checked(const musa_aiter_hip_copy_rows_paged_call* call, void* stream);

/* Block tables [batch, max_blocks] and seq_lens [batch] (device, int64) of a dense call, read on the
 * device: out[0] / out[1] receive the smallest and largest length, out[2] is 1 when a sequence uses a
 * block id outside [0, num_blocks) (ids past ceil(len / block_size), and columns the table does not
 * have, are not read), else 0.  report, report_words, stamp: as above (the words may be shared with
 * the calls above); values: 2 * report_words further words of pinned host memory, for the lengths,
 * in which no verdict is looked for.  Returns when the values are there. */
int musa_aiter_hip_block_tables_check(const int64_t* block_tables, const int64_t* seq_lens, int64_t batch,
                                      int64_t max_blocks, int64_t num_blocks, int64_t block_size, int64_t* report,
                                      int64_t report_words, int64_t* values, int64_t stamp, int64_t* out,
                                      void* stream);

/* hipThreadExchangeStreamCaptureMode: *mode becomes this thread's capture mode, and receives the one before. */
int musa_aiter_hip_exchange_capture_mode(int* mode);

#ifdef __cplusplus
}
#endif

#endif
