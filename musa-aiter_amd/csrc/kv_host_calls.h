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
 * host memory; `guard` is a device word (0 at first), `stamp` > 0 differs from every earlier call on
 * the same guard, and calls sharing a guard are issued one after another on one stream.  The entry
 * returns when the verdict is there, which does not wait for the copy. */
typedef struct musa_aiter_hip_paged_tiles_call {
  int32_t scatter, codec, cache_elt, lin_elt, lin_dtype, scale_mode, fill_zeros, dedupe;
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

#ifdef __cplusplus
}
#endif

#endif
