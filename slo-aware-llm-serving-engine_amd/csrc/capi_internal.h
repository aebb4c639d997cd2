// Error reporting shared by the C-ABI entry points.
#pragma once
#include <hip/hip_runtime.h>
#include "../../include/slo_attn.h"

namespace slo {

// Records `msg` as the calling thread's last error and returns `code`.
int fail(int code, const char* msg);

// Checks the launch that was just enqueued; never synchronises.
int check_launch(const char* what);

// Argument checks of a KV write (SLO_OK or an error, recorded): those of
// slo_store_kvcache, for every launch that writes the pool.
int check_store(const void* key, int64_t key_row_stride, const void* value, int64_t value_row_stride,
                const int32_t* slot_mapping, int32_t num_tokens, int32_t num_kv_heads, int32_t head_dim,
                int32_t kv_dtype, const void* k_cache, const void* v_cache, const float* k_scale, const float* v_scale,
                float scale_floor);

}  // namespace slo
