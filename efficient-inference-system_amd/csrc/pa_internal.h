// What this package's own wrappers use of the library beside its public entry points (paged_hip.h).
#pragma once
#include <stddef.h>
#include <stdint.h>

extern "C" {
// Identifier of the graph capture that `stream` (not the default stream) is part of; 0: none.
unsigned long long paged_internal_capture_id(void* stream);

// pa_prefill_workspace_size for one KV dtype: a call over bf16 KV that runs unbalanced needs none, also
// where one over fp32 KV would be balanced.
size_t paged_internal_prefill_workspace(int kv_dtype, int32_t batch, int32_t num_heads, int32_t query_len,
                                        int32_t head_dim, int32_t max_pages, int32_t split_blocks);
}
