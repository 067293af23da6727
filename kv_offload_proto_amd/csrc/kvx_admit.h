// Entry point between the library and its Python module, beside the C ABI of
// kvx/kvx.h (the reference has no call of its own for it).
#pragma once

#include <cstdint>

extern "C" {

/* Admission of one request in every layer (xds_offload.py:56-77) in one
 * launch: slot s holds token s for s < min(prefill_len, device_buffer_size)
 * and -1 past it, visited bits and hand record cleared, the tables built,
 * prefill_lens[req_pool_idx] and req_host_base[req_batch_idx] (int64) set.
 * Tensors as sieve_update takes them, from layer 0.  ht_size a power of two in
 * [1024, 2^20], padded_buffer_size a multiple of 16 below 65536 and ht_size. */
int kvx_admit_request(uint64_t device_buffer_tokens, uint64_t device_buffer_visited, uint64_t device_buffer_ht,
                      uint64_t sieve_hand, uint64_t prefill_lens, uint64_t req_host_base, uint32_t req_batch_idx,
                      uint32_t req_pool_idx, int32_t prefill_len, int64_t host_base_row, uint32_t layer_num,
                      uint32_t pool_size, uint32_t device_buffer_size, uint32_t padded_buffer_size,
                      uint32_t visited_stride_b, uint32_t ht_size, uint64_t stream);

}  // extern "C"
