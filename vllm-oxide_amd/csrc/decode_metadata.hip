// Device-side decode metadata: cu_seqlens_k and the slot of each sequence's
// new token, built on the GPU from context lengths and the padded block table.
//
// Semantics are the reference's decode-step preparation
// (crates/vllm-oxide/src/engine/mod.rs:247-267): for sequence b with
// L = context_lens[b] (the new token included),
//   cu_seqlens_k[b+1] = cu_seqlens_k[b] + L                   (metadata.rs:30-37)
//   slot_mapping[b]   = compute_slot_mapping(seq, L - 1, 1)   (kv_cache_manager.rs:115-135)
//                     = table[b][(L-1)/BS] * BS + (L-1) % BS, or -1 when that
//                       block index is past the row (>= max_blocks) or L == 0.
// The reference builds these on the host and uploads them in every layer; an
// engine that keeps context lengths and block tables on the device can run
// this once per step and feed every layer's append and attention from it.
//
// One workgroup, a lane per sequence up to 1024 of them: each lane sums a contiguous
// run of sequences, the run totals are scanned -- inside the waves by shuffles, the
// waves' totals through LDS -- and each lane writes its run's prefix sums and slots.
// Batches of up to 65535 sequences.  Its time is latency (the lengths, then the table
// entries they select, and the scan): 3.2 -> 1.9 us at 4 sequences against a scan of
// 1024 lanes through LDS with two barriers a step.
#include "oxide_common.hpp"

namespace {

constexpr int kLanes = 1024;

__global__ __launch_bounds__(kLanes) void decode_metadata_kernel(const uint32_t* __restrict__ context_lens,
                                                                 const int32_t* __restrict__ block_table,
                                                                 int64_t max_blocks, int batch,
                                                                 int block_size,
                                                                 uint32_t* __restrict__ cu_seqlens_k,
                                                                 int64_t* __restrict__ slot_mapping) {
  __shared__ uint32_t s_wave[kLanes / 64];
  const int t = threadIdx.x;
  const int per = (batch + blockDim.x - 1) / blockDim.x;
  const int b0 = t * per;
  const int b1 = min(batch, b0 + per);
  uint32_t run = 0;
  for (int b = b0; b < b1; ++b) run += context_lens[b];
  uint32_t acc = run;  // inclusive over the wave's runs
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t add = __shfl_up(acc, off);
    if ((t & 63) >= off) acc += add;
  }
  acc -= run;  // exclusive
  if (blockDim.x > 64) {
    if ((t & 63) == 63) s_wave[t >> 6] = acc + run;
    __syncthreads();
    for (int w = 0; w < t >> 6; ++w) acc += s_wave[w];
  }
  if (t == 0) cu_seqlens_k[0] = 0;
  for (int b = b0; b < b1; ++b) {
    const uint32_t L = context_lens[b];
    acc += L;
    cu_seqlens_k[b + 1] = acc;
    int64_t slot = -1;
    if (L > 0) {
      const uint32_t bs = static_cast<uint32_t>(block_size);
      const uint32_t blk = (L - 1) / bs;
      if (blk < max_blocks)
        slot = static_cast<int64_t>(block_table[static_cast<int64_t>(b) * max_blocks + blk]) * block_size +
               (L - 1) % bs;
    }
    slot_mapping[b] = slot;
  }
}

}  // namespace

extern "C" void build_decode_metadata_device(const uint32_t* context_lens, const int32_t* block_table,
                                             int64_t max_blocks_per_seq, int64_t batch,
                                             int64_t block_size, uint32_t* cu_seqlens_k,
                                             int64_t* slot_mapping, void* stream) {
  if (batch < 0 || max_blocks_per_seq < 0 || block_size <= 0 || batch > 65535 ||
      block_size > INT32_MAX) {
    oxide::set_error(OXIDE_ERR_INVALID_ARGUMENT);
    return;
  }
  if (!cu_seqlens_k || (batch > 0 && (!context_lens || !slot_mapping ||
                                      (max_blocks_per_seq > 0 && !block_table)))) {
    oxide::set_error(OXIDE_ERR_INVALID_ARGUMENT);
    return;
  }
  const int lanes = batch >= kLanes ? kLanes : static_cast<int>((batch + 63) / 64 * 64);
  hipLaunchKernelGGL(decode_metadata_kernel, dim3(1), dim3(lanes > 0 ? lanes : 64), 0, oxide::as_stream(stream),
                     context_lens, block_table, max_blocks_per_seq, static_cast<int>(batch),
                     static_cast<int>(block_size), cu_seqlens_k, slot_mapping);
  oxide::check_launch();
}
