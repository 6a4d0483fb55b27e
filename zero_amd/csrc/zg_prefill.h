// zg_prefill.h -- launchers of the batched prefill's own kernels (internal).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace zg {

// Causal attention of a chunk of prompt rows over the fp32 KV cache: row z
// sits at position pos0 + z, its normalised and rotated query heads at
// q + z * nq * HD, and attends to cache rows 0..pos0 + z (all written).  Its
// output row goes to out as fp32 when out is set, else Q8_0-encoded to qs
// (int8) and qsd (fp16 d bits).  A head whose max score or exp-sum is not
// finite sets bit 2 of *err.
struct PrefillAttnArgs {
  const float* q;
  const float* kcache;  // [max_ctx][nkv * HD], this layer's K rows
  const float* vcache;
  float* out;
  int8_t* qs;
  uint16_t* qsd;
  uint32_t* err;
  int nq, nkv, n, pos0;
  float scale;
  float* part;        // scratch of part_bytes (16-byte aligned), or null
  size_t part_bytes;
};
// Scratch with which few rows at a long context run on more CUs (0: they have
// no such form); the results do not depend on it.
size_t attn_prefill_scratch(int nq, int nkv, int head_dim, int n);
// head_dim 64 or 128
hipError_t launch_attn_prefill(const PrefillAttnArgs& a, int head_dim, hipStream_t st);

}  // namespace zg
