// kh_attn_args.hpp - kernel arguments and helpers shared by the attention kernels.
#pragma once

#include "kh_common.hpp"

namespace kh {

constexpr int kQB = 32;  // queries per workgroup
constexpr int kKB = 32;  // keys per block
// buffer resource word 3 for gfx9-family raw buffers: 32-bit data format
constexpr int kBufferFlags = 0x00020000;

struct AttnArgs {
  const float *q, *k, *v;
  float *o;                // (a bf16 array when o16)
  const float *mask;
  int64_t q_b, q_t, k_b, k_t, v_b, v_t, o_b, o_t, m_b, m_q, m_k;
  int32_t batch, tq, tk, n_qblocks;
  int32_t mask_mode, scale_mode;
  float scale;
  int32_t o16;             // the output is bf16 (its consumer is a bf16 matmul)
  int32_t o_pair;          // the output is bf16 pair words (1) or fp16 pairs (2), as its consumer reads it
  float o_scale;           // fp16 pairs: the power of two the output is scaled by
  float qk_inv, v_inv;     // q, k, v in fp16 pairs: 1 / (scale of q * scale of k), 1 / scale of v
  uint64_t *rec;           // timeline probe only: 8 words per wave (kh_probe_attn_timeline)
};

// Exchange between the two lane halves (lanes l and l ^ 32): returns
// (x[l & 31], x[32 + (l & 31)]), the low half's value first in every lane,
// so a combine of the two is the same in both halves. One v_permlane32_swap.
__device__ __forceinline__ float2 halves(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return make_float2(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// Launch the fp16-pair kernel (kh_attn_f16.hip) for head dimension dh with nw
// key-split waves (hipErrorInvalidValue for a pair it is not compiled for).
hipError_t launch_attn_f16(const AttnArgs &a, int dh, int nw, dim3 grid, hipStream_t stream);

}  // namespace kh
