// kh_gemm_f16.hip - fp32 products on the fp16 matrix cores (configuration
// kind 8): C[b] = epilogue(A[b] @ B[b]) with both operands held as fp16 pairs
// (kh_common.hpp): A written that way by its producer, B the build-time
// [batch][N][K'] pair copy of a constant weight, each column n scaled by its
// own power of two. A product is three v_mfma_f32_16x16x32_f16 passes,
// l.h + h.l + h.h, accumulated in fp32, times the column's power of two.
//
// Same contract as the rest of the matmul family (the reference's tl.dot
// kernel with fused epilogue, kiln/gpu/codegen.py:484-530). The fp32 MFMA
// runs at 157 TFLOP/s; three fp16 passes are worth 840. Operands keep 23 bits
// where the plan sends a product here: activations down to 2^-27 of the bound
// their scale is chosen for, weights down to 2^-15 of their column's largest
// (kh_common.hpp, kiln/hip/bounds.py). On GPT-2 blocks the error against
// float64 is below that of the fp32 MFMA products, whose sums round once per
// four terms instead of once per 32.
//
// A pair row has the bytes of an fp32 row, and an MFMA operand (8 consecutive
// K values of one row) is one 16-byte chunk of h and one of l, so the LDS
// layout is like the K-contiguous fp32 kernel's: rows of 32 values = 8 chunks,
// chunk c of row r at c ^ swz_p(r). The MFMA time of a step is 3/16 of the
// fp32 kernel's, so what surrounds the MFMAs decides:
//   * fragments in two register sets: step s + 1's are read while step s's
//     feed the matrix cores, and every read and copy is issued between MFMAs;
//   * copies NS - 1 steps ahead: at the barrier of step s every wave holds
//     stage s in registers, so its slot is refilled with stage s + NS;
//   * the weights enter as the MFMA's row operand, so a lane's accumulator
//     is 4 consecutive output columns of one row and the epilogue needs no
//     staging: bias, residual and output are 16-byte accesses;
//   * 128x192 tiles for the largest products (8 waves, one workgroup per CU),
//     64x96 down to 32x64 with 2-3 workgroups per CU otherwise.
// Measured (fp32 configuration before, plan timing): 2048x3072x768 81.7 ->
// 31.9 us, 2048x768x3072 81.8 -> 35.5, 2048x2304x768 67.3 -> 29.5,
// 1024x3072x768 45.4 -> 18.8, 777x3072x768 44.8 -> 19.4. A probe of the
// 128x192 step (36 MFMAs, 14 reads and 5 copies per wave, one barrier) takes
// 1466 cycles where its MFMAs alone take 1180, and the clock falls to 1.6 -
// 1.9 GHz under it: 0.76 us a step against 0.97 here; 9 us of a launch are
// outside the steps (launch, first loads, the output written at once).
// K must be a positive multiple of 32 and the operands' spans below 2^29
// elements (the host checks both).
#include <algorithm>
#include <type_traits>

#include "kh_common.hpp"
#include "kh_gemm_args.hpp"
#include "kh_gemm_dev.hpp"
#include "kh_internal.hpp"

namespace kh {
namespace {

// LDS swizzle of a row's chunks, alike for rows 16 apart, so the fragment
// reads of a wave's 16-row blocks share their address registers. Free of bank
// conflicts: the 16 lanes of one LDS cycle (kh_gemm_dev.hpp) are rows li in
// {0-3, 12-15} reading chunk c and li in {4-11} reading chunk c + 2 (c of 0,
// 1, 4, 5); of the even rows the swizzles are 0 2 5 7 and 4 6 1 3, and c + 2
// is c ^ 2, so they meet chunks c ^ {0 2 5 7 6 4 3 1}; likewise the odd rows.
__device__ __forceinline__ int swz_p(int r) { return (r ^ ((r >> 3) & 1)) & 7; }

// TAPE = false: the direct epilogue (bias, residual, no activation, ReLU or
// GELU tanh) from registers; TAPE = true: any other epilogue, one loop over
// the wave's tile staged through LDS (one copy of the tape interpreter).
// Waves per SIMD that the LDS of the workgroups on a CU allows, at most 3
// (the register budget the compiler is held to).
template <int BM, int BN, int WAVES, int NS>
constexpr int waves_per_simd() {
  constexpr int groups = 160 * 1024 / (NS * (BM + BN) * 32 * 4);
  return groups * WAVES / 4 < 3 ? groups * WAVES / 4 : 3;
}

template <int BM, int BN, int WM, int WN, int NS, bool TAPE>
__global__ __launch_bounds__(64 * WM * WN) __attribute__((amdgpu_waves_per_eu(waves_per_simd<BM, BN, WM * WN, NS>())))
void gemm_f16_kernel(const GemmArgs a) {
  constexpr int BK = 32, MT = 16, CH = BK / 4;
  constexpr int kWaves = WM * WN;
  constexpr int TM = BM / WM, TN = BN / WN, FM = TM / MT, FN = TN / MT;
  constexpr int A_WORDS = BM * BK, STAGE = (BM + BN) * BK;
  constexpr int A_PER_WAVE = BM * CH / 64 / kWaves, B_PER_WAVE = BN * CH / 64 / kWaves;
  constexpr int COPIES = A_PER_WAVE + B_PER_WAVE;
  // SPLIT: the small products (b.l a.h, b.h a.l) accumulate apart from h.h and
  // join it at the end, so two thirds of the roundings happen at 2^-11 of the
  // sum's size (K = 768: error 3.2e-7 -> 1.9e-7 of the result, the fp32 MFMA
  // chain 5.0e-7), and apart from each other: A's l halves are stored times
  // 2^11. Not where two waves per SIMD leave no registers for it (92 spilled
  // with one more set): there B's h is multiplied by 2^-11 for that pass.
  constexpr bool SPLIT = kWaves == 4 || FM * FN <= 8;
  constexpr int ACCS = SPLIT ? 3 : 1;
  constexpr int CS = TN + 4;   // TAPE staging row stride (floats, 16-byte aligned rows)
  static_assert(TM % MT == 0 && TN % MT == 0, "wave tile of whole MFMA blocks");
  static_assert((BM * CH) % (64 * kWaves) == 0 && (BN * CH) % (64 * kWaves) == 0, "copy mapping");
  static_assert(NS >= 2 && NS <= 4 && (NS - 2) * COPIES < 64, "ring depth / vmcnt range");
  static_assert(NS * STAGE * 4 <= 160 * 1024, "LDS");
  static_assert(kWaves * MT * CS <= NS * STAGE, "epilogue staging fits the ring");

  __shared__ float4 ring[NS * STAGE / 4];

  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);
  const int wm = wave / WN, wn = wave % WN;
  const int li = lane & 15, g = lane >> 4;
  const int bidx = blockIdx.y;
  const float *Ab = a.A + (int64_t)bidx * a.sa_b;
  const float *Bb = a.B + (int64_t)bidx * a.sb_b;
  const int n_steps = a.K / BK;   // the host checks K % 32 == 0 and K > 0
  int tm, tn;
  tile_coords(blockIdx.x, a, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;

  // per-lane copy sources: byte offsets from the step's first K column (rows
  // past M / N clamped to the last one; their results are never stored)
  uint32_t a_off[A_PER_WAVE], b_off[B_PER_WAVE];
#pragma unroll
  for (int i = 0; i < A_PER_WAVE; ++i) {
    const int p = (wave * A_PER_WAVE + i) * 64 + lane, r = p / CH;
    a_off[i] = (uint32_t)(min(m0 + r, a.M - 1) * (int)a.sa_m + ((p % CH) ^ swz_p(r)) * 4) * 4u;
  }
#pragma unroll
  for (int i = 0; i < B_PER_WAVE; ++i) {
    const int p = (wave * B_PER_WAVE + i) * 64 + lane, r = p / CH;
    b_off[i] = (uint32_t)(min(n0 + r, a.N - 1) * (int)a.sb_n + ((p % CH) ^ swz_p(r)) * 4) * 4u;
  }
  const uint32_t ring_lds = (uint32_t)(uintptr_t)(lds_void_t *)ring;
  auto issue = [&](int step) {
    const float *abase = uniform_ptr(Ab + step * BK);
    const float *bbase = uniform_ptr(Bb + step * BK);
    const uint32_t lds = ring_lds + (uint32_t)((step % NS) * STAGE * 4);
#pragma unroll
    for (int i = 0; i < A_PER_WAVE; ++i) copy_to_lds<4>(abase, a_off[i], lds + (wave_u * A_PER_WAVE + i) * 1024);
#pragma unroll
    for (int i = 0; i < B_PER_WAVE; ++i)
      copy_to_lds<4>(bbase, b_off[i], lds + A_WORDS * 4 + (wave_u * B_PER_WAVE + i) * 1024);
  };
  // this wave's copies of a step have landed, `later` steps' copies being
  // issued after them
  auto wait_landed = [&](int later) {
    if (later <= 0) wait_vmcnt<0>();
    else if (later == 1 || NS < 4) wait_vmcnt<COPIES>();
    else wait_vmcnt<2 * COPIES>();
  };

  // fragment reads: chunk 2g + h of the lane's rows, at the wave's base plus
  // a constant per 16-row block (the swizzle repeats every 16 rows)
  const float *ringf = reinterpret_cast<const float *>(ring);
  const int chunk[2] = {((2 * g) ^ swz_p(li)) * 4, ((2 * g + 1) ^ swz_p(li)) * 4};
  const int fa_off = (wm * TM + li) * BK, fb_off = A_WORDS + (wn * TN + li) * BK;

  struct Frags {
    f16x8_t a[FM][2], b[FN][2];
  };
  // fragment i of a stage, in the order the passes want them (l of B and h of
  // A first)
  constexpr int READS = 2 * (FM + FN);
  auto read_one = [&](const float *st, int i, Frags &f) {
    if (i < FN) f.b[i][1] = *reinterpret_cast<const f16x8_t *>(st + fb_off + i * MT * BK + chunk[1]);
    else if (i < FN + FM) f.a[i - FN][0] = *reinterpret_cast<const f16x8_t *>(st + fa_off + (i - FN) * MT * BK + chunk[0]);
    else if (i < 2 * FN + FM)
      f.b[i - FN - FM][0] = *reinterpret_cast<const f16x8_t *>(st + fb_off + (i - FN - FM) * MT * BK + chunk[0]);
    else
      f.a[i - 2 * FN - FM][1] = *reinterpret_cast<const f16x8_t *>(st + fa_off + (i - 2 * FN - FM) * MT * BK + chunk[1]);
  };
  auto stage_words = [&](int step) { return ringf + (step % NS) * STAGE; };

  f32x4 accs[ACCS][FM][FN];
#pragma unroll
  for (int i = 0; i < ACCS; ++i)
#pragma unroll
    for (int fm = 0; fm < FM; ++fm)
#pragma unroll
      for (int fn = 0; fn < FN; ++fn) accs[i][fm][fn] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto &acc = accs[0];
  // the MFMAs of one column block in one pass: l.h, h.l, then h.h (the small
  // products first; a block's three passes are FM x FN MFMAs apart)
  f16x8_t down;   // !SPLIT: B's h times 2^-11 for the next group
  auto mfma_group = [&](int q, const Frags &f) {
    const int p = q / FN, fn = q % FN;
    const f16x8_t b = p == 1 && !SPLIT ? down : f.b[fn][p == 0];
#pragma unroll
    for (int fm = 0; fm < FM; ++fm) {
      f32x4 &c = accs[SPLIT ? 2 - p : 0][fm][fn];
      c = __builtin_amdgcn_mfma_f32_16x16x32_f16(b, f.a[fm][p == 1], c, 0, 0, 0);
    }
    if (!SPLIT && (q + 1) / FN == 1) down = f.b[(q + 1) % FN][0] * kPairDown;
  };
  auto mfmas = [&](const Frags &f) {
#pragma unroll
    for (int q = 0; q < 3 * FN; ++q) mfma_group(q, f);
  };
  auto join = [&] {
    if constexpr (SPLIT) {
#pragma unroll
      for (int fm = 0; fm < FM; ++fm)
#pragma unroll
        for (int fn = 0; fn < FN; ++fn) acc[fm][fn] += accs[1][fm][fn] * (float)kPairDown + accs[2][fm][fn];
    }
  };

  for (int p = 0; p < NS && p < n_steps; ++p) issue(p);
  wait_landed(min(NS, n_steps) - 1);
  stage_barrier();
  Frags fx, fy;
#pragma unroll
  for (int i = 0; i < READS; ++i) read_one(stage_words(0), i, fx);

  // Step s: stage s + 1 landed everywhere, and every wave's fragments of
  // stage s are in its registers (stage_barrier waits for this wave's LDS
  // reads), so its slot takes stage s + NS. The reads of stage s + 1 and the
  // copies are spread between the MFMA groups: issued in one run ahead of
  // them they left the matrix cores idle while both waves of a SIMD issued
  // (2048x3072x768: 33.7 us).
  constexpr int GROUPS = 3 * FN;
  auto step = [&](int s, const Frags &cur, Frags &next, auto steady) {
    constexpr bool kSteady = decltype(steady)::value;   // stage s + NS exists
    if constexpr (kSteady) wait_vmcnt<(NS - 2) * COPIES>();
    else wait_landed(min(NS - 2, n_steps - 2 - s));
    stage_barrier();
    if constexpr (!kSteady)
      if (s + NS < n_steps) issue(s + NS);
    const float *st = stage_words(s + 1);
    const float *abase = nullptr, *bbase = nullptr;
    uint32_t lds = 0;
    if constexpr (kSteady) {
      abase = uniform_ptr(Ab + (s + NS) * BK), bbase = uniform_ptr(Bb + (s + NS) * BK);
      lds = ring_lds + (uint32_t)((s % NS) * STAGE * 4);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < GROUPS; ++q) {
      mfma_group(q, cur);
      // copies one per so many groups over the whole step, reads over its
      // first three quarters
      if constexpr (kSteady) {
#pragma unroll
        for (int c = 0; c < COPIES; ++c) {
          if (c * GROUPS / COPIES != q) continue;
          if (c < A_PER_WAVE) copy_to_lds<4>(abase, a_off[c], lds + (wave_u * A_PER_WAVE + c) * 1024);
          else copy_to_lds<4>(bbase, b_off[c - A_PER_WAVE], lds + A_WORDS * 4 + (wave_u * B_PER_WAVE + c - A_PER_WAVE) * 1024);
        }
      }
#pragma unroll
      for (int i = 0; i < READS; ++i)
        if (i * (GROUPS * 3 / 4) / READS == q) read_one(st, i, next);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  int s = 0;
  for (; s + NS + 1 < n_steps; s += 2) {
    step(s, fx, fy, std::true_type{});
    step(s + 1, fy, fx, std::true_type{});
  }
  bool in_y = false;
  for (; s + 1 < n_steps; ++s) {
    step(s, fx, fy, std::false_type{});
    in_y = ++s + 1 >= n_steps;
    if (in_y) break;
    step(s, fy, fx, std::false_type{});
  }

  const int row0 = m0 + wm * TM, col0 = n0 + wn * TN;
  auto load4 = [&](int j, int m, int n, int valid) {
    const float *p = a.eptr[j] + (int64_t)bidx * a.estride[j][0] + (int64_t)m * a.estride[j][1];
    if ((a.e_vec_mask >> j & 1) && valid == 4) return *reinterpret_cast<const float4 *>(p + n);
    float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int i = 0; i < valid; ++i) v[i] = p[(int64_t)(n + i) * a.estride[j][2]];
    return make_float4(v[0], v[1], v[2], v[3]);
  };
  auto act = [&](float v) {
    if (a.d_act == KH_OP_GELU_TANH) return op_gelu_tanh(v);
    if constexpr (TAPE)
      if (a.d_act == KH_OP_GELU_ERF) return op_gelu_erf(v);
    if (a.d_act == KH_OP_RELU) return v != v ? v : fmaxf(v, 0.0f);
    return v;
  };
  auto store4 = [&](int m, int n, int valid, const float (&v)[4]) {
    float *o = a.eptr[a.d_out] + (int64_t)bidx * a.estride[a.d_out][0] + (int64_t)m * a.estride[a.d_out][1];
    if (a.o_pair) {
      store_f16_pairs4(o, n, make_float4(v[0], v[1], v[2], v[3]), a.o_scale);
    } else if ((a.e_vec_mask >> a.d_out & 1) && valid == 4) {
      *reinterpret_cast<float4 *>(o + n) = make_float4(v[0], v[1], v[2], v[3]);
    } else {
      for (int i = 0; i < valid; ++i) o[(int64_t)(n + i) * a.estride[a.d_out][2]] = v[i];
    }
  };

  if constexpr (!TAPE) {
    // the column scales and the bias are loaded ahead of the last step's MFMAs
    float4 cs[FN], bias[FN];
#pragma unroll
    for (int fn = 0; fn < FN; ++fn) {
      const int n = col0 + fn * MT + 4 * g, valid = min(4, a.N - n);
      cs[fn] = load4(a.d_cs, 0, n, valid);
      bias[fn] = a.d_bias >= 0 ? load4(a.d_bias, 0, n, valid) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (in_y) mfmas(fy);
    else mfmas(fx);
    join();
#pragma unroll
    for (int fm = 0; fm < FM; ++fm) {
      const int m = row0 + fm * MT + li;
      float4 res[FN];
      if (a.d_res >= 0) {
#pragma unroll
        for (int fn = 0; fn < FN; ++fn) {
          const int n = col0 + fn * MT + 4 * g;
          if (m < a.M && n < a.N) res[fn] = load4(a.d_res, m, n, min(4, a.N - n));
        }
      }
#pragma unroll
      for (int fn = 0; fn < FN; ++fn) {
        const int n = col0 + fn * MT + 4 * g;
        if (m >= a.M || n >= a.N) continue;
        // out = act((acc [+ bias]) [+ res]), in the tape's order
        float v[4] = {acc[fm][fn][0] * cs[fn].x, acc[fm][fn][1] * cs[fn].y, acc[fm][fn][2] * cs[fn].z,
                      acc[fm][fn][3] * cs[fn].w};
        if (a.d_bias >= 0) v[0] += bias[fn].x, v[1] += bias[fn].y, v[2] += bias[fn].z, v[3] += bias[fn].w;
        if (a.d_res >= 0)
          v[0] = res[fn].x + v[0], v[1] = res[fn].y + v[1], v[2] = res[fn].z + v[2], v[3] = res[fn].w + v[3];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = act(v[i]);
        store4(m, n, min(4, a.N - n), v);
      }
    }
  } else {
    if (in_y) mfmas(fy);
    else mfmas(fx);
    join();
    __syncthreads();   // every wave is done with the ring
    float *Cw = reinterpret_cast<float *>(ring) + wave * MT * CS;
#pragma unroll
    for (int fm = 0; fm < FM; ++fm) {
      // the slice is the wave's own: LDS operations of a wave complete in order
#pragma unroll
      for (int fn = 0; fn < FN; ++fn) *reinterpret_cast<f32x4 *>(Cw + li * CS + fn * MT + 4 * g) = acc[fm][fn];
      __builtin_amdgcn_wave_barrier();
#pragma unroll 1
      for (int q = lane; q < MT * TN / 4; q += 64) {
        const int r = q / (TN / 4), c = (q % (TN / 4)) * 4;
        const int m = row0 + fm * MT + r, n = col0 + c;
        if (m >= a.M || n >= a.N) continue;
        const int valid = min(4, a.N - n);
        const float4 p = *reinterpret_cast<const float4 *>(Cw + r * CS + c), cs = load4(a.d_cs, 0, n, valid);
        float v[4] = {p.x * cs.x, p.y * cs.y, p.z * cs.z, p.w * cs.w};
        if (!a.direct) {
          Vec<4> t;
          t.v[0] = v[0], t.v[1] = v[1], t.v[2] = v[2], t.v[3] = v[3];
          run_epilogue(a, bidx, m, n, valid, t);
          continue;
        }
        if (a.d_bias >= 0) {
          const float4 b = load4(a.d_bias, m, n, valid);
          v[0] += b.x, v[1] += b.y, v[2] += b.z, v[3] += b.w;
        }
        for (int i = 0; i < 4; ++i) v[i] = act(v[i]);   // (an activation excludes a residual)
        store4(m, n, valid, v);
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
}

}  // namespace

hipError_t launch_gemm_f16(int id, const GemmArgs &a, dim3 grid, hipStream_t stream) {
  const bool tape = !a.direct || a.d_act == KH_OP_GELU_ERF;
  switch (id) {
#define KH_CFGF16_CASE(cid, bm, bn, wm, wn, ns)                                                                \
  case cid:                                                                                                  \
    if (tape)                                                                                                \
      hipLaunchKernelGGL((gemm_f16_kernel<bm, bn, wm, wn, ns, true>), grid, dim3(64 * wm * wn), 0, stream, a); \
    else                                                                                                     \
      hipLaunchKernelGGL((gemm_f16_kernel<bm, bn, wm, wn, ns, false>), grid, dim3(64 * wm * wn), 0, stream, a); \
    break;
    KH_GEMM_F16_CONFIGS(KH_CFGF16_CASE)
#undef KH_CFGF16_CASE
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace kh
