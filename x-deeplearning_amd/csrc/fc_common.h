// fc_common.h -- what the FC kernels of fc_fused.hip and fc_pieces.hip share: the epilogue (Gemm's alpha / beta / bias,
// then the folded activation) and the MFMA element traits.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

#include <type_traits>

#include "bz_common.h"

namespace bz {
struct CewP;  // bz_pieces.h
namespace fc {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr float kDiceEps = 1e-8f;  // blaze/operator/common_helper.h:90

struct Epilogue {
  const float* bias;
  const float* p0;
  const float* p1;
  const float* p2;
  int bias_rows;
  int act;
  int act_size;
  int dice_nosqrt;
  float alpha, beta, act_alpha;
  // the N columns are `split_n`-wide slices (sibling FCs stacked along N): column n belongs to slice n / split_n, whose
  // output matrix [M, split_n] (row pitch ldy) starts split_stride elements after the previous slice's; a full bias is
  // laid out the same way, slice after slice.  split_n == 0: one matrix.
  int split_n;
  int64_t split_stride;
};

// element offset of output (m, n) in Y, and of the same element in a full [.., N] bias
__device__ __forceinline__ int64_t out_index(const Epilogue& ep, int64_t m, int n, int64_t ldy) {
  if (ep.split_n == 0) return m * ldy + n;
  const int p = n / ep.split_n;
  return p * ep.split_stride + m * ldy + (n - p * ep.split_n);
}
__device__ __forceinline__ int64_t full_bias_index(const Epilogue& ep, int64_t m, int n, int M, int N) {
  if (ep.split_n == 0) return m * N + n;
  const int p = n / ep.split_n;
  return ((int64_t)p * M + m) * ep.split_n + (n - p * ep.split_n);
}

// Dice as the standalone kernel computes it: the denominator of a column, and an output
__device__ __forceinline__ float dice_den(const Epilogue& e, float var) { return e.dice_nosqrt ? var : sqrtf(var + kDiceEps); }
__device__ __forceinline__ float dice_exact(float v, float gamma, float mean, float den) {
  const float t = expf(-1.f * (v - mean) / den);
  const float p = 1.f / (1.f + t);
  return (1.f - p) * gamma * v + p * v;
}

__device__ __forceinline__ float apply_act(float v, int n, const Epilogue& e) {
  switch (e.act) {
    case BZ_ACT_PRELU: {
      const float w = e.p0[e.act_size == 1 ? 0 : n];
      return v * ((float)(v > 0.f) + (float)(v < 0.f) * w);  // math/activation.h:37-42
    }
    case BZ_ACT_DICE:
      return dice_exact(v, e.p0[n], e.p1[n], dice_den(e, e.p2[n]));
    case BZ_ACT_LEAKY_RELU:
      return v >= 0.f ? v : e.act_alpha * v;
    case BZ_ACT_SIGMOID: {
      const float t = expf(v);
      return t / (1.f + t);
    }
    default:
      return v;
  }
}

// the same with the column's parameters already in registers (p0 = slope | gamma, p1 = mean, p2 = var)
__device__ __forceinline__ float apply_act_regs(float v, const Epilogue& e, float p0, float p1, float p2) {
  switch (e.act) {
    case BZ_ACT_PRELU:
      return v * ((float)(v > 0.f) + (float)(v < 0.f) * p0);
    case BZ_ACT_DICE:
      return dice_exact(v, p0, p1, dice_den(e, p2));
    case BZ_ACT_LEAKY_RELU:
      return v >= 0.f ? v : e.act_alpha * v;
    case BZ_ACT_SIGMOID: {
      const float t = expf(v);
      return t / (1.f + t);
    }
    default:
      return v;
  }
}

// log2(e) / (the Dice denominator of a column): computed once per column, before the K loop
__device__ __forceinline__ float dice_inv_den(const Epilogue& e, float var) {
  return 1.44269504088896341f / dice_den(e, var);
}

// The tile kernels' epilogue, activation fixed at compile time.  For Dice p2 is dice_inv_den() of the column, not its
// variance, and the element costs five plain instructions, one v_exp_f32 and one v_rcp_f32 (the attention MLP applies
// Dice to 120 outputs a history position: at 51200 x 50 positions the activation arithmetic alone is microseconds of
// every SIMD): a lane applies the activation to 32..128 outputs one after the other with one or two waves on its SIMD, so
// the exact expf and the two divisions per element (some 80 dependent instructions) were a third to a half of the run
// time of the attention layers (51200 x 216 -> 80: 23.6 us with Dice, 13.2 without).  v_exp_f32 and v_rcp_f32 are
// good to about 1 ulp of fp32 each; what they change in the result is far below the rounding of a 2-byte output and
// below 1e-6 relative for fp32 outputs.
template <int ACT>
__device__ __forceinline__ float apply_act_t(float v, const Epilogue& e, float p0, float p1, float p2) {
  if constexpr (ACT == BZ_ACT_PRELU) {
    return v * ((float)(v > 0.f) + (float)(v < 0.f) * p0);
  } else if constexpr (ACT == BZ_ACT_DICE) {
    const float t = __builtin_amdgcn_exp2f((p1 - v) * p2);  // e^((mean - v) / den)
    const float p = __builtin_amdgcn_rcpf(1.f + t);
    return fmaf(p, 1.f - p0, p0) * v;  // ((1 - p) gamma + p) v; 1 - gamma is the column's, hoisted out of the rows
  } else if constexpr (ACT == BZ_ACT_LEAKY_RELU) {
    return v >= 0.f ? v : e.act_alpha * v;
  } else if constexpr (ACT == BZ_ACT_SIGMOID) {
    const float t = expf(v);
    return t / (1.f + t);
  } else {
    return v;
  }
}

// f with the layer's activation as a constant
template <typename F>
__device__ __forceinline__ void with_act(int act, const F& f) {
  switch (act) {
    case BZ_ACT_PRELU: f(std::integral_constant<int, BZ_ACT_PRELU>()); break;
    case BZ_ACT_DICE: f(std::integral_constant<int, BZ_ACT_DICE>()); break;
    case BZ_ACT_LEAKY_RELU: f(std::integral_constant<int, BZ_ACT_LEAKY_RELU>()); break;
    case BZ_ACT_SIGMOID: f(std::integral_constant<int, BZ_ACT_SIGMOID>()); break;
    default: f(std::integral_constant<int, BZ_ACT_NONE>()); break;
  }
}

template <typename OutT>
__device__ __forceinline__ void store_out(OutT* p, float v);
template <>
__device__ __forceinline__ void store_out<float>(float* p, float v) {
  *p = v;
}
template <>
__device__ __forceinline__ void store_out<__half>(__half* p, float v) {
  *p = __float2half_rn(v);
}
template <>
__device__ __forceinline__ void store_out<__hip_bfloat16>(__hip_bfloat16* p, float v) {
  *p = __float2bfloat16(v);
}

// ---------------------------------------------------------------------------------------------
// element traits
// ---------------------------------------------------------------------------------------------
template <int DT>
struct In;
template <>
struct In<BZ_F16> {
  static constexpr int kSize = 2;
  static constexpr int kChunk = 8;   // elements per 16 bytes
  static constexpr int kStepK = 16;  // K consumed per fragment pair (both lane halves)
  static __device__ __forceinline__ void mma(const uint4& a, const uint4& b, floatx16& acc) {
    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(*(const half8*)&a, *(const half8*)&b, acc, 0, 0, 0);
  }
  // 16x16 block, K of 64 bytes: lane l holds row l % 16, bytes 16 * (l / 16) ..; result: column l % 16, rows 4 * (l / 16) ..
  static __device__ __forceinline__ void mma16(const uint4& a, const uint4& b, floatx4& acc) {
    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(*(const half8*)&a, *(const half8*)&b, acc, 0, 0, 0);
  }
};
template <>
struct In<BZ_BF16> {
  static constexpr int kSize = 2;
  static constexpr int kChunk = 8;
  static constexpr int kStepK = 16;
  static __device__ __forceinline__ void mma(const uint4& a, const uint4& b, floatx16& acc) {
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*(const bf16x8*)&a, *(const bf16x8*)&b, acc, 0, 0, 0);
  }
  static __device__ __forceinline__ void mma16(const uint4& a, const uint4& b, floatx4& acc) {
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8*)&a, *(const bf16x8*)&b, acc, 0, 0, 0);
  }
};
template <>
struct In<BZ_F32> {
  static constexpr int kSize = 4;
  static constexpr int kChunk = 4;
  static constexpr int kStepK = 8;
  // lane half h holds k = 4h..4h+3 of the 8-wide step; instruction i multiplies element i of both
  // halves, i.e. k in {i, 4+i}: a permutation of k applied equally to A and W.
  static __device__ __forceinline__ void mma(const uint4& a, const uint4& b, floatx16& acc) {
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a.x), __uint_as_float(b.x), acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a.y), __uint_as_float(b.y), acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a.z), __uint_as_float(b.z), acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a.w), __uint_as_float(b.w), acc, 0, 0, 0);
  }
  // (instruction i multiplies element i of the four lane groups: again one permutation of k for both operands)
  static __device__ __forceinline__ void mma16(const uint4& a, const uint4& b, floatx4& acc) {
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.x), __uint_as_float(b.x), acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.y), __uint_as_float(b.y), acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.z), __uint_as_float(b.z), acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.w), __uint_as_float(b.w), acc, 0, 0, 0);
  }
};

// A float as the sum of three bf16s: each the nearest to what the ones before leave over, 8 significant bits and a sign a
// piece, so that nothing is left over (|x| from 2^-110 up; below, what is left over is at most 2^-134, and 2^-126 where the matrix
// instructions take a piece that small for zero: whoever uses this looks for sums that may be of such products).  A product of two
// such sums, without the three of its nine products that are below 2^-25 of it, comes from the bf16 matrix instructions: six of
// them multiply 32x32x16 in 192 clocks, the fp32 ones in 512.
// A float that is no bf16 to be rounded to, an infinity or one within 2^-9 of it, makes infinite or undefined pieces, which
// make infinite or undefined sums: whoever uses this looks for them, too, and computes them with fp32 instructions.
struct Bf16x3 {
  uint4 hi, mid, lo;  // eight floats: element i in half i % 2 of word i / 2
};
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t nearest_bf16x2(float x0, float x1) {
  const bf16x2 h = __builtin_convertvector((floatx2{x0, x1}), bf16x2);  // v_cvt_pk_bf16_f32
  return *(const uint32_t*)&h;
}
__device__ __forceinline__ void split_pair(float x0, float x1, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
  hi = nearest_bf16x2(x0, x1);
  x0 -= __uint_as_float(hi << 16);
  x1 -= __uint_as_float(hi & 0xffff0000u);
  mid = nearest_bf16x2(x0, x1);
  x0 -= __uint_as_float(mid << 16);
  x1 -= __uint_as_float(mid & 0xffff0000u);
  lo = nearest_bf16x2(x0, x1);
}
__device__ __forceinline__ Bf16x3 split_floats(const uint4& a, const uint4& b) {
  Bf16x3 s;
  split_pair(__uint_as_float(a.x), __uint_as_float(a.y), s.hi.x, s.mid.x, s.lo.x);
  split_pair(__uint_as_float(a.z), __uint_as_float(a.w), s.hi.y, s.mid.y, s.lo.y);
  split_pair(__uint_as_float(b.x), __uint_as_float(b.y), s.hi.z, s.mid.z, s.lo.z);
  split_pair(__uint_as_float(b.z), __uint_as_float(b.w), s.hi.w, s.mid.w, s.lo.w);
  return s;
}

constexpr int kSkinnyMaxN = 8;

// the optional skinny second layer computed from the first layer's output tile while it is still in LDS
struct HeadArgs {
  const char* w;      // [n, ldw], K contiguous, the dtype of the first layer's operands
  const float* bias;  // [n] or null
  void* y;            // [M, ldy]
  int64_t ldw, ldy;
  int n, act, out_dtype;
  void* copy;         // the outputs once more, [M, n], or null (fc_fused)
};

// The code that is unrolled over a head's outputs exists for two (the usual heads) and for kSkinnyMaxN: a short kernel
// runs through code that no CU has at hand, and unrolled for eight with two used most of what it fetches is skipped.
inline int head_unroll(int n) { return n <= 2 ? 2 : kSkinnyMaxN; }

// the head's bias, asked for where a kernel starts: loaded at its end the whole of a small launch waits for it
template <int HN>
struct HeadBias {
  float b[HN];
  HeadBias() = default;
  __device__ __forceinline__ explicit HeadBias(const HeadArgs& head) { ask(head); }
  __device__ __forceinline__ void ask(const HeadArgs& head) {
#pragma unroll
    for (int j = 0; j < HN; ++j) b[j] = 0.f;
    if (head.bias != nullptr) {
#pragma unroll
      for (int j = 0; j < HN; ++j) b[j] = head.bias[j < head.n ? j : head.n - 1];
    }
  }
};

// the head's outputs of row m from its dot products: bias, activation, store
template <int HN>
__device__ __forceinline__ void head_finish(const HeadArgs& head, const HeadBias<HN>& bias, int m, const float (&dot)[HN]) {
  float v[HN];
#pragma unroll
  for (int j = 0; j < HN; ++j) v[j] = (j < head.n) ? dot[j] + bias.b[j] : 0.f;
  if (head.act == BZ_ACT_SOFTMAX) {  // softmax_op.cc:21-78: subtract max, exp, sum in order, divide
    float mx = v[0];
#pragma unroll
    for (int j = 1; j < HN; ++j)
      if (j < head.n) mx = v[j] > mx ? v[j] : mx;
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < HN; ++j)
      if (j < head.n) {
        v[j] = expf(v[j] - mx);
        sum += v[j];
      }
#pragma unroll
    for (int j = 0; j < HN; ++j)
      if (j < head.n) v[j] = v[j] / sum;
  } else if (head.act == BZ_ACT_SIGMOID) {
#pragma unroll
    for (int j = 0; j < HN; ++j) {
      const float t = expf(v[j]);
      v[j] = t / (1.f + t);
    }
  }
  auto store = [&](void* y, int64_t ld) {
#pragma unroll
    for (int j = 0; j < HN; ++j) {
      if (j < head.n) {
        const int64_t at = m * ld + j;
        if (head.out_dtype == BZ_F32)
          store_out<float>((float*)y + at, v[j]);
        else if (head.out_dtype == BZ_F16)
          store_out<__half>((__half*)y + at, v[j]);
        else
          store_out<__hip_bfloat16>((__hip_bfloat16*)y + at, v[j]);
      }
    }
  };
  store(head.y, head.ldy);
  if (head.copy != nullptr) store(head.copy, head.n);
}

// The sum over each aligned group of W lanes, in the group's first lane (the others hold parts): the halves added to each
// other down to one, as a butterfly of __shfl_xor adds them up for that lane.  Those go through the LDS unit, some 100
// clocks each; these are plain vector instructions.  All lanes of the wave have to be there.
template <int N>
__device__ __forceinline__ float row_shl(float v) {  // lane i of a row of 16: lane i + N's
  return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v), 0x100 + N, 0xf, 0xf, true));
}
__device__ __forceinline__ float row_quarters_sum(float v) {  // of lanes l, l ^ 16, l ^ 32, l ^ 48, in all four
  const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(h[0]) + __uint_as_float(h[1]);
  const auto q = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(q[0]) + __uint_as_float(q[1]);
}
template <int W>
__device__ __forceinline__ float group_sum(float v) {
  static_assert(W == 2 || W == 4 || W == 8 || W == 16 || W == 64, "a power of two within a row, or the wave");
  if constexpr (W == 64) v = row_quarters_sum(v);
  if constexpr (W >= 16) v += row_shl<8>(v);
  if constexpr (W >= 8) v += row_shl<4>(v);
  if constexpr (W >= 4) v += row_shl<2>(v);
  return v + row_shl<1>(v);
}

// The descriptor's head; all zero without one, whatever its other head_* fields hold: kernels that may do without a head
// ask for its bias before they look at head.n, and bias[head.n - 1] would lie in front of it.
inline HeadArgs head_args(const bz_fc_desc& d, void* copy = nullptr) {
  HeadArgs head = {};
  if (d.head_n <= 0) return head;
  head.w = (const char*)d.head_w;
  head.bias = d.head_bias;
  head.y = d.head_y;
  head.ldw = d.head_ldw;
  head.ldy = d.head_ldy;
  head.n = d.head_n;
  head.act = d.head_act;
  head.out_dtype = d.head_out_dtype;
  head.copy = copy;
  return head;
}

}  // namespace fc

// fc_pieces.hip: the layer whose A operand is given as pieces (bz_fc_desc.a_pieces); called by bz_fc_fused after its
// argument checks
int fc_pieces_launch(const bz_fc_desc& d, const fc::Epilogue& ep, hipStream_t st);
// fc_attention.hip: the layer on pieces [x, y, x - y, x * y] with a second and a skinny third one, all 2-byte; called by
// fc_pieces.hip, which has checked the descriptor.  BZ_ENOTSUP, with nothing launched, for a width it does not take.
int fc_attention(const bz_fc_desc& d, const CewP& p, const fc::Epilogue& ep1, const fc::Epilogue& ep2, hipStream_t st);
// the epilogue of a checked descriptor's (first) layer
fc::Epilogue fc_epilogue(const bz_fc_desc& d);
// The layer on a stored A, one function per operand type (fc_fused_f16.hip, fc_fused_bf16.hip, fc_fused_f32.hip): with a
// head when d.head_n != 0, else the skinny, tile or streaming kernel.  bz_fc_fused has checked the descriptor.
int fc_run_f16(const bz_fc_desc& d, const fc::Epilogue& ep, bool vec_a, bool vec_w, void* copy, hipStream_t st);
int fc_run_bf16(const bz_fc_desc& d, const fc::Epilogue& ep, bool vec_a, bool vec_w, void* copy, hipStream_t st);
int fc_run_f32(const bz_fc_desc& d, const fc::Epilogue& ep, bool vec_a, bool vec_w, void* copy, hipStream_t st);

}  // namespace bz
