// fc_attention.hip -- the attention MLP of a 2-byte DIN model as one launch: its input [x, y, x - y, x * y] computed in
// registers, two layers and a skinny third (the reference's Concat of elementwise results followed by 3-D Gemms and their
// activations, tools/example_model/din/model/graph_ulf.txt; blaze/operator/op/concat_op.h:46-121, gemm_op.h:52-58,77-91).
// Called by fc_pieces.hip, which has checked the descriptor and takes other pieces and shorter chains; fp32 models run
// theirs in fc_attention_f32.hip.
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

#include <algorithm>
#include <mutex>
#include <type_traits>

#include "bz_common.h"
#include "bz_pieces.h"
#include "fc_common.h"

namespace {

using namespace bz::fc;

// A launch lasts some ten microseconds, most of them latency: trips to memory, chains of dependent instructions, code that no
// CU has at hand.  So a wave works for itself on 16 rows, from loading them to storing their scores, with nothing in LDS
// but what all waves read (both weights, arranged as the fragments they are read as, and the layers' parameters), behind the
// one barrier there is.
//  - Products are taken as weight times input (D = W * A^T): a lane holds four consecutive columns of one row of a layer's
//    output.  That is, but for the order of K, how the next product takes its input, and the order of K is free as long as
//    the weight is laid out in the same: the layers hand each other their rows in registers, converted in place.
//  - x and y are loaded as fragments, 16 bytes a lane.  A piece is padded to whole steps of K; the chunk it ends in is read
//    from where it lies wholly inside the row, its elements that belong to the chunk before are zero, in the weight too.
//  - A pass of the loop makes 32 columns of the first layer and multiplies them into the second: short code that stays at
//    hand, and registers for four waves to a SIMD.
// What bounds it alone: a third of a wave's 20 000 clocks are the weights' and parameters' trips to memory, the rest chains of
// instructions with two or three waves on a SIMD to fill them; beside others, the instructions (half of them in the layers'
// activations).  us alone / with eight streams of the same, in brackets the 128-row tiles of fc_pieces.hip that took
// these before: 1024 x 50 rows of 216 -> 80 -> 40 -> 1 fp16 11.5 / 6.6 (16.4 / 10.9), 2000 x 60 18.1 / 14.3 (30.1 / 26.6), 153 x 29 8.7 / 2.5
// (13.7 / 3.9), 300 x 40 of 96 -> 80 -> 40 -> 1 7.2 / 2.3 (11.1 / 3.1).  32 rows a wave read the weights from LDS half as often,
// but only two waves fit a SIMD: 10.9 / 7.8 and 17.4 / 15.3 at the first two sizes, and slower below.  The model on eight
// serving threads, 1024 samples 21.3 -> 16.1 us a pass, 201 12.4 -> 10.6, one pass alone 58.8 -> 50.0 and 50.2 -> 42.5.
constexpr int kMaxNB2 = 4;  // 16-column blocks of the second layer

struct Attention {
  const char *x, *y;
  int64_t xs0, xs1, ys0, ys1;  // row m is x[m / r1 * xs0 + m % r1 * xs1 ..]
  uint32_t r1;
  int w, m, n, n2;
  const char *w1, *w2;
  int64_t ldw1, ldw2;
  char *o1, *o2;  // the layers' outputs [m, ldo], or null
  int64_t ldo1, ldo2;
  Epilogue ep1, ep2;
  HeadArgs head;
};

// What a workgroup keeps in LDS, in bytes: the first layer's weight [pairs * 2 blocks of 16 columns][steps] fragments of 1 KB,
// the second's [nb2][pairs], and as words [5][kCols1], [5][kCols2] the parameters of either (beta * bias, slope or gamma, mean,
// log2(e) / den, all ones or zero beyond the layer's columns), [unrolled][kCols2] the third layer's weight
constexpr int kCols1 = 96, kCols2 = 16 * kMaxNB2;
struct Layout {
  int pairs, nb2;
  int w2, ps1, ps2, w3, all;
};
__host__ __device__ inline Layout layout(int steps, int n, int n2, int hn) {
  Layout l;
  l.pairs = (n + 31) / 32;
  l.nb2 = (n2 + 15) / 16;
  l.w2 = l.pairs * 2 * steps * 1024;
  l.ps1 = l.w2 + l.nb2 * l.pairs * 1024;
  l.ps2 = l.ps1 + 5 * kCols1 * 4;
  l.w3 = l.ps2 + 5 * kCols2 * 4;
  l.all = l.w3 + hn * kCols2 * 4;
  return l;
}

// x op y of a chunk, each element rounded to the type as bz_concat_ew would store it.  (fp16: the difference or product of
// two in fp32, rounded to fp16, is the one rounded once.)
template <int DT, int OP>
__device__ __forceinline__ uint4 piece(const uint4& x, const uint4& y) {
  if constexpr (DT == BZ_F16) {
    const half8 r = OP == BZ_EW_SUB ? *(const half8*)&x - *(const half8*)&y : *(const half8*)&x * *(const half8*)&y;
    return *(const uint4*)&r;
  } else {
    using Pack = bz::CewPack<__hip_bfloat16, 8>;
    const Pack r = bz::cew_piece<__hip_bfloat16, 8>(OP, *(const Pack*)&x, *(const Pack*)&y);
    return *(const uint4*)&r;
  }
}

// the first `skip` elements of a chunk are not kept
__device__ __forceinline__ uint4 keep_from(int skip) {
  auto word = [&](int i) { return skip >= 2 * i + 2 ? 0u : skip == 2 * i + 1 ? 0xffff0000u : 0xffffffffu; };
  return make_uint4(word(0), word(1), word(2), word(3));
}
__device__ __forceinline__ uint4 mask(const uint4& a, const uint4& m) { return make_uint4(a.x & m.x, a.y & m.y, a.z & m.z, a.w & m.w); }

// four elements from column k of a row, `ld` of them there to be read (a multiple of four)
__device__ __forceinline__ uint2 load_four(const char* row, int k, int64_t ld) { return *(const uint2*)(row + (k + 4 <= ld ? k : 0) * 2); }
// the first n of the four
__device__ __forceinline__ uint2 first(uint2 v, int n) {
  auto bits = [](int n) { return (uint32_t)(0xffffffffull >> (32 - 16 * min(max(n, 0), 2))); };
  return make_uint2(v.x & bits(n), v.y & bits(n - 2));
}

// One of a layer's four parameters, chosen by the wave: its source (`any`, memory that is there, where the layer has none), the
// columns it is read at, and what is kept of it.  No branches: everything is asked for before anything is waited for.
struct Param {
  const float* src;
  int last, which;
  uint32_t use;
  __device__ __forceinline__ Param(const Epilogue& ep, int which_, int n, const char* any) : which(which_) {
    const bool dice = ep.act == BZ_ACT_DICE, prelu = ep.act == BZ_ACT_PRELU;
    const float* s = which == 0 ? ep.bias : which == 1 ? ep.p0 : which == 2 ? ep.p1 : ep.p2;
    const bool have = which == 0 ? ep.bias_rows == 1 : which == 1 ? dice || prelu : dice;
    src = have ? s : (const float*)any;
    use = have ? 0xffffffffu : 0u;
    last = !have || (which == 1 && prelu && ep.act_size == 1) ? 0 : n - 1;
  }
  __device__ __forceinline__ float load(int c) const { return src[min(c, last)]; }
  __device__ __forceinline__ float finish(const Epilogue& ep, float v) const {
    const float r = which == 0 ? ep.beta * v : which == 3 ? dice_inv_den(ep, v) : v;
    return __uint_as_float(__float_as_uint(r) & use);
  }
};

// four columns of a layer's output, activated; ps: the first one's parameters, [5][cols]
template <int ACT>
__device__ __forceinline__ void finish_four(const Epilogue& ep, const floatx4& v, const float* ps, int cols, float (&out)[4]) {
  const float4 b = *(const float4*)ps, p0 = *(const float4*)(ps + cols), p1 = *(const float4*)(ps + 2 * cols), p2 = *(const float4*)(ps + 3 * cols);
  const uint4 keep = *(const uint4*)(ps + 4 * cols);
  out[0] = apply_act_t<ACT>(fmaf(ep.alpha, v[0], b.x), ep, p0.x, p1.x, p2.x);
  out[1] = apply_act_t<ACT>(fmaf(ep.alpha, v[1], b.y), ep, p0.y, p1.y, p2.y);
  out[2] = apply_act_t<ACT>(fmaf(ep.alpha, v[2], b.z), ep, p0.z, p1.z, p2.z);
  out[3] = apply_act_t<ACT>(fmaf(ep.alpha, v[3], b.w), ep, p0.w, p1.w, p2.w);
  out[0] = __uint_as_float(__float_as_uint(out[0]) & keep.x);
  out[1] = __uint_as_float(__float_as_uint(out[1]) & keep.y);
  out[2] = __uint_as_float(__float_as_uint(out[2]) & keep.z);
  out[3] = __uint_as_float(__float_as_uint(out[3]) & keep.w);
}

// four columns from n0 of a row of a stored output of n columns
template <typename ET>
__device__ __forceinline__ void store_four(char* out, int64_t ld, int m, int n0, int n, const ET* e) {
  ET* o = (ET*)out + m * ld + n0;
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (n0 + r < n) o[r] = e[r];
}

// S: steps of K a piece takes (32 elements each); HN: outputs of the third layer the code is unrolled for; STORE: the
// first two layers' outputs may be asked for, and the third layer may be missing
template <int DT, int S, int HN, bool STORE>
__global__ __launch_bounds__(512, STORE ? 2 : 4) void bz_fc_attention_kernel(const Attention a) {
  using T = In<DT>;
  using ET = typename std::conditional<DT == BZ_F16, __half, __hip_bfloat16>::type;
  constexpr int STEPS = 4 * S;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = blockDim.x >> 6;
  const int row = lane & 15, g = lane >> 4;
  const Layout l = layout(STEPS, a.n, a.n2, HN);
  float *ps1 = (float*)(lds + l.ps1), *ps2 = (float*)(lds + l.ps2), *w3 = (float*)(lds + l.w3);

  // this lane's columns of step s of a piece; of the last step's chunk only what the one before does not hold
  auto col = [&](int s) { return min(s * 32 + g * 8, a.w - 8); };
  const uint4 keep = keep_from((S - 1) * 32 + g * 8 - col(S - 1));

  const int tiles = (a.m + 15) / 16, stride = (int)gridDim.x * waves;
  uint4 x[S], y[S];
  auto load = [&](int tile) {
    const uint32_t m = min((uint32_t)tile * 16 + row, (uint32_t)a.m - 1);
    const uint32_t i0 = m / a.r1, i1 = m - i0 * a.r1;
    const char* px = a.x + ((int64_t)i0 * a.xs0 + (int64_t)i1 * a.xs1) * 2;
    const char* py = a.y + ((int64_t)i0 * a.ys0 + (int64_t)i1 * a.ys1) * 2;
#pragma unroll
    for (int s = 0; s < S; ++s) {
      __builtin_memcpy(&x[s], px + col(s) * 2, 16);
      __builtin_memcpy(&y[s], py + col(s) * 2, 16);
    }
  };
  int tile = blockIdx.x * waves + wave;
  load(tile);

  // the parameters, the third layer's weight and bias, the second's weight: asked for before anything is put away
  const HeadBias<HN> hbias(a.head);
  const Param p1(a.ep1, wave & 3, a.n, a.w1), p2(a.ep2, wave & 3, a.n2, a.w1);
  const float v1a = p1.load(lane), v1b = p1.load(lane + 64), v2 = p2.load(lane);
  constexpr int P3 = (HN + 3) / 4, P2 = (kMaxNB2 * 3 + 3) / 4;  // passes, of four waves at least
  float v3[P3];
#pragma unroll
  for (int i = 0; i < P3; ++i)
    v3[i] = bz::ldv<ET>((const ET*)(STORE && a.head.n == 0 ? a.w1 : a.head.w) + (STORE && a.head.n == 0 ? 0 : min(wave + i * waves, a.head.n - 1) * a.head.ldw + min(lane, a.n2 - 1)));
  // (the second layer's K in the order that the first one's outputs are held in: a chunk of eight is a lane's four of one
  // block and its four of the next)
  const int all2 = l.nb2 * l.pairs;
  uint2 w2v[P2][2];
#pragma unroll
  for (int i = 0; i < P2; ++i) {
    const int f = min(wave + i * waves, all2 - 1), j = f / l.pairs, t = f - j * l.pairs;
    const char* r = a.w2 + min(j * 16 + row, a.n2 - 1) * a.ldw2 * 2;
    w2v[i][0] = load_four(r, t * 32 + 4 * g, a.ldw2);
    w2v[i][1] = load_four(r, t * 32 + 16 + 4 * g, a.ldw2);
  }
  // fragments: a lane's chunk of fragment f is at f * 1 KB + lane * 16
  constexpr int B = 6;
  const int all1 = l.pairs * 2 * STEPS;
  for (int f0 = wave; f0 < all1; f0 += B * waves) {
    uint4 v[B];
#pragma unroll
    for (int i = 0; i < B; ++i) {
      const int f = min(f0 + i * waves, all1 - 1), j = f / STEPS, t = f - j * STEPS, p = t / S, s = t - p * S;
      __builtin_memcpy(&v[i], a.w1 + (min(j * 16 + row, a.n - 1) * a.ldw1 + p * a.w + col(s)) * 2, 16);
    }
#pragma unroll
    for (int i = 0; i < B; ++i) {
      const int f = f0 + i * waves, j = f / STEPS, t = f - j * STEPS;
      const uint32_t in = j * 16 + row < a.n ? 0xffffffffu : 0u, all = t % S == S - 1 ? 0u : 0xffffffffu;
      v[i] = make_uint4(v[i].x & (keep.x | all) & in, v[i].y & (keep.y | all) & in, v[i].z & (keep.z | all) & in, v[i].w & (keep.w | all) & in);
      if (f < all1) *(uint4*)(lds + f * 1024 + lane * 16) = v[i];
    }
  }
#pragma unroll
  for (int i = 0; i < P2; ++i) {
    const int f = wave + i * waves, j = f / l.pairs, t = f - j * l.pairs;
    const int n = (j * 16 + row < a.n2 ? a.n : 0) - (t * 32 + 4 * g);
    const uint2 lo = first(w2v[i][0], n), hi = first(w2v[i][1], n - 16);
    if (f < all2) *(uint4*)(lds + l.w2 + f * 1024 + lane * 16) = make_uint4(lo.x, lo.y, hi.x, hi.y);
  }
  if (wave < 4) {
    ps1[wave * kCols1 + lane] = p1.finish(a.ep1, v1a);
    if (lane + 64 < kCols1) ps1[wave * kCols1 + lane + 64] = p1.finish(a.ep1, v1b);
    ps2[wave * kCols2 + lane] = p2.finish(a.ep2, v2);
  }
  if (tid < kCols1) ps1[4 * kCols1 + tid] = __uint_as_float(tid < a.n ? 0xffffffffu : 0u);
  if (tid < kCols2) ps2[4 * kCols2 + tid] = __uint_as_float(tid < a.n2 ? 0xffffffffu : 0u);
#pragma unroll
  for (int i = 0; i < P3; ++i)
    if (wave + i * waves < HN) w3[(wave + i * waves) * kCols2 + lane] = wave + i * waves < a.head.n && lane < a.n2 ? v3[i] : 0.f;
  __syncthreads();

  for (; tile < tiles; tile += stride) {
    uint4 f[STEPS];
    x[S - 1] = mask(x[S - 1], keep);
    y[S - 1] = mask(y[S - 1], keep);
#pragma unroll
    for (int s = 0; s < S; ++s) {
      f[s] = x[s];
      f[S + s] = y[s];
      f[2 * S + s] = piece<DT, BZ_EW_SUB>(x[s], y[s]);
      f[3 * S + s] = piece<DT, BZ_EW_MUL>(x[s], y[s]);
    }
    const int m = tile * 16 + row;
    if (tile + stride < tiles) load(tile + stride);
    floatx4 acc2[kMaxNB2];
#pragma unroll
    for (int j = 0; j < kMaxNB2; ++j) acc2[j] = floatx4{0.f, 0.f, 0.f, 0.f};
    for (int pair = 0; pair < l.pairs; ++pair) {
      const char* w1 = lds + pair * (2 * STEPS * 1024) + lane * 16;
      floatx4 acc[2];
      acc[0] = acc[1] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < STEPS; ++t) {
#pragma unroll
        for (int h = 0; h < 2; ++h) T::mma16(*(const uint4*)(w1 + (h * STEPS + t) * 1024), f[t], acc[h]);
        if (t % 4 == 3) __builtin_amdgcn_sched_barrier(0);  // (the fragments of all steps at once do not fit the registers)
      }
      uint4 next;  // the two blocks as the second layer takes them
      with_act(a.ep1.act, [&](auto act) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          float o[4];
          finish_four<decltype(act)::value>(a.ep1, acc[h], ps1 + pair * 32 + h * 16 + 4 * g, kCols1, o);
#pragma unroll
          for (int r = 0; r < 4; ++r) store_out<ET>((ET*)&next + 4 * h + r, o[r]);
        }
      });
      if constexpr (STORE) {
        if (a.o1 != nullptr && m < a.m) {
          store_four<ET>(a.o1, a.ldo1, m, pair * 32 + 4 * g, a.n, (const ET*)&next);
          store_four<ET>(a.o1, a.ldo1, m, pair * 32 + 16 + 4 * g, a.n, (const ET*)&next + 4);
        }
      }
#pragma unroll
      for (int j = 0; j < kMaxNB2; ++j)
        if (j < l.nb2) T::mma16(*(const uint4*)(lds + l.w2 + (j * l.pairs + pair) * 1024 + lane * 16), next, acc2[j]);
    }
    // the third layer: a lane's columns, then the four lanes that share the row
    // (an opaque zero: the parameters are read here, not kept in 100 registers from tile to tile)
    int here = 0;
    asm volatile("" : "+s"(here));
    const float *ps = ps2 + 4 * g + here, *w = w3 + 4 * g + here;
    float dot[HN];
#pragma unroll
    for (int k = 0; k < HN; ++k) dot[k] = 0.f;
    with_act(a.ep2.act, [&](auto act) {
#pragma unroll
      for (int j = 0; j < kMaxNB2; ++j) {
        if (j < l.nb2) {
          float o[4];
          ET e[4];
          finish_four<decltype(act)::value>(a.ep2, acc2[j], ps + j * 16, kCols2, o);
#pragma unroll
          for (int r = 0; r < 4; ++r) store_out<ET>(&e[r], o[r]);
          if constexpr (STORE) {
            if (a.o2 != nullptr && m < a.m) store_four<ET>(a.o2, a.ldo2, m, j * 16 + 4 * g, a.n2, e);
          }
#pragma unroll
          for (int r = 0; r < 4; ++r) o[r] = bz::ldv<ET>(&e[r]);
#pragma unroll
          for (int k = 0; k < HN; ++k) {
            const float4 u = *(const float4*)(w + k * kCols2 + j * 16);
            dot[k] = fmaf(o[3], u.w, fmaf(o[2], u.z, fmaf(o[1], u.y, fmaf(o[0], u.x, dot[k]))));
          }
        }
      }
    });
    if (STORE && a.head.n == 0) continue;
#pragma unroll
    for (int k = 0; k < HN; ++k) dot[k] = row_quarters_sum(dot[k]);
    if (g == 0 && m < a.m) head_finish(a.head, hbias, m, dot);
  }
}

template <int DT, int S, int HN, bool STORE>
int launch(const Attention& a, hipStream_t st) {
  static std::mutex mu;
  static bool raised[64] = {};
  int dev = 0;
  BZ_HIP_OK(hipGetDevice(&dev));
  {
    std::lock_guard<std::mutex> lock(mu);
    if (dev >= 0 && dev < 64 && !raised[dev]) {
      BZ_HIP_OK(hipFuncSetAttribute((const void*)bz_fc_attention_kernel<DT, S, HN, STORE>, hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024));
      raised[dev] = true;
    }
  }
  // (at most 66 KB: two workgroups a CU)
  const int lds = layout(4 * S, a.n, a.n2, HN).all;
  const int tiles = (a.m + 15) / 16;
  // four waves a workgroup until every CU has one: a wave's share of the weights is larger, but more CUs work
  const int waves = tiles <= 4 * 256 ? 4 : 8;
  const int grid = std::min((tiles + waves - 1) / waves, 256 * (STORE ? 8 : 16) / waves);
  hipLaunchKernelGGL((bz_fc_attention_kernel<DT, S, HN, STORE>), dim3(grid), dim3(waves * 64), lds, st, a);
  BZ_LAUNCH_OK("bz_fc_attention_kernel");
  return BZ_OK;
}

template <int DT, int S>
int dispatch(const Attention& a, hipStream_t st) {
  if (a.o1 != nullptr || a.o2 != nullptr) return launch<DT, S, kSkinnyMaxN, true>(a, st);
  return head_unroll(a.head.n) == 2 ? launch<DT, S, 2, false>(a, st) : launch<DT, S, kSkinnyMaxN, false>(a, st);
}

}  // namespace

int bz::fc_attention(const bz_fc_desc& d, const bz::CewP& p, const fc::Epilogue& ep1, const fc::Epilogue& ep2, hipStream_t st) {
  if (p.col0[1] < 8 || p.r1 >= (1ll << 31) || d.m >= (1ll << 31) - 32 * 16 * 256) return BZ_ENOTSUP;
  if (d.m == 0) return BZ_OK;
  Attention a = {};
  a.x = (const char*)p.x[0];
  a.y = (const char*)p.x[1];
  a.xs0 = p.xs[0][0];
  a.xs1 = p.xs[0][1];
  a.ys0 = p.xs[1][0];
  a.ys1 = p.xs[1][1];
  a.r1 = (uint32_t)p.r1;
  a.w = p.col0[1];
  a.m = d.m;
  a.n = d.n;
  a.n2 = d.next->n;
  a.w1 = (const char*)d.w;
  a.w2 = (const char*)d.next->w;
  a.ldw1 = d.ldw;
  a.ldw2 = d.next->ldw;
  a.o1 = (char*)d.y;
  a.o2 = (char*)d.next->y;
  a.ldo1 = d.ldy;
  a.ldo2 = d.next->ldy;
  a.ep1 = ep1;
  a.ep2 = ep2;
  a.head = head_args(d);
  if (d.in_dtype == BZ_F16) return a.w <= 32 ? dispatch<BZ_F16, 1>(a, st) : dispatch<BZ_F16, 2>(a, st);
  return a.w <= 32 ? dispatch<BZ_BF16, 1>(a, st) : dispatch<BZ_BF16, 2>(a, st);
}
