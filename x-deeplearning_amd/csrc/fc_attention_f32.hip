// fc_attention_f32.hip -- the attention MLP of a DIN model in fp32 as one launch: its input [x, y, x - y, x * y] computed
// while it is loaded, two layers and a skinny third (the reference's Concat of elementwise results followed by 3-D Gemms and
// their activations, tools/example_model/din/model/graph_ulf.txt; blaze/operator/op/concat_op.h:46-121, gemm_op.h:52-58,77-91).
// 2-byte models run theirs in fc_attention.hip.
#include <hip/hip_runtime.h>

#include <mutex>
#include <type_traits>

#include "bz_common.h"
#include "bz_pieces.h"
#include "fc_common.h"

namespace {

using namespace bz::fc;

// A launch of its own for the input, one for the first layer and one for the rest take their latency three times, and the
// input's 4 * w columns go to memory and back.  Here a workgroup of eight waves keeps both layers' weights in LDS and walks
// tiles of 32 rows, the next tile's operands on their way meanwhile: the waves share a tile's 16x16 blocks, and the layers
// hand each other 32 rows through LDS.  With 100 to 160 KB a workgroup there is one on a CU, so tiles are small and a launch is
// as many workgroups as there are tiles, up to the CUs.  An output is added up in four sums: scores against 64 bits
// 1.2e-7 to 2.2e-7, by the layers' own kernels 1.5e-7 to 2.3e-7.  201 x 23 rows, 192 -> 80 -> 40 -> 1: 6.4 + 6.8 + 7.6 us, 12.4
// this way; a request of that model 80.5 -> 70.5, of 1000 x 50 rows 172 -> 150; eight serving threads, us a pass, 201 samples
// 16.6 -> 11.9, 1024 35.0 -> 26.7, 2000 56.8 -> 49.3 (history lookups included).
constexpr int kRows = 32, kThreads = 512, kSums = 4;
constexpr int kMaxLds = 160 * 1024;

struct Layout {  // in floats
  int pa, ph, p2;                        // pitches: input tile and first weight; first outputs and second weight; second outputs
  int nb, nb2;                           // blocks of 16 columns
  int w1, h1, w2, h2, ps1, ps2, w3, all;  // beginnings (the input tile's is 0)
};

// Pitches of 4 floats more than a multiple of 16: the 16 rows of a fragment read start on 16 different groups of banks.
__host__ __device__ inline Layout layout(int k, int n, int n2) {
  Layout l;
  l.nb = (n + 15) / 16;
  l.nb2 = (n2 + 15) / 16;
  l.pa = (k + 15) / 16 * 16 + 4;
  l.ph = l.nb * 16 + 4;
  l.p2 = l.nb2 * 16 + 4;
  l.w1 = kRows * l.pa;
  l.h1 = l.w1 + l.nb * 16 * l.pa;
  l.w2 = l.h1 + kRows * l.ph;
  l.h2 = l.w2 + l.nb2 * 16 * l.ph;
  l.ps1 = l.h2 + kRows * l.p2;
  l.ps2 = l.ps1 + 4 * l.nb * 16;
  l.w3 = l.ps2 + 4 * l.nb2 * 16;
  l.all = l.w3 + kSkinnyMaxN * l.nb2 * 16;
  return l;
}

struct Attention {
  const float *x, *y;
  int64_t xs0, xs1, ys0, ys1;  // row m is x[m / r1 * xs0 + m % r1 * xs1 ..]
  int w, r1, m, n, k, n2;      // k = 4 * w
  const float *w1, *w2;
  int64_t ldw1, ldw2;
  Epilogue ep1, ep2;
  HeadArgs head;
};

// acc <- 16 rows of a times 16 rows of w over `steps` steps of 16, in kSums sums; a, w: this lane's first chunk
__device__ __forceinline__ floatx4 block_product(const float* a, const float* w, int steps) {
  floatx4 s[kSums];
#pragma unroll
  for (int i = 0; i < kSums; ++i) s[i] = floatx4{0.f, 0.f, 0.f, 0.f};
  for (int k = 0; k < steps; k += kSums) {
#pragma unroll
    for (int i = 0; i < kSums; ++i)
      if (k + i < steps) In<BZ_F32>::mma16(*(const uint4*)(a + (k + i) * 16), *(const uint4*)(w + (k + i) * 16), s[i]);
  }
  return (s[0] + s[1]) + (s[2] + s[3]);
}

// four outputs of a lane, rows 4 * (lane / 16) .. of column n of a block: activation, into LDS; zero in the columns beyond N
__device__ __forceinline__ void finish_block(const Epilogue& ep, const floatx4& v, const float* ps, int cols, int n, bool inside, float* out,
                                             int pitch) {
  const float b = ps[n], p0 = ps[cols + n], p1 = ps[2 * cols + n], p2 = ps[3 * cols + n];
  with_act(ep.act, [&](auto act) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float o = apply_act_t<decltype(act)::value>(fmaf(ep.alpha, v[r], b), ep, p0, p1, p2);
      out[r * pitch] = inside ? o : 0.f;
    }
  });
}

// A matrix of [rows, cols] floats into LDS rows `pitch` apart, 16 bytes a thread and pass: asked for first, put away later, so
// that everything a workgroup needs is on its way at once.  Chunks from `have_cols` on and rows from `have_rows` on are zero.
template <int PASSES>
struct Staged {
  uint4 r[PASSES];
  __device__ __forceinline__ void load(const float* src, int64_t ld, int rows, int cols, int have_rows, int have_cols) {
    const int per = cols / 4;
#pragma unroll
    for (int i = 0; i < PASSES; ++i) {
      const int q = threadIdx.x + i * kThreads, row = q / per, c = (q - row * per) * 4;
      const bool have = row < have_rows && c < have_cols;
      r[i] = *(const uint4*)(src + (have ? row * ld + c : 0));  // (no branch round the load)
      if (!have) r[i] = make_uint4(0, 0, 0, 0);
    }
  }
  __device__ __forceinline__ void store(float* dst, int pitch, int rows, int cols) const {
    const int per = cols / 4;
#pragma unroll
    for (int i = 0; i < PASSES; ++i) {
      const int q = threadIdx.x + i * kThreads, row = q / per, c = (q - row * per) * 4;
      if (row < rows) *(uint4*)(dst + row * pitch + c) = r[i];
    }
  }
};

// a layer's column parameters as the epilogue takes them, [4][cols], cols <= kThreads / 4: thread t's is t / cols of column t % cols
struct StagedParams {
  float v;
  __device__ __forceinline__ void load(const Epilogue& ep, int cols, int n, const float* any) {
    const int which = threadIdx.x / cols, c = min((int)threadIdx.x - which * cols, n - 1);
    const bool dice = ep.act == BZ_ACT_DICE, prelu = ep.act == BZ_ACT_PRELU;
    const float* src = which == 0 ? ep.bias : which == 1 ? ep.p0 : which == 2 ? ep.p1 : ep.p2;
    const bool use = which == 0 ? ep.bias_rows == 1 : which == 1 ? dice || prelu : which < 4 && dice;
    v = *(use ? src + (which == 1 && prelu && ep.act_size == 1 ? 0 : c) : any);
    if (!use) v = 0.f;
  }
  __device__ __forceinline__ void store(const Epilogue& ep, float* ps, int cols) const {
    const int which = threadIdx.x / cols;
    if (which < 4) ps[threadIdx.x] = which == 0 ? ep.beta * v : which == 3 && ep.act == BZ_ACT_DICE ? dice_inv_den(ep, v) : v;
  }
};

// VEC: columns of x and y a lane loads at once; HN: outputs of the third layer the code is unrolled for
template <int VEC, int HN>
__global__ __launch_bounds__(kThreads, 2) void bz_fc_attention_f32_kernel(const Attention a) {
  using Pack = bz::CewPack<float, VEC>;
  constexpr int kLoads = (kRows * 56 / VEC + kThreads - 1) / kThreads;  // w is at most 56
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const Layout l = layout(a.k, a.n, a.n2);
  float *h1 = lds + l.h1, *w1 = lds + l.w1, *w2 = lds + l.w2, *h2 = lds + l.h2, *w3 = lds + l.w3;
  const int tiles = (a.m + kRows - 1) / kRows;

  // this thread's share of a tile of x and y: the same columns of the same rows in every tile
  const int cw = a.w / VEC;
  int row[kLoads], col[kLoads];
  Pack x[kLoads], y[kLoads];
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int e = tid + i * kThreads;
    row[i] = e / cw;
    col[i] = (e - row[i] * cw) * VEC;
  }
  auto load = [&](int tile) {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int m = min(tile * kRows + min(row[i], kRows - 1), a.m - 1);
      const int i0 = m / a.r1, i1 = m - i0 * a.r1;
      x[i] = *(const Pack*)(a.x + i0 * a.xs0 + i1 * a.xs1 + col[i]);
      y[i] = *(const Pack*)(a.y + i0 * a.ys0 + i1 * a.ys1 + col[i]);
    }
  };
  load(blockIdx.x);
  const HeadBias<HN> hbias(a.head);

  // both weights, zero beyond their rows and columns, the third layer's, the parameters
  Staged<(96 * 56 + kThreads - 1) / kThreads> s1;
  Staged<64 * 24 / kThreads> s2;
  StagedParams p1, p2;
  s1.load(a.w1, a.ldw1, l.nb * 16, l.pa - 4, a.n, a.k);
  s2.load(a.w2, a.ldw2, l.nb2 * 16, l.ph - 4, a.n2, (int)a.ldw2);
  p1.load(a.ep1, l.nb * 16, a.n, a.w1);
  p2.load(a.ep2, l.nb2 * 16, a.n2, a.w1);
  const int w3r = tid / (l.nb2 * 16), w3c = tid - w3r * (l.nb2 * 16);
  const bool w3have = w3r < a.head.n && w3c < a.n2;
  const float w3v = *(w3have ? (const float*)a.head.w + w3r * a.head.ldw + w3c : a.w1);
  s1.store(w1, l.pa, l.nb * 16, l.pa - 4);
  s2.store(w2, l.ph, l.nb2 * 16, l.ph - 4);
  p1.store(a.ep1, lds + l.ps1, l.nb * 16);
  p2.store(a.ep2, lds + l.ps2, l.nb2 * 16);
  if (w3r < kSkinnyMaxN) w3[tid] = w3have ? w3v : 0.f;
  const int pad = l.pa - 4 - a.k;  // columns of the input tile that are always zero
  if (pad > 0)
    for (int q = tid; q < kRows * pad; q += kThreads) lds[q / pad * l.pa + a.k + q % pad] = 0.f;

  const int rb = (wave & 1) * 16, frow = lane & 15, fk = (lane >> 4) * 4;
  for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    // (nobody reads the input tile any more: the barrier behind the first layer)
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      if (row[i] < kRows) {
        float* o = lds + row[i] * l.pa + col[i];
        *(Pack*)o = x[i];
        *(Pack*)(o + a.w) = y[i];
        *(Pack*)(o + 2 * a.w) = bz::cew_piece<float, VEC>(BZ_EW_SUB, x[i], y[i]);
        *(Pack*)(o + 3 * a.w) = bz::cew_piece<float, VEC>(BZ_EW_MUL, x[i], y[i]);
      }
    }
    if (tile + (int)gridDim.x < tiles) load(tile + gridDim.x);
    __syncthreads();
    for (int b = wave >> 1; b < l.nb; b += 4) {
      const int n = b * 16 + frow;
      const floatx4 v = block_product(lds + (rb + frow) * l.pa + fk, w1 + n * l.pa + fk, (l.pa - 4) / 16);
      finish_block(a.ep1, v, lds + l.ps1, l.nb * 16, n, n < a.n, h1 + (rb + fk) * l.ph + n, l.ph);
    }
    __syncthreads();
    if (wave >> 1 < l.nb2) {
      const int n = (wave >> 1) * 16 + frow;
      const floatx4 v = block_product(h1 + (rb + frow) * l.ph + fk, w2 + n * l.ph + fk, l.nb);
      finish_block(a.ep2, v, lds + l.ps2, l.nb2 * 16, n, n < a.n2, h2 + (rb + fk) * l.p2 + n, l.p2);
    }
    __syncthreads();
    // the third layer: sixteen lanes a row, four columns each
    const int r = tid >> 4, c = (tid & 15) * 4, m = tile * kRows + r;
    float dot[HN];
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (c < l.nb2 * 16) v = *(const float4*)(h2 + r * l.p2 + c);
#pragma unroll
    for (int j = 0; j < HN; ++j) {
      dot[j] = 0.f;
      if (j < a.head.n) {
        float4 u = make_float4(0.f, 0.f, 0.f, 0.f);
        if (c < l.nb2 * 16) u = *(const float4*)(w3 + j * l.nb2 * 16 + c);
        dot[j] = group_sum<16>(fmaf(v.w, u.w, fmaf(v.z, u.z, fmaf(v.y, u.y, v.x * u.x))));
      }
    }
    if ((tid & 15) == 0 && m < a.m) head_finish(a.head, hbias, m, dot);
  }
}

template <int VEC, int HN>
int launch(const Attention& a, int lds, hipStream_t st) {
  static std::mutex mu;
  static bool raised[64] = {};
  int dev = 0;
  BZ_HIP_OK(hipGetDevice(&dev));
  {
    std::lock_guard<std::mutex> lock(mu);
    if (dev >= 0 && dev < 64 && !raised[dev]) {
      BZ_HIP_OK(hipFuncSetAttribute((const void*)bz_fc_attention_f32_kernel<VEC, HN>, hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds));
      raised[dev] = true;
    }
  }
  const int tiles = (a.m + kRows - 1) / kRows;
  hipLaunchKernelGGL((bz_fc_attention_f32_kernel<VEC, HN>), dim3(tiles < 256 ? tiles : 256), dim3(kThreads), lds, st, a);
  BZ_LAUNCH_OK("bz_fc_attention_f32_kernel");
  return BZ_OK;
}

}  // namespace

bool bz::fc_attention_f32_takes(int64_t k, int64_t n, int64_t n2) {
  return k <= 4 * 56 && n <= 96 && n2 <= 64 && layout((int)k, (int)n, (int)n2).all * (int)sizeof(float) <= kMaxLds;
}

int bz::fc_attention_f32(const bz_fc_desc& d, bz_stream_t stream) {
  if (d.a_pieces == nullptr || d.next == nullptr) return bz::fail(BZ_ENOTSUP, "attention MLP: no pieces or no second layer");
  const bz_fc_next& x = *d.next;
  bz::CewP p;
  int vec = 1;
  const int rc = bz::cew_build(*d.a_pieces, false, &p, &vec, "attention MLP");
  if (rc != BZ_OK) return rc;
  BZ_REQUIRE(p.rows == d.m && p.col0[p.n] == d.k, "attention MLP: the pieces describe [%lld, %d], the layer takes [%d, %d]", (long long)p.rows,
             p.col0[p.n], d.m, d.k);
  auto same = [&](int k, bool second, int src) {
    const void* ptr = second ? p.y[k] : p.x[k];
    const int64_t* s = second ? p.ys[k] : p.xs[k];
    return ptr == p.x[src] && s[0] == p.xs[src][0] && s[1] == p.xs[src][1];
  };
  const bool xy = bz::cew_uniform(p) && p.n == 4 && p.op[0] == BZ_EW_ASSIGN && p.op[1] == BZ_EW_ASSIGN && p.op[2] == BZ_EW_SUB &&
                  p.op[3] == BZ_EW_MUL && same(2, false, 0) && same(2, true, 1) && same(3, false, 0) && same(3, true, 1);
  auto plain = [](int act) { return act == BZ_ACT_NONE || act == BZ_ACT_PRELU || act == BZ_ACT_DICE || act == BZ_ACT_LEAKY_RELU || act == BZ_ACT_SIGMOID; };
  const bool aligned = (uintptr_t)d.w % 16 == 0 && d.ldw % 4 == 0 && (uintptr_t)x.w % 16 == 0 && x.ldw % 4 == 0;
  if (d.in_dtype != BZ_F32 || d.out_dtype != BZ_F32 || d.a_pieces->dtype != BZ_F32 || !xy || !fc_attention_f32_takes(d.k, d.n, x.n) || !aligned || d.y != nullptr || x.y != nullptr || d.head_n < 1 || d.head_n > kSkinnyMaxN || d.n_split != 0 ||
      d.bias_rows > 1 || !plain(d.act) || !plain(x.act) || p.r1 >= (1ll << 31) || d.m >= (1ll << 31) - 256 * kRows)
    return bz::fail(BZ_ENOTSUP, "attention MLP: a shape or form outside the kernel's");
  BZ_REQUIRE(d.w != nullptr && x.w != nullptr && d.head_w != nullptr && d.head_y != nullptr && d.ldw >= d.k && x.ldw >= d.n &&
                 d.head_ldw >= x.n && d.head_ldy >= d.head_n,
             "attention MLP: null operand or a leading dimension below its row");
  BZ_REQUIRE(d.bias_rows == 0 || d.bias != nullptr, "attention MLP: bias_rows=%d without bias", d.bias_rows);
  BZ_REQUIRE(d.act != BZ_ACT_PRELU || (d.act_p0 && (d.act_size == 1 || d.act_size == d.n)), "attention MLP: PRelu slope size %d", d.act_size);
  BZ_REQUIRE(d.act != BZ_ACT_DICE || (d.act_p0 && d.act_p1 && d.act_p2), "attention MLP: Dice needs gamma, mean and var");
  BZ_REQUIRE(x.act != BZ_ACT_PRELU || (x.act_p0 && (x.act_size == 1 || x.act_size == x.n)), "attention MLP: PRelu slope size %d", x.act_size);
  BZ_REQUIRE(x.act != BZ_ACT_DICE || (x.act_p0 && x.act_p1 && x.act_p2), "attention MLP: Dice needs gamma, mean and var");
  if (d.m == 0) return BZ_OK;
  Attention a = {};
  a.x = (const float*)p.x[0];
  a.y = (const float*)p.x[1];
  a.xs0 = p.xs[0][0];
  a.xs1 = p.xs[0][1];
  a.ys0 = p.xs[1][0];
  a.ys1 = p.xs[1][1];
  a.w = p.col0[1];
  a.r1 = (int)p.r1;
  a.m = d.m;
  a.n = d.n;
  a.k = d.k;
  a.n2 = x.n;
  a.w1 = (const float*)d.w;
  a.w2 = (const float*)x.w;
  a.ldw1 = d.ldw;
  a.ldw2 = x.ldw;
  a.ep1 = fc_epilogue(d);
  a.ep2.bias = x.bias;
  a.ep2.bias_rows = x.bias != nullptr ? 1 : 0;
  a.ep2.p0 = x.act_p0;
  a.ep2.p1 = x.act_p1;
  a.ep2.p2 = x.act_p2;
  a.ep2.act = x.act;
  a.ep2.act_size = x.act_size;
  a.ep2.dice_nosqrt = x.dice_nosqrt;
  a.ep2.alpha = x.alpha;
  a.ep2.beta = x.beta;
  a.ep2.act_alpha = x.act_alpha;
  a.head = head_args(d);
  hipStream_t st = bz::as_stream(stream);
  const int lds = layout(d.k, d.n, x.n).all * (int)sizeof(float);
  const bool two = head_unroll(d.head_n) == 2;
  if (vec >= 4) return two ? launch<4, 2>(a, lds, st) : launch<4, kSkinnyMaxN>(a, lds, st);
  if (vec == 2) return two ? launch<2, 2>(a, lds, st) : launch<2, kSkinnyMaxN>(a, lds, st);
  return two ? launch<1, 2>(a, lds, st) : launch<1, kSkinnyMaxN>(a, lds, st);
}
