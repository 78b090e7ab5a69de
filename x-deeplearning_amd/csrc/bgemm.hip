// bgemm.hip -- strided-batched small GEMM for gfx950: C[i] = alpha*op(A[i])*op(B[i]) + beta*C[i].
//
// Stands in for GemmStridedBatched (blaze/math/gemm.cc:82-139, gemm.cu:251-336) as the
// reference reaches it from MatMul / BroadcastGemm_NxN (blaze/operator/op/matmul_op.h:77-89,
// blaze/math/broadcast.h:157-222), FusedParallelGemm (fused_parallel_gemm_op.h:96-129) and
// FusedParallelMatMul / BatchedBroadcastGemm_NxN (blaze/math/broadcast.h:267-381).
//
// Two kernels.  A row times a matrix (M = 1, B stored [K, N]: the DIN attention sum, 1xT . TxD) is one pass over B with
// nothing to reuse: bz_bgemm_row_kernel.  Everything else is a contraction whose operands are used M or N times, on the
// matrix cores: bz_bgemm_mfma_kernel.  fp32 accumulate in both.
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>

#include "bz_common.h"
#include "fc_common.h"

namespace {

template <typename T>
__device__ __forceinline__ float ld(const T* p);
template <>
__device__ __forceinline__ float ld<float>(const float* p) {
  return *p;
}
template <>
__device__ __forceinline__ float ld<__half>(const __half* p) {
  return __half2float(*p);
}
template <typename T>
__device__ __forceinline__ void st(T* p, float v);
template <>
__device__ __forceinline__ void st<float>(float* p, float v) {
  *p = v;
}
template <>
__device__ __forceinline__ void st<__half>(__half* p, float v) {
  *p = __float2half_rn(v);
}

// One wave per batch item, one lane per output column; K is walked in steps of kUnroll with all loads of a step issued
// before the first multiply-add.  The products are added in ascending k, the order bz_weighted_pool_kernel keeps as well.
constexpr int kUnroll = 32;

template <typename T>
__global__ __launch_bounds__(256) void bz_bgemm_row_kernel(const T* __restrict__ A, const T* __restrict__ B, T* __restrict__ C,
                                                           int64_t sa, int64_t sb, int64_t sc, int N, int K, int batch, float alpha,
                                                           float beta) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t item = (int64_t)blockIdx.x * 4 + wave;
  if (item >= batch) return;
  const T* a = A + sa * item;  // (a single row: [1, K] and [K, 1] are the same memory)
  const T* b = B + sb * item;
  T* c = C + sc * item;
  for (int n = lane; n < N; n += 64) {
    float acc = 0.f;
    for (int k0 = 0; k0 < K; k0 += kUnroll) {
      float av[kUnroll], bv[kUnroll];
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        const int k = k0 + u < K ? k0 + u : K - 1;  // clamped address; the product is skipped below
        av[u] = ld<T>(a + k);
        bv[u] = ld<T>(b + (int64_t)k * N + n);
      }
#pragma unroll
      for (int u = 0; u < kUnroll; ++u)
        if (k0 + u < K) acc = fmaf(av[u], bv[u], acc);
    }
    float v = alpha * acc;
    if (beta != 0.f) v += beta * ld<T>(c + n);  // beta == 0: C is not read (BLAS rule)
    st<T>(c + n, v);
  }
}

// ---------------------------------------------------------------------------------------------
// matrix-core kernel
// ---------------------------------------------------------------------------------------------
// The matrices are small (tens of rows and columns) and there are many: the work is one pass over A, B and C, and an
// item's operands fit LDS whole.  A workgroup of four waves owns G items (G = 1: a C tile of 64 x 64, a wave per 32 x 32
// block; G = 4: items of at most 32 x 32, a wave each), stages K in pieces of 128 bytes a row -- both operands K contiguous,
// rows padded by 16 bytes so that the fragment reads (16 bytes a lane) spread over the banks -- and stores C straight from
// the accumulators (a store instruction covers 32 neighbouring columns of two rows).  The next piece of K is loaded into
// registers while the present one is multiplied.
// An operand stored K contiguous is read 16 bytes a lane wherever its rows start (an item's matrix is contiguous, so most
// rows start on 2 bytes; the memory system takes such loads), the few chunks that would reach past the operand's last
// element by elements.  An operand stored the other way round is read 16 bytes a lane along its rows with neighbouring
// lanes on neighbouring k, so that the transposing LDS writes of a wave are contiguous.
// 1024 x [50,54]x[54,50] fp16 (16 MB, 3.3 us at the copy's rate): a lane per output element with scalar loads took 184 us.
constexpr int kRowB = 128;            // bytes of K staged per row
constexpr int kPitch = kRowB + 16;    // LDS pitch of a staged row

template <int DT>
struct Elem;
template <>
struct Elem<BZ_F16> {
  typedef __half T;
};
template <>
struct Elem<BZ_F32> {
  typedef float T;
};

// 16 bytes from any element-aligned address
__device__ __forceinline__ uint4 load16(const char* p) {
  uint4 v;
  __builtin_memcpy(&v, p, 16);
  return v;
}

// 16 bytes of which only the first `n` elements count (n <= 0: none): the rest come back as zeros.  `end`: one past the
// operand's last byte.
template <int ES>
__device__ __forceinline__ uint4 load_part(const char* p, int n, const char* end) {
  constexpr int CH = 16 / ES;
  uint4 v = make_uint4(0, 0, 0, 0);
  if (n <= 0) return v;
  if (p + 16 <= end) {
    v = load16(p);
  } else {
    uint32_t w[4] = {0, 0, 0, 0};
    for (int i = 0; i < CH; ++i)
      if (i < n) {
        if constexpr (ES == 4)
          w[i] = *(const uint32_t*)(p + 4 * i);
        else
          w[i / 2] |= (uint32_t) * (const unsigned short*)(p + 2 * i) << (16 * (i & 1));
      }
    v = make_uint4(w[0], w[1], w[2], w[3]);
  }
  if (n < CH) {
    uint32_t* w = (uint32_t*)&v;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if constexpr (ES == 4)
        w[j] = j < n ? w[j] : 0u;
      else
        w[j] = 2 * j + 1 < n ? w[j] : (2 * j < n ? w[j] & 0xffffu : 0u);
    }
  }
  return v;
}

// one operand's tile: ROWS rows (of M or N) by kRowB bytes of K, NT threads.  KC: the operand is stored K contiguous.
template <int DT, int ROWS, int NT, bool KC>
struct Stage {
  static constexpr int ES = bz::fc::In<DT>::kSize;
  static constexpr int CH = 16 / ES;                // elements per chunk
  static constexpr int BK = kRowB / ES;             // K per piece
  static constexpr int CHUNKS = ROWS * kRowB / 16;  // per piece
  static constexpr int PER = CHUNKS / NT;
  static_assert(CHUNKS % NT == 0, "tile");
  uint4 r[PER];
  // base: the item's matrix; ld: its row length; rows r0 .. of `rows`, k0 .. of K
  __device__ __forceinline__ void load(const char* base, const char* end, int t, int r0, int rows, int k0, int K) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int q = t + i * NT;
      if constexpr (KC) {
        const int row = r0 + q / (kRowB / 16), k = k0 + (q % (kRowB / 16)) * CH;
        r[i] = load_part<ES>(base + ((int64_t)row * K + k) * ES, row < rows ? K - k : 0, end);
      } else {
        const int k = k0 + q % BK, row = r0 + (q / BK) * CH;
        r[i] = load_part<ES>(base + ((int64_t)k * rows + row) * ES, k < K ? rows - row : 0, end);
      }
    }
  }
  __device__ __forceinline__ void store(char* lds, int t) const {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int q = t + i * NT;
      if constexpr (KC) {
        *(uint4*)(lds + (q / (kRowB / 16)) * kPitch + (q % (kRowB / 16)) * 16) = r[i];
      } else {
        const uint32_t w[4] = {r[i].x, r[i].y, r[i].z, r[i].w};
        char* p = lds + (q / BK) * CH * kPitch + (q % BK) * ES;
#pragma unroll
        for (int e = 0; e < CH; ++e) {
          if constexpr (ES == 4)
            *(uint32_t*)(p + e * kPitch) = w[e];
          else
            *(unsigned short*)(p + e * kPitch) = (unsigned short)(w[e / 2] >> (16 * (e & 1)));
        }
      }
    }
  }
};

template <int DT, bool TA, bool TB, int G>
__global__ __launch_bounds__(256) void bz_bgemm_mfma_kernel(const char* __restrict__ A, const char* __restrict__ B, int64_t sa, int64_t sb,
                                                            int M, int N, int K, int tiles, int total_wg, int wg_per_xcd, int batch,
                                                            typename Elem<DT>::T* __restrict__ C, int64_t sc, float alpha, float beta) {
  typedef typename Elem<DT>::T T;
  typedef bz::fc::In<DT> IN;
  constexpr int ES = IN::kSize;
  constexpr int BK = kRowB / ES;
  constexpr int TILE = G == 1 ? 64 : 32, NT = 256 / G;
  __shared__ __attribute__((aligned(16))) char lds[G][2 * TILE * kPitch];
  // the tiles of an item share its operands: neighbouring workgroups of one XCD (workgroups are dealt round robin)
  const int v = (int)(blockIdx.x % bz::kNumXcd) * wg_per_xcd + (int)(blockIdx.x / bz::kNumXcd);
  if (v >= total_wg) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int tiles_n = (N + TILE - 1) / TILE;
  const int tile = v % tiles;
  const int mine = v / tiles * G + (G == 1 ? 0 : wave);
  const bool live = G == 1 || mine < batch;
  const int64_t item = live ? mine : batch - 1;  // (a wave without an item of its own meets the barriers and stores nothing)
  const int t = G == 1 ? threadIdx.x : lane;
  const int m0 = tile / tiles_n * TILE, n0 = tile % tiles_n * TILE;
  const char* a = A + item * sa * ES;
  const char* b = B + item * sb * ES;
  const char* a_end = a + (int64_t)M * K * ES;
  const char* b_end = b + (int64_t)N * K * ES;
  char* la = lds[G == 1 ? 0 : wave];
  char* lb = la + TILE * kPitch;
  Stage<DT, TILE, NT, !TA> ga;
  Stage<DT, TILE, NT, TB> gb;
  ga.load(a, a_end, t, m0, M, 0, K);
  gb.load(b, b_end, t, n0, N, 0, K);
  bz::fc::floatx16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  const int wm = G == 1 ? (wave >> 1) * 32 : 0, wn = G == 1 ? (wave & 1) * 32 : 0;
  const char* fa = la + (wm + (lane & 31)) * kPitch + (lane >> 5) * 16;
  const char* fb = lb + (wn + (lane & 31)) * kPitch + (lane >> 5) * 16;
  // a block wholly outside C leaves the matrix cores to the other workgroups of the CU (fp32 5x150x64: half of the blocks)
  const bool works = m0 + wm < M && n0 + wn < N;
  for (int k0 = 0; k0 < K; k0 += BK) {
    ga.store(la, t);
    gb.store(lb, t);
    __syncthreads();
    if (k0 + BK < K) {
      ga.load(a, a_end, t, m0, M, k0 + BK, K);
      gb.load(b, b_end, t, n0, N, k0 + BK, K);
    }
    const int steps = works ? (min(K - k0, BK) + IN::kStepK - 1) / IN::kStepK : 0;
#pragma unroll
    for (int ks = 0; ks < BK / IN::kStepK; ++ks)
      if (ks < steps) IN::mma(*(const uint4*)(fa + ks * 32), *(const uint4*)(fb + ks * 32), acc);
    __syncthreads();
  }
  // a lane owns column n and rows 8 * (r / 4) + 4 * (lane / 32) + r % 4 of its block
  const int n = n0 + wn + (lane & 31);
  if (!live || n >= N) return;
  T* c = C + item * sc + n;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int m = m0 + wm + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
    if (m < M) {
      float x = alpha * acc[r];
      if (beta != 0.f) x += beta * ld<T>(c + (int64_t)m * N);  // beta == 0: C is not read (BLAS rule)
      st<T>(c + (int64_t)m * N, x);
    }
  }
}

template <int DT>
int launch_bgemm(const bz_bgemm_desc& d, hipStream_t s) {
  typedef typename Elem<DT>::T T;
  // A single row on a matrix stored [K, N] reads every element of B once: no tile, no transposition.
  if (d.m == 1 && !d.trans_b) {
    const int grid = (d.batch + 3) / 4;
    hipLaunchKernelGGL((bz_bgemm_row_kernel<T>), dim3(grid), dim3(256), 0, s, (const T*)d.a, (const T*)d.b, (T*)d.c, d.stride_a,
                       d.stride_b, d.stride_c, d.n, d.k, d.batch, d.alpha, d.beta);
    BZ_LAUNCH_OK("bz_bgemm_row_kernel");
    return BZ_OK;
  }
  const bool small = d.m <= 32 && d.n <= 32;
  const int tile = small ? 32 : 64;
  const int64_t tiles_m = (d.m + tile - 1) / tile, tiles_n = (d.n + tile - 1) / tile;
  const int64_t total = small ? (d.batch + 3) / 4 : tiles_m * tiles_n * d.batch;
  BZ_REQUIRE(total < (1ll << 30), "bz_gemm_strided_batched: m=%d n=%d batch=%d make too many tiles", d.m, d.n, d.batch);
  const int per_xcd = (int)((total + bz::kNumXcd - 1) / bz::kNumXcd);
#define BZ_BGEMM(TA, TB, G)                                                                                                        \
  hipLaunchKernelGGL((bz_bgemm_mfma_kernel<DT, TA, TB, G>), dim3(per_xcd * bz::kNumXcd), dim3(256), 0, s, (const char*)d.a,        \
                     (const char*)d.b, d.stride_a, d.stride_b, d.m, d.n, d.k, (int)(tiles_m * tiles_n), (int)total, per_xcd,        \
                     d.batch, (T*)d.c, d.stride_c, d.alpha, d.beta)
#define BZ_BGEMM_G(TA, TB) \
  if (small)               \
    BZ_BGEMM(TA, TB, 4);   \
  else                     \
    BZ_BGEMM(TA, TB, 1)
  if (d.trans_a && d.trans_b) {
    BZ_BGEMM_G(true, true);
  } else if (d.trans_a) {
    BZ_BGEMM_G(true, false);
  } else if (d.trans_b) {
    BZ_BGEMM_G(false, true);
  } else {
    BZ_BGEMM_G(false, false);
  }
#undef BZ_BGEMM_G
#undef BZ_BGEMM
  BZ_LAUNCH_OK("bz_bgemm_mfma_kernel");
  return BZ_OK;
}

// One wave per batch item, lanes over the channels.  Both sums walk t in ascending order, the weighted one with the
// fused multiply-add bz_bgemm_row_kernel uses for C = A^T * B, the plain one with separate adds like bz_reduce_sum_kernel,
// and the weight is rounded to the tensor type first, as the Mul operator would have stored it: the results are the
// three operators' results bit for bit.
// (a history of 50 in one round of loads: with one wave per item and four waves per CU the kernel is a chain of
// round trips to memory, 10 us at 16 steps per round on [1024, 50, 54])
constexpr int kPoolUnroll = 64;

template <typename T>
__global__ __launch_bounds__(256) void bz_weighted_pool_kernel(const T* __restrict__ w, const T* __restrict__ mask,
                                                               const T* __restrict__ x, T* __restrict__ att, T* __restrict__ sum,
                                                               int64_t batch, int t_len, int c_len, int64_t ld_att, int64_t ld_sum,
                                                               const T* __restrict__ copy_src, T* __restrict__ copy_dst, int copy_c,
                                                               int64_t ld_copy_src, int64_t ld_copy_dst) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t item = (int64_t)blockIdx.x * 4 + wave;
  if (item >= batch) return;
  // the piece copied alongside (asked for first: its loads travel with the history's)
  for (int c = lane; c < copy_c; c += 64) copy_dst[item * ld_copy_dst + c] = copy_src[item * ld_copy_src + c];
  const T* wp = w + item * t_len;
  const T* mp = mask ? mask + item * t_len : nullptr;
  const T* xp = x + item * (int64_t)t_len * c_len;
  // The channel loop is uniform over the wave: every lane runs every pass, so that lane u holds the weight of step
  // t0 + u when it is read with v_readlane below, whatever c_len is; a lane past the last channel reads the last
  // channel's address and stores nothing.
  for (int c0 = 0; c0 < c_len; c0 += 64) {
    const bool live = c0 + lane < c_len;
    const int c = live ? c0 + lane : c_len - 1;
    float acc_w = 0.f, acc_s = 0.f;
    for (int t0 = 0; t0 < t_len; t0 += kPoolUnroll) {
      // lane l fetches the weight of step t0 + l (every lane needs every weight: they are handed round below), then
      // its own channel of all the steps; nothing is used before everything has been asked for
      const int tl = t0 + lane < t_len ? t0 + lane : t_len - 1;
      const float w_raw = ld<T>(wp + tl);
      const float m_raw = mp ? ld<T>(mp + tl) : 1.f;
      float xv[kPoolUnroll];
#pragma unroll
      for (int u = 0; u < kPoolUnroll; ++u) {
        const int t = t0 + u < t_len ? t0 + u : t_len - 1;  // clamped address; the term is skipped below
        xv[u] = ld<T>(xp + (int64_t)t * c_len + c);
      }
      float w_mine = w_raw;
      if (mp) {
        T r;
        st<T>(&r, __fmul_rn(w_raw, m_raw));
        w_mine = ld<T>(&r);
      }
#pragma unroll
      for (int u = 0; u < kPoolUnroll; ++u)
        if (t0 + u < t_len) {
          const float wu = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(w_mine), u));
          acc_w = fmaf(wu, xv[u], acc_w);
          acc_s = __fadd_rn(acc_s, xv[u]);
        }
    }
    if (live && att) st<T>(att + item * ld_att + c, acc_w);
    if (live && sum) st<T>(sum + item * ld_sum + c, acc_s);
  }
}

}  // namespace

extern "C" int bz_weighted_pool(const bz_weighted_pool_desc* desc, bz_stream_t stream) {
  BZ_REQUIRE(desc != nullptr, "bz_weighted_pool: null descriptor");
  const bz_weighted_pool_desc& d = *desc;
  BZ_REQUIRE(d.x != nullptr && (d.att != nullptr || d.sum != nullptr), "bz_weighted_pool: null x, or neither output asked for");
  BZ_REQUIRE(d.att == nullptr || d.w != nullptr, "bz_weighted_pool: the weighted sum needs w");
  BZ_REQUIRE(d.batch >= 0 && d.t > 0 && d.c > 0, "bz_weighted_pool: bad shape batch=%lld t=%d c=%d", (long long)d.batch, d.t, d.c);
  const int64_t ld_att = d.ld_att ? d.ld_att : d.c, ld_sum = d.ld_sum ? d.ld_sum : d.c;
  const int64_t ld_cs = d.ld_copy_src ? d.ld_copy_src : d.copy_c, ld_cd = d.ld_copy_dst ? d.ld_copy_dst : d.copy_c;
  BZ_REQUIRE(ld_att >= d.c && ld_sum >= d.c, "bz_weighted_pool: ld_att=%lld / ld_sum=%lld below c=%d", (long long)ld_att, (long long)ld_sum, d.c);
  BZ_REQUIRE(d.copy_c >= 0 && (d.copy_c == 0 || (d.copy_src != nullptr && d.copy_dst != nullptr && ld_cs >= d.copy_c && ld_cd >= d.copy_c)),
             "bz_weighted_pool: copied piece of %d elements with a null pointer or a leading dimension below it", d.copy_c);
  if (d.batch == 0) return BZ_OK;
  BZ_REQUIRE((d.batch + 3) / 4 < (1ll << 31), "bz_weighted_pool: batch %lld too large", (long long)d.batch);
  const int grid = (int)((d.batch + 3) / 4);
  hipStream_t s = bz::as_stream(stream);
  const void* w = d.att ? d.w : d.x;  // no weighted sum: any readable address of t elements per item will do
  if (d.dtype == BZ_F32)
    hipLaunchKernelGGL(bz_weighted_pool_kernel<float>, dim3(grid), dim3(256), 0, s, (const float*)w, (const float*)(d.att ? d.mask : nullptr),
                       (const float*)d.x, (float*)d.att, (float*)d.sum, d.batch, d.t, d.c, ld_att, ld_sum, (const float*)d.copy_src,
                       (float*)d.copy_dst, d.copy_c, ld_cs, ld_cd);
  else if (d.dtype == BZ_F16)
    hipLaunchKernelGGL(bz_weighted_pool_kernel<__half>, dim3(grid), dim3(256), 0, s, (const __half*)w,
                       (const __half*)(d.att ? d.mask : nullptr), (const __half*)d.x, (__half*)d.att, (__half*)d.sum, d.batch, d.t, d.c,
                       ld_att, ld_sum, (const __half*)d.copy_src, (__half*)d.copy_dst, d.copy_c, ld_cs, ld_cd);
  else
    return bz::fail(BZ_ENOTSUP, "bz_weighted_pool: unsupported dtype %d", d.dtype);
  BZ_LAUNCH_OK("bz_weighted_pool_kernel");
  return BZ_OK;
}

extern "C" int bz_gemm_strided_batched(const bz_bgemm_desc* desc, bz_stream_t stream) {
  BZ_REQUIRE(desc != nullptr, "bz_gemm_strided_batched: null descriptor");
  const bz_bgemm_desc& d = *desc;
  BZ_REQUIRE(d.a && d.b && d.c, "bz_gemm_strided_batched: null a/b/c");
  BZ_REQUIRE(d.m > 0 && d.n > 0 && d.k > 0 && d.batch >= 0, "bz_gemm_strided_batched: bad shape m=%d n=%d k=%d batch=%d",
             d.m, d.n, d.k, d.batch);
  BZ_REQUIRE((int64_t)d.m * d.n < (1ll << 31), "bz_gemm_strided_batched: m*n too large");
  BZ_REQUIRE(d.stride_c >= (int64_t)d.m * d.n || d.batch <= 1, "bz_gemm_strided_batched: outputs overlap (stride_c=%lld)",
             (long long)d.stride_c);
  if (d.batch == 0) return BZ_OK;
  hipStream_t s = bz::as_stream(stream);
  if (d.dtype == BZ_F32) return launch_bgemm<BZ_F32>(d, s);
  if (d.dtype == BZ_F16) return launch_bgemm<BZ_F16>(d, s);
  return bz::fail(BZ_ENOTSUP, "bz_gemm_strided_batched: unsupported dtype %d", d.dtype);
}
