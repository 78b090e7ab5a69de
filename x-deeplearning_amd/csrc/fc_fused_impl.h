// fc_fused_impl.h -- FC layer = GEMM + bias + activation in one kernel, for gfx950 MFMA.
//
// Stands in for the reference's pair  Gemm op (blaze/operator/op/gemm_op.h:33-107:
// Y <- broadcast(bias); Y = alpha*A*B + beta*Y via cblas/cuBLAS, blaze/math/gemm.cc:13-27,
// gemm.cu:35-104)  +  the separate PRelu / Dice / LeakyRelu / Sigmoid / Softmax op that
// follows it (prelu_op.cc:11-30, dice_op.cc:15-34, leaky_relu_op.cc:15-21,
// sigmoid_op.cc:15-21, softmax_op.cc:21-78).  The result equals the composition
// Activation(Gemm(x, W, b)) evaluated in fp32.
//
// Main kernel: C tile BM x BN per workgroup, K stepped by BK through double-buffered LDS
// (global -> registers -> LDS, one barrier per step) with the global loads of the next D
// tiles in flight in D register sets while the current tile is multiplied.  Operands are both "K contiguous" (A row major, W packed [N,K]) so
// a lane's MFMA fragment is one 16-byte LDS read; rows are padded by 16 bytes, which
// spreads the 16 lanes of a ds_read_b128 phase over all 64 banks.  fp16/bf16 use
// v_mfma_f32_32x32x16 (K=16 per instruction, fp32 accumulate); fp32 uses
// v_mfma_f32_32x32x2 with a K permutation inside each 8-wide step so its fragments are
// 16-byte reads as well.  In the accumulator a lane owns one output column and 16
// rows, so per-column epilogue parameters (bias, PReLU slope, Dice gamma/mean/var) are
// lane constants.
//
// Skinny kernel (N <= 8: the 256->2 softmax head, the 40->1 attention score, the 256->1
// sigmoid head): bandwidth bound on A; a lane group of pow2(K/8) lanes owns a row, the
// weight fragments live in registers, the N dot products are added up over it by lane swaps and DPP operands.
//
// Compiled once per operand type (fc_fused_f16.hip, fc_fused_bf16.hip, fc_fused_f32.hip include this file and define
// that type's entry, bz::fc_run_*): three translation units that build side by side instead of one that takes three
// times as long.  bz_fc_fused itself (argument checks, the choice of path) is in fc_fused.hip.
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

#include <mutex>
#include <type_traits>

#include "bz_common.h"
#include "fc_common.h"

namespace {

using namespace bz::fc;

// one 16-byte chunk of a K-contiguous operand row that may start anywhere; a chunk that reaches beyond K is read by
// elements and zero there
template <int DT>
__device__ __forceinline__ uint4 load_chunk(const char* base, int64_t row, int64_t ld, int k, int K) {
  constexpr int ES = In<DT>::kSize;
  constexpr int CH = In<DT>::kChunk;
  const char* p = base + (row * ld + k) * ES;
  uint4 out = make_uint4(0, 0, 0, 0);
  if (k + CH <= K) {
    __builtin_memcpy(&out, p, 16);
  } else if (k < K) {
    uint32_t e[4] = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < CH - 1; ++i)
      if (k + i < K) {
        if constexpr (ES == 2)
          e[i / 2] |= (uint32_t) * (const unsigned short*)(p + 2 * i) << (16 * (i & 1));
        else
          e[i] = *(const uint32_t*)(p + 4 * i);
      }
    out = make_uint4(e[0], e[1], e[2], e[3]);
  }
  return out;
}

// The same without a branch, for K of at least a chunk: the chunk is read from where it lies wholly inside the row, and
// shift_chunk drops the elements before k (and brings zeros in behind) when it is put into LDS.  The memory system takes
// 16-byte loads at any element; by elements and with one K tile in flight, 4096 x 3071 -> 1024 fp16 took 159 us and
// 600 x 900 -> 512 16.4.
template <int DT>
__device__ __forceinline__ uint4 load_chunk_anywhere(const char* base, int64_t row, int64_t ld, int k, int K) {
  uint4 out;
  __builtin_memcpy(&out, base + (row * ld + min(k, K - In<DT>::kChunk)) * In<DT>::kSize, 16);
  return out;
}
// `n` elements out at the front, zeros in at the back (n >= the chunk: all zeros)
template <int DT>
__device__ __forceinline__ uint4 shift_chunk(uint4 v, int n) {
  const int b = n * In<DT>::kSize;
  if (b & 4) v = make_uint4(v.y, v.z, v.w, 0u);
  if (b & 8) v = make_uint4(v.z, v.w, 0u, 0u);
  if (b & 2) v = make_uint4(v.x >> 16 | v.y << 16, v.y >> 16 | v.z << 16, v.z >> 16 | v.w << 16, v.w >> 16);
  if (b >= 16) v = make_uint4(0, 0, 0, 0);
  return v;
}

// The same for operands whose rows are 16-byte aligned and K a multiple of the chunk (a chunk is either wholly inside
// K or absent): no branches and nothing done to the loaded value, so the loads of several K tiles can stay in
// flight.  A chunk beyond K is read from 16 bytes of zeros instead of being masked after the load: a mask is an
// instruction on the loaded register, and the scheduler is free to place it - and the wait for the load it implies -
// right behind the load (it did so in the 128x256 tile: one exposed trip to memory in every K tile).
__device__ uint4 kZeroChunk = {0u, 0u, 0u, 0u};  // never written; not const, so that it lives in the global address space like the operands (a select between a global and a constant-space pointer would be loaded through FLAT)

template <int DT>
__device__ __forceinline__ uint4 load_chunk_aligned(const char* base, int64_t row, int64_t ld, int k, int K) {
  constexpr int ES = In<DT>::kSize;
  const char* p = k < K ? base + (row * ld + k) * ES : (const char*)&kZeroChunk;
  return *(const uint4*)p;
}

// The variant that reads a clamped address and leaves the zeroing of chunks beyond K to the consumer.  The eight-wave
// tile with the skinny head keeps it: there the address select costs more (11.1 against 10.5 us on config 2's
// 512 -> 256 -> 2) than the mask, which the scheduler leaves at the LDS store in that kernel.
template <int DT>
__device__ __forceinline__ uint4 load_chunk_clamped(const char* base, int64_t row, int64_t ld, int k, int K) {
  constexpr int ES = In<DT>::kSize;
  constexpr int CH = In<DT>::kChunk;
  const int kc = k < K ? k : K - CH;
  return *(const uint4*)(base + (row * ld + kc) * ES);
}


template <int DT>
__device__ __forceinline__ void chunk_to_float(const uint4& c, float (&f)[In<DT>::kChunk]) {
  const uint32_t r[4] = {c.x, c.y, c.z, c.w};
  if constexpr (DT == BZ_F32) {
#pragma unroll
    for (int i = 0; i < 4; ++i) f[i] = __uint_as_float(r[i]);
  } else if constexpr (DT == BZ_F16) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      f[2 * i] = __half2float(__ushort_as_half((unsigned short)(r[i] & 0xffffu)));
      f[2 * i + 1] = __half2float(__ushort_as_half((unsigned short)(r[i] >> 16)));
    }
  } else {  // bf16: the upper 16 bits of the fp32 pattern
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      f[2 * i] = __uint_as_float(r[i] << 16);
      f[2 * i + 1] = __uint_as_float(r[i] & 0xffff0000u);
    }
  }
}

// ---------------------------------------------------------------------------------------------
// tiled MFMA kernel
// ---------------------------------------------------------------------------------------------
// Sums an output is added up in where a wave owns one 32x32 block.  fp32: one for each step of a K tile, which also makes
// them shorter (error against 64 bits of 4096 x 896 -> 512, when these tiles computed it, 2.7e-7, 3.8e-7 with two).  Two otherwise, and in the tiles with
// a head, whose other registers are many: with four the 64x64 one takes 10.7 us for 17000 x 80 -> 40 instead of 10.3.
template <int DT, int BM, int BN, int BK, int WM, int WN, int HEAD>
constexpr int default_sums() {
  constexpr int steps = BK / In<DT>::kStepK;
  return BM / WM / 32 * (BN / WN / 32) > 1 ? 1 : DT == BZ_F32 && !HEAD ? steps : steps >= 2 ? 2 : 1;
}

// HEAD: outputs the code of the skinny second layer is unrolled for, 0 without one
template <int DT, typename OutT, int BM, int BN, int BK, int WM, int WN, int D, bool ALIGNED, int HEAD, int KACC>
__global__ __launch_bounds__(WM* WN * 64) void bz_fc_mfma_kernel(const char* __restrict__ A, const char* __restrict__ W,
                                                                  OutT* __restrict__ Y, int M, int N, int K, int64_t lda,
                                                                  int64_t ldw, int64_t ldy, bool vec_y, int tiles_m, Epilogue ep,
                                                                  HeadArgs head) {
  using T = In<DT>;
  constexpr int NT = WM * WN * 64;
  constexpr int ES = T::kSize;
  constexpr int ROWB = BK * ES;        // bytes of one tile row
  constexpr int PITCH = ROWB + 16;     // padded LDS pitch
  constexpr int CPR = ROWB / 16;       // 16-byte chunks per row
  constexpr int A_CHUNKS = BM * CPR, W_CHUNKS = BN * CPR;
  constexpr int A_PER = (A_CHUNKS + NT - 1) / NT, W_PER = (W_CHUNKS + NT - 1) / NT;
  constexpr int WTM = BM / WM, WTN = BN / WN;  // wave tile
  constexpr int TM = WTM / 32, TN = WTN / 32;  // 32x32 blocks per wave
  static_assert(WTM % 32 == 0 && WTN % 32 == 0 && BK % T::kStepK == 0, "tile shape");

  __shared__ __attribute__((aligned(16))) char lds[2][(BM + BN) * PITCH];
  // HEAD: the second layer's weight [HEAD, BN], requested now into registers, parked in LDS after the K loop
  constexpr int HW_ROW = BN * ES;  // bytes
  constexpr int HW_CHUNKS = HEAD ? HEAD * HW_ROW / 16 : 1;
  constexpr int HW_PER = (HW_CHUNKS + NT - 1) / NT;
  __shared__ __attribute__((aligned(16))) char lds_hw[HEAD ? HEAD * HW_ROW : 16];
  uint4 rhw[HW_PER];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave / WN, wn = wave % WN;
  // consecutive workgroups walk down M within one N panel: the W panel stays hot in L2
  const int tile_m = blockIdx.x % tiles_m, tile_n = blockIdx.x / tiles_m;
  const int m0 = tile_m * BM, n0 = tile_n * BN;

  // D register sets: K tiles kt+1 .. kt+D are in flight from global memory while tile kt is multiplied out of
  // LDS.  The kernel is latency bound at CTR sizes (a tile's MFMAs take ~0.1 us, a round trip ~1 us), so the
  // number of exposed round trips, ceil(KT / D), is what sets its duration.
  // which aligned loader: the head tile (see load_chunk_clamped) and the 256x256 tile, whose 256 registers have no room
  // for the zero-chunk select's addresses (it spilled 75 of them)
  constexpr bool CLAMPED = HEAD != 0 || BM * BN >= 256 * 256;
  uint4 ra[D][A_PER], rw[D][W_PER];
  auto gload = [&](int set, int k0) {
#pragma unroll
    for (int i = 0; i < A_PER; ++i) {
      const int q = tid + i * NT;
      if (A_CHUNKS % NT == 0 || q < A_CHUNKS) {
        const int r = q / CPR, ch = q % CPR;
        int m = m0 + r;
        m = m < M ? m : M - 1;
        ra[set][i] = !ALIGNED ? load_chunk_anywhere<DT>(A, m, lda, k0 + ch * T::kChunk, K)
                     : CLAMPED ? load_chunk_clamped<DT>(A, m, lda, k0 + ch * T::kChunk, K)
                            : load_chunk_aligned<DT>(A, m, lda, k0 + ch * T::kChunk, K);
      }
    }
#pragma unroll
    for (int i = 0; i < W_PER; ++i) {
      const int q = tid + i * NT;
      if (W_CHUNKS % NT == 0 || q < W_CHUNKS) {
        const int r = q / CPR, ch = q % CPR;
        int n = n0 + r;
        n = n < N ? n : N - 1;
        rw[set][i] = !ALIGNED ? load_chunk_anywhere<DT>(W, n, ldw, k0 + ch * T::kChunk, K)
                     : CLAMPED ? load_chunk_clamped<DT>(W, n, ldw, k0 + ch * T::kChunk, K)
                            : load_chunk_aligned<DT>(W, n, ldw, k0 + ch * T::kChunk, K);
      }
    }
  };
  // registers -> LDS (chunks beyond K already arrived as zeros, except from the clamped loaders)
  auto masked = [&](uint4 v, int k, bool inside) {
    if (!ALIGNED && !inside) return shift_chunk<DT>(v, k - min(k, K - T::kChunk));
    if (ALIGNED && CLAMPED) {
      const uint32_t keep = k < K ? 0xffffffffu : 0u;
      v.x &= keep;
      v.y &= keep;
      v.z &= keep;
      v.w &= keep;
    }
    return v;
  };
  auto lstore = [&](int set, int buf, int k0) {
    const bool inside = k0 + BK <= K;
#pragma unroll
    for (int i = 0; i < A_PER; ++i) {
      const int q = tid + i * NT;
      if (A_CHUNKS % NT == 0 || q < A_CHUNKS)
        *(uint4*)&lds[buf][(q / CPR) * PITCH + (q % CPR) * 16] = masked(ra[set][i], k0 + (q % CPR) * T::kChunk, inside);
    }
#pragma unroll
    for (int i = 0; i < W_PER; ++i) {
      const int q = tid + i * NT;
      if (W_CHUNKS % NT == 0 || q < W_CHUNKS)
        *(uint4*)&lds[buf][(BM + q / CPR) * PITCH + (q % CPR) * 16] = masked(rw[set][i], k0 + (q % CPR) * T::kChunk, inside);
    }
  };

  const HeadBias<HEAD == 0 ? 1 : HEAD> hbias(head);  // (without a head its bias is null)
  if constexpr (HEAD != 0) {
    const int present = N * ES / 16;  // chunks of a weight row that exist (N is a whole number of chunks)
#pragma unroll
    for (int i = 0; i < HW_PER; ++i) {
      const int q = tid + i * NT;
      const int j = q / (HW_ROW / 16), ch = q % (HW_ROW / 16);
      rhw[i] = make_uint4(0, 0, 0, 0);
      if (q < HW_CHUNKS && j < head.n && ch < present) rhw[i] = *(const uint4*)(head.w + (int64_t)j * head.ldw * ES + ch * 16);
    }
  }

  // with a single 32x32 block per wave, back-to-back MFMAs into one accumulator would each wait for the
  // previous result; alternate K steps between KACC accumulators and add them at the end
  floatx16 acc[KACC][TM][TN];
#pragma unroll
  for (int a = 0; a < KACC; ++a)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[a][i][j][r] = 0.f;

  // per-column epilogue parameters, requested before anything else so their latency hides under the K loop; nothing
  // is computed from them before the epilogue (an instruction on a loaded value here is a wait for memory here)
  float cbias[TN], cp0[TN], cp1[TN], cp2[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    int n = n0 + wn * WTN + j * 32 + (lane & 31);
    n = n < N ? n : N - 1;
    cbias[j] = ep.bias_rows == 1 ? ep.bias[n] : 0.f;
    cp0[j] = cp1[j] = cp2[j] = 0.f;
    if (ep.act == BZ_ACT_PRELU) cp0[j] = ep.p0[ep.act_size == 1 ? 0 : n];
    if (ep.act == BZ_ACT_DICE) {
      cp0[j] = ep.p0[n];
      cp1[j] = ep.p1[n];
      cp2[j] = ep.p2[n];
    }
  }

  // The K loop runs over KT rounded up to a multiple of D with no conditionals inside: tiles beyond K are
  // loaded from a clamped address and zeroed by the mask, so they add nothing.  Straight-line code lets the
  // compiler count outstanding loads exactly (s_waitcnt vmcnt(n) waits for the oldest set only).
  const int KT = (K + BK - 1) / BK;
  const int KTR = (KT + D - 1) / D * D;
#pragma unroll
  for (int d = 0; d < D; ++d) gload(d, d * BK);
  lstore(0, 0, 0);
  __syncthreads();
  const int frag_row = lane & 31, frag_half = lane >> 5;
  // Tiles are bound by how well LDS traffic hides behind the MFMAs, and a barrier lines all waves up in the same
  // phase: a burst of fragment reads right after it (matrix pipes idle), a burst of tile stores right before it.  PIPE
  // reorders a K tile: the next tile goes to the other LDS buffer first (its registers arrived long ago), fragments
  // are read one sub-step ahead of the MFMAs that use them, and the barrier sits before the last sub-step's MFMAs,
  // which then cover the read of the next tile's first fragments.
  // (not the 256x256 tile: with 128 accumulator registers a wave has no room for a second set of fragments; measured on
  // the other tiles: 128x256 245 -> 238 us on 8192x12800x1024, 64x64 9.6 -> 9.2 us on config 2's first layer)
  constexpr bool PIPE = !HEAD && BM * BN >= 64 * 64 && BM * BN < 256 * 256;
  constexpr int KS = BK / T::kStepK;  // sub-steps of a K tile
  if constexpr (PIPE) {
    static_assert(KS % 2 == 0, "fragment double buffer needs an even number of sub-steps");
    uint4 fa[2][TM], fw[2][TN];
    auto fread = [&](int slot, int buf, int ks) {
      const char* la = &lds[buf][(wm * WTM + frag_row) * PITCH + frag_half * 16];
      const char* lw = &lds[buf][(BM + wn * WTN + frag_row) * PITCH + frag_half * 16];
#pragma unroll
      for (int i = 0; i < TM; ++i) fa[slot][i] = *(const uint4*)(la + i * 32 * PITCH + ks * 32);
#pragma unroll
      for (int j = 0; j < TN; ++j) fw[slot][j] = *(const uint4*)(lw + j * 32 * PITCH + ks * 32);
    };
    auto fmma = [&](int slot, int ks) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) T::mma(fa[slot][i], fw[slot][j], acc[ks % KACC][i][j]);
    };
    fread(0, 0, 0);
    for (int kt0 = 0; kt0 < KTR; kt0 += D) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        const int kt = kt0 + d;
        const int buf = kt & 1;
        gload(d, (kt + D) * BK);  // set d held tile kt, which already sits in LDS
        // the other buffer was last read before the previous barrier: tile kt+1 can go there now
        lstore((d + 1) % D, buf ^ 1, (kt + 1) * BK);
#pragma unroll
        for (int ks = 0; ks + 1 < KS; ++ks) {
          fread((ks + 1) & 1, buf, ks + 1);
          fmma(ks & 1, ks);
        }
        __syncthreads();           // tile kt+1 is complete; every read of this buffer has returned
        fread(0, buf ^ 1, 0);      // KS is even: the next tile's first fragments take slot 0 again
        fmma((KS - 1) & 1, KS - 1);
      }
    }
    __syncthreads();  // the fragments read ahead for a tile that does not exist are dropped; LDS is free for the epilogue
  } else {
  for (int kt0 = 0; kt0 < KTR; kt0 += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int kt = kt0 + d;
      const int buf = kt & 1;
      gload(d, (kt + D) * BK);  // set d held tile kt, which already sits in LDS
      const char* la = &lds[buf][(wm * WTM + frag_row) * PITCH + frag_half * 16];
      const char* lw = &lds[buf][(BM + wn * WTN + frag_row) * PITCH + frag_half * 16];
#pragma unroll
      for (int ks = 0; ks < BK / T::kStepK; ++ks) {
        uint4 fa[TM], fw[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) fa[i] = *(const uint4*)(la + i * 32 * PITCH + ks * 32);
#pragma unroll
        for (int j = 0; j < TN; ++j) fw[j] = *(const uint4*)(lw + j * 32 * PITCH + ks * 32);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) T::mma(fa[i], fw[j], acc[ks % KACC][i][j]);
      }
      lstore((d + 1) % D, buf ^ 1, (kt + 1) * BK);
      __syncthreads();
    }
  }
  }

#pragma unroll
  for (int a = 1; a < KACC; ++a)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[0][i][j][r] += acc[a][i][j][r];
  // epilogue: lane owns column n, rows 8*(r/4) + 4*(lane/32) + r%4 of each 32x32 block.  The activated tile
  // goes through LDS (free after the K loop) so that global stores are 16 bytes per lane along rows.
  constexpr int OS = (int)sizeof(OutT);
  constexpr int OPITCH = BN * OS + 16;
  static_assert(BM * OPITCH <= (int)sizeof(lds), "output tile must fit the operand buffers");
  char* lout = &lds[0][0];
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    cbias[j] *= ep.beta;
    if (ep.act == BZ_ACT_DICE) cp2[j] = dice_inv_den(ep, cp2[j]);
  }
  // A bias of one row per sample, the rare form, is folded into the accumulators first, so that the element loop below
  // has no index to compute and nothing to decide per element.
  // (The 256x256 tile has no registers to spare for it and is not chosen for such a layer.)
  float alpha_e = ep.alpha;
  if (BM * BN < 256 * 256 && ep.bias_rows > 1) {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int n = n0 + wn * WTN + j * 32 + (lane & 31);
#pragma unroll
      for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int m = m0 + wm * WTM + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
          const float b = (m < M && n < N) ? ep.beta * ep.bias[full_bias_index(ep, m, n, M, N)] : 0.f;
          acc[0][i][j][r] = fmaf(ep.alpha, acc[0][i][j][r], b);
        }
      }
    }
    alpha_e = 1.f;
  }
  // The activation is a compile-time parameter of the element loop: a run-time switch per element would turn the
  // unrolled epilogue into a string of taken branches over far more code than the loop needs.  Every output goes
  // into the LDS tile, rows and columns beyond the matrix included (they are not copied out): a bounds check and a
  // 64-bit address per element cost several times the activation.
  auto epilogue = [&](auto act_c) {
    constexpr int ACT = decltype(act_c)::value;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int nl = wn * WTN + j * 32 + (lane & 31);
#pragma unroll
      for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int ml = wm * WTM + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
          float v = fmaf(alpha_e, acc[0][i][j][r], cbias[j]);  // (cbias: beta * bias of the column, or 0)
          v = apply_act_t<ACT>(v, ep, cp0[j], cp1[j], cp2[j]);
          store_out<OutT>((OutT*)(lout + ml * OPITCH) + nl, v);
        }
      }
    }
  };
  switch (ep.act) {
    case BZ_ACT_PRELU:
      epilogue(std::integral_constant<int, BZ_ACT_PRELU>());
      break;
    case BZ_ACT_DICE:
      epilogue(std::integral_constant<int, BZ_ACT_DICE>());
      break;
    case BZ_ACT_LEAKY_RELU:
      epilogue(std::integral_constant<int, BZ_ACT_LEAKY_RELU>());
      break;
    case BZ_ACT_SIGMOID:
      epilogue(std::integral_constant<int, BZ_ACT_SIGMOID>());
      break;
    default:
      epilogue(std::integral_constant<int, BZ_ACT_NONE>());
      break;
  }
  if constexpr (HEAD != 0) {
#pragma unroll
    for (int i = 0; i < HW_PER; ++i) {
      const int q = tid + i * NT;
      if (q < HW_CHUNKS) *(uint4*)&lds_hw[q * 16] = rhw[i];
    }
  }
  __syncthreads();
  if (vec_y) {
    constexpr int OCPR = BN * OS / 16;  // 16-byte chunks per tile row
    for (int q = tid; q < BM * OCPR; q += NT) {
      const int ml = q / OCPR, ch = q % OCPR;
      const int m = m0 + ml, n = n0 + ch * (16 / OS);
      if (m < M && n < N) *(uint4*)((char*)(Y + out_index(ep, m, n, ldy))) = *(const uint4*)(lout + ml * OPITCH + ch * 16);
    }
  } else if (Y != nullptr) {  // an output that takes no 16-byte stores: element by element, along rows
    for (int q = tid; q < BM * BN; q += NT) {
      const int ml = q / BN, nl = q % BN;
      if (m0 + ml < M && n0 + nl < N) Y[out_index(ep, m0 + ml, n0 + nl, ldy)] = ((const OutT*)(lout + ml * OPITCH))[nl];
    }
  }
  if constexpr (HEAD != 0) {
    // z[m, j] = head_act(sum_n y[m, n] * w2[j, n] + b2[j]) from the rounded tile, as the separate skinny launch
    // computes it from the stored tensor.  NT / BM lanes share a row; this workgroup owns whole rows (n0 == 0).
    static_assert(OS == ES, "the head reads the tile with the operand type");
    constexpr int LPRH = NT / BM;
    constexpr int CH = In<DT>::kChunk;
    const int r = tid / LPRH, hl = tid % LPRH;
    const int m = m0 + r;
    const int nch = N / CH;
    float hacc[HEAD];
#pragma unroll
    for (int j = 0; j < HEAD; ++j) hacc[j] = 0.f;
    for (int ch = hl; ch < nch; ch += LPRH) {
      float a[CH];
      chunk_to_float<DT>(*(const uint4*)(lout + r * OPITCH + ch * 16), a);
#pragma unroll
      for (int j = 0; j < HEAD; ++j) {
        if (j < head.n) {
          float w[CH];
          chunk_to_float<DT>(*(const uint4*)(lds_hw + j * HW_ROW + ch * 16), w);
#pragma unroll
          for (int i = 0; i < CH; ++i) hacc[j] = fmaf(a[i], w[i], hacc[j]);
        }
      }
    }
#pragma unroll
    for (int j = 0; j < HEAD; ++j) hacc[j] = group_sum<LPRH>(hacc[j]);
    if (hl == 0 && m < M) head_finish(head, hbias, m, hacc);
  }
}


// ---------------------------------------------------------------------------------------------
// streaming kernel: large layers (a 256x128 tile per CU fills the chip, K deep)
// ---------------------------------------------------------------------------------------------
// At this size the limit is how fast operands reach a CU, not latency: a 256x128x64 step is 1024 MFMA cycles per SIMD
// and 48 KB of operands, which the path from L2 into a CU (64 bytes a clock) needs 768 cycles for.  So the tile is the
// largest one that still gives every CU a workgroup with one wave per SIMD multiplying (128x64 per wave, 128 accumulator
// registers), and nothing else may stand in the loads' way:
//  - operands go from global memory straight into LDS (global_load_lds_dwordx4: no registers, no LDS store
//    instructions), three stages of 48 KB, two tiles in flight;
//  - four more waves, one per SIMD, do nothing but issue those loads and wait for them; the multiplying waves issue
//    only LDS reads and MFMAs and meet the loaders at one barrier per K tile (the same wave doing both measured 237 us
//    on 8192 x 12800 -> 1024 bf16, this split 203 us);
//  - a tile row is 128 bytes, half of the 64 banks; chunk c of row r is stored at position c ^ ((r >> 1) & 7), so the
//    16 lanes of a ds_read_b128 phase (16 rows, one logical chunk) hit 16 different bank groups (203 -> 195 us: with
//    the 32-bank pattern c ^ (r & 7) every other cycle of the LDS was a conflict);
//  - the scheduler is told to alternate MFMA and fragment read, and not to move either across a phase (195 -> 192 us).
constexpr int kStreamBM = 256, kStreamBN = 128, kStreamBK = 64, kStreamStages = 3;
constexpr int kStreamRowB = kStreamBK * 2;
constexpr int kStreamStageBytes = (kStreamBM + kStreamBN) * kStreamRowB;  // 49152
constexpr int kStreamLds = kStreamStages * kStreamStageBytes;            // 147456 of the CU's 160 KB
constexpr int kStreamCompute = 256;                                       // threads that multiply; as many again load

typedef __attribute__((address_space(3))) char lds_char;

// 16 bytes per lane from global memory to LDS at lds_addr + 16 * lane (lds_addr is the same in all lanes).  A scalar write of M0
// needs a wait state before a load to LDS reads it; the compiler puts one between its own instructions, in an asm's text nobody does.
__device__ __forceinline__ void load_to_lds(const char* g, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "s"(lds_addr) : "memory", "m0");
}

// one phase = 6 fragment reads for the phase after next and 8 MFMAs on fragments read a phase ago
#define BZ_PIN_PHASE()                                     \
  do {                                                     \
    _Pragma("unroll") for (int q_ = 0; q_ < 6; ++q_) {     \
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   \
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   \
    }                                                      \
    __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);     \
    __builtin_amdgcn_sched_barrier(0);                     \
  } while (0)

template <int DT, typename OutT>
__global__ __launch_bounds__(2 * kStreamCompute, 1) void bz_fc_stream_kernel(const char* __restrict__ A,
                                                                              const char* __restrict__ W, OutT* __restrict__ Y,
                                                                              int M, int N, int K, int64_t lda, int64_t ldw,
                                                                              int64_t ldy, int tiles_m, int tiles_n, Epilogue ep) {
  using T = In<DT>;
  static_assert(T::kSize == 2 && sizeof(OutT) == 2, "2-byte operands and outputs");
  constexpr int BM = kStreamBM, BN = kStreamBN, ROWB = kStreamRowB, STAGES = kStreamStages, NT = kStreamCompute;
  constexpr int STAGE_BYTES = kStreamStageBytes;
  constexpr int LOADS = (BM + BN) * (ROWB / 16) / NT;  // 12 chunks per loader thread per stage
  constexpr int TM = 4, TN = 2;                        // 32x32 blocks per wave tile (128 x 64)
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const bool loader = threadIdx.x >= NT;
  const int tid = threadIdx.x & (NT - 1), lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  // The 8 XCDs take turns at consecutive workgroup ids.  XCD x walks its own band of M tiles, the N tiles of an M tile
  // next to each other in time: an A tile is fetched into that XCD's L2 once, the W panel streams through it.
  const int xcd = blockIdx.x & 7, j = blockIdx.x >> 3;
  const int per_xcd = (tiles_m + 7) / 8;
  const int tile_m = xcd * per_xcd + j / tiles_n, tile_n = j % tiles_n;
  if (tile_m >= tiles_m) return;
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_char*)smem;
  const int KT = K / kStreamBK;

  if (loader) {
    // chunk p = i*256 + tid of a stage: row p >> 3 (A rows, then W rows), position p & 7
    const char* src[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int p = i * NT + tid;
      const int r = p >> 3, c = (p & 7) ^ ((r >> 1) & 7);
      if (r < BM) {
        int m = m0 + r;
        m = m < M ? m : M - 1;
        src[i] = A + ((int64_t)m * lda) * 2 + c * 16;
      } else {
        int n = n0 + (r - BM);
        n = n < N ? n : N - 1;
        src[i] = W + ((int64_t)n * ldw) * 2 + c * 16;
      }
    }
    auto issue = [&](int kt) {
      const uint32_t base = __builtin_amdgcn_readfirstlane(lds0 + (kt % STAGES) * STAGE_BYTES + wave * 1024);
      const int64_t koff = (int64_t)kt * ROWB;
#pragma unroll
      for (int i = 0; i < LOADS; ++i) load_to_lds(src[i] + koff, base + i * (NT * 16));
    };
    // Barrier kt (counted from 0) says: tile kt has landed, and nobody reads the stage tile kt+2 goes to any more.
    // The waits are written out because only this code knows how many loads may stay in flight.
    issue(0);
    if (KT > 1) issue(1);
    if (KT > 1)
      asm volatile("s_waitcnt vmcnt(12)\n\ts_barrier" ::: "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    for (int kt = 0; kt < KT; ++kt) {
      if (kt + 2 < KT) {
        issue(kt + 2);
        asm volatile("s_waitcnt vmcnt(12)\n\ts_barrier" ::: "memory");
      } else {
        asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
      }
    }
    __syncthreads();  // the two barriers of the epilogue
    __syncthreads();
    return;
  }

  // per-column epilogue parameters, requested before the K loop
  float cbias[TN], cp0[TN], cp1[TN], cp2[TN];
#pragma unroll
  for (int jn = 0; jn < TN; ++jn) {
    int n = n0 + wn * 64 + jn * 32 + (lane & 31);
    n = n < N ? n : N - 1;
    cbias[jn] = ep.bias_rows == 1 ? ep.bias[n] : 0.f;
    cp0[jn] = cp1[jn] = cp2[jn] = 0.f;
    if (ep.act == BZ_ACT_PRELU) cp0[jn] = ep.p0[ep.act_size == 1 ? 0 : n];
    if (ep.act == BZ_ACT_DICE) {
      cp0[jn] = ep.p0[n];
      cp1[jn] = ep.p1[n];
      cp2[jn] = ep.p2[n];  // (finished in the epilogue: an instruction on a loaded value here is a wait for memory here)
    }
  }

  floatx16 acc[TM][TN];
#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int b = 0; b < TN; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.f;

  // lane (row = lane & 31, half = lane >> 5) reads logical chunk 2*ks + half of its row
  const int frow = lane & 31, fhalf = lane >> 5;
  int foff[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) foff[ks] = frow * ROWB + (((2 * ks + fhalf) ^ ((frow >> 1) & 7)) << 4);
  const int a_base = (wm * 128) * ROWB, w_base = (BM + wn * 64) * ROWB;
  uint4 fa[2][TM], fw[2][TN];
  auto fread = [&](int slot, int stage, int ks) {
    const char* s = smem + stage * STAGE_BYTES + foff[ks];
#pragma unroll
    for (int i = 0; i < TM; ++i) fa[slot][i] = *(const uint4*)(s + a_base + i * 32 * ROWB);
#pragma unroll
    for (int jn = 0; jn < TN; ++jn) fw[slot][jn] = *(const uint4*)(s + w_base + jn * 32 * ROWB);
  };
  auto fmma = [&](int slot) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int jn = 0; jn < TN; ++jn) T::mma(fa[slot][i], fw[slot][jn], acc[i][jn]);
  };

  asm volatile("s_barrier" ::: "memory");  // tile 0 landed
  fread(0, 0, 0);
  for (int kt = 0; kt < KT; ++kt) {
    const int stage = kt % STAGES;
    fread(1, stage, 1);
    fmma(0);
    BZ_PIN_PHASE();
    fread(0, stage, 2);
    fmma(1);
    BZ_PIN_PHASE();
    fread(1, stage, 3);
    fmma(0);
    BZ_PIN_PHASE();
    // every read of this stage has returned (the last were issued 8 MFMAs ago); past the barrier tile kt+1 is complete
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (kt + 1 < KT) fread(0, (kt + 1) % STAGES, 0);
    fmma(1);
    BZ_PIN_PHASE();
  }

  // epilogue: lane owns column n of each 32x32 block, rows 8*(r/4) + 4*(lane/32) + r%4; the activated tile goes through
  // LDS so that global stores are 16 bytes per lane along rows
  __syncthreads();
#pragma unroll
  for (int jn = 0; jn < TN; ++jn) {
    cbias[jn] *= ep.beta;
    if (ep.act == BZ_ACT_DICE) cp2[jn] = dice_inv_den(ep, cp2[jn]);
  }
  constexpr int OPITCH = BN * 2 + 16;
  char* lout = smem;
  auto epilogue = [&](auto act_c) {
    constexpr int ACT = decltype(act_c)::value;
#pragma unroll
    for (int jn = 0; jn < TN; ++jn) {
      const int nl = wn * 64 + jn * 32 + (lane & 31);
#pragma unroll
      for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int ml = wm * 128 + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
          float v = fmaf(ep.alpha, acc[i][jn][r], cbias[jn]);  // (cbias: beta * bias of the column, or 0)
          v = apply_act_t<ACT>(v, ep, cp0[jn], cp1[jn], cp2[jn]);
          store_out<OutT>((OutT*)(lout + ml * OPITCH) + nl, v);
        }
      }
    }
  };
  switch (ep.act) {
    case BZ_ACT_PRELU:
      epilogue(std::integral_constant<int, BZ_ACT_PRELU>());
      break;
    case BZ_ACT_DICE:
      epilogue(std::integral_constant<int, BZ_ACT_DICE>());
      break;
    case BZ_ACT_LEAKY_RELU:
      epilogue(std::integral_constant<int, BZ_ACT_LEAKY_RELU>());
      break;
    case BZ_ACT_SIGMOID:
      epilogue(std::integral_constant<int, BZ_ACT_SIGMOID>());
      break;
    default:
      epilogue(std::integral_constant<int, BZ_ACT_NONE>());
      break;
  }
  __syncthreads();
  constexpr int OCPR = BN * 2 / 16;
  for (int q = tid; q < BM * OCPR; q += NT) {
    const int ml = q / OCPR, ch = q % OCPR;
    const int m = m0 + ml, n = n0 + ch * 8;
    if (m < M && n < N) *(uint4*)((char*)(Y + out_index(ep, m, n, ldy))) = *(const uint4*)(lout + ml * OPITCH + ch * 16);
  }
}
#undef BZ_PIN_PHASE

// ---------------------------------------------------------------------------------------------
// split kernel: few tiles
// ---------------------------------------------------------------------------------------------
// A workgroup owns a 32 x 32 tile of C and its eight or four waves (NW) share the K range: unit u (128 bytes of every row)
// is wave u % NW's.  A wave works for itself: it loads a unit with eight lanes on a row, turns it in LDS of its own into MFMA
// fragments, the next unit's loads in flight meanwhile, and meets the others only when the partial tiles are added up.
//  - Few tiles leave the chip idle and the chain of K tiles sets the time: eight waves walk it in an eighth of the steps.
//  - A lane's 16 bytes may start anywhere (a row pitch of 445 fp16 elements): the memory system takes such loads, and
//    the lines they share are L1 hits.  So rows that start on no 16 bytes need no path of their own here.
// Loaded straight into fragments a group of 16 lanes touches 16 lines, and the path into the CU takes a line a clock:
// 128 x 4096 -> 1024 fp16 18.7 us, 9.1 this way (21.9 on the staged tile).
constexpr int kSplitUnit = 128;
// Where chunk `chunk` of row `row` lies.  2-byte operands: rows 16 bytes further apart than they are long, so that a fragment
// read's sixteen lanes (one chunk of sixteen rows) are on all banks.  fp32, which moves twice the bytes for as many products:
// rows side by side, their chunks in an order of the row's own, so that a write's (two rows) are as well (2048 x 512 -> 256 with a
// head in its launch 18.1 us, 17.2 this way; fp16 1024 x 896 -> 512 5.8 and 5.9).
template <int DT>
constexpr int kSplitPitch = DT == BZ_F32 ? kSplitUnit : kSplitUnit + 16;
template <int DT>
__device__ __forceinline__ int split_at(int row, int chunk) {
  return row * kSplitPitch<DT> + (DT == BZ_F32 ? (chunk ^ (row >> 1)) & 7 : chunk) * 16;
}

// One wave's 8 * P rows of an operand, a unit of K at a time: global memory -> registers (lane: row l / 8 of each pass,
// chunk l % 8) -> LDS as split_at has it.
// CHUNKS: K is a whole number of chunks (a layer with a head's is)
template <int DT, int P, bool CHUNKS = false>
struct SplitRows {
  static constexpr int ES = In<DT>::kSize, CH = In<DT>::kChunk;
  const char* p[P];
  uint4 r[P];
  bool part = false;  // the unit is the one that K ends in: `back` elements in front of what is wanted were loaded with it (as in shift_chunk)
  int back = 0;
  __device__ __forceinline__ void init(const char* base, int64_t ld, int row0, int rows, int lane) {
#pragma unroll
    for (int i = 0; i < P; ++i) p[i] = base + (int64_t)min(row0 + i * 8 + (lane >> 3), rows - 1) * ld * ES;
  }
  // a whole unit
  __device__ __forceinline__ void load(int u, int lane) {
    part = false;
#pragma unroll
    for (int i = 0; i < P; ++i) __builtin_memcpy(&r[i], p[i] + (int64_t)u * kSplitUnit + (lane & 7) * 16, 16);
  }
  // The unit that K ends in, zeros beyond K.  (Ragged rows are shifted when they are stored: where they are loaded, each was a trip of its
  // own, eight for the wave whose unit it is.  300 x 445 -> 256 fp16 4.9 -> 4.3 us, one row 4.2 -> 3.6, 2000 x 901 -> 128 7.2 -> 6.4.)
  __device__ __forceinline__ void load_last(int u, int K, int lane) {
    const int k = u * (kSplitUnit / ES) + (lane & 7) * CH;
    if constexpr (CHUNKS) {
      const uint32_t have = k < K ? 0xffffffffu : 0u;
#pragma unroll
      for (int i = 0; i < P; ++i) __builtin_memcpy(&r[i], p[i] + (int64_t)min(k, K - CH) * ES, 16);
#pragma unroll
      for (int i = 0; i < P; ++i) r[i] = make_uint4(r[i].x & have, r[i].y & have, r[i].z & have, r[i].w & have);
      return;
    }
    part = K >= CH;
    if (part) {
      const int at = min(k, K - CH);
      back = k - at;
#pragma unroll
      for (int i = 0; i < P; ++i) __builtin_memcpy(&r[i], p[i] + (int64_t)at * ES, 16);
    } else {
#pragma unroll
      for (int i = 0; i < P; ++i) r[i] = load_chunk<DT>(p[i], 0, 0, k, K);
    }
  }
  __device__ __forceinline__ void store(char* lds, int lane) const {
    uint4 v[P];
#pragma unroll
    for (int i = 0; i < P; ++i) v[i] = r[i];
    if (!CHUNKS && part) {
#pragma unroll
      for (int i = 0; i < P; ++i) v[i] = shift_chunk<DT>(r[i], back);
    }
#pragma unroll
    for (int i = 0; i < P; ++i) *(uint4*)(lds + split_at<DT>(i * 8 + (lane >> 3), lane & 7)) = v[i];
  }
};

template <int DT, typename OutT, int NW, bool CHUNKS>
__global__ __launch_bounds__(NW * 64, 4) void bz_fc_split_kernel(const char* __restrict__ A, const char* __restrict__ W,
                                                                 int M, int N, int K, int tiles_m, int64_t lda, int64_t ldw,
                                                                 OutT* __restrict__ Y, int64_t ldy, Epilogue ep) {
  using T = In<DT>;
  constexpr int STEPS = kSplitUnit / 32;  // a step: 16 bytes of K in each half of the lanes
  constexpr int PITCH = 33;
  __shared__ __attribute__((aligned(16))) char lds[NW][64 * kSplitPitch<DT>];
  static_assert(32 * PITCH * 4 <= 64 * kSplitPitch<DT>, "a partial tile fits where its wave's operands were");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m0 = (int)(blockIdx.x % tiles_m) * 32, n0 = (int)(blockIdx.x / tiles_m) * 32;
  const int frow = lane & 31, fhalf = lane >> 5;
  char* la = lds[wave];
  char* lw = la + 32 * kSplitPitch<DT>;
  SplitRows<DT, 4, CHUNKS> ra, rw;
  ra.init(A, lda, m0, M, lane);
  rw.init(W, ldw, n0, N, lane);
  floatx16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  const int whole = (int)((int64_t)K * T::kSize / kSplitUnit), units = (int)(((int64_t)K * T::kSize + kSplitUnit - 1) / kSplitUnit);
  auto load = [&](int u) {
    if (u < whole) {
      ra.load(u, lane);
      rw.load(u, lane);
    } else if (u < units) {
      ra.load_last(u, K, lane);
      rw.load_last(u, K, lane);
    }
  };
  load(wave);
  // the parameters of the column that this thread finishes: asked for now, looked at at the end.  (Behind the operands, whose addresses come
  // with the wave: the parameters' are still on their way.)
  float cbias = 0.f, cp0 = 0.f, cp1 = 0.f, cp2 = 0.f;
  {
    const int c = min(n0 + tid % 32, N - 1);
    if (ep.bias_rows == 1) cbias = ep.bias[c];
    if (ep.act == BZ_ACT_PRELU) cp0 = ep.p0[ep.act_size == 1 ? 0 : c];
    if (ep.act == BZ_ACT_DICE) {
      cp0 = ep.p0[c];
      cp1 = ep.p1[c];
      cp2 = ep.p2[c];
    }
  }
  for (int u = wave; u < units; u += NW) {
    // (a wave's own LDS operations keep their order: nobody to wait for)
    ra.store(la, lane);
    rw.store(lw, lane);
    __builtin_amdgcn_wave_barrier();
    load(u + NW);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < STEPS; ++ks)
      T::mma(*(const uint4*)(la + split_at<DT>(frow, fhalf + ks * 2)), *(const uint4*)(lw + split_at<DT>(frow, fhalf + ks * 2)), acc);
    __builtin_amdgcn_wave_barrier();
  }
  // a lane owns column lane & 31 and rows 8 * (r / 4) + 4 * (lane / 32) + r % 4: the upper half of the waves leave theirs
  // where their operands were, the lower half add their own
  float* mine = (float*)lds[wave] + 4 * fhalf * PITCH + frow;
  if (wave >= NW / 2) {
#pragma unroll
    for (int r = 0; r < 16; ++r) mine[(8 * (r >> 2) + (r & 3)) * PITCH] = acc[r];
  }
  __syncthreads();
  if (wave < NW / 2) {
    const float* other = (const float*)lds[wave + NW / 2] + 4 * fhalf * PITCH + frow;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int at = (8 * (r >> 2) + (r & 3)) * PITCH;
      mine[at] = acc[r] + other[at];
    }
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < 32 * 32 / (NW * 64); ++e) {
    const int q = tid + e * NW * 64, ml = q / 32, nl = q % 32;
    const int m = m0 + ml, n = n0 + nl;
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < NW / 2; ++w) v += ((const float*)lds[w])[ml * PITCH + nl];
    if (m < M && n < N) {
      const float b = ep.bias_rows <= 1 ? cbias : ep.bias[full_bias_index(ep, m, n, M, N)];
      store_out<OutT>(Y + out_index(ep, m, n, ldy), apply_act_regs(fmaf(ep.alpha, v, ep.beta * b), ep, cp0, cp1, cp2));
    }
  }
}

// ---------------------------------------------------------------------------------------------
// fp32 layers on the bf16 matrix cores
// ---------------------------------------------------------------------------------------------
// A workgroup owns a tile of 32 * TM x 32 * TN outputs and its NW waves share K, 16 at a time (stage t is wave t % NW's), each
// working for itself: it loads a stage of the tile's rows straight into LDS of its own, reads fragments from there, splits them
// into three bf16s a float (Bf16x3) and multiplies those; the partial tiles meet once, at the end.
//  - The conversion, 11 vector instructions for two floats and one that keeps the largest of them, is what bounds it, not the products:
//    between 32-clock MFMAs the SIMD issues a vector instruction every five clocks, where 8 come to each MFMA of a 64x64 tile, and it does
//    so only if a wave's own instructions alternate (beside another wave's MFMAs a wave of vector instructions gets one in 18 clocks).  So a step
//    multiplies one stage, converts the next and reads the one after, and tells the scheduler to alternate (with all conversions
//    in front of the products, as they came, 2048 x 896 -> 512 took 17.5 us, with the read in front of them 16.2, this way 14.5).
//  - That takes two sets of pieces in registers, and none are left for loads in flight: they go to LDS without any.
//  - 2048 x 896 -> 512 by clocks, eight waves: 4 500 to the first stage, 15 000 for two waves' seven steps a SIMD (11 000 of MFMAs), 1 500
//    to add up, 3 000 to finish and store.
constexpr int kF32Stage = 16;                   // of K
constexpr int kF32RowB = kF32Stage * 4;         // bytes of a row of a stage
constexpr uint32_t kF32RowsWithin = 0x80000000u;  // bytes that a tile's rows lie within
inline bool f32_rows_fit(int64_t ld, int k) { return k >= 4 && (64 * ld + k) * 4 < (int64_t)kF32RowsWithin; }

// 16 bytes per lane from base + off to LDS at lds_addr + 16 * lane where `left`, as base and lds_addr the same in all lanes, is
// above 0.  (The branch stands in the assembler: one that the compiler sees ends the block in which it may alternate products
// and conversions.)
__device__ __forceinline__ void load_to_lds_from(const char* base, uint32_t off, uint32_t lds_addr, int left) {
  asm volatile("s_cmp_lt_i32 %3, 1\n\ts_cbranch_scc1 .Lnone%=\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1\n.Lnone%=:" ::"v"(off),
               "s"(base), "s"(lds_addr), "s"(left)
               : "memory", "m0", "scc");
}

// m = the largest of m, |x| and |y|.  (NaNs are passed over, and make their sums NaNs anyway.  In assembly, so that it stands where the
// products have ended: alternated with them, 2048 x 896 -> 512 took 0.8 us more.)
__device__ __forceinline__ void largest(float& m, float x, float y) { asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(m) : "v"(x), "v"(y)); }
// Whether a sum of K split products may be off, max_a and max_w being the largest |operands| of its two rows: it is not finite, or so
// small that what a split may drop of operands below 2^-110, at most 2^-126 of each, times the other row's largest counts in it.
// (What the matrix instructions may flush of the products, 2^-126 of each of the six, is less than that for 1.)
constexpr float kSplitDrops = 0x1p-98f;
__device__ __forceinline__ bool doubtful(float v, int K, float max_a, float max_w) {
  const float least = (float)K * kSplitDrops * fmaxf(1.f, fmaxf(max_a, max_w));
  const bool off = !(fabsf(v) >= least && fabsf(v) < __builtin_huge_valf());
  return off && !(v == 0.f && (max_a == 0.f || max_w == 0.f));
}
// Where no operand of a tile is beyond this, and no sum of it doubtful for this, nothing is: one look at the tile.  (Each sum by its own
// rows' largest operands, without it, made 2048 x 896 -> 512 16.9 us, the tile's at once 16.0; without any of this it was 15.8.)
constexpr float kOrdinary = 0x1p40f;

// EXACT: Dice as apply_act computes it, not as the tile kernels do
template <typename OutT, int NW, int TM, int TN, int SUMS, bool EXACT>
__global__ __launch_bounds__(NW * 64, 2) void bz_fc_f32_kernel(const char* __restrict__ A, const char* __restrict__ W, int M, int N, int K,
                                                            int tiles_m, int64_t lda, int64_t ldw, OutT* __restrict__ Y, int64_t ldy,
                                                            Epilogue ep) {
  constexpr int BM = 32 * TM, BN = 32 * TN, NT = NW * 64, ROWS = BM + BN;
  constexpr int LOADS = ROWS / 16;  // a load instruction brings 16 rows of a stage
  constexpr int SLOT = ROWS * kF32RowB;
  static_assert(BM * BN * 4 <= 2 * SLOT, "a partial tile fits where its wave's operands were");
  __shared__ __attribute__((aligned(16))) char lds[NW][2][SLOT];
  __shared__ float most[NW][2][ROWS];  // the largest |operand| of each row that a half of the wave saw
  __shared__ __attribute__((aligned(16))) uint32_t beyond[NW];  // whether any of them is beyond kOrdinary
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m0 = (int)(blockIdx.x % tiles_m) * BM, n0 = (int)(blockIdx.x / tiles_m) * BN;
  const int frow = lane & 31, fhalf = lane >> 5;
  // Row r of a stage lies at 64 * r, its chunk c at position c ^ ((r >> 2) & 3): sixteen lanes that read one chunk of sixteen rows
  // are on all banks.  Lane l of a load has position l % 4 of row l / 4 of its sixteen.
  const int lrow = lane >> 2, lchunk = (lane & 3) ^ (lane >> 4);
  const char* abase = A + (int64_t)m0 * lda * 4;
  const char* wbase = W + (int64_t)n0 * ldw * 4;
  uint32_t off[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    if (i * 16 < BM)
      off[i] = (uint32_t)min(i * 16 + lrow, M - 1 - m0) * (uint32_t)(lda * 4) + lchunk * 16;
    else
      off[i] = (uint32_t)min(i * 16 - BM + lrow, N - 1 - n0) * (uint32_t)(ldw * 4) + lchunk * 16;
  }
  const int stages = (K + kF32Stage - 1) / kF32Stage;
  const int n = wave < stages ? (stages - 1 - wave) / NW + 1 : 0;  // this wave's
  // The wave's stages in descending order, so that the one that K ends in comes first
  auto stage_at = [&](int i) { return wave + (n - 1 - i) * NW; };
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_char*)&lds[0][0][0] + wave * (2 * SLOT);
  auto issue = [&](int i) {
    const int64_t k = (int64_t)stage_at(i) * kF32RowB;
    const uint32_t to = __builtin_amdgcn_readfirstlane(lds0 + (i & 1) * SLOT);
#pragma unroll
    for (int q = 0; q < LOADS; ++q) load_to_lds_from((q * 16 < BM ? abase : wbase) + k, off[q], to + q * 1024, n - i);
  };
  // the same through registers, for a stage that reaches beyond K: zeros there
  auto issue_part = [&](int i) {
    const int k = stage_at(i) * kF32Stage + lchunk * 4, back = k - min(k, K - 4);
    uint4 r[LOADS];
#pragma unroll
    for (int q = 0; q < LOADS; ++q) __builtin_memcpy(&r[q], (q * 16 < BM ? abase : wbase) + (int64_t)(k - back) * 4 + (off[q] - lchunk * 16), 16);
#pragma unroll
    for (int q = 0; q < LOADS; ++q) *(uint4*)(&lds[wave][i & 1][q * 1024 + lane * 16]) = shift_chunk<BZ_F32>(r[q], back);
  };
  const bool part = n > 0 && (stage_at(0) + 1) * kF32Stage > K;
  if (n > 0) {
    if (!part) issue(0);
    issue(1);
    if (part) issue_part(0);
  }
  // the parameters of the column that this thread finishes: asked for now, looked at at the end
  float cbias = 0.f, cp0 = 0.f, cp1 = 0.f, cp2 = 0.f;
  {
    const int c = min(n0 + tid % BN, N - 1);
    if (ep.bias_rows == 1) cbias = ep.bias[c];
    if (ep.act == BZ_ACT_PRELU) cp0 = ep.p0[ep.act_size == 1 ? 0 : c];
    if (ep.act == BZ_ACT_DICE) {
      cp0 = ep.p0[c];
      cp1 = ep.p1[c];
      cp2 = ep.p2[c];
    }
  }
  // (the sums that an output is added up in, stage by stage in turn)
  floatx16 acc[SUMS][TM][TN];
#pragma unroll
  for (int a = 0; a < SUMS; ++a)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[a][i][j][r] = 0.f;

  struct Pieces {
    Bf16x3 a[TM], w[TN];
  };
  struct Raw {
    uint4 a[TM][2], w[TN][2];
  };
  // chunks h and h + 2 of its row are the lane's in half h
  auto read = [&](int i, Raw& raw) {
    const char* from = &lds[wave][i & 1][0] + frow * kF32RowB;
    const int p0 = (fhalf ^ ((frow >> 2) & 3)) * 16, p1 = p0 ^ 32;
#pragma unroll
    for (int b = 0; b < TM; ++b) {
      raw.a[b][0] = *(const uint4*)(from + b * 32 * kF32RowB + p0);
      raw.a[b][1] = *(const uint4*)(from + b * 32 * kF32RowB + p1);
    }
#pragma unroll
    for (int b = 0; b < TN; ++b) {
      raw.w[b][0] = *(const uint4*)(from + (BM + b * 32) * kF32RowB + p0);
      raw.w[b][1] = *(const uint4*)(from + (BM + b * 32) * kF32RowB + p1);
    }
  };
  // (the largest operands so far of the rows whose fragments the lane has)
  float max_a[TM], max_w[TN];
#pragma unroll
  for (int b = 0; b < TM; ++b) max_a[b] = 0.f;
#pragma unroll
  for (int b = 0; b < TN; ++b) max_w[b] = 0.f;
  auto split = [&](const uint4 (&raw)[2], float& most) {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      largest(most, __uint_as_float(raw[c].x), __uint_as_float(raw[c].y));
      largest(most, __uint_as_float(raw[c].z), __uint_as_float(raw[c].w));
    }
    return split_floats(raw[0], raw[1]);
  };
  auto convert = [&](const Raw& raw, Pieces& p) {
#pragma unroll
    for (int b = 0; b < TM; ++b) p.a[b] = split(raw.a[b], max_a[b]);
#pragma unroll
    for (int b = 0; b < TN; ++b) p.w[b] = split(raw.w[b], max_w[b]);
  };
  // the smallest products first
  auto multiply = [&](const Pieces& p, auto parity) {
    constexpr int SUM = decltype(parity)::value % SUMS;
    auto each = [&](auto f) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) f(p.a[i], p.w[j], acc[SUM][i][j]);
    };
    each([](const Bf16x3& x, const Bf16x3& y, floatx16& c) { In<BZ_BF16>::mma(x.lo, y.hi, c); });
    each([](const Bf16x3& x, const Bf16x3& y, floatx16& c) { In<BZ_BF16>::mma(x.hi, y.lo, c); });
    each([](const Bf16x3& x, const Bf16x3& y, floatx16& c) { In<BZ_BF16>::mma(x.mid, y.mid, c); });
    each([](const Bf16x3& x, const Bf16x3& y, floatx16& c) { In<BZ_BF16>::mma(x.mid, y.hi, c); });
    each([](const Bf16x3& x, const Bf16x3& y, floatx16& c) { In<BZ_BF16>::mma(x.hi, y.mid, c); });
    each([](const Bf16x3& x, const Bf16x3& y, floatx16& c) { In<BZ_BF16>::mma(x.hi, y.hi, c); });
  };
  // Stage i has landed where every load but the last stage's is waited for; the waits are written out because only this code
  // knows how many loads may stay in flight.
  auto landed = [&](int i) {
    asm volatile("s_cmp_gt_i32 %0, 1\n\ts_cbranch_scc1 .Lmore%=\n\ts_waitcnt vmcnt(0)\n.Lmore%=:\n\ts_waitcnt vmcnt(%1)" ::"s"(n - i), "n"(LOADS)
                 : "memory", "scc");
  };
  // the stage after next goes where stage i was, once every read of it has returned
  auto refill = [&](int i) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    issue(i + 2);
  };
  // multiplies stage i, converts stage i + 1, reads stage i + 2
  auto step = [&](const Pieces& now, Pieces& next, const Raw& raw, Raw& raw_next, int i, auto parity) {
    landed(i + 2);
    read(i + 2, raw_next);
    __builtin_amdgcn_sched_barrier(0);
    multiply(now, parity);
    convert(raw, next);
    constexpr int MFMAS = 6 * TM * TN, VALU = 88 * (TM + TN) / 2, EACH = VALU / MFMAS;
#pragma unroll
    for (int q = 0; q < MFMAS; ++q) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, EACH, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    refill(i + 2);
  };
  if (n > 0) {
    Pieces p0, p1;
    Raw r0, r1;
    landed(0);
    read(0, r0);
    refill(0);
    landed(1);
    read(1, r1);
    convert(r0, p0);
    refill(1);
    const std::integral_constant<int, 0> even;
    const std::integral_constant<int, 1> odd;
    int i = 0;
    for (; i + 2 < n; i += 2) {
      step(p0, p1, r1, r0, i, even);
      step(p1, p0, r0, r1, i + 1, odd);
    }
    if (i + 1 < n) {
      step(p0, p1, r1, r0, i, even);
      multiply(p1, odd);
    } else {
      multiply(p0, even);
    }
  }
  // A lane owns column lane & 31 of each block and rows 8 * (r / 4) + 4 * (lane / 32) + r % 4: four rows of a column are a chunk.  Every
  // wave leaves its partial tile where its operands were, column by column, the chunks of a column in an order of its own, so
  // that writes and reads are on all banks; then a thread adds up and finishes chunks of one column.
  constexpr int CHUNKS = BM / 4, EACH = (CHUNKS * BN + NT - 1) / NT;  // of a column; of a thread
  static_assert((BN == 64 || (BN == 32 && EACH == 1)) && EACH <= 4, "the rows of a wave's threads are sixteen or fewer");
  static_assert(NT % BN == 0 && (CHUNKS * BN % NT == 0 || EACH == 1) && (CHUNKS & (CHUNKS - 1)) == 0, "threads share the tile's chunks evenly");
  auto chunk_at = [&](int col, int chunk) { return (col * CHUNKS + (chunk ^ (col & (CHUNKS - 1)))) * 16; };
  const int col = tid % BN, nn = n0 + col;
  float v[EACH][4];
  auto add_up = [&]() {
#pragma unroll
    for (int a = 1; a < SUMS; ++a)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[0][i][j][r] += acc[a][i][j][r];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *(float4*)(&lds[wave][0][0] + chunk_at(j * 32 + frow, i * 8 + q * 2 + fhalf)) =
              make_float4(acc[0][i][j][4 * q], acc[0][i][j][4 * q + 1], acc[0][i][j][4 * q + 2], acc[0][i][j][4 * q + 3]);
    __syncthreads();
#pragma unroll
    for (int e = 0; e < EACH; ++e)
#pragma unroll
      for (int c = 0; c < 4; ++c) v[e][c] = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w)
#pragma unroll
      for (int e = 0; e < EACH; ++e) {
        const float4 p = *(const float4*)(&lds[w][0][0] + chunk_at(col, tid / BN + e * (NT / BN)));
        v[e][0] += p.x;
        v[e][1] += p.y;
        v[e][2] += p.z;
        v[e][3] += p.w;
      }
  };
  {
    float all = 0.f;
#pragma unroll
    for (int b = 0; b < TM + TN; ++b) {
      const float m = b < TM ? max_a[b < TM ? b : 0] : max_w[b < TM ? 0 : b - TM];
      most[wave][fhalf][b * 32 + frow] = m;
      all = fmaxf(all, m);
    }
    const uint64_t any = __builtin_amdgcn_ballot_w64(all > kOrdinary);
    if (lane == 0) beyond[wave] = any != 0;
  }
  add_up();
  if (tid / BN >= CHUNKS) return;  // (whole waves)
  // |v| from what is doubtful for kOrdinary up to infinity, as bits without the sign's
  uint32_t again = 0, worst = 0, large = 0;
  const uint32_t least = __float_as_uint((float)K * (kSplitDrops * kOrdinary)) << 1;
#pragma unroll
  for (int e = 0; e < EACH; ++e)
#pragma unroll
    for (int c = 0; c < 4; ++c) worst = max(worst, (__float_as_uint(v[e][c]) << 1) - least);
#pragma unroll
  for (int w = 0; w < NW; ++w) large |= beyond[w];
  if (__builtin_expect(large != 0 || worst >= 0xff000000u - least, 0)) {
    auto row_most = [&](int row) {
      float m = 0.f;
      for (int w = 0; w < NW; ++w) m = fmaxf(m, fmaxf(most[w][0][row], most[w][1][row]));
      return m;
    };
    const float max_w = row_most(BM + col);
#pragma unroll
    for (int e = 0; e < EACH; ++e)
#pragma unroll
      for (int c = 0; c < 4; ++c)
        again |= doubtful(v[e][c], K, row_most((tid / BN + e * (NT / BN)) * 4 + c), max_w) ? 1u << (e * 4 + c) : 0u;
  }
  if (__builtin_expect(__any(again != 0), 0)) {
    // The wave's rows times all columns once more, with fp32 instructions; of these products the doubtful ones are taken.  A row of sixteen
    // operands is four rows of chunk i / 4, in the order the wave's threads have them; an instruction's four inputs have a sum of their own.
    // (It waits for its operands, 64 inputs of all rows at a time.  2048 x 896 -> 512, 16.0 us without: a NaN in one row 42 us, in every 32nd 42,
    // in all 53; as dot products of the threads, a sum at a time, 42, 65 and 504.)
    const int i = lane & 15, q = i >> 2;
    const int chunk = BN == 64 ? wave + min(q, EACH - 1) * (NT / BN) : wave * 2 + (q & 1);
    const float* const a = (const float*)A + min(m0 + chunk * 4 + (i & 3), M - 1) * lda;
    const float* w[BN / 16];
    floatx4 sums[BN / 16][4];
#pragma unroll
    for (int b = 0; b < BN / 16; ++b) {
      w[b] = (const float*)W + min(n0 + b * 16 + i, N - 1) * ldw;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) sums[b][t][r] = 0.f;
    }
    constexpr int kAhead = 4;  // steps of sixteen inputs asked for together
    for (int k0 = 0; k0 < K; k0 += 16 * kAhead) {
      uint4 x[kAhead], y[kAhead][BN / 16];
      int beyond_k[kAhead];
#pragma unroll
      for (int s = 0; s < kAhead; ++s) {
        const int k = k0 + s * 16 + (lane >> 4) * 4, from = min(k, K - 4);
        beyond_k[s] = k - from;
        __builtin_memcpy(&x[s], a + from, 16);
#pragma unroll
        for (int b = 0; b < BN / 16; ++b) __builtin_memcpy(&y[s][b], w[b] + from, 16);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < kAhead; ++s) {
        const uint4 xs = shift_chunk<BZ_F32>(x[s], beyond_k[s]);
#pragma unroll
        for (int b = 0; b < BN / 16; ++b) {
          const uint4 ys = shift_chunk<BZ_F32>(y[s][b], beyond_k[s]);
          sums[b][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(xs.x), __uint_as_float(ys.x), sums[b][0], 0, 0, 0);
          sums[b][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(xs.y), __uint_as_float(ys.y), sums[b][1], 0, 0, 0);
          sums[b][2] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(xs.z), __uint_as_float(ys.z), sums[b][2], 0, 0, 0);
          sums[b][3] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(xs.w), __uint_as_float(ys.w), sums[b][3], 0, 0, 0);
        }
      }
    }
#pragma unroll
    for (int b = 0; b < BN / 16; ++b)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const float s = (sums[b][0][c] + sums[b][1][c]) + (sums[b][2][c] + sums[b][3][c]);
#pragma unroll
        for (int e = 0; e < EACH; ++e) {
          const float t = __shfl(s, (col & 15) + 16 * (BN == 64 ? e : lane >> 5), bz::kWave);
          if ((col >> 4) == b && (again >> (e * 4 + c) & 1) != 0) v[e][c] = t;
        }
      }
  }
  if (nn >= N) return;
  cbias *= ep.beta;
  if (ep.act == BZ_ACT_DICE) cp2 = EXACT ? dice_den(ep, cp2) : dice_inv_den(ep, cp2);
  OutT* const y = Y + out_index(ep, m0, nn, ldy);
  with_act(ep.act, [&](auto act) {
#pragma unroll
    for (int e = 0; e < EACH; ++e)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int ml = (tid / BN + e * (NT / BN)) * 4 + c;
        if (m0 + ml >= M) continue;
        const float b = ep.bias_rows > 1 ? ep.beta * ep.bias[full_bias_index(ep, m0 + ml, nn, M, N)] : cbias;
        const float z = fmaf(ep.alpha, v[e][c], b);
        constexpr int ACT = decltype(act)::value;
        if constexpr (EXACT && ACT == BZ_ACT_DICE)
          store_out<OutT>(y + ml * ldy, dice_exact(z, cp0, cp1, cp2));
        else
          store_out<OutT>(y + ml * ldy, apply_act_t<ACT>(z, ep, cp0, cp1, cp2));
      }
  });
}

// ---------------------------------------------------------------------------------------------
// split kernel with the skinny head
// ---------------------------------------------------------------------------------------------
// A layer with a head keeps whole rows in one workgroup, so M sets how many CUs work: 16 rows a workgroup where the staged
// tile takes 32, and sixteen waves that share its columns (32 each) and, for N below 256, K, each working for itself as in
// the split kernel above.  After the partial blocks are added up, wave r owns
// row r: its lanes hold the row's outputs in registers, and the head is a dot product within the wave.
constexpr int kHeadWaves = 16;

template <int DT, typename OutT, int HN>
__global__ __launch_bounds__(kHeadWaves * 64) void bz_fc_split_head_kernel(const char* __restrict__ A, const char* __restrict__ W,
                                                                           int M, int N, int K, int64_t lda, int64_t ldw,
                                                                           OutT* __restrict__ Y, int64_t ldy, Epilogue ep, HeadArgs head) {
  using T = In<DT>;
  static_assert(sizeof(OutT) == T::kSize, "the head reads the tile with the operand type");
  constexpr int ES = T::kSize, STEPS = kSplitUnit / 64, COLS = 256 / 64;
  constexpr int kHeadStage = 48 * kSplitPitch<DT>;
  __shared__ __attribute__((aligned(16))) char lds[kHeadWaves * kHeadStage];
  static_assert(16 * 33 * 4 <= kHeadStage, "the partial blocks fit");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m0 = blockIdx.x * 16;
  // the row's columns of this lane: their parameters and the head's weights, asked for first
  float cb[COLS], q0[COLS], q1[COLS], q2[COLS];
  OutT hw[HN == 2 ? HN : 1][COLS];  // (eight outputs' beside the operands do not fit the registers: read at the end)
  const HeadBias<HN> hbias(head);
#pragma unroll
  for (int c = 0; c < COLS; ++c) {
    const int n = min(lane + 64 * c, N - 1);
    cb[c] = ep.bias_rows == 1 ? ep.bias[n] : 0.f;
    q0[c] = q1[c] = q2[c] = 0.f;
    if (ep.act == BZ_ACT_PRELU) q0[c] = ep.p0[ep.act_size == 1 ? 0 : n];
    if (ep.act == BZ_ACT_DICE) {
      q0[c] = ep.p0[n];
      q1[c] = ep.p1[n];
      q2[c] = ep.p2[n];
    }
    if constexpr (HN == 2) {
#pragma unroll
      for (int j = 0; j < HN; ++j) hw[j][c] = ((const OutT*)head.w + n)[(j < head.n ? j : head.n - 1) * head.ldw];
    }
  }
  const int nb = (N + 31) / 32, parts = kHeadWaves / nb, pitch = nb * 32 + 1;
  const int part = wave / nb, block = wave - part * nb;
  const int frow = lane & 15, fq = lane >> 4;
  floatx4 acc[2];
#pragma unroll
  for (int r = 0; r < 4; ++r) acc[0][r] = acc[1][r] = 0.f;
  if (part < parts) {
    char* la = lds + wave * kHeadStage;
    char* lw = la + 16 * kSplitPitch<DT>;
    SplitRows<DT, 2, true> ra;
    SplitRows<DT, 4, true> rw;
    ra.init(A, lda, m0, M, lane);
    rw.init(W, ldw, block * 32, N, lane);
    const int64_t kbytes = (int64_t)K * ES;
    const int whole = (int)(kbytes / kSplitUnit), units = (int)((kbytes + kSplitUnit - 1) / kSplitUnit);
    auto load = [&](int u) {
      if (u < whole) {
        ra.load(u, lane);
        rw.load(u, lane);
      } else if (u < units) {
        ra.load_last(u, K, lane);
        rw.load_last(u, K, lane);
      }
    };
    load(part);
    for (int u = part; u < units; u += parts) {
      ra.store(la, lane);
      rw.store(lw, lane);
      __builtin_amdgcn_wave_barrier();
      load(u + parts);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < STEPS; ++s) {
        const uint4 a = *(const uint4*)(la + split_at<DT>(frow, s * 4 + fq));
        T::mma16(a, *(const uint4*)(lw + split_at<DT>(frow, s * 4 + fq)), acc[0]);
        T::mma16(a, *(const uint4*)(lw + split_at<DT>(16 + frow, s * 4 + fq)), acc[1]);
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
  __syncthreads();  // the operands' LDS becomes the partial blocks'
  float* red = (float*)lds;
  if (part < parts) {
    float* mine = red + (part * 16 + 4 * fq) * pitch + block * 32 + frow;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      mine[r * pitch] = acc[0][r];
      mine[r * pitch + 16] = acc[1][r];
    }
  }
  __syncthreads();
  const int m = m0 + wave;
  if (m >= M) return;
  // (read for all columns at once, and beyond N as well: nothing waits in turn)
  float sum[COLS];
#pragma unroll
  for (int c = 0; c < COLS; ++c) sum[c] = 0.f;
#pragma unroll 4
  for (int p = 0; p < parts; ++p) {
#pragma unroll
    for (int c = 0; c < COLS; ++c) sum[c] += red[(p * 16 + wave) * pitch + min(lane + 64 * c, N - 1)];
  }
  float dot[HN];
#pragma unroll
  for (int j = 0; j < HN; ++j) dot[j] = 0.f;
#pragma unroll
  for (int c = 0; c < COLS; ++c) {
    const int n = lane + 64 * c;
    if (n < N) {
      OutT y;
      store_out<OutT>(&y, apply_act_regs(fmaf(ep.alpha, sum[c], ep.beta * cb[c]), ep, q0[c], q1[c], q2[c]));
      if (Y != nullptr) Y[(int64_t)m * ldy + n] = y;
#pragma unroll
      for (int j = 0; j < HN; ++j) {
        const OutT w = HN == 2 ? hw[HN == 2 ? j : 0][c] : ((const OutT*)head.w + n)[(j < head.n ? j : head.n - 1) * head.ldw];
        dot[j] = fmaf((float)y, (float)w, dot[j]);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < HN; ++j) dot[j] = group_sum<64>(dot[j]);
  if (lane == 0) head_finish(head, hbias, m, dot);
}

// ---------------------------------------------------------------------------------------------
// skinny kernel: N <= 8
// ---------------------------------------------------------------------------------------------
// NMAX: outputs the code is unrolled for
template <int DT, typename OutT, int NMAX>
__global__ __launch_bounds__(256) void bz_fc_skinny_kernel(const char* __restrict__ A, const char* __restrict__ W,
                                                           int M, int N, int K, int lpr_log, int64_t lda, int64_t ldw,
                                                           OutT* __restrict__ Y, OutT* __restrict__ copy, int64_t ldy, Epilogue ep) {
  constexpr int CH = In<DT>::kChunk, ES = In<DT>::kSize;
  const int tid = threadIdx.x;
  const int g = tid >> lpr_log, lpr = 1 << lpr_log, l = tid & (lpr - 1);
  const int rows_per_wg = 256 >> lpr_log;
  const int nchunks = (K + CH - 1) / CH;
  const int64_t stride = (int64_t)gridDim.x * rows_per_wg;
  // A lane's chunk of a row and of every output's weights, all asked for at once: loaded where they are multiplied they were a trip each.
  // The chunk that K ends in is read from in front of its start, and shifted.  us with that, and with sums over the lanes by vector
  // instructions and not through LDS: 2048 x 256 -> 2 fp32 3.26 -> 3.05, 300 x 101 -> 2 fp16 4.06 -> 3.16, 8192 x 512 -> 1 5.5 -> 5.1, 20000 x 300 -> 8
  // 39.1 -> 37.4.  (The first row's asked for in front of the parameters, and each next one's in front of the sums: 5.9, 46.)
  uint4 ra, rw[NMAX];
  int back = 0;
  auto ask = [&](int64_t m, int c) {
    const int k = c * CH;
    if (K >= CH) {
      const int at = min(k, K - CH);
      back = k - at;
      __builtin_memcpy(&ra, A + (m * lda + at) * ES, 16);
#pragma unroll
      for (int n = 0; n < NMAX; ++n)
        if (n < N) __builtin_memcpy(&rw[n], W + (n * ldw + at) * ES, 16);
    } else {
      ra = load_chunk<DT>(A, m, lda, k, K);
#pragma unroll
      for (int n = 0; n < NMAX; ++n)
        if (n < N) rw[n] = load_chunk<DT>(W, n, ldw, k, K);
    }
  };
  int64_t m = (int64_t)blockIdx.x * rows_per_wg + g;
  // per-column parameters first: their latency hides under the row loads
  float cb[NMAX], q0[NMAX], q1[NMAX], q2[NMAX];
#pragma unroll
  for (int n = 0; n < NMAX; ++n) {
    const int nn = n < N ? n : N - 1;
    cb[n] = ep.bias_rows == 1 ? ep.bias[nn] : 0.f;
    q0[n] = q1[n] = q2[n] = 0.f;
    if (ep.act == BZ_ACT_PRELU) q0[n] = ep.p0[ep.act_size == 1 ? 0 : nn];
    if (ep.act == BZ_ACT_DICE) {
      q0[n] = ep.p0[nn];
      q1[n] = ep.p1[nn];
      q2[n] = ep.p2[nn];
    }
  }
  for (int64_t first = (int64_t)blockIdx.x * rows_per_wg; first < M; first += stride, m += stride) {  // (all lanes come along: group_sum's)
    float acc[NMAX];
#pragma unroll
    for (int n = 0; n < NMAX; ++n) acc[n] = 0.f;
    for (int c = l; c < nchunks; c += lpr) {
      ask(m < M ? m : M - 1, c);
      float a[CH];
      chunk_to_float<DT>(back != 0 ? shift_chunk<DT>(ra, back) : ra, a);
#pragma unroll
      for (int n = 0; n < NMAX; ++n) {
        if (n < N) {
          float w[CH];
          chunk_to_float<DT>(back != 0 ? shift_chunk<DT>(rw[n], back) : rw[n], w);
#pragma unroll
          for (int i = 0; i < CH; ++i) acc[n] = fmaf(a[i], w[i], acc[n]);
        }
      }
    }
    // reduce over the lane group, which is aligned, for its first lane, halves first
#pragma unroll
    for (int n = 0; n < NMAX; ++n) {
      if (lpr == 64) {
        const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[n]), __float_as_uint(acc[n]), false, false);
        acc[n] = __uint_as_float(h[0]) + __uint_as_float(h[1]);
      }
      if (lpr >= 32) {
        const auto h = __builtin_amdgcn_permlane16_swap(__float_as_uint(acc[n]), __float_as_uint(acc[n]), false, false);
        acc[n] = __uint_as_float(h[0]) + __uint_as_float(h[1]);
      }
      if (lpr >= 16) acc[n] += row_shl<8>(acc[n]);
      if (lpr >= 8) acc[n] += row_shl<4>(acc[n]);
      if (lpr >= 4) acc[n] += row_shl<2>(acc[n]);
      if (lpr >= 2) acc[n] += row_shl<1>(acc[n]);
    }
    if (l == 0 && m < M) {
      float v[NMAX];
#pragma unroll
      for (int n = 0; n < NMAX; ++n) {
        v[n] = 0.f;
        if (n < N) {
          float x = ep.alpha * acc[n];
          if (ep.bias_rows == 1)
            x += ep.beta * cb[n];
          else if (ep.bias_rows > 1)
            x += ep.beta * ep.bias[full_bias_index(ep, m, n, M, N)];
          v[n] = x;
        }
      }
      if (ep.act == BZ_ACT_SOFTMAX) {  // softmax_op.cc:21-78: subtract max, exp, sum in order, divide
        float mx = v[0];
#pragma unroll
        for (int n = 1; n < NMAX; ++n)
          if (n < N) mx = v[n] > mx ? v[n] : mx;
        float sum = 0.f;
#pragma unroll
        for (int n = 0; n < NMAX; ++n)
          if (n < N) {
            v[n] = expf(v[n] - mx);
            sum += v[n];
          }
#pragma unroll
        for (int n = 0; n < NMAX; ++n)
          if (n < N) v[n] = v[n] / sum;
      } else {
#pragma unroll
        for (int n = 0; n < NMAX; ++n)
          if (n < N) v[n] = apply_act_regs(v[n], ep, q0[n], q1[n], q2[n]);
      }
#pragma unroll
      for (int n = 0; n < NMAX; ++n)
        if (n < N) store_out<OutT>(Y + out_index(ep, m, n, ldy), v[n]);
      if (copy != nullptr) {
#pragma unroll
        for (int n = 0; n < NMAX; ++n)
          if (n < N) store_out<OutT>(copy + m * N + n, v[n]);
      }
    }
  }
}

template <int DT, typename OutT, int BM, int BN, int BK, int WM, int WN, int D, bool ALIGNED, int HEAD = 0,
          int KACC = default_sums<DT, BM, BN, BK, WM, WN, HEAD>()>
int launch_mfma(const bz_fc_desc& d, const Epilogue& ep, hipStream_t st, void* copy = nullptr) {
  const int tiles_m = (d.m + BM - 1) / BM, tiles_n = (d.n + BN - 1) / BN;
  // output rows 16-byte aligned and N a whole number of 16-byte chunks: coalesced stores through LDS
  // (with split outputs every slice must start on a chunk boundary as well)
  const bool vec_y = d.y != nullptr && ((uintptr_t)d.y % 16 == 0) && ((d.ldy * (int64_t)sizeof(OutT)) % 16 == 0) &&
                     (d.n % (16 / (int)sizeof(OutT)) == 0) &&
                     (d.n_split == 0 || (d.n_split % (16 / (int)sizeof(OutT)) == 0 && (d.y_split_stride * (int64_t)sizeof(OutT)) % 16 == 0));
  const HeadArgs head = HEAD != 0 ? head_args(d, copy) : HeadArgs{};
  hipLaunchKernelGGL((bz_fc_mfma_kernel<DT, OutT, BM, BN, BK, WM, WN, D, ALIGNED, HEAD, KACC>), dim3(tiles_m * tiles_n), dim3(WM * WN * 64), 0,
                     st, (const char*)d.a, (const char*)d.w, (OutT*)d.y, d.m, d.n, d.k, d.lda, d.ldw, d.ldy, vec_y, tiles_m, ep, head);
  BZ_LAUNCH_OK("bz_fc_mfma_kernel");
  return BZ_OK;
}


template <int DT, typename OutT, int NW>
int launch_split(const bz_fc_desc& d, const Epilogue& ep, hipStream_t st) {
  const int tiles_m = (d.m + 31) / 32, tiles_n = (d.n + 31) / 32;
  // (K of whole chunks has a tail without shifts and branches.  fp32 layers come here with less than a chunk only.)
  auto kernel = bz_fc_split_kernel<DT, OutT, NW, false>;
  if constexpr (DT != BZ_F32)
    if (d.k % In<DT>::kChunk == 0) kernel = bz_fc_split_kernel<DT, OutT, NW, true>;
  hipLaunchKernelGGL(kernel, dim3(tiles_m * tiles_n), dim3(NW * 64), 0, st, (const char*)d.a,
                     (const char*)d.w, d.m, d.n, d.k, tiles_m, d.lda, d.ldw, (OutT*)d.y, d.ldy, ep);
  BZ_LAUNCH_OK("bz_fc_split_kernel");
  return BZ_OK;
}


template <typename OutT, int NW, int TM, int TN, int SUMS, bool EXACT>
int launch_f32(const bz_fc_desc& d, const Epilogue& ep, hipStream_t st) {
  const int tiles_m = (d.m + 32 * TM - 1) / (32 * TM), tiles_n = (d.n + 32 * TN - 1) / (32 * TN);
  hipLaunchKernelGGL((bz_fc_f32_kernel<OutT, NW, TM, TN, SUMS, EXACT>), dim3(tiles_m * tiles_n), dim3(NW * 64), 0, st, (const char*)d.a, (const char*)d.w, d.m, d.n, d.k, tiles_m,
                     d.lda, d.ldw, (OutT*)d.y, d.ldy, ep);
  BZ_LAUNCH_OK("bz_fc_f32_kernel");
  return BZ_OK;
}

// 2-byte operands and outputs, 16-byte aligned rows on all three, K a whole number of 64-wide tiles
template <int DT, typename OutT>
int launch_stream(const bz_fc_desc& d, const Epilogue& ep, hipStream_t st) {
  const int tiles_m = (d.m + kStreamBM - 1) / kStreamBM, tiles_n = (d.n + kStreamBN - 1) / kStreamBN;
  const int grid = (tiles_m + 7) / 8 * 8 * tiles_n;
  // more dynamic LDS than the default limit: raised once per kernel and device
  static std::mutex mu;
  static bool raised[64] = {};
  int dev = 0;
  BZ_HIP_OK(hipGetDevice(&dev));
  {
    std::lock_guard<std::mutex> lock(mu);
    if (dev >= 0 && dev < 64 && !raised[dev]) {
      BZ_HIP_OK(hipFuncSetAttribute((const void*)bz_fc_stream_kernel<DT, OutT>, hipFuncAttributeMaxDynamicSharedMemorySize, kStreamLds));
      raised[dev] = true;
    }
  }
  hipLaunchKernelGGL((bz_fc_stream_kernel<DT, OutT>), dim3(grid), dim3(2 * kStreamCompute), kStreamLds, st, (const char*)d.a,
                     (const char*)d.w, (OutT*)d.y, d.m, d.n, d.k, d.lda, d.ldw, d.ldy, tiles_m, tiles_n, ep);
  BZ_LAUNCH_OK("bz_fc_stream_kernel");
  return BZ_OK;
}


// Layer + skinny head in one launch: a workgroup owns whole rows of the first layer's output (N <= 256).
template <int DT, typename OutT, int HN>
int dispatch_head(const bz_fc_desc& d, const Epilogue& ep, void* copy, hipStream_t st) {
  constexpr int BK = In<DT>::kSize == 2 ? 64 : 32;
  // fp32 is bound by the matrix cores of the CUs that work, so the staged tile's 32 rows waste time while they are few: 16
  // rows a workgroup up to 2048 rows (us alone / with eight streams of the same, the tile's behind: 1024 x 512 -> 256
  // 17.1 / 4.4 and 24.6 / 6.3, 2048 x 512 -> 256 17.3 / 9.1 and 24.6 / 6.3, 2000 x 512 -> 128 10.9 / 4.7 and 16.7 / 5.9,
  // 201 x 200 -> 80 6.9 / 1.9 and 10.4 / 2.8; before that kernel's chunks had an order of their own, 4096 x 512 -> 256 18.2 / 16.5 and 24.6 / 15.2).  A row's operands cost more
  // this way, which shows where other kernels fill the chip: of a tower on eight serving threads a pass of 1024 rows took
  // 20.4 us and 21.7 with the tile, of 2048 32.1 and 30.7 (64.0 and 69.1 alone), of 4096 63.6 and 57.0 (84.8 and 89.8).
  // 2-byte layers are not bound by the matrix cores (2048 x 512 -> 256 fp16 8.3 / 3.6, the tile 8.2 / 2.2; 201 x 200 -> 80
  // 5.8 / 2.1 and 5.8 / 2.3).
  //
  // HN: outputs the head's code is unrolled for.  Two instead of eight, its bias asked for at the start and its sums taken
  // by vector instructions, and each launch ends 1.5 to 2 us earlier: 2048 x 512 -> 256 fp16 9.7 -> 8.1 us alone, 2.5 -> 2.2
  // with eight streams, fp32 19.9 -> 18.0 / 9.0 -> 8.1; one row of 200 -> 80 fp32 7.9 -> 6.2.
  if constexpr (DT == BZ_F32) {
    if (d.m <= 2048) {
      hipLaunchKernelGGL((bz_fc_split_head_kernel<DT, OutT, HN>), dim3((d.m + 15) / 16), dim3(kHeadWaves * 64), 0, st, (const char*)d.a,
                         (const char*)d.w, d.m, d.n, d.k, d.lda, d.ldw, (OutT*)d.y, d.ldy, ep, head_args(d, copy));
      BZ_LAUNCH_OK("bz_fc_split_head_kernel");
      return BZ_OK;
    }
    // Up to 4096 rows four sums an output, as short as that kernel's (3000 x 512 -> 128 17.9 / 8.3, with two 17.8 / 9.3;
    // 8000 x 512 -> 128 18.1 / 12.7 and 17.9 / 11.6; measured with the head's code unrolled for eight)
    if (d.m <= 4096 && d.n <= 64) return launch_mfma<DT, OutT, 32, 64, BK, 1, 2, 4, true, HN, 4>(d, ep, st, copy);
    if (d.m <= 4096 && d.n <= 128) return launch_mfma<DT, OutT, 32, 128, BK, 1, 4, 4, true, HN, 4>(d, ep, st, copy);
  } else if constexpr (DT == BZ_F16) {  // (bz::fc_fused takes such columns, for a net's layers, none of which is bf16)
    if (d.n % In<DT>::kChunk != 0) {  // (the tiles read a head's weight in whole chunks)
      hipLaunchKernelGGL((bz_fc_split_head_kernel<DT, OutT, HN>), dim3((d.m + 15) / 16), dim3(kHeadWaves * 64), 0, st, (const char*)d.a,
                         (const char*)d.w, d.m, d.n, d.k, d.lda, d.ldw, (OutT*)d.y, d.ldy, ep, head_args(d, copy));
      BZ_LAUNCH_OK("bz_fc_split_head_kernel");
      return BZ_OK;
    }
  }
  if (d.n <= 64) {
    if ((d.m + 63) / 64 >= 256) return launch_mfma<DT, OutT, 64, 64, BK, 2, 2, 4, true, HN>(d, ep, st, copy);
    return launch_mfma<DT, OutT, 32, 64, BK, 1, 2, 4, true, HN>(d, ep, st, copy);
  }
  if (d.n <= 128) return launch_mfma<DT, OutT, 32, 128, BK, 1, 4, 4, true, HN>(d, ep, st, copy);
  // eight waves: with one workgroup per 32 rows only M / 32 CUs work, and each has 288 KB of operands to pull in
  // (two K tiles in flight: with eight waves taking turns that hides the loads, and it was faster than four both alone,
  // 10.5 against 11.3 us on config 2's 512 -> 256 -> 2, and next to other kernels)
  return launch_mfma<DT, OutT, 32, 256, BK, 1, 8, 2, true, HN>(d, ep, st, copy);
}

// The tiles of the staged kernel that both kinds of rows take (ALIGNED: every row starts on 16 bytes and K is a whole
// number of chunks)
template <int DT, typename OutT, bool ALIGNED>
int dispatch_mid(const bz_fc_desc& d, const Epilogue& ep, hipStream_t st) {
  constexpr int BK = In<DT>::kSize == 2 ? 64 : 32;
  const int64_t wg128 = (int64_t)((d.m + 127) / 128) * ((d.n + 127) / 128);
  const int64_t wg64 = (int64_t)((d.m + 63) / 64) * ((d.n + 63) / 64);
  const int64_t wg64x128 = (int64_t)((d.m + 63) / 64) * ((d.n + 127) / 128);
  // tall and narrow (the attention MLP over batch x history rows): one 96-wide tile reads A once
  if (d.n > 64 && d.n <= 96 && (d.m + 127) / 128 >= 256)
    return launch_mfma<DT, OutT, 128, 96, BK, 4, 1, 2, ALIGNED>(d, ep, st);
  // 2-byte operands: eight waves with two K tiles in flight as soon as 64x64 tiles make more than one round of the CUs: 64x128
  // then, 128x64 where that covers the columns, and 128x128 from 129 tiles on, where another round of the smaller ones
  // would cost as much as the first.  us alone / with eight streams of the same: four waves on 64x64 with two K tiles in flight,
  // 64x128, 128x64, 128x128:
  //  2048 x 896 -> 512, 256 tiles of 64x64, 7.6 / 4.9, 8.5 / 4.4, 8.6 / 4.8, 11.3 / 5.4; 1100 x 512 -> 1000, 288, 7.3 / 4.0, 6.5 / 3.9,
  //  6.6 / 3.8; 1500 x 896 -> 704, 264, 9.6 / 5.1, 8.5 / 5.1, 8.6 / 4.8; 2048 x 896 -> 1024, 128 of 128x128, 10.6 / 7.8, 9.6 / 7.3,
  //  9.8 / 7.1, 11.9 / 6.8; 2176 rows, 136, 13.3 / 8.9, 13.6 / 8.5, 14.4 / 9.1, 12.7 / 7.5; 2048 x 2048 -> 1024 17.9 / 14.3 (64x128) and 22.5 / 13.2,
  //  2176 rows 26.2 / 17.4 and 23.1 / 16.3; 20000 x 896 -> 64 10.1 / 6.4, 13.2 / 8.5, 9.2 / 6.2; 17000 x 512 -> 64, 266, 7.2 / 4.4, 9.1 / 5.4,
  //  6.6 / 4.0; 6000 rows of 2048 -> 64, 94, 11.8 / 6.5, 14.6 / 7.7, 14.6 / 7.3.
  // Before, four waves on 64x64 with four K tiles in flight up to 256 tiles of 64x128: 1500 x 896 -> 704 10.7 / 5.5, 2500 x 640 -> 400 9.1 / 4.7
  // and now 7.1 / 4.3, 50000 x 128 -> 64 9.0 / 5.9 and 5.8 / 4.3.
  // Where K is shallow the second round is short and the line to 128x128 lies a little higher (2176 x 128 -> 1024 5.7 / 3.1 and
  // 6.5 / 3.1, 2304 rows, 288 tiles of 64x128, 5.7 / 3.1 and 6.0 / 3.1).
  // Rows that start anywhere: 128x64 (64x64, 64x128, 128x64: 3000 x 901 -> 400 16.5 / 9.7, 13.4 / 8.5, 12.8 / 7.6; 20000 x 901 -> 64 15.7 / 9.4, 20.9 / 13.0,
  // 12.8 / 8.1; 12000 x 301 -> 100 10.4 / 6.0, 9.0 / 5.1, 9.4 / 5.5), up to four K tiles one in flight, as below (4000 x 61 -> 512 5.5 / 3.7
  // and 5.2 / 3.3, with two 6.1 / 3.9; 10000 x 162 -> 200 6.9 / 4.3 and 6.9 / 4.2, 8.1 / 4.6).  At 257 to 272 tiles of 64x64 with deep rows
  // that start anywhere the line is not sharp: 4288 x 1501 -> 200 19.1 / 9.7 (64x64) and 16.6 / 9.1, 4352 rows 15.9 / 9.3 and 16.7 / 9.2.
  if constexpr (In<DT>::kSize == 2) {
    if (d.n > 64 && wg128 >= (d.k > 256 ? 129 : 140)) return launch_mfma<DT, OutT, 128, 128, BK, 2, 4, 2, ALIGNED>(d, ep, st);
    if (wg64 > 256) {
      if constexpr (ALIGNED) {
        if (d.n > 64) return launch_mfma<DT, OutT, 64, 128, BK, 2, 4, 2, ALIGNED>(d, ep, st);
      } else if (d.k <= 4 * BK) {
        return launch_mfma<DT, OutT, 128, 64, BK, 4, 2, 1, ALIGNED>(d, ep, st);
      }
      return launch_mfma<DT, OutT, 128, 64, BK, 4, 2, 2, ALIGNED>(d, ep, st);
    }
  } else if constexpr (ALIGNED) {
    if (d.n > 64 && wg128 >= 512) return launch_mfma<DT, OutT, 128, 128, BK, 2, 2, 3, ALIGNED>(d, ep, st);
    if (d.n > 64 && wg64x128 >= 512) return launch_mfma<DT, OutT, 64, 128, BK, 2, 2, 4, ALIGNED>(d, ep, st);
  }
  // Rows that start anywhere: K is seldom a whole number of tiles, and a tile that is loaded only to be dropped costs as
  // much as any other, so few are in flight: one while K is at most four tiles of 2-byte operands, else two.  64x64,
  // 4-byte rows however many there are (us alone / with eight streams of the same; 32x64 or 64x64 with four in flight: fp16
  // 3000 x 162 -> 200 8.1 / 3.7, now 6.0 / 2.8, 10000 x 50 -> 64 8.8 / 3.6 and 4.5 / 2.1, 2000 x 901 -> 400 14.9 / 9.2 and
  // 10.3 / 5.8).
  if constexpr (!ALIGNED) {
    if constexpr (In<DT>::kSize == 2)
      if (d.k <= 4 * BK) return launch_mfma<DT, OutT, 64, 64, BK, 2, 2, 1, ALIGNED>(d, ep, st);
    return launch_mfma<DT, OutT, 64, 64, BK, 2, 2, 2, ALIGNED>(d, ep, st);
  } else {
    if constexpr (DT == BZ_F32) {
      // (two K tiles in flight; with four waves sharing each, 10000 x 64 -> 200 14.5 / 9.4 and this way 9.6 / 5.8)
      return launch_mfma<DT, OutT, 64, 64, BK, 2, 2, 2, ALIGNED>(d, ep, st);
    } else {
      // Two K tiles in flight, or the one that there is (2048 x 896 -> 512 7.6 us alone / 4.9 with eight streams of the same, with
      // four in flight 8.4 / 4.9, and the model of that layer on eight serving threads 14.2 us a pass with either; 1500 x 896 -> 512
      // 7.9 / 4.0, 32x64 with four 10.8 / 5.8; 730 x 64 -> 512 with one 3.7 / 1.7, with two 4.0 / 1.8)
      if (d.k <= BK) return launch_mfma<DT, OutT, 64, 64, BK, 2, 2, 1, ALIGNED>(d, ep, st);
      return launch_mfma<DT, OutT, 64, 64, BK, 2, 2, 2, ALIGNED>(d, ep, st);
    }
  }
}

template <int DT, typename OutT>
int dispatch_tiles(const bz_fc_desc& d, const Epilogue& ep, bool vec_a, bool vec_w, hipStream_t st) {
  constexpr int BK = In<DT>::kSize == 2 ? 64 : 32;
  // rows 16-byte aligned and K a whole number of chunks
  const bool aligned = vec_a && vec_w && d.k % In<DT>::kChunk == 0;
  // Few tiles: the split kernel (and K below a chunk, which the other loaders cannot read).  Its workgroups are large for
  // what they do, so beyond a line they cost other streams more than they save a lone launch.
  //  2-byte: 256 tiles of 32x32 (us alone / with eight streams of the same, against 64x64: 512 x 896 -> 512, 256 tiles,
  //   4.4 / 2.6 and 7.3 / 3.3; 1024 x 256 -> 512, 512, 4.1 / 2.9 and 4.7 / 2.1);
  //   K above 256 up to 512 with four waves, half the LDS (1024 x 896 -> 512, 512 tiles, eight waves, four, the 64x64 tile:
  //   6.2 / 4.3, 6.0 / 3.7, 7.4 / 3.5; 742 x 2179 -> 512, 384, 12.2 / 8.1, 12.9 / 7.9, 16.5 / 8.7).  Models on eight serving
  //   threads, us a pass, a lone pass in brackets, in the same order: that first layer at batch 1024 11.2 (35.3),
  //   9.8 (35.2), 8.7 (36.8), 1984 -> 512 at 700 10.2 (40.2), 9.9 (39.7), 11.1 (45.3), at 1000 12.3 (38.8), 11.1 (38.3),
  //   10.8 (42.9).
  //  2-byte rows that start anywhere, K at most 256: 192 (850 x 162 -> 200, 189 tiles, 4.3 / 2.2 and 5.1 / 2.2 with one K
  //   tile in flight; 1024 x 162 -> 200, 224, 4.4 / 2.2 and 5.1 / 2.2, but the attention model of that layer, batch 1024, on
  //   eight serving threads 41.1 M samples/s this way and 43.1 on the tile, 63.2 and 63.7 us a lone pass).
  const int64_t wg32 = (int64_t)((d.m + 31) / 32) * ((d.n + 31) / 32);
  if constexpr (DT == BZ_F32) {
    // The bf16 matrix cores, but for rows of shallow K in more tiles than CUs.  32x32 tiles of eight waves while there are few,
    // 32x64 of four up to a 64x64 one for half the CUs, and where K is shallow; else 64x64 (us alone / with eight streams of
    // the same, in that order; with eight waves a 64x64 tile is a little faster alone, 2048 x 896 -> 512 14.5 / 13.7, and slower beside others):
    //  500 x 600 -> 500, 256 tiles of 32x32, 6.7 / 4.1, 8.6 / 3.8, 11.2 / 4.3; 520 rows -> 520, 289, 9.0 / 4.5, 8.6 / 4.0, 11.3 / 4.5;
    //  700 x 200 -> 512, 352, 5.5 / 3.4, 5.9 / 3.2, 8.0 / 3.3; 2000 x 144 -> 200, 441, 5.3 / 4.0, 5.8 / 4.0, 7.3 / 4.1;
    //  1000 x 600 -> 500, 128 of 64x64, 9.4 / 7.1, 9.4 / 5.8, 11.6 / 5.3; 1100 rows, 144, 12.6 / 8.0, 12.7 / 6.6, 11.8 / 5.9;
    //  20000 x 162 -> 256 36.9 / 31.5, 24.8 / 20.4, 26.2 / 19.5; 2000 x 200 -> 800 14.5 / 10.8, 12.7 / 8.0, 11.3 / 7.4.
    // The fp32 tiles / 32x64: 50000 x 80 -> 80 20.8 / 14.4 and 22.0 / 17.1, 20000 x 80 -> 512 37.3 / 24.2 and 32.3 / 27.2,
    // 50000 x 100 -> 200 68 / 47 and 43 / 38, 20000 x 128 -> 512 53 / 38 and 36 / 33.
    // Before, the split kernel below and those tiles: 300 x 445 -> 256 6.8 / 4.0 and now 4.9 / 3.1, 32 x 2075 -> 768 14.8 / 6.0 and
    // 10.2 / 4.0, 1024 x 896 -> 512 13.7 / 10.8 and 11.9 / 8.2, 2048 x 896 -> 512 19.6 / 15.9 and 14.9 / 12.1, 8192 rows 65 / 62 and 49 / 49,
    // 16384 x 301 -> 512 55 / 52 and 43 / 42, 5000 x 3000 -> 1024 380 / 250 and 213 / 220.  Errors against 64 bits, in the
    // same order: 1.5e-7 and 1.2e-7, 2.9e-7 and 2.5e-7, 2.0e-7 and 1.6e-7, 2.7e-7 and 2.3e-7, 5.4e-7 and 2.3e-7, 1.6e-7 and 1.3e-7, 9.7e-7 and 4.2e-7.
    // They grow with what one sum takes in, K over the waves, so beyond 256 inputs the 32x64 tiles, four waves where the split kernel has
    // eight, add every output up in two sums, stage by stage in turn (1024 x 896 -> 512 with one 11.1 / 7.4 and 2.3e-7, 1024 x 4096 -> 512 35.9 / 33
    // and 5.0e-7, with two 38.3 / 32 and 3.5e-7, before 49.8 / 45 and 4.1e-7), and up to 32 columns eight waves stay with
    // 32x32 (12000 x 512 -> 20 9.9 / 6.0, 64x64 11.1 / 6.0, now 8.7 / 5.3; 16384 x 1024 -> 32 17.3 / 13.1, 16.9 / 13.7 and 15.9 / 11.7).
    // Ragged layers of up to 512 tiles of 32x32 and more than 128 of 64x64, which the split kernel had, too, have eight sums from eight waves
    // on 64x64 (four waves, four sums / 32x64, two sums each / this: 2200 x 896 -> 200 16.0 / 7.0 and 2.2e-7, 17.9 / 8.8 and 1.6e-7, 15.6 / 8.5
    // and 1.6e-7; 1700 x 2048 -> 270 26.8 / 14.5, 31.0 / 17.8, 26.0 / 15.7; 4500 x 512 -> 96 11.4 / 5.9, 12.1 / 6.1, 11.4 / 6.2).
    // Up to 512 tiles of 32x32 Dice is exact, as it was in the split kernels (the activation's own error 3.6e-8 of the outputs, with v_exp_f32 and
    // v_rcp_f32 3.9e-8; 1024 x 896 -> 512 with Dice 11.9 us and 11.1, without 10.8); with more, as it was in the tiles.
    const int64_t wg64 = (int64_t)((d.m + 63) / 64) * ((d.n + 63) / 64);
    if (f32_rows_fit(d.lda, d.k) && f32_rows_fit(d.ldw, d.k) && (d.k > 96 || wg64 <= 128 || wg32 <= 512)) {
      if (wg32 <= 256 || (wg32 <= 512 && (d.k <= 256 || d.n <= 32))) return launch_f32<OutT, 8, 1, 1, 1, true>(d, ep, st);
      if (wg64 <= 128) return launch_f32<OutT, 4, 1, 2, 2, true>(d, ep, st);
      if (wg32 <= 512) return launch_f32<OutT, 8, 2, 2, 1, true>(d, ep, st);
      if (d.k < 200) return launch_f32<OutT, 4, 1, 2, 1, false>(d, ep, st);
      return launch_f32<OutT, 4, 2, 2, 1, false>(d, ep, st);
    }
  }
  if (d.k < In<DT>::kChunk || (In<DT>::kSize == 2 && wg32 <= (aligned || d.k > 256 ? 256 : 192))) return launch_split<DT, OutT, 8>(d, ep, st);
  if constexpr (In<DT>::kSize == 2)
    if (wg32 <= 512 && d.k > 256) return launch_split<DT, OutT, 4>(d, ep, st);
  if (!aligned) return dispatch_mid<DT, OutT, false>(d, ep, st);
  // Largest first, and never a tile much wider than N.  128x256 with eight waves and three K tiles in flight fills the
  // chip once it has a workgroup per CU (its fp32 output tile would not fit the operand buffers it is staged in, so
  // 2-byte outputs only); below that the tiles of dispatch_mid.
  const int64_t wg128x256 = (int64_t)((d.m + 127) / 128) * ((d.n + 255) / 256);
  if constexpr (sizeof(OutT) == 2 && In<DT>::kSize == 2) {
    // the streaming kernel once its 256x128 tiles keep most CUs busy and K is deep enough to pay for filling its ring
    // (8192 x 12800 -> 1024 bf16: 192 against 238 us; 4096^3: 128 against 139 us)
    const int64_t wg_stream = (int64_t)((d.m + kStreamBM - 1) / kStreamBM) * ((d.n + kStreamBN - 1) / kStreamBN);
    const bool vec_y = d.y != nullptr && ((uintptr_t)d.y % 16 == 0) && ((d.ldy * 2) % 16 == 0) && d.n % 8 == 0 &&
                       (d.n_split == 0 || (d.n_split % 8 == 0 && (d.y_split_stride * 2) % 16 == 0));
    // (a bias of one row per sample stays with the tile kernels: the streaming kernel's epilogue handles 128 outputs a
    // lane, and an index and a bounds check per output for that rare form cost every layer ten times the activation)
    if (wg_stream >= 200 && d.k % kStreamBK == 0 && d.k >= 8 * kStreamBK && vec_y && d.bias_rows <= 1)
      return launch_stream<DT, OutT>(d, ep, st);
  }
  if constexpr (sizeof(OutT) == 2 && In<DT>::kSize == 2) {
    // (256x256 once even that fills the chip: 4096^3 bf16 987 against 885 TFLOP/s; with fp32 operands these two tiles
    // do not fit the registers)
    const int64_t wg256 = (int64_t)((d.m + 255) / 256) * ((d.n + 255) / 256);
    if (wg256 >= 256 && d.bias_rows <= 1) return launch_mfma<DT, OutT, 256, 256, BK, 4, 2, 2, true>(d, ep, st);
    if (d.n > 128 && wg128x256 >= 256) return launch_mfma<DT, OutT, 128, 256, BK, 2, 4, 3, true>(d, ep, st);
  }
  return dispatch_mid<DT, OutT, true>(d, ep, st);
}

template <int DT, typename OutT>
int dispatch_skinny(const bz_fc_desc& d, const Epilogue& ep, void* copy, hipStream_t st) {
  const int nchunks = (d.k + In<DT>::kChunk - 1) / In<DT>::kChunk;
  int lpr_log = 0;
  while ((1 << lpr_log) < nchunks && lpr_log < 6) ++lpr_log;
  const int rows_per_wg = 256 >> lpr_log;
  int64_t grid = ((int64_t)d.m + rows_per_wg - 1) / rows_per_wg;
  if (grid > 256 * 32) grid = 256 * 32;
  // One and two outputs are the usual heads: unrolled for eight, each wave ran through four times the code and kept 94
  // scalars in vector registers (300 x 100 -> 2 fp16 7.4 us, now 4.8; 8192 x 512 -> 1 11.6 and 6.2; 50000 x 40 -> 1 fp32
  // 15.2 and 7.1).
  if (d.n <= 2)
    hipLaunchKernelGGL((bz_fc_skinny_kernel<DT, OutT, 2>), dim3((int)grid), dim3(256), 0, st, (const char*)d.a, (const char*)d.w,
                       d.m, d.n, d.k, lpr_log, d.lda, d.ldw, (OutT*)d.y, (OutT*)copy, d.ldy, ep);
  else
    hipLaunchKernelGGL((bz_fc_skinny_kernel<DT, OutT, kSkinnyMaxN>), dim3((int)grid), dim3(256), 0, st, (const char*)d.a,
                       (const char*)d.w, d.m, d.n, d.k, lpr_log, d.lda, d.ldw, (OutT*)d.y, (OutT*)copy, d.ldy, ep);
  BZ_LAUNCH_OK("bz_fc_skinny_kernel");
  return BZ_OK;
}

template <int DT>
int dispatch_out(const bz_fc_desc& d, const Epilogue& ep, bool vec_a, bool vec_w, void* copy, hipStream_t st) {
  const bool skinny = d.n <= kSkinnyMaxN;
  switch (d.out_dtype) {
    case BZ_F32:
      return skinny ? dispatch_skinny<DT, float>(d, ep, copy, st) : dispatch_tiles<DT, float>(d, ep, vec_a, vec_w, st);
    case BZ_F16:
      return skinny ? dispatch_skinny<DT, __half>(d, ep, copy, st)
                    : dispatch_tiles<DT, __half>(d, ep, vec_a, vec_w, st);
    case BZ_BF16:
      return skinny ? dispatch_skinny<DT, __hip_bfloat16>(d, ep, copy, st)
                    : dispatch_tiles<DT, __hip_bfloat16>(d, ep, vec_a, vec_w, st);
    default:
      return bz::fail(BZ_EINVAL, "bz_fc_fused: unsupported out dtype %d", d.out_dtype);
  }
}


// one operand type's entry: the layer with a head, or the plain layer (skinny / tile / streaming kernel)
template <int DT, typename T>
int run_typed(const bz_fc_desc& d, const Epilogue& ep, bool vec_a, bool vec_w, void* copy, hipStream_t st) {
  if (d.head_n != 0) return bz::fc::head_unroll(d.head_n) == 2 ? dispatch_head<DT, T, 2>(d, ep, copy, st) : dispatch_head<DT, T, kSkinnyMaxN>(d, ep, copy, st);
  return dispatch_out<DT>(d, ep, vec_a, vec_w, copy, st);
}

}  // namespace
