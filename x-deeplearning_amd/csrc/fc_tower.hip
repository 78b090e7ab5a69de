// fc_tower.hip -- two layers and the skinny one behind them in one launch, fp16: a workgroup takes 32 rows through all three, and what
// the first two put out stays in LDS, rounded to fp16 as it would be stored.
//
// Two launches are two starts, two ends and a trip of the first layer's outputs to memory and back, with many workgroups that each
// last a few us.  Here a workgroup needs nothing from others, few of them do the work of many, and what bounds one is how fast all the
// weights reach its CU: 64 bytes a clock, 917 KB in 14,300 clocks at 896 -> 512, of which it reaches 54.  So weights go from memory to
// the matrix cores' registers, laid out once in the order these take them (through LDS they would cross it twice), 128 KB a CU on their
// way; the rows, which all eight waves read, are in LDS.
// us alone / a launch on four streams, two launches and this: 1024 of 198 -> 200 -> 80 -> 2 11.7 / 5.5 and 7.5 / 3.0, 300 of 445 -> 256 -> 100
// 10.9 / 5.2 and 8.4 / 3.2, 2048 of 896 -> 512 -> 256 16.4 / 6.5 and 14.9 / 4.5 (of these 14.9: rows to LDS 2.9, first layer 6.3, its
// activation 1.1, second layer and activation 2.1, skinny layer 0.9; since then 0.7 more with weights hot in L2, for a second sum an output and for
// what WarmWeights takes, which gives 3.5 where they are not).  fp16 model of 2048 x 26 lists, us a lone pass / of eight serving threads: 43.6 / 13.9
// and 41.8 / 11.9.
#include <mutex>

#include "fc_common.h"

using namespace bz::fc;

namespace {

constexpr int kWaves = 8, kThreads = kWaves * 64, kRows = 32;
constexpr int kGroup = 4;                                  // K steps of 16 whose weights are asked for together
constexpr int kMaxWide = 512, kMaxNarrow = 256;            // outputs of the first and of the second layer
constexpr int kMaxLds = 152 * 1024;

__host__ __device__ constexpr int up(int v, int to) { return (v + to - 1) / to * to; }

// Weights as the matrix instructions take them: block by block of 32 outputs, step by step of 16 inputs, 1 KB each, lane l's
// eight inputs 8 * (l / 32) .. of output l % 32 in its 16 bytes; outputs and inputs filled up with zeros to 64.  A wave then
// reads whole lines, and no weight goes through LDS.
size_t weight_bytes(int64_t k, int64_t n) { return (size_t)(k + 63) / 64 * 64 * ((size_t)(n + 63) / 64 * 64) * 2; }

__global__ __launch_bounds__(256) void bz_fc_tower_pack_kernel(const uint16_t* __restrict__ w, uint4* __restrict__ out, int k, int n, int64_t sk,
                                                               int64_t sn, int units) {
  const int u = blockIdx.x * 256 + threadIdx.x;
  if (u >= units) return;
  const int steps = up(k, 64) / 16, lane = u % 64, step = u / 64 % steps, block = u / 64 / steps;
  const int o = block * 32 + lane % 32, i0 = step * 16 + lane / 32 * 8;
  uint16_t v[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = o < n && i0 + i < k ? w[(i0 + i) * sk + o * sn] : (uint16_t)0;
  out[u] = *(const uint4*)v;
}

struct Tower {
  const char* x;  // [m, lda]
  int lda;        // bytes
  int m, k, n1, n2;
  const char *w1, *w2;
};
// what is needed later than that
struct Finish {
  Epilogue ep1, ep2;
  HeadArgs head;
};

// LDS, in bytes.  Rows of operands as 16-byte units, unit (c, r) = inputs 8 c .. of row r at (c * kRows + r) * 16: fragment
// reads and the epilogue's writes are each 1 KB without a bank conflict.
struct Layout {
  int rows2, params, head_w, dots, all;
};
__host__ __device__ inline Layout layout(int k, int n1, int n2, int hn) {
  const int k1 = up(k, 64), k2 = up(n1, 64), k3 = up(n2, 64);
  Layout l;
  l.rows2 = kRows * (k1 > k2 ? k1 : k2) * 2;  // the input, then the first layer's outputs over it
  l.params = l.rows2 + kRows * k3 * 2;
  l.head_w = l.params + 4 * (k2 + k3) * 4;
  l.dots = l.head_w + hn * k3 * 2;
  l.all = l.dots + kWaves * kRows * hn * 4;
  return l;
}

// The kernel's start is short straight-line code: loads through buffer resources, which give zeros behind what they cover, need no
// branches and no 64-bit addresses.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)bytes, 0x00020000);
}
constexpr int kBeyond = 1 << 30;  // an offset behind any of them

// A thread's column of a layer: its parameters, asked for at the kernel's start and put into LDS behind the rows: beta * bias, then as
// apply_act_t takes them; zeros behind the layer's columns.
struct Column {
  float bias, p0, p1, p2;
  __device__ __forceinline__ void ask(const Epilogue& ep, int n) {
    const int at = threadIdx.x * 4;
    auto load = [&](const float* from, int size, int off) {
      return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(buffer_of(from, from != nullptr ? size * 4 : 0), off, 0, 0));
    };
    bias = load(ep.bias_rows != 0 ? ep.bias : nullptr, n, at);
    p0 = load(ep.p0, ep.act_size == 1 ? 1 : n, ep.act_size == 1 ? 0 : at);
    p1 = load(ep.p1, n, at);
    p2 = load(ep.p2, n, at);
  }
  __device__ __forceinline__ void put(const Epilogue& ep, int padded, float* to) const {
    const int i = threadIdx.x;
    if (i >= padded) return;
    to[i] = ep.beta * bias;
    to[padded + i] = p0;
    to[2 * padded + i] = p1;
    to[3 * padded + i] = ep.act == BZ_ACT_DICE ? dice_inv_den(ep, p2) : 0.f;
  }
};

// a layer's weights: where they are, blocks of 32 outputs, steps of 16 inputs
struct Weights {
  __amdgpu_buffer_rsrc_t from;
  int blocks, steps;
  __device__ __forceinline__ Weights(const char* w, int k, int n) : blocks(up(n, 64) / 32), steps(up(k, 64) / 16) {
    from = buffer_of(w, blocks * steps * 1024);
  }
};

// The weights of blocks `block` and, with TN == 2, block + kWaves, as they stream through registers.  (The last block's where there
// is no such one: nothing is made of them.)
template <int TN>
struct WeightStream {
  uint4 w[kGroup][TN];
  __device__ __forceinline__ void ask(const Weights& from, int block, int group) {
    const int lane = threadIdx.x & 63, groups = from.steps / kGroup;
    // (behind the last group nothing is read, and the loop's waits count the same loads all the same)
    const int at = group < groups ? lane * 16 : kBeyond;
    group = min(group, groups - 1);
#pragma unroll
    for (int j = 0; j < kGroup; ++j)
#pragma unroll
      for (int t = 0; t < TN; ++t) {
        const int b = min(block + t * kWaves, from.blocks - 1);
        const auto v = __builtin_amdgcn_raw_buffer_load_b128(from.from, at, (b * from.steps + group * kGroup + j) * 1024, 0);
        w[j][t] = *(const uint4*)&v;
      }
    __builtin_amdgcn_sched_barrier(0);  // (they stay ahead of what the wave multiplies meanwhile)
  }
};

// The weights on their way into the XCD's L2: its workgroups ask for a share each, a word of every line, while the rows are staged.  In a
// pass of a whole model the lookups have been through L2 since the last one, all workgroups walk the weights in step, and each waits for
// every line as if it were alone: 128 KB under way are too few for the memory's latency.  (A lone pass of 2048 x 26 lists, 896 -> 512 -> 256 -> 2,
// without this 45.4 us, 43.5 in two launches, 41.7 this way; on eight threads 12.4, 13.8 and 11.9 a pass.)
struct WarmWeights {
  static constexpr int kEach = 2;  // of the first layer, a thread's: its 0.9 MB where eight workgroups share an XCD
  uint32_t w[kEach + 1];
  __device__ __forceinline__ void ask(const Weights& w1, const Weights& w2) {
    // (shares of a wave's 64 lines, so that few weights, too, are as many loads for each)
    const uint32_t sharers = (gridDim.x + bz::kNumXcd - 1) / bz::kNumXcd, mine = blockIdx.x / bz::kNumXcd, wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    auto line = [&](uint32_t i) { return (int)((((i * kWaves + wave) * sharers + mine) * 64 + lane) * 128u); };
#pragma unroll
    for (int i = 0; i < kEach; ++i) w[i] = __builtin_amdgcn_raw_buffer_load_b32(w1.from, line(i), 0, 0);
    w[kEach] = __builtin_amdgcn_raw_buffer_load_b32(w2.from, line(0), 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  }
  // (they have arrived by now; until here nobody has waited for them)
  __device__ __forceinline__ void done() const {
#pragma unroll
    for (int i = 0; i <= kEach; ++i) asm volatile("" ::"v"(w[i]));
  }
};

// Not for a layer of one block of columns a wave: the loads of a word a line, and the registers, cost its short workgroups what they spare (eight
// serving threads, 64 passes of 2595 rows, 104 -> 100 -> 100, 380 us with them and 360 without; a lone pass of 2048 x 26 lists, 896 -> 256 -> 104, 33.2
// either way).
struct NoWarming {
  __device__ __forceinline__ void ask(const Weights&, const Weights&) {}
  __device__ __forceinline__ void done() const {}
};

// the rows' side of a group
struct RowFragments {
  uint4 x[kGroup];
  __device__ __forceinline__ void read(const char* rows, int group) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int j = 0; j < kGroup; ++j) x[j] = *(const uint4*)(rows + (((group * kGroup + j) * 2 + lane / 32) * kRows + lane % 32) * 16);
    __builtin_amdgcn_sched_barrier(0);
  }
};

// A layer's weights on their way through three sets of registers: two groups are asked for at its start, and one ahead of each
// that is multiplied, 128 KB a CU under way; the rows' fragments are read a group ahead.  (2048 x 896 -> 512 -> 256 with two sets 15.1 us
// alone as with three, 64 passes on eight serving threads 877 and 857; with four and five 16.0 and 15.9.)
template <int TN>
struct Layer {
  WeightStream<TN> w[3];
  RowFragments r[3];
  // An output's two sums, of every other step of 16 inputs, as in the tiles.  (896 -> 512 -> 256 -> 2: the model's error is that of two
  // launches; with one sum 20 % more outputs are rounded to the other side.)
  floatx16 acc[TN], odd[TN];
  __device__ __forceinline__ void start(const Weights& from, int block) {
    w[0].ask(from, block, 0);
    w[1].ask(from, block, 1);
  }
  __device__ __forceinline__ void multiply(int i) {
#pragma unroll
    for (int j = 0; j < kGroup; ++j)
#pragma unroll
      for (int t = 0; t < TN; ++t) In<BZ_F16>::mma(w[i].w[j][t], r[i].x[j], j % 2 == 0 ? acc[t] : odd[t]);
    __builtin_amdgcn_sched_barrier(0);
  }
  // acc = the weights' blocks times the rows.  (Behind the last group's fragments lie others: read, and not used.)
  __device__ __forceinline__ void run(const Weights& from, const char* rows, int block) {
    const int groups = from.steps / kGroup;
    r[0].read(rows, 0);
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[t][i] = odd[t][i] = 0.f;
    int g = 0;
    for (; g + 3 <= groups; g += 3) {  // (no branch around an ask: the waits behind it would be for everything)
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        w[(i + 2) % 3].ask(from, block, g + i + 2);
        r[(i + 1) % 3].read(rows, g + i + 1);
        multiply(i);
      }
    }
    if (g < groups) {
      r[1].read(rows, g + 1);
      multiply(0);
      if (g + 1 < groups) multiply(1);
    }
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[t][i] += odd[t][i];
  }
};

__device__ __forceinline__ uint32_t round_pair(float x, float y) {
  typedef _Float16 half2v __attribute__((ext_vector_type(2)));
  const half2v h = __builtin_convertvector((floatx2{x, y}), half2v);  // v_cvt_pk_f16_f32
  return *(const uint32_t*)&h;
}

// bias and activation, rounded, as the next layer's rows; zeros behind the layer's columns.  Lane l holds row l % 32, columns
// 8 * (i / 4) + 4 * (l / 32) + i % 4 of a block.
template <int TN>
__device__ __forceinline__ void finish(const Epilogue& ep, const float* params, int n, int padded, int block, const floatx16 (&acc)[TN], char* rows) {
  const int lane = threadIdx.x & 63;
  with_act(ep.act, [&](auto act) {
#pragma unroll
    for (int t = 0; t < TN; ++t) {
      const int n0 = (block + t * kWaves) * 32;
      if (n0 >= padded) continue;
      const float* of = params + n0 + lane / 32 * 4;
      char* to = rows + (n0 / 8 * kRows + lane % 32) * 16 + lane / 32 * 8;
      uint2 v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float4 bias = *(const float4*)(of + q * 8), p0 = *(const float4*)(of + padded + q * 8), p1 = *(const float4*)(of + 2 * padded + q * 8),
                     p2 = *(const float4*)(of + 3 * padded + q * 8);
        float z[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
          z[i] = apply_act_t<decltype(act)::value>(fmaf(ep.alpha, acc[t][q * 4 + i], (&bias.x)[i]), ep, (&p0.x)[i], (&p1.x)[i], (&p2.x)[i]);
        v[q] = make_uint2(round_pair(z[0], z[1]), round_pair(z[2], z[3]));
      }
      if (n0 + 32 > n) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int left = n - n0 - q * 8 - lane / 32 * 4;
          v[q].x = left >= 2 ? v[q].x : left == 1 ? v[q].x & 0xffffu : 0u;
          v[q].y = left >= 4 ? v[q].y : left == 3 ? v[q].y & 0xffffu : 0u;
        }
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) *(uint2*)(to + q * kRows * 16) = v[q];
    }
  });
}

// The workgroup's rows of the input to LDS, inputs filled up with zeros to 64.  `meanwhile` runs when the first are asked for, `then`
// when they are written.  16-byte loads need addresses that are multiples of 4 only; ODD: rows may start 2 bytes behind one, and every
// unit is put together from the 16 bytes before its start and the next 4 (300 x 445 -> 256 -> 100: 9.2 us with eight 2-byte loads a
// unit, 8.4 this way).  Inputs that fill no unit come one by one, the last wave's lanes a row each.
template <bool ODD, typename F, typename G>
__device__ __forceinline__ void stage_rows(const Tower& a, int m0, char* rows, const F& meanwhile, const G& then) {
  constexpr int kAhead = 8;
  const int lane = threadIdx.x & 63, wave = threadIdx.x / 64;
  const int here = min(a.m - m0, kRows), groups = up(a.k, 64) / 64, whole = a.k / 8, rest = a.k % 8;
  const char* from = a.x + (int64_t)m0 * a.lda;
  const int start = ODD ? (int)((uintptr_t)from & 2) : 0;
  const auto x = buffer_of(from - start, (uint32_t)up(start + (here - 1) * a.lda + a.k * 2, 4));
  // A wave has eight of the rows (lane % 8), every other 64 inputs (unit lane / 8): whole lines read, and 128 bytes a quarter wave
  // written
  const int r = wave % 4 * 8 + lane % 8, c0 = wave / 4 * 8 + lane / 8;
  const bool last = rest != 0 && wave == kWaves - 1 && lane < kRows;
  uint16_t tail[8];
  auto batch = [&](int g0, const F* meanwhile) {
    uint4 v[kAhead];
    uint32_t next[kAhead];
    const int base = start + r * a.lda, odd = ODD ? base & 2 : 0;
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      const int c = g0 * 8 + c0 + i * 16;
      const int at = r < here && c < whole ? base - odd + c * 16 : kBeyond;
      const auto u = __builtin_amdgcn_raw_buffer_load_b128(x, at, 0, 0);
      v[i] = *(const uint4*)&u;
      if constexpr (ODD) next[i] = __builtin_amdgcn_raw_buffer_load_b32(x, odd != 0 ? at : kBeyond, 16, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (meanwhile != nullptr) (*meanwhile)();
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      if constexpr (ODD) {
        v[i].x = __builtin_amdgcn_alignbyte(v[i].y, v[i].x, odd);
        v[i].y = __builtin_amdgcn_alignbyte(v[i].z, v[i].y, odd);
        v[i].z = __builtin_amdgcn_alignbyte(v[i].w, v[i].z, odd);
        v[i].w = __builtin_amdgcn_alignbyte(next[i], v[i].w, odd);
      }
      const int g = g0 + wave / 4 + i * 2, c = g0 * 8 + c0 + i * 16;
      if (g < groups && (rest == 0 || c != whole)) *(uint4*)(rows + (c * kRows + r) * 16) = v[i];
    }
  };
  if (last) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      tail[i] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(x, i < rest && lane < here ? start + lane * a.lda + (whole * 8 + i) * 2 : kBeyond, 0, 0);
  }
  batch(0, &meanwhile);
  then();
  if (last) {
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = tail[2 * i] | (uint32_t)tail[2 * i + 1] << 16;
    *(uint4*)(rows + (whole * kRows + lane) * 16) = make_uint4(w[0], w[1], w[2], w[3]);
  }
  for (int g = kAhead * 2; g < groups; g += kAhead * 2) batch(g, nullptr);
}

// TN: blocks of 32 columns a wave holds of the first layer; with one, two workgroups share a CU (with more registers than that leaves, the
// attention model on eight serving threads, whose 162 -> 200 -> 80 it is, comes to 62 M samples/s for 66).  HN: outputs the skinny layer's code is unrolled for.  ODD: stage_rows'.
template <int TN, int HN, bool ODD>
__global__ __launch_bounds__(kThreads, TN == 1 ? 4 : 2) void bz_fc_tower_kernel(const char* x, const char* w1_, const char* w2_, int lda, int m, int k, int n1,
                                                                                int n2, const Finish f) {
  typedef __half T;
  const Tower a = {x, lda, m, k, n1, n2, w1_, w2_};
  extern __shared__ __align__(16) char lds[];
  const Layout at = layout(a.k, a.n1, a.n2, HN);
  const int k2 = up(a.n1, 64), k3 = up(a.n2, 64);
  const int m0 = blockIdx.x * kRows, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const Weights w1(a.w1, a.k, a.n1), w2(a.w2, a.n1, a.n2);
  char* rows2 = lds + at.rows2;
  float *params1 = (float*)(lds + at.params), *params2 = params1 + 4 * k2, *dots = (float*)(lds + at.dots);
  T* head_w = (T*)(lds + at.head_w);

  // The rows first, whose addresses come with the wave (the kernel's first arguments are preloaded); then, once the other arguments have
  // arrived, the parameters, and the weights behind them
  Layer<TN> first;
  HeadBias<HN> hbias;
  Column col1, col2;
  constexpr int kHeadPer = HN * kMaxNarrow / kThreads;  // of the skinny layer's weights, a thread's
  const int hc = threadIdx.x % kMaxNarrow, hj = threadIdx.x / kMaxNarrow;
  uint16_t hw[kHeadPer];
  std::conditional_t<(TN > 1), WarmWeights, NoWarming> warm;
  stage_rows<ODD>(
      a, m0, lds,
      [&]() {
        hbias.ask(f.head);
        col1.ask(f.ep1, a.n1);
        col2.ask(f.ep2, a.n2);
        const auto from_head = buffer_of(f.head.w, (uint32_t)(((f.head.n - 1) * (int)f.head.ldw + a.n2) * 2));
#pragma unroll
        for (int i = 0; i < kHeadPer; ++i) {
          const int j = hj + i * (kThreads / kMaxNarrow);
          hw[i] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(from_head, j < f.head.n && hc < a.n2 ? (j * (int)f.head.ldw + hc) * 2 : kBeyond, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        first.start(w1, wave);
        warm.ask(w1, w2);
      },
      [&]() {
        col1.put(f.ep1, k2, params1);
        col2.put(f.ep2, k3, params2);
#pragma unroll
        for (int i = 0; i < kHeadPer; ++i)
          if (hc < k3) ((uint16_t*)head_w)[(hj + i * (kThreads / kMaxNarrow)) * k3 + hc] = hw[i];
      });
  __syncthreads();

  const bool busy1 = wave * 32 < k2, busy2 = wave * 32 < k3;
  if (busy1) first.run(w1, lds, wave);
  warm.done();
  Layer<1> second;
  second.start(w2, wave);
  __syncthreads();
  if (busy1) finish<TN>(f.ep1, params1, a.n1, k2, wave, first.acc, lds);
  __syncthreads();
  if (busy2) {
    second.run(w2, lds, wave);
    finish<1>(f.ep2, params2, a.n2, k3, wave, second.acc, rows2);
  }
  __syncthreads();

  // the skinny layer from the rounded outputs: sixteen lanes share a row, eight columns at a time
  float dot[HN];
#pragma unroll
  for (int j = 0; j < HN; ++j) dot[j] = 0.f;
  const int r = threadIdx.x % kRows;
  for (int c = threadIdx.x / kRows; c < k3 / 8; c += kThreads / kRows) {
    const uint4 y = *(const uint4*)(rows2 + (c * kRows + r) * 16);
#pragma unroll
    for (int j = 0; j < HN; ++j) {
      const uint4 w = *(const uint4*)(head_w + j * k3 + c * 8);
#pragma unroll
      for (int i = 0; i < 8; ++i) dot[j] = fmaf((float)((const T*)&y)[i], (float)((const T*)&w)[i], dot[j]);
    }
  }
#pragma unroll
  for (int j = 0; j < HN; ++j) {
    const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(dot[j]), __float_as_uint(dot[j]), false, false);
    dot[j] = __uint_as_float(h[0]) + __uint_as_float(h[1]);
    if ((threadIdx.x & 32) == 0) dots[(wave * HN + j) * kRows + r] = dot[j];
  }
  __syncthreads();
  if (threadIdx.x < kRows && m0 + r < a.m) {
#pragma unroll
    for (int j = 0; j < HN; ++j) {
      dot[j] = 0.f;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) dot[j] += dots[(w * HN + j) * kRows + r];
    }
    head_finish(f.head, hbias, m0 + r, dot);
  }
}

template <int TN, int HN, bool ODD>
int launch(const Tower& a, const Finish& f, int lds, hipStream_t st) {
  // more dynamic LDS than the default limit: raised once per kernel and device
  static std::mutex mu;
  static bool raised[64] = {};
  int dev = 0;
  BZ_HIP_OK(hipGetDevice(&dev));
  {
    std::lock_guard<std::mutex> lock(mu);
    if (dev >= 0 && dev < 64 && !raised[dev]) {
      BZ_HIP_OK(hipFuncSetAttribute((const void*)bz_fc_tower_kernel<TN, HN, ODD>, hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds));
      raised[dev] = true;
    }
  }
  hipLaunchKernelGGL((bz_fc_tower_kernel<TN, HN, ODD>), dim3((a.m + kRows - 1) / kRows), dim3(kThreads), lds, st, a.x, a.w1, a.w2, a.lda, a.m, a.k, a.n1, a.n2,
                     f);
  BZ_LAUNCH_OK("bz_fc_tower_kernel");
  return BZ_OK;
}

template <int TN, int HN>
int with_rows(const Tower& a, const Finish& f, int lds, hipStream_t st) {
  return (((uintptr_t)a.x | (uintptr_t)a.lda) & 3) != 0 ? launch<TN, HN, true>(a, f, lds, st) : launch<TN, HN, false>(a, f, lds, st);
}

}  // namespace

size_t bz::fc_tower_weight_bytes(int64_t k, int64_t n) { return weight_bytes(k, n); }

int bz::fc_tower_pack(const void* w, bool transposed, int k, int n, void* out, bz_stream_t stream) {
  const int units = (int)(weight_bytes(k, n) / 16);
  hipLaunchKernelGGL(bz_fc_tower_pack_kernel, dim3((units + 255) / 256), dim3(256), 0, bz::as_stream(stream), (const uint16_t*)w, (uint4*)out, k, n,
                     transposed ? (int64_t)1 : (int64_t)n, transposed ? (int64_t)k : (int64_t)1, units);
  BZ_LAUNCH_OK("bz_fc_tower_pack_kernel");
  return BZ_OK;
}

bool bz::fc_tower_takes(int64_t k, int64_t n1, int64_t n2) {
  return k >= 1 && k <= 1280 && n1 > kSkinnyMaxN && n1 <= kMaxWide && n2 > kSkinnyMaxN && n2 <= kMaxNarrow &&
         layout((int)k, (int)n1, (int)n2, kSkinnyMaxN).all <= kMaxLds;
}

// One launch against two, in models that look 32-wide rows up for the input, us of a lone pass / of eight serving threads (weights in units
// of 1024): one where a lone pass is no longer, or by 2 % where the threads gain more.  From 1200 rows on that is with inputs up to 1024:
//  896 -> 512 -> 256 (576) 1100 rows 37.8 / 9.9 and 37.7 / 9.3, 1300 39.0 / 9.2 and 39.2 / 10.5, 2048 39.4 / 10.3 and 39.6 / 11.9, 4096 47.2 / 18.8
//  and 50.4 / 21.7; 1024 -> 512 -> 256 (640) 1600 41.1 / 10.5 and 40.8 / 12.1, 3000 45.0 / 16.2 and 47.6 / 18.8; 1024 -> 256 -> 128 (288) 1300
//  34.2 / 8.6 and 36.1 / 10.3; but 2048 of 1152 -> 512 -> 256 47.0 / 13.2 and 45.8 / 14.8, of 1216 -> 200 -> 80 41.9 / 11.6 and 40.4 / 13.2.
// With fewer rows, and few workgroups to pull all the weights, where these are few:
//  (256) with inputs up to 768, or up to 1024 from 600 rows on: 600 rows of 640 -> 256 -> 100 (185) 29.1 / 6.4 and 30.2 / 7.4, 768 -> 256 -> 100
//   (217) 30.4 / 6.8 and 31.0 / 7.7, 352 -> 512 -> 100 (226) 30.1 / 6.6 and 31.1 / 7.6; 300 of them 29.2 / 6.2 and 29.7 / 6.8, 30.2 / 6.6 and
//   30.2 / 7.0, 30.5 / 6.9 and 29.6 / 7.1; 64 (longer alone in the model, but not in a whole request: two samples of 730 -> 256 -> 256 looked up by key
//   36.4 and 38.2) 27.4 / 5.5 and 26.7 / 6.0, 28.7 / 6.0 and 27.5 / 6.4, 29.2 / 5.6 and 26.7 / 6.2; 900 of 896 -> 200 -> 80 (190) 31.9 / 7.4 and
//   32.5 / 7.9; but 300 of 896 -> 256 -> 104 (250) 32.6 / 7.4 and 31.7 / 7.0, 600 of 640 -> 400 -> 128 (300) 33.5 / 8.5 and 31.9 / 7.6;
//  (144) any: 256 -> 200 -> 80 (65) 300 rows 24.0 / 5.3 and 26.5 / 6.2; 448 -> 256 -> 100 (137) one row 23.0 / 5.0 and 23.4 / 5.3, 300 26.6 / 5.8
//   and 28.4 / 6.9; 640 -> 100 -> 256 (87) 203 27.3 / 5.8 and 31.6 / 7.3; 640 -> 200 -> 80 (140) 64 27.7 / 5.5 and 27.0 / 6.1; 1024 -> 128 -> 100 (140) 64
//   28.7 / 6.0 and 28.2 / 6.2; 1280 -> 100 -> 40 (128) 300 33.2 / 7.1 and 35.3 / 7.8; but 64 of 1152 -> 128 -> 64 (152) 30.6 / 6.1 and 28.8 / 6.7.
// (Alone on hot weights one launch wins far beyond these lines: 300 of 896 -> 256 -> 104 9.8 and 10.4.)  Beyond 4096 rows two launches leave
// more to others (6000 of 896 -> 400 -> 128 on hot weights 15.5 us alone, 11.5 on four streams, and 21.4, 10.9).
bool bz::fc_tower_pays(int64_t rows, int64_t k, int64_t n1, int64_t n2) {
  if (rows < 1 || rows > 4096 || k > 1280) return false;
  const bool more = k <= 768 || (k <= 1024 && rows >= 600);
  return (rows >= 1200 && k <= 1024) || k * n1 + n1 * n2 <= (more ? 256 << 10 : 144 << 10);
}

int bz::fc_tower(const bz_fc_desc& d, void* copy, bz_stream_t stream) {
  BZ_REQUIRE(d.next != nullptr, "tower: no second layer");
  const bz_fc_next& x = *d.next;
  auto plain = [](int act) { return act == BZ_ACT_NONE || act == BZ_ACT_PRELU || act == BZ_ACT_DICE || act == BZ_ACT_LEAKY_RELU || act == BZ_ACT_SIGMOID; };
  if (d.in_dtype != BZ_F16 || d.out_dtype != d.in_dtype || !fc_tower_takes(d.k, d.n, x.n) || d.y != nullptr || x.y != nullptr ||
      d.head_n < 1 || d.head_n > kSkinnyMaxN || d.n_split != 0 || d.a_pieces != nullptr || d.bias_rows > 1 || !plain(d.act) || !plain(x.act))
    return bz::fail(BZ_ENOTSUP, "tower: a shape or form outside the kernel's");
  BZ_REQUIRE(d.a != nullptr && d.w != nullptr && x.w != nullptr && d.head_w != nullptr && d.head_y != nullptr && d.lda >= d.k && d.head_ldw >= x.n &&
                 d.head_ldy >= d.head_n,
             "tower: null operand or a leading dimension below its row");
  BZ_REQUIRE(d.bias_rows == 0 || d.bias != nullptr, "tower: bias_rows=%d without bias", d.bias_rows);
  BZ_REQUIRE(d.act != BZ_ACT_PRELU || (d.act_p0 && (d.act_size == 1 || d.act_size == d.n)), "tower: PRelu slope size %d", d.act_size);
  BZ_REQUIRE(d.act != BZ_ACT_DICE || (d.act_p0 && d.act_p1 && d.act_p2), "tower: Dice needs gamma, mean and var");
  BZ_REQUIRE(x.act != BZ_ACT_PRELU || (x.act_p0 && (x.act_size == 1 || x.act_size == x.n)), "tower: PRelu slope size %d", x.act_size);
  BZ_REQUIRE(x.act != BZ_ACT_DICE || (x.act_p0 && x.act_p1 && x.act_p2), "tower: Dice needs gamma, mean and var");
  if (d.lda > 1 << 20 || d.head_ldw > 1 << 20) return bz::fail(BZ_ENOTSUP, "tower: rows further apart than the kernel's offsets reach");
  BZ_REQUIRE(d.m >= 0 && d.m < (1ll << 31) - kRows, "tower: %lld rows", (long long)d.m);
  if (d.m == 0) return BZ_OK;
  Tower a = {};
  Finish f = {};
  a.x = (const char*)d.a;
  a.lda = (int)d.lda * 2;
  a.m = d.m;
  a.k = d.k;
  a.n1 = d.n;
  a.n2 = x.n;
  a.w1 = (const char*)d.w;
  a.w2 = (const char*)x.w;
  f.ep1 = fc_epilogue(d);
  f.ep2.bias = x.bias;
  f.ep2.bias_rows = x.bias != nullptr ? 1 : 0;
  f.ep2.p0 = x.act_p0;
  f.ep2.p1 = x.act_p1;
  f.ep2.p2 = x.act_p2;
  f.ep2.act = x.act;
  f.ep2.act_size = x.act_size;
  f.ep2.dice_nosqrt = x.dice_nosqrt;
  f.ep2.alpha = x.alpha;
  f.ep2.beta = x.beta;
  f.ep2.act_alpha = x.act_alpha;
  // (a layer without these activations may have their pointers set all the same)
  for (Epilogue* e : {&f.ep1, &f.ep2}) {
    if (e->act != BZ_ACT_PRELU && e->act != BZ_ACT_DICE) e->p0 = nullptr;
    if (e->act != BZ_ACT_DICE) e->p1 = e->p2 = nullptr;
  }
  f.head = head_args(d, copy);
  hipStream_t st = bz::as_stream(stream);
  const int lds = layout(d.k, d.n, x.n, head_unroll(d.head_n)).all;
  const bool two = head_unroll(d.head_n) == 2;
  if (a.n1 <= kWaves * 32) return two ? with_rows<1, 2>(a, f, lds, st) : with_rows<1, kSkinnyMaxN>(a, f, lds, st);
  return two ? with_rows<2, 2>(a, f, lds, st) : with_rows<2, kSkinnyMaxN>(a, f, lds, st);
}
