// fc_rows.hip -- two layers and the skinny one behind them in one launch, for few rows: a workgroup takes one to four rows through all of
// them, and nothing but the last layer's outputs goes to memory.
//
// With few rows a layer is a chain and not work: each launch starts, waits for operands, adds up, ends.  Here there is one chain; what bounds
// it is the instructions in front of the first products and, with more weights, how fast these reach a CU, 64 bytes a clock.  So weights are laid out once as the lanes take them and asked
// for as early as there are registers for them (128 KB a CU under way; the second layer's follow the first's, ahead of the first's
// outputs), and no instruction is spent on them but the load and the products: a lane has one output's 16 bytes, and
// v_mfma_f32_4x4x1 (sixteen blocks of four outputs and four rows) multiplies four rows at a time by them; waves share K.
//
// us of the kernels, before (layer, and layer with head; 1.5 to 2 between the two) and now: one row of 192 -> 200 -> 80 -> 2 4.5 + 6.1 and 7.0, 201 of 144
// -> 200 -> 80 -> 2 4.8 + 8.5 and 8.5; a request with them 30.9 -> 28.6 and 54.3 -> 48.9.  Of one row's 14,600 clocks the first loads are under way
// at 2,200, the rows are in LDS at 4,600, the first layer's sums are there at 9,500, its activation at 10,600, the second's sums at 12,400.  What
// is kept short is the code, which every CU has to fetch: with the splits worked out in the kernel and sixteen waves it took 9.3, with outputs
// beside each other in a lane's block, each load's bounds checked and a reduction every 64 outputs 14.7.
#include "fc_common.h"

using namespace bz::fc;

namespace {

constexpr int kWaves = 8, kThreads = kWaves * 64, kRows = 4, kPerRow = kThreads / kRows;
constexpr int kGroup = 4;  // chunks of 16 bytes (a lane's, of its output) asked for together
constexpr int kRing = 4;   // such groups under way
constexpr int kMaxIn = bz::kRowsMaxIn, kMaxWide = bz::kRowsMaxColumns, kMaxLast = bz::kRowsMaxColumns;
constexpr int kBeyond = 1 << 30;  // an offset behind any operand

__host__ __device__ constexpr int up(int v, int to) { return (v + to - 1) / to * to; }

// How a layer's waves share it: blocks of 64 outputs, and of each block's K slices of whole groups.  (Made on the host: a kernel this
// short would spend as long on the divisions as on a layer.)
struct Split {
  int chunks, blocks, slices, groups;  // groups: of a slice
  int per_block;                       // 2^16 / blocks, rounded up: wave / blocks is wave * per_block / 2^16
  Split() = default;
  Split(int k, int n)
      : chunks((k + 3) / 4), blocks((n + 63) / 64), slices(kWaves / blocks), groups(((chunks + slices - 1) / slices + kGroup - 1) / kGroup),
        per_block(65535 / blocks + 1) {}
};

// Weights as the lanes take them: block by block of 64 outputs (the last of what is left), chunk by chunk of 16 bytes of inputs, an output's
// 16 bytes after the other's; zeros behind K.
__global__ __launch_bounds__(256) void bz_fc_rows_pack_kernel(const float* __restrict__ w, float4* __restrict__ out, int k, int n, int64_t sk, int64_t sn, int units) {
  const int u = blockIdx.x * 256 + threadIdx.x;
  if (u >= units) return;
  const int chunks = (k + 3) / 4, block = u / (64 * chunks), width = min(64, n - block * 64);
  const int c = (u - block * 64 * chunks) / width, o = block * 64 + (u - block * 64 * chunks) % width;
  float v[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = c * 4 + i < k ? w[(c * 4 + i) * sk + o * sn] : 0.f;
  out[u] = make_float4(v[0], v[1], v[2], v[3]);
}

// LDS, in bytes: rows of operands, 16 bytes further apart than whole groups, so that four rows' reads of one chunk are on different
// banks; the waves' sums, lane by lane; parameters
struct Layout {
  int pitch1, pitch2, x2, sums, params1, params2, head_w, all;
  Layout() = default;
  constexpr Layout(int k, int n1, int n2, int hn) : pitch1(), pitch2(), x2(), sums(), params1(), params2(), head_w(), all() {
    pitch1 = up((k + 3) / 4, kGroup) * 16 + 16;
    pitch2 = up((n1 + 3) / 4, kGroup) * 16 + 16;
    x2 = kRows * pitch1;
    sums = x2 + kRows * pitch2;
    params1 = sums + kThreads * 16;
    params2 = params1 + 4 * n1 * 4;
    head_w = params2 + 4 * n2 * 4;
    all = head_w + hn * kMaxLast * 4;
  }
};

static_assert(Layout(kMaxIn, kMaxWide, kMaxLast, kSkinnyMaxN).all <= 64 * 1024, "what a launch gets without asking for more");
static_assert(kMaxWide <= kWaves / 2 * 64 && kMaxLast <= kWaves / 2 * 64, "eight, four or two slices of K");

// what the kernel's first loads need comes first, as plain arguments (they are in registers when a wave starts); the rest
struct Finish {
  Layout at;
  Split by2;
  Epilogue ep1, ep2;
  HeadArgs head;
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)bytes, 0x00020000);
}

// a column's parameters: beta * bias, then as apply_act_regs takes them.  (What is not there is asked for at `some` address and dropped:
// a load under a branch would make later waits longer.)
struct Column {
  float bias, p0, p1, p2;
  __device__ __forceinline__ void ask(const Epilogue& ep, int n, const float* some) {
    const int col = min((int)threadIdx.x, n - 1);
    bias = (ep.bias_rows != 0 ? ep.bias : some)[ep.bias_rows != 0 ? col : 0];
    p0 = (ep.p0 != nullptr ? ep.p0 : some)[ep.p0 == nullptr || ep.act_size == 1 ? 0 : col];
    p1 = (ep.p1 != nullptr ? ep.p1 : some)[ep.p1 != nullptr ? col : 0];
    p2 = (ep.p2 != nullptr ? ep.p2 : some)[ep.p2 != nullptr ? col : 0];
  }
  __device__ __forceinline__ void put(const Epilogue& ep, int n, float* to) const {
    if ((int)threadIdx.x < n) *(float4*)(to + threadIdx.x * 4) = make_float4(ep.bias_rows != 0 ? ep.beta * bias : 0.f, p0, p1, p2);
  }
};

// output `col` of row `row` from the waves' sums
__device__ __forceinline__ float finished(const Epilogue& ep, const float* params, const Split& by, int row, int col, const float* sums) {
  const float* of = sums + (col / 4 * 4 + row) * 4 + col % 4;  // (block by block of 64 lanes, a lane's four outputs of row lane % 4)
  const int next = by.blocks * 256;
  const float4 p = *(const float4*)(params + col * 4);
  float sum;
  if (by.slices == 8)
    sum = ((of[0] + of[next]) + (of[2 * next] + of[3 * next])) + ((of[4 * next] + of[5 * next]) + (of[6 * next] + of[7 * next]));
  else if (by.slices == 4)
    sum = (of[0] + of[next]) + (of[2 * next] + of[3 * next]);
  else
    sum = of[0] + of[next];
  return apply_act_regs(fmaf(ep.alpha, sum, p.x), ep, p.y, p.z, p.w);
}

// A wave's share of a layer's weights
struct Share {
  __amdgpu_buffer_rsrc_t from;  // the share
  int lane, step;               // the lane's bytes of the first chunk (or beyond), from one chunk to the next
  int first, groups;            // the share's first chunk, its groups
  __device__ __forceinline__ Share(const char* w, const Split& by, int n, int wave) {
    const int slice = wave * by.per_block >> 16, block = wave - slice * by.blocks, width = min(64, n - block * 64), l = threadIdx.x & 63;
    first = slice * by.groups * kGroup;
    const int mine = slice < by.slices ? max(0, min(by.groups * kGroup, by.chunks - first)) : 0;  // chunks
    groups = (mine + kGroup - 1) / kGroup;
    step = width * 16;
    lane = l < width ? l * 16 : kBeyond;
    from = buffer_of(w + (block * 64 * by.chunks + first * width) * 16, (uint32_t)(mine * step));
  }
  // (what is behind the share reads as zeros)
  __device__ __forceinline__ void ask(uint4 (&w)[kGroup], int group) const {
    int at = lane + group * kGroup * step;
#pragma unroll
    for (int i = 0; i < kGroup; ++i) {
      const auto v = __builtin_amdgcn_raw_buffer_load_b128(from, at, 0, 0);
      w[i] = *(const uint4*)&v;
      at += step;
    }
    __builtin_amdgcn_sched_barrier(0);
  }
};

// sixteen blocks of 4 outputs x 4 rows: lane l has 16 bytes of output l in w and of row l % 4 in x; a block's sums of row l % 4 are in lane l
__device__ __forceinline__ void mma4(const uint4& w, const uint4& x, floatx4 (&acc)[4]) {
  acc[0] = __builtin_amdgcn_mfma_f32_4x4x1f32(__uint_as_float(w.x), __uint_as_float(x.x), acc[0], 0, 0, 0);
  acc[1] = __builtin_amdgcn_mfma_f32_4x4x1f32(__uint_as_float(w.y), __uint_as_float(x.y), acc[1], 0, 0, 0);
  acc[2] = __builtin_amdgcn_mfma_f32_4x4x1f32(__uint_as_float(w.z), __uint_as_float(x.z), acc[2], 0, 0, 0);
  acc[3] = __builtin_amdgcn_mfma_f32_4x4x1f32(__uint_as_float(w.w), __uint_as_float(x.w), acc[3], 0, 0, 0);
}

// The wave's sums of a layer, whose first kRing groups are on their way; `then` asks for others behind the layer's own
template <typename Then>
__device__ __forceinline__ void multiply(uint4 (&w)[kRing][kGroup], const Share& of, const char* x, int pitch, floatx4* sums, const Then& then) {
  const char* row = x + (threadIdx.x % kRows) * pitch + of.first * 16;
  // A group has sums of its own, four an output, which are added to the output's: sums over all of K that one float takes up one
  // product after the other were up to 1.4 times as far off 64 bits as the launches that this one stands for (771 -> 129 -> 65 -> 2).
  floatx4 all = {0.f, 0.f, 0.f, 0.f};
  auto one = [&](int slot, int group) {
    if (group >= of.groups) return;
    uint4 f[kGroup];
#pragma unroll
    for (int i = 0; i < kGroup; ++i) f[i] = *(const uint4*)(row + (slot * kGroup + i) * 16);
    floatx4 acc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < kGroup; ++i) mma4(w[slot][i], f[i], acc);
    all += (acc[0] + acc[1]) + (acc[2] + acc[3]);
  };
  int g = 0;
  for (; g + kRing < of.groups; g += kRing) {
#pragma unroll
    for (int i = 0; i < kRing; ++i) {
      one(i, g + i);
      of.ask(w[i], g + i + kRing);
    }
    row += kRing * kGroup * 16;
  }
#pragma unroll
  for (int i = 0; i < kRing; ++i) {
    one(i, g + i);
    then(w[i], i);
  }
  sums[threadIdx.x] = all;
}

// a workgroup's rows to LDS, a quarter of the threads each, at any alignment of their elements; zeros behind K and for rows that are not there
struct Input {
  static constexpr int kEach = up(kMaxIn / 4, kPerRow) / kPerRow;
  uint4 q[kEach];
  __device__ __forceinline__ void ask(const float* x, int64_t row, bool there, int k) {
    const auto from = buffer_of(x + (there ? row : 0), there ? (uint32_t)k * 4u : 0u);
    const int c = threadIdx.x % kPerRow;
#pragma unroll
    for (int i = 0; i < kEach; ++i) {
      const auto v = __builtin_amdgcn_raw_buffer_load_b128(from, (c + i * kPerRow) * 16, 0, 0);
      q[i] = *(const uint4*)&v;
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  __device__ __forceinline__ void put(char* to, int bytes, int k) {
    const int c = threadIdx.x % kPerRow;
#pragma unroll
    for (int i = 0; i < kEach; ++i) {
      const int at = c + i * kPerRow;
      if (at * 4 < k && at * 4 + 4 > k) {  // (the chunk that K ends in)
        if (at * 4 + 1 >= k) q[i].y = 0;
        if (at * 4 + 2 >= k) q[i].z = 0;
        q[i].w = 0;
      }
      if (at * 16 < bytes) *(uint4*)(to + at * 16) = q[i];
    }
  }
};

// HN: outputs the skinny layer's code is unrolled for.  rows: of a workgroup.  by1: the first layer's.
template <int HN>
__global__ __launch_bounds__(kThreads) void bz_fc_rows_kernel(const float* x, const char* w1_, int lda, int m, int k, int n1, int rows, int chunks, int blocks,
                                                              int slices, int groups, int per_block, const char* w2_, int n2, const Finish f) {
  extern __shared__ __align__(16) char lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x & 63;
  const int m0 = blockIdx.x * rows, here = min(rows, m - m0), r = wave / (kWaves / kRows), c = threadIdx.x % kPerRow;
  Input in;
  in.ask(x, (int64_t)(m0 + r) * lda, r < here, k);
  Split by1;
  by1.chunks = chunks;
  by1.blocks = blocks;
  by1.slices = slices;
  by1.groups = groups;
  by1.per_block = per_block;
  const Share of1(w1_, by1, n1, wave);
  uint4 w[kRing][kGroup];
#pragma unroll
  for (int i = 0; i < kRing; ++i) of1.ask(w[i], i);

  // the columns' parameters and the skinny layer's weights, whose addresses are still on their way
  const Layout& at = f.at;
  float *sums = (float*)(lds + at.sums), *params1 = (float*)(lds + at.params1), *params2 = (float*)(lds + at.params2), *head_w = (float*)(lds + at.head_w);
  HeadBias<HN> hbias(f.head);
  Column col1, col2;
  col1.ask(f.ep1, n1, (const float*)w1_);
  col2.ask(f.ep2, n2, (const float*)w1_);
  constexpr int kHeadPer = HN * kMaxLast / kThreads;
  float hw[kHeadPer];
#pragma unroll
  for (int i = 0; i < kHeadPer; ++i) {
    const int j = (threadIdx.x + i * kThreads) / kMaxLast, hc = threadIdx.x % kMaxLast;
    hw[i] = ((const float*)f.head.w)[min(j, f.head.n - 1) * (int)f.head.ldw + min(hc, n2 - 1)];
  }
  __builtin_amdgcn_sched_barrier(0);
  in.put(lds + r * at.pitch1, at.pitch1 - 16, k);
  __syncthreads();
  const Share of2(w2_, f.by2, n2, wave);
  multiply(w, of1, lds, at.pitch1, (floatx4*)sums, [&](uint4 (&slot)[kGroup], int group) { of2.ask(slot, group); });
  col1.put(f.ep1, n1, params1);
  col2.put(f.ep2, n2, params2);
#pragma unroll
  for (int i = 0; i < kHeadPer; ++i) head_w[threadIdx.x + i * kThreads] = hw[i];
  __syncthreads();
  if (r < rows)
    for (int o = c; o * 4 < at.pitch2 - 16; o += kPerRow)
      ((float*)(lds + at.x2 + r * at.pitch2))[o] = o < n1 ? finished(f.ep1, params1, by1, r, o, sums) : 0.f;
  __syncthreads();
  multiply(w, of2, lds + at.x2, at.pitch2, (floatx4*)sums, [](uint4 (&)[kGroup], int) {});
  __syncthreads();
  // a wave a row: the second layer's activation and the skinny layer
  if (wave < here) {
    float dot[HN];
#pragma unroll
    for (int j = 0; j < HN; ++j) dot[j] = 0.f;
    for (int o = lane; o < n2; o += 64) {
      const float v = finished(f.ep2, params2, f.by2, wave, o, sums);
#pragma unroll
      for (int j = 0; j < HN; ++j) dot[j] = fmaf(v, head_w[j * kMaxLast + o], dot[j]);
    }
#pragma unroll
    for (int j = 0; j < HN; ++j) dot[j] = group_sum<64>(dot[j]);
    if (lane == 0) head_finish(f.head, hbias, m0 + wave, dot);
  }
}

struct Rows {
  const float* x;
  const char *w1, *w2;
  int lda, m, k, n1, n2, rows;
};

template <int HN>
int launch(const Rows& a, Finish& f, hipStream_t st) {
  const Split by1(a.k, a.n1);
  f.by2 = Split(a.n1, a.n2);
  f.at = Layout(a.k, a.n1, a.n2, HN);
  hipLaunchKernelGGL((bz_fc_rows_kernel<HN>), dim3((a.m + a.rows - 1) / a.rows), dim3(kThreads), f.at.all, st, a.x, a.w1, a.lda, a.m, a.k, a.n1, a.rows,
                     by1.chunks, by1.blocks, by1.slices, by1.groups, by1.per_block, a.w2, a.n2, f);
  BZ_LAUNCH_OK("bz_fc_rows_kernel");
  return BZ_OK;
}

}  // namespace

size_t bz::fc_rows_weight_bytes(int64_t k, int64_t n) { return (size_t)n * ((k + 3) / 4) * 16; }

int bz::fc_rows_pack(const void* w, bool transposed, int k, int n, void* out, bz_stream_t stream) {
  const int units = (int)(fc_rows_weight_bytes(k, n) / 16);
  hipLaunchKernelGGL(bz_fc_rows_pack_kernel, dim3((units + 255) / 256), dim3(256), 0, bz::as_stream(stream), (const float*)w, (float4*)out, k, n,
                     transposed ? (int64_t)1 : (int64_t)n, transposed ? (int64_t)k : (int64_t)1, units);
  BZ_LAUNCH_OK("bz_fc_rows_pack_kernel");
  return BZ_OK;
}

int bz::fc_rows(const bz_fc_desc& d, void* copy, bz_stream_t stream) {
  BZ_REQUIRE(d.next != nullptr, "rows: no second layer");
  const bz_fc_next& x = *d.next;
  auto plain = [](int act) { return act == BZ_ACT_NONE || act == BZ_ACT_PRELU || act == BZ_ACT_DICE || act == BZ_ACT_LEAKY_RELU || act == BZ_ACT_SIGMOID; };
  if (d.in_dtype != BZ_F32 || d.out_dtype != d.in_dtype || !fc_rows_takes(d.k, d.n, x.n) || d.y != nullptr || x.y != nullptr ||
      d.head_n < 1 || d.head_n > kSkinnyMaxN || d.n_split != 0 || d.a_pieces != nullptr || d.bias_rows > 1 || !plain(d.act) || !plain(x.act))
    return bz::fail(BZ_ENOTSUP, "rows: a shape or form outside the kernel's");
  BZ_REQUIRE(d.a != nullptr && d.w != nullptr && x.w != nullptr && d.head_w != nullptr && d.head_y != nullptr && d.lda >= d.k && d.head_ldw >= x.n &&
                 d.head_ldy >= d.head_n,
             "rows: null operand or a leading dimension below its row");
  BZ_REQUIRE(d.bias_rows == 0 || d.bias != nullptr, "rows: bias_rows=%d without bias", d.bias_rows);
  BZ_REQUIRE(d.act != BZ_ACT_PRELU || (d.act_p0 && (d.act_size == 1 || d.act_size == d.n)), "rows: PRelu slope size %d", d.act_size);
  BZ_REQUIRE(d.act != BZ_ACT_DICE || (d.act_p0 && d.act_p1 && d.act_p2), "rows: Dice needs gamma, mean and var");
  BZ_REQUIRE(x.act != BZ_ACT_PRELU || (x.act_p0 && (x.act_size == 1 || x.act_size == x.n)), "rows: PRelu slope size %d", x.act_size);
  BZ_REQUIRE(x.act != BZ_ACT_DICE || (x.act_p0 && x.act_p1 && x.act_p2), "rows: Dice needs gamma, mean and var");
  // (offsets within a workgroup's rows are 32-bit)
  if (d.lda > 1 << 20 || d.head_ldw > 1 << 20) return bz::fail(BZ_ENOTSUP, "rows: rows further apart than the kernel's offsets reach");
  BZ_REQUIRE(d.m >= 0, "rows: %lld rows", (long long)d.m);
  if (d.m == 0) return BZ_OK;
  Rows a = {};
  a.x = (const float*)d.a;
  a.w1 = (const char*)d.w;
  a.w2 = (const char*)x.w;
  a.lda = (int)d.lda;
  a.m = d.m;
  a.k = d.k;
  a.n1 = d.n;
  a.n2 = x.n;
  // (up to 128 workgroups of one row each; beyond, the weights that every workgroup pulls would cost others more than rows cost it.  201 rows of
  // 192 -> 200 -> 80 and 468 -> 256 -> 100, one row a workgroup and four: a lone request 31.1 and 32.5, 37.6 and 38.2 us, a pass on eight
  // serving threads 5.6 and 5.3, 6.9 and 6.3)
  a.rows = (int)((d.m + 127) / 128 < kRows ? (d.m + 127) / 128 : kRows);
  Finish f = {};
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
  return head_unroll(d.head_n) == 2 ? launch<2>(a, f, st) : launch<kSkinnyMaxN>(a, f, st);
}
