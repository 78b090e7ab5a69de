// feed.hip -- request inputs from pinned host memory to where the net reads them, for gfx950.
//
// Stands in for the cudaMemcpyAsync calls of the reference's Feed (blaze/api/cpp_api/predictor_impl.cc:110-138).  A
// request brings tens of inputs; most are staged side by side and land side by side (one contiguous range), a few live
// inside a Concat's output, where their rows are a pitch apart.  One kernel reads the pinned memory over PCIe and writes
// both kinds in place.
//
// What bounds it: the link (57 GB/s), or at small sizes one trip over it.  The strided rows are what this kernel is for: the copy
// engine takes them row by row (hipMemcpy2DAsync of 300 rows of 26 bytes: 2.1 ms; here 4 us), and a contiguous copy
// beside them would cost another launch and a hand-over between engines.
#include <hip/hip_runtime.h>

#include <stdint.h>

#include "bz_common.h"

namespace {

// Units (16 bytes of the range, or `unit` bytes of a piece) a lane asks for before it stores any: one in a small launch, whose
// requests then leave from as many CUs as there are 4 KB; two where the link is full anyway and half the workgroups drain
// sooner.  us from the call to the end of the wait for it, with 1, 2, 4 (an empty kernel 11.6): 4 KB 12.9 15.2 14.9, 64 KB 13.9
// 16.1 16.0, 256 KB 17.9 18.9 19.1, 320 KB 19.6 19.8, 384 KB 21.3 20.9, 512 KB 24.5 23.2, 1 MB 37.4 32.6 35.4, 2 MB 61.7 53.6
// 57.8, 2048 rows of 128 bytes 18.6 19.8 19.8.
constexpr int kFeedThreads = 256;
constexpr int64_t kFeedOneUnit = 320 << 10;  // bytes up to which a lane asks for one

// 16-byte stores of a lane in a range of one repeated word, which reads nothing
constexpr int kSameUnits = 4;

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));  // (arrays of HIP's uint4 ended up in LDS, one load waited for at a time)

struct FeedRange {
  const char* src;
  char* dst;
  int64_t chunks;  // 16-byte chunks at dst
  int32_t form;
  uint32_t word;
  int32_t wg_begin;  // workgroups of the ranges before it
};

// N: ranges that the launch has room for
template <int N>
struct FeedArgs {
  FeedRange r[N];
  int wg_end[N];  // workgroups of the ranges up to and including this one
  int n;
  bz_feed_rows p[BZ_FEED_MAX_ROWS];
  int unit[BZ_FEED_MAX_ROWS];     // widest power of two (<= 16) that divides addresses, pitches and row length
  int row_end[BZ_FEED_MAX_ROWS];  // workgroups of the ranges and of the strided pieces up to and including this one
};

template <typename U, int UNITS>
__device__ __forceinline__ void feed_rows(const bz_feed_rows& p, int64_t first) {
  const uint64_t per_row = (uint64_t)p.row_bytes / sizeof(U), total = (uint64_t)p.rows * per_row;
  // where the workgroup's first unit lies: one 64-bit division for all lanes
  const uint64_t row0 = (uint64_t)first / per_row, col0 = (uint64_t)first - row0 * per_row;
  U v[UNITS];
  char* to[UNITS];
#pragma unroll
  for (int k = 0; k < UNITS; ++k) {
    const uint32_t i = k * kFeedThreads + threadIdx.x;
    const uint32_t ahead = (uint64_t)first + i < total ? i : (uint32_t)(total - 1 - (uint64_t)first);  // (first is below total)
    const uint64_t at = col0 + ahead;
    // (a row of 2^31 units and more ends at most once on the way)
    const uint32_t rows = per_row < (1u << 31) ? (uint32_t)at / (uint32_t)per_row : at >= per_row;
    const uint64_t row = row0 + rows, col = at - rows * per_row;
    v[k] = *(const U*)((const char*)p.src + row * (uint64_t)p.src_pitch + col * sizeof(U));
    to[k] = (char*)p.dst + row * (uint64_t)p.dst_pitch + col * sizeof(U);
  }
#pragma unroll
  for (int k = 0; k < UNITS; ++k)
    if ((uint64_t)first + k * kFeedThreads + threadIdx.x < total) *(U*)to[k] = v[k];
}

template <int UNITS>
__device__ __forceinline__ void feed_raw(const FeedRange& r, int wg) {
  const u32x4* src = (const u32x4*)r.src;
  u32x4* dst = (u32x4*)r.dst;
  const int64_t i0 = (int64_t)wg * (kFeedThreads * UNITS) + (int)threadIdx.x;
  u32x4 v[UNITS];
#pragma unroll
  for (int k = 0; k < UNITS; ++k) v[k] = src[min(i0 + k * kFeedThreads, r.chunks - 1)];
#pragma unroll
  for (int k = 0; k < UNITS; ++k)
    if (i0 + k * kFeedThreads < r.chunks) dst[i0 + k * kFeedThreads] = v[k];
}

template <int UNITS>
__device__ __forceinline__ void feed_low32(const FeedRange& r, int wg) {
  const u32x4* src = (const u32x4*)r.src;
  u32x4* dst = (u32x4*)r.dst;
  const int64_t units = (r.chunks + 1) >> 1;  // 16 bytes at the source are 32 here
  const int64_t i0 = (int64_t)wg * (kFeedThreads * UNITS) + (int)threadIdx.x;
  u32x4 v[UNITS];
#pragma unroll
  for (int k = 0; k < UNITS; ++k) v[k] = src[min(i0 + k * kFeedThreads, units - 1)];
#pragma unroll
  for (int k = 0; k < UNITS; ++k) {
    const int64_t i = i0 + k * kFeedThreads;
    if (i < units) dst[2 * i] = u32x4{v[k].x, 0, v[k].y, 0};
    if (2 * i + 1 < r.chunks) dst[2 * i + 1] = u32x4{v[k].z, 0, v[k].w, 0};
  }
}

__device__ __forceinline__ void feed_same32(const FeedRange& r, int wg) {
  u32x4* dst = (u32x4*)r.dst;
  const int64_t i0 = (int64_t)wg * (kFeedThreads * kSameUnits) + (int)threadIdx.x;
#pragma unroll
  for (int k = 0; k < kSameUnits; ++k)
    if (i0 + k * kFeedThreads < r.chunks) dst[i0 + k * kFeedThreads] = u32x4{r.word, r.word, r.word, r.word};
}

// (the first four arguments are there when a wave starts: N == 1 reads over the link at once)
template <int UNITS, int N>
__global__ __launch_bounds__(kFeedThreads) void bz_feed_kernel(int range_wg, const char* src, char* dst, int64_t chunks, const FeedArgs<N> a) {
  const int wg = (int)blockIdx.x;
  if (wg < range_wg) {
    if (N == 1) {
      feed_raw<UNITS>({src, dst, chunks, BZ_FEED_RAW, 0, 0}, wg);
      return;
    }
    // which range: every lane brings one, and where it ends, in one trip to the arguments (ranges that are not there end with the last)
    const int lane = min((int)threadIdx.x & (bz::kWave - 1), N - 1);
    const FeedRange mine = a.r[lane];
    const int q = __popcll(__ballot(wg >= a.wg_end[lane]));
    auto of = [&](uint32_t v) { return (uint32_t)__builtin_amdgcn_readlane((int)v, q); };
    auto of64 = [&](uint64_t v) { return (uint64_t)of((uint32_t)(v >> 32)) << 32 | of((uint32_t)v); };
    const FeedRange r = {(const char*)of64((uint64_t)mine.src), (char*)of64((uint64_t)mine.dst), (int64_t)of64((uint64_t)mine.chunks),
                         (int32_t)of((uint32_t)mine.form), of(mine.word), (int32_t)of((uint32_t)mine.wg_begin)};
    if (r.form == BZ_FEED_RAW)
      feed_raw<UNITS>(r, wg - r.wg_begin);
    else if (r.form == BZ_FEED_LOW32)
      feed_low32<UNITS>(r, wg - r.wg_begin);
    else
      feed_same32(r, wg - r.wg_begin);
    return;
  }
  int q = 0;
  while (q < a.n - 1 && wg >= a.row_end[q]) ++q;  // (uniform; at most BZ_FEED_MAX_ROWS steps)
  const bz_feed_rows p = a.p[q];
  const int64_t first = (int64_t)(wg - (q == 0 ? range_wg : a.row_end[q - 1])) * (kFeedThreads * UNITS);
  switch (a.unit[q]) {
    case 16: feed_rows<u32x4, UNITS>(p, first); break;
    case 8: feed_rows<u32x2, UNITS>(p, first); break;
    case 4: feed_rows<uint32_t, UNITS>(p, first); break;
    case 2: feed_rows<uint16_t, UNITS>(p, first); break;
    default: feed_rows<uint8_t, UNITS>(p, first); break;
  }
}

// the arguments from checked pieces, and the launch
template <int N>
int launch_feed(const bz_feed_piece* pieces, int n_pieces, const bz_feed_rows* rows, int n_rows, bz_stream_t stream) {
  FeedArgs<N> a = {};
  int64_t all = 0;  // what is read
  for (int i = 0; i < n_pieces; ++i) all += pieces[i].form == BZ_FEED_RAW ? pieces[i].bytes : pieces[i].form == BZ_FEED_LOW32 ? pieces[i].bytes / 2 : 0;
  for (int i = 0; i < n_rows; ++i) {
    const bz_feed_rows& p = rows[i];
    if (p.rows > 0 && p.row_bytes > 0) all += p.rows < (1ll << 40) / p.row_bytes ? p.rows * p.row_bytes : 1ll << 40;
  }
  const int units = all <= kFeedOneUnit ? 1 : all <= (1ll << 30) ? 2 : 4;  // (four for the sake of the grid's size)
  const int64_t span = kFeedThreads * units;
  int64_t wg = 0;
  int n_ranges = 0;
  for (int i = 0; i < n_pieces; ++i) {
    const bz_feed_piece& p = pieces[i];
    if (p.bytes == 0) continue;
    const int64_t chunks = p.bytes / 16;
    FeedRange& r = a.r[n_ranges];
    r = {(const char*)p.src, (char*)p.dst, chunks, p.form, p.word, (int32_t)wg};
    if (p.form == BZ_FEED_SAME32)
      wg += (chunks + kFeedThreads * kSameUnits - 1) / (kFeedThreads * kSameUnits);
    else
      wg += ((p.form == BZ_FEED_LOW32 ? (chunks + 1) / 2 : chunks) + span - 1) / span;
    BZ_REQUIRE(wg < (1ll << 30), "bz_feed: %lld bytes make too many workgroups", (long long)p.bytes);
    a.wg_end[n_ranges++] = (int)wg;
  }
  const int range_wg = (int)wg;
  for (int i = n_ranges; i < N; ++i) a.wg_end[i] = range_wg;
  for (int i = 0; i < n_rows; ++i) {
    const bz_feed_rows& p = rows[i];
    BZ_REQUIRE(p.rows >= 0 && p.row_bytes >= 0 && p.src_pitch >= p.row_bytes && p.dst_pitch >= p.row_bytes,
               "bz_feed: piece %d of %lld rows of %lld bytes, pitches %lld and %lld", i, (long long)p.rows, (long long)p.row_bytes,
               (long long)p.src_pitch, (long long)p.dst_pitch);
    if (p.rows == 0 || p.row_bytes == 0) continue;
    BZ_REQUIRE(p.src != nullptr && p.dst != nullptr, "bz_feed: piece %d without memory", i);
    const uintptr_t all = (uintptr_t)p.src | (uintptr_t)p.dst | (uintptr_t)p.row_bytes | (uintptr_t)p.src_pitch | (uintptr_t)p.dst_pitch;
    int unit = 16;
    while (all & (uintptr_t)(unit - 1)) unit >>= 1;
    BZ_REQUIRE(p.rows <= (1ll << 40) / p.row_bytes, "bz_feed: piece %d of %lld rows of %lld bytes", i, (long long)p.rows, (long long)p.row_bytes);
    wg += (p.rows * (p.row_bytes / unit) + span - 1) / span;
    BZ_REQUIRE(wg < (1ll << 30), "bz_feed: piece %d makes too many workgroups", i);
    a.p[a.n] = p;
    a.unit[a.n] = unit;
    a.row_end[a.n] = (int)wg;
    ++a.n;
  }
  if (wg == 0) return BZ_OK;
  hipLaunchKernelGGL((units == 1 ? bz_feed_kernel<1, N> : units == 2 ? bz_feed_kernel<2, N> : bz_feed_kernel<4, N>), dim3((int)wg),
                     dim3(kFeedThreads), 0, bz::as_stream(stream), range_wg, a.r[0].src, a.r[0].dst, a.r[0].chunks, a);
  BZ_LAUNCH_OK("bz_feed_kernel");
  return BZ_OK;
}

}  // namespace

extern "C" int bz_feed(const void* src, void* dst, int64_t bytes, const bz_feed_rows* rows, int n_rows, bz_stream_t stream) {
  const bz_feed_piece range = {src, dst, bytes, BZ_FEED_RAW, 0};
  return bz_feed_pieces(&range, 1, rows, n_rows, stream);
}

extern "C" int bz_feed_pieces(const bz_feed_piece* pieces, int n_pieces, const bz_feed_rows* rows, int n_rows, bz_stream_t stream) {
  BZ_REQUIRE(n_rows >= 0 && n_rows <= BZ_FEED_MAX_ROWS && (n_rows == 0 || rows != nullptr), "bz_feed: n_rows=%d (at most %d)", n_rows,
             BZ_FEED_MAX_ROWS);
  BZ_REQUIRE(n_pieces >= 0 && n_pieces <= BZ_FEED_MAX_PIECES && (n_pieces == 0 || pieces != nullptr), "bz_feed: n_pieces=%d (at most %d)", n_pieces,
             BZ_FEED_MAX_PIECES);
  bool one = true;
  for (int i = 0; i < n_pieces; ++i) {
    const bz_feed_piece& p = pieces[i];
    BZ_REQUIRE(p.form == BZ_FEED_RAW || p.form == BZ_FEED_LOW32 || p.form == BZ_FEED_SAME32, "bz_feed: form %d", p.form);
    BZ_REQUIRE(p.bytes >= 0 && p.bytes < (1ll << 44), "bz_feed: %lld bytes make too many workgroups", (long long)p.bytes);
    const bool read = p.form != BZ_FEED_SAME32;
    BZ_REQUIRE(p.bytes == 0 || (p.dst != nullptr && (!read || p.src != nullptr) && p.bytes % 16 == 0 && ((uintptr_t)p.dst & 15) == 0 &&
                                (!read || ((uintptr_t)p.src & 15) == 0)),
               "bz_feed: a contiguous range needs 16-byte aligned addresses and a multiple of 16 bytes (%lld)", (long long)p.bytes);
    one = one && p.form == BZ_FEED_RAW;
  }
  return n_pieces <= 1 && one ? launch_feed<1>(pieces, n_pieces, rows, n_rows, stream)
                              : launch_feed<BZ_FEED_MAX_PIECES>(pieces, n_pieces, rows, n_rows, stream);
}
