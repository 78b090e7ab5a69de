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

struct FeedArgs {
  const char* src;
  char* dst;
  int64_t chunks;  // 16-byte chunks of the contiguous range
  int range_wg;    // workgroups that copy it
  int n;
  bz_feed_rows p[BZ_FEED_MAX_ROWS];
  int unit[BZ_FEED_MAX_ROWS];    // widest power of two (<= 16) that divides addresses, pitches and row length
  int wg_end[BZ_FEED_MAX_ROWS];  // workgroups of the range and of the pieces up to and including this one
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
__global__ __launch_bounds__(kFeedThreads) void bz_feed_kernel(const FeedArgs a) {
  const int wg = (int)blockIdx.x;
  if (wg < a.range_wg) {
    const uint4* src = (const uint4*)a.src;
    uint4* dst = (uint4*)a.dst;
    const int64_t i0 = (int64_t)wg * (kFeedThreads * UNITS) + threadIdx.x;
    uint4 v[UNITS];
#pragma unroll
    for (int k = 0; k < UNITS; ++k) {
      const int64_t i = i0 + k * kFeedThreads;
      v[k] = src[i < a.chunks ? i : a.chunks - 1];
    }
#pragma unroll
    for (int k = 0; k < UNITS; ++k) {
      const int64_t i = i0 + k * kFeedThreads;
      if (i < a.chunks) dst[i] = v[k];
    }
    return;
  }
  int q = 0;
  while (q < a.n - 1 && wg >= a.wg_end[q]) ++q;  // (uniform; at most BZ_FEED_MAX_ROWS steps)
  const bz_feed_rows p = a.p[q];
  const int64_t first = (int64_t)(wg - (q == 0 ? a.range_wg : a.wg_end[q - 1])) * (kFeedThreads * UNITS);
  switch (a.unit[q]) {
    case 16: feed_rows<uint4, UNITS>(p, first); break;
    case 8: feed_rows<uint2, UNITS>(p, first); break;
    case 4: feed_rows<uint32_t, UNITS>(p, first); break;
    case 2: feed_rows<uint16_t, UNITS>(p, first); break;
    default: feed_rows<uint8_t, UNITS>(p, first); break;
  }
}

}  // namespace

extern "C" int bz_feed(const void* src, void* dst, int64_t bytes, const bz_feed_rows* rows, int n_rows, bz_stream_t stream) {
  BZ_REQUIRE(bytes >= 0 && n_rows >= 0 && n_rows <= BZ_FEED_MAX_ROWS && (n_rows == 0 || rows != nullptr),
             "bz_feed: bytes=%lld n_rows=%d (at most %d)", (long long)bytes, n_rows, BZ_FEED_MAX_ROWS);
  BZ_REQUIRE(bytes == 0 || (src != nullptr && dst != nullptr && bytes % 16 == 0 && (((uintptr_t)src | (uintptr_t)dst) & 15) == 0),
             "bz_feed: the contiguous range needs 16-byte aligned addresses and a multiple of 16 bytes (%lld)", (long long)bytes);
  FeedArgs a = {};
  a.src = (const char*)src;
  a.dst = (char*)dst;
  a.chunks = bytes / 16;
  int64_t all = bytes;
  for (int i = 0; i < n_rows; ++i) {
    const bz_feed_rows& p = rows[i];
    if (p.rows > 0 && p.row_bytes > 0) all += p.rows < (1ll << 40) / p.row_bytes ? p.rows * p.row_bytes : 1ll << 40;
  }
  const int units = all <= kFeedOneUnit ? 1 : all <= (1ll << 30) ? 2 : 4;  // (four for the sake of the grid's size)
  const int64_t span = kFeedThreads * units;
  int64_t wg = (a.chunks + span - 1) / span;
  BZ_REQUIRE(wg < (1ll << 30), "bz_feed: %lld bytes make too many workgroups", (long long)bytes);
  a.range_wg = (int)wg;
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
    a.wg_end[a.n] = (int)wg;
    ++a.n;
  }
  if (wg == 0) return BZ_OK;
  hipLaunchKernelGGL(units == 1 ? bz_feed_kernel<1> : units == 2 ? bz_feed_kernel<2> : bz_feed_kernel<4>, dim3((int)wg), dim3(kFeedThreads), 0, bz::as_stream(stream), a);
  BZ_LAUNCH_OK("bz_feed_kernel");
  return BZ_OK;
}
