// feed.hip -- request inputs from pinned host memory to where the net reads them, for gfx950.
//
// Stands in for the cudaMemcpyAsync calls of the reference's Feed (blaze/api/cpp_api/predictor_impl.cc:110-138).  A
// request brings tens of inputs; most are staged side by side and land side by side (one contiguous range), a few live
// inside a Concat's output, where their rows are a pitch apart.  One kernel reads the pinned memory over PCIe and writes
// both kinds in place.
//
// What bounds it: the link (57 GB/s), or at small sizes one trip over it.  64 bytes a lane are requested before any is
// stored, so a 1 MB launch has all its reads on the way at once.  The strided rows are what this kernel is for: the copy
// engine takes them row by row (hipMemcpy2DAsync of 300 rows of 26 bytes: 2.1 ms; here 4 us), and a contiguous copy
// beside them would cost another launch and a hand-over between engines.
#include <hip/hip_runtime.h>

#include <stdint.h>

#include "bz_common.h"

namespace {

constexpr int kFeedThreads = 256;
constexpr int kFeedUnroll = 4;
constexpr int kFeedSpan = kFeedThreads * kFeedUnroll;  // units (16 bytes of the range, or `unit` bytes of a piece) a workgroup

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

template <typename U>
__device__ __forceinline__ void feed_rows(const bz_feed_rows& p, int64_t first) {
  const uint64_t per_row = (uint64_t)p.row_bytes / sizeof(U), total = (uint64_t)p.rows * per_row;
  U v[kFeedUnroll];
  uint64_t row[kFeedUnroll], col[kFeedUnroll];
#pragma unroll
  for (int k = 0; k < kFeedUnroll; ++k) {
    const uint64_t i = (uint64_t)first + k * kFeedThreads + threadIdx.x;
    const uint64_t at = i < total ? i : total - 1;
    // (a 64-bit division is some 150 instructions: taken only by inputs of 2^32 units and more)
    row[k] = total <= 0xffffffffull ? (uint64_t)((uint32_t)at / (uint32_t)per_row) : at / per_row;
    col[k] = at - row[k] * per_row;
    v[k] = *(const U*)((const char*)p.src + row[k] * (uint64_t)p.src_pitch + col[k] * sizeof(U));
  }
#pragma unroll
  for (int k = 0; k < kFeedUnroll; ++k)
    if ((uint64_t)first + k * kFeedThreads + threadIdx.x < total)
      *(U*)((char*)p.dst + row[k] * (uint64_t)p.dst_pitch + col[k] * sizeof(U)) = v[k];
}

__global__ __launch_bounds__(kFeedThreads) void bz_feed_kernel(const FeedArgs a) {
  const int wg = (int)blockIdx.x;
  if (wg < a.range_wg) {
    const uint4* src = (const uint4*)a.src;
    uint4* dst = (uint4*)a.dst;
    const int64_t i0 = (int64_t)wg * kFeedSpan + threadIdx.x;
    uint4 v[kFeedUnroll];
#pragma unroll
    for (int k = 0; k < kFeedUnroll; ++k) {
      const int64_t i = i0 + k * kFeedThreads;
      v[k] = src[i < a.chunks ? i : a.chunks - 1];
    }
#pragma unroll
    for (int k = 0; k < kFeedUnroll; ++k) {
      const int64_t i = i0 + k * kFeedThreads;
      if (i < a.chunks) dst[i] = v[k];
    }
    return;
  }
  int q = 0;
  while (q < a.n - 1 && wg >= a.wg_end[q]) ++q;  // (uniform; at most BZ_FEED_MAX_ROWS steps)
  const bz_feed_rows p = a.p[q];
  const int64_t first = (int64_t)(wg - (q == 0 ? a.range_wg : a.wg_end[q - 1])) * kFeedSpan;
  switch (a.unit[q]) {
    case 16: feed_rows<uint4>(p, first); break;
    case 8: feed_rows<uint2>(p, first); break;
    case 4: feed_rows<uint32_t>(p, first); break;
    case 2: feed_rows<uint16_t>(p, first); break;
    default: feed_rows<uint8_t>(p, first); break;
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
  int64_t wg = (a.chunks + kFeedSpan - 1) / kFeedSpan;
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
    wg += (p.rows * (p.row_bytes / unit) + kFeedSpan - 1) / kFeedSpan;
    BZ_REQUIRE(wg < (1ll << 30), "bz_feed: piece %d makes too many workgroups", i);
    a.p[a.n] = p;
    a.unit[a.n] = unit;
    a.wg_end[a.n] = (int)wg;
    ++a.n;
  }
  if (wg == 0) return BZ_OK;
  hipLaunchKernelGGL(bz_feed_kernel, dim3((int)wg), dim3(kFeedThreads), 0, bz::as_stream(stream), a);
  BZ_LAUNCH_OK("bz_feed_kernel");
  return BZ_OK;
}
