// feed_pack.h -- what of a fed input need not cross the link: the upper halves of ids that fit 32 bits, and all but one of
// values that are all the same (a multi-hot feature's weights are mostly 1).
//
// Both functions look at their input once, block by block, and stop in front of the first block that does not have that form: the
// caller stages the rest as it is.  What it costs where nothing has it is a look at the first few words.
#pragma once

#include <immintrin.h>
#include <stdint.h>
#include <string.h>

#include <algorithm>

namespace blaze {

constexpr size_t kPackBlock = 1024;  // words looked at before the answer counts: 8 KB, which stay in L1 for the copy of a refused block

// What is looked at is asked for this many bytes ahead: the hardware's own prefetching ends with each 4 KB page.  Requests of 5.6 MB
// that take turns and no longer fit the caches, us to pack one: without 145, 2 KB 136, 4 KB 126, 8 KB 115, 16 KB 120; from the caches 61..64
// either way.  (A plain copy in blocks with the same hints was no faster, 165 to 185..210.)
constexpr int kPrefetch = 8 << 10;

// Copies the lower halves of n words and returns the bits that any upper half has.
inline uint64_t CopyLow32Plain(uint32_t* dst, const uint64_t* src, size_t n) {
  uint64_t any = 0;
  for (size_t i = 0; i < n; ++i) {
    uint64_t v;
    memcpy(&v, (const char*)src + 8 * i, 8);  // (the caller's buffer need not be aligned)
    any |= v;
    dst[i] = (uint32_t)v;
  }
  return any >> 32;
}

__attribute__((target("avx2"))) inline uint64_t CopyLow32Avx2(uint32_t* dst, const uint64_t* src, size_t n) {
  __m256i any = _mm256_setzero_si256();
  size_t i = 0;
  for (; i + 8 <= n; i += 8) {
    _mm_prefetch((const char*)(src + i) + kPrefetch, _MM_HINT_T0);
    const __m256i a = _mm256_loadu_si256((const __m256i*)(src + i)), b = _mm256_loadu_si256((const __m256i*)(src + i + 4));
    any = _mm256_or_si256(any, _mm256_or_si256(a, b));
    const __m256 low = _mm256_shuffle_ps(_mm256_castsi256_ps(a), _mm256_castsi256_ps(b), 0x88);  // words 0 1 4 5 2 3 6 7
    _mm256_storeu_si256((__m256i*)(dst + i), _mm256_permute4x64_epi64(_mm256_castps_si256(low), 0xd8));
  }
  const bool fits = _mm256_testz_si256(any, _mm256_set1_epi64x((long long)0xffffffff00000000ull));
  return (fits ? 0 : 1) | CopyLow32Plain(dst + i, src + i, n - i);
}

// How many of the n words at src have an upper half of zero, up to the end of a block: their lower halves are at dst, and up to a
// block behind them at dst has been written over.
inline size_t PackLow32(uint32_t* dst, const uint64_t* src, size_t n) {
  static const bool avx2 = __builtin_cpu_supports("avx2");
  uint32_t first[8];
  if (CopyLow32Plain(first, src, std::min<size_t>(n, 8)) != 0) return 0;
  for (size_t i = 0; i < n; i += kPackBlock) {
    const size_t len = std::min(kPackBlock, n - i);
    if ((avx2 ? CopyLow32Avx2(dst + i, src + i, len) : CopyLow32Plain(dst + i, src + i, len)) != 0) return i;
  }
  return n;
}

// How many of the n 32-bit words at src are `word`, up to the end of a block.
inline size_t CountSame32(const void* src, size_t n, uint32_t word) {
  const char* p = (const char*)src;
  for (size_t i = 0; i < n; i += kPackBlock) {
    const size_t end = std::min(i + kPackBlock, n);
    const __m128i w = _mm_set1_epi32((int)word);
    size_t k = i;
    for (; k + 16 <= end; k += 16) {
      const __m128i* v = (const __m128i*)(p + 4 * k);
      _mm_prefetch((const char*)v + kPrefetch, _MM_HINT_T0);
      const __m128i a = _mm_and_si128(_mm_cmpeq_epi32(_mm_loadu_si128(v), w), _mm_cmpeq_epi32(_mm_loadu_si128(v + 1), w));
      const __m128i b = _mm_and_si128(_mm_cmpeq_epi32(_mm_loadu_si128(v + 2), w), _mm_cmpeq_epi32(_mm_loadu_si128(v + 3), w));
      if (_mm_movemask_epi8(_mm_and_si128(a, b)) != 0xffff) return i;
    }
    for (; k < end; ++k) {
      uint32_t v;
      memcpy(&v, p + 4 * k, 4);
      if (v != word) return i;
    }
  }
  return n;
}

}  // namespace blaze
