// feed_pack.h -- how a request's inputs are staged: in parts, whose transfers start as soon as they are there, and without what need not
// cross the link: the upper halves of ids that fit 32 bits, and all but one of values that are all the same (a multi-hot feature's weights
// are mostly 1).
//
// PackLow32 and CountSame32 look at their input once, block by block, and stop in front of the first block that does not have that form:
// the rest of the input is staged as it is.  What it costs where nothing has it is a look at the first few words, or one block.
#pragma once

#include <immintrin.h>
#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <vector>

#include "blaze_hip.h"

namespace blaze {

constexpr size_t kPackBlock = 256;  // words looked at before the answer counts; the copy of a refused block finds them in L1

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

// A request is moved in parts, each launched as soon as it is staged.  Up to 4 MB the link is what bounds it (the kernel moves
// 47 GB/s and leaves a gap behind each launch, staging runs at 58), so it starts early: 384 KB first, each part half as large
// again as the one before until 1 MB.  Beyond, staging is (35 GB/s, the copies no longer fit the caches between requests), and a
// launch costs the host 2.9 us: even parts of 1 MB or more.  The last part takes what would be left of it below half a part.  us to the end of a
// request among others, even parts of 1 MB or more / these: 0.74 MB 79.3 / 78.5, 1.07 92.8 / 88.5, 1.8 125 / 112, 2.5 115 / 112,
// 3 135 / 127, 4 162 / 158, 4.6 180..191 / 184..194 (not taken), 5.1 203 / 217 (not taken).  (The copy engine moves 57 GB/s, but each copy costs 10 us until
// what follows it on the stream may start: 5 MB in ten parts arrived 230 us after the first byte was staged, in one part behind
// the whole staging 210, through five launches of the kernel 162.)
constexpr size_t kFeedFirst = 384 << 10, kFeedMost = 1 << 20, kFeedLong = 4 << 20;
// An input of this many bytes is staged in the form that crosses in fewest, if one fits: words of 8 bytes, which lose half, and of 4, which lose
// all, in a request that may lose kPackLeast.  Each such input makes a range, and another one of what lies raw behind it (some 0.05 us each), and
// a launch of several ranges takes about half a microsecond longer than one of one.  A launch has room for BZ_FEED_MAX_PIECES: what is left
// of the part is raw then.  us of a request with lists of 8 ids below 2^32 and values of 1, as it is / packed / with keys of 62 bits for ids: 26 lists
// x 128 samples 41.6 / 41.6 / 45.1 and 45.1, x 200 50.1 / 45.5 / 54.0 and 50.7, x 400 66.6 / 59.7 / 69.6 and 64.9, 40 x 160 56.9 / 55.6 / 62.0 and 61.4, 64 x 200 76.1 /
// 75.5 / 86.2 and 85.9, 64 x 400 108 / 95 / 122 and 113.  From 2 KB on, with a second launch where the ranges did not fit: 26 x 80 34.7 / 39.2, 26 x 128 38.3 /
// 41.4, 40 x 100 46.5 / 51.5, 64 x 64 53.6 / 62.6, 64 x 256 86.0 / 92.2.  Few inputs, 33 KB to lose: 8 x 128 30.4 / 31.0; 101 KB: 8 x 200 32.8 / 32.7.
// An input crosses packed up to the first block that does not have the form: 26 x 2048 with one id in a hundred -1 186 / 146, with one id and one value
// in a thousand other than the rest 186 / 180, one in a hundred 185 / 184.
constexpr size_t kPackWide = 12 << 10, kPackFrom = 4 << 10, kPackLeast = 48 << 10;

struct FeedInput {
  const void* data;
  size_t len;
  size_t offset;  // its slice of the arena: they lie side by side, multiples of 256 bytes each
  size_t word;    // bytes of an element
  // what the link may be spared of it
  size_t Spares() const { return word == 8 && len >= kPackWide ? len / 2 : word == 4 && len >= kPackFrom ? len : 0; }
};

// Stages the inputs, which are FeedInputs and whose slices are `plain` bytes, from `staging` on, which has as many, and has
// launch(pieces, how many) move them to `arena`.
template <typename Input, typename Launch>
void StageInputs(const std::vector<Input>& inputs, size_t plain, char* staging, char* arena, const Launch& launch) {
  bz_feed_piece pieces[BZ_FEED_MAX_PIECES];
  int n = 0;
  size_t moved = 0, staged = 0;  // bytes of the arena whose transfer has been launched; of the staging memory in use
  size_t part = plain < kFeedLong ? kFeedFirst : (plain / (plain / kFeedMost) / 256 + 1) * 256;
  auto end_of_part = [&]() { return plain - moved < part + part / 2 ? plain : moved + part; };
  size_t end = end_of_part();
  auto next_part = [&]() {
    moved = end;
    if (plain < kFeedLong) part = std::min(part + part / 2, kFeedMost);
    end = end_of_part();
  };
  size_t least = 0;
  for (const Input& in : inputs) least += in.Spares();
  // As it is, a request of few bytes above all, whose many inputs are no more than a copy each here (one sample of 18 lists: 5.95 us
  // in the call with the loop below, 5.5 with this one).
  if (least < kPackLeast) {
    auto launch_part = [&]() {
      pieces[0] = {staging + moved, arena + moved, (int64_t)(end - moved), BZ_FEED_RAW, 0};
      launch(pieces, 1);
      next_part();
    };
    for (const Input& in : inputs)
      for (size_t at = 0; at < in.len;) {
        // (a part ends on a multiple of 256 bytes, as every slice begins: never before this byte)
        const size_t now = std::min(in.len - at, end - (in.offset + at));
        memcpy(staging + in.offset + at, (const char*)in.data + at, now);
        at += now;
        if (in.offset + at == end) launch_part();
      }
    if (plain > moved) launch_part();
    return;
  }
  auto up = [](size_t bytes, size_t to) { return (bytes + to - 1) / to * to; };
  // `bytes` of the arena from `at` on, of which `source` bytes have been staged
  auto add = [&](size_t at, size_t bytes, int form, uint32_t word, size_t source) {
    char *from = staging + staged, *to = arena + at;
    staged += source;
    bz_feed_piece* last = n > 0 ? &pieces[n - 1] : nullptr;
    if (last && form == BZ_FEED_RAW && last->form == BZ_FEED_RAW)  // (what is raw lies side by side at both ends)
      last->bytes += bytes;
    else
      pieces[n++] = {from, to, (int64_t)bytes, form, word};
  };
  for (const Input& in : inputs) {
    bool packs = in.Spares() > 0;
    uint32_t first = 0;
    if (packs) memcpy(&first, in.data, 4);
    for (size_t at = 0; at < in.len;) {
      // (staged <= in.offset + at)
      const char* from = (const char*)in.data + at;
      const size_t left = std::min(in.len - at, end - (in.offset + at));
      size_t now = 0;
      // (with room for this range and a raw one behind it, to which all further ones of the part then belong)
      if (packs && n + 2 <= BZ_FEED_MAX_PIECES) {
        now = in.word * (in.word == 8 ? PackLow32((uint32_t*)(staging + staged), (const uint64_t*)from, left / 8) : CountSame32(from, left / 4, first));
        packs = now == left;
        if (now > 0) add(in.offset + at, up(now, 16), in.word == 8 ? BZ_FEED_LOW32 : BZ_FEED_SAME32, first, in.word == 8 ? up(now / 2, 256) : 0);
      }
      if (now == 0) {
        now = left;
        memcpy(staging + staged, from, now);
        add(in.offset + at, up(now, 256), BZ_FEED_RAW, 0, up(now, 256));
      }
      at += now;
      if (in.offset + at == end) {
        launch(pieces, n);
        n = 0;
        next_part();
      }
    }
  }
  if (n > 0) launch(pieces, n);
}

}  // namespace blaze
