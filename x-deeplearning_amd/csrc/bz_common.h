// bz_common.h -- shared helpers of the gfx950 kernel layer (error plumbing, small device utilities).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "blaze_hip.h"

namespace bz {

// Records the message returned by bz_last_error() for this thread and returns `code`.
int fail(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));

#define BZ_REQUIRE(cond, ...)                       \
  do {                                              \
    if (!(cond)) return ::bz::fail(BZ_EINVAL, __VA_ARGS__); \
  } while (0)

#define BZ_HIP_OK(expr)                                                                                   \
  do {                                                                                                    \
    hipError_t e_ = (expr);                                                                               \
    if (e_ != hipSuccess) return ::bz::fail(BZ_EHIP, "%s failed: %s", #expr, hipGetErrorString(e_));      \
  } while (0)

// A kernel launch reports configuration errors through hipGetLastError.
#define BZ_LAUNCH_OK(what)                                                                                \
  do {                                                                                                    \
    hipError_t e_ = hipGetLastError();                                                                    \
    if (e_ != hipSuccess) return ::bz::fail(BZ_EHIP, "launch of %s failed: %s", what, hipGetErrorString(e_)); \
  } while (0)

inline hipStream_t as_stream(bz_stream_t s) { return reinterpret_cast<hipStream_t>(s); }

inline int dtype_size(int dt) {
  switch (dt) {
    case BZ_F32: return 4;
    case BZ_I32: return 4;
    case BZ_F16: return 2;
    case BZ_BF16: return 2;
    case BZ_I8: return 1;
    case BZ_I64: return 8;
    default: return 0;
  }
}

constexpr int kWave = 64;       // CDNA wavefront
constexpr int kNumXcd = 8;      // MI355X: 8 accelerator complex dies, workgroups are dealt to them round robin

// fc_attention_f32.hip, for the host layer: bz_fc_fused of an fp32 layer on pieces [x, y, x - y, x * y] with a second and a
// skinny third layer, of whose outputs only the last is stored.  BZ_ENOTSUP, with nothing launched, for anything else.
int fc_attention_f32(const bz_fc_desc& d, bz_stream_t stream);
// whether it takes layers k -> n -> n2
bool fc_attention_f32_takes(int64_t k, int64_t n, int64_t n2);
// fc_tower.hip, for the host layer: an fp16 layer on a stored input, a second one (d.next) and a skinny third (the head) in one
// launch, of whose outputs only the last is stored, once more at `copy` unless that is null.  d.w and d.next->w are weights that
// fc_tower_pack laid out, fc_tower_weight_bytes each.  BZ_ENOTSUP, with nothing launched, for anything else.
int fc_tower(const bz_fc_desc& d, void* copy, bz_stream_t stream);
bool fc_tower_takes(int64_t k, int64_t n1, int64_t n2);  // whether it takes layers k -> n1 -> n2
bool fc_tower_pays(int64_t rows, int64_t k, int64_t n1, int64_t n2);  // whether that is faster than the first and the others in two
size_t fc_tower_weight_bytes(int64_t k, int64_t n);
int fc_tower_pack(const void* w, bool transposed, int k, int n, void* out, bz_stream_t stream);  // from [k, n], or [n, k] when transposed
// fc_rows.hip, for the host layer: the same for few rows, fp32; d.w and d.next->w as fc_rows_pack laid them out
int fc_rows(const bz_fc_desc& d, void* copy, bz_stream_t stream);
size_t fc_rows_weight_bytes(int64_t k, int64_t n);
int fc_rows_pack(const void* w, bool transposed, int k, int n, void* out, bz_stream_t stream);
// fc_fused.hip, for the host layer: bz_fc_fused that stores the outputs of a head, or of a layer of at most eight columns,
// once more at `copy`, [m, columns] without gaps (pinned host memory: results that are there when the launch has ended)
int fc_fused(const bz_fc_desc& d, void* copy, bz_stream_t stream);
// Whether it takes a head behind an fp16 or fp32 layer of columns that are no whole number of 16-byte chunks (bz_fc_fused does not; the
// kernel is the one of sixteen rows a workgroup).  That saves a launch, 2 us alone, and costs the whole weight for every
// sixteen rows: a lone launch gets longer with k * n, which one workgroup multiplies, and takes more of the chip from others
// with rows * k.  A model's forward alone / us a pass on eight serving threads, one launch and two, below and beyond each line:
//  k * n, fp16  300 of 256 -> 250 26.9 / 6.7 and 28.2 / 7.2, 400 -> 250 28.5 / 7.4 and 28.7 / 7.4; the two layers by themselves
//               768 -> 250 21.2 / 5.1 and 19.9 / 4.9
//         fp32  1024 of 128 -> 250 28.7 / 7.3 and 29.2 / 7.5, 400 -> 100 32.7 / 9.7 and 32.1 / 9.3, 200 -> 250 31.4 / 7.9 and 30.2 / 8.3;
//               the two layers by themselves 300 of 400 -> 250 25.5 / 6.2 and 20.9 / 5.6
//  rows * k, fp16  1500 of 512 -> 100 29.3 / 7.4 and 31.6 / 8.2, 2048 of 400 -> 250 31.1 / 9.3 and 32.0 / 8.7, 512 -> 100 29.9 / 9.3 and
//                  31.5 / 8.3
//            fp32  1024 of 200 -> 100 28.7 / 7.0 and 29.2 / 7.8, of 256 -> 50 27.6 / 7.8 and 29.3 / 7.7, 2048 of 128 -> 100 27.7 / 8.2 and
//                  28.6 / 8.0
//  rows  fp16  2048 of 256 -> 50 27.4 / 7.0 and 29.7 / 7.6, 2600 28.0 / 8.2 and 30.7 / 8.0; the two layers by themselves, 4096 of
//              64 -> 50 with others 1.28 times as long in one
inline bool head_behind_any_columns(int64_t rows, int64_t k, int64_t n, int element_size) {
  return rows <= 2048 && (element_size == 4 ? rows * k <= 240 << 10 && k * n <= 36 << 10 : rows * k <= 768 << 10 && k * n <= 96 << 10);
}

// Whether an fp32 layer's head is better off behind it, in a launch of its own.  In the layer's launch a workgroup owns whole rows,
// multiplies all of k * n for them, and the rows set how many CUs work; by itself the layer is on all of them.  One launch / two,
// us alone (errors against 64 bits are smaller in two): 300 of 256 -> 100 (25 K) 7.1 / 7.3, 201 of 200 -> 80 6.4 / 7.4, 2048 of
// 256 -> 64 6.1 / 7.5, 16384 of 200 -> 80 14.9 / 18.5; 1000 and 2000 of 512 -> 128 (64 K) 10.4 / 8.4 and 10.6 / 9.5, 64 of 2000 -> 48
// 16.1 / 12.5, 1024 of 512 -> 256 16.6 / 8.8, 2048 17.0 / 11.8, 4096 25.3 / 16.4, 8192 26.1 / 25.2, 2000 of 4096 -> 256 102 / 41.
inline bool head_apart(int64_t k, int64_t n, int element_size) { return element_size == 4 && k * n > 48 << 10; }

// What fc_rows takes: no more columns than four blocks of 64, so that at least two waves share K (with one each, 896 -> 400 -> 128, us of one lone row /
// a pass on eight serving threads, apart and in one launch 41.0 / 6.3 and 43.0 / 7.5), and weights that it does not lose with at any number of rows
// (322 K, 1032 -> 256 -> 256, 40.8 / 6.5 and 38.1 / 6.8).
constexpr int kRowsMaxIn = 1280, kRowsMaxColumns = 256;
inline bool fc_rows_takes(int64_t k, int64_t n1, int64_t n2) {
  return k >= 1 && k <= kRowsMaxIn && n1 > 8 && n1 <= kRowsMaxColumns && n2 > 8 && n2 <= kRowsMaxColumns && k * n1 + n1 * n2 <= 208 << 10;
}

// Whether few rows of a fp32 tower that it takes, k -> n1 -> n2 -> skinny, are better off in one launch (fc_rows.hip: one row a workgroup up to 128 rows, two to
// 256, three to 384, then four) than in two or three.  Models that look rows up for the input, us of a lone request / a pass on eight serving
// threads, apart and in one launch, by weights in units of 1024 and by rows:
//    5 (48 -> 64 -> 32)    1: 31.2 / 5.0 and 30.8 / 5.0, 300: 34.6 / 6.0 and 34.4 / 6.0, 600: 35.3 / 6.1 and 35.1 / 6.1, 1024: 37.2 / 6.2 and 37.1 / 6.2:
//      level, serving within 2 % either way from one run to the next
//   53 (192 -> 200 -> 80)  1: 32.8 / 5.7 and 30.2 / 4.9, 300: 38.4 / 6.8 and 35.5 / 5.9, 600: 43.3 / 7.0 and 39.1 / 5.6, 1024: 47.9 / 7.2 and 44.8 / 6.4
//   87 (328 -> 256 -> 16)  1024: 65.1 / 8.6 and 61.1 / 7.5
//  142 (468 -> 256 -> 100) 1: 36.9 / 6.1 and 34.7 / 5.4, 300: 45.0 / 7.3 and 40.2 / 6.4, 600: 53.0 / 7.8 and 46.6 / 7.1, 896: 62.4 / 8.7 and 57.2 / 8.3,
//      1024: 58.5 / 8.8 and 54.9 / 9.1
//  173 (592 -> 256 -> 100) 450: 56.0 / 7.8 and 50.2 / 7.2, 768: 63.4 / 8.9 and 59.3 / 8.6, 832: 65.3 / 9.0 and 60.2 / 9.0, 896: 66.1 / 9.1 and 61.8 / 9.4,
//      1024: 62.6 / 9.4 and 59.8 / 10.4
//  208 (732 -> 256 -> 100) 1: 38.9 / 6.2 and 37.6 / 6.1, 300: 56.0 / 7.7 and 51.0 / 7.4, 640: 62.8 / 8.7 and 58.0 / 8.5, 700: 67.6 / 9.0 and 62.4 / 9.1,
//      768: 69.1 / 9.5 and 65.3 / 9.7, 896: 73.6 / 9.9 and 68.4 / 10.6, 1024: 74.4 / 10.4 and 71.5 / 11.6
// A lone request is no slower in one; what it takes from others grows with rows times weights, and the line is where serving has begun
// to lose: 3 % at 142 x 1024, level at 173 x 832 and 208 x 700.  Beyond 1024 rows (with four a workgroup): 53 x 2000 59.9 / 9.2 and 59.6 / 9.1, 61 x 2000 89.0 / 10.1 and 86.3 / 11.1, 142 x 2000 85.2 / 13.5 and 79.5 / 15.4.
inline bool fc_rows_pays(int64_t rows, int64_t k, int64_t n1, int64_t n2) {
  return rows >= 1 && rows <= 1024 && rows * (k * n1 + n1 * n2) <= 144 << 20;
}

}  // namespace bz
