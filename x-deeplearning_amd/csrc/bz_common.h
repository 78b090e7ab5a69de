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
bool fc_rows_takes(int64_t k, int64_t n1, int64_t n2);
bool fc_rows_pays(int64_t rows, int64_t k, int64_t n1, int64_t n2);
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

}  // namespace bz
