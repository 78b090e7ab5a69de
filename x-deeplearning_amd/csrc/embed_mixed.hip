// embed_mixed.hip -- Embedding launches whose slots are not all sums over equal numbers of samples: kassign, numbers of
// samples that differ (one row shape: bz_embed_mixed_kernel), row shapes or table types that differ (bz_embed_pool_generic_kernel).
#include <limits.h>
#include <string.h>

#include "embed_common.h"

namespace {

constexpr int kUnroll = 4;  // rows in flight per lane group in the generic kernel (8 held 118 VGPRs and was no faster)

// ksum / kavg for one lane: chunk `c` of the segment [start, end) of sample b.
template <int DT>
__device__ __forceinline__ void pool_sum(const bz_embed_slot& s, int64_t start, int64_t end, int c, int64_t b) {
  constexpr int CE = RowTraits<DT>::kElems;
  float acc[CE];
#pragma unroll
  for (int i = 0; i < CE; ++i) acc[i] = 0.f;
  const char* table = (const char*)s.table + (int64_t)c * 16;
  for (int64_t j = start; j < end; j += kUnroll) {
    const int n = (int)((end - j) < kUnroll ? (end - j) : kUnroll);
    int64_t row[kUnroll];
    float val[kUnroll];
    uint4 raw[kUnroll];
    float sc[kUnroll];
    // clamp instead of branching: the tail repeats the last id (cache hit), results ignored
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      const int64_t jj = (u < n) ? j + u : end - 1;
      row[u] = resolve_row(s, s.ids[jj]);
      val[u] = s.values[jj];
    }
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      const int64_t r = row[u] < 0 ? 0 : row[u];
      raw[u] = *(const uint4*)(table + r * (int64_t)s.pitch);
      sc[u] = (DT == BZ_I8) ? load_scale(s, r) : 1.f;
    }
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      if (u < n && row[u] >= 0) {
        float w[CE];
        widen<DT>(raw[u], sc[u], w);
        // out = out + value * w: two roundings, never an FMA (udf_processor.h:66)
#pragma unroll
        for (int i = 0; i < CE; ++i) acc[i] = __fadd_rn(acc[i], __fmul_rn(val[u], w[i]));
      }
    }
  }
  if (s.udf == BZ_AVG) {
    const int64_t num = end - start;
    if (num != 0) {
      const float inv = (float)(1.0 / (double)num);  // ValueType(1.0 / size), udf_processor.h:88
#pragma unroll
      for (int i = 0; i < CE; ++i) acc[i] = __fmul_rn(acc[i], inv);
    }
  }
  const int e0 = c * CE;
  const int nvalid = (s.dim - e0) < CE ? (s.dim - e0) : CE;
  store_elems<CE>(s.out, b * s.out_stride + e0, acc, nvalid, s.out_dtype);
}
template <int DT>
__device__ __forceinline__ void pool_assign(const bz_embed_slot& s, int64_t start, int64_t end, int c, int64_t b, int p0) {
  constexpr int CE = RowTraits<DT>::kElems;
  constexpr int R = kAssignRun;
  const int64_t num = end - start;
  const int e0 = c * CE;
  const int nvalid = (s.dim - e0) < CE ? (s.dim - e0) : CE;
  const char* table = (const char*)s.table + (int64_t)c * 16;
  const int64_t shift = (s.trunc_dir == BZ_ORDER) ? 0 : num - (int64_t)s.trunc_num;
  // no branch round the loads: a position without an id reads id 0 of the slot (there is one whenever any position
  // has an id) and row 0 of the table, and the result is dropped
  bool live[R];
  int64_t row[R];
  float val[R];
  uint4 raw[R];
  float sc[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int64_t j = shift + p0 + r;
    live[r] = p0 + r < s.trunc_num && j >= 0 && j < num;
    const int64_t at = live[r] ? start + j : 0;
    row[r] = -1;
    val[r] = 0.f;
    if (num > 0) {  // (uniform over the group's positions: they belong to one sample)
      row[r] = resolve_row(s, s.ids[at]);
      val[r] = s.values[at];
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    live[r] = live[r] && row[r] >= 0;
    const int64_t rr = live[r] ? row[r] : 0;
    raw[r] = *(const uint4*)(table + rr * (int64_t)s.pitch);
    sc[r] = (DT == BZ_I8) ? load_scale(s, rr) : 1.f;
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (p0 + r < s.trunc_num) {
      float out[CE];
      float w[CE];
      widen<DT>(raw[r], sc[r], w);
#pragma unroll
      for (int i = 0; i < CE; ++i) out[i] = live[r] ? __fmul_rn(val[r], w[i]) : 0.f;
      store_elems<CE>(s.out, b * s.out_stride + (int64_t)(p0 + r) * assign_pitch(s) + e0, out, nvalid, s.out_dtype);
    }
  }
}

// zero fill of one item's columns (unknown table name: quick_embedding_dict.cc:95 leaves the
// memset block untouched)
__device__ __forceinline__ void pool_zero(const bz_embed_slot& s, int64_t b, int p0, int l, int lpr) {
  const int run = s.udf == BZ_ASSIGN ? kAssignRun : 1;  // p0 = 0 unless kassign
  for (int p = p0; p < p0 + run && (p == 0 || p < s.trunc_num); ++p) {
    const int64_t base = b * s.out_stride + (int64_t)p * assign_pitch(s);
    for (int e = l; e < s.dim; e += lpr) {
      if (s.out_dtype == BZ_F32)
        ((float*)s.out)[base + e] = 0.f;
      else
        ((__half*)s.out)[base + e] = __ushort_as_half(0);
    }
  }
}
__device__ __forceinline__ int chunk_elems(int dt) { return dt == BZ_F32 ? 4 : (dt == BZ_F16 ? 8 : 16); }

// one workgroup of the generic path: workgroup v of the launch, owned by slot s
__device__ __forceinline__ void pool_generic(const bz_embed_slot& s, int v, const int64_t* __restrict__ offsets, int64_t* s_off,
                                             int64_t* s_part) {
  const int ce = chunk_elems(s.table_dtype);
  const int nchunks = (s.dim + ce - 1) / ce;
  // lpr, a power of two: shifts, not divisions (a 64-bit division is some 150 instructions, and this kernel's threads
  // each do little else than one or four row gathers)
  int lpr_log = 0;
  while ((1 << lpr_log) < nchunks && (1 << lpr_log) < bz::kWave) ++lpr_log;
  const int lpr = 1 << lpr_log;
  const int groups = kThreads >> lpr_log;
  const int tid = threadIdx.x;
  const int g = tid >> lpr_log;
  const int l = tid - (g << lpr_log);
  // a lane group owns one item: a sample (ksum / kavg) or kAssignRun output positions of a sample (kassign)
  const int64_t per = items_per_sample(s);
  const int64_t n_items = (int64_t)s.batch * per;
  const int64_t i0 = (int64_t)(v - s.wg_begin) * groups;
  int64_t i_last = i0 + groups - 1;
  if (i_last >= n_items) i_last = n_items - 1;
  // item -> sample: no division for pooled slots (per == 1), a 32-bit one while the item count allows it
  auto sample_of = [&](int64_t item) -> int64_t {
    if (per == 1) return item;
    if (n_items < (1ll << 31)) return (int64_t)((uint32_t)item / (uint32_t)per);
    return item / per;
  };
  const int64_t b_first = sample_of(i0);
  const int n_samples = (int)(sample_of(i_last) - b_first) + 1;  // <= groups
  stage_offsets(s, offsets, b_first, n_samples, s_off, s_part);
  const int64_t item = i0 + g;
  if (item >= n_items) return;
  const int64_t b = sample_of(item);
  const int p = (int)(item - b * per) * (s.udf == BZ_ASSIGN ? kAssignRun : 1);
  if (s.table == nullptr) {
    pool_zero(s, b, p, l, lpr);
    return;
  }
  const int64_t start = s_off[b - b_first], end = s_off[b - b_first + 1];
  for (int c = l; c < nchunks; c += lpr) {
    if (s.udf == BZ_ASSIGN) {
      switch (s.table_dtype) {
        case BZ_F32: pool_assign<BZ_F32>(s, start, end, c, b, p); break;
        case BZ_F16: pool_assign<BZ_F16>(s, start, end, c, b, p); break;
        default: pool_assign<BZ_I8>(s, start, end, c, b, p); break;
      }
    } else {
      switch (s.table_dtype) {
        case BZ_F32: pool_sum<BZ_F32>(s, start, end, c, b); break;
        case BZ_F16: pool_sum<BZ_F16>(s, start, end, c, b); break;
        default: pool_sum<BZ_I8>(s, start, end, c, b); break;
      }
    }
  }
}

// The slot that owns workgroup v = the last one with wg_begin <= v (empty slots share a begin with their successor).
// Begins never decrease, so that is (number of begins <= v) - 1: every wave counts them 64 at a time with one load
// and a ballot - one trip to memory where a binary search would make log2(n_slots) dependent ones.
__device__ __forceinline__ int slot_of(const bz_embed_slot* __restrict__ slots, int n_slots, int v) {
  const int lane = threadIdx.x & (bz::kWave - 1);
  int cnt = 0;
  for (int base = 0; base < n_slots; base += bz::kWave) {
    const int i = base + lane;
    const bool le = i < n_slots && slots[i].wg_begin <= v;
    cnt += __popcll(__ballot(le));
  }
  return __builtin_amdgcn_readfirstlane(cnt - 1);
}

// the same with the slot records as kernel arguments: no trip for the begins, none for the record
struct SlotBegins {
  int b[16];  // wg_begin of every slot, INT_MAX behind the last: read with one wide scalar load
};
__device__ __forceinline__ int slot_of(const SlotBegins& begins, int v) {
  int lo = -1;
#pragma unroll
  for (int i = 0; i < 16; ++i) lo += begins.b[i] <= v ? 1 : 0;  // uniform: scalar compares
  return lo;
}

__global__ __launch_bounds__(kThreads) void bz_embed_pool_generic_kernel(const bz_embed_slot* __restrict__ slots,
                                                                         int n_slots, int total_wg, int wg_per_xcd,
                                                                         int wg_per_slot, const int64_t* __restrict__ ext_off,
                                                                         int64_t ext_stride) {
  __shared__ int64_t s_off[kThreads + 1];
  __shared__ int64_t s_part[2 * kThreads / bz::kWave];
  // XCD-aware order: hardware deals consecutive workgroup ids round robin over the 8 XCDs; give
  // each XCD a contiguous range of the logical workgroup space (= a contiguous range of slots).
  const int v = (int)(blockIdx.x % bz::kNumXcd) * wg_per_xcd + (int)(blockIdx.x / bz::kNumXcd);
  if (v >= total_wg) return;
  const int lo = wg_per_slot > 0 ? v / wg_per_slot : slot_of(slots, n_slots, v);
  // slots with wg_count == 0 sharing this begin come before the one that owns the workgroup
  const bz_embed_slot s = slots[lo];
  pool_generic(s, v, ext_off != nullptr ? ext_off + (int64_t)lo * ext_stride : s.offsets, s_off, s_part);
}

__global__ __launch_bounds__(kThreads) void bz_embed_pool_generic_args_kernel(int total_wg, int wg_per_xcd, int wg_per_slot,
                                                                              const SlotPack pack, const SlotBegins begins) {
  __shared__ int64_t s_off[kThreads + 1];
  __shared__ int64_t s_part[2 * kThreads / bz::kWave];
  const int v = (int)(blockIdx.x % bz::kNumXcd) * wg_per_xcd + (int)(blockIdx.x / bz::kNumXcd);
  if (v >= total_wg) return;
  const int lo = wg_per_slot > 0 ? v / wg_per_slot : slot_of(begins, v);
  const bz_embed_slot s = pack.s[lo];
  pool_generic(s, v, s.offsets, s_off, s_part);
}

// ---------------------------------------------------------------------------------------------
// slots of one table dtype and LPR lanes per row whose items differ: kassign, or numbers of samples
// ---------------------------------------------------------------------------------------------
// The lanes of a group know their row shape, so kassign takes the walk's loads (ids one a lane, rows through a buffer resource
// without a branch, 60 registers where the generic kernel holds 110) and a chunk leaves in one store at any 4-byte address
// where it took four; an fp16 row whose value is 1 leaves as it came.  Generic kernel / this one, us: 3 histories of 50 x 1024
// samples, 36-byte fp16 rows 12.0 / 6.7; 20 x 4096 of 128-byte rows 289 / 187 (1 GB written); int8 rows of 100, 20 x 2048,
// 312 / 190; keyed 192-byte fp32 rows, 16 x 1000, 187 / 75.
// Positions p0 .. p0 + kAssignRun - 1 of sample b, whose ids are [start, start + num): one step of the walk, stored position
// by position.
template <int DT, int LPR, bool HASH>
__device__ __forceinline__ void assign_step(const bz_embed_slot& s, int64_t first, uint32_t from, int num, int l, int64_t b, int p0) {
  constexpr int CE = RowTraits<DT>::kElems;
  static_assert(kAssignRun == kBlockIds, "a run of positions is a step of ids");
  const int skip = (s.trunc_dir == BZ_ORDER ? 0 : num - s.trunc_num) + p0;  // of the sample's ids, to position p0's
  RowStream<DT, LPR, HASH, true> rows(s, first, from + (uint32_t)skip, min(num - skip, s.trunc_num - p0), l);
  rows.low = -skip - l % StepShape<LPR>::kSrc;
  StepRows<DT, LPR> st;
  rows.fetch();
  rows.template request<false>(st, l);
  const int e0 = l * CE;
  const int64_t at = b * s.out_stride + (int64_t)p0 * assign_pitch(s) + e0;
  each_id([&](auto u) {
    constexpr int U = decltype(u)::value, K = U / StepShape<LPR>::kSrc;
    // (handed on by lanes that may have no chunk of the row themselves: before any lane is left out)
    const float val = __uint_as_float(of_id<LPR, U>(__float_as_uint(st.val[K])));
    const float scale = DT == BZ_I8 ? __uint_as_float(of_id<LPR, U>(st.scale[K])) : 1.f;
    if (e0 >= s.dim || p0 + U >= s.trunc_num) return;
    const uint4 raw = make_uint4(st.raw[U].x, st.raw[U].y, st.raw[U].z, st.raw[U].w);
    if (DT == BZ_F16 && s.out_dtype == BZ_F16 && st.weighted == 0) {  // the row's own bits
      const uint32_t pk[4] = {raw.x, raw.y, raw.z, raw.w};
      store_halves<4>((__half*)s.out + at + U * assign_pitch(s), pk, s.dim - e0);
    } else {
      float w[CE];
      widen<DT>(raw, scale, w);
#pragma unroll
      for (int i = 0; i < CE; ++i) w[i] = __fmul_rn(val, w[i]);
      store_elems<CE>(s.out, at + U * assign_pitch(s), w, s.dim - e0, s.out_dtype);
    }
  });
}

// Start and end of sample b_first + i, 0 <= i < n_samples <= kThreads, i the caller's own, from the counts: the counts
// before b_first are added up, the workgroup's own scanned, one barrier.  Every thread of the workgroup calls it; nnz < 2^31.
struct SegmentLds {
  uint32_t incl[kThreads];                  // within a wave's 64 samples
  uint32_t tot[2 * kThreads / bz::kWave];  // the waves' shares of the counts before b_first, then their own samples' sums
};
__device__ __forceinline__ void segment_of(const bz_embed_slot& s, int64_t b_first, int n_samples, int i, SegmentLds& lds, int64_t* start,
                                           int64_t* end) {
  constexpr int WAVES = kThreads / bz::kWave;
  const int tid = threadIdx.x;
  const int lane = tid & (bz::kWave - 1), wave = tid / bz::kWave;
  const uint32_t cap = (uint32_t)s.nnz;
  const int32_t own = tid < n_samples ? s.segments[b_first + tid] : 0;
  const uint32_t quads = (uint32_t)b_first / 4;
  const int32_t odd = tid < (int)(b_first & 3) ? s.segments[4 * quads + tid] : 0;
  uint32_t part = 0;
  for (uint32_t i0 = tid; i0 < quads; i0 += kThreads) part = add_counts_sat(part, ((const i32x4a4*)s.segments)[i0], cap);
  part = sat_add(part, count_sat(odd, cap), cap);
  const uint32_t incl = wave_scan_sat(count_sat(own, cap), cap);
  const uint32_t earlier = wave_scan_sat(part, cap);
  lds.incl[tid] = incl;
  if (lane == bz::kWave - 1) {
    lds.tot[wave] = earlier;
    lds.tot[WAVES + wave] = incl;
  }
  __syncthreads();
  const uint32_t t = waves_scan_sat<WAVES>(lds.tot, cap);
  const uint32_t before = (uint32_t)__shfl((int)t, WAVES - 1 + i / bz::kWave, bz::kWave);
  const uint32_t excl = i % bz::kWave == 0 ? 0u : lds.incl[i - 1];
  *start = (int64_t)sat_add(before, excl, cap);
  *end = (int64_t)sat_add(before, lds.incl[i], cap);
}

// one workgroup of such a launch: workgroup v, owned by slot s
template <int DT, int LPR, bool KEYED>
__device__ __forceinline__ void pool_mixed(const bz_embed_slot& s, int v, const int64_t* __restrict__ offsets) {
  constexpr int GROUPS = kThreads / LPR;
  __shared__ union {
    SegmentLds lds;
    struct {
      int64_t off[kThreads + 1], part[2 * kThreads / bz::kWave];
    } wide;
  } sh;
  const int tid = threadIdx.x;
  const int g = tid / LPR, l = tid % LPR;
  // a lane group owns one item: a sample (ksum / kavg) or kAssignRun output positions of a sample (kassign)
  const int64_t per = items_per_sample(s);
  const int64_t n_items = (int64_t)s.batch * per;
  const int64_t i0 = (int64_t)(v - s.wg_begin) * GROUPS;
  auto sample_of = [&](int64_t item) -> int64_t {
    if (per == 1) return item;
    if (n_items < (1ll << 31)) return (int64_t)((uint32_t)item / (uint32_t)per);
    return item / per;
  };
  const int64_t last = n_items - 1, item = i0 + g;
  if (i0 > last) return;  // (of the whole workgroup: a record whose batch disagrees with the plan)
  const int64_t b_first = sample_of(i0);
  const int n_samples = (int)(sample_of(i0 + GROUPS - 1 < last ? i0 + GROUPS - 1 : last) - b_first) + 1;  // <= GROUPS
  const int64_t b = sample_of(item < last ? item : last);
  int64_t start, end;
  if (offsets == nullptr && s.nnz < (1ll << 31)) {
    segment_of(s, b_first, n_samples, (int)(b - b_first), sh.lds, &start, &end);
  } else {
    stage_offsets(s, offsets, b_first, n_samples, sh.wide.off, sh.wide.part);
    start = sh.wide.off[b - b_first];
    end = sh.wide.off[b - b_first + 1];
  }
  if (s.udf != BZ_ASSIGN) {
    sum_samples<DT, LPR, KEYED>(s, start, end, l, b, item <= last);
    return;
  }
  if (item > last) return;
  const int p0 = (int)(item - b * per) * kAssignRun;
  int64_t first;
  const bool hash = s.hash_buckets != nullptr;
  if (wave_is_near(start, end, &first) && table_fits<DT>(s) && (KEYED || !hash)) {
    const uint32_t from = (uint32_t)(start - first);
    const int num = end > start ? (int)(end - start) : 0;
    if (KEYED && hash)
      assign_step<DT, LPR, true>(s, first, from, num, l, b, p0);
    else
      assign_step<DT, LPR, false>(s, first, from, num, l, b, p0);
  } else if (l < (s.dim + RowTraits<DT>::kElems - 1) / RowTraits<DT>::kElems) {
    pool_assign<DT>(s, start, end, l, b, p0);
  }
}

template <int DT, int LPR, bool KEYED>
__global__ __launch_bounds__(kThreads) void bz_embed_mixed_kernel(const bz_embed_slot* __restrict__ slots, int n_slots, int total_wg,
                                                                  int wg_per_xcd, int wg_per_slot, const int64_t* __restrict__ ext_off,
                                                                  int64_t ext_stride) {
  const int v = (int)(blockIdx.x % bz::kNumXcd) * wg_per_xcd + (int)(blockIdx.x / bz::kNumXcd);
  if (v >= total_wg) return;
  const int lo = wg_per_slot > 0 ? v / wg_per_slot : slot_of(slots, n_slots, v);
  const bz_embed_slot s = slots[lo];
  pool_mixed<DT, LPR, KEYED>(s, v, ext_off != nullptr ? ext_off + (int64_t)lo * ext_stride : s.offsets);
}

template <int DT, int LPR, bool KEYED>
__global__ __launch_bounds__(kThreads) void bz_embed_mixed_args_kernel(int total_wg, int wg_per_xcd, int wg_per_slot,
                                                                       const SlotPack pack, const SlotBegins begins) {
  const int v = (int)(blockIdx.x % bz::kNumXcd) * wg_per_xcd + (int)(blockIdx.x / bz::kNumXcd);
  if (v >= total_wg) return;
  const int lo = wg_per_slot > 0 ? v / wg_per_slot : slot_of(begins, v);
  const bz_embed_slot s = pack.s[lo];
  pool_mixed<DT, LPR, KEYED>(s, v, s.offsets);
}
}  // namespace

namespace bz {

int embed_launch_mixed(const bz_embed_slot* slots_dev, const bz_embed_launch& L, const int64_t* ext_off, int64_t ext_stride, hipStream_t st) {
  const int per_xcd = (L.total_wg + kNumXcd - 1) / kNumXcd;
  const dim3 grid(per_xcd * kNumXcd), block(kThreads);
  const int per_slot = ((int64_t)L.wg_per_slot * L.n_slots == L.total_wg) ? L.wg_per_slot : 0;
  if (L.shape != 0) {
    const int rc = with_shape(L.shape & ~kShapeKeyed, (L.shape & kShapeKeyed) != 0, [&](auto dt, auto lpr, auto keyed) {
      hipLaunchKernelGGL((bz_embed_mixed_kernel<decltype(dt)::value, decltype(lpr)::value, decltype(keyed)::value>), grid, block, 0, st, slots_dev, L.n_slots,
                         L.total_wg, per_xcd, per_slot, ext_off, ext_stride);
    });
    if (rc != BZ_OK) return rc;
    BZ_LAUNCH_OK("bz_embed_mixed_kernel");
    return BZ_OK;
  }
  hipLaunchKernelGGL(bz_embed_pool_generic_kernel, grid, block, 0, st, slots_dev, L.n_slots, L.total_wg, per_xcd, per_slot, ext_off,
                     ext_stride);
  BZ_LAUNCH_OK("bz_embed_pool_generic_kernel");
  return BZ_OK;
}

int embed_launch_mixed_args(const bz_embed_slot* slots_host, const bz_embed_launch& L, hipStream_t st) {
  SlotPack pack;
  memcpy(pack.s, slots_host, (size_t)L.n_slots * sizeof(bz_embed_slot));
  memset(pack.s + L.n_slots, 0, (size_t)(BZ_EMBED_ARG_SLOTS - L.n_slots) * sizeof(bz_embed_slot));
  const int per_xcd = (L.total_wg + kNumXcd - 1) / kNumXcd;
  const dim3 grid(per_xcd * kNumXcd), block(kThreads);
  if (L.n_slots > 16) return fail(BZ_ENOTSUP, "bz_embed_pool_args: a plan of mixed row shapes takes at most 16 slots");
  for (int i = 0; i < L.n_slots; ++i)
    BZ_REQUIRE(pack.s[i].offsets == nullptr, "bz_embed_pool_args: slot %d brings offsets, but the plan says the scan is fused in", i);
  SlotBegins begins;
  for (int i = 0; i < 16; ++i) begins.b[i] = i < L.n_slots ? pack.s[i].wg_begin : INT_MAX;
  const int per_slot = ((int64_t)L.wg_per_slot * L.n_slots == L.total_wg) ? L.wg_per_slot : 0;
  if (L.shape != 0) {
    const int rc = with_shape(L.shape & ~kShapeKeyed, (L.shape & kShapeKeyed) != 0, [&](auto dt, auto lpr, auto keyed) {
      hipLaunchKernelGGL((bz_embed_mixed_args_kernel<decltype(dt)::value, decltype(lpr)::value, decltype(keyed)::value>), grid, block, 0, st, L.total_wg, per_xcd, per_slot, pack,
                         begins);
    });
    if (rc != BZ_OK) return rc;
    BZ_LAUNCH_OK("bz_embed_mixed_args_kernel");
    return BZ_OK;
  }
  hipLaunchKernelGGL(bz_embed_pool_generic_args_kernel, grid, block, 0, st, L.total_wg, per_xcd, per_slot, pack, begins);
  BZ_LAUNCH_OK("bz_embed_pool_generic_args_kernel");
  return BZ_OK;
}

}  // namespace bz
