// embed_common.h -- what the Embedding kernels of embed_pool.hip (one row shape, sums) and embed_mixed.hip (kassign, slots of
// different shapes) share: offsets from segment counts, rows through buffer resources, the walk over a segment, the stores.
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>

#include <type_traits>

#include "bz_common.h"
#include "embed_groups.h"

namespace {

constexpr int kThreads = 512;  // measured at 128 / 256 / 512 / 1024 on config 2: 14.7 / 13.5 / 13.3 / 13.4 us per launch,
                               // 127 / 131 / 135 / 129 M samples/s with eight serving threads

__device__ __forceinline__ int64_t wave_incl_scan(int64_t v, int lane) {
#pragma unroll
  for (int d = 1; d < bz::kWave; d <<= 1) {
    int64_t t = __shfl_up(v, d, bz::kWave);
    if (lane >= d) v += t;
  }
  return v;
}

// All sums saturate at cap (< 2^31): every term is >= 0 and <= cap, so min(a + b, cap) is associative and gives the
// clamped offsets whatever the order of the additions, in 32 bits.
__device__ __forceinline__ uint32_t sat_add(uint32_t a, uint32_t b, uint32_t cap) {
  const uint32_t t = a + b;  // a, b <= cap < 2^31: no wrap
  return t < cap ? t : cap;
}

// Inclusive scan over the 64 lanes with data-parallel primitives (row_shr within rows of 16 lanes, then lane 15 and
// lane 31 handed on to the following rows): a dozen VALU instructions, where the same scan through ds_bpermute
// (__shfl_up) is six dependent trips to LDS per 32 bits.
__device__ __forceinline__ uint32_t row_scan_sat(uint32_t v, uint32_t cap) {  // within each row of 16 lanes
  v = sat_add(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false), cap);  // row_shr:1
  v = sat_add(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false), cap);  // row_shr:2
  v = sat_add(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false), cap);  // row_shr:4
  v = sat_add(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false), cap);  // row_shr:8
  return v;
}
__device__ __forceinline__ uint32_t wave_scan_sat(uint32_t v, uint32_t cap) {
  v = row_scan_sat(v, cap);
  v = sat_add(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false), cap);  // row_bcast:15 -> rows 1, 3
  v = sat_add(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false), cap);  // row_bcast:31 -> rows 2, 3
  return v;
}
// ---------------------------------------------------------------------------------------------
// pooling
// ---------------------------------------------------------------------------------------------
template <int DT>
struct RowTraits;
template <>
struct RowTraits<BZ_F32> {
  static constexpr int kElems = 4;  // per 16-byte chunk
};
template <>
struct RowTraits<BZ_F16> {
  static constexpr int kElems = 8;
};
template <>
struct RowTraits<BZ_I8> {
  static constexpr int kElems = 16;
};

// widen one 16-byte chunk to fp32 weights.  int8: w = scale * (float)q, one rounding.
template <int DT>
__device__ __forceinline__ void widen(const uint4& raw, float scale, float (&w)[RowTraits<DT>::kElems]) {
  const uint32_t r[4] = {raw.x, raw.y, raw.z, raw.w};
  if constexpr (DT == BZ_F32) {
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = __uint_as_float(r[i]);
  } else if constexpr (DT == BZ_F16) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      w[2 * i] = __half2float(__ushort_as_half((unsigned short)(r[i] & 0xffffu)));
      w[2 * i + 1] = __half2float(__ushort_as_half((unsigned short)(r[i] >> 16)));
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        int q = (int)(int8_t)((r[i] >> (8 * b)) & 0xffu);
        w[4 * i + b] = __fmul_rn(scale, (float)q);
      }
    }
  }
}

// scale of row r of an int8 table (a dense float array, or a field inside the table's rows)
__device__ __forceinline__ float load_scale(const bz_embed_slot& s, int64_t r) {
  return *(const float*)((const char*)s.row_scale + r * (int64_t)(s.scale_pitch != 0 ? s.scale_pitch : 4));
}

// acc += value * (the weights of one 16-byte chunk), the product rounded, then the sum rounded (udf_processor.h:66: never
// one fused operation).  For fp16 rows the widening rides in the multiply: fma(widen(h), value, +0) is the correctly
// rounded product (a product of -0 comes out as +0, which adds the same).  UNIT: the caller knows value == 1, so the
// product is the weight itself and acc + w is a single rounding, fma(widen(h), 1, acc) -- one instruction per element
// where the general form takes three.
// (int8 rows: and that every |scale| is below kFoldedScale)
constexpr float kFoldedScale = 0x1p120f;
template <int DT, bool UNIT>
__device__ __forceinline__ void accum_chunk(float (&acc)[RowTraits<DT>::kElems], const uint4& raw, float scale, float value) {
  const uint32_t r[4] = {raw.x, raw.y, raw.z, raw.w};
  if constexpr (DT == BZ_F32) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float w = __uint_as_float(r[i]);
      acc[i] = __fadd_rn(acc[i], UNIT ? w : __fmul_rn(value, w));
    }
  } else if constexpr (DT == BZ_F16) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float w = __half2float(__ushort_as_half((unsigned short)((r[i / 2] >> (16 * (i & 1))) & 0xffffu)));
      // (UNIT: `value` is a 1.0 the compiler cannot see through, so that the widening and the add stay one
      // v_fma_mix_f32; with a literal 1 it splits them into a convert and an add)
      acc[i] = UNIT ? __builtin_fmaf(w, value, acc[i]) : __fadd_rn(acc[i], __builtin_fmaf(w, value, 0.0f));
    }
  } else if constexpr (UNIT) {
    // q * scale from q + 128, a byte without a sign: fma(q + 128, scale, -128 * scale) is that product, rounded once, as long as 128 * scale is
    // finite.  A signed byte's conversion takes an operand selector, and twice the turns of an addition; and an instruction that waits
    // for the one before it takes longer also where eight waves share the SIMD, so they come eight of a kind: 7.7 clocks an element, 12.3
    // before.  4096 x 50 lists of 20 ids, 64-byte rows, 2000 a table, 50.4 -> 46.5 us (a million a table 70, memory's), 1024 of 200 bytes 45.9 -> 43.4.
    const float least = -128.f * scale;
    constexpr int G = 8;
#pragma unroll
    for (int g = 0; g < 16; g += G) {
      float w[G];
#pragma unroll
      for (int i = 0; i < G; ++i) w[i] = (float)(((r[(g + i) / 4] ^ 0x80808080u) >> (8 * (i & 3))) & 0xffu);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < G; ++i) w[i] = __builtin_fmaf(w[i], scale, least);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < G; ++i) acc[g + i] = __fadd_rn(acc[g + i], w[i]);
      __builtin_amdgcn_sched_barrier(0);
    }
  } else {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float w = __fmul_rn(scale, (float)(int)(int8_t)((r[i / 4] >> (8 * (i & 3))) & 0xffu));
      acc[i] = __fadd_rn(acc[i], __fmul_rn(value, w));
      if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
  }
}

typedef unsigned long long u64x2a8 __attribute__((ext_vector_type(2), aligned(8)));

// key / id -> table row, or -1 when absent.  Hash path = HashTable::Lookup
// (hashtable.cc:45-64): bucket record {offset:40, size:24}, (key,row) pairs.
__device__ __forceinline__ int64_t resolve_row(const bz_embed_slot& s, int64_t id) {
  if (s.hash_buckets != nullptr) {
    const uint64_t key = (uint64_t)id;
    const uint32_t h = (uint32_t)key;
    const uint64_t rec = s.hash_buckets[h % s.hash_bucket_size];
    const uint32_t cnt = (uint32_t)(rec >> 40);
    const uint64_t* p = s.hash_pairs + ((rec & 0xffffffffffull) >> 3);
    // (a pair in one load: the row number is there with the key, not a trip after it.  1000 x 24 lists of 6 keys, 400-byte
    // rows 21.0 -> 19.5 us, 8000 x 24 lists of 48-byte rows 34.5 -> 30.4)
    uint64_t row = ~0ull;
    for (uint32_t i = 0; i < cnt; ++i) {
      const u64x2a8 pair = *(const u64x2a8*)(p + 2 * i);
      if (pair.x == key) {
        row = pair.y;
        break;
      }
    }
    return row < (uint64_t)s.rows ? (int64_t)row : -1;
  }
  return (id >= 0 && id < s.rows) ? id : -1;
}

// fp32 -> bf16 bit pattern, round to nearest even; NaN stays a quiet NaN
__device__ __forceinline__ uint32_t f32_to_bf16_bits(float f) {
  const uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (u >> 16) | 0x40u;
  return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
}

// 16 and 8 bytes at any 4-byte address: the memory system takes such stores
typedef unsigned int u32x4a4 __attribute__((ext_vector_type(4), aligned(4)));
typedef unsigned int u32x2a4 __attribute__((ext_vector_type(2), aligned(4)));

// `nvalid` of 2 * W 2-byte elements, packed two a word, to `dst`: whole chunks in one store while every active lane's
// address is a multiple of 4 (lanes of one wave that took different ways would run them one after the other), a row's last
// chunk word by word.
template <int W>
__device__ __forceinline__ void store_halves(__half* dst, const uint32_t (&pk)[W], int nvalid) {
  if (__all(((uintptr_t)dst & 3) == 0)) {
    uint32_t* d = (uint32_t*)dst;
    if (nvalid >= 2 * W) {
#pragma unroll
      for (int i = 0; i + 4 <= W; i += 4) *(u32x4a4*)(d + i) = u32x4a4{pk[i], pk[i + 1], pk[i + 2], pk[i + 3]};
      if (W % 4 != 0) *(u32x2a4*)(d + W / 4 * 4) = u32x2a4{pk[W / 4 * 4], pk[W / 4 * 4 + 1]};
    } else {
#pragma unroll
      for (int i = 0; i < W; ++i) {
        if (2 * i + 1 < nvalid)
          d[i] = pk[i];
        else if (2 * i < nvalid)
          dst[2 * i] = __ushort_as_half((unsigned short)(pk[i] & 0xffffu));
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < 2 * W; ++i)
      if (i < nvalid) dst[i] = __ushort_as_half((unsigned short)((pk[i / 2] >> (16 * (i & 1))) & 0xffffu));
  }
}

// Store `nvalid` fp32 results as the slot's output dtype at element `elem_off`.
template <int N>
__device__ __forceinline__ void store_elems(void* dst_base, int64_t elem_off, const float (&v)[N], int nvalid,
                                            int out_dtype) {
  if (out_dtype == BZ_F32) {
    float* dst = (float*)dst_base + elem_off;
    if (nvalid >= N) {
#pragma unroll
      for (int i = 0; i < N; i += 4)
        *(u32x4a4*)(dst + i) =
            u32x4a4{__float_as_uint(v[i]), __float_as_uint(v[i + 1]), __float_as_uint(v[i + 2]), __float_as_uint(v[i + 3])};
    } else {
#pragma unroll
      for (int i = 0; i < N; ++i)
        if (i < nvalid) dst[i] = v[i];
    }
  } else {  // BZ_F16 / BZ_BF16, round to nearest even (a 16-bit slot; bf16 bits travel through the same stores)
    uint32_t pk[N / 2];
#pragma unroll
    for (int i = 0; i < N / 2; ++i) {
      uint32_t lo, hi;
      if (out_dtype == BZ_F16) {
        lo = __half_as_ushort(__float2half_rn(v[2 * i]));
        hi = __half_as_ushort(__float2half_rn(v[2 * i + 1]));
      } else {
        lo = f32_to_bf16_bits(v[2 * i]);
        hi = f32_to_bf16_bits(v[2 * i + 1]);
      }
      pk[i] = lo | (hi << 16);
    }
    store_halves<N / 2>((__half*)dst_base + elem_off, pk, nvalid);
  }
}

// elements between the output positions of a kassign sample
__device__ __forceinline__ int assign_pitch(const bz_embed_slot& s) { return s.assign_pitch != 0 ? s.assign_pitch : s.dim; }
// kassign: position p of the output holds id j = p (in order) or num - trunc + p (reverse);
// positions without an id, and ids absent from the table, are zero (udf_processor.h:103-131).
// One call fills chunk c of positions p0 .. p0 + kAssignRun - 1 of sample b: the positions of a sample are independent
// of each other, so the kernel spreads them over lane groups instead of walking them one dependent load after the
// other, and a group keeps kAssignRun of them in flight (their ids are neighbours in memory): with one position a
// group, DIN's 50-position histories were bounded by the four dependent trips to memory each group makes for a
// single 36-byte row.
constexpr int kAssignRun = 4;
__host__ __device__ inline int64_t items_per_sample(const bz_embed_slot& s) {
  return s.udf == BZ_ASSIGN ? (s.trunc_num + kAssignRun - 1) / kAssignRun : 1;
}
// ---------------------------------------------------------------------------------------------
// offsets of one workgroup's samples, derived from the segment counts
// ---------------------------------------------------------------------------------------------
// s_off[0..groups] <- exclusive offsets of samples b0 .. b0+groups (clipped to batch).
// Every thread of the workgroup calls it; ends with a barrier.
// `offsets`: the slot's precomputed offsets (slot.offsets, or its share of a buffer the launch brings), or nullptr.
template <int THREADS = kThreads>
__device__ __forceinline__ void stage_offsets(const bz_embed_slot& s, const int64_t* __restrict__ offsets, int64_t b0,
                                              int groups, int64_t* s_off, int64_t* s_part) {
  const int tid = threadIdx.x;
  const int lane = tid & (bz::kWave - 1), wave = tid / bz::kWave;
  if (offsets != nullptr) {
    for (int t = tid; t <= groups; t += THREADS)
      if (b0 + t <= s.batch) {
        const int64_t o = offsets[b0 + t];
        s_off[t] = o < 0 ? 0 : (o < s.nnz ? o : s.nnz);  // caller-made offsets get the same bounds as the scan's
      }
    __syncthreads();
    return;
  }
  // base = sum of the counts before b0 (independent coalesced reads), local = this thread's sample
  // (8 loads in flight per thread: a rolled loop would wait for each load before issuing the next)
  // this thread's own count is requested first so that it travels with the counts summed below
  // (a negative count is taken as 0 and the offsets below stop at nnz: see bz_embed_slot.nnz)
  const int64_t mine = (tid < groups && b0 + tid < s.batch) ? (int64_t)max(s.segments[b0 + tid], 0) : 0;
  int64_t part = 0;
  const int64_t ahead = bz::counts_before(b0, s.batch);
  for (int64_t i0 = 0; i0 < ahead; i0 += 8 * THREADS) {
    int32_t c[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int64_t i = i0 + k * THREADS + tid;
      c[k] = i < ahead ? max(s.segments[i], 0) : 0;
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) part += c[k];
  }
  int64_t base = part;
#pragma unroll
  for (int d = bz::kWave / 2; d > 0; d >>= 1) base += __shfl_xor(base, d, bz::kWave);
  const int64_t incl = wave_incl_scan(mine, lane);
  if (lane == bz::kWave - 1) {
    s_part[wave] = base;
    s_part[THREADS / bz::kWave + wave] = incl;
  }
  __syncthreads();
  int64_t before = 0;
#pragma unroll
  for (int w = 0; w < THREADS / bz::kWave; ++w) {
    before += s_part[w];
    if (w < wave) before += s_part[THREADS / bz::kWave + w];
  }
  if (tid < groups) s_off[tid + 1] = (before + incl) < s.nnz ? (before + incl) : s.nnz;
  if (tid == 0) s_off[0] = before < s.nnz ? before : s.nnz;
  __syncthreads();
}

typedef int i32x4a4 __attribute__((ext_vector_type(4), aligned(4)));  // four counts, from any count on

// a count as the scans take it, and a sum with four more of them
__device__ __forceinline__ uint32_t count_sat(int32_t c, uint32_t cap) { return (uint32_t)min(max(c, 0), (int)cap); }
__device__ __forceinline__ uint32_t add_counts_sat(uint32_t sum, const i32x4a4& c, uint32_t cap) {
#pragma unroll
  for (int j = 0; j < 4; ++j) sum = sat_add(sum, count_sat(c[j], cap), cap);
  return sum;
}

// What lies before wave w of a workgroup of WAVES, given in LDS each wave's share of the counts before the workgroup's first
// sample, then each wave's own sum: entry WAVES - 1 + w of the inclusive scan over the 2 * WAVES values, done in one row of
// 16 lanes, in lane WAVES - 1 + w of each row.
template <int WAVES>
__device__ __forceinline__ uint32_t waves_scan_sat(const uint32_t* tot, uint32_t cap) {
  static_assert(2 * WAVES <= 16, "the waves' totals are scanned within one row of lanes");
  const int i = threadIdx.x & 15;
  return row_scan_sat(i < 2 * WAVES ? tot[i] : 0u, cap);
}

constexpr int kShapeKeyed = 1 << 16;  // in a plan's `shape`: a slot is looked up by key

constexpr int kBlockIds = 4;  // ids walked per step (measured at 2, 4, 8, 16: 4 is best or equal on segments of 1-4, 8 and 20 ids)

// Slot records handed over as kernel arguments: a workgroup then has its record after the one scalar load every
// kernel starts with, instead of after a second trip to memory for slots[si] (measured on config 2: 1050 cycles from
// the start of a wave to its kernel arguments, 2200 more to the record).
struct SlotPack {
  bz_embed_slot s[BZ_EMBED_ARG_SLOTS];
};
static_assert(sizeof(SlotPack) + 4 * 16 + 32 <= 4096, "the records and the other arguments fit the 4 KB kernel-argument segment");

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
constexpr uint32_t kBeyondTable = 0xF0000000u;  // a byte offset that nothing read through a buffer resource reaches
constexpr int64_t kWalkIds = 1ll << 28;         // ids of one wave's segments: their byte offsets and twice kBeyondTable stay apart

// Which lane of a row's group holds what of a step of kBlockIds ids: id u of the step is held by lane u % kSrc of every
// quad of the group (u / kSrc: which of the lane's kPerLane ids), so that handing it to the group's lanes is one DPP
// operand of the instruction that uses it.
template <int LPR>
struct StepShape {
  static constexpr int kSrc = LPR < kBlockIds ? LPR : kBlockIds;
  static constexpr int kPerLane = kBlockIds / kSrc;
};

// what the lane that holds id U of the step has in v
template <int LPR, int U>
__device__ __forceinline__ uint32_t of_id(uint32_t v) {
  if constexpr (LPR == 1) return v;
  constexpr int w = U % StepShape<LPR>::kSrc;
  constexpr int ctrl = LPR >= 4 ? w * 0x55 : (w | w << 2 | (2 + w) << 4 | (2 + w) << 6);  // quad_perm
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, ctrl, 0xf, 0xf, true);
}

template <typename F>
__device__ __forceinline__ void each_id(const F& f) {
  static_assert(kBlockIds == 4, "");
  f(std::integral_constant<int, 0>{});
  f(std::integral_constant<int, 1>{});
  f(std::integral_constant<int, 2>{});
  f(std::integral_constant<int, 3>{});
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)bytes, 0x00020000);
}

// ids of one step that a lane holds, on their way
template <int LPR>
struct StepIds {
  u32x2 id[StepShape<LPR>::kPerLane];
  float val[StepShape<LPR>::kPerLane];
};

// rows of one step, on their way
template <int DT, int LPR>
struct StepRows {
  u32x4 raw[kBlockIds];
  float val[StepShape<LPR>::kPerLane];    // of the ids the lane holds
  uint32_t scale[StepShape<LPR>::kPerLane];  // int8 tables: of the same ids, a float's bits
  uint64_t weighted;                      // the wave's lanes that hold a value other than 1 (uniform)
};

template <int DT, int LPR>
__device__ __forceinline__ void add_rows(float (&acc)[RowTraits<DT>::kElems], const StepRows<DT, LPR>& st, float one) {
  using S = StepShape<LPR>;
  auto add = [&](auto u, auto unit) {
    constexpr int U = decltype(u)::value, K = U / S::kSrc;
    constexpr bool kUnit = decltype(unit)::value;
    uint4 raw = make_uint4(st.raw[U].x, st.raw[U].y, st.raw[U].z, st.raw[U].w);
    // (opaque, or the compiler moves the conversions that both forms begin with in front of them: 64 registers more)
    if (!kUnit) asm volatile("" : "+v"(raw.x), "+v"(raw.y), "+v"(raw.z), "+v"(raw.w));
    const float scale = DT == BZ_I8 ? __uint_as_float(of_id<LPR, U>(st.scale[K])) : 1.f;
    accum_chunk<DT, kUnit>(acc, raw, scale, kUnit ? one : __uint_as_float(of_id<LPR, U>(__float_as_uint(st.val[K]))));
    __builtin_amdgcn_sched_barrier(0);
  };
  // two conditions that the compiler cannot tell to exclude each other: as two branches of one condition the forms' sums
  // would live in registers of their own
  uint64_t general = st.weighted;
  if constexpr (DT == BZ_I8) {
    bool folded = true;
#pragma unroll
    for (int k = 0; k < S::kPerLane; ++k) folded &= fabsf(__uint_as_float(st.scale[k])) < kFoldedScale;
    general |= __builtin_amdgcn_ballot_w64(!folded);
  }
  uint64_t weighted = general;
  asm volatile("" : "+s"(weighted));
  if (general == 0) each_id([&](auto u) { add(u, std::true_type{}); });
  if (weighted != 0) each_id([&](auto u) { add(u, std::false_type{}); });
}

// One wave's reading of ids, a step of kBlockIds a lane group at a time, and of their rows: every operand comes through a
// buffer resource (the hardware checks every access and returns zeros beyond the end), so that what a lane does not need is
// asked for beyond the end and no load sits under a branch.
// LOW: a lane's ids may begin `low` ids after its first (positions of a kassign sample that come before its first id).
template <int DT, int LPR, bool HASH, bool LOW = false>
struct RowStream {
  using S = StepShape<LPR>;
  __amdgpu_buffer_rsrc_t ids, values, table, scales;
  const bz_embed_slot& s;
  uint32_t scale_pitch, at, pos;
  int rest, low;  // of the step at hand: this lane's ids k * kSrc with low <= k * kSrc < rest are there
  StepIds<LPR> next;

  // `first`: the wave's first id; this lane group's ids start `from` (in the first step, for its lane 0) after it
  __device__ __forceinline__ RowStream(const bz_embed_slot& slot, int64_t first, uint32_t from, int n, int l) : s(slot) {
    constexpr int CE = RowTraits<DT>::kElems;
    const int q = l % S::kSrc;
    const int nchunks = (s.dim + CE - 1) / CE;
    at = l < nchunks ? (uint32_t)l * 16u : 0u;  // (a lane without a chunk reads the group's first and drops it)
    const int64_t left = s.nnz - first;
    const uint32_t avail = left < kWalkIds ? (uint32_t)left : (uint32_t)kWalkIds;
    ids = buffer_of(s.ids + first, avail * 8u);
    values = buffer_of(s.values + first, avail * 4u);
    table = buffer_of(s.table, (uint32_t)(s.rows * (int64_t)s.pitch));
    scale_pitch = s.scale_pitch != 0 ? (uint32_t)s.scale_pitch : 4u;
    scales = buffer_of(s.row_scale, DT == BZ_I8 ? (uint32_t)(s.rows - 1) * scale_pitch + 4u : 0u);
    // with a hash index only the group's first quad holds ids: a probe is a request of its own
    const bool holds = !HASH || LPR <= 4 || l < S::kSrc;
    pos = (from + (uint32_t)q) * 4u;
    rest = holds ? n - q : 0;
    low = 0;
  }
  __device__ __forceinline__ bool there(int k) const { return (!LOW || k * S::kSrc >= low) && k * S::kSrc < rest; }
  __device__ __forceinline__ void fetch() {
#pragma unroll
    for (int k = 0; k < S::kPerLane; ++k) {
      const uint32_t o = there(k) ? pos + 4u * k * S::kSrc : kBeyondTable;
      next.id[k] = __builtin_amdgcn_raw_buffer_load_b64(ids, (int)(o << 1), 0, 0);
      next.val[k] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(values, (int)o, 0, 0));
    }
    pos += 4u * kBlockIds;
  }
  // asks for the rows of the ids fetched last, and, NEXT, for the ids behind them
  template <bool NEXT>
  __device__ __forceinline__ void request(StepRows<DT, LPR>& st, int l) {
    const int lane = threadIdx.x & (bz::kWave - 1);
    uint32_t off[S::kPerLane], soff[S::kPerLane];
    bool unit = true;
#pragma unroll
    for (int k = 0; k < S::kPerLane; ++k) {
      const uint64_t id = (uint64_t)next.id[k].y << 32 | next.id[k].x;
      bool ok = there(k);
      uint32_t row = (uint32_t)id;
      if constexpr (HASH) {
        const int64_t r = ok ? resolve_row(s, (int64_t)id) : -1;
        ok = r >= 0;
        row = (uint32_t)r;
      } else {
        ok = ok && id < (uint64_t)s.rows;
      }
      uint32_t at_row = __umul24(row, (uint32_t)s.pitch), at_scale = DT == BZ_I8 ? __umul24(row, scale_pitch) : 0u;
      float val = next.val[k];
      // (opaque, or the selects below become a divergent branch, and every uniform branch of the loop with them a pair
      // of masked blocks with sums of their own)
      asm volatile("" : "+v"(at_row), "+v"(at_scale), "+v"(val));
      off[k] = ok ? at_row : kBeyondTable;
      if (DT == BZ_I8) soff[k] = ok ? at_scale : kBeyondTable;
      // an id without a row contributes a zero row (times the value 1): adding +0 leaves the running sum as it is (the
      // sum starts at +0 and so is never -0)
      st.val[k] = ok ? val : 1.f;
      unit &= st.val[k] == 1.f;
    }
    st.weighted = __builtin_amdgcn_ballot_w64(!unit);
    if constexpr (HASH && LPR > 4) {
      const int holder = lane - l + l % S::kSrc;
#pragma unroll
      for (int k = 0; k < S::kPerLane; ++k) {
        off[k] = (uint32_t)__shfl((int)off[k], holder, bz::kWave);
        if (DT == BZ_I8) soff[k] = (uint32_t)__shfl((int)soff[k], holder, bz::kWave);
        st.val[k] = __shfl(st.val[k], holder, bz::kWave);
      }
    }
    if constexpr (NEXT) {
      rest -= kBlockIds;
      fetch();
    }
    each_id([&](auto u) {
      constexpr int U = decltype(u)::value, K = U / S::kSrc;
      st.raw[U] = __builtin_amdgcn_raw_buffer_load_b128(table, (int)(of_id<LPR, U>(off[K]) + at), 0, 0);
    });
    if (DT == BZ_I8) {
#pragma unroll
      for (int k = 0; k < S::kPerLane; ++k) st.scale[k] = __builtin_amdgcn_raw_buffer_load_b32(scales, (int)soff[k], 0, 0);
    }
    asm volatile("" ::: "memory");  // (the loads stay in this order on every path, or the loop's waits count too many)
  }
};

// Steps of the wave's longest segment, n being this lane's (the same in the LPR lanes of a group; every lane of the wave takes
// part).  The maximum ends up in lane 63, by DPP operands as in wave_scan_sat: through LDS it was up to six dependent trips of 120
// clocks in front of every walk.
template <int LPR>
__device__ __forceinline__ int wave_steps(int n) {
  n = max(n, 0);
  if (LPR < 2) n = max(n, __builtin_amdgcn_update_dpp(0, n, 0x111, 0xf, 0xf, false));   // row_shr:1
  if (LPR < 4) n = max(n, __builtin_amdgcn_update_dpp(0, n, 0x112, 0xf, 0xf, false));   // row_shr:2
  if (LPR < 8) n = max(n, __builtin_amdgcn_update_dpp(0, n, 0x114, 0xf, 0xf, false));   // row_shr:4
  if (LPR < 16) n = max(n, __builtin_amdgcn_update_dpp(0, n, 0x118, 0xf, 0xf, false));  // row_shr:8
  if (LPR < 32) n = max(n, __builtin_amdgcn_update_dpp(0, n, 0x142, 0xa, 0xf, false));  // row_bcast:15 -> rows 1, 3
  if (LPR < 64) n = max(n, __builtin_amdgcn_update_dpp(0, n, 0x143, 0xc, 0xf, false));  // row_bcast:31 -> rows 2, 3
  return (__builtin_amdgcn_readlane(n, bz::kWave - 1) + kBlockIds - 1) / kBlockIds;
}

// The walk over a segment: straight-line code that the whole wave runs as often as its longest segment takes, the rows of a
// step under way while those of the step before are added up.  (Waits count outstanding loads in order: after a join of a
// path with loads and one without, the compiler waits for all of them.)
// Measured with this walk, before / after: 26 slots x 2048 of 8 ids, 64-byte rows 9.0 /
// 8.8 us, half the vector instructions; with offsets given 16384 samples 48.4 / 45.9, 200 slots x 8192 of 2.5 ids, 128-byte
// rows 181 / 157 to 168; int8 rows of 64, 20 ids, 83 / 80; eight serving threads 15.2 / 14.9 us a pass of 2048.  Rows that
// are found in the caches are bound by the lanes' idle turns (a wave walks as far as its longest segment) and, int8, by the
// three instructions an element takes (92 % of the vector units' time); rows that are not by memory, 4.7 TB/s of lines.
// Positions are relative to `first`, the wave's first id; n ids from position `from` on.
template <int DT, int LPR>
__device__ __forceinline__ void walk(const bz_embed_slot& s, int64_t first, uint32_t from, int n, int l, float (&acc)[RowTraits<DT>::kElems]) {
  RowStream<DT, LPR, false> rows(s, first, from, n, l);
  float one = 1.f;  // (opaque: see accum_chunk)
  asm volatile("" : "+v"(one));
  int steps = wave_steps<LPR>(n);
  if (steps <= 0) return;
  StepRows<DT, LPR> a, b;
  rows.fetch();
  rows.template request<true>(a, l);
  for (; steps > 2; steps -= 2) {
    rows.template request<true>(b, l);
    add_rows<DT, LPR>(acc, a, one);
    rows.template request<true>(a, l);
    add_rows<DT, LPR>(acc, b, one);
  }
  if (steps == 2) {
    rows.template request<true>(b, l);
    add_rows<DT, LPR>(acc, a, one);
    a = b;
  }
  add_rows<DT, LPR>(acc, a, one);
}

// The same for tables looked up by key.  A probe is two dependent trips to memory (bucket, then pair) before the row's own, so
// keys are resolved kKeyBatch at a time, one or more a lane: every lane of a group probes, where four did a step's four, and a
// segment of up to kKeyBatch ids makes those two trips once instead of once a step.  Its rows then follow as in the walk above.
// What bounds it is that chain (counts, ids, bucket, pair, row).  1000 x 24 lists of 6 keys, 400-byte fp32 rows: 19.1 -> 15.1 us.
template <int DT, int LPR>
__device__ __forceinline__ void walk_keyed(const bz_embed_slot& s, int64_t first, uint32_t from, int n, int l, float (&acc)[RowTraits<DT>::kElems]) {
  using S = StepShape<LPR>;
  constexpr int kKeyBatch = LPR > 8 ? LPR : 8, kPer = kKeyBatch / LPR;  // lane l holds keys k * LPR + l of a batch
  const RowStream<DT, LPR, true> rows(s, first, from, n, l);           // (its resources and chunk)
  float one = 1.f;  // (opaque: see accum_chunk)
  asm volatile("" : "+v"(one));
  int steps = wave_steps<LPR>(n);
  if (steps <= 0) return;
  const int gbase = (threadIdx.x & (bz::kWave - 1)) - l;
  u32x2 id[kPer];
  float val[kPer];
  int at = l;  // this lane's first id of the batch at hand
  auto fetch = [&]() {
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const uint32_t o = at + k * LPR < n ? (from + (uint32_t)(at + k * LPR)) * 4u : kBeyondTable;
      id[k] = __builtin_amdgcn_raw_buffer_load_b64(rows.ids, (int)(o << 1), 0, 0);
      val[k] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rows.values, (int)o, 0, 0));
    }
  };
  fetch();
  for (;; steps -= kKeyBatch / kBlockIds) {
    uint32_t off[kPer], soff[kPer];
    float v[kPer];
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int64_t r = at + k * LPR < n ? resolve_row(s, (int64_t)((uint64_t)id[k].y << 32 | id[k].x)) : -1;
      off[k] = r >= 0 ? __umul24((uint32_t)r, (uint32_t)s.pitch) : kBeyondTable;
      soff[k] = DT == BZ_I8 && r >= 0 ? __umul24((uint32_t)r, rows.scale_pitch) : kBeyondTable;
      v[k] = r >= 0 ? val[k] : 1.f;  // (an id without a row adds a zero row: see RowStream::request)
    }
    if (steps > kKeyBatch / kBlockIds) {
      at += kKeyBatch;
      fetch();
    }
    // step s of the batch
    auto request = [&](StepRows<DT, LPR>& st, int step) {
      uint32_t so[S::kPerLane], of[S::kPerLane];
      bool unit = true;
#pragma unroll
      for (int k = 0; k < S::kPerLane; ++k) {
        if constexpr (LPR <= kBlockIds) {  // the lane's own (`step` is a constant here)
          of[k] = off[step * S::kPerLane + k];
          so[k] = soff[step * S::kPerLane + k];
          st.val[k] = v[step * S::kPerLane + k];
        } else {
          const int holder = gbase + step * kBlockIds + l % kBlockIds;
          of[k] = (uint32_t)__shfl((int)off[0], holder, bz::kWave);
          if (DT == BZ_I8) so[k] = (uint32_t)__shfl((int)soff[0], holder, bz::kWave);
          st.val[k] = __shfl(v[0], holder, bz::kWave);
        }
        unit &= st.val[k] == 1.f;
      }
      st.weighted = __builtin_amdgcn_ballot_w64(!unit);
      each_id([&](auto u) {
        constexpr int U = decltype(u)::value, K = U / S::kSrc;
        st.raw[U] = __builtin_amdgcn_raw_buffer_load_b128(rows.table, (int)(of_id<LPR, U>(of[K]) + rows.at), 0, 0);
      });
      if (DT == BZ_I8) {
#pragma unroll
        for (int k = 0; k < S::kPerLane; ++k) st.scale[k] = __builtin_amdgcn_raw_buffer_load_b32(rows.scales, (int)so[k], 0, 0);
      }
      asm volatile("" ::: "memory");
    };
    StepRows<DT, LPR> a, b;
    const int here = min(steps, kKeyBatch / kBlockIds);
    request(a, 0);
    if constexpr (LPR <= 8) {
      if (here > 1) {
        request(b, 1);
        add_rows<DT, LPR>(acc, a, one);
        a = b;
      }
    } else {
      int i = 1;
      for (; i + 1 < here; i += 2) {
        request(b, i);
        add_rows<DT, LPR>(acc, a, one);
        request(a, i + 1);
        add_rows<DT, LPR>(acc, b, one);
      }
      if (i < here) {
        request(b, i);
        add_rows<DT, LPR>(acc, a, one);
        a = b;
      }
    }
    add_rows<DT, LPR>(acc, a, one);
    if (steps <= kKeyBatch / kBlockIds) return;
  }
}

// The same for tables and segments beyond what buffer resources address: plain loads under branches.  26 slots x 4096 of 20
// ids from 2^24 + 999 rows, values of 1 in a form of their own / all multiplied: int8 rows of 64 66.0 / 67.7 us, of 20000 hot
// rows 41.5 / 46.6, 300 samples of 8 ids 10.1 / 11.2; fp16 rows of 32 63.0 / 63.7 and 24.0 / 25.2, 2048 of 8 ids, rows of 18, 8.9 / 9.7.
template <int DT, int LPR>
__device__ __forceinline__ void walk_plain(const bz_embed_slot& s, int64_t start, int64_t end, int l, float (&acc)[RowTraits<DT>::kElems]) {
  using S = StepShape<LPR>;
  constexpr int CE = RowTraits<DT>::kElems;
  const int gbase = (threadIdx.x & (bz::kWave - 1)) - l;  // first lane of this group within the wave
  const bool has_chunk = l < (s.dim + CE - 1) / CE;
  const char* table = (const char*)s.table + (int64_t)l * 16;
  float one = 1.f;  // (opaque: see accum_chunk)
  asm volatile("" : "+v"(one));
  // the next step's ids are requested before this step's rows, so the two round trips overlap
  int64_t id_next[S::kPerLane];  // raw ids: resolved to rows only when consumed, so the wait lands after the row loads
  float val_next[S::kPerLane];
  auto fetch_ids = [&](int64_t j) {
#pragma unroll
    for (int k = 0; k < S::kPerLane; ++k) {
      const int idx = k * S::kSrc + l;
      id_next[k] = -1;
      val_next[k] = 0.f;
      if (l < S::kSrc && idx < end - j) {
        id_next[k] = s.ids[j + idx];
        val_next[k] = s.values[j + idx];
      }
    }
  };
  if (start < end) fetch_ids(start);
  for (int64_t j = start; j < end; j += kBlockIds) {
    int row_own[S::kPerLane];
    float val_own[S::kPerLane];
#pragma unroll
    for (int k = 0; k < S::kPerLane; ++k) {
      row_own[k] = (l < S::kSrc && k * S::kSrc + l < end - j) ? (int)resolve_row(s, id_next[k]) : -1;
      val_own[k] = row_own[k] >= 0 ? val_next[k] : 1.f;
    }
    if (j + kBlockIds < end) fetch_ids(j + kBlockIds);
    // (whether all values of the wave's ids are 1; two conditions for one, as in add_rows)
    bool unit = true;
#pragma unroll
    for (int k = 0; k < S::kPerLane; ++k) unit &= val_own[k] == 1.f;
    uint64_t weighted = __builtin_amdgcn_ballot_w64(!unit);
    int row[kBlockIds];
    float val[kBlockIds];
    uint4 raw[kBlockIds];
    float sc[kBlockIds];
#pragma unroll
    for (int u = 0; u < kBlockIds; ++u) {  // (all before the first load: 69.0 -> 66.0 us for the int8 rows above)
      row[u] = __shfl(row_own[u / S::kSrc], gbase + (u % S::kSrc), bz::kWave);
      val[u] = __shfl(val_own[u / S::kSrc], gbase + (u % S::kSrc), bz::kWave);
    }
#pragma unroll
    for (int u = 0; u < kBlockIds; ++u) {
      raw[u] = make_uint4(0, 0, 0, 0);
      sc[u] = 1.f;
      if (has_chunk && row[u] >= 0) {
        raw[u] = *(const uint4*)(table + (int64_t)row[u] * s.pitch);
        if (DT == BZ_I8) sc[u] = load_scale(s, row[u]);
      }
    }
    if constexpr (DT == BZ_I8) {
      bool folded = true;
#pragma unroll
      for (int u = 0; u < kBlockIds; ++u) folded &= fabsf(sc[u]) < kFoldedScale;
      weighted |= __builtin_amdgcn_ballot_w64(!folded);
    }
    uint64_t weighted_too = weighted;
    asm volatile("" : "+s"(weighted_too));
    auto add = [&](int u, float v, auto unit_form) {
      constexpr bool kUnit = decltype(unit_form)::value;
      uint4 r = raw[u];
      if (!kUnit) asm volatile("" : "+v"(r.x), "+v"(r.y), "+v"(r.z), "+v"(r.w));
      accum_chunk<DT, kUnit>(acc, r, sc[u], v);
      __builtin_amdgcn_sched_barrier(0);  // (all conversions of a step's int8 rows at once would hold 64 more registers)
    };
    if (weighted == 0) {
#pragma unroll
      for (int u = 0; u < kBlockIds; ++u) add(u, one, std::true_type{});
    }
    if (weighted_too != 0) {
#pragma unroll
      for (int u = 0; u < kBlockIds; ++u) add(u, val[u], std::false_type{});
    }
  }
  // No load is under way here, but the compiler takes both forms above to be skipped and the rows' loads to be pending, also
  // where the other walk's code begins, whose waits for ids, values and rows then are for everything: 1000 x 24 lists of keyed
  // 400-byte rows 19.2 us, 19.6 without this wait.  (vmcnt 0, the other counters anything)
  __builtin_amdgcn_s_waitcnt(0x0f70);
}

// whether the table is one that buffer resources address
template <int DT>
__device__ __forceinline__ bool table_fits(const bz_embed_slot& s) {
  return s.rows <= (1ll << 24) && s.pitch < (1 << 24) && (uint64_t)s.rows * (uint64_t)s.pitch <= (uint64_t)kBeyondTable &&
         (DT != BZ_I8 || (s.scale_pitch < (1 << 24) && (uint64_t)s.rows * (uint64_t)(uint32_t)s.scale_pitch <= (uint64_t)kBeyondTable));
}

// the wave's first id, and whether all of the wave's segments lie close behind it: offsets never decrease when the scan
// makes them (caller-made ones may, and take the other path)
__device__ __forceinline__ bool wave_is_near(int64_t start, int64_t end, int64_t* first) {
  *first = (int64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)start) |
           (int64_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)((uint64_t)start >> 32)) << 32;
  return __all(start >= *first && end - *first < kWalkIds);
}

// acc: the sum of the segment [start, end), for one chunk of the row.  KEYED: the kernel is one for slots with a hash index.
// In the others the keyed walk's code is left out, and with it 7 to 15 registers (200 slots x 8192 of 2.5 ids 184.5 us with
// both walks in one kernel, 180.3 without; eight serving threads 976 and 949); a slot that is keyed all the same is right there,
// by plain loads.
template <int DT, int LPR, bool KEYED>
__device__ __forceinline__ void sum_segment(const bz_embed_slot& s, int64_t start, int64_t end, int l, float (&acc)[RowTraits<DT>::kElems]) {
#pragma unroll
  for (int i = 0; i < RowTraits<DT>::kElems; ++i) acc[i] = 0.f;
  int64_t first;
  const bool hash = s.hash_buckets != nullptr;
  if (wave_is_near(start, end, &first) && table_fits<DT>(s) && (KEYED || !hash)) {
    const uint32_t from = (uint32_t)(start - first);
    const int n = (int)(end - start);
    if (KEYED && hash)
      walk_keyed<DT, LPR>(s, first, from, n, l, acc);
    else
      walk<DT, LPR>(s, first, from, n, l, acc);
  } else {
    walk_plain<DT, LPR>(s, start, end, l, acc);
  }
}

template <int DT>
__device__ __forceinline__ void finish_sum(const bz_embed_slot& s, int64_t num, int l, int64_t b, float (&acc)[RowTraits<DT>::kElems]) {
  constexpr int CE = RowTraits<DT>::kElems;
  if (s.udf == BZ_AVG && num != 0) {
    const float inv = (float)(1.0 / (double)num);  // ValueType(1.0 / size), udf_processor.h:88
#pragma unroll
    for (int i = 0; i < CE; ++i) acc[i] = __fmul_rn(acc[i], inv);
  }
  const int e0 = l * CE;
  if (e0 < s.dim) store_elems<CE>(s.out, b * s.out_stride + e0, acc, s.dim - e0, s.out_dtype);
}

// The sum of sample b, `inside`: whether there is such a sample.  All lanes of a wave with one come along (wave_steps).
template <int DT, int LPR, bool KEYED>
__device__ __forceinline__ void sum_samples(const bz_embed_slot& s, int64_t start, int64_t end, int l, int64_t b, bool inside) {
  if (__builtin_amdgcn_ballot_w64(inside) == 0) return;
  if (!inside) end = start;
  float acc[RowTraits<DT>::kElems];
  sum_segment<DT, LPR, KEYED>(s, start, end, l, acc);
  if (inside) finish_sum<DT>(s, end - start, l, b, acc);
}

// f(table dtype, lanes per row, whether a slot is keyed), all as constants, for a (dtype << 8) | lanes code of a plan
template <typename F>
int with_shape(int code, bool keyed, const F& with_keyed) {
  auto f = [&](auto dt, auto lpr) {
    if (keyed)
      with_keyed(dt, lpr, std::true_type{});
    else
      with_keyed(dt, lpr, std::false_type{});
  };
  auto lanes = [&](auto dt) -> int {
    switch (code & 0xff) {
      case 1: f(dt, std::integral_constant<int, 1>{}); return BZ_OK;
      case 2: f(dt, std::integral_constant<int, 2>{}); return BZ_OK;
      case 4: f(dt, std::integral_constant<int, 4>{}); return BZ_OK;
      case 8: f(dt, std::integral_constant<int, 8>{}); return BZ_OK;
      case 16: f(dt, std::integral_constant<int, 16>{}); return BZ_OK;
      case 32: f(dt, std::integral_constant<int, 32>{}); return BZ_OK;
      case 64: f(dt, std::integral_constant<int, 64>{}); return BZ_OK;
      default: return bz::fail(BZ_EINVAL, "bz_embed_pool: bad lanes-per-row %d in variant", code & 0xff);
    }
  };
  switch (code >> 8) {
    case BZ_F32: return lanes(std::integral_constant<int, BZ_F32>{});
    case BZ_F16: return lanes(std::integral_constant<int, BZ_F16>{});
    case BZ_I8: return lanes(std::integral_constant<int, BZ_I8>{});
    default: return bz::fail(BZ_EINVAL, "bz_embed_pool: bad table dtype %d in variant", code >> 8);
  }
}

}  // namespace

namespace bz {
// embed_mixed.hip: the launches of plans without the specialised kernel (launch.variant == 0)
int embed_launch_mixed(const bz_embed_slot* slots_dev, const bz_embed_launch& L, const int64_t* ext_off, int64_t ext_stride, hipStream_t st);
int embed_launch_mixed_args(const bz_embed_slot* slots_host, const bz_embed_launch& L, hipStream_t st);
}  // namespace bz
