// embed_pool.hip -- Embedding gather + segmented pooling for gfx950 (MI355X).
//
// Replaces, for device-resident tables, the CPU loop of
// blaze/store/quick_embedding/quick_embedding_dict.cc:89-148 (QuickEmbeddingDict::Get)
// with its pooling processors blaze/store/quick_embedding/udf_processor.h:43-133 and
// the key lookup blaze/store/quick_embedding/hashtable.cc:45-64.
//
// Work decomposition.  The workload is memory bound: per id one random table row
// (36..256 bytes) plus 12 bytes of id/value.  A row is cut into 16-byte chunks
// (one 128-bit load); a *lane group* of `lpr` = pow2(chunks per row) lanes owns one
// (sample, slot) segment and walks its ids in order, so every output element is
// summed in exactly the reference's order (bit-identical fp32).  A workgroup of 512
// or 256 threads (small_groups) holds 512/lpr or 256/lpr segments of consecutive samples of one slot.  One launch
// covers every slot of the operator; the linear workgroup id is remapped so that
// each of the 8 XCDs (each with its own L2) serves a contiguous range of slots and
// therefore caches the hot rows of only those tables.
//
// The kernel is latency bound before it is bandwidth bound (a batch-2048 launch moves
// ~36 MB), so the dependent chain is kept at: slot record -> segments -> ids -> rows.
//   * segments -> offsets is fused: a workgroup sums the counts before its first
//     sample and scans its own in registers (no separate scan launch, no
//     offsets round trip);
//   * with equal work per slot the slot index is a division, not a search;
//   * the specialised ksum/kavg kernel walks a segment kBlockIds ids at a time: the lanes
//     of a group load disjoint ids/values (one coalesced read), resolve them to rows,
//     pass the rows around as DPP operands, and the rows of a step are requested before
//     those of the step before are added (walk).  The block is short on purpose: the
//     memory-level parallelism comes from eight resident waves per SIMD, not from a deep
//     unroll in each.
// embed_mixed.hip covers kassign, slots that differ in their numbers of samples or row
// shapes, and rows wider than 64 chunks.
//
// The memory system fetches 128-byte lines: a table whose rows sit inside lines
// (bz_table_pitch) costs one request per id, and an int8 row's scale lives in the
// row's own line.  Counts come from the caller and are not trusted: negative counts
// are zero and offsets stop at the slot's nnz.
#include <string.h>

#include <limits.h>

#include <mutex>

#include "embed_common.h"

namespace {

// Workgroups of the specialised kernel when the offsets are given: they share nothing then, and smaller ones fill the chip
// more evenly (200 slots x 8192 samples, 64 threads 166.5, 128 167.2, 256 168.2, 512 176 us; 1000 x 24 and 1024 x 26 shortest
// lists 18.2 / 5.4 us at 256 against 17.5 / 6.6 at 64).
constexpr int kOffsetThreads = 256;

// ---------------------------------------------------------------------------------------------
// segments -> offsets (exclusive scan), one workgroup per array
// ---------------------------------------------------------------------------------------------
// A wave holds kScanRows rows of 64 consecutive counts, one count a lane, so that every load and store is one coalesced
// access and the scan runs within the registers: DPP scans of the rows, the rows' totals added up on the way, one barrier
// for the waves' totals.  (Before, every thread owned a run of 8 counts and the layout was turned in 55 KB of LDS, five
// barriers a tile of 4096 and a scan of six dependent trips to LDS: 200 slots x 8192 counts 9.0 us, 7.4-8.0 now.)
constexpr int kScanThreads = 256;
constexpr int kScanRows = 8;
constexpr int kScanWaves = kScanThreads / bz::kWave;
constexpr int kScanTile = kScanThreads * kScanRows;
// the sums of a scan: 32 bits that saturate where the limit allows it, 64 bits without a limit else
struct ScanSat {
  typedef uint32_t T;
  uint32_t cap;
  __device__ T take(int32_t c) const { return (uint32_t)min(max(c, 0), (int)cap); }
  __device__ T add(T a, T b) const { return sat_add(a, b, cap); }
  __device__ T scan(T v, int) const { return wave_scan_sat(v, cap); }
  __device__ T last(T v) const { return (uint32_t)__builtin_amdgcn_readlane((int)v, bz::kWave - 1); }
  __device__ int64_t offset(T v) const { return (int64_t)v; }
};
struct ScanWide {
  typedef int64_t T;
  int64_t limit;
  __device__ T take(int32_t c) const { return max(c, 0); }
  __device__ T add(T a, T b) const { return a + b; }
  __device__ T scan(T v, int lane) const { return wave_incl_scan(v, lane); }
  __device__ T last(T v) const { return __shfl(v, bz::kWave - 1, bz::kWave); }
  __device__ int64_t offset(T v) const { return v < limit ? v : limit; }
};

// Counts below zero are taken as zero and the running offset stops at the limit (the length of the ids / values arrays),
// so no offset this scan produces points outside them.
// Tiles [first_tile, first_tile + n_tiles) of the array (n_tiles < 0: all of them from first_tile on).  A workgroup that
// does not start at tile 0 first adds up the counts before its first tile - all those loads are independent, so a slot's
// scan split over several workgroups takes one tile's time, not the array's.
template <typename S>
__device__ __forceinline__ void scan_tiles(const S sums, const int32_t* __restrict__ seg, int64_t* __restrict__ off, int64_t n,
                                           int64_t first_tile, int64_t n_tiles, int64_t* lds) {
  typedef typename S::T T;
  T* tot = (T*)lds;  // [2][kScanWaves]: tiles take turns, so that one barrier a tile is enough
  const int tid = threadIdx.x;
  const int lane = tid & (bz::kWave - 1), wave = tid / bz::kWave;
  const int64_t begin = first_tile * kScanTile;
  const int64_t end = (n_tiles < 0 || begin + n_tiles * kScanTile > n) ? n : begin + n_tiles * kScanTile;
  if (begin > n || (begin == n && n != 0)) return;  // nothing here; whoever scans the last tile writes off[n]
  // The first tile's counts and those before it, eight times four of these a thread, are all on their way before any is added up.  (One count a
  // load, a trip for every 2048 of them, and the tile's own behind those: 200 slots x 8192 counts in front of their lookups 13.1 us, 8.4 this way.)
  int32_t c[kScanRows];
  auto ask = [&](int64_t base) {
    const int64_t at = base + wave * (kScanRows * bz::kWave) + lane;
#pragma unroll
    for (int k = 0; k < kScanRows; ++k) c[k] = at + k * bz::kWave < n ? seg[at + k * bz::kWave] : 0;
  };
  ask(begin);
  T carry = 0;
  if (begin > 0) {
    T part = 0;
    const i32x4a4* before = (const i32x4a4*)seg;
    const int64_t quads = begin / 4;  // (begin is a whole number of tiles)
    constexpr int kQuads = 8;
    static_assert(kScanTile / 4 % kScanThreads == 0, "a row of quads is there or not for the whole workgroup");
    for (int64_t i = 0; i < quads; i += kQuads * kScanThreads) {
      i32x4a4 q[kQuads];
#pragma unroll
      for (int k = 0; k < kQuads; ++k) {
        q[k] = 0;
        if (i + k * kScanThreads < quads) q[k] = before[i + k * kScanThreads + tid];
      }
#pragma unroll
      for (int k = 0; k < kQuads; ++k)
#pragma unroll
        for (int j = 0; j < 4; ++j) part = sums.add(part, sums.take(q[k][j]));
    }
    part = sums.last(sums.scan(part, lane));
    if (lane == 0) tot[kScanWaves + wave] = part;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kScanWaves; ++w) carry = sums.add(carry, tot[kScanWaves + w]);
  }
  int turn = 0;
  for (int64_t base = begin; base < end; base += kScanTile, turn ^= kScanWaves) {
    const int64_t at = base + wave * (kScanRows * bz::kWave) + lane;
    T excl[kScanRows], run = 0;
#pragma unroll
    for (int k = 0; k < kScanRows; ++k) {
      const T v = sums.take(c[k]);
      const T incl = sums.scan(v, lane);
      // (saturated sums have no inverse: the sum before this lane is the scan's value one lane back)
      T before = __shfl_up(incl, 1, bz::kWave);
      if (lane == 0) before = 0;
      excl[k] = sums.add(run, before);
      run = sums.add(run, sums.last(incl));
    }
    if (base + kScanTile < end) ask(base + kScanTile);
    if (lane == 0) tot[turn + wave] = run;
    __syncthreads();
    T before = carry;
#pragma unroll
    for (int w = 0; w < kScanWaves; ++w) {
      const T t = tot[turn + w];
      if (w < wave) before = sums.add(before, t);
      carry = sums.add(carry, t);
    }
#pragma unroll
    for (int k = 0; k < kScanRows; ++k)
      if (at + k * bz::kWave < n) off[at + k * bz::kWave] = sums.offset(sums.add(before, excl[k]));
  }
  if (tid == 0 && end == n) off[n] = sums.offset(carry);
}

__device__ __forceinline__ void scan_segments(const int32_t* __restrict__ seg, int64_t* __restrict__ off, int64_t n, int64_t limit,
                                              int64_t first_tile, int64_t n_tiles) {
  __shared__ int64_t lds[2 * kScanWaves];
  if (limit < (1ll << 31))
    scan_tiles(ScanSat{(uint32_t)limit}, seg, off, n, first_tile, n_tiles, lds);
  else
    scan_tiles(ScanWide{limit}, seg, off, n, first_tile, n_tiles, lds);
}

// Grid (parts): part p scans tile p, the last part every tile from its own on.
__global__ __launch_bounds__(kScanThreads) void bz_scan_segments_kernel(const int32_t* __restrict__ seg,
                                                                        int64_t* __restrict__ off, int64_t n) {
  scan_segments(seg, off, n, INT64_MAX, blockIdx.x, blockIdx.x + 1 == gridDim.x ? -1 : 1);
}

// ext_off != nullptr: slot i's offsets go to ext_off + i * ext_stride instead of slot.offsets (at most ext_stride - 1
// samples of a slot are scanned, so a record whose batch disagrees with the plan cannot write past its share)
// Grid (slots, parts): parts as above.
__global__ __launch_bounds__(kScanThreads) void bz_scan_segments_slots_kernel(const bz_embed_slot* __restrict__ slots,
                                                                              int64_t* __restrict__ ext_off, int64_t ext_stride) {
  const bz_embed_slot* s = &slots[blockIdx.x];
  const int64_t first = blockIdx.y, count = blockIdx.y + 1 == gridDim.y ? -1 : 1;
  // (all of the record in one trip to memory)
  const int32_t* seg = s->segments;
  int64_t* off = s->offsets;
  int64_t n = s->batch;
  const int64_t nnz = s->nnz;
  if (ext_off != nullptr) {
    off = ext_off + (int64_t)blockIdx.x * ext_stride;
    n = n < ext_stride - 1 ? n : ext_stride - 1;
  }
  scan_segments(seg, off, n, nnz, first, count);
}

// parts a slot's scan is split into: one per tile of the largest batch, at most 8 (a part re-reads the counts before it)
inline int scan_parts(int64_t max_batch) {
  const int64_t tiles = (max_batch + kScanTile - 1) / kScanTile;
  return (int)(tiles < 1 ? 1 : (tiles > 8 ? 8 : tiles));
}
// ---------------------------------------------------------------------------------------------
// the same for the specialised kernel, where lane group g of the workgroup owns sample b0 + g: every lane ends up with
// its own segment [start, end) in registers
// ---------------------------------------------------------------------------------------------
// (sums saturate at cap = nnz, below 2^31 here; larger arrays take stage_offsets.  The counts before b0 in loads of four:
// 26 slots x 16384 samples 66.6 -> 57.9 us with single loads, eight in flight, before)
// start / end of sample b = b0 + g for every lane of lane group g (LPR lanes, g = tid / LPR); lanes of samples beyond
// the batch get an empty segment.  Every thread of the workgroup calls it; one barrier.
template <int LPR, int THREADS>
__device__ __forceinline__ void own_segment(const bz_embed_slot& s, int64_t b0, uint32_t* s_tot, int64_t* start, int64_t* end) {
  constexpr int WAVES = THREADS / bz::kWave;
  static_assert(THREADS / LPR % 4 == 0, "the counts before a workgroup's first sample come in fours");
  const int tid = threadIdx.x;
  const int lane = tid & (bz::kWave - 1), wave = tid / bz::kWave;
  const int g = tid / LPR, l = tid % LPR;
  const int64_t b = b0 + g;
  const uint32_t cap = (uint32_t)s.nnz;
  // this group's own count first (all its lanes ask for the same word), then the counts before b0, four loads of four
  // in flight a thread: everything is requested before anything is used
  const int32_t own = b < s.batch ? s.segments[b] : 0;
  // (b0 is below 2^31: batch is an int32.  A workgroup near the head of its slot has few counts before it: the rounds
  // stop, for the whole workgroup, where b0 ends)
  const uint32_t quads = (uint32_t)bz::counts_before(b0, s.batch) / 4;
  const i32x4a4* before_b0 = (const i32x4a4*)s.segments;
  uint32_t part = 0;
  for (uint32_t i0 = 0; i0 < quads; i0 += 4 * THREADS) {
    i32x4a4 c[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t i = i0 + k * THREADS + tid;
      c[k] = 0;
      if (i0 + k * THREADS < quads) c[k] = before_b0[i < quads ? i : quads - 1];  // (uniform test; a lane past b0 reads the last counts, dropped below)
      if (i >= quads) c[k] = 0;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) part = add_counts_sat(part, c[k], cap);
  }
  const uint32_t mine = min((uint32_t)max(own, 0), cap);
  // the group's count sits in its last lane: after the scan that lane holds the inclusive sum and the group's other
  // lanes the exclusive one (they add nothing)
  const uint32_t scan = wave_scan_sat(l == LPR - 1 ? mine : 0u, cap);
  const uint32_t earlier = wave_scan_sat(part, cap);
  if (lane == bz::kWave - 1) {
    s_tot[wave] = earlier;
    s_tot[WAVES + wave] = scan;
  }
  __syncthreads();
  const uint32_t t = waves_scan_sat<WAVES>(s_tot, cap);
  const uint32_t before = (uint32_t)__builtin_amdgcn_readlane((int)t, WAVES - 1 + wave);
  const uint32_t x = sat_add(before, scan, cap);
  if constexpr (LPR == 1) {
    uint32_t excl = (uint32_t)__shfl_up((int)scan, 1, bz::kWave);
    if (lane == 0) excl = 0;
    *start = (int64_t)sat_add(before, excl, cap);
    *end = (int64_t)x;
  } else if constexpr (LPR == 2 || LPR == 4) {  // (an operand, where a shuffle is a trip to LDS)
    *start = (int64_t)(uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, LPR == 4 ? 0x00 : 0xa0, 0xf, 0xf, true);  // quad_perm
    *end = (int64_t)(uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, LPR == 4 ? 0xff : 0xf5, 0xf, 0xf, true);
  } else {
    const int gbase = lane - l;
    *start = (int64_t)(uint32_t)__shfl((int)x, gbase, bz::kWave);
    *end = (int64_t)(uint32_t)__shfl((int)x, gbase + LPR - 1, bz::kWave);
  }
}

// ---------------------------------------------------------------------------------------------
// specialised ksum / kavg kernel: every slot has table dtype DT and LPR lanes per row
// ---------------------------------------------------------------------------------------------
template <int DT, int LPR, int THREADS, bool KEYED>
__device__ __forceinline__ void pool_samples(const bz_embed_slot& s, int64_t b0, const int64_t* __restrict__ offsets) {
  constexpr int GROUPS = THREADS / LPR;
  __shared__ int64_t s_off[GROUPS + 1];
  __shared__ int64_t s_part[2 * THREADS / bz::kWave];
  const int tid = threadIdx.x;
  const int g = tid / LPR, l = tid % LPR;
  int64_t start, end;
  if (offsets == nullptr && s.nnz < (1ll << 31)) {
    own_segment<LPR, THREADS>(s, b0, (uint32_t*)s_part, &start, &end);
  } else if (offsets != nullptr) {
    // every lane of a group asks for its sample's two offsets itself (one address a group): nothing goes through LDS
    // and no wave waits for another's.  Caller-made offsets get the same bounds as the scan's.
    const int64_t bb = b0 + g < s.batch ? b0 + g : s.batch - 1;  // (lanes past the batch: any)
    const int64_t o0 = offsets[bb], o1 = offsets[bb + 1];
    start = o0 < 0 ? 0 : (o0 < s.nnz ? o0 : s.nnz);
    end = o1 < 0 ? 0 : (o1 < s.nnz ? o1 : s.nnz);
  } else {
    stage_offsets<THREADS>(s, offsets, b0, GROUPS, s_off, s_part);
    start = s_off[g];
    end = s_off[g + 1];
  }
  const int64_t b = b0 + g;
  sum_samples<DT, LPR, KEYED>(s, start, end, l, b, b < s.batch);
}

template <int DT, int LPR, int THREADS, bool KEYED>
__global__ __launch_bounds__(THREADS) void bz_embed_pool_kernel(const bz_embed_slot* __restrict__ slots, int n_slots,
                                                                 int total_wg, int wg_per_xcd, int wg_per_slot,
                                                                 const int64_t* __restrict__ ext_off, int64_t ext_stride) {
  constexpr int GROUPS = THREADS / LPR;
  const int v = (int)(blockIdx.x % bz::kNumXcd) * wg_per_xcd + (int)(blockIdx.x / bz::kNumXcd);
  if (v >= total_wg) return;
  const int si = v / wg_per_slot;
  const bz_embed_slot s = slots[si];
  const int64_t b0 = (int64_t)(v - si * wg_per_slot) * GROUPS;
  pool_samples<DT, LPR, THREADS, KEYED>(s, b0, ext_off != nullptr ? ext_off + (int64_t)si * ext_stride : s.offsets);
}

template <int DT, int LPR, int THREADS, bool KEYED>
__global__ __launch_bounds__(THREADS) void bz_embed_pool_args_kernel(int total_wg, int wg_per_xcd, int wg_per_slot,
                                                                      const SlotPack pack) {
  constexpr int GROUPS = THREADS / LPR;
  const int v = (int)(blockIdx.x % bz::kNumXcd) * wg_per_xcd + (int)(blockIdx.x / bz::kNumXcd);
  if (v >= total_wg) return;
  const int si = v / wg_per_slot;
  const bz_embed_slot s = pack.s[si];
  const int64_t b0 = (int64_t)(v - si * wg_per_slot) * GROUPS;
  pool_samples<DT, LPR, THREADS, KEYED>(s, b0, s.offsets);
}

// When workgroups that find their offsets themselves have 256 threads instead of 512: where the larger ones would leave CUs without any, and
// for the forms whose walk takes more than 64 registers (int8 rows, slots looked up by key), of which three of the larger ones share a CU
// and not four; unless the counts in front of each workgroup, which twice as many then read, are more than 32 MB.
// us with 512 / 256 threads, by workgroups of 512: 6 (223 x 3 lists of 9 ids, fp16) 4.7 / 4.4, 10 (108 x 10 of 22, int8) 9.7 / 7.5, 72 (380 x 3 of 22,
// fp32 rows of 128) 5.4 / 4.5, 95 (1058 x 19 of 12, fp16) 6.3 / 5.0, 119 (1050 x 7 of 21) 5.9 / 4.8, 208 (1024 x 26 of 8) 5.0 / 4.9; but 400 (100 x 200
// of 10) 6.4 / 6.8, 416 (2048 x 26 of 8) 7.0 / 7.0 and on eight serving threads 12.1 / 12.2 a pass.  int8: 580 (7193 x 20 of 17) 42.0 / 36.7, 1600 (4096
// x 50 of 20) 52.6 / 49.8, 3486 (10539 x 83 of 21, 146 MB of counts) 295 / 297.  By key: 1512 (1000 x 24 of 6, fp32 rows of 100) 14.7 / 13.8, 54
// (300 x 18 of 3, fp16) 5.6 / 5.2, a request with them 39.4 / 38.8; 1011 (10782 x 6 of 20, 43 MB of counts) 29.3 / 30.3.
constexpr int kSmallThreads = 256;
constexpr int kSmallGroups = 256;
constexpr int64_t kSmallBytes = 32ll << 20;
inline bool small_groups(const bz_embed_launch& L, int dtype, bool keyed) {
  const int64_t groups = (int64_t)L.total_wg * (kThreads / kSmallThreads);
  return (L.total_wg < kSmallGroups || dtype == BZ_I8 || keyed) && groups * L.max_batch * 2 <= kSmallBytes;
}

// When a separate scan launch (4.2-8 us, and 3-4 between the launches) is cheaper than the fused scan, whose cost is one
// preamble a workgroup and, with long batches, the counts read again and again: above this many workgroups of 512 threads
// of the specialised kernel, or above this many bytes of repeated reads.  Fused / scan + pool in us, by workgroups: 1600 (int8, 20 ids) 80 / 84, 1664
// (26 slots x 8192 of 64-byte rows) 23 / 27, 3328 (16384) 57 / 59.5, 3840 (60 slots x 16384, 32-byte rows) 76 / 81, 5040 40 /
// 41.7 and 75 / 70, 5120 38.5 / 34, 7560 (120 slots x 1000, 400-byte rows) 60.5 / 57, 15360 117 / 96, 25600 (200 slots x 8192)
// 219 / 180.  A plan whose records may travel as kernel arguments needs no upload of them when fused: twice as many there.
constexpr int64_t kScanFirstGroups = 5000;
constexpr int64_t kScanFirstBytes = 128ll << 20;

int groups_per_wg(const bz_embed_slot& s) {
  const int ce = s.table_dtype == BZ_F32 ? 4 : (s.table_dtype == BZ_F16 ? 8 : 16);
  const int nchunks = (s.dim + ce - 1) / ce;
  int lpr = 1;
  while (lpr < nchunks && lpr < bz::kWave) lpr <<= 1;
  return kThreads / lpr;
}

// ---------------------------------------------------------------------------------------------
// scratch of the entry point that allocates nothing: every slot's offsets, inside the library's own device image
// ---------------------------------------------------------------------------------------------
constexpr int64_t kStaticScratchEntries = BZ_EMBED_STATIC_SCRATCH_BYTES / sizeof(int64_t);
static __device__ __align__(256) int64_t scratch[kStaticScratchEntries];

// Device address of `scratch` on the current device.  In host code the array's name is only a handle: the address
// comes from hipGetSymbolAddress, asked once per device with that device current (every GPU holds its own copy of the
// array at its own address), and only that pointer is ever handed to a kernel.
constexpr int kMaxDevices = 64;
int static_scratch_ptr(int64_t** out) {
  static std::mutex mu;
  static int64_t* ptr[kMaxDevices] = {};
  int dev = -1;
  BZ_HIP_OK(hipGetDevice(&dev));
  BZ_REQUIRE(dev >= 0 && dev < kMaxDevices, "device ordinal %d outside [0, %d)", dev, kMaxDevices);
  std::lock_guard<std::mutex> lock(mu);
  if (ptr[dev] == nullptr) {
    void* p = nullptr;
    BZ_HIP_OK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    BZ_REQUIRE(p != nullptr, "hipGetSymbolAddress gave no address for the scratch buffer on device %d", dev);
    ptr[dev] = static_cast<int64_t*>(p);
  }
  *out = ptr[dev];
  return BZ_OK;
}

}  // namespace

extern "C" {

int32_t bz_table_pitch(int64_t row_bytes, int scale_bytes) {
  if (row_bytes <= 0 || row_bytes > (1 << 24)) return 0;
  int64_t need = (row_bytes + 3) / 4 * 4 + (scale_bytes > 0 ? 4 : 0);
  need = (need + 15) / 16 * 16;
  if (need <= 128) {
    int64_t p = 16;
    while (p < need) p <<= 1;
    return (int32_t)p;
  }
  const int64_t lines = (need + 127) / 128 * 128;
  return (int32_t)(lines * 3 <= need * 4 ? lines : need);
}

int bz_embed_plan(bz_embed_slot* slots, int n_slots, bz_embed_launch* launch) {
  BZ_REQUIRE(slots != nullptr && launch != nullptr && n_slots > 0, "bz_embed_plan: null argument or n_slots=%d", n_slots);
  int64_t total = 0;
  bool uniform_wg = true, uniform_shape = true, one_shape = true, any_offsets = false, all_offsets = true, keyed = false;
  int lpr0 = 0;
  for (int i = 0; i < n_slots; ++i) {
    bz_embed_slot& s = slots[i];
    BZ_REQUIRE(s.table_dtype == BZ_F32 || s.table_dtype == BZ_F16 || s.table_dtype == BZ_I8,
               "slot %d: unsupported table dtype %d", i, s.table_dtype);
    BZ_REQUIRE(s.out_dtype == BZ_F32 || s.out_dtype == BZ_F16 || s.out_dtype == BZ_BF16, "slot %d: unsupported out dtype %d", i,
               s.out_dtype);
    BZ_REQUIRE(s.udf == BZ_SUM || s.udf == BZ_AVG || s.udf == BZ_ASSIGN, "slot %d: Unsupported udf type: %d", i, s.udf);
    BZ_REQUIRE(s.dim > 0 && s.batch >= 0 && s.nnz >= 0, "slot %d: dim=%d batch=%d nnz=%lld", i, s.dim, s.batch, (long long)s.nnz);
    if (s.udf == BZ_ASSIGN)
      BZ_REQUIRE(s.trunc_num > 0 && (s.trunc_dir == BZ_ORDER || s.trunc_dir == BZ_REVERSE),
                 "slot %d: kAssign needs trunc_num > 0 and a trunc direction (trunc_num=%d dir=%d)", i, s.trunc_num,
                 s.trunc_dir);
    BZ_REQUIRE(s.assign_pitch == 0 || (s.udf == BZ_ASSIGN && s.assign_pitch >= s.dim),
               "slot %d: assign_pitch=%d is for kAssign items and at least dim=%d", i, s.assign_pitch, s.dim);
    BZ_REQUIRE(s.out != nullptr && (s.batch == 0 || s.segments != nullptr), "slot %d: null out/segments", i);
    if (s.table != nullptr) {
      const int esz = bz::dtype_size(s.table_dtype);
      BZ_REQUIRE(s.pitch % 16 == 0 && s.pitch >= ((s.dim * esz + 15) / 16) * 16,
                 "slot %d: row pitch %d must be a multiple of 16 covering dim*elem=%d", i, s.pitch, s.dim * esz);
      BZ_REQUIRE(((uintptr_t)s.table & 15) == 0, "slot %d: table base not 16-byte aligned", i);
      BZ_REQUIRE(s.table_dtype != BZ_I8 || s.row_scale != nullptr, "slot %d: int8 table without row_scale", i);
      BZ_REQUIRE(s.scale_pitch >= 0 && s.scale_pitch % 4 == 0 && ((uintptr_t)s.row_scale & 3) == 0,
                 "slot %d: scale_pitch=%d / row_scale must be multiples of 4", i, s.scale_pitch);
      BZ_REQUIRE(s.rows > 0 && s.rows < (1ll << 31), "slot %d: rows=%lld outside (0, 2^31)", i, (long long)s.rows);
      BZ_REQUIRE(s.nnz == 0 || (s.ids != nullptr && s.values != nullptr), "slot %d: null ids/values", i);
      if (s.hash_buckets != nullptr)
        BZ_REQUIRE(s.hash_pairs != nullptr && s.hash_bucket_size > 0, "slot %d: incomplete hash index", i);
    }
    keyed |= s.table != nullptr && s.hash_buckets != nullptr;
    any_offsets |= s.offsets != nullptr;
    all_offsets &= s.offsets != nullptr;
    const int g = groups_per_wg(s);
    const int lpr = kThreads / g;
    const int ce = s.table_dtype == BZ_F32 ? 4 : (s.table_dtype == BZ_F16 ? 8 : 16);
    s.wg_begin = (int32_t)total;
    const int64_t items = (int64_t)s.batch * items_per_sample(s);  // lane groups needed
    BZ_REQUIRE((items + g - 1) / g < (1ll << 30), "slot %d: too many workgroups", i);
    s.wg_count = (int32_t)((items + g - 1) / g);
    total += s.wg_count;
    BZ_REQUIRE(total < (1ll << 30), "too many workgroups");
    if (i == 0) lpr0 = lpr;
    uniform_wg &= s.wg_count == slots[0].wg_count;
    one_shape &= s.table != nullptr && lpr == lpr0 && s.table_dtype == slots[0].table_dtype && (s.dim + ce - 1) / ce <= lpr;
    uniform_shape &= s.udf != BZ_ASSIGN;
  }
  BZ_REQUIRE(all_offsets || !any_offsets, "either every slot carries offsets or none does");
  launch->n_slots = n_slots;
  launch->total_wg = (int32_t)total;
  launch->wg_per_slot = (uniform_wg && slots[0].wg_count > 0) ? slots[0].wg_count : 0;
  launch->variant = (one_shape && uniform_shape && launch->wg_per_slot > 0) ? ((slots[0].table_dtype << 8) | lpr0) : 0;
  launch->fused_scan = any_offsets ? 0 : 1;
  // the fused scan reads, per workgroup, the counts before its first sample: on average batch/2 counts of 4 bytes
  int64_t prefix_bytes = 0;
  for (int i = 0; i < n_slots; ++i) prefix_bytes += (int64_t)slots[i].wg_count * slots[i].batch * 2;
  const int64_t most = n_slots <= BZ_EMBED_ARG_SLOTS ? 2 * kScanFirstGroups : kScanFirstGroups;
  launch->scan_first = (launch->fused_scan && ((launch->variant != 0 && total > most) || prefix_bytes > kScanFirstBytes)) ? 1 : 0;
  int32_t max_batch = 0;
  for (int i = 0; i < n_slots; ++i) max_batch = slots[i].batch > max_batch ? slots[i].batch : max_batch;
  launch->max_batch = max_batch;
  launch->shape = (launch->variant == 0 && one_shape) ? ((slots[0].table_dtype << 8) | lpr0) : 0;
  if (keyed && (launch->variant != 0 || launch->shape != 0)) launch->shape |= kShapeKeyed;
  return BZ_OK;
}

int bz_segments_to_offsets(const int32_t* segments, int64_t* offsets, int64_t n, bz_stream_t stream) {
  BZ_REQUIRE(offsets != nullptr && n >= 0 && (n == 0 || segments != nullptr), "bz_segments_to_offsets: null argument");
  BZ_REQUIRE(n <= (1ll << 24), "bz_segments_to_offsets: n=%lld exceeds 2^24", (long long)n);
  hipLaunchKernelGGL(bz_scan_segments_kernel, dim3(scan_parts(n)), dim3(kScanThreads), 0, bz::as_stream(stream), segments, offsets, n);
  BZ_LAUNCH_OK("bz_scan_segments_kernel");
  return BZ_OK;
}

int bz_segments_to_offsets_slots(const bz_embed_slot* slots_dev, int n_slots, bz_stream_t stream) {
  BZ_REQUIRE(slots_dev != nullptr && n_slots > 0, "bz_segments_to_offsets_slots: null argument or n_slots=%d", n_slots);
  // the batch sizes are in device memory: always 8 parts a slot; a part beyond its slot's batch returns at once
  hipLaunchKernelGGL(bz_scan_segments_slots_kernel, dim3(n_slots, 8), dim3(kScanThreads), 0, bz::as_stream(stream), slots_dev,
                     (int64_t*)nullptr, (int64_t)0);
  BZ_LAUNCH_OK("bz_scan_segments_slots_kernel");
  return BZ_OK;
}

// launches the pooling kernel the plan chose; ext_off (may be nullptr) replaces slot.offsets as described at the kernels
static int launch_pool(const bz_embed_slot* slots_dev, const bz_embed_launch& L, const int64_t* ext_off, int64_t ext_stride,
                       hipStream_t st) {
  BZ_REQUIRE(L.n_slots > 0 && L.total_wg >= 0 && L.wg_per_slot >= 0, "bz_embed_pool: bad launch record (n_slots=%d total_wg=%d)",
             L.n_slots, L.total_wg);
  if (L.total_wg == 0) return BZ_OK;
  if (L.variant == 0) return bz::embed_launch_mixed(slots_dev, L, ext_off, ext_stride, st);
  BZ_REQUIRE(L.wg_per_slot > 0 && (int64_t)L.wg_per_slot * L.n_slots == L.total_wg,
             "bz_embed_pool: variant %#x needs equal work per slot", L.variant);
  // with offsets given: smaller workgroups, each with its share of a planned workgroup's samples
  const bool scanned = ext_off != nullptr || !L.fused_scan;
  const int rc = with_shape(L.variant, (L.shape & kShapeKeyed) != 0, [&](auto dt, auto lpr, auto keyed) {
    auto launch = [&](auto threads) {
      constexpr int kEach = decltype(threads)::value;
      const bz::PoolGrid grid(L.total_wg, L.wg_per_slot, kThreads / kEach);
      hipLaunchKernelGGL((bz_embed_pool_kernel<decltype(dt)::value, decltype(lpr)::value, kEach, decltype(keyed)::value>), dim3(grid.blocks), dim3(kEach),
                         0, st, slots_dev, L.n_slots, grid.total_wg, grid.wg_per_xcd, grid.wg_per_slot, ext_off, ext_stride);
    };
    static_assert(kOffsetThreads == kSmallThreads, "one kernel for both");
    if (scanned || small_groups(L, decltype(dt)::value, decltype(keyed)::value))
      launch(std::integral_constant<int, kSmallThreads>{});
    else
      launch(std::integral_constant<int, kThreads>{});
  });
  if (rc != BZ_OK) return rc;
  BZ_LAUNCH_OK("bz_embed_pool_kernel");
  return BZ_OK;
}

int bz_embed_pool(const bz_embed_slot* slots_dev, const bz_embed_launch* launch, bz_stream_t stream) {
  BZ_REQUIRE(slots_dev != nullptr && launch != nullptr, "bz_embed_pool: null argument");
  return launch_pool(slots_dev, *launch, nullptr, 0, bz::as_stream(stream));
}

int bz_embed_pool_args(const bz_embed_slot* slots_host, const bz_embed_launch* launch, bz_stream_t stream) {
  BZ_REQUIRE(slots_host != nullptr && launch != nullptr, "bz_embed_pool_args: null argument");
  const bz_embed_launch& L = *launch;
  BZ_REQUIRE(L.n_slots > 0 && L.total_wg >= 0 && L.wg_per_slot >= 0, "bz_embed_pool_args: bad launch record (n_slots=%d total_wg=%d)",
             L.n_slots, L.total_wg);
  if (L.n_slots > BZ_EMBED_ARG_SLOTS || !L.fused_scan || L.scan_first)
    return bz::fail(BZ_ENOTSUP, "bz_embed_pool_args: takes plans with at most %d slots and the scan fused in", BZ_EMBED_ARG_SLOTS);
  BZ_REQUIRE(L.variant == 0 || (L.wg_per_slot > 0 && (int64_t)L.wg_per_slot * L.n_slots == L.total_wg),
             "bz_embed_pool_args: variant %#x needs equal work per slot", L.variant);
  if (L.total_wg == 0) return BZ_OK;
  if (L.variant == 0) return bz::embed_launch_mixed_args(slots_host, L, bz::as_stream(stream));
  SlotPack pack;
  memcpy(pack.s, slots_host, (size_t)L.n_slots * sizeof(bz_embed_slot));
  memset(pack.s + L.n_slots, 0, (size_t)(BZ_EMBED_ARG_SLOTS - L.n_slots) * sizeof(bz_embed_slot));
  hipStream_t st = bz::as_stream(stream);
  const int rc = with_shape(L.variant, (L.shape & kShapeKeyed) != 0, [&](auto dt, auto lpr, auto keyed) {
    auto launch = [&](auto threads) {
      constexpr int kEach = decltype(threads)::value;
      const bz::PoolGrid grid(L.total_wg, L.wg_per_slot, kThreads / kEach);
      hipLaunchKernelGGL((bz_embed_pool_args_kernel<decltype(dt)::value, decltype(lpr)::value, kEach, decltype(keyed)::value>), dim3(grid.blocks),
                         dim3(kEach), 0, st, grid.total_wg, grid.wg_per_xcd, grid.wg_per_slot, pack);
    };
    if (small_groups(L, decltype(dt)::value, decltype(keyed)::value))
      launch(std::integral_constant<int, kSmallThreads>{});
    else
      launch(std::integral_constant<int, kThreads>{});
  });
  if (rc != BZ_OK) return rc;
  BZ_LAUNCH_OK("bz_embed_pool_args_kernel");
  return BZ_OK;
}

int bz_embed_pool_static_scratch(const bz_embed_slot* slots_dev, const bz_embed_launch* launch, bz_stream_t stream) {
  BZ_REQUIRE(slots_dev != nullptr && launch != nullptr, "bz_embed_pool_static_scratch: null argument");
  const bz_embed_launch& L = *launch;
  BZ_REQUIRE(L.n_slots > 0 && L.max_batch >= 0, "bz_embed_pool_static_scratch: bad launch record (n_slots=%d max_batch=%d)",
             L.n_slots, L.max_batch);
  const int64_t stride = (int64_t)L.max_batch + 1;  // int64 entries per slot
  BZ_REQUIRE((int64_t)L.n_slots * stride <= kStaticScratchEntries,
             "bz_embed_pool_static_scratch: %d slots x (batch %d + 1) offsets = %lld bytes exceed the library's %u-byte buffer",
             L.n_slots, L.max_batch, (long long)((int64_t)L.n_slots * stride * 8), BZ_EMBED_STATIC_SCRATCH_BYTES);
  int64_t* off = nullptr;
  const int rc = static_scratch_ptr(&off);
  if (rc != BZ_OK) return rc;
  hipStream_t st = bz::as_stream(stream);
  // nothing to clear: the scan writes entries [0, batch] of every slot's share, the only ones the pooling kernel reads
  hipLaunchKernelGGL(bz_scan_segments_slots_kernel, dim3(L.n_slots, scan_parts(L.max_batch)), dim3(kScanThreads), 0, st, slots_dev, off,
                     stride);
  BZ_LAUNCH_OK("bz_scan_segments_slots_kernel");
  return launch_pool(slots_dev, L, off, stride, st);
}

const char* bz_embed_pool_kernel_name(void) { return "bz_embed_pool_kernel"; }

}  // extern "C"
