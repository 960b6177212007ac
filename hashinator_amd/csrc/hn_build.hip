// hn_build.hip -- bulk insert into an empty table, written directly in Robin
// Hood order.
//
// An insert of n keys into an empty linear-probing table (kernels_AMD.h
// insert_kernel on a fresh map) followed by the reorder pass gives one image
// that depends on the key set alone: in every cluster the keys stand in order
// of home slot, ties by key.  That image is also what a max-plus scan gives
// over the keys sorted by (home, key):  position_j = max(home_j,
// position_{j-1} + 1), taken cyclically.  This file computes it without
// probing:
//
//   1. stable radix partition of the (key, value) pairs by region
//      (region = home >> log2 R, R = 2048 slots): per pass a per-tile digit
//      count, an exclusive scan of the digit-major count matrix, and a stable
//      multisplit scatter through LDS (digits of at most 9 bits, 1-3 passes);
//   2. region boundaries in the partitioned array (a binary search per
//      region; after a single pass, whose digits are the regions, the digits'
//      own offsets);
//   3. per region, in LDS: sort by (home, key), drop all but the last
//      occurrence of a repeated key (the value a serial insert leaves), and
//      summarise the region as the carry function g(c) = max(a, c + b), where
//      c is the number of keys spilling into the region from before it;
//   4. a workgroup walks 16 consecutive regions, handing the carry from one
//      to the next (carry out = max(a, c + b); the walk starts from the
//      region before it, taken with no carry in), places each region's keys
//      with a max-scan and writes its slot range (keys and EMPTY slots)
//      once, coalesced;
//   5. one scan composes the carry functions (g2 after g1 is
//      (max(a2, a1 + b2), b1 + b2)) into the true carries (the carry into
//      region 0 is the least fixed point of the whole-table composition,
//      max(A, c + B) with B = n - N < 0, i.e. c0 = A), and the regions whose
//      carry was wrong, or whose range wraps past the table's end, are
//      placed again.
//
// A build of a small table is mostly its launches, so what can ride along
// does: the first count decides whether the build runs and clears the words
// of the scan behind it, the only scatter leaves the region boundaries, one
// workgroup does the carries of up to 4,096 regions, and the fix-up kernel
// empties the table for the fallback (15 launches -> 9: 2^20 u32 slots at
// load factor 0.5 0.086 -> 0.061 ms, 2^18 u64 at 0.9 0.090 -> 0.069 ms).
//
// Traffic per key: the first partition pass reads the key for its count,
// each pass reads and writes the 16 (u64) or 8 (u32) byte pair, and a pass
// whose successor's digit fits a byte also writes that digit at the pair's
// output position, so the successor counts from one byte per pair instead of
// the pair; the region step reads the pair once more and the table is
// written once.  No atomics on the table, no probing.
//
// The table's memory is the output of the first partition pass when there
// are two, so the scratch holds one pair array, not two.  A region holding
// more than kRegionCap keys (only with strongly skewed keys) abandons the
// placement on the device: the table is emptied and the probing insert
// places the partitioned pairs (by k_region_fix, then k_insert), so the
// call still ends with err = SUCCESS (or FAIL if a key found no slot), the
// same live set in arrival order, and HN_INFO_ORDERED not set.  A table that
// is not empty (fill or tombstones nonzero) is answered with err = INVALID
// and left untouched.
#include <algorithm>
#include <atomic>

#include "hn_device.hpp"
#include "hn_host.hpp"
#include "hn_probe.hpp"

namespace hn {

constexpr int kRegionLog = 11;   // 2048 slots per region
constexpr int kPartBS = 256;     // count workgroup
constexpr int kPartBSS = 512, kPartRoundsS = 8;   // 4,096-pair scatter tiles: threads, pairs per thread
constexpr int kPartBSL = 1024, kPartRoundsL = 8;  // 8,192-pair scatter tiles
// Scatter tiles: 8,192 pairs (16-pair runs per 9-bit digit, one block per CU)
// for inputs of at least kPartLargeMin pairs, 4,096 (two blocks per CU) below.
// The scatter is bound by its scattered writes: longer runs per digit mean
// fewer partial lines (2^28 u64 slots at LF 0.9, 242 M pairs: 7.97 ms against
// 8.66 ms with the small tile; 2^26, 60 M: 2.01 against 2.07 ms), while the
// small tile's two blocks keep a CU busy where the table stays in the caches
// (2^24, 15 M pairs: 0.56 against 0.60 ms).  The small tile's 512 threads of
// 8 pairs (88 VGPRs, four waves per SIMD) instead of 256 of 16 (151 VGPRs,
// two) took the 2^20-slot build from 0.120 to 0.115 ms, 2^22 from 0.218 to
// 0.202.  The next tile's loads issued a whole tile ahead, with nothing that
// waits for a tile's stores, left the 2^28 scatters at 2.68 + 2.08 ms: the
// memory, not the wait for it, is the bound.
constexpr uint32_t kPartTileS = 4096;
constexpr uint32_t kPartTileL = 8192;
constexpr uint64_t kPartLargeMin = 1ull << 25;
constexpr int kPartSub = 8;      // tiles per partition block at most (fewer for small inputs)
constexpr int kMaxDigitBits = 9; // 512 digits per pass at most
constexpr int kRegionBS = 512;
constexpr int kRegionIPT = 5;
constexpr int kRegionCap = kRegionBS * kRegionIPT; // keys per region held in LDS

struct BuildHeader {
   uint32_t go;        // the table was empty: the build runs
   uint32_t fail;      // a region over capacity: the build is abandoned
   uint32_t max_probe; // longest probe (displacement + 1) of the placed keys
   uint32_t pad0;
   int64_t c0;         // carry into region 0
   uint64_t n_distinct;
   uint32_t n_fix;     // regions placed again after the carries are known
   int32_t fb_fail;    // the fallback insert found no slot for a key
   uint64_t n;         // pairs after the first partition pass (the live slots when the input is a table)
   uint64_t fb_len;    // pairs the fallback insert takes from the partitioned array (0: none)
   uint64_t prior_fill; // rehash: the old table's fill, which the new one must hold
   uint64_t grow_old, grow_new; // rehash with a batch: the old table's slots, the batch's length (else 0)
   uint64_t fb_new;     // its fallback: pairs taken from the batch (fb_len then counts old slots)
   uint32_t pad[42];
};
static_assert(sizeof(BuildHeader) == 256, "header is one 256-byte line");

struct RegionSum {
   int64_t a, b; // carry out = max(a, carry in + b)
};

struct BuildPlan {
   int sp;
   uint64_t n;          // input pairs
   uint64_t N;          // slots
   int rlog;            // log2 slots per region
   uint64_t R;          // slots per region
   uint64_t NR;         // regions
   int rbits;           // log2 NR
   int passes;          // partition passes
   int dbits[3];        // digit bits per pass (low digit first)
   uint32_t nblocks;    // partition blocks
   uint32_t tile;       // pairs per scatter tile (kPartTileS or kPartTileL)
   uint32_t sub;        // tiles per partition block
   size_t off_pairs, off_mat, off_scan, off_start, off_word, off_spec, off_carry, off_mark, off_list, off_blk, off_dig,
       total;
};

inline size_t align256(size_t x) { return (x + 255) / 256 * 256; }

// The scratch layouts place their arrays at 256-byte offsets from the start
// and read them with 16-byte loads, so the start must be 256-byte aligned
// (hipMalloc's and hipMallocAsync's are).
inline bool scratch_aligned(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 255u) == 0; }

// dcap: widest partition digit (1..9 bits); narrower digits mean more passes.
template <typename K>
bool build_plan(int sp, uint64_t n, int dcap, BuildPlan* P) {
   if (dcap < 1 || dcap > kMaxDigitBits) return false;
   if (sp < 1 || sp > std::min(max_size_power<K>(), 32)) return false;
   P->sp = sp;
   P->n = n;
   P->N = 1ull << sp;
   if (n == 0 || n >= P->N) return false;
   P->rlog = std::min(sp, kRegionLog);
   P->R = 1ull << P->rlog;
   P->rbits = sp - P->rlog;
   P->NR = 1ull << P->rbits;
   P->passes = std::max(1, (P->rbits + dcap - 1) / dcap);
   if (P->passes > 3) return false;
   int left = P->rbits;
   for (int i = 0; i < P->passes; ++i) {
      P->dbits[i] = left / (P->passes - i) + ((left % (P->passes - i)) ? 1 : 0);
      left -= P->dbits[i];
   }
   // Tiles per block: kPartSub, or as few as keep the blocks within one
   // resident round (2 small-tile or 1 large-tile scatter blocks per CU):
   // more blocks than that would leave a partial second round.
   P->tile = n >= kPartLargeMin ? kPartTileL : kPartTileS;
   const uint64_t tiles = (n + P->tile - 1) / P->tile;
   const uint64_t slots = static_cast<uint64_t>(cu_count()) * (P->tile == kPartTileL ? 1 : 2);
   const uint64_t per = (tiles + slots - 1) / slots;
   P->sub = static_cast<uint32_t>(per < 1 ? 1 : (per > kPartSub ? kPartSub : per));
   const uint64_t super = static_cast<uint64_t>(P->tile) * P->sub;
   const uint64_t nb = (n + super - 1) / super;
   if (nb > 0xFFFFFFFFull) return false;
   P->nblocks = static_cast<uint32_t>(nb);
   // Sized for the default digit width, so any narrower one fits the same scratch.
   const uint64_t mat = (1ull << kMaxDigitBits) * nb;
   size_t o = sizeof(BuildHeader);
   P->off_pairs = o;
   o = align256(o + n * sizeof(Slot<K>));
   P->off_mat = o;
   o = align256(o + mat * sizeof(uint32_t));
   P->off_scan = o;
   o = align256(o + hn_compact_scratch_bytes(mat));
   P->off_start = o;
   o = align256(o + (P->NR + 1) * sizeof(uint64_t));
   P->off_word = o;
   o = align256(o + P->NR * sizeof(uint64_t));
   P->off_spec = o;
   o = align256(o + P->NR * sizeof(int64_t));
   P->off_carry = o;
   o = align256(o + P->NR * sizeof(int64_t));
   P->off_mark = o;
   o = align256(o + P->NR * sizeof(uint32_t));
   P->off_list = o;
   o = align256(o + P->NR * sizeof(uint32_t));
   P->off_blk = o;
   o = align256(o + ((P->NR + 1023) / 1024) * sizeof(RegionSum));
   // One byte per pair: the next pass's digit, written by a scatter pass
   // whose successor's digit fits a byte (reserved for every plan of more
   // than one region, so the size does not depend on the digit width).
   P->off_dig = o;
   if (P->NR > 1) o = align256(o + n);
   P->total = o;
   return true;
}

// Input of a partition pass: the caller's arrays (pass 0) or a pair array.
template <typename K>
struct PartIn {
   const K* keys;        // SRC_SOA / SRC_INDEX
   const K* vals;        // SRC_SOA
   const Slot<K>* pairs; // SRC_PAIRS / SRC_TABLE (a pair array)
   // SRC_GROW: the n_table slots of `table`, then the batch in one of the forms above
   const Slot<K>* table;
   uint64_t n_table;
};
constexpr int SRC_GROW = SRC_TABLE + 1;

template <typename K, int SRC>
__device__ __forceinline__ K part_key(const PartIn<K>& in, uint64_t e) {
   if constexpr (SRC == SRC_SOA || SRC == SRC_INDEX) {
      return in.keys[e];
   } else if constexpr (SRC == SRC_GROW) {
      if (e < in.n_table) return in.table[e].key;
      return in.pairs ? in.pairs[e - in.n_table].key : in.keys[e - in.n_table];
   } else {
      return in.pairs[e].key;
   }
}

template <typename K, int SRC>
__device__ __forceinline__ Slot<K> part_pair(const PartIn<K>& in, uint64_t e) {
   Slot<K> s;
   if constexpr (SRC == SRC_SOA) {
      s.key = in.keys[e];
      s.val = in.vals[e];
   } else if constexpr (SRC == SRC_INDEX) {
      s.key = in.keys[e];
      s.val = static_cast<K>(e);
   } else if constexpr (SRC == SRC_GROW) {
      const uint64_t q = e - in.n_table;
      if (e < in.n_table) {
         s = in.table[e];
      } else if (in.pairs) {
         s = in.pairs[q];
      } else {
         s.key = in.keys[q];
         s.val = in.vals ? in.vals[q] : static_cast<K>(q);
      }
   } else {
      s = in.pairs[e];
   }
   return s;
}

// A table's EMPTY and TOMBSTONE slots are left out, and a batch's EMPTY keys
// (a padded batch's: the probing insert finds such a key in the first EMPTY
// slot and places nothing).
template <typename K, int SRC>
__device__ __forceinline__ bool part_live(const PartIn<K>& in, uint64_t e, K key) {
   return key != empty_key<K>() && (key != tomb_key<K>() || (SRC == SRC_GROW && e >= in.n_table));
}

template <typename K>
__device__ __forceinline__ uint32_t region_of(K key, int sp, int rlog) {
   const uint64_t mask = (1ull << sp) - 1;
   return static_cast<uint32_t>((fib_home(key, sp) & mask) >> rlog);
}

// Build from caller arrays into an empty table, (rehash) from the live
// slots of another, smaller table into a new one, (grow) from those and
// caller arrays, or (merge) from caller arrays and an ordered table into a
// second array of the table's size.
enum BuildMode { BUILD_EMPTY = 0, BUILD_REHASH = 2, BUILD_MERGE = 3, BUILD_GROW = 4 };

// What the first kernel of a build does besides its own work: with `info`
// set, decide whether the build runs and set up its header (a launch of its
// own otherwise, k_build_begin); and clear the look-back words of the scan
// that follows.
struct BuildBegin {
   const hn_info* info;
   int sp, mode;
   uint64_t len;
   uint64_t* scan_words;
   uint32_t n_scan_words;
};

__device__ __forceinline__ bool build_go(const hn_info* info, int sp, int mode) {
   if (mode == BUILD_REHASH || mode == BUILD_GROW) return true; // k_rehash_info has just set the Info up for the new table
   const bool sp_ok = info->size_power == sp;
   // a merge's batch is partitioned whether the merge or its fallback runs
   return sp_ok && (mode == BUILD_MERGE || (info->fill == 0 && info->tombstone_counter == 0));
}
__device__ __forceinline__ void build_header(BuildHeader* h, bool go, uint64_t n, uint64_t grow_old = 0,
                                             uint64_t grow_new = 0) {
   h->go = go ? 1u : 0u;
   h->fail = 0;
   h->max_probe = 0;
   h->c0 = 0;
   h->n_distinct = 0;
   h->n_fix = 0;
   h->fb_fail = 0;
   h->fb_len = 0;
   h->fb_new = 0;
   h->grow_old = grow_old;
   h->grow_new = grow_new;
   h->n = n;
}

// A rehash counts the live slots in its first pass, so its header is set up
// before that.
__global__ void k_build_begin(const hn_info* info, BuildHeader* h, int sp, int mode, uint64_t grow_old,
                              uint64_t grow_new) {
   if (threadIdx.x == 0) build_header(h, build_go(info, sp, mode), 0, grow_old, grow_new);
}

// Per-block digit counts, written digit-major: mat[d * nblocks + block].  A
// block covers `sub` consecutive tiles of `tile` pairs, which keeps the
// count matrix -- and its scan -- small.
// DIG: the digits come from the byte array the previous scatter pass wrote
// (one byte per pair, 16 per load) instead of from the pairs' keys.
template <typename K, int SRC, bool FILTER, bool DIG = false>
__global__ __launch_bounds__(kPartBS) void k_part_count(PartIn<K> in, uint64_t n_in, const uint64_t* d_n, uint32_t* mat,
                                                        uint32_t nblocks, uint32_t tile, uint32_t nsub, int sp,
                                                        int rlog, int dshift, int dbits, BuildHeader* h,
                                                        const uint8_t* dig, BuildBegin bg) {
   __shared__ uint32_t hist[1 << kMaxDigitBits];
   __shared__ uint32_t live_s;
   if (blockIdx.x == 0)
      for (uint32_t i = threadIdx.x; i < bg.n_scan_words; i += kPartBS) bg.scan_words[i] = 0;
   if (bg.info) {
      const bool go = build_go(bg.info, bg.sp, bg.mode); // the Info does not change before the build's last kernel
      if (blockIdx.x == 0 && threadIdx.x == 0) build_header(h, go, bg.len);
      if (!go) return;
   } else if (!h->go) {
      return;
   }
   const uint64_t n = d_n ? *d_n : n_in;
   const uint32_t D = 1u << dbits, dmask = D - 1;
   for (uint32_t d = threadIdx.x; d < D; d += kPartBS) hist[d] = 0;
   if (threadIdx.x == 0) live_s = 0;
   __syncthreads();
   const uint64_t super = static_cast<uint64_t>(tile) * nsub;
   const uint64_t t0 = static_cast<uint64_t>(blockIdx.x) * super;
   const uint64_t t1 = std::min<uint64_t>(t0 + super, n);
   uint32_t live = 0;
   if constexpr (DIG) {
      static_assert(!FILTER, "digit bytes follow a pass that kept only live pairs");
      // t0 is a multiple of the block's span, so the 16-byte loads are aligned.
      for (uint64_t e = t0 + 16ull * threadIdx.x; e < t1; e += 16ull * kPartBS) {
         if (e + 16 <= t1) {
            const uint4 w = *reinterpret_cast<const uint4*>(dig + e);
            const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
               for (int b = 0; b < 4; ++b) atomicAdd(&hist[(ws[q] >> (8 * b)) & 0xFFu], 1u);
         } else {
            for (uint64_t x = e; x < t1; ++x) atomicAdd(&hist[dig[x]], 1u);
         }
      }
   } else {
      // Four keys loaded before their four counts: more loads in flight per thread.
      constexpr int U = 4;
      for (uint64_t e0 = t0 + threadIdx.x; e0 < t1; e0 += U * kPartBS) {
         K key[U];
#pragma unroll
         for (int u = 0; u < U; ++u) {
            const uint64_t e = e0 + static_cast<uint64_t>(u) * kPartBS;
            if (e < t1) key[u] = part_key<K, SRC>(in, e);
         }
#pragma unroll
         for (int u = 0; u < U; ++u) {
            const uint64_t e = e0 + static_cast<uint64_t>(u) * kPartBS;
            if (e >= t1 || (FILTER && !part_live<K, SRC>(in, e, key[u]))) continue;
            atomicAdd(&hist[(region_of(key[u], sp, rlog) >> dshift) & dmask], 1u);
            ++live;
         }
      }
   }
   if (FILTER) {
      live = wave_sum(live);
      if (__lane_id() == 0 && live) atomicAdd(&live_s, live);
   }
   __syncthreads();
   for (uint32_t d = threadIdx.x; d < D; d += kPartBS) mat[static_cast<uint64_t>(d) * nblocks + blockIdx.x] = hist[d];
   if (FILTER && threadIdx.x == 0 && live_s) atomic_add_relaxed(&h->n, static_cast<uint64_t>(live_s));
}

// Carry bookkeeping over regions: each region's carry function, the carry
// it was placed with (spec), the true carry, and the regions to place again.
struct RegionLB {
   uint64_t* word;  // [NR] the region's carry function, packed
   int64_t* spec;   // [NR] carry the region was placed with
   int64_t* carry;  // [NR] true carry
   uint32_t* mark;  // [NR] 1: place again
   uint32_t* list;  // [NR] regions to place again (count in the header)
};

// Stable multisplit.  A block walks its `nsub` tiles in order, keeping the
// running output offset of every digit in LDS.  In a tile, wave w ranks the
// pairs [64*ROUNDS*w, 64*ROUNDS*(w+1)) in ROUNDS rounds of 64: lanes with equal
// digits are found with one ballot per digit bit, and the wave's own LDS
// counters carry the earlier rounds (no block barrier per round).  Per-wave
// counts then give each pair's rank among equal digits in tile order; the
// tile is staged in LDS in digit order and leaves in runs.  The per-wave
// counters are 16-bit (a count or an offset within a tile is below 2^16),
// which leaves room in LDS for 16 waves beside an 8,192-pair tile.  `start`
// (nullable): the pass is the only one, its digits are the regions, and block
// 0 does what k_region_starts does otherwise.
template <typename K, int SRC, bool FILTER, int BS, int ROUNDS>
__global__ __launch_bounds__(BS) void k_part_scatter(PartIn<K> in, uint64_t n_in, const uint64_t* d_n,
                                                          Slot<K>* out, const uint32_t* offs, uint32_t nblocks,
                                                          uint32_t nsub, int sp, int rlog, int dshift, int dbits,
                                                          const BuildHeader* h, uint8_t* dig, int ndshift,
                                                          uint32_t nmask, uint64_t* start, RegionLB lb) {
   constexpr int NW = BS / kWave;
   constexpr int TILE = BS * ROUNDS;
   constexpr uint32_t DMAX = 1u << kMaxDigitBits;
   constexpr int DPT = DMAX >= BS ? DMAX / BS : 1; // digits per thread in the digit loops
   static_assert(DPT * BS >= DMAX && TILE < 65536, "digit split; 16-bit counters");
   __shared__ Slot<K> tile_s[TILE];
   __shared__ uint16_t wcnt_s[NW][DMAX];
   __shared__ uint32_t lstart_s[DMAX];
   __shared__ uint32_t goff_s[DMAX];
   __shared__ uint32_t wsum_s[NW];
   if (!h->go) return;
   const uint64_t n = d_n ? *d_n : n_in;
   const uint32_t D = 1u << dbits, dmask = D - 1;
   const int lane = __lane_id(), wave = threadIdx.x / kWave;
   const uint64_t lt = (1ull << lane) - 1ull;
   const uint32_t d0 = threadIdx.x * DPT; // this thread's digits in the digit loops
   for (uint32_t d = d0; d < d0 + DPT && d < D; ++d) {
      const uint32_t o = offs[static_cast<uint64_t>(d) * nblocks + blockIdx.x];
      goff_s[d] = o;
      if (start && blockIdx.x == 0) {
         start[d] = o;
         if (d == D - 1) start[D] = FILTER ? h->n : n;
         lb.mark[d] = 0;
      }
   }
   const uint64_t base = static_cast<uint64_t>(blockIdx.x) * TILE * nsub;
   // The pairs of tile `sub` are loaded while tile sub-1 is written out.
   Slot<K> el[ROUNDS];
   auto load_tile = [&](int sub) {
      const uint64_t w0 = base + static_cast<uint64_t>(sub) * TILE + static_cast<uint64_t>(wave) * (TILE / NW) +
                          static_cast<uint64_t>(lane);
#pragma unroll
      for (int r = 0; r < ROUNDS; ++r) {
         const uint64_t e = w0 + static_cast<uint64_t>(r) * kWave;
         if (e < n) el[r] = part_pair<K, SRC>(in, e);
      }
   };
   load_tile(0);
   for (int sub = 0; sub < static_cast<int>(nsub); ++sub) {
      const uint64_t t0 = base + static_cast<uint64_t>(sub) * TILE;
      if (t0 >= n) break;
      for (uint32_t d = d0; d < d0 + DPT && d < D; ++d) {
#pragma unroll
         for (int w = 0; w < NW; ++w) wcnt_s[w][d] = 0;
      }
      __syncthreads();
      uint32_t dg[ROUNDS], rk[ROUNDS];
      bool ok[ROUNDS];
      const uint64_t w0 = t0 + static_cast<uint64_t>(wave) * (TILE / NW) + lane;
#pragma unroll
      for (int r = 0; r < ROUNDS; ++r) {
         const uint64_t e = w0 + static_cast<uint64_t>(r) * kWave;
         dg[r] = 0;
         ok[r] = false;
         if (e < n) {
            ok[r] = !FILTER || part_live<K, SRC>(in, e, el[r].key);
            dg[r] = (region_of(el[r].key, sp, rlog) >> dshift) & dmask;
         }
      }
      uint16_t* wc = wcnt_s[wave];
#pragma unroll
      for (int r = 0; r < ROUNDS; ++r) {
         const bool valid = ok[r];
         uint64_t m = __ballot(valid);
         for (int b = 0; b < dbits; ++b) {
            const bool bit = (dg[r] >> b) & 1u;
            const uint64_t bal = __ballot(bit);
            m &= bit ? bal : ~bal;
         }
         // All lanes read the counter before its one writer (the group's
         // first lane) updates it; a wave's LDS operations run in order.
         if (valid) rk[r] = wc[dg[r]] + static_cast<uint32_t>(__popcll(m & lt));
         if (valid && first_bit(m) == lane) wc[dg[r]] += static_cast<uint16_t>(__popcll(m));
      }
      __syncthreads();
      // Per digit: waves' counts -> exclusive offsets over waves; tile totals -> exclusive scan.
      uint32_t tot[DPT];
      uint32_t acc = 0;
#pragma unroll
      for (int i = 0; i < DPT; ++i) {
         tot[i] = 0;
         const uint32_t d = d0 + i;
         if (d < D) {
#pragma unroll
            for (int w = 0; w < NW; ++w) {
               const uint32_t c = wcnt_s[w][d];
               wcnt_s[w][d] = static_cast<uint16_t>(tot[i]);
               tot[i] += c;
            }
         }
         acc += tot[i];
      }
      {
         uint32_t inc = acc;
#pragma unroll
         for (int o = 1; o < kWave; o <<= 1) {
            const uint32_t y = __shfl_up(inc, o, kWave);
            if (lane >= o) inc += y;
         }
         if (lane == kWave - 1) wsum_s[wave] = inc;
         __syncthreads();
         uint32_t bse = inc - acc;
         for (int w = 0; w < wave; ++w) bse += wsum_s[w];
#pragma unroll
         for (int i = 0; i < DPT; ++i) {
            if (d0 + i < D) lstart_s[d0 + i] = bse;
            bse += tot[i];
         }
      }
      __syncthreads();
#pragma unroll
      for (int r = 0; r < ROUNDS; ++r) {
         if (ok[r]) {
            const uint32_t p = lstart_s[dg[r]] + wcnt_s[wave][dg[r]] + rk[r];
            tile_s[p] = el[r];
         }
      }
      if (sub + 1 < static_cast<int>(nsub)) load_tile(sub + 1);
      __syncthreads();
      uint32_t cnt = 0; // pairs of this tile that are written: the digit scan's total
      for (int w = 0; w < NW; ++w) cnt += wsum_s[w];
      for (uint32_t p = threadIdx.x; p < cnt; p += BS) {
         const Slot<K> e = tile_s[p];
         const uint32_t rg = region_of(e.key, sp, rlog);
         const uint32_t d = (rg >> dshift) & dmask; // recomputed: cheaper than LDS for it
         const uint64_t pos = static_cast<uint64_t>(goff_s[d]) + (p - lstart_s[d]);
         out[pos] = e;
         if (nmask) dig[pos] = static_cast<uint8_t>((rg >> ndshift) & nmask); // the next pass's digit
      }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < DPT; ++i)
         if (d0 + i < D) goff_s[d0 + i] += tot[i];
   }
}

// Exclusive scan of x[0..m) in LDS by a whole workgroup; returns the total.
template <int BS>
__device__ uint32_t lds_exclusive_scan(uint32_t* x, uint32_t m, uint32_t* wsum) {
   const int lane = __lane_id(), wave = threadIdx.x / kWave;
   const uint32_t per = (m + BS - 1) / BS;
   const uint32_t c0 = std::min<uint32_t>(threadIdx.x * per, m), c1 = std::min<uint32_t>(c0 + per, m);
   uint32_t acc = 0;
   for (uint32_t i = c0; i < c1; ++i) acc += x[i];
   const uint32_t inc = wave_incl_add(acc);
   if (lane == kWave - 1) wsum[wave] = inc;
   __syncthreads();
   uint32_t run = inc - acc, total = 0;
#pragma unroll
   for (int w = 0; w < BS / kWave; ++w) {
      const uint32_t c = wsum[w];
      run += w < wave ? c : 0u;
      total += c;
   }
   for (uint32_t i = c0; i < c1; ++i) {
      const uint32_t v = x[i];
      x[i] = run;
      run += v;
   }
   __syncthreads();
   return total;
}

// Carry functions g(c) = max(a, c + b): `first` applied, then `then`.
constexpr int64_t kNegInf = INT64_MIN / 4; // identity: max(-inf, c + 0) = c
__host__ __device__ __forceinline__ RegionSum compose(RegionSum first, RegionSum then) {
   RegionSum g;
   g.a = first.a + then.b > then.a ? first.a + then.b : then.a;
   g.b = first.b + then.b;
   return g;
}

// A region's carry function in one 64-bit word: a <= keys in the region
// < 2^24; b + R in [0, 2^24).
__device__ __forceinline__ uint64_t pack_sum(RegionSum g, int64_t R) {
   return (static_cast<uint64_t>(g.b + R) << 24) | static_cast<uint64_t>(g.a);
}
__device__ __forceinline__ RegionSum unpack_sum(uint64_t w, int64_t R) {
   RegionSum g;
   g.a = static_cast<int64_t>(w & 0xFFFFFFull);
   g.b = static_cast<int64_t>((w >> 24) & 0xFFFFFFull) - R;
   return g;
}
__device__ __forceinline__ RegionSum load_sum(const RegionLB& lb, uint64_t r, int64_t R) {
   return unpack_sum(lb.word[r], R);
}

// start[r] = first index of region r in the partitioned array (the first
// index whose region is >= r, so an empty region starts where the next one
// does), start[NR] = n: a binary search per region over the sorted array.
// Neighbouring lanes search neighbouring regions and share the upper levels
// of their searches in cache; the array itself is not streamed.  The same
// launch clears the regions' marks; their sums are written by the placing step
// before any kernel reads them.
template <typename K>
__global__ __launch_bounds__(256) void k_region_starts(const Slot<K>* S, uint64_t* start, RegionLB lb, uint64_t NR,
                                                       int sp, int rlog, BuildHeader* h) {
   if (!h->go) return;
   const uint64_t n = h->n;
   const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
   for (uint64_t r = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; r <= NR; r += stride) {
      uint64_t lo = 0, hi = n;
      while (lo < hi) {
         const uint64_t mid = lo + (hi - lo) / 2;
         if (region_of(S[mid].key, sp, rlog) < r) lo = mid + 1;
         else hi = mid;
      }
      start[r] = lo;
      if (r < NR) lb.mark[r] = 0;
   }
}

constexpr int kRegionNW = kRegionBS / kWave;
constexpr uint32_t kRegionMax = 1u << kRegionLog;

// LDS of one region of at most IPT keys per thread: the sort tables are dead
// once each key knows its sorted index, so the placement arrays reuse their
// space.
constexpr uint32_t kStage = kRegionMax + 512; // slots of a region's write span held at a time
template <typename K, int IPT>
struct RegionLds {
   static constexpr uint32_t kCap = kRegionBS * IPT;
   union {
      struct {
         K key[kCap];
         uint16_t order[kCap];
         uint8_t dup[kCap];
      } s;
      Slot<K> out[kStage];
   } u1;
   union {
      struct {
         uint32_t cnt[kRegionMax + 1];  // keys per home offset, then their exclusive starts
         uint32_t scnt[kRegionMax + 1]; // the same over the surviving keys
      } c;
      int32_t v[kCap]; // by sorted index f: home offset - f, then its running max
   } u2;
   static_assert(sizeof(int32_t) * kCap <= 2 * sizeof(uint32_t) * (kRegionMax + 1), "v fits the count tables");
   uint32_t wsum[kRegionNW];
   int32_t wmax[kRegionNW];
   uint32_t r;
   int64_t carry;
};
// Pairs S[lo, lo + m) of a region: thread t owns keys t + k*kRegionBS, kk/vv
// the pairs, uu[k] the key's home offset in the region.  PRE: kk
// and vv hold the pairs (loaded ahead by the caller), S is not read.
template <typename K, bool PRE = false>
__device__ __forceinline__ void region_pairs(const Slot<K>* S, uint64_t lo, uint32_t m, int sp, uint64_t R, K* kk,
                                             K* vv, uint32_t* uu) {
#pragma unroll
   for (int k = 0; k < kRegionIPT; ++k) {
      const uint32_t e = threadIdx.x + k * kRegionBS;
      if (e < m) {
         if (!PRE) {
            const Slot<K> s = S[lo + e];
            kk[k] = s.key;
            vv[k] = s.val;
         }
         uu[k] = static_cast<uint32_t>((fib_home(kk[k], sp) & ((1ull << sp) - 1)) & (R - 1));
      }
   }
}

// has() of region_sort where the first m elements are the keys.
__device__ __forceinline__ auto in_first(uint32_t m) {
   return [m](int k) { return threadIdx.x + k * kRegionBS < m; };
}

// Sort a region's keys in LDS by (home, key), keeping the last occurrence of
// a repeated key.  Thread t owns the keys of input index t + k*kRegionBS for
// which has(k); ff[k] = its sorted index among the survivors, or -1.
// Leaves v[f] = home offset - f.  Returns the number of survivors.  Called by
// the whole workgroup.
//
// A counting sort by home slot puts the keys, with their input indices, in
// home order in LDS; a key's rank among its home's keys is then one pass over
// that home's few entries (0.9 others on average at load factor 0.9), which
// also spots repeated keys.  Without repeats in the region (the block agrees
// with one __syncthreads_or) every key survives and the sorted index is
// home start + rank; otherwise the survivors are counted per home and ranked
// again among survivors.
template <typename K, int IPT, typename F>
__device__ uint32_t region_sort(uint64_t R, RegionLds<K, IPT>& L, F has, const K* kk, const uint32_t* uu, int32_t* ff) {
   __syncthreads(); // the previous user of L is done
   for (uint32_t i = threadIdx.x; i <= R; i += kRegionBS) L.u2.c.cnt[i] = 0;
   __syncthreads();
   uint32_t sub[IPT];
#pragma unroll
   for (int k = 0; k < IPT; ++k) {
      ff[k] = -1;
      if (has(k)) sub[k] = atomicAdd(&L.u2.c.cnt[uu[k]], 1u);
   }
   __syncthreads();
   const uint32_t m = lds_exclusive_scan<kRegionBS>(L.u2.c.cnt, static_cast<uint32_t>(R) + 1, L.wsum);
   // keys and input indices in home order
#pragma unroll
   for (int k = 0; k < IPT; ++k) {
      const uint32_t e = threadIdx.x + k * kRegionBS;
      if (has(k)) {
         const uint32_t pos = L.u2.c.cnt[uu[k]] + sub[k];
         L.u1.s.key[pos] = kk[k];
         L.u1.s.order[pos] = static_cast<uint16_t>(e);
      }
   }
   __syncthreads();
   // Rank among the home's keys, several of a thread's keys side by side: the
   // homes' entries are read one round after another, one wait each (a loop
   // per key waited for each key's entries in turn; absent keys read entry 0).
   // Two where there are eight, most of whose last rows are empty.
   constexpr int SIDE = IPT <= 5 ? IPT : 2;
   uint32_t twice = 0; // bit k: key k's home holds it more than once
#pragma unroll
   for (int b = 0; b < IPT; b += SIDE) {
      uint32_t j0[SIDE], jn[SIDE], eq[SIDE];
#pragma unroll
      for (int i = 0; i < SIDE; ++i) {
         const bool h = b + i < IPT && has(b + i);
         j0[i] = h ? L.u2.c.cnt[uu[b + i]] : 0;
         jn[i] = h ? L.u2.c.cnt[uu[b + i] + 1] - j0[i] : 0;
         eq[i] = 0;
         if (b + i < IPT) ff[b + i] = h ? static_cast<int32_t>(j0[i]) : -1;
      }
      for (uint32_t r = 0;; ++r) {
         bool any = false;
#pragma unroll
         for (int i = 0; i < SIDE; ++i) any = any || r < jn[i];
         if (!__ballot(any)) break;
         K kj[SIDE];
#pragma unroll
         for (int i = 0; i < SIDE; ++i) kj[i] = L.u1.s.key[j0[i] + (r < jn[i] ? r : 0)];
#pragma unroll
         for (int i = 0; i < SIDE; ++i) {
            if (b + i >= IPT) continue;
            ff[b + i] += r < jn[i] && kj[i] < kk[b + i] ? 1 : 0;
            eq[i] += r < jn[i] && kj[i] == kk[b + i] ? 1 : 0;
         }
      }
#pragma unroll
      for (int i = 0; i < SIDE; ++i) twice |= eq[i] > 1 ? 1u << (b + i) : 0u;
   }
   uint32_t ms;
   if (!__syncthreads_or(twice != 0)) {
      ms = m;
   } else {
      uint32_t dupm = 0; // bit k: a later copy of key k drops it
#pragma unroll
      for (int k = 0; k < IPT; ++k) {
         const uint32_t e = threadIdx.x + k * kRegionBS;
         if ((twice >> k) & 1u)
            for (uint32_t j = L.u2.c.cnt[uu[k]]; j < L.u2.c.cnt[uu[k] + 1]; ++j)
               if (L.u1.s.key[j] == kk[k] && L.u1.s.order[j] > e) dupm |= 1u << k;
      }
      for (uint32_t i = threadIdx.x; i <= R; i += kRegionBS) L.u2.c.scnt[i] = 0;
#pragma unroll
      for (int k = 0; k < IPT; ++k) {
         const uint32_t e = threadIdx.x + k * kRegionBS;
         if (has(k)) L.u1.s.dup[e] = (dupm >> k) & 1u;
      }
      __syncthreads();
#pragma unroll
      for (int k = 0; k < IPT; ++k)
         if (ff[k] >= 0 && !((dupm >> k) & 1u)) atomicAdd(&L.u2.c.scnt[uu[k]], 1u);
      __syncthreads();
      ms = lds_exclusive_scan<kRegionBS>(L.u2.c.scnt, static_cast<uint32_t>(R) + 1, L.wsum);
#pragma unroll
      for (int k = 0; k < IPT; ++k) {
         if (ff[k] < 0) continue;
         if ((dupm >> k) & 1u) {
            ff[k] = -1;
            continue;
         }
         int32_t rank = 0;
         for (uint32_t j = L.u2.c.cnt[uu[k]]; j < L.u2.c.cnt[uu[k] + 1]; ++j)
            rank += (!L.u1.s.dup[L.u1.s.order[j]] && L.u1.s.key[j] < kk[k]) ? 1 : 0;
         ff[k] = static_cast<int32_t>(L.u2.c.scnt[uu[k]]) + rank;
      }
   }
   __syncthreads(); // count tables dead from here; v takes their place
#pragma unroll
   for (int k = 0; k < IPT; ++k)
      if (ff[k] >= 0) L.u2.v[ff[k]] = static_cast<int32_t>(uu[k]) - ff[k];
   __syncthreads();
   return ms;
}

template <typename K, int IPT>
__device__ RegionSum region_summary(RegionLds<K, IPT>& L, uint32_t ms, uint64_t R, const int32_t* ff) {
   int32_t M = INT32_MIN;
#pragma unroll
   for (int k = 0; k < IPT; ++k)
      if (ff[k] >= 0) M = std::max(M, L.u2.v[ff[k]]);
   M = wave_max(M);
   if (__lane_id() == 0) L.wmax[threadIdx.x / kWave] = M;
   __syncthreads();
   int32_t Mb = INT32_MIN;
   for (int w = 0; w < kRegionNW; ++w) Mb = std::max(Mb, L.wmax[w]);
   __syncthreads();
   RegionSum g;
   const int64_t mp = static_cast<int64_t>(ms), Ri = static_cast<int64_t>(R);
   g.b = mp - Ri;
   g.a = mp > 0 ? std::max<int64_t>(0, mp - Ri + Mb) : 0;
   return g;
}

// Place a sorted region after carry c: key f at p = f + max(running max of v, c),
// and write the span [c, max(R, last p + 1)) of slots (keys and EMPTY) at
// base + offset.  `keep` picks by unwrapped position: 0 = below N only, 1 =
// all, 2 = N and above only.  Returns this thread's longest probe.
template <typename K, int IPT>
__device__ uint32_t region_place(RegionLds<K, IPT>& L, uint32_t ms, int64_t c, uint64_t base, int sp, uint64_t R,
                                 int keep, const K* kk, const K* vv, const uint32_t* uu, const int32_t* ff,
                                 Slot<K>* b) {
   const int lane = __lane_id(), wave = threadIdx.x / kWave;
   const uint64_t N = 1ull << sp, mask = N - 1;
   {
      const uint32_t per = (ms + kRegionBS - 1) / kRegionBS;
      const uint32_t j0 = std::min<uint32_t>(threadIdx.x * per, ms), j1 = std::min<uint32_t>(j0 + per, ms);
      int32_t acc = INT32_MIN;
      for (uint32_t j = j0; j < j1; ++j) acc = std::max(acc, L.u2.v[j]);
      const int32_t inc = wave_incl_max(acc);
      if (lane == kWave - 1) L.wmax[wave] = inc;
      __syncthreads();
      int32_t run = __shfl_up(inc, 1, kWave);
      if (lane == 0) run = INT32_MIN;
#pragma unroll
      for (int w = 0; w < kRegionNW; ++w) {
         const int32_t c = L.wmax[w];
         run = std::max(run, w < wave ? c : INT32_MIN);
      }
      for (uint32_t j = j0; j < j1; ++j) {
         run = std::max(run, L.u2.v[j]);
         L.u2.v[j] = run;
      }
   }
   __syncthreads();
   const int64_t last = ms ? static_cast<int64_t>(ms - 1) + std::max<int64_t>(L.u2.v[ms - 1], c) : -1;
   const int64_t end = std::max<int64_t>(static_cast<int64_t>(R), last + 1);
   const int64_t span = end - c;
   auto kept = [&](uint64_t pos) { return keep == 1 || (keep == 0 ? pos < N : pos >= N); };
   uint32_t probe = 0;
   // The span leaves in slot order from LDS: stored from the threads that
   // sorted them, a wave's 64 slots went to as many lines.  With the ranks
   // side by side (region_sort) the builds of 2^28 slots at load .9 went from
   // 7.94 to 7.67 ms (u64) and 5.82 to 5.56 (u32), a merge of 2^22 keys into
   // 2^26 u32 slots from 0.93 to 0.83, into u64 slots 1.07 to 1.04.
   for (int64_t s0 = 0; s0 < span; s0 += kStage) {
      const uint32_t m = static_cast<uint32_t>(std::min<int64_t>(span - s0, kStage));
      if (s0) __syncthreads(); // the pass before has been written out
      for (uint32_t q = threadIdx.x; q < m; q += kRegionBS) {
         L.u1.out[q].key = empty_key<K>();
         L.u1.out[q].val = 0;
      }
      __syncthreads();
#pragma unroll
      for (int k = 0; k < IPT; ++k) {
         if (ff[k] >= 0) {
            const int64_t p = ff[k] + std::max<int64_t>(L.u2.v[ff[k]], c);
            const int64_t q = p - c - s0;
            if (q >= 0 && q < m) {
               L.u1.out[q].key = kk[k];
               L.u1.out[q].val = vv[k];
               probe = std::max<uint32_t>(probe, static_cast<uint32_t>(p - static_cast<int64_t>(uu[k]) + 1));
            }
         }
      }
      __syncthreads();
      for (uint32_t q = threadIdx.x; q < m; q += kRegionBS) {
         const uint64_t pos = base + static_cast<uint64_t>(c + s0 + q);
         if (kept(pos)) b[pos & mask] = L.u1.out[q];
      }
   }
   return probe;
}

template <typename K, int IPT>
__device__ void probe_to_header(RegionLds<K, IPT>& L, uint32_t probe, BuildHeader* h) {
   probe = wave_max(probe);
   __syncthreads();
   if (__lane_id() == 0) L.wmax[threadIdx.x / kWave] = static_cast<int32_t>(probe);
   __syncthreads();
   if (threadIdx.x == 0) {
      uint32_t pb = 0;
      for (int w = 0; w < kRegionNW; ++w) pb = std::max(pb, static_cast<uint32_t>(L.wmax[w]));
      if (pb > __hip_atomic_load(&h->max_probe, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
         atomic_max_relaxed(&h->max_probe, pb);
   }
}

// One workgroup walks `chunk` consecutive regions in order: sort a
// region, record its carry function, place it with the carry handed on from
// the region before, and hand on max(a, c + b).  The walk starts from the
// carry out of the region before the chunk taken with no carry in (that
// region is sorted once more for its summary).  Slots at unwrapped positions
// >= N are skipped.  Nothing waits on another workgroup; the carry kernels
// finds the regions whose carry was wrong (a spill crossing a whole region
// into a chunk, or the wrap past the table's end) and k_region_fix places
// them again.  The carries do not depend on the chunk: a shorter one only
// means more walks and more regions sorted twice.
constexpr uint32_t kRegionChunk = 16;

// Regions per walk: kRegionChunk, or fewer when that would leave the device
// short of workgroups (tables below 2^24 slots): a 2^20-slot table has 512
// regions, 32 walks of 16 but 512 of 1.
inline uint32_t region_chunk(uint64_t NR) {
   const uint64_t c = NR / (static_cast<uint64_t>(cu_count()) * 2);
   return static_cast<uint32_t>(c < 1 ? 1 : (c > kRegionChunk ? kRegionChunk : c));
}

// The next region's pairs are loaded while the current one is placed (no
// walk waits on another, so nothing depends on the order of completion);
// held to 128 VGPRs for two workgroups per CU: 8.68 ms against 9.19 ms for
// the 2^28-slot build, 10.2 ms when the extra registers left one per CU.
template <typename K>
__global__ __launch_bounds__(kRegionBS) __attribute__((amdgpu_waves_per_eu(4))) void k_region_build(
    const Slot<K>* S, const uint64_t* start, RegionLB lb, Slot<K>* b, int sp, int rlog, uint64_t NR, uint32_t chunk,
    BuildHeader* h) {
   __shared__ RegionLds<K, kRegionIPT> L;
   if (!h->go) return;
   const uint64_t R = 1ull << rlog;
   const int64_t Ri = static_cast<int64_t>(R);
   const uint64_t r0 = static_cast<uint64_t>(blockIdx.x) * chunk;
   const uint64_t r1 = std::min<uint64_t>(r0 + chunk, NR);
   K kk[kRegionIPT], vv[kRegionIPT];
   K nk[kRegionIPT], nv[kRegionIPT]; // the next region's pairs, loaded while this one is placed
   uint32_t uu[kRegionIPT];
   int32_t ff[kRegionIPT];
   uint32_t probe = 0;
   int64_t c = 0;
   auto prefetch = [&](uint64_t r) {
      const uint64_t lo = start[r], m = start[r + 1] - lo;
#pragma unroll
      for (int k = 0; k < kRegionIPT; ++k) {
         const uint32_t e = threadIdx.x + k * kRegionBS;
         if (e < m && m <= static_cast<uint64_t>(kRegionCap)) {
            const Slot<K> s = S[lo + e];
            nk[k] = s.key;
            nv[k] = s.val;
         }
      }
   };
   if (r0 < r1) prefetch(r0);
   if (r0 > 0) {
      // Seed the walk with the carry out of the region before the chunk, that
      // region taken with no carry in: exact unless a spill crosses it whole.
      const uint64_t lo = start[r0 - 1], m = start[r0] - lo;
      if (m <= static_cast<uint64_t>(kRegionCap)) {
         region_pairs<K>(S, lo, static_cast<uint32_t>(m), sp, R, kk, vv, uu);
         const uint32_t ms = region_sort(R, L, in_first(static_cast<uint32_t>(m)), kk, uu, ff);
         const RegionSum g = region_summary(L, ms, R, ff);
         c = std::max(g.a, g.b);
      }
   }
   for (uint64_t r = r0; r < r1; ++r) {
      const uint64_t lo = start[r], m = start[r + 1] - lo;
      if (m > static_cast<uint64_t>(kRegionCap)) { // abandon the build
         if (threadIdx.x == 0) __hip_atomic_store(&h->fail, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
         return;
      }
#pragma unroll
      for (int k = 0; k < kRegionIPT; ++k) {
         kk[k] = nk[k];
         vv[k] = nv[k];
      }
      region_pairs<K, true>(S, lo, static_cast<uint32_t>(m), sp, R, kk, vv, uu);
      const uint32_t ms = region_sort(R, L, in_first(static_cast<uint32_t>(m)), kk, uu, ff);
      if (r + 1 < r1) prefetch(r + 1);
      probe = std::max(probe, region_place(L, ms, c, r * R, sp, R, 0, kk, vv, uu, ff, b));
      // The region's summary from the prefix max the placement left in v:
      // v[ms - 1] = max over its keys of (home offset - sorted index).
      RegionSum g;
      g.b = static_cast<int64_t>(ms) - Ri;
      g.a = ms > 0 ? std::max<int64_t>(0, static_cast<int64_t>(ms) - Ri + L.u2.v[ms - 1]) : 0;
      if (threadIdx.x == 0) {
         lb.word[r] = pack_sum(g, Ri);
         lb.spec[r] = c;
      }
      c = std::max(g.a, c + g.b);
   }
   probe_to_header(L, probe, h);
}

// True carries.  The carry into region 0 is the least fixed point of the
// whole-table composition max(A, c + B), B = n - N < 0: c0 = A; region r's
// carry is the composition over regions 0..r-1 applied to c0.  Three small
// kernels: per block of kCarryTile regions the composition (k_carry_local),
// the blocks' prefixes and c0 (k_carry_top, one workgroup), each region's
// carry (k_carry_apply); then k_carry_mark lists the regions to place again.
constexpr int kCarryBS = 256;
constexpr int kCarryPer = 4;
constexpr uint64_t kCarryTile = kCarryBS * kCarryPer;

// Block-wide inclusive scan (composition) of one RegionSum per thread, in LDS.
__device__ RegionSum carry_block_scan(RegionSum mine, int64_t* fa, int64_t* fb) {
   fa[threadIdx.x] = mine.a;
   fb[threadIdx.x] = mine.b;
   __syncthreads();
   for (int o = 1; o < static_cast<int>(blockDim.x); o <<= 1) {
      const RegionSum cur{fa[threadIdx.x], fb[threadIdx.x]};
      RegionSum prev{kNegInf, 0};
      if (static_cast<int>(threadIdx.x) >= o) prev = RegionSum{fa[threadIdx.x - o], fb[threadIdx.x - o]};
      __syncthreads();
      if (static_cast<int>(threadIdx.x) >= o) {
         const RegionSum c = compose(prev, cur);
         fa[threadIdx.x] = c.a;
         fb[threadIdx.x] = c.b;
      }
      __syncthreads();
   }
   return RegionSum{fa[threadIdx.x], fb[threadIdx.x]};
}

__global__ __launch_bounds__(kCarryBS) void k_carry_local(RegionLB lb, RegionSum* blk, uint64_t NR, int64_t R,
                                                           const BuildHeader* h) {
   __shared__ int64_t fa[kCarryBS], fb[kCarryBS];
   if (!h->go || h->fail) return;
   const uint64_t r0 = blockIdx.x * kCarryTile + threadIdx.x * kCarryPer;
   RegionSum g{kNegInf, 0};
   for (uint64_t r = r0; r < r0 + kCarryPer && r < NR; ++r) g = compose(g, load_sum(lb, r, R));
   const RegionSum inc = carry_block_scan(g, fa, fb);
   if (threadIdx.x == kCarryBS - 1) blk[blockIdx.x] = inc;
}

// One workgroup: blk[i] becomes the carry into block i (as RegionSum{c, 0}).
__global__ __launch_bounds__(1024) void k_carry_top(RegionSum* blk, uint64_t nblk, uint64_t N, BuildHeader* h) {
   __shared__ int64_t fa[1024], fb[1024];
   if (!h->go || h->fail) return;
   const uint64_t per = (nblk + 1023) / 1024;
   const uint64_t b0 = std::min<uint64_t>(threadIdx.x * per, nblk), b1 = std::min<uint64_t>(b0 + per, nblk);
   RegionSum g{kNegInf, 0};
   for (uint64_t i = b0; i < b1; ++i) g = compose(g, blk[i]);
   const RegionSum inc = carry_block_scan(g, fa, fb);
   const RegionSum T{fa[1023], fb[1023]};
   const int64_t c0 = std::max<int64_t>(T.a, 0);
   RegionSum P{kNegInf, 0}; // composition over the blocks before b0
   if (threadIdx.x > 0) P = RegionSum{fa[threadIdx.x - 1], fb[threadIdx.x - 1]};
   (void)inc;
   __syncthreads();
   int64_t c = std::max(P.a, c0 + P.b);
   for (uint64_t i = b0; i < b1; ++i) {
      const RegionSum gi = blk[i];
      blk[i] = RegionSum{c, 0};
      c = std::max(gi.a, c + gi.b);
   }
   if (threadIdx.x == 0) {
      h->c0 = c0;
      h->n_distinct = static_cast<uint64_t>(T.b + static_cast<int64_t>(N));
      if (T.b >= 0) h->fail = 1; // a merge's union would fill the table: there is no carry to place it with
   }
}

__global__ __launch_bounds__(kCarryBS) void k_carry_apply(RegionLB lb, const RegionSum* blk, uint64_t NR, int64_t R,
                                                           const BuildHeader* h) {
   __shared__ int64_t fa[kCarryBS], fb[kCarryBS];
   if (!h->go || h->fail) return;
   const uint64_t r0 = blockIdx.x * kCarryTile + threadIdx.x * kCarryPer;
   RegionSum gs[kCarryPer];
   RegionSum g{kNegInf, 0};
#pragma unroll
   for (int k = 0; k < kCarryPer; ++k) {
      gs[k] = r0 + k < NR ? load_sum(lb, r0 + k, R) : RegionSum{kNegInf, 0};
      g = compose(g, gs[k]);
   }
   carry_block_scan(g, fa, fb);
   RegionSum P{kNegInf, 0};
   if (threadIdx.x > 0) P = RegionSum{fa[threadIdx.x - 1], fb[threadIdx.x - 1]};
   const int64_t cin = blk[blockIdx.x].a;
   int64_t c = std::max(P.a, cin + P.b);
#pragma unroll
   for (int k = 0; k < kCarryPer; ++k) {
      if (r0 + k < NR) {
         lb.carry[r0 + k] = c;
         c = std::max(gs[k].a, c + gs[k].b);
      }
   }
}

// Placed again: every region whose spec carry differs, the regions whose
// true slot ranges cover the slots such a region wrote wrongly
// ([rR + spec, rR + carry)), and the regions whose range reaches past N
// (those slots were skipped).  Regions r0, r0 + stride, ...
__device__ __forceinline__ void carry_mark(const RegionLB& lb, uint64_t NR, int64_t R, int64_t N, int64_t c0,
                                           BuildHeader* h, uint64_t r0, uint64_t stride) {
   auto start_of = [&](uint64_t r) { return static_cast<int64_t>(r) * R + lb.carry[r]; };
   auto mark = [&](uint64_t r) {
      if (atomicExch(&lb.mark[r], 1u) == 0) lb.list[atomicAdd(&h->n_fix, 1u)] = static_cast<uint32_t>(r);
   };
   for (uint64_t r = r0; r < NR; r += stride) {
      const int64_t cr = lb.carry[r], sr = lb.spec[r];
      const int64_t next = r + 1 < NR ? start_of(r + 1) : N + c0; // end of r's true range
      if (next > N) mark(r);                                      // reaches past N
      if (cr != sr) {
         mark(r);
         const int64_t lo = static_cast<int64_t>(r) * R + sr;
         for (int64_t q = static_cast<int64_t>(r) - 1; q >= 0; --q) {
            mark(static_cast<uint64_t>(q));
            if (start_of(static_cast<uint64_t>(q)) <= lo) break;
         }
      }
   }
}

__global__ __launch_bounds__(256) void k_carry_mark(RegionLB lb, uint64_t NR, int64_t R, int64_t N, BuildHeader* h) {
   if (!h->go || h->fail) return;
   carry_mark(lb, NR, R, N, h->c0, h, static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x,
              static_cast<uint64_t>(gridDim.x) * blockDim.x);
}

// The four carry kernels as one launch of one workgroup, for tables of at
// most kCarrySmall regions (2^23 slots): there each of the four was mostly
// its launch (2^20 u32 slots: 4.0 + 4.7 + 2.6 + 2.5 us).
constexpr uint64_t kCarrySmall = 4096;
__global__ __launch_bounds__(1024) void k_carry_small(RegionLB lb, uint64_t NR, int64_t R, uint64_t N, BuildHeader* h) {
   __shared__ int64_t fa[1024], fb[1024];
   if (!h->go || h->fail) return;
   constexpr int PER = static_cast<int>(kCarrySmall / 1024);
   const uint64_t r0 = static_cast<uint64_t>(threadIdx.x) * PER;
   RegionSum gs[PER];
   RegionSum g{kNegInf, 0};
#pragma unroll
   for (int k = 0; k < PER; ++k) {
      gs[k] = r0 + k < NR ? load_sum(lb, r0 + k, R) : RegionSum{kNegInf, 0};
      g = compose(g, gs[k]);
   }
   carry_block_scan(g, fa, fb);
   const RegionSum T{fa[1023], fb[1023]};
   const int64_t c0 = std::max<int64_t>(T.a, 0);
   RegionSum P{kNegInf, 0};
   if (threadIdx.x > 0) P = RegionSum{fa[threadIdx.x - 1], fb[threadIdx.x - 1]};
   int64_t c = std::max(P.a, c0 + P.b);
#pragma unroll
   for (int k = 0; k < PER; ++k) {
      if (r0 + k < NR) {
         lb.carry[r0 + k] = c;
         c = std::max(gs[k].a, c + gs[k].b);
      }
   }
   if (threadIdx.x == 0) {
      h->c0 = c0;
      h->n_distinct = static_cast<uint64_t>(T.b + static_cast<int64_t>(N));
      if (T.b >= 0) h->fail = 1; // as in k_carry_top
   }
   if (T.b >= 0) return;
   __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
   __syncthreads();
   __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
   carry_mark(lb, NR, R, static_cast<int64_t>(N), c0, h, threadIdx.x, 1024);
}

// A region over capacity abandons the placement: the table is emptied and
// the probing insert takes the partitioned pairs (all of them, in S); a
// rehash with a batch inserts the old table and then the batch, whose values
// win.
template <typename K>
__device__ void build_fallback_prep(Slot<K>* b, uint64_t N, hn_info* info, BuildHeader* h) {
   if (blockIdx.x == 0 && threadIdx.x == 0) {
      h->fb_len = h->grow_old ? h->grow_old : h->n;
      h->fb_new = h->grow_new;
      info->fill = 0;
      info->current_max_bucket_overflow = kBucketOverflow;
   }
   const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
   for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < N; i += stride) {
      Slot<K> s;
      s.key = empty_key<K>();
      s.val = 0;
      b[i] = s;
   }
}

// Place the listed regions again with their true carries, all slots of
// their ranges (wrapping past N); or, when the placement was abandoned, empty
// the table for the probing insert.
template <typename K>
__global__ __launch_bounds__(kRegionBS) void k_region_fix(const Slot<K>* S, const uint64_t* start, RegionLB lb,
                                                         Slot<K>* b, int sp, int rlog, hn_info* info, BuildHeader* h) {
   __shared__ RegionLds<K, kRegionIPT> L;
   if (!h->go) return;
   if (h->fail) {
      build_fallback_prep<K>(b, 1ull << sp, info, h);
      return;
   }
   const uint64_t R = 1ull << rlog;
   K kk[kRegionIPT], vv[kRegionIPT];
   uint32_t uu[kRegionIPT];
   int32_t ff[kRegionIPT];
   uint32_t probe = 0;
   const uint32_t nfix = h->n_fix;
   for (uint32_t i = blockIdx.x; i < nfix; i += gridDim.x) {
      const uint32_t r = lb.list[i];
      const uint64_t lo = start[r];
      const uint32_t m = static_cast<uint32_t>(start[r + 1] - lo);
      region_pairs<K>(S, lo, m, sp, R, kk, vv, uu);
      const uint32_t ms = region_sort(R, L, in_first(m), kk, uu, ff);
      probe = std::max(probe, region_place(L, ms, lb.carry[r], static_cast<uint64_t>(r) * R, sp, R, 1, kk, vv,
                                              uu, ff, b));
   }
   probe_to_header(L, probe, h);
}

// Finish the Info.  Not run (go = 0): an empty-table build reports
// err = INVALID with the table untouched (so does a merge whose size power is
// not the table's).  Placed: fill, overflow of the layout, ordered.
// Fallback: the insert has set fill and overflow; a merge's keeps the old
// table's TOMBSTONEs.
__global__ void k_build_end(hn_info* info, const BuildHeader* h, int mode) {
   if (threadIdx.x != 0) return;
   if (!h->go) {
      info->err = HN_STATUS_INVALID; // (a rehash always goes)
      return;
   }
   info->reserved0 = 0;
   if (!(mode == BUILD_MERGE && h->fail)) info->tombstone_counter = 0;
   if (h->fail) {
      info->err = h->fb_fail ? HN_STATUS_FAIL : HN_STATUS_SUCCESS;
      info->reserved1 = 0;
   } else {
      info->fill = h->n_distinct;
      info->current_max_bucket_overflow =
          std::max<uint64_t>(kBucketOverflow, next_overflow(h->max_probe, kBucketOverflow));
      info->err = HN_STATUS_SUCCESS;
      info->reserved1 = kInfoOrdered;
   }
   // device_rehash reports success iff the new table holds the old fill (hashinator.h:333)
   if (mode == BUILD_REHASH && info->err == HN_STATUS_SUCCESS && info->fill != h->prior_fill)
      info->err = HN_STATUS_FAIL;
}

// Rehash: remember the old fill and give the Info the new table's size
// (Info(newSizePower), hashinator.h:328).  The build writes every slot of the
// new table, so it needs no initialisation.
__global__ void k_rehash_info(hn_info* info, int new_sp, BuildHeader* h) {
   if (threadIdx.x != 0) return;
   h->prior_fill = info->fill;
   info->size_power = new_sp;
   info->reserved0 = 0;
   info->fill = 0;
   info->current_max_bucket_overflow = kBucketOverflow;
   info->tombstone_counter = 0;
   info->err = HN_STATUS_SUCCESS;
   info->reserved1 = 0;
}

// A pass's digits come from the byte array when the pass before it wrote
// them: a pass after the first whose digit fits a byte.
inline bool digits_in_bytes(const BuildPlan& P, int pass) { return pass > 0 && pass < P.passes && P.dbits[pass] <= 8; }

// The exclusive scan of hn_compact.hip over look-back words that an earlier
// kernel has cleared, and those words.
uint64_t* scan_words_u32(void* scr, uint64_t n, uint32_t* count);
int scan_u32_cleared(uint32_t* x, uint64_t n, void* scr, size_t bytes, hipStream_t s);

template <typename K, int SRC, bool FILTER>
int launch_part(const BuildPlan& P, int pass, PartIn<K> in, uint64_t n_in, const uint64_t* d_n, Slot<K>* out,
                uint32_t* mat, void* scan_scratch, size_t scan_bytes, BuildHeader* h, uint8_t* dig, BuildBegin bg,
                uint64_t* start, RegionLB lb, hipStream_t s) {
   int dshift = 0;
   for (int i = 0; i < pass; ++i) dshift += P.dbits[i];
   const int dbits = P.dbits[pass];
   const uint64_t D = 1ull << dbits;
   const int ndshift = dshift + dbits;
   const uint32_t nmask = digits_in_bytes(P, pass + 1) ? (1u << P.dbits[pass + 1]) - 1u : 0u;
   bg.scan_words = scan_words_u32(scan_scratch, D * P.nblocks, &bg.n_scan_words);
   auto count = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(P.nblocks), dim3(kPartBS), 0, s, in, n_in, d_n, mat, P.nblocks, P.tile, P.sub,
                         P.sp, P.rlog, dshift, dbits, h, dig, bg);
   };
   if constexpr (SRC == SRC_TABLE && !FILTER) {
      if (digits_in_bytes(P, pass))
         count(k_part_count<K, SRC, FILTER, true>);
      else
         count(k_part_count<K, SRC, FILTER>);
   } else {
      count(k_part_count<K, SRC, FILTER>);
   }
   int rc = scan_u32_cleared(mat, D * P.nblocks, scan_scratch, scan_bytes, s);
   if (rc) return rc;
   static_assert(kPartBSL * kPartRoundsL == kPartTileL && kPartBSS * kPartRoundsS == kPartTileS, "scatter tiles");
   auto scatter = [&](auto kernel, int bs) {
      hipLaunchKernelGGL(kernel, dim3(P.nblocks), dim3(bs), 0, s, in, n_in, d_n, out, mat, P.nblocks, P.sub, P.sp,
                         P.rlog, dshift, dbits, h, dig, ndshift, nmask, P.passes == 1 ? start : nullptr, lb);
   };
   if (P.tile == kPartTileL)
      scatter(k_part_scatter<K, SRC, FILTER, kPartBSL, kPartRoundsL>, kPartBSL);
   else
      scatter(k_part_scatter<K, SRC, FILTER, kPartBSS, kPartRoundsS>, kPartBSS);
   return static_cast<int>(hipGetLastError());
}

// Defined with the insert kernels (hn_map.hip): the probing insert of
// pairs[0, *d_len), failures OR-ed into *fail_sink, Info left to the caller.
template <typename K>
int launch_insert_pairs_dlen(const Slot<K>* pairs, Slot<K>* buckets, hn_info* info, uint64_t max_len,
                             const uint64_t* d_len, int32_t* fail_sink, hipStream_t s);
// The same from a table's slots, and from a batch in any of its forms.
template <typename K>
int launch_insert_table_dlen(const Slot<K>* table, Slot<K>* buckets, hn_info* info, uint64_t max_len,
                             const uint64_t* d_len, int32_t* fail_sink, hipStream_t s);
template <typename K>
int launch_insert_batch_dlen(const K* keys, const K* vals, const Slot<K>* pairs, Slot<K>* buckets, hn_info* info,
                             uint64_t max_len, const uint64_t* d_len, int32_t* fail_sink, hipStream_t s);

inline RegionLB region_lb(const BuildPlan& P, char* base) {
   RegionLB lb;
   lb.word = reinterpret_cast<uint64_t*>(base + P.off_word);
   lb.spec = reinterpret_cast<int64_t*>(base + P.off_spec);
   lb.carry = reinterpret_cast<int64_t*>(base + P.off_carry);
   lb.mark = reinterpret_cast<uint32_t*>(base + P.off_mark);
   lb.list = reinterpret_cast<uint32_t*>(base + P.off_list);
   return lb;
}

// The partition passes and the region starts: the input pairs end in S,
// stably partitioned by region, with start[r] the first of region r.  src0
// picks the first pass's input kind; n_in is its element count (the old
// table's slot count for a rehash, whose first pass keeps live slots only).
// Pass i writes S when (passes - 1 - i) is even, `alt` (memory of the same
// size that is written later anyway: the output table) otherwise, so the
// last pass lands in S.
template <typename K>
int partition_regions(const BuildPlan& P, int mode, const hn_info* info, int src0, PartIn<K> in0, uint64_t n_in,
                      Slot<K>* alt, void* scratch, hipStream_t s) {
   char* base = static_cast<char*>(scratch);
   BuildHeader* h = reinterpret_cast<BuildHeader*>(base);
   Slot<K>* S = reinterpret_cast<Slot<K>*>(base + P.off_pairs);
   uint32_t* mat = reinterpret_cast<uint32_t*>(base + P.off_mat);
   void* scan_scratch = base + P.off_scan;
   const size_t scan_bytes = P.off_start - P.off_scan;
   uint64_t* start = reinterpret_cast<uint64_t*>(base + P.off_start);
   uint8_t* dig = reinterpret_cast<uint8_t*>(base + P.off_dig);
   const RegionLB lb = region_lb(P, base);
   BuildBegin bg{};
   if (mode == BUILD_REHASH || mode == BUILD_GROW)
      hipLaunchKernelGGL(k_build_begin, dim3(1), dim3(64), 0, s, info, h, P.sp, mode, in0.n_table,
                         mode == BUILD_GROW ? n_in - in0.n_table : 0);
   else
      bg = BuildBegin{info, P.sp, mode, P.n, nullptr, 0};
   const Slot<K>* src = nullptr;
   for (int pass = 0; pass < P.passes; ++pass) {
      Slot<K>* dst = ((P.passes - 1 - pass) % 2 == 0) ? S : alt;
      int rc;
      if (pass == 0) {
         switch (src0) {
         case SRC_PAIRS:
            rc = launch_part<K, SRC_PAIRS, false>(P, 0, in0, n_in, nullptr, dst, mat, scan_scratch, scan_bytes, h, dig, bg,
                                                  start, lb, s);
            break;
         case SRC_SOA:
            rc = launch_part<K, SRC_SOA, false>(P, 0, in0, n_in, nullptr, dst, mat, scan_scratch, scan_bytes, h, dig, bg,
                                                  start, lb, s);
            break;
         case SRC_INDEX:
            rc = launch_part<K, SRC_INDEX, false>(P, 0, in0, n_in, nullptr, dst, mat, scan_scratch, scan_bytes, h, dig, bg,
                                                  start, lb, s);
            break;
         case SRC_GROW:
            rc = launch_part<K, SRC_GROW, true>(P, 0, in0, n_in, nullptr, dst, mat, scan_scratch, scan_bytes, h, dig, bg,
                                                start, lb, s);
            break;
         default:
            rc = launch_part<K, SRC_TABLE, true>(P, 0, in0, n_in, nullptr, dst, mat, scan_scratch, scan_bytes, h, dig, bg,
                                                 start, lb, s);
            break;
         }
      } else {
         PartIn<K> in{nullptr, nullptr, src, nullptr, 0};
         rc = launch_part<K, SRC_TABLE, false>(P, pass, in, 0, &h->n, dst, mat, scan_scratch, scan_bytes, h, dig,
                                               BuildBegin{}, start, lb, s);
      }
      if (rc) return rc;
      src = dst;
   }
   if (P.passes > 1)
      hipLaunchKernelGGL(k_region_starts<K>, dim3(stream_blocks(P.NR + 1, 256)), dim3(256), 0, s, S, start, lb, P.NR,
                         P.sp, P.rlog, h);
   return static_cast<int>(hipGetLastError());
}

// True carries, and the regions to place again.
inline void launch_carry(const BuildPlan& P, RegionLB lb, char* base, BuildHeader* h, hipStream_t s) {
   RegionSum* blk = reinterpret_cast<RegionSum*>(base + P.off_blk);
   const uint64_t nblk = (P.NR + kCarryTile - 1) / kCarryTile;
   const int64_t Ri = static_cast<int64_t>(P.R), Ni = static_cast<int64_t>(P.N);
   if (P.NR <= kCarrySmall) {
      hipLaunchKernelGGL(k_carry_small, dim3(1), dim3(1024), 0, s, lb, P.NR, Ri, P.N, h);
   } else {
      hipLaunchKernelGGL(k_carry_local, dim3(static_cast<uint32_t>(nblk)), dim3(kCarryBS), 0, s, lb, blk, P.NR, Ri, h);
      hipLaunchKernelGGL(k_carry_top, dim3(1), dim3(1024), 0, s, blk, nblk, P.N, h);
      hipLaunchKernelGGL(k_carry_apply, dim3(static_cast<uint32_t>(nblk)), dim3(kCarryBS), 0, s, lb, blk, P.NR, Ri, h);
      hipLaunchKernelGGL(k_carry_mark, dim3(stream_blocks(P.NR, 256)), dim3(256), 0, s, lb, P.NR, Ri, Ni, h);
   }
}

// Everything after the first partition pass's input is chosen (see
// partition_regions for src0 and n_in).
template <typename K>
int build_core(const BuildPlan& P, int mode, int src0, PartIn<K> in0, uint64_t n_in, void* buckets, hn_info* info,
               void* scratch, hipStream_t s) {
   char* base = static_cast<char*>(scratch);
   BuildHeader* h = reinterpret_cast<BuildHeader*>(base);
   Slot<K>* S = reinterpret_cast<Slot<K>*>(base + P.off_pairs);
   uint64_t* start = reinterpret_cast<uint64_t*>(base + P.off_start);
   const RegionLB lb = region_lb(P, base);
   Slot<K>* T = static_cast<Slot<K>*>(buckets);

   int rc = partition_regions<K>(P, mode, info, src0, in0, n_in, T, scratch, s);
   if (rc) return rc;
   const uint32_t chunk = region_chunk(P.NR);
   hipLaunchKernelGGL(k_region_build<K>, dim3(static_cast<uint32_t>((P.NR + chunk - 1) / chunk)), dim3(kRegionBS), 0,
                      s, S, start, lb, T, P.sp, P.rlog, P.NR, chunk, h);
   launch_carry(P, lb, base, h, s);
   const uint32_t gfix = static_cast<uint32_t>(std::min<uint64_t>(P.NR, static_cast<uint64_t>(cu_count()) * 2));
   hipLaunchKernelGGL(k_region_fix<K>, dim3(gfix), dim3(kRegionBS), 0, s, S, start, lb, T, P.sp, P.rlog, info, h);
   if (mode == BUILD_GROW) {
      rc = launch_insert_table_dlen<K>(in0.table, T, info, in0.n_table, &h->fb_len, &h->fb_fail, s);
      if (!rc)
         rc = launch_insert_batch_dlen<K>(in0.keys, in0.vals, in0.pairs, T, info, n_in - in0.n_table, &h->fb_new,
                                          &h->fb_fail, s);
   } else {
      rc = launch_insert_pairs_dlen<K>(S, T, info, P.n, &h->fb_len, &h->fb_fail, s);
   }
   if (rc) return rc;
   hipLaunchKernelGGL(k_build_end, dim3(1), dim3(64), 0, s, info, h, mode);
   return static_cast<int>(hipGetLastError());
}

template <typename K>
int build(const void* keys, const void* vals, const void* pairs, void* buckets, hn_info* info, size_t len, int sp,
          void* scratch, size_t bytes, hipStream_t s, const hn_tune* t) {
   if (!buckets || !info) return HN_EINVAL;
   if (len == 0) return 0;
   if (!keys && !pairs) return HN_EINVAL;
   const int dcap = (t && t->reserved) ? t->reserved : kMaxDigitBits;
   BuildPlan P;
   if (!build_plan<K>(sp, len, dcap, &P)) return HN_EINVAL;
   if (!scratch || bytes < P.total) return HN_ESCRATCH;
   if (!scratch_aligned(scratch)) return HN_EINVAL;
   PartIn<K> in{static_cast<const K*>(keys), static_cast<const K*>(vals), static_cast<const Slot<K>*>(pairs), nullptr, 0};
   const int src0 = pairs ? SRC_PAIRS : (vals ? SRC_SOA : SRC_INDEX);
   return build_core<K>(P, BUILD_EMPTY, src0, in, len, buckets, info, scratch, s);
}

template <typename K>
size_t build_scratch_bytes(int sp, size_t len) {
   BuildPlan P;
   return build_plan<K>(sp, len, kMaxDigitBits, &P) ? P.total : 0;
}

// device_rehash into a larger table as a build: the first partition pass
// reads the old table's live slots (extractPattern + insert in the reference,
// hashinator.h:284-336, without the intermediate array).  The new table is
// Robin Hood ordered.  Growing only: the live pairs then fill at most half of
// the new table.
template <typename K>
bool rehash_plan(int old_sp, int new_sp, BuildPlan* P) {
   if (old_sp < 1 || new_sp <= old_sp || new_sp > std::min(max_size_power<K>(), 32)) return false;
   return build_plan<K>(new_sp, 1ull << old_sp, kMaxDigitBits, P);
}

template <typename K>
size_t rehash_build_scratch_bytes(int old_sp, int new_sp) {
   BuildPlan P;
   return rehash_plan<K>(old_sp, new_sp, &P) ? P.total : 0;
}

template <typename K>
int rehash_build(const void* old_b, int old_sp, void* new_b, int new_sp, hn_info* info, void* scratch, size_t bytes,
                 hipStream_t s) {
   if (!old_b || !new_b || !info) return HN_EINVAL;
   BuildPlan P;
   if (!rehash_plan<K>(old_sp, new_sp, &P)) return HN_EINVAL;
   const char* o0 = static_cast<const char*>(old_b);
   const char* n0 = static_cast<const char*>(new_b);
   if (o0 < n0 + P.N * sizeof(Slot<K>) && n0 < o0 + (1ull << old_sp) * sizeof(Slot<K>)) return HN_EINVAL;
   if (!scratch || bytes < P.total) return HN_ESCRATCH;
   if (!scratch_aligned(scratch)) return HN_EINVAL;
   hipLaunchKernelGGL(k_rehash_info, dim3(1), dim3(64), 0, s, info, new_sp, static_cast<BuildHeader*>(scratch));
   PartIn<K> in{nullptr, nullptr, static_cast<const Slot<K>*>(old_b), nullptr, 0};
   return build_core<K>(P, BUILD_REHASH, SRC_TABLE, in, 1ull << old_sp, new_b, info, scratch, s);
}

// An insert that grows the table (hashinator.h:1329-1335: resize, then
// insert) as one build: the first partition pass reads the old table's live
// slots and then the batch, so the sort's last copy of a key is the newest.
// A rehash, the probing insert and the reorder go through the new table twice
// more: 3 million u64 keys to 3 million of 2^23 slots 0.73 ms, here 0.43; 1.1
// million 0.59 and 0.39; 60,000 to 60,000 of 2^17 0.098 and 0.074.
template <typename K>
bool grow_plan(int old_sp, int new_sp, uint64_t len, BuildPlan* P) {
   if (old_sp < 1 || new_sp <= old_sp || new_sp > std::min(max_size_power<K>(), 32)) return false;
   if (len == 0 || len >= 1ull << new_sp) return false;
   return build_plan<K>(new_sp, (1ull << old_sp) + len, kMaxDigitBits, P);
}

template <typename K>
size_t grow_scratch_bytes(int old_sp, int new_sp, size_t len) {
   BuildPlan P;
   return grow_plan<K>(old_sp, new_sp, len, &P) ? P.total : 0;
}

template <typename K>
int grow(const void* keys, const void* vals, const void* pairs, const void* old_b, int old_sp, void* new_b, int new_sp,
         hn_info* info, size_t len, void* scratch, size_t bytes, hipStream_t s) {
   if (!old_b || !new_b || !info || (!keys && !pairs)) return HN_EINVAL;
   BuildPlan P;
   if (!grow_plan<K>(old_sp, new_sp, len, &P)) return HN_EINVAL;
   const char* o0 = static_cast<const char*>(old_b);
   const char* n0 = static_cast<const char*>(new_b);
   if (o0 < n0 + P.N * sizeof(Slot<K>) && n0 < o0 + (1ull << old_sp) * sizeof(Slot<K>)) return HN_EINVAL;
   if (!scratch || bytes < P.total) return HN_ESCRATCH;
   if (!scratch_aligned(scratch)) return HN_EINVAL;
   const uint64_t nt = 1ull << old_sp;
   hipLaunchKernelGGL(k_rehash_info, dim3(1), dim3(64), 0, s, info, new_sp, static_cast<BuildHeader*>(scratch));
   PartIn<K> in{static_cast<const K*>(keys), static_cast<const K*>(vals), static_cast<const Slot<K>*>(pairs),
                static_cast<const Slot<K>*>(old_b), nt};
   return build_core<K>(P, BUILD_GROW, SRC_GROW, in, nt + len, new_b, info, scratch, s);
}

// ------------------------------------------------------------------ merge insert
//
// Hasher::insert (hashers.h:55-70, kernels_AMD.h insert_kernel) into a table
// that already holds keys, followed by the reorder: the image as a function
// of the live set, written into a second bucket array of the same size.  The
// old table must be free of TOMBSTONEs and in Robin Hood order; then its live
// keys stand in slot order sorted by (home, key), unwrapped from an EMPTY
// slot, and the keys whose home lies in region r fill one run of slots
// [s_r, s_{r+1}): s_r is the first slot at or after rR that is EMPTY or holds
// a key whose home is at or after rR (k_merge_bounds).  The new pairs take
// the build's partition passes.  Then the build's walk over regions, its
// carries and its second placement, with a region's keys taken from both: the
// old run first, the new pairs in batch order behind it, so that the last
// copy of a key, which the sort keeps, is the newest (an insert of a present
// key overwrites its value, a key repeated in the batch keeps its last
// value).  When the table has TOMBSTONEs or no order flag, a region exceeds
// its capacity (2,560 old slots or 1,536 new pairs), the old table is not in
// order after all (a key outside its region's run), or the union would fill
// the table, the output is made the other way, on the device: the old table
// copied, then the probing insert of the partitioned batch (the partition
// keeps the batch order of equal keys), so the output is hn_insert_*'s result
// and the order flag is cleared.
//
// 2,560 old slots per 2,048-slot region: a region's run is its 2,048 slots
// plus the difference of the spills across its two ends (tens of slots at
// load factor 0.9).
constexpr uint32_t kMergeCapO = 2560, kMergeCapN = 1536;
constexpr uint32_t kAbsent = 0xFFFFFFFFu;
constexpr int kMergeIPT = static_cast<int>((kMergeCapO + kMergeCapN) / kRegionBS);

// sb[r] = s_r (unwrapped, < rR + kMergeCapO), sb[NR] = N + s_0.  One wave per
// region.
template <typename K>
__global__ __launch_bounds__(256) void k_merge_bounds(const Slot<K>* ob, const hn_info* info, int sp, int rlog,
                                                      uint64_t NR, uint64_t* sb, BuildHeader* h) {
   if (!h->go) return;
   if (info->tombstone_counter != 0 || !(info->reserved1 & kInfoOrdered)) {
      if (blockIdx.x == 0 && threadIdx.x == 0) h->fail = 1;
      return;
   }
   const int lane = __lane_id();
   const uint64_t N = 1ull << sp, mask = N - 1;
   const uint64_t waves = static_cast<uint64_t>(gridDim.x) * (blockDim.x / kWave);
   for (uint64_t r = static_cast<uint64_t>(blockIdx.x) * (blockDim.x / kWave) + threadIdx.x / kWave; r < NR;
        r += waves) {
      const int64_t lo = static_cast<int64_t>(r << rlog);
      int64_t found = -1;
      for (uint32_t o = 0; o < kMergeCapO; o += kWave) {
         const int64_t p = lo + o + lane;
         const K k = ob[static_cast<uint64_t>(p) & mask].key;
         bool stop = k == empty_key<K>();
         if (!stop) {
            const int64_t d = static_cast<int64_t>((static_cast<uint64_t>(p) - fib_home(k, sp)) & mask);
            stop = p - d >= lo;
         }
         const uint64_t m = __ballot(stop);
         if (m) {
            found = lo + o + first_bit(m);
            break;
         }
      }
      if (lane == 0) {
         if (found < 0) {
            __hip_atomic_store(&h->fail, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            found = lo;
         }
         sb[r] = static_cast<uint64_t>(found);
         if (r == 0) sb[NR] = N + static_cast<uint64_t>(found);
      }
   }
}

// A region's two inputs: Lo old slots from o0 (EMPTY ones among them), then
// Ln new pairs from n0.  Element e < Lo + Ln.
template <typename K>
struct MergeRegion {
   uint64_t o0, n0;
   uint32_t Lo, m; // m = Lo + Ln; both 0 when the region is over capacity
   bool fits;
   __device__ MergeRegion(const uint64_t* sb, const uint64_t* start, uint64_t r) : o0(sb[r]), n0(start[r]) {
      const uint64_t lo = sb[r + 1] - o0, ln = start[r + 1] - n0;
      fits = lo <= kMergeCapO && ln <= kMergeCapN;
      Lo = fits ? static_cast<uint32_t>(lo) : 0;
      m = fits ? static_cast<uint32_t>(lo + ln) : 0;
   }
   // Thread t owns elements t + k * kRegionBS: f(k, element).  Three bases that
   // are the same for every lane and a 32-bit index (one address per element
   // and lane took the u64 kernel over its registers).
   template <typename F>
   __device__ __forceinline__ void each(const Slot<K>* ob, const Slot<K>* S, uint64_t mask, F f) const {
      const uint64_t first = o0 & mask;
      const uint32_t turn = static_cast<uint32_t>(std::min<uint64_t>(mask + 1 - first, Lo)); // old slots before the wrap
      const Slot<K>* const p0 = ob + first;
      const Slot<K>* const p1 = ob - turn;
      const Slot<K>* const p2 = S + n0 - Lo;
#pragma unroll
      for (int k = 0; k < kMergeIPT; ++k) {
         const uint32_t e = threadIdx.x + k * kRegionBS;
         if (e < turn)
            f(k, p0[e]);
         else if (e < Lo)
            f(k, p1[e]);
         else if (e < m)
            f(k, p2[e]);
      }
   }
   __device__ __forceinline__ void keys(const Slot<K>* ob, const Slot<K>* S, uint64_t mask, K* kk) const {
      each(ob, S, mask, [&](int k, const Slot<K>& s) { kk[k] = s.key; });
   }
   __device__ __forceinline__ void vals(const Slot<K>* ob, const Slot<K>* S, uint64_t mask, K* vv) const {
      each(ob, S, mask, [&](int k, const Slot<K>& s) { vv[k] = s.val; });
   }
   // Home offsets of the loaded keys, EMPTY ones (a padded batch's too) left
   // out; false in a thread whose old key does not belong to the region.
   __device__ __forceinline__ bool homes(const K* kk, uint64_t rb, int sp, uint64_t R, uint32_t* uu) const {
      const uint64_t mask = (1ull << sp) - 1;
      bool ok = true;
#pragma unroll
      for (int k = 0; k < kMergeIPT; ++k) {
         const uint32_t e = threadIdx.x + k * kRegionBS;
         uu[k] = kAbsent;
         if (e < m && kk[k] != empty_key<K>()) {
            const uint64_t hr = (fib_home(kk[k], sp) - rb) & mask;
            if (hr >= R || (e < Lo && kk[k] == tomb_key<K>()))
               ok = false;
            else
               uu[k] = static_cast<uint32_t>(hr);
         }
      }
      return ok;
   }
};

// k_region_build over both inputs.  Only the next region's keys are held in
// registers ahead (with the values the u64 kernel spilled 88 VGPRs); the values
// come from L2, where the keys' lines already are.  A workgroup per region in
// ticket order, each waiting for its carry by a look-back over the regions in
// flight, took 20.7 us a region where the walk takes 11: 2^24 keys into 2^26
// u64 slots up to load .9 the whole merge 1.71 -> 1.36 ms, 2^22 up to load .5
// 1.31 -> 0.96, u32 1.42 -> 1.12 and 1.13 -> 0.84.
template <typename K>
__global__ __launch_bounds__(kRegionBS) __attribute__((amdgpu_waves_per_eu(4))) void k_merge_build(
    const Slot<K>* ob, const uint64_t* sb, const Slot<K>* S, const uint64_t* start, RegionLB lb, Slot<K>* b, int sp,
    int rlog, uint64_t NR, uint32_t chunk, BuildHeader* h) {
   __shared__ RegionLds<K, kMergeIPT> L;
   if (__syncthreads_or(!h->go || h->fail)) return; // a workgroup may see another's failure: all its threads do
   const uint64_t R = 1ull << rlog, mask = (1ull << sp) - 1;
   const int64_t Ri = static_cast<int64_t>(R);
   const uint64_t r0 = static_cast<uint64_t>(blockIdx.x) * chunk;
   const uint64_t r1 = std::min<uint64_t>(r0 + chunk, NR);
   K kk[kMergeIPT], vv[kMergeIPT];
   K nk[kMergeIPT]; // the next region's keys, loaded while this one is placed; the values then come from L2
   uint32_t uu[kMergeIPT];
   int32_t ff[kMergeIPT];
   uint32_t probe = 0;
   int64_t c = 0;
   if (r0 < r1) MergeRegion<K>(sb, start, r0).keys(ob, S, mask, nk);
   if (r0 > 0) { // the carry out of the region before, as in k_region_build
      const MergeRegion<K> g(sb, start, r0 - 1);
      if (g.fits) {
         g.keys(ob, S, mask, kk);
         g.homes(kk, (r0 - 1) << rlog, sp, R, uu); // its own walk reports a key out of place
         const uint32_t ms = region_sort(R, L, [&](int k) { return uu[k] != kAbsent; }, kk, uu, ff);
         const RegionSum gs = region_summary(L, ms, R, ff);
         c = std::max(gs.a, gs.b);
      }
   }
   for (uint64_t r = r0; r < r1; ++r) {
      const MergeRegion<K> g(sb, start, r);
#pragma unroll
      for (int k = 0; k < kMergeIPT; ++k) kk[k] = nk[k];
      g.vals(ob, S, mask, vv);
      if (__syncthreads_or(!g.fits || !g.homes(kk, r << rlog, sp, R, uu))) { // abandon the merge
         if (threadIdx.x == 0) __hip_atomic_store(&h->fail, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
         return;
      }
      const uint32_t ms = region_sort(R, L, [&](int k) { return uu[k] != kAbsent; }, kk, uu, ff);
      if (r + 1 < r1) MergeRegion<K>(sb, start, r + 1).keys(ob, S, mask, nk);
      probe = std::max(probe, region_place(L, ms, c, r * R, sp, R, 0, kk, vv, uu, ff, b));
      RegionSum gs;
      gs.b = static_cast<int64_t>(ms) - Ri;
      gs.a = ms > 0 ? std::max<int64_t>(0, static_cast<int64_t>(ms) - Ri + L.u2.v[ms - 1]) : 0;
      if (threadIdx.x == 0) {
         lb.word[r] = pack_sum(gs, Ri);
         lb.spec[r] = c;
      }
      c = std::max(gs.a, c + gs.b);
   }
   probe_to_header(L, probe, h);
}

// The listed regions again with their true carries; or, where the merge does
// not stand, the old table copied for the probing insert of the batch.
template <typename K>
__global__ __launch_bounds__(kRegionBS) void k_merge_fix(const Slot<K>* ob, const uint64_t* sb, const Slot<K>* S,
                                                         const uint64_t* start, RegionLB lb, Slot<K>* b, int sp,
                                                         int rlog, BuildHeader* h) {
   __shared__ RegionLds<K, kMergeIPT> L;
   if (!h->go) return;
   const uint64_t R = 1ull << rlog, N = 1ull << sp;
   if (h->fail) {
      if (blockIdx.x == 0 && threadIdx.x == 0) h->fb_len = h->n;
      const uint64_t stride = static_cast<uint64_t>(gridDim.x) * kRegionBS;
      for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * kRegionBS + threadIdx.x; i < N; i += stride) b[i] = ob[i];
      return;
   }
   K kk[kMergeIPT], vv[kMergeIPT];
   uint32_t uu[kMergeIPT];
   int32_t ff[kMergeIPT];
   uint32_t probe = 0;
   const uint32_t nfix = h->n_fix;
   for (uint32_t i = blockIdx.x; i < nfix; i += gridDim.x) {
      const uint64_t r = lb.list[i];
      const MergeRegion<K> g(sb, start, r);
      g.keys(ob, S, N - 1, kk);
      g.vals(ob, S, N - 1, vv);
      g.homes(kk, r << rlog, sp, R, uu);
      const uint32_t ms = region_sort(R, L, [&](int k) { return uu[k] != kAbsent; }, kk, uu, ff);
      probe = std::max(probe, region_place(L, ms, lb.carry[r], r * R, sp, R, 1, kk, vv, uu, ff, b));
   }
   probe_to_header(L, probe, h);
}

struct MergePlan {
   BuildPlan P;
   size_t off_sb, total;
};

template <typename K>
bool merge_plan(int sp, uint64_t len, MergePlan* M) {
   if (sp < 1 || sp > 30 || len == 0) return false;
   if (!build_plan<K>(sp, len, kMaxDigitBits, &M->P)) return false;
   M->off_sb = align256(M->P.total);
   M->total = align256(M->off_sb + (M->P.NR + 1) * sizeof(uint64_t));
   return true;
}

template <typename K>
size_t merge_scratch_bytes(int sp, size_t len) {
   MergePlan M;
   return merge_plan<K>(sp, len, &M) ? M.total : 0;
}

template <typename K>
int merge(const void* keys, const void* vals, const void* pairs, const void* old_b, void* new_b, hn_info* info,
          size_t len, int sp, void* scratch, size_t bytes, hipStream_t s) {
   if (!old_b || !new_b || !info) return HN_EINVAL;
   if (len > 0 && !keys && !pairs) return HN_EINVAL;
   if (sp < 1 || sp > 30) return HN_EINVAL;
   const uint64_t N = 1ull << sp;
   const char* o0 = static_cast<const char*>(old_b);
   const char* n0 = static_cast<const char*>(new_b);
   if (o0 < n0 + N * sizeof(Slot<K>) && n0 < o0 + N * sizeof(Slot<K>)) return HN_EINVAL;
   if (len == 0) // nothing to merge: the output is the table
      return static_cast<int>(hipMemcpyAsync(new_b, old_b, N * sizeof(Slot<K>), hipMemcpyDeviceToDevice, s));
   MergePlan M;
   if (!merge_plan<K>(sp, len, &M)) return HN_EINVAL;
   if (!scratch || bytes < M.total) return HN_ESCRATCH;
   if (!scratch_aligned(scratch)) return HN_EINVAL;
   const BuildPlan& P = M.P;
   char* base = static_cast<char*>(scratch);
   BuildHeader* h = reinterpret_cast<BuildHeader*>(base);
   const Slot<K>* S = reinterpret_cast<const Slot<K>*>(base + P.off_pairs);
   const uint64_t* start = reinterpret_cast<const uint64_t*>(base + P.off_start);
   uint64_t* sb = reinterpret_cast<uint64_t*>(base + M.off_sb);
   const RegionLB lb = region_lb(P, base);
   const Slot<K>* ob = static_cast<const Slot<K>*>(old_b);
   Slot<K>* nb = static_cast<Slot<K>*>(new_b);

   PartIn<K> in{static_cast<const K*>(keys), static_cast<const K*>(vals), static_cast<const Slot<K>*>(pairs), nullptr, 0};
   const int src0 = pairs ? SRC_PAIRS : (vals ? SRC_SOA : SRC_INDEX);
   int rc = partition_regions<K>(P, BUILD_MERGE, info, src0, in, len, nb, scratch, s);
   if (rc) return rc;
   hipLaunchKernelGGL(k_merge_bounds<K>, dim3(static_cast<uint32_t>(std::min<uint64_t>((P.NR + 3) / 4, 65536))),
                      dim3(256), 0, s, ob, info, sp, P.rlog, P.NR, sb, h);
   const uint32_t chunk = region_chunk(P.NR);
   hipLaunchKernelGGL(k_merge_build<K>, dim3(static_cast<uint32_t>((P.NR + chunk - 1) / chunk)), dim3(kRegionBS), 0, s,
                      ob, sb, S, start, lb, nb, sp, P.rlog, P.NR, chunk, h);
   launch_carry(P, lb, base, h, s);
   const uint32_t gfix = static_cast<uint32_t>(std::min<uint64_t>(P.NR, static_cast<uint64_t>(cu_count()) * 2));
   hipLaunchKernelGGL(k_merge_fix<K>, dim3(gfix), dim3(kRegionBS), 0, s, ob, sb, S, start, lb, nb, sp, P.rlog, h);
   rc = launch_insert_pairs_dlen<K>(S, nb, info, len, &h->fb_len, &h->fb_fail, s);
   if (rc) return rc;
   hipLaunchKernelGGL(k_build_end, dim3(1), dim3(64), 0, s, info, h, BUILD_MERGE);
   return static_cast<int>(hipGetLastError());
}

} // namespace hn

using namespace hn;
extern "C" {
size_t hn_rehash_build_scratch_bytes_u32(int old_sp, int new_sp) {
   return rehash_build_scratch_bytes<uint32_t>(old_sp, new_sp);
}
size_t hn_rehash_build_scratch_bytes_u64(int old_sp, int new_sp) {
   return rehash_build_scratch_bytes<uint64_t>(old_sp, new_sp);
}
int hn_rehash_build_u32(const void* ob, int osp, void* nb, int nsp, hn_info* i, void* sc, size_t bytes, hn_stream_t s) {
   return rehash_build<uint32_t>(ob, osp, nb, nsp, i, sc, bytes, s);
}
int hn_rehash_build_u64(const void* ob, int osp, void* nb, int nsp, hn_info* i, void* sc, size_t bytes, hn_stream_t s) {
   return rehash_build<uint64_t>(ob, osp, nb, nsp, i, sc, bytes, s);
}
size_t hn_build_scratch_bytes_u32(int sp, size_t len) { return build_scratch_bytes<uint32_t>(sp, len); }
size_t hn_build_scratch_bytes_u64(int sp, size_t len) { return build_scratch_bytes<uint64_t>(sp, len); }
int hn_build_u32(const void* k, const void* v, void* b, hn_info* i, size_t n, int sp, void* sc, size_t sb,
                 hn_stream_t s, const hn_tune* t) {
   return build<uint32_t>(k, v, nullptr, b, i, n, sp, sc, sb, s, t);
}
int hn_build_u64(const void* k, const void* v, void* b, hn_info* i, size_t n, int sp, void* sc, size_t sb,
                 hn_stream_t s, const hn_tune* t) {
   return build<uint64_t>(k, v, nullptr, b, i, n, sp, sc, sb, s, t);
}
int hn_build_pairs_u32(const void* p, void* b, hn_info* i, size_t n, int sp, void* sc, size_t sb, hn_stream_t s,
                       const hn_tune* t) {
   return build<uint32_t>(nullptr, nullptr, p, b, i, n, sp, sc, sb, s, t);
}
int hn_build_pairs_u64(const void* p, void* b, hn_info* i, size_t n, int sp, void* sc, size_t sb, hn_stream_t s,
                       const hn_tune* t) {
   return build<uint64_t>(nullptr, nullptr, p, b, i, n, sp, sc, sb, s, t);
}
size_t hn_grow_scratch_bytes_u32(int osp, int nsp, size_t len) { return grow_scratch_bytes<uint32_t>(osp, nsp, len); }
size_t hn_grow_scratch_bytes_u64(int osp, int nsp, size_t len) { return grow_scratch_bytes<uint64_t>(osp, nsp, len); }
int hn_grow_u32(const void* k, const void* v, const void* ob, int osp, void* nb, int nsp, hn_info* i, size_t n,
                void* sc, size_t sb, hn_stream_t s) {
   return grow<uint32_t>(k, v, nullptr, ob, osp, nb, nsp, i, n, sc, sb, s);
}
int hn_grow_u64(const void* k, const void* v, const void* ob, int osp, void* nb, int nsp, hn_info* i, size_t n,
                void* sc, size_t sb, hn_stream_t s) {
   return grow<uint64_t>(k, v, nullptr, ob, osp, nb, nsp, i, n, sc, sb, s);
}
int hn_grow_pairs_u32(const void* p, const void* ob, int osp, void* nb, int nsp, hn_info* i, size_t n, void* sc,
                      size_t sb, hn_stream_t s) {
   return grow<uint32_t>(nullptr, nullptr, p, ob, osp, nb, nsp, i, n, sc, sb, s);
}
int hn_grow_pairs_u64(const void* p, const void* ob, int osp, void* nb, int nsp, hn_info* i, size_t n, void* sc,
                      size_t sb, hn_stream_t s) {
   return grow<uint64_t>(nullptr, nullptr, p, ob, osp, nb, nsp, i, n, sc, sb, s);
}
size_t hn_merge_scratch_bytes_u32(int sp, size_t len) { return merge_scratch_bytes<uint32_t>(sp, len); }
size_t hn_merge_scratch_bytes_u64(int sp, size_t len) { return merge_scratch_bytes<uint64_t>(sp, len); }
int hn_merge_u32(const void* k, const void* v, const void* ob, void* nb, hn_info* i, size_t n, int sp, void* sc,
                 size_t sb, hn_stream_t s) {
   return merge<uint32_t>(k, v, nullptr, ob, nb, i, n, sp, sc, sb, s);
}
int hn_merge_u64(const void* k, const void* v, const void* ob, void* nb, hn_info* i, size_t n, int sp, void* sc,
                 size_t sb, hn_stream_t s) {
   return merge<uint64_t>(k, v, nullptr, ob, nb, i, n, sp, sc, sb, s);
}
int hn_merge_pairs_u32(const void* p, const void* ob, void* nb, hn_info* i, size_t n, int sp, void* sc, size_t sb,
                       hn_stream_t s) {
   return merge<uint32_t>(nullptr, nullptr, p, ob, nb, i, n, sp, sc, sb, s);
}
int hn_merge_pairs_u64(const void* p, const void* ob, void* nb, hn_info* i, size_t n, int sp, void* sc, size_t sb,
                       hn_stream_t s) {
   return merge<uint64_t>(nullptr, nullptr, p, ob, nb, i, n, sp, sc, sb, s);
}
} // extern "C"
