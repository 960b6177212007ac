// hn_map.hip -- gfx950 kernels and C-ABI for the hash-map operations.
//
// The probe loops themselves (probe groups, aligned windows, block I/O) are
// in hn_probe.hpp; this file holds the single-map kernels around them, the
// full-table passes (clear, clean_tombstones, rehash) and the C-ABI.
//
// Reference: kstppd/hashinator include/hashinator/kernels_AMD.h (insert_kernel
// 272-405, insert_index_kernel 507-641, delete_kernel 412-505, retrieve_kernel
// 647-752, reset_all_to_empty 26-43, reset_to_empty 65-134) and the host
// wrappers in hashers.h / hashinator.h cited at each entry point.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstring>

#include "hn_device.hpp"
#include "hn_host.hpp"
#include "hn_probe.hpp"
#include "hn_region.hpp"

namespace hn {

// The segment pass of clean_tombstones (hn_clean.hip) and the reorder that
// follows the region path when the segment pass hands a table to it
// (hn_reorder.hip).
size_t seg_clean_fixed_bytes(int sp);
template <typename K>
size_t seg_clean_default_pool(int sp);
template <typename K>
size_t seg_clean_full_pool(int sp);
size_t seg_clean_min_pool();
const uint32_t* seg_clean_gate(const void* scratch);
template <typename K>
int seg_clean(void* buckets, hn_info* info, int sp, void* scratch, void* pool, size_t pool_bytes, bool region_ok,
              hipStream_t s);
size_t reorder_scratch_bytes(int sp);
template <typename K>
int reorder_gated(void* buckets, hn_info* info, int sp, void* scratch, size_t bytes, const uint32_t* gate,
                  hipStream_t s);

// Entries that a group takes at a time: one while there is a group for every
// entry (a group resolves its entries one after another, so the others would
// only wait: 8,000 u64 keys into 2^18 slots, a quarter of the groups at work,
// 21.2 us, all of them 15.4; 10^3 into 2^14 at load .9 147 and 90).
template <int G>
__device__ __forceinline__ uint32_t entries_per_group(uint64_t len, uint64_t groups) {
   const uint64_t per = (len + groups - 1) / groups;
   return per < 1 ? 1 : per < G ? static_cast<uint32_t>(per) : G;
}

// insert_kernel / insert_index_kernel (kernels_AMD.h:136-405, 507-641)
template <typename K, int G, int SRC>
__global__ __launch_bounds__(1024) void k_insert(InsertArgs<K> a) {
   const int sp = a.info->size_power;
   const bool sp_ok = sp >= 1 && sp <= max_size_power<K>();
   if (a.d_len && *a.d_len == 0) return; // a build's fallback that is not needed
   const uint64_t len = !sp_ok ? 0 : (a.d_len ? *a.d_len : a.len);
   const uint64_t gstride = static_cast<uint64_t>(gridDim.x) * (blockDim.x / G);
   const uint64_t blk = (static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x) / G;
   InsertCounters c;
   c.failed = sp_ok ? 0 : 1;
   if (sp_ok) insert_range<K, G, SRC>(a, sp, len, blk, gstride, c, entries_per_group<G>(len, gstride));
   insert_fold_block(a.info, a.fail_sink ? a.fail_sink : &a.info->reserved1, c.placed, c.max_probe, c.failed);
}

// A workgroup that ran a whole insert: err and the reserved words, as
// k_insert_finish leaves them.  Thread 0 wrote the fold's atomics itself.
__device__ __forceinline__ void insert_publish(hn_info* info) {
   if (threadIdx.x != 0) return;
   const int32_t f = __hip_atomic_load(&info->reserved1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & kInfoFail;
   info->err = f ? HN_STATUS_FAIL : HN_STATUS_SUCCESS;
   info->reserved0 = 0;
   info->reserved1 = 0;
}

// An insert of at most kSmallInsert keys.  Into a table of one region (64 KiB
// of slots, known on the device only), workgroup 0 runs it with the table in
// LDS where the probe chains are long enough to pay for the table's way in
// (lds_insert_pays); otherwise as k_insert.  Up to kSoloInsert keys take one
// workgroup, which finishes the Info too: a launch less (200 keys into 2^18
// slots 19.1 -> 13.0 us; more keys want more CUs, whose address translations
// run side by side: 10^3 keys on one workgroup took 21 us, on eight 14).
constexpr uint64_t kSmallInsert = 8192, kSoloInsert = 256;
// Direct and LDS, us a call, from a 64th of the slots on.  Tables of up to 16
// KiB always (2^10 u32 slots: 64 keys at load .1 8.5 and 8.8, at .6 13.1 and
// 10.4, 896 into an empty one 46 and 35).  Larger ones by the load over and
// after the insert where one workgroup runs it (64 keys into 2^12 u64 slots
// empty 7.4 and 10.8, at load .6 15.1 and 14.9, at .85 44 and 38).  Several
// workgroups must agree whatever the fill is when each starts, so by the sizes
// alone: from a quarter of the slots on, into tables of 32 KiB (512 into 2^12
// u32 slots empty 11.0 and 14.1, at load .6 24 and 24, 1,024 at .7 99 and 77)
// and of 64 KiB in 64 bits (2^12: 1,024 into an empty one 13 and 16, at .7 110
// and 93); not in 32 (2^13: 2,048 into an empty one 13 and 19, at .6 46 and 44,
// 6,200 into an empty one 29 and 36, at .1 48 and 55, at .2 163 and 150).
template <typename K>
__device__ __forceinline__ bool lds_insert_pays(const hn_info* info, int sp, uint64_t len, int solo) {
   constexpr int kLog = kRegionLogB<K>;
   const uint64_t R = 1ull << sp;
   if (sp > kLog || len * 64 < R) return false;
   if (sp <= kLog - 2) return true;
   if (!solo) return len * 4 >= R && (sp < kLog || sizeof(K) == 8);
   const uint64_t used = info->fill + info->tombstone_counter;
   return (2 * used + len) * 8 >= R * 9 || (used + len) * 4 >= R * 3;
}
template <typename K, int G, int SRC>
__global__ __launch_bounds__(kRgBS) void k_insert_small(InsertArgs<K> a, int solo) {
   __shared__ RegionMem<K> L;
   const int sp = a.info->size_power;
   const bool sp_ok = sp >= 1 && sp <= max_size_power<K>();
   if (!(sp_ok && lds_insert_pays<K>(a.info, sp, a.len, solo))) {
      InsertCounters c;
      c.failed = sp_ok ? 0 : 1;
      const uint64_t gstride = static_cast<uint64_t>(gridDim.x) * (blockDim.x / G);
      if (sp_ok)
         insert_range<K, G, SRC>(a, sp, a.len, (static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x) / G,
                                 gstride, c, entries_per_group<G>(a.len, gstride));
      insert_fold_block(a.info, &a.info->reserved1, c.placed, c.max_probe, c.failed);
      if (solo) insert_publish(a.info);
      return;
   }
   if (blockIdx.x > 0) return;
   const uint32_t R = 1u << sp, W = R < kRgWin ? R : kRgWin;
   for (uint32_t i = threadIdx.x; i < R; i += blockDim.x) {
      const Slot<K> s = a.buckets[i];
      L.key[i] = s.key;
      L.val[i] = s.val;
   }
   for (uint32_t i = threadIdx.x; i < (R + 31) / 32; i += blockDim.x) L.from[i] = 0;
   __syncthreads();
   InsertCounters c;
   auto step = [&](K key, uint32_t idx, uint32_t& pos, uint32_t& off) -> bool {
      uint32_t at;
      const InsertStep r = lds_insert_step<K>(L, R, W, key, idx, pos, off, &at);
      if (r == STEP_PLACED) {
         ++c.placed;
         const uint64_t pr = off + (at - pos) + 1;
         c.max_probe = pr > c.max_probe ? pr : c.max_probe;
      }
      if (r != STEP_NEXT) return r != STEP_AGAIN;
      if (pos == R) pos = 0;
      if (off >= R) c.failed = 1;
      return off >= R;
   };
   auto take = [](uint32_t, K, uint32_t) { return true; };
   auto home = [](uint32_t h) { return h; };
   const uint32_t len = static_cast<uint32_t>(a.len);
   if constexpr (SRC == SRC_PAIRS)
      lds_probe<K>(L, SlotKeys<K>{a.pairs, len}, sp, take, home, step);
   else
      lds_probe<K>(L, KeyList<K>(a.keys, len), sp, take, home, step);
   insert_fold_block(a.info, &a.info->reserved1, c.placed, c.max_probe, c.failed); // and every key is placed
   if (solo) insert_publish(a.info);
   for (uint32_t i = threadIdx.x; i < R; i += blockDim.x) {
      if (!((L.from[i >> 5] >> (i & 31)) & 1u)) continue; // as it was
      const uint32_t q = static_cast<uint32_t>(L.val[i]);
      Slot<K> s;
      s.key = L.key[i];
      s.val = SRC == SRC_PAIRS ? a.pairs[q].val : SRC == SRC_SOA ? a.vals[q] : static_cast<K>(q);
      a.buckets[i] = s;
   }
}

// After an insert kernel: err = FAIL if a key found no slot (or the fill is
// not the expected one), else SUCCESS; reserved words cleared (an insert does
// not keep Robin Hood order).
__global__ void k_insert_finish(hn_info* info, const uint64_t* expected_fill) {
   int32_t f = info->reserved1 & kInfoFail;
   if (expected_fill && info->fill != *expected_fill) f = 1;
   info->err = f ? HN_STATUS_FAIL : HN_STATUS_SUCCESS;
   info->reserved0 = 0;
   info->reserved1 = 0;
}

// The Info and, of kLookKeys keys at equal distances in a batch, how many the
// table does not hold: what the choice between a merge and a probing insert
// needs, in one read-back with the Info.  Eight lanes a key, whose windows
// start at its home slot; a chain of a few loads, so one workgroup.
constexpr uint32_t kLookKeys = 128;
template <typename K>
__global__ __launch_bounds__(kLookKeys * 8) void k_insert_look(const char* keys, uint64_t stride, uint64_t len,
                                                               const Slot<K>* b, const hn_info* info,
                                                               hn_insert_look* out) {
   __shared__ uint32_t absent_s;
   if (threadIdx.x == 0) absent_s = 0;
   __syncthreads();
   const hn_info i = *info;
   const int sp = i.size_power;
   const bool run = sp >= 1 && sp <= max_size_power<K>() && (i.reserved1 & kInfoOrdered) && i.tombstone_counter == 0;
   const uint32_t m = len < kLookKeys ? static_cast<uint32_t>(len) : kLookKeys;
   const uint32_t g = threadIdx.x / 8, gl = threadIdx.x & 7u;
   const int gbase = __lane_id() & ~7;
   const uint32_t mask = slot_mask32(sp);
   const uint64_t nsl = static_cast<uint64_t>(mask) + 1;
   const uint64_t bound = i.current_max_bucket_overflow < nsl ? i.current_max_bucket_overflow : nsl;
   const bool mine = run && g < m;
   K key = 0;
   uint32_t home = 0;
   if (mine) {
      key = *reinterpret_cast<const K*>(keys + g * (len / m) * stride);
      home = home_slot(key, sp);
   }
   bool active = mine, found = false;
   for (uint64_t off = 0; __ballot(active); off += 8) {
      const uint64_t p = off + gl;
      const uint32_t slot = (home + static_cast<uint32_t>(p)) & mask;
      K k = empty_key<K>();
      if (active && p < bound) k = b[slot].key;
      const bool stop = k == empty_key<K>() || ((slot - home_slot(k, sp)) & mask) < p; // Robin Hood order
      const uint32_t hit = group_bits32<8>(__ballot(active && k == key), gbase);
      const uint32_t end = group_bits32<8>(__ballot(stop), gbase);
      if (active && (hit | end)) {
         found = hit && (!end || __ffs(hit) < __ffs(end));
         active = false;
      }
   }
   if (mine && gl == 0 && !found) atomicAdd(&absent_s, 1u);
   __syncthreads();
   if (threadIdx.x == 0) {
      out->info = i;
      out->sampled = run ? m : 0;
      out->absent = absent_s;
   }
}

// A size power that no table has: nothing is found, and a caller that left its
// values to the kernel gets its zeros all the same.
template <typename K, bool PAIRS, int MODE>
__device__ __forceinline__ void zero_vals(const LookupArgs<K>& a) {
   if constexpr (MODE == LK_RETRIEVE && !PAIRS) {
      if (!a.zero) return;
      const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
      for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < a.len; i += stride)
         a.vals[i] = 0;
   }
}

// retrieve_kernel (kernels_AMD.h:647-752), delete_kernel (412-505), reset_to_empty (65-134)
template <typename K, int G, bool PAIRS, int MODE>
__global__ __launch_bounds__(1024) void k_lookup(LookupArgs<K> a) {
   const int sp = a.info->size_power;
   const bool sp_ok = sp >= 1 && sp <= max_size_power<K>();
   const uint64_t gstride = static_cast<uint64_t>(gridDim.x) * (blockDim.x / G);
   const uint64_t blk = (static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x) / G;
   uint64_t erased = 0;
   if (sp_ok)
      erased = lookup_range<K, G, PAIRS, MODE>(a, sp, a.info->current_max_bucket_overflow, a.len, blk, gstride,
                                               (a.info->reserved1 & kInfoOrdered) != 0);
   else
      zero_vals<K, PAIRS, MODE>(a);
   if constexpr (MODE == LK_ERASE) {
      erased = wave_sum(erased);
      if (__lane_id() == 0 && erased) {
         atomic_add_relaxed(&a.info->tombstone_counter, erased);
         __hip_atomic_fetch_sub(&a.info->fill, erased, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
   }
   if constexpr (MODE == LK_RESET) {
      if (blockIdx.x == 0 && threadIdx.x == 0)
         __hip_atomic_fetch_sub(&a.info->fill, a.len, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
   }
}

// Lane-window lookups (one key per lane, see lane_lookup): each wave with its
// own LDS and its own contiguous share of the queries.  Tables smaller than
// one 128-byte window (and a zero probe bound) take the group loop with one
// lane per key.  One wave per block, four for an erase, which adds its count
// to the Info once per block (two atomics, some 16 ns each one after another:
// 2^24 u64 erases in 2^26 slots 0.89 -> 0.85 ms).
constexpr int lane_block(int mode) { return mode == LK_ERASE ? 256 : kWave; }
template <typename K, bool PAIRS, int MODE>
__global__ __launch_bounds__(lane_block(MODE)) void k_lookup_lane(LookupArgs<K> a, uint32_t cus) {
   constexpr int kWaves = lane_block(MODE) / kWave;
   __shared__ LaneLds<K, MODE> L[kWaves];
   const int sp = a.info->size_power;
   const bool sp_ok = sp >= 1 && sp <= max_size_power<K>();
   const uint64_t ovf = a.info->current_max_bucket_overflow;
   const bool ordered = (a.info->reserved1 & kInfoOrdered) != 0;
   uint64_t erased = 0;
   if (sp_ok) {
      if (sp >= LaneWin<K>::kLog && ovf > 0) {
         const int wv = threadIdx.x / kWave;
         // Waves on a CU, where the grid is the automatic one: 16 for a table in
         // the L2s, 8 for one in the last-level cache, 12 beyond, where more only
         // queue for the memory.  At load .9, 8 million queries and up to as many
         // erases, 8 / 12 / 16 waves, us: 16 MiB u64 queries 219 / - / 208, u32
         // 187 / - / 168; 32 MiB 240 / - / 249, u32 196 / - / 199; 64 MiB 262 / 270
         // / 270, erases 66 / 73 / 76, u32 queries 206 / 214 / 215, erases 100 / 101
         // / 105; 256 MiB 279 / 290 / 288, erases 217 / 214 / 211, u32 220 / 228 /
         // 231, erases 363 / 374 / 373; 1 GiB 337 / 316 / 313, erases 475 each, u32
         // of 512 MiB 233 / 224 / 227, erases 369 / 387 / 388.  The size is known on
         // the device only: the waves over that number end at once.
         const uint64_t bytes = sizeof(Slot<K>) << sp;
         const uint64_t per_cu = bytes <= 1ull << 25 ? 16 : bytes <= 1ull << 28 ? 8 : 12;
         uint64_t nwaves = static_cast<uint64_t>(gridDim.x) * kWaves;
         if (cus) nwaves = std::min<uint64_t>(nwaves, cus * per_cu);
         const uint64_t w = static_cast<uint64_t>(blockIdx.x) * kWaves + wv;
         const uint64_t per = a.len / nwaves, rem = a.len % nwaves;
         const uint64_t q0 = w * per + (w < rem ? w : rem);
         const uint64_t q1 = q0 + per + (w < rem ? 1 : 0);
         if (w < nwaves) erased = lane_lookup<K, PAIRS, MODE>(a, sp, ovf, ordered, q0, q1, L[wv]);
      } else {
         const uint64_t gstride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
         const uint64_t blk = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
         erased = lookup_range<K, 1, PAIRS, MODE>(a, sp, ovf, a.len, blk, gstride, ordered);
      }
   } else {
      zero_vals<K, PAIRS, MODE>(a);
   }
   if constexpr (MODE == LK_ERASE) {
      __shared__ unsigned long long erased_s;
      if (threadIdx.x == 0) erased_s = 0;
      __syncthreads();
      erased = wave_sum(erased);
      if (__lane_id() == 0 && erased) atomicAdd(&erased_s, static_cast<unsigned long long>(erased));
      __syncthreads();
      if (threadIdx.x == 0 && erased_s) {
         const uint64_t e = erased_s;
         atomic_add_relaxed(&a.info->tombstone_counter, e);
         __hip_atomic_fetch_sub(&a.info->fill, e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
   }
}

// reset_all_to_empty (kernels_AMD.h:26-43): keys -> EMPTY, values untouched.
template <typename K>
__global__ __launch_bounds__(256) void k_reset_all(Slot<K>* b, hn_info* info, uint64_t len) {
   const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
   for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < len; i += stride) {
      Slot<K> s = b[i];
      s.key = empty_key<K>();
      b[i] = s;
   }
   if (blockIdx.x == 0 && threadIdx.x == 0) info->fill = 0;
}

// Fresh table: every slot {EMPTYBUCKET, V()} (splitvec.h:233-238).
template <typename K>
__global__ __launch_bounds__(256) void k_table_init(Slot<K>* b, uint64_t n) {
   const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
   for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride) {
      Slot<K> s;
      s.key = empty_key<K>();
      s.val = 0;
      b[i] = s;
   }
}

__global__ void k_info_init(hn_info* info, int sp) {
   info->size_power = sp;
   info->reserved0 = 0;
   info->fill = 0;
   info->current_max_bucket_overflow = kBucketOverflow;
   info->tombstone_counter = 0;
   info->err = HN_STATUS_INVALID;
   info->reserved1 = 0;
}

// ------------------------------------------------------------ clean_tombstones

struct CleanHeader {
   uint64_t start;   // first slot of region 0 (an EMPTY slot), ~0 = none found yet
   uint64_t total;   // elements lifted out over all regions
   int32_t skip;     // no tombstones (or no usable start): do nothing
   int32_t fail;     // a reinsertion failed
   int32_t no_empty; // no EMPTY slot and scratch too small for the whole table
   int32_t pad;
   uint64_t counters[1]; // [n_regions]
};

constexpr uint64_t kNone = ~0ull;

// `gate` (nullable): run only when *gate is nonzero (the segment pass's flag).
__global__ void k_clean_begin(const hn_info* info, CleanHeader* h, uint32_t n_regions, const uint32_t* gate) {
   for (uint32_t r = threadIdx.x; r < n_regions; r += blockDim.x) h->counters[r] = 0;
   if (threadIdx.x == 0) {
      h->start = kNone;
      h->total = 0;
      h->skip = ((gate && *gate == 0) || info->tombstone_counter == 0) ? 1 : 0;
      h->fail = 0;
      h->no_empty = 0;
   }
}

// Any EMPTY slot will do as the start; the lowest one among the blocks that
// look is taken.  Blocks past an already-found slot stop at once.
template <typename K>
__global__ __launch_bounds__(256) void k_find_empty(const Slot<K>* b, uint64_t n, CleanHeader* h) {
   if (h->skip) return;
   const uint64_t chunk = static_cast<uint64_t>(blockDim.x) * 16;
   const uint64_t lo = static_cast<uint64_t>(blockIdx.x) * chunk;
   if (__hip_atomic_load(&h->start, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < lo) return;
   uint64_t best = kNone;
   for (uint64_t i = lo + threadIdx.x; i < lo + chunk && i < n; i += blockDim.x) {
      if (b[i].key == empty_key<K>()) {
         best = i;
         break;
      }
   }
   if (best != kNone) atomic_min_u64(&h->start, best);
}

__global__ void k_clean_commit(hn_info* info, CleanHeader* h, uint64_t n, uint64_t region_slots) {
   if (h->skip) return;
   if (h->start == kNone) {
      if (region_slots < n) { // cannot order the regions: leave the table as it is
         h->skip = 1;
         h->no_empty = 1;
         return;
      }
      h->start = 0;
   }
   info->tombstone_counter = 0;
   info->current_max_bucket_overflow = kBucketOverflow;
   info->reserved1 = 0; // the reinsertion does not keep Robin Hood order
}

// One region: TOMBSTONE -> EMPTY; a live element away from its home slot is
// copied to scratch and its slot emptied (the isOverflown rule at
// hashinator.h:1285-1297 followed by reset_to_empty).
template <typename K>
__global__ __launch_bounds__(256) void k_clean_extract(Slot<K>* b, int sp, hn_info* info, CleanHeader* h,
                                                        uint32_t region, uint64_t region_slots, Slot<K>* out) {
   if (h->skip) return;
   const uint64_t n = 1ull << sp, mask = n - 1;
   const uint64_t r0 = static_cast<uint64_t>(region) * region_slots;
   if (r0 >= n) return;
   const uint64_t rlen = std::min(region_slots, n - r0);
   const uint64_t start = h->start;
   const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
   const uint64_t iters = (rlen + stride - 1) / stride;
   uint64_t lifted = 0;
   for (uint64_t it = 0; it < iters; ++it) {
      const uint64_t i = it * stride + static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
      bool take = false;
      Slot<K> s{};
      uint64_t slot = 0;
      if (i < rlen) {
         slot = (start + r0 + i) & mask;
         s = b[slot];
         if (s.key == tomb_key<K>()) {
            Slot<K> e = s;
            e.key = empty_key<K>();
            b[slot] = e;
         } else if (s.key != empty_key<K>() && (fib_home(s.key, sp) & mask) != slot) {
            take = true;
         }
      }
      const uint64_t m = __ballot(take);
      if (m) {
         uint64_t wbase = 0;
         const int leader = first_bit(m);
         if (__lane_id() == leader) wbase = atomic_add_relaxed(&h->counters[region], static_cast<uint64_t>(__popcll(m)));
         wbase = __shfl(wbase, leader, kWave);
         if (take) {
            const uint64_t rank = __popcll(m & ((1ull << __lane_id()) - 1ull));
            out[wbase + rank] = s;
            Slot<K> e = s;
            e.key = empty_key<K>();
            b[slot] = e;
         }
         lifted += take ? 1 : 0;
      }
   }
   lifted = wave_sum(lifted);
   if (__lane_id() == 0 && lifted) {
      __hip_atomic_fetch_sub(&info->fill, lifted, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      atomic_add_relaxed(&h->total, lifted);
   }
}

__global__ void k_clean_end(hn_info* info, const CleanHeader* h) {
   if (h->no_empty) {
      info->err = HN_STATUS_FAIL;
      return;
   }
   if (h->skip || h->total == 0) return;
   info->err = h->fail ? HN_STATUS_FAIL : HN_STATUS_SUCCESS;
}

// ------------------------------------------------------------ device_rehash

struct RehashHeader {
   uint64_t prior_fill;
};

template <typename K>
__global__ __launch_bounds__(256) void k_rehash_begin(Slot<K>* nb, uint64_t n, hn_info* info, int new_sp,
                                                       RehashHeader* h) {
   const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
   for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride) {
      Slot<K> s;
      s.key = empty_key<K>();
      s.val = 0;
      nb[i] = s;
   }
   if (blockIdx.x == 0 && threadIdx.x == 0) {
      h->prior_fill = info->fill;
      info->size_power = new_sp;
      info->reserved0 = 0;
      info->fill = 0;
      info->current_max_bucket_overflow = kBucketOverflow;
      info->tombstone_counter = 0;
      info->err = HN_STATUS_INVALID;
      info->reserved1 = 0;
   }
}

// ------------------------------------------------------------ launch helpers

template <typename K, int SRC>
using InsertKernel = void (*)(InsertArgs<K>);

template <typename K, int SRC>
InsertKernel<K, SRC> pick_insert(int G) {
   switch (G) {
   case 1: return k_insert<K, 1, SRC>;
   case 2: return k_insert<K, 2, SRC>;
   case 4: return k_insert<K, 4, SRC>;
   case 8: return k_insert<K, 8, SRC>;
   case 16: return k_insert<K, 16, SRC>;
   case 32: return k_insert<K, 32, SRC>;
   case 64: return k_insert<K, 64, SRC>;
   default: return nullptr;
   }
}

template <typename K, bool PAIRS, int MODE>
using LookupKernel = void (*)(LookupArgs<K>);

template <typename K, bool PAIRS, int MODE>
LookupKernel<K, PAIRS, MODE> pick_lookup(int G) {
   switch (G) {
   case 1: return k_lookup<K, 1, PAIRS, MODE>;
   case 2: return k_lookup<K, 2, PAIRS, MODE>;
   case 4: return k_lookup<K, 4, PAIRS, MODE>;
   case 8: return k_lookup<K, 8, PAIRS, MODE>;
   case 16: return k_lookup<K, 16, PAIRS, MODE>;
   case 32: return k_lookup<K, 32, PAIRS, MODE>;
   case 64: return k_lookup<K, 64, PAIRS, MODE>;
   default: return nullptr;
   }
}

template <typename K, int SRC>
int launch_insert(InsertArgs<K> a, uint64_t grid_len, hipStream_t s, const hn_tune* t, OpKind op) {
   const bool tuned = t && (t->probe_width || t->block_size || t->grid_blocks);
   bool small = false;
   if constexpr (SRC != SRC_TABLE) small = !tuned && !a.d_len && !a.fail_sink && a.len <= kSmallInsert;
   if (small) {
      if constexpr (SRC != SRC_TABLE) {
         constexpr int G = default_probe_width<K>(OP_INSERT);
         if (a.len <= kSoloInsert) {
            hipLaunchKernelGGL((k_insert_small<K, G, SRC>), dim3(1), dim3(kRgBS), 0, s, a, 1);
            return static_cast<int>(hipGetLastError());
         }
         const uint32_t blocks = static_cast<uint32_t>((a.len + kRgBS / G - 1) / (kRgBS / G));
         hipLaunchKernelGGL((k_insert_small<K, G, SRC>), dim3(blocks), dim3(kRgBS), 0, s, a, 0);
      }
   } else {
      Launch L;
      // Up to 2^23 entries 1,024 threads: the fold at a block's end costs about
      // 16 ns on the Info's one line, one block after another (300,000 u64 keys
      // into 2^20 slots: folded per wave 135 us, per 256 threads 70, per 512 58,
      // per 1,024 45; 8 million into 2^24 768, 682, 650 and 634).  Beyond, the
      // smaller blocks, whose CU takes no pause for its longest chain (16 million
      // into 2^26, load .9: 2.42 ms at 256, 2.49 at 1,024).
      hn_tune wide = t ? *t : hn_tune{};
      if (!wide.block_size && grid_len <= 1ull << 23) wide.block_size = 1024;
      int rc = resolve_launch<K>(&wide, op, grid_len, &L);
      if (rc) return rc;
      InsertKernel<K, SRC> k = pick_insert<K, SRC>(L.probe_width);
      if (!k) return HN_EINVAL;
      hipLaunchKernelGGL(k, dim3(L.blocks), dim3(L.block_size), 0, s, a);
   }
   if (!a.fail_sink) hipLaunchKernelGGL(k_insert_finish, dim3(1), dim3(1), 0, s, a.info, a.expected_fill);
   return static_cast<int>(hipGetLastError());
}

template <typename K, bool PAIRS, int MODE>
int launch_lookup(LookupArgs<K> a, hipStream_t s, const hn_tune* t, OpKind op) {
   if constexpr (MODE != LK_RESET) {
      if (!t || t->probe_width == 0) { // automatic: lane windows
         // block_size does not apply: the lane kernel's blocks are lane_block()
         // One query per lane and up (at least 256 per wave left most of the
         // device idle: 1,000 queries of a 2^20-slot table took 17.8 us on four
         // waves, events included, and 10.5 us on 16).
         constexpr int kBlock = lane_block(MODE);
         uint64_t need = (a.len + kBlock - 1) / kBlock;
         if (need == 0) need = 1;
         // one resident wave per block slot: the waves split the queries
         // statically, so a block that waits for a free slot would finish late
         static std::atomic<int> occ{0};
         // at most 16 waves on a CU; the kernel may use fewer (see there)
         const int per_cu =
             std::min(resident_blocks_per_cu(k_lookup_lane<K, PAIRS, MODE>, kBlock, occ), 16 * kWave / kBlock);
         uint64_t cap = (t && t->grid_blocks > 0) ? static_cast<uint64_t>(t->grid_blocks)
                                                  : static_cast<uint64_t>(cu_count()) * per_cu;
         if (cap > (1u << 20)) cap = 1u << 20;
         const uint32_t blocks = static_cast<uint32_t>(need < cap ? need : cap);
         hipLaunchKernelGGL((k_lookup_lane<K, PAIRS, MODE>), dim3(blocks), dim3(kBlock), 0, s, a,
                            t && t->grid_blocks > 0 ? 0u : static_cast<uint32_t>(cu_count()));
         return static_cast<int>(hipGetLastError());
      }
   }
   Launch L;
   int rc = resolve_launch<K>(t, op, a.len, &L);
   if (rc) return rc;
   LookupKernel<K, PAIRS, MODE> k = pick_lookup<K, PAIRS, MODE>(L.probe_width);
   if (!k) return HN_EINVAL;
   hipLaunchKernelGGL(k, dim3(L.blocks), dim3(L.block_size), 0, s, a);
   return static_cast<int>(hipGetLastError());
}

template <typename K>
int insert_soa(const K* keys, const K* vals, void* buckets, hn_info* info, size_t len, hipStream_t s,
               const hn_tune* t) {
   if (!buckets || !info || (len && (!keys || !vals))) return HN_EINVAL;
   InsertArgs<K> a{keys, vals, nullptr, static_cast<Slot<K>*>(buckets), info, len, nullptr, nullptr, nullptr};
   return launch_insert<K, SRC_SOA>(a, len, s, t, OP_INSERT);
}

template <typename K>
int insert_index(const K* keys, void* buckets, hn_info* info, size_t len, hipStream_t s, const hn_tune* t) {
   if (!buckets || !info || (len && !keys)) return HN_EINVAL;
   InsertArgs<K> a{keys, nullptr, nullptr, static_cast<Slot<K>*>(buckets), info, len, nullptr, nullptr, nullptr};
   return launch_insert<K, SRC_INDEX>(a, len, s, t, OP_INSERT);
}

template <typename K>
int insert_pairs(const void* pairs, void* buckets, hn_info* info, size_t len, hipStream_t s, const hn_tune* t) {
   if (!buckets || !info || (len && !pairs)) return HN_EINVAL;
   InsertArgs<K> a{nullptr, nullptr, static_cast<const Slot<K>*>(pairs), static_cast<Slot<K>*>(buckets), info, len,
                   nullptr, nullptr, nullptr};
   return launch_insert<K, SRC_PAIRS>(a, len, s, t, OP_INSERT);
}

template <typename K>
int insert_look(const void* keys, size_t stride, size_t len, const void* buckets, const hn_info* info,
                hn_insert_look* out, hipStream_t s) {
   if (!buckets || !info || !out || (len && (!keys || stride < sizeof(K)))) return HN_EINVAL;
   hipLaunchKernelGGL(k_insert_look<K>, dim3(1), dim3(kLookKeys * 8), 0, s, static_cast<const char*>(keys), stride, len,
                      static_cast<const Slot<K>*>(buckets), info, out);
   return static_cast<int>(hipGetLastError());
}

template <typename K>
int retrieve_soa(const K* keys, K* vals, uint8_t* hit, const void* buckets, const hn_info* info, size_t len,
                 hipStream_t s, const hn_tune* t, bool zero) {
   if (!buckets || !info || (len && (!keys || !vals))) return HN_EINVAL;
   if (len == 0) return 0;
   LookupArgs<K> a{keys, vals, nullptr, hit, const_cast<Slot<K>*>(static_cast<const Slot<K>*>(buckets)),
                   const_cast<hn_info*>(info), len, zero};
   return launch_lookup<K, false, LK_RETRIEVE>(a, s, t, OP_RETRIEVE);
}

template <typename K>
int retrieve_pairs(void* pairs, uint8_t* hit, const void* buckets, const hn_info* info, size_t len, hipStream_t s,
                   const hn_tune* t) {
   if (!buckets || !info || (len && !pairs)) return HN_EINVAL;
   if (len == 0) return 0;
   LookupArgs<K> a{nullptr, nullptr, static_cast<Slot<K>*>(pairs), hit,
                   const_cast<Slot<K>*>(static_cast<const Slot<K>*>(buckets)), const_cast<hn_info*>(info), len, false};
   return launch_lookup<K, true, LK_RETRIEVE>(a, s, t, OP_RETRIEVE);
}

template <typename K>
int erase_keys(const K* keys, void* buckets, hn_info* info, size_t len, hipStream_t s, const hn_tune* t) {
   if (!buckets || !info || (len && !keys)) return HN_EINVAL;
   if (len == 0) return 0;
   LookupArgs<K> a{keys, nullptr, nullptr, nullptr, static_cast<Slot<K>*>(buckets), info, len, false};
   return launch_lookup<K, false, LK_ERASE>(a, s, t, OP_ERASE);
}

template <typename K>
int reset_keys(const void* pairs, void* buckets, hn_info* info, size_t len, hipStream_t s) {
   if (!buckets || !info || (len && !pairs)) return HN_EINVAL;
   if (len == 0) return 0;
   LookupArgs<K> a{nullptr, nullptr, const_cast<Slot<K>*>(static_cast<const Slot<K>*>(pairs)), nullptr,
                   static_cast<Slot<K>*>(buckets), info, len, false};
   return launch_lookup<K, true, LK_RESET>(a, s, nullptr, OP_ERASE);
}

template <typename K>
int reset_all(void* buckets, hn_info* info, size_t len, hipStream_t s) {
   if (!buckets || !info) return HN_EINVAL;
   if (len == 0) return 0; // the reference launches no block for len 0 (hashers.h:155-163): fill stays
   const uint32_t blocks = stream_blocks(len, 256);
   hipLaunchKernelGGL(k_reset_all<K>, dim3(blocks), dim3(256), 0, s, static_cast<Slot<K>*>(buckets), info,
                      static_cast<uint64_t>(len));
   return static_cast<int>(hipGetLastError());
}

template <typename K>
int table_init(void* buckets, size_t n, hipStream_t s) {
   if (!buckets && n) return HN_EINVAL;
   if (n == 0) return 0;
   hipLaunchKernelGGL(k_table_init<K>, dim3(stream_blocks(n, 256)), dim3(256), 0, s, static_cast<Slot<K>*>(buckets),
                      static_cast<uint64_t>(n));
   return static_cast<int>(hipGetLastError());
}

constexpr size_t kHeaderAlign = 256;

size_t clean_header_bytes(uint64_t n_regions) {
   size_t b = sizeof(CleanHeader) + (n_regions ? n_regions - 1 : 0) * sizeof(uint64_t);
   return (b + kHeaderAlign - 1) / kHeaderAlign * kHeaderAlign;
}

// Largest region (in slots) that fits `bytes` of scratch, and the header
// size that goes with it.
template <typename K>
bool clean_plan(uint64_t n, size_t bytes, uint64_t* region_slots, uint64_t* n_regions, size_t* header) {
   const size_t slot = sizeof(Slot<K>);
   for (uint64_t regions = 1; regions <= n; regions *= 2) {
      const uint64_t rs = (n + regions - 1) / regions;
      const size_t hb = clean_header_bytes(regions);
      if (hb + rs * slot <= bytes) {
         *region_slots = rs;
         *n_regions = regions;
         *header = hb;
         return true;
      }
   }
   return false;
}

// Scratch of clean_tombstones.  With room for the segment pass (its header
// and lists, the reorder's, and a pool of at least seg_clean_min_pool()
// bytes) it takes that path; the pool holds segments too long for LDS, and
// when it also holds a whole-table region clean, a table with no EMPTY slot
// is cleaned too.  With less, the region clean alone runs in what there is.
// budget 0: the segment pass with a pool for long segments covering 1/32 of
// the table.  budget SIZE_MAX: enough for any table -- a full one, or one
// segment over the whole table.
template <typename K>
size_t clean_scratch_bytes(int sp, size_t budget) {
   if (sp < 1 || sp > max_size_power<K>()) return 0;
   const uint64_t n = 1ull << sp;
   const size_t fixed = seg_clean_fixed_bytes(sp) + reorder_scratch_bytes(sp);
   const size_t whole = clean_header_bytes(1) + n * sizeof(Slot<K>);
   const size_t pool = seg_clean_default_pool<K>(sp);
   if (budget == 0) return fixed + pool;
   if (budget == SIZE_MAX) return fixed + std::max(std::max(pool, whole), seg_clean_full_pool<K>(sp));
   if (budget >= fixed + seg_clean_min_pool()) return budget;
   uint64_t rs, nr;
   size_t hb;
   for (size_t b = budget; b >= hn_clean_tombstones_min_scratch(); b /= 2)
      if (clean_plan<K>(n, b, &rs, &nr, &hb)) return hb + rs * sizeof(Slot<K>);
   return hn_clean_tombstones_min_scratch();
}

// Probing insert of pairs[0, *d_len) with failures OR-ed into *fail_sink
// (used by the bulk build's fallback, hn_build.hip).
template <typename K>
int launch_insert_pairs_dlen(const Slot<K>* pairs, Slot<K>* buckets, hn_info* info, uint64_t max_len,
                             const uint64_t* d_len, int32_t* fail_sink, hipStream_t s) {
   InsertArgs<K> a{nullptr, nullptr, pairs, buckets, info, max_len, d_len, nullptr, fail_sink};
   return launch_insert<K, SRC_PAIRS>(a, max_len, s, nullptr, OP_REINSERT);
}
template <typename K>
int launch_insert_table_dlen(const Slot<K>* table, Slot<K>* buckets, hn_info* info, uint64_t max_len,
                             const uint64_t* d_len, int32_t* fail_sink, hipStream_t s) {
   InsertArgs<K> a{nullptr, nullptr, table, buckets, info, max_len, d_len, nullptr, fail_sink};
   return launch_insert<K, SRC_TABLE>(a, max_len, s, nullptr, OP_REINSERT);
}
template <typename K>
int launch_insert_batch_dlen(const K* keys, const K* vals, const Slot<K>* pairs, Slot<K>* buckets, hn_info* info,
                             uint64_t max_len, const uint64_t* d_len, int32_t* fail_sink, hipStream_t s) {
   InsertArgs<K> a{keys, vals, pairs, buckets, info, max_len, d_len, nullptr, fail_sink};
   if (pairs) return launch_insert<K, SRC_PAIRS>(a, max_len, s, nullptr, OP_INSERT);
   if (vals) return launch_insert<K, SRC_SOA>(a, max_len, s, nullptr, OP_INSERT);
   return launch_insert<K, SRC_INDEX>(a, max_len, s, nullptr, OP_INSERT);
}
#define HN_DLEN(K)                                                                                                    \
   template int launch_insert_table_dlen<K>(const Slot<K>*, Slot<K>*, hn_info*, uint64_t, const uint64_t*, int32_t*,  \
                                            hipStream_t);                                                             \
   template int launch_insert_batch_dlen<K>(const K*, const K*, const Slot<K>*, Slot<K>*, hn_info*, uint64_t,         \
                                            const uint64_t*, int32_t*, hipStream_t);
HN_DLEN(uint32_t)
HN_DLEN(uint64_t)
#undef HN_DLEN
template int launch_insert_pairs_dlen<uint32_t>(const Slot<uint32_t>*, Slot<uint32_t>*, hn_info*, uint64_t,
                                                const uint64_t*, int32_t*, hipStream_t);
template int launch_insert_pairs_dlen<uint64_t>(const Slot<uint64_t>*, Slot<uint64_t>*, hn_info*, uint64_t,
                                                const uint64_t*, int32_t*, hipStream_t);

// The region clean: TOMBSTONE -> EMPTY and displaced elements lifted out and
// reinserted, region by region from an EMPTY slot; `gate` as in k_clean_begin.
template <typename K>
int region_clean(void* buckets, hn_info* info, int sp, void* scratch, size_t bytes, const uint32_t* gate,
                 hipStream_t s) {
   const uint64_t n = 1ull << sp;
   uint64_t rs = 0, nr = 0;
   size_t hb = 0;
   if (!clean_plan<K>(n, bytes, &rs, &nr, &hb)) return HN_ESCRATCH;
   CleanHeader* h = static_cast<CleanHeader*>(scratch);
   Slot<K>* pairs = reinterpret_cast<Slot<K>*>(static_cast<char*>(scratch) + hb);
   Slot<K>* b = static_cast<Slot<K>*>(buckets);
   hipLaunchKernelGGL(k_clean_begin, dim3(1), dim3(256), 0, s, info, h, static_cast<uint32_t>(nr), gate);
   const uint64_t chunk = 256 * 16;
   hipLaunchKernelGGL(k_find_empty<K>, dim3(static_cast<uint32_t>((n + chunk - 1) / chunk)), dim3(256), 0, s, b, n, h);
   hipLaunchKernelGGL(k_clean_commit, dim3(1), dim3(1), 0, s, info, h, n, rs);
   for (uint64_t r = 0; r < nr; ++r) {
      hipLaunchKernelGGL(k_clean_extract<K>, dim3(stream_blocks(rs, 256)), dim3(256), 0, s, b, sp, info, h,
                         static_cast<uint32_t>(r), rs, pairs);
      InsertArgs<K> a{nullptr, nullptr, pairs, b, info, rs, &h->counters[r], nullptr, &h->fail};
      int rc = launch_insert<K, SRC_PAIRS>(a, rs, s, nullptr, OP_REINSERT);
      if (rc) return rc;
   }
   hipLaunchKernelGGL(k_clean_end, dim3(1), dim3(1), 0, s, info, h);
   return static_cast<int>(hipGetLastError());
}

// Hashmap::clean_tombstones (hashinator.h:1261-1315).
template <typename K>
int clean_tombstones(void* buckets, hn_info* info, int sp, void* scratch, size_t bytes, hipStream_t s) {
   if (!buckets || !info || !scratch) return HN_EINVAL;
   if (sp < 1 || sp > max_size_power<K>()) return HN_EINVAL;
   const uint64_t n = 1ull << sp;
   const size_t seg = seg_clean_fixed_bytes(sp), ro = reorder_scratch_bytes(sp);
   if (bytes < seg + ro + seg_clean_min_pool()) return region_clean<K>(buckets, info, sp, scratch, bytes, nullptr, s);
   char* base = static_cast<char*>(scratch);
   char* pool = base + seg + ro;
   const size_t pool_bytes = bytes - seg - ro;
   uint64_t rs = 0, nr = 0;
   size_t hb = 0;
   const bool region_ok = clean_plan<K>(n, pool_bytes, &rs, &nr, &hb) && nr == 1;
   int rc = seg_clean<K>(buckets, info, sp, base, pool, pool_bytes, region_ok, s);
   if (rc || !region_ok) return rc;
   // a table with no EMPTY slot: one region over the whole table, then the reorder
   const uint32_t* gate = seg_clean_gate(base);
   rc = region_clean<K>(buckets, info, sp, pool, pool_bytes, gate, s);
   if (rc) return rc;
   return reorder_gated<K>(buckets, info, sp, base + seg, ro, gate, s);
}

template <typename K>
int rehash(const void* old_b, int old_sp, void* new_b, int new_sp, hn_info* info, void* scratch, hipStream_t s) {
   if (!old_b || !new_b || !info || !scratch) return HN_EINVAL;
   if (old_sp < 1 || old_sp > max_size_power<K>() || new_sp < 1 || new_sp > max_size_power<K>()) return HN_EINVAL;
   if (new_sp > 32) return HN_EINVAL; // hashinator.h:288-290 throws beyond 32 bits
   const uint64_t on = 1ull << old_sp, nn = 1ull << new_sp;
   const char* o0 = static_cast<const char*>(old_b);
   const char* n0 = static_cast<const char*>(new_b);
   if (o0 < n0 + nn * sizeof(Slot<K>) && n0 < o0 + on * sizeof(Slot<K>)) return HN_EINVAL;
   RehashHeader* h = static_cast<RehashHeader*>(scratch);
   hipLaunchKernelGGL(k_rehash_begin<K>, dim3(stream_blocks(nn, 256)), dim3(256), 0, s, static_cast<Slot<K>*>(new_b),
                      nn, info, new_sp, h);
   InsertArgs<K> a{nullptr, nullptr, static_cast<const Slot<K>*>(old_b), static_cast<Slot<K>*>(new_b), info, on,
                   nullptr, &h->prior_fill, nullptr};
   return launch_insert<K, SRC_TABLE>(a, on, s, nullptr, OP_REINSERT);
}

} // namespace hn

using namespace hn;

extern "C" {

int hn_info_init(hn_info* info, int sp, hn_stream_t s) {
   if (!info) return HN_EINVAL;
   hipLaunchKernelGGL(k_info_init, dim3(1), dim3(1), 0, s, info, sp);
   return static_cast<int>(hipGetLastError());
}

int hn_table_init_u32(void* b, size_t n, hn_stream_t s) { return table_init<uint32_t>(b, n, s); }
int hn_table_init_u64(void* b, size_t n, hn_stream_t s) { return table_init<uint64_t>(b, n, s); }

int hn_insert_u32(const uint32_t* k, const uint32_t* v, void* b, hn_info* i, size_t n, hn_stream_t s,
                  const hn_tune* t) {
   return insert_soa<uint32_t>(k, v, b, i, n, s, t);
}
int hn_insert_u64(const uint64_t* k, const uint64_t* v, void* b, hn_info* i, size_t n, hn_stream_t s,
                  const hn_tune* t) {
   return insert_soa<uint64_t>(k, v, b, i, n, s, t);
}
int hn_insert_index_u32(const uint32_t* k, void* b, hn_info* i, size_t n, hn_stream_t s, const hn_tune* t) {
   return insert_index<uint32_t>(k, b, i, n, s, t);
}
int hn_insert_index_u64(const uint64_t* k, void* b, hn_info* i, size_t n, hn_stream_t s, const hn_tune* t) {
   return insert_index<uint64_t>(k, b, i, n, s, t);
}
int hn_insert_pairs_u32(const void* p, void* b, hn_info* i, size_t n, hn_stream_t s, const hn_tune* t) {
   return insert_pairs<uint32_t>(p, b, i, n, s, t);
}
int hn_insert_pairs_u64(const void* p, void* b, hn_info* i, size_t n, hn_stream_t s, const hn_tune* t) {
   return insert_pairs<uint64_t>(p, b, i, n, s, t);
}
int hn_insert_look_u32(const void* k, size_t stride, size_t n, const void* b, const hn_info* i, hn_insert_look* out,
                       hn_stream_t s) {
   return insert_look<uint32_t>(k, stride, n, b, i, out, s);
}
int hn_insert_look_u64(const void* k, size_t stride, size_t n, const void* b, const hn_info* i, hn_insert_look* out,
                       hn_stream_t s) {
   return insert_look<uint64_t>(k, stride, n, b, i, out, s);
}
int hn_retrieve_u32(const uint32_t* k, uint32_t* v, uint8_t* h, const void* b, const hn_info* i, size_t n,
                    hn_stream_t s, const hn_tune* t) {
   return retrieve_soa<uint32_t>(k, v, h, b, i, n, s, t, false);
}
int hn_retrieve_u64(const uint64_t* k, uint64_t* v, uint8_t* h, const void* b, const hn_info* i, size_t n,
                    hn_stream_t s, const hn_tune* t) {
   return retrieve_soa<uint64_t>(k, v, h, b, i, n, s, t, false);
}
int hn_retrieve_zero_u32(const uint32_t* k, uint32_t* v, uint8_t* h, const void* b, const hn_info* i, size_t n,
                         hn_stream_t s, const hn_tune* t) {
   return retrieve_soa<uint32_t>(k, v, h, b, i, n, s, t, true);
}
int hn_retrieve_zero_u64(const uint64_t* k, uint64_t* v, uint8_t* h, const void* b, const hn_info* i, size_t n,
                         hn_stream_t s, const hn_tune* t) {
   return retrieve_soa<uint64_t>(k, v, h, b, i, n, s, t, true);
}
int hn_retrieve_pairs_u32(void* p, uint8_t* h, const void* b, const hn_info* i, size_t n, hn_stream_t s,
                          const hn_tune* t) {
   return retrieve_pairs<uint32_t>(p, h, b, i, n, s, t);
}
int hn_retrieve_pairs_u64(void* p, uint8_t* h, const void* b, const hn_info* i, size_t n, hn_stream_t s,
                          const hn_tune* t) {
   return retrieve_pairs<uint64_t>(p, h, b, i, n, s, t);
}
int hn_erase_u32(const uint32_t* k, void* b, hn_info* i, size_t n, hn_stream_t s, const hn_tune* t) {
   return erase_keys<uint32_t>(k, b, i, n, s, t);
}
int hn_erase_u64(const uint64_t* k, void* b, hn_info* i, size_t n, hn_stream_t s, const hn_tune* t) {
   return erase_keys<uint64_t>(k, b, i, n, s, t);
}
int hn_reset_all_u32(void* b, hn_info* i, size_t n, hn_stream_t s) { return reset_all<uint32_t>(b, i, n, s); }
int hn_reset_u32(const void* p, void* b, hn_info* i, size_t n, hn_stream_t s) { return reset_keys<uint32_t>(p, b, i, n, s); }
int hn_reset_u64(const void* p, void* b, hn_info* i, size_t n, hn_stream_t s) { return reset_keys<uint64_t>(p, b, i, n, s); }
int hn_reset_all_u64(void* b, hn_info* i, size_t n, hn_stream_t s) { return reset_all<uint64_t>(b, i, n, s); }

size_t hn_clean_tombstones_min_scratch(void) { return 64 * 1024; }
size_t hn_clean_tombstones_scratch_bytes_u32(int sp, size_t budget) { return clean_scratch_bytes<uint32_t>(sp, budget); }
size_t hn_clean_tombstones_scratch_bytes_u64(int sp, size_t budget) { return clean_scratch_bytes<uint64_t>(sp, budget); }
int hn_clean_tombstones_u32(void* b, hn_info* i, int sp, void* sc, size_t sb, hn_stream_t s) {
   return clean_tombstones<uint32_t>(b, i, sp, sc, sb, s);
}
int hn_clean_tombstones_u64(void* b, hn_info* i, int sp, void* sc, size_t sb, hn_stream_t s) {
   return clean_tombstones<uint64_t>(b, i, sp, sc, sb, s);
}

size_t hn_rehash_scratch_bytes(void) { return 256; }
int hn_rehash_u32(const void* ob, int osp, void* nb, int nsp, hn_info* i, void* sc, hn_stream_t s) {
   return rehash<uint32_t>(ob, osp, nb, nsp, i, sc, s);
}
int hn_rehash_u64(const void* ob, int osp, void* nb, int nsp, hn_info* i, void* sc, hn_stream_t s) {
   return rehash<uint64_t>(ob, osp, nb, nsp, i, sc, s);
}

const char* hn_version(void) { return "hashinator_amd 0.1 gfx950"; }

} // extern "C"
