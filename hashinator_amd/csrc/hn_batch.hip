// hn_batch.hip -- many independent maps in a few launches.
//
// No counterpart kernel in the reference (its API is one launch per map per
// operation, hashers.h:46-163); the per-map semantics are the reference's:
// for each map, in order, insert (insert_kernel, kernels_AMD.h:272-405),
// retrieve (retrieve_kernel 647-697), erase (delete_kernel 412-505), then
// clean_tombstones (hashinator.h:1261-1315).
//
// The default (no launch tuning asked for): every map is cut into regions of
// 64 KiB of slots (8,192 u32, 4,096 u64), and a workgroup runs a phase on one
// region in LDS (k_region_insert, k_region_lookup, k_region_clean).  It reads
// the map's whole key list and takes the keys whose home lies in its region;
// what probes past the region's end is left to the kernels that follow
// (k_boundary_insert, k_map_insert_end; k_map_clean_end) or, for lookups, goes
// on in global memory.  One workgroup per map left the call waiting for the
// largest maps' probe chains (1,024 u32 maps of 2^8..2^16 slots at load
// factor 0.6, velocity-grid ids: 4.99 ms, two launches of 2.16 ms among them;
// by regions 1.04 ms: insert 0.32 + 0.08, lookups 0.35, clean 0.15 + 0.05 ms.
// 4,096 such maps: 10.3 -> 4.2 ms; one u64 map of 2^20 slots: 13.8 -> 1.3
// ms).  What is few keys for its map goes another way (map_ways): the insert
// and the erase by one workgroup that probes the table where it stands
// (k_batch_group), lookups one key per lane (k_batch_retrieve_lane), as do
// query lists much longer than the table.  A small call is launches only, so
// the set-up (batch_prep) is a workgroup of the first of them, and an insert
// is 4 launches, lookups and erases 3 (one map of 2^13 slots, 16 keys updated
// 38 us by 6 launches and 19 us by 4; one workgroup in 2 launches 15).
//
// Maps of more than kMaxRegions regions, maps that a call barely touches, and
// calls with explicit tuning: one workgroup owns one map at a time and runs
// insert, and erase + clean, on it back to back, separated by workgroup
// barriers with workgroup-scope fences (no other workgroup touches the map
// during the launch).  With tuning, maps are handed out by an atomic ticket in
// the order the caller lists them (largest first balances the grid).  Retrieve
// runs between the two, one key per lane over units of every map's queries.
// The probe loops are the single-map ones (hn_probe.hpp), so a map's results
// are those of the plain calls.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "hn_device.hpp"
#include "hn_host.hpp"
#include "hn_probe.hpp"
#include "hn_region.hpp"

namespace hn {

template <typename K>
struct BatchArgs {
   const hn_batch_map* maps;
   uint32_t n_maps;
   uint32_t ops;
   const K* ins_keys;
   const K* ins_vals;
   const K* qry_keys;
   K* qry_vals;
   uint8_t* qry_hit;
   const K* ers_keys;
   Slot<K>* clean_scratch;
   uint64_t* ticket;
   uint32_t req; // the call's phases (ops is the launch's)
};

// ------------------------------------------------------- ways of a map
constexpr uint64_t kMaxRegions = 1024;

// Whether a map's queries are looked up by units, although it has regions.
// Each of its regions' workgroups reads the whole list (0.43 ns a query) and
// looks up its own share (2.2 ns each) on the CU that it has; the units go over
// the whole device, but wait for memory, and for clustered keys' long probes.
// So by units: lists that a region takes long for, over 30 us where it is alone,
// over 100 where the regions of as many such maps as the call has would give
// every CU one; and maps of more than 32 regions, whose reading
// costs more than the lookups.  By regions and by units, us a call: one u32 map
// of 2^13 slots, 8,192 queries 45 and 46, 2^22 9,480 and 75; 100 such maps,
// 30,011 each 97 and 64; 256, 8,192 each 55 and 67, 32,768 each 122 and 143; one
// of 2^16 slots with 65,536 73 and 46, 64 with 78,643 ids of a grid each 130 and
// 296; one of 2^20 with 262,144 144 and 54; one u64 map of 2^22 slots, 2^24
// queries 19,300 and 449.
constexpr uint64_t kRegionsByUnits = 32, kRegionsFill = 256;
__device__ __forceinline__ bool by_units(uint64_t nq, uint64_t regions, uint32_t n_maps) {
   const uint64_t wgs = n_maps * regions;
   const uint64_t limit_ns = 30000 + 70000 * (wgs < kRegionsFill ? wgs : kRegionsFill) / kRegionsFill;
   return regions == 0 || regions > kRegionsByUnits || nq * (430 * regions + 2200) > 1000 * limit_ns * regions;
}

// How a map's phases run: by its regions, or else by one workgroup (insert,
// erase, clean) and by units (retrieve).
enum : uint32_t { kWayIns = 1, kWayQry = 2, kWayErs = 4, kWayClean = 8 };

// The map's regions, or 0: a size power out of range; more than kMaxRegions of
// them (every region reads the map's whole key lists, so the reads grow with the
// square of the map: a u64 map of 1,024 regions at load factor 0.6 takes 13.9
// ms, one of 256 1.3 ms, against 54 and 13.8 ms for one workgroup per map); or
// lists too long for 32-bit indices.
template <typename K>
__device__ __forceinline__ uint32_t map_regions(const hn_batch_map& M, int sp, uint32_t ops) {
   if (sp < 1 || sp > max_size_power<K>()) return 0;
   const uint64_t nreg = sp <= kRegionLogB<K> ? 1 : 1ull << (sp - kRegionLogB<K>);
   const uint64_t longest = ((ops & HN_BATCH_INSERT) ? M.ins_len : 0) | ((ops & HN_BATCH_RETRIEVE) ? M.qry_len : 0) |
                            ((ops & HN_BATCH_ERASE) ? M.ers_len : 0);
   return nreg > kMaxRegions || (longest >> 31) ? 0 : static_cast<uint32_t>(nreg);
}
// A map of several regions goes by them unless its lists hold fewer keys than a
// sixteenth of the slots, where loading the table costs more than probing it.
__device__ __forceinline__ bool several_pay(const hn_batch_map& M, uint32_t nreg, uint64_t n, uint32_t ops,
                                            uint32_t n_maps) {
   const uint64_t nq = (ops & HN_BATCH_RETRIEVE) && !by_units(M.qry_len, nreg, n_maps) ? M.qry_len : 0;
   const uint64_t keys = ((ops & HN_BATCH_INSERT) ? M.ins_len : 0) + nq + ((ops & HN_BATCH_ERASE) ? M.ers_len : 0);
   return (ops & HN_BATCH_CLEAN) || keys * 16 >= n;
}
// Whether a map is inserted into by regions.  A map of one region is above an
// eighth of its slots; up to there, its one workgroup probes the table where it
// stands (4,096 u32 maps of 2^13 slots, 16 keys each 56 us, through LDS 188,
// 1,024 of their keys updated 179 and 245; 1,024 maps, a quarter of the slots
// into empty ones 117 and 62), unless TOMBSTONEs make the probes long (a table
// full of them: 24 ms and 0.2).  By what an insert does not change, so that two
// workgroups that ask agree.
template <typename K>
__device__ __forceinline__ bool ins_by_regions(const hn_batch_map& M, const hn_info* info, int sp, uint32_t ops,
                                               uint32_t n_maps) {
   const uint32_t nreg = map_regions<K>(M, sp, ops);
   if (!(ops & HN_BATCH_INSERT) || nreg == 0 || M.ins_len == 0) return false;
   const uint64_t n = 1ull << sp;
   return nreg > 1 ? several_pay(M, nreg, n, ops, n_maps) : M.ins_len * 8 > n || info->tombstone_counter * 4 >= n;
}
// All of a map's ways, decided once a call (batch_prep).  The keys of a map of
// one region are looked up and erased where the table stands while they are few,
// since indexing the region costs more than their probes, and by the region as
// the probes get long.  Measured at u32, so / by the region:
// - lookups, from 512 queries or as many as slots on, and where seven eighths of
//   the slots are taken: 256 maps of 2^12 slots, 128 queries, load factor 0.6 23
//   and 27 us, 0.9 74 and 29, 4,096 maps 53 and 147, 129 and 152, 512 queries at
//   0.6 80 and 155 but one map of 2^10 27 and 24; fewer than 2^10 slots 62 and
//   113 also at 0.9;
// - erases, from a tenth of the slots on (256 maps of 2^13 slots, 0.6: a
//   sixteenth 29 and 36 us, a quarter 55 and 37), where five eighths are taken
//   from a 64th on (0.8: 49 and 36; of 2^10 slots 35 and 26; 4 keys each of 4,096
//   maps of 2^8 83 and 105);
// - both where nearly all are: a table full of TOMBSTONEs is probed slot by slot.
// The lines lie lower than lists like these alone would have them (4,096 maps of
// 2^8, an eighth erased at 0.6: 99 and 110 us), since among larger maps both
// ways run and each waits for its last map (1,024 maps of 2^8..2^16 slots, all
// phases: a quarter of the slots of small maps as the line 1,108 us, a tenth
// 1,081).
template <typename K>
__device__ __forceinline__ uint32_t map_ways(const hn_batch_map& M, const hn_info* info, int sp, uint32_t ops,
                                             uint32_t n_maps) {
   const uint32_t nreg = map_regions<K>(M, sp, ops);
   if (nreg == 0) return 0;
   const uint64_t n = 1ull << sp, nq = (ops & HN_BATCH_RETRIEVE) ? M.qry_len : 0;
   const uint64_t ne = (ops & HN_BATCH_ERASE) ? M.ers_len : 0;
   bool qry = nq && !by_units(nq, nreg, n_maps), ers = ne != 0;
   if (nreg > 1) {
      if (!several_pay(M, nreg, n, ops, n_maps)) return 0;
   } else {
      const uint64_t used = info->fill + info->tombstone_counter + ((ops & HN_BATCH_INSERT) ? M.ins_len : 0);
      const bool full = used * 16 >= n * 15;
      qry = qry && (nq >= 512 || nq >= n || full || (sp >= 10 && used * 8 >= n * 7));
      ers = ers && (ne * 10 >= n || full || (used * 8 >= n * 5 && ne >= 16 && ne * 64 >= n));
   }
   return (ins_by_regions<K>(M, info, sp, ops, n_maps) ? kWayIns : 0u) | (qry ? kWayQry : 0u) | (ers ? kWayErs : 0u) |
          ((ops & HN_BATCH_CLEAN) ? kWayClean : 0u);
}

__device__ __forceinline__ void phase_barrier() {
   __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
   __syncthreads();
   __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// One workgroup runs `ops` on one map.
struct GroupMem {
   unsigned long long placed, max, erased, lifted;
   int failed;
};
template <typename K, int G>
__device__ __forceinline__ void map_phases(const BatchArgs<K>& a, const hn_batch_map& M, uint32_t ops, GroupMem& S) {
   const uint64_t groups = blockDim.x / G;
   const uint64_t g = threadIdx.x / G;
   const int lane = __lane_id();
   hn_info* info = M.info;
   Slot<K>* b = static_cast<Slot<K>*>(M.buckets);
   const int sp = info->size_power;
   const bool sp_ok = sp >= 1 && sp <= max_size_power<K>();
   const uint64_t nsl = sp_ok ? (1ull << sp) : 0;
   auto fold_insert = [&](const InsertCounters& c) {
      const uint64_t p = wave_sum(c.placed);
      const uint64_t m = wave_max(c.max_probe);
      const int f = wave_max(c.failed);
      if (lane == 0) {
         if (p) atomicAdd(&S.placed, static_cast<unsigned long long>(p));
         if (m) atomicMax(&S.max, static_cast<unsigned long long>(m));
         if (f) atomicOr(&S.failed, 1);
      }
   };
   if (threadIdx.x == 0) S = GroupMem{0, 0, 0, 0, 0};
   __syncthreads();
   if (ops & HN_BATCH_INSERT) {
      InsertCounters c;
      if (sp_ok) {
         InsertArgs<K> ia{a.ins_keys + M.ins_off, a.ins_vals + M.ins_off, nullptr, b, info, M.ins_len,
                          nullptr, nullptr, nullptr};
         insert_range<K, G, SRC_SOA>(ia, sp, M.ins_len, g, groups, c);
      }
      fold_insert(c);
      __syncthreads();
      if (threadIdx.x == 0) {
         info->fill += S.placed;
         if (S.max) {
            const uint64_t o = next_overflow(S.max, kBucketOverflow);
            if (o > info->current_max_bucket_overflow) info->current_max_bucket_overflow = o;
         }
         info->err = (S.failed || !sp_ok) ? HN_STATUS_FAIL : HN_STATUS_SUCCESS;
         info->reserved1 = 0; // inserts do not keep Robin Hood order
         S.placed = 0;
         S.max = 0;
         S.failed = 0;
      }
      phase_barrier();
   }
   if ((ops & HN_BATCH_RETRIEVE) && sp_ok) {
      LookupArgs<K> la{a.qry_keys + M.qry_off, a.qry_vals + M.qry_off, nullptr,
                       a.qry_hit ? a.qry_hit + M.qry_off : nullptr, b, info, M.qry_len, false};
      lookup_range<K, G, false, LK_RETRIEVE>(la, sp, info->current_max_bucket_overflow, M.qry_len, g, groups,
                                             (info->reserved1 & kInfoOrdered) != 0);
      phase_barrier();
   }
   if ((ops & HN_BATCH_ERASE) && sp_ok) {
      LookupArgs<K> la{a.ers_keys + M.ers_off, nullptr, nullptr, nullptr, b, info, M.ers_len, false};
      const uint64_t e =
          wave_sum(lookup_range<K, G, false, LK_ERASE>(la, sp, info->current_max_bucket_overflow, M.ers_len, g, groups,
                                                       (info->reserved1 & kInfoOrdered) != 0));
      if (lane == 0 && e) atomicAdd(&S.erased, static_cast<unsigned long long>(e));
      __syncthreads();
      if (threadIdx.x == 0) {
         info->tombstone_counter += S.erased;
         info->fill -= S.erased;
      }
      phase_barrier();
   }
   if ((ops & HN_BATCH_CLEAN) && sp_ok && info->tombstone_counter > 0) {
      if (info->fill > M.scratch_cap) {
         // not enough scratch to lift the displaced elements out: leave the map as it is
         if (threadIdx.x == 0) info->err = HN_STATUS_FAIL;
      } else {
         // TOMBSTONE -> EMPTY; live elements away from home are lifted into scratch (one region: the map)
         Slot<K>* out = a.clean_scratch + M.scratch_off;
         const uint64_t mask = nsl - 1;
         for (uint64_t base = 0; base < nsl; base += blockDim.x) {
            const uint64_t i = base + threadIdx.x;
            bool take = false;
            Slot<K> s{};
            if (i < nsl) {
               s = b[i];
               if (s.key == tomb_key<K>()) {
                  Slot<K> e = s;
                  e.key = empty_key<K>();
                  b[i] = e;
               } else if (s.key != empty_key<K>() && (fib_home(s.key, sp) & mask) != i) {
                  take = true;
               }
            }
            const uint64_t m = __ballot(take);
            if (m) {
               unsigned long long wb = 0;
               const int leader = first_bit(m);
               if (lane == leader) wb = atomicAdd(&S.lifted, static_cast<unsigned long long>(__popcll(m)));
               wb = __shfl(wb, leader, kWave);
               if (take) {
                  out[wb + __popcll(m & ((1ull << lane) - 1ull))] = s;
                  Slot<K> e = s;
                  e.key = empty_key<K>();
                  b[i] = e;
               }
            }
         }
         phase_barrier();
         const uint64_t lifted = S.lifted;
         if (threadIdx.x == 0) {
            info->tombstone_counter = 0;
            info->current_max_bucket_overflow = kBucketOverflow;
            info->fill -= lifted;
            info->reserved1 = 0; // the reinsertion does not keep Robin Hood order
         }
         phase_barrier();
         InsertCounters c;
         if (lifted) {
            InsertArgs<K> ia{nullptr, nullptr, out, b, info, lifted, nullptr, nullptr, nullptr};
            insert_range<K, G, SRC_PAIRS>(ia, sp, lifted, g, groups, c);
         }
         fold_insert(c);
         __syncthreads();
         if (threadIdx.x == 0) {
            info->fill += S.placed;
            if (S.max) {
               const uint64_t o = next_overflow(S.max, kBucketOverflow);
               if (o > info->current_max_bucket_overflow) info->current_max_bucket_overflow = o;
            }
            if (lifted) info->err = S.failed ? HN_STATUS_FAIL : HN_STATUS_SUCCESS;
         }
      }
      phase_barrier();
   }
   __syncthreads(); // S is set again by thread 0 next
}

template <typename K, int G>
__global__ __launch_bounds__(1024) void k_batch(BatchArgs<K> a) {
   __shared__ uint64_t s_map;
   __shared__ GroupMem S;
   for (;;) {
      if (threadIdx.x == 0) s_map = __hip_atomic_fetch_add(a.ticket, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __syncthreads();
      const uint64_t mi = s_map;
      if (mi >= a.n_maps) break;
      map_phases<K, G>(a, a.maps[mi], a.ops, S);
   }
}

__global__ void k_zero_u64(uint64_t* p) { *p = 0; }

// ---------------------------------------------------------- retrieve phase
//
// The queries of maps without regions, and of those with regions whose lists
// are long (by_units), run on their own, one key per lane (lane_lookup): they
// are cut into units of kBatchUnit, numbered map after map (map m owns units
// [unit_start[m], unit_start[m+1]), so units come in the caller's map order,
// largest maps first), and dealt to the waves in turn: units are alike, a
// ticket for each wave and unit took 16 ns apiece (53 us of any call), and with
// units of 4,096 the last one alone took 130.  No unit is empty.  Results per
// map are those of the plain retrieve: maps are independent, and the phases
// still run insert -> retrieve -> erase -> clean for each of them.
constexpr uint64_t kBatchUnit = 1024;

struct BatchScratch {
   uint64_t ticket;  // map ticket of k_batch
   uint64_t units;   // retrieve units of all maps
   uint64_t items;   // regions of all maps
   uint32_t several; // maps of several regions
   uint32_t any;     // kAny*: what there is to do for whole launches
   uint64_t pad[4];
   // followed by unit_start[n_maps + 1], item_start[n_maps + 1], MapState[n_maps], the spill lists
};
static_assert(sizeof(BatchScratch) == 64, "header of hn_batch_scratch_bytes");
enum : uint32_t {
   kAnyIns = 1,     // a map is inserted into by regions
   kAnyLook = 2,    // a map is looked up, or erased from, by regions
   kAnyGroup = 4,   // a map is erased from, or cleaned, by one workgroup
   kAnySpill = 8,   // an insert ran past its region's end
   kAnyLeft = 16,   // k_boundary_insert left some of those
   kAnyListed = 32, // clean: a map of several regions has listed keys
};
// Read first: 2,280 regions' atomics on the one word took 35 us.
__device__ __forceinline__ void set_any(BatchScratch* sc, uint32_t bits) {
   if (!(__hip_atomic_load(&sc->any, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & bits))
      __hip_atomic_fetch_or(&sc->any, bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// What the region kernels leave for the per-map kernels.
struct MapState {
   uint32_t ways;      // kWay*
   uint32_t list;      // a map of several regions: its spill list, if below spill_lists(n_maps)
   uint32_t spilled;   // 1: an insert ran past its region's end; 2: k_boundary_insert left some keys
   uint32_t n_spill;   // such keys; the first ones are listed by index
   uint32_t listed;    // clean: keys in the map's scratch slice, to be placed by k_map_clean_end
   uint32_t max_probe; // clean: longest probe of the keys placed by the regions
   uint32_t displaced; // clean: a live key stood away from its home slot
   uint32_t placed;    // clean: keys placed by the regions and their borders
};
// Indices in a spill list.  Only maps of several regions can spill, and only
// the first kSpillLists of them have a list (a list a map made a batch of a
// million maps of one region take 1 GB of workspace; now 48 MB): without one,
// or when it is full, k_boundary_insert looks through all of the map's keys.
constexpr uint32_t kSpillCap = 248, kSpillLists = 4096;
__host__ __device__ inline uint32_t spill_lists(uint32_t n_maps) { return n_maps < kSpillLists ? n_maps : kSpillLists; }

__host__ __device__ inline uint64_t* unit_start(BatchScratch* sc) { return reinterpret_cast<uint64_t*>(sc + 1); }
__host__ __device__ inline uint64_t* item_start(BatchScratch* sc, uint32_t n_maps) {
   return unit_start(sc) + n_maps + 1;
}
__host__ __device__ inline MapState* map_state(BatchScratch* sc, uint32_t n_maps) {
   return reinterpret_cast<MapState*>(item_start(sc, n_maps) + n_maps + 1);
}
// A map's spill list and how many indices it holds.
struct SpillList {
   uint32_t* idx;
   uint32_t cap;
   __device__ SpillList(BatchScratch* sc, uint32_t n_maps, const MapState& st)
       : idx(reinterpret_cast<uint32_t*>(map_state(sc, n_maps) + n_maps) + static_cast<uint64_t>(st.list) * kSpillCap),
         cap(st.list < spill_lists(n_maps) ? kSpillCap : 0) {}
};

size_t batch_scratch_bytes(uint32_t n_maps) {
   const size_t b = sizeof(BatchScratch) + (static_cast<size_t>(n_maps) + 1) * 2 * sizeof(uint64_t) +
                    static_cast<size_t>(n_maps) * sizeof(MapState) +
                    static_cast<size_t>(spill_lists(n_maps)) * kSpillCap * sizeof(uint32_t);
   return (b + 255) & ~static_cast<size_t>(255);
}

// Block-wide exclusive prefixes of N values per thread (kRgBS threads, sums
// below 2^32); total receives the sums.  wsum: one entry per wave.
template <int N>
__device__ __forceinline__ void block_excl_scan(uint32_t (&v)[N], uint32_t (*wsum)[N], uint32_t (&total)[N]) {
   const int lane = __lane_id(), w = threadIdx.x / kWave;
   static_assert(kRgWaves <= 16, "a row of 16 lanes scans the waves' sums");
#pragma unroll
   for (int k = 0; k < N; ++k) {
      const uint32_t x = wave_incl_add(v[k]);
      if (lane == kWave - 1) wsum[w][k] = x;
      v[k] = x - v[k];
   }
   __syncthreads();
#pragma unroll
   for (int k = 0; k < N; ++k) {
      const uint32_t mine = (lane & 15) < kRgWaves ? wsum[lane & 15][k] : 0;
      int x = static_cast<int>(mine);
      x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false); // row_shr:1, 2, 4, 8
      x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);
      x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);
      x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);
      total[k] = static_cast<uint32_t>(__shfl(x, 15, kWave));
      v[k] += static_cast<uint32_t>(__shfl(x, w, kWave) - __shfl(static_cast<int>(mine), w, kWave));
   }
   __syncthreads();
}

// A call's set-up, by one workgroup of kRgBS threads, as many maps per step:
// exclusive prefix sums over the maps of the retrieve units (every map's when
// `regions` is 0) and of the regions; the maps' states; err of the maps that
// are inserted into by regions, to be set to FAIL by a region that fails.
template <typename K>
__device__ __forceinline__ void batch_prep(const BatchArgs<K>& a, int regions, BatchScratch* sc) {
   __shared__ uint32_t wsum[kRgWaves][4];
   __shared__ uint32_t any_s;
   const uint32_t n_maps = a.n_maps;
   uint64_t* us = unit_start(sc);
   uint64_t* is = item_start(sc, n_maps);
   MapState* st = map_state(sc, n_maps);
   constexpr int kLow = 22; // a step's units in two parts, whose sums stay below 2^32
   uint64_t units = 0, items = 0;
   uint32_t several = 0;
   if (threadIdx.x == 0) any_s = 0;
   for (uint64_t base = 0; base < n_maps; base += kRgBS) {
      const uint64_t m = base + threadIdx.x;
      uint64_t u = 0;
      uint32_t ways = 0, nreg = 0;
      bool group = false;
      if (m < n_maps) {
         const hn_batch_map M = a.maps[m];
         if (regions) {
            const int sp = M.info->size_power;
            ways = map_ways<K>(M, M.info, sp, a.req, n_maps);
            nreg = ways ? map_regions<K>(M, sp, a.req) : 0;
         }
         if ((a.req & HN_BATCH_RETRIEVE) && !(ways & kWayQry)) u = (M.qry_len + kBatchUnit - 1) / kBatchUnit;
         group = ((a.req & HN_BATCH_ERASE) && !(ways & kWayErs) && M.ers_len) ||
                 ((a.req & HN_BATCH_CLEAN) && !(ways & kWayClean));
         if (ways & kWayIns) {
            M.info->err = HN_STATUS_SUCCESS;
            M.info->reserved1 = 0; // inserts do not keep Robin Hood order
         }
      }
      uint32_t v[4] = {static_cast<uint32_t>(u & ((1u << kLow) - 1)), static_cast<uint32_t>(u >> kLow), nreg,
                       nreg > 1 ? 1u : 0u};
      uint32_t total[4];
      block_excl_scan<4>(v, wsum, total);
      const uint32_t any = (__ballot(ways & kWayIns) ? kAnyIns : 0u) |
                           (__ballot(ways & (kWayQry | kWayErs)) ? kAnyLook : 0u) | (__ballot(group) ? kAnyGroup : 0u);
      if (__lane_id() == 0 && any) atomicOr(&any_s, any);
      if (m < n_maps) {
         us[m] = units + v[0] + (static_cast<uint64_t>(v[1]) << kLow);
         is[m] = items + v[2];
         MapState z{};
         z.ways = ways;
         z.list = several + v[3];
         st[m] = z;
      }
      units += total[0] + (static_cast<uint64_t>(total[1]) << kLow);
      items += total[2];
      several += total[3];
   }
   __syncthreads();
   if (threadIdx.x == 0) {
      us[n_maps] = units;
      is[n_maps] = items;
      sc->units = units;
      sc->items = items;
      sc->several = several;
      sc->any = any_s;
   }
}

// The phases that do not run by regions, a workgroup per map.  With `prep` the
// call's set-up runs beside an insert phase, in workgroup 0 (both are mostly a
// few waits for memory, and a launch is another 4 us).
template <typename K>
__global__ __launch_bounds__(kRgBS) void k_batch_group(BatchArgs<K> a, BatchScratch* sc, int prep, int regions) {
   __shared__ GroupMem S;
   if (prep && blockIdx.x == 0) {
      batch_prep<K>(a, regions, sc);
      return;
   }
   if (!prep && !(sc->any & kAnyGroup)) return;
   for (uint64_t m = blockIdx.x - prep; m < a.n_maps; m += gridDim.x - prep) {
      const hn_batch_map M = a.maps[m];
      uint32_t ops;
      if (prep) {
         ops = ins_by_regions<K>(M, M.info, M.info->size_power, a.req, a.n_maps) ? 0 : a.ops;
      } else {
         const uint32_t ways = map_state(sc, a.n_maps)[m].ways;
         ops = ((ways & kWayErs) || !M.ers_len ? 0 : a.ops & HN_BATCH_ERASE) |
               ((ways & kWayClean) ? 0 : a.ops & HN_BATCH_CLEAN);
      }
      if (ops) map_phases<K, default_probe_width<K>(OP_INSERT)>(a, M, ops, S);
   }
}

template <typename K>
__global__ __launch_bounds__(kWave) void k_batch_retrieve_lane(BatchArgs<K> a, BatchScratch* sc) {
   __shared__ LaneLds<K, LK_RETRIEVE> L;
   const uint64_t units = sc->units;
   if (units == 0) return;
   const uint64_t* us = unit_start(sc);
   for (uint64_t u = blockIdx.x; u < units; u += gridDim.x) {
      // the map holding unit u: us[lo] <= u < us[hi] throughout, so map lo has units
      uint32_t lo = 0, hi = a.n_maps;
      while (hi - lo > 1) {
         const uint32_t mid = lo + (hi - lo) / 2;
         if (us[mid] <= u)
            lo = mid;
         else
            hi = mid;
      }
      const hn_batch_map M = a.maps[lo];
      const uint64_t q0 = (u - us[lo]) * kBatchUnit;
      hn_info* info = M.info;
      const int sp = info->size_power;
      if (sp >= 1 && sp <= max_size_power<K>()) {
         const uint64_t q1 = q0 + kBatchUnit < M.qry_len ? q0 + kBatchUnit : M.qry_len;
         const uint64_t ovf = info->current_max_bucket_overflow;
         const bool ordered = (info->reserved1 & kInfoOrdered) != 0;
         LookupArgs<K> la{a.qry_keys + M.qry_off, a.qry_vals + M.qry_off, nullptr,
                          a.qry_hit ? a.qry_hit + M.qry_off : nullptr, static_cast<Slot<K>*>(M.buckets), info,
                          M.qry_len, false};
         if (sp >= LaneWin<K>::kLog && ovf > 0) {
            lane_lookup<K, false, LK_RETRIEVE>(la, sp, ovf, ordered, q0, q1, L);
         } else {
            lookup_range<K, 1, false, LK_RETRIEVE>(la, sp, ovf, q1, q0 + __lane_id(), kWave, ordered);
         }
         wave_lds_sync();
      }
   }
}

// ------------------------------------------------------------ region kernels

// The map of region `item`: the last one whose first region is <= item (it
// has regions, since the next map's first is above).  A whole wave searches
// 64 ways, so a batch of thousands of maps takes two or three loads.
__device__ __forceinline__ uint64_t find_map(const uint64_t* start, uint32_t n_maps, uint64_t item) {
   const int lane = __lane_id();
   uint64_t lo = 0, hi = n_maps;
   while (hi - lo > 1) {
      const uint64_t step = (hi - lo + kWave - 1) / kWave;
      const uint64_t i = lo + static_cast<uint64_t>(lane) * step;
      const uint64_t m = __ballot(i < hi && start[i] <= item);
      const uint64_t nlo = lo + static_cast<uint64_t>(__popcll(m) - 1) * step;
      hi = nlo + step < hi ? nlo + step : hi;
      lo = nlo;
   }
   return lo;
}

// The workgroup's next region, `item` and every gridDim.x-th after it: false
// when there is none left.  The largest maps' regions come first and regions
// of a map are alike, so dealing them out in turn balances the grid; a ticket
// per region took 2,280 serial atomics per launch.
template <typename Mem>
__device__ __forceinline__ bool next_region(Mem& L, BatchScratch* sc, uint32_t n_maps, uint64_t* item, uint64_t* map,
                                            uint64_t* region) {
   const uint64_t it = *item;
   if (it >= sc->items) return false;
   *item = it + gridDim.x;
   const uint64_t* is = item_start(sc, n_maps);
   *map = find_map(is, n_maps, it);
   *region = it - is[*map];
   __syncthreads(); // the previous region's LDS is no longer read
   if (threadIdx.x == 0) {
      L.n = 0;
      L.max_probe = 0;
      L.flag = 0;
   }
   __syncthreads();
   return true;
}

// err = FAIL, whatever other workgroups do to it (SUCCESS is 0).
__device__ __forceinline__ void set_fail(hn_info* info) {
   __hip_atomic_fetch_or(&info->err, HN_STATUS_FAIL, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Insert phase on one region.  Bound by LDS probing and by the lists a region
// has to read; the table passes through LDS once each way.  While keys are
// placed a slot holds its value's index in the list, so that no probe waits
// for a value; the values come in as the region is written back.
template <typename K>
__global__ __launch_bounds__(kRgBS) void k_region_insert(BatchArgs<K> a, BatchScratch* sc) {
   __shared__ RegionMem<K> L;
   if (!(sc->any & kAnyIns)) return;
   uint64_t mi, r, item = blockIdx.x;
   while (next_region(L, sc, a.n_maps, &item, &mi, &r)) {
      MapState* const st = &map_state(sc, a.n_maps)[mi];
      if (!(st->ways & kWayIns)) continue;
      const hn_batch_map M = a.maps[mi];
      const int sp = M.info->size_power;
      const int rlog = sp < kRegionLogB<K> ? sp : kRegionLogB<K>;
      const uint32_t R = 1u << rlog, W = R < kRgWin ? R : kRgWin;
      const uint64_t nreg = 1ull << (sp - rlog);
      const SpillList spill(sc, a.n_maps, *st);
      Slot<K>* b = static_cast<Slot<K>*>(M.buckets) + (r << rlog);
      for (uint32_t i = threadIdx.x; i < R; i += kRgBS) {
         const Slot<K> s = b[i];
         L.key[i] = s.key;
         L.val[i] = s.val;
      }
      for (uint32_t i = threadIdx.x; i < (R + 31) / 32; i += kRgBS) L.from[i] = 0;
      __syncthreads();
      uint32_t placed = 0, max_probe = 0;
      bool spilled = false, failed = false;
      lds_probe<K>(
          L, KeyList<K>(a.ins_keys + M.ins_off, static_cast<uint32_t>(M.ins_len)), sp,
          [&](uint32_t, K, uint32_t home) { return (home >> rlog) == r; },
          [&](uint32_t home) { return home & (R - 1); },
          [&](K key, uint32_t idx, uint32_t& pos, uint32_t& off) -> bool {
             uint32_t at;
             const InsertStep did = lds_insert_step<K>(L, R, W, key, idx, pos, off, &at);
             if (did == STEP_PLACED) {
                ++placed;
                const uint32_t pr = off + (at - pos) + 1;
                max_probe = pr > max_probe ? pr : max_probe;
             }
             if (did != STEP_NEXT) return did != STEP_AGAIN;
             if (pos == R) {
                if (nreg > 1) { // k_boundary_insert's
                   spilled = true;
                   const uint32_t n = atomic_add_relaxed(&st->n_spill, 1u);
                   if (n < spill.cap) spill.idx[n] = idx;
                   return true;
                }
                pos = 0;
             }
             failed = failed || off >= R;
             return off >= R;
          });
      placed = wave_sum(placed);
      max_probe = wave_max(max_probe);
      const bool ws = __ballot(spilled) != 0, wf = __ballot(failed) != 0;
      if (__lane_id() == 0) {
         if (placed) atomicAdd(&L.n, static_cast<unsigned long long>(placed));
         if (max_probe) atomicMax(&L.max_probe, max_probe);
         if (ws || wf) atomicOr(&L.flag, (ws ? 1u : 0u) | (wf ? 2u : 0u));
      }
      __syncthreads();
      const K* vals = a.ins_vals + M.ins_off;
      for (uint32_t i = threadIdx.x; i < R; i += kRgBS) {
         Slot<K> s;
         s.key = L.key[i];
         s.val = L.val[i];
         if ((L.from[i >> 5] >> (i & 31)) & 1u) s.val = vals[static_cast<uint32_t>(s.val)];
         b[i] = s;
      }
      if (threadIdx.x == 0) {
         if (L.n) atomic_add_relaxed(&M.info->fill, static_cast<uint64_t>(L.n));
         if (L.max_probe)
            atomic_max_relaxed(&M.info->current_max_bucket_overflow,
                               next_overflow(L.max_probe, kBucketOverflow));
         if (L.flag & 1u) {
            __hip_atomic_fetch_or(&st->spilled, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            set_any(sc, kAnySpill);
         }
         if (L.flag & 2u) set_fail(M.info);
      }
   }
}

// One key into a table in global memory by one lane (other lanes of the
// workgroup insert into it too): insert_range's steps for a group of one,
// with its window rule.
template <typename K>
__device__ __forceinline__ void insert_one(Slot<K>* b, int sp, K key, K val, InsertCounters& c) {
   constexpr K kEmpty = empty_key<K>();
   const uint64_t n = 1ull << sp, mask = n - 1;
   const uint64_t W = n < kRgWin ? n : kRgWin;
   const uint64_t home = fib_home(key, sp) & mask;
   for (uint64_t off = 0; off < n; ++off) {
      const uint64_t p = (home + off) & mask;
      const K k = b[p].key;
      if (k == key) {
         b[p].val = val;
         return;
      }
      if (k != kEmpty) continue;
      for (uint64_t q = p + 1; q <= (p | (W - 1)); ++q) {
         if (b[q].key == key) {
            b[q].val = val;
            return;
         }
      }
      const K old = atomic_cas(&b[p].key, kEmpty, key);
      if (old == kEmpty || old == key) {
         b[p].val = val;
         if (old == kEmpty) {
            ++c.placed;
            c.max_probe = off + 1 > c.max_probe ? off + 1 : c.max_probe;
         }
         return;
      }
   }
   c.failed = 1;
}

// The keys that probe past the end of region r, tried in LDS over the kRgHalf
// slots before the end and as many after it (the halves of neighbouring
// regions do not meet).
//
// After k_region_insert (maps of several regions where a key did): the keys
// that k_region_insert listed or, when it met more than the list holds, all
// keys of the map that may be among them: such a key has every slot from its
// home to the region's end occupied, so its home lies in the region's last
// run of occupied slots.  After k_region_clean (CLEAN): the map's listed keys with a home
// in the region.  A home further than kRgHalf before the end, or a key that
// finds no slot in the window, is left to the per-map kernel that follows.
constexpr uint32_t kRgHalf = 1024;
template <typename K, bool CLEAN>
__global__ __launch_bounds__(kRgBS) void k_boundary_insert(BatchArgs<K> a, BatchScratch* sc) {
   __shared__ RegionMem<K> L;
   constexpr K kEmpty = empty_key<K>();
   constexpr uint32_t kSpan = 2 * kRgHalf;
   static_assert(kSpan <= RegionMem<K>::kSlots, "the window fits a region's arrays; windows are disjoint");
   if (!(sc->any & (CLEAN ? kAnyListed : kAnySpill))) return;
   uint64_t mi, r, item = blockIdx.x;
   while (next_region(L, sc, a.n_maps, &item, &mi, &r)) {
      MapState* const st = &map_state(sc, a.n_maps)[mi];
      const hn_batch_map M = a.maps[mi];
      const int sp = M.info->size_power;
      if (CLEAN ? (st->listed == 0 || sp <= kRegionLogB<K>) : st->spilled == 0) continue;
      const uint32_t mask = slot_mask32(sp);
      Slot<K>* const b = static_cast<Slot<K>*>(M.buckets);
      const uint32_t end = static_cast<uint32_t>((r + 1) << kRegionLogB<K>);
      const uint32_t lo = end - kRgHalf; // slots [lo, lo + kSpan), taken mod 2^sp
      uint32_t last = 0;                 // 1 + the last EMPTY slot of the first half
      for (uint32_t i = threadIdx.x; i < kSpan; i += kRgBS) {
         const Slot<K> s = b[(lo + i) & mask];
         L.key[i] = s.key;
         L.val[i] = s.val;
         if (i < kRgHalf && s.key == kEmpty) last = i + 1;
      }
      for (uint32_t i = threadIdx.x; i < kSpan / 32; i += kRgBS) L.from[i] = 0;
      last = wave_max(last);
      if (__lane_id() == 0 && last) atomicMax(&L.max_probe, last);
      __syncthreads();
      uint32_t tail = L.max_probe; // the run starts at window slot `tail`
      __syncthreads();
      if (threadIdx.x == 0) L.max_probe = 0;
      if (CLEAN) {
         tail = 0;
      } else {
         if (tail == kRgHalf) continue; // the region's last slot is EMPTY
         if (tail == 0) {               // the run may reach back further
            if (threadIdx.x == 0) {
               __hip_atomic_fetch_or(&st->spilled, 2u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
               set_any(sc, kAnyLeft);
            }
            continue;
         }
      }
      __syncthreads();
      uint32_t placed = 0, max_probe = 0;
      bool left = false;
      auto put = [&](uint32_t at, uint32_t idx) {
         L.val[at] = static_cast<K>(idx);
         atomicOr(&L.from[at >> 5], 1u << (at & 31));
      };
      auto take = [&](uint32_t, K, uint32_t home) {
         if (CLEAN && home >> kRegionLogB<K> == r && home < lo) left = true;
         return home - lo >= tail && home - lo < kRgHalf;
      };
      auto step = [&](K key, uint32_t idx, uint32_t& pos, uint32_t& off) -> bool {
         uint32_t mm, em;
         window_bits<K>(L.key, pos, kRgWin, key, &mm, &em);
         const uint32_t w = pos & ~3u;
         if (mm) { // (clean: a second copy of the key, dropped)
            if (!CLEAN && pos >= kRgHalf) put(w + __ffs(mm) - 1, idx); // one before its region's end was set there
            return true;
         }
         if (em) {
            const uint32_t at = w + __ffs(em) - 1;
            const K old = lds_cas(&L.key[at], kEmpty, key);
            if (old != kEmpty && old != key) return false;
            put(at, idx);
            if (old == kEmpty) {
               ++placed;
               const uint32_t pr = off + (at - pos) + 1;
               max_probe = pr > max_probe ? pr : max_probe;
            }
            return true;
         }
         const uint32_t next = w + kRgWin;
         off += next - pos;
         pos = next;
         if (pos == kSpan) {
            left = true;
            return true;
         }
         return false;
      };
      auto place = [&](uint32_t home) { return home - lo; };
      const Slot<K>* const list = CLEAN ? a.clean_scratch + M.scratch_off : nullptr;
      const SpillList spill(sc, a.n_maps, *st);
      if constexpr (CLEAN)
         lds_probe<K>(L, SlotKeys<K>{list, st->listed}, sp, take, place, step);
      else if (st->n_spill <= spill.cap)
         lds_probe<K>(L, PickedKeys<K>{a.ins_keys + M.ins_off, spill.idx, st->n_spill}, sp, take, place, step);
      else
         lds_probe<K>(L, KeyList<K>(a.ins_keys + M.ins_off, static_cast<uint32_t>(M.ins_len)), sp, take, place, step);
      placed = wave_sum(placed);
      max_probe = wave_max(max_probe);
      const bool wl = __ballot(left) != 0;
      if (__lane_id() == 0) {
         if (placed) atomicAdd(&L.n, static_cast<unsigned long long>(placed));
         if (max_probe) atomicMax(&L.max_probe, max_probe);
         if (wl) L.flag = 1;
      }
      __syncthreads();
      for (uint32_t i = threadIdx.x; i < kSpan; i += kRgBS) {
         if (!((L.from[i >> 5] >> (i & 31)) & 1u)) continue;
         const uint32_t at = static_cast<uint32_t>(L.val[i]);
         Slot<K> s;
         s.key = L.key[i];
         s.val = CLEAN ? list[at].val : a.ins_vals[M.ins_off + at];
         b[(lo + i) & mask] = s;
      }
      if (threadIdx.x == 0) {
         if (L.flag) {
            __hip_atomic_fetch_or(&st->spilled, 2u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            set_any(sc, kAnyLeft);
         }
         if constexpr (CLEAN) {
            if (L.n) atomic_add_relaxed(&st->placed, static_cast<uint32_t>(L.n));
            if (L.max_probe) atomic_max_relaxed(&st->max_probe, L.max_probe);
         } else {
            if (L.n) atomic_add_relaxed(&M.info->fill, static_cast<uint64_t>(L.n));
            if (L.max_probe)
               atomic_max_relaxed(&M.info->current_max_bucket_overflow, next_overflow(L.max_probe, kBucketOverflow));
         }
      }
   }
}

// After k_region_insert and k_boundary_insert, a workgroup per map: the keys
// that k_boundary_insert left (every key with a home in a region's last run of
// occupied slots is tried in global memory).
template <typename K>
__global__ __launch_bounds__(kRgBS) void k_map_insert_end(BatchArgs<K> a, BatchScratch* sc) {
   __shared__ uint64_t tail[kMaxRegions]; // first slot of each region's last run of occupied slots
   if (!(sc->any & kAnyLeft)) return;
   for (uint32_t m = blockIdx.x; m < a.n_maps; m += gridDim.x) {
      MapState* const st = &map_state(sc, a.n_maps)[m];
      if (!(st->spilled & 2u)) continue;
      const hn_batch_map M = a.maps[m];
      const int sp = M.info->size_power, rlog = kRegionLogB<K>; // only maps of several regions spill
      const uint32_t nreg = 1u << (sp - rlog);
      const uint64_t R = 1ull << rlog;
      Slot<K>* b = static_cast<Slot<K>*>(M.buckets);
      const int lane = __lane_id();
      for (uint32_t r = threadIdx.x / kWave; r < nreg; r += kRgWaves) {
         const uint64_t base = static_cast<uint64_t>(r) << rlog;
         uint64_t first = base;
         for (uint64_t o = R; o > 0; o -= kWave) {
            const uint64_t e = __ballot(b[base + o - kWave + lane].key == empty_key<K>());
            if (e) {
               first = base + o - __clzll(static_cast<long long>(e));
               break;
            }
         }
         if (lane == 0) tail[r] = first;
      }
      __syncthreads();
      InsertCounters c;
      for (uint64_t i = threadIdx.x; i < M.ins_len; i += kRgBS) {
         const K key = a.ins_keys[M.ins_off + i];
         const uint64_t home = home_slot(key, sp);
         if (home >= tail[home >> rlog]) insert_one<K>(b, sp, key, a.ins_vals[M.ins_off + i], c);
      }
      const uint64_t placed = wave_sum(c.placed), max_probe = wave_max(c.max_probe);
      if (lane == 0) {
         if (placed) atomic_add_relaxed(&M.info->fill, placed);
         if (max_probe) atomic_max_relaxed(&M.info->current_max_bucket_overflow, next_overflow(max_probe, kBucketOverflow));
      }
      if (__ballot(c.failed) && lane == 0) set_fail(M.info);
      __syncthreads(); // tail is rewritten for the next map; the state has been read
      if (threadIdx.x == 0) st->spilled = 0; // the clean's from here
   }
}

// Lookups on a region go through an index of it: its keys sorted by home slot
// (a counting sort in LDS), so a query compares the keys of its own home slot
// alone, however long the cluster it falls into.  kOver slots after the
// region's end are held too, for the keys that probed past it.
template <typename K>
struct IndexMem {
   static constexpr uint32_t kSlots = 1u << kRegionLogB<K>;
   static constexpr uint32_t kOver = sizeof(K) == 4 ? 512 : 1024; // what the LDS of half a CU leaves
   static constexpr uint32_t kHeld = kSlots + kOver;
   K key[kHeld];                // by home slot
   uint16_t slot[kHeld];        // and the held slot of each
   uint32_t start[kSlots / 2 + 1]; // first key of each home slot, two 16-bit entries a word
   uint32_t empty[kHeld / 32];  // EMPTY slots, one bit each
   K qkey[kRgWaves][kRgQueue];
   uint32_t qidx[kRgWaves][kRgQueue];
   uint32_t wsum[kRgWaves];
   unsigned long long n;
   uint32_t max_probe, flag; // flag: held slots from there on hold no EMPTY one
};

// fn(i, key) for the keys of list[0, len) whose home lies in region r, a full
// wave of them at a time while there are that many; lanes without one call
// with on = false.  Every lane of the workgroup calls.
template <typename K, typename Fn>
__device__ __forceinline__ void region_keys(IndexMem<K>& L, const KeyList<K> src, int sp, int rlog, uint64_t nreg,
                                            uint32_t r, Fn fn) {
   const uint32_t lane = __lane_id();
   const int wave = threadIdx.x / kWave;
   const uint32_t len = src.entries();
   K* const qk = L.qkey[wave];
   uint32_t* const qi = L.qidx[wave];
   uint32_t have = 0;
   K k0[4], k1[4];
   auto load = [&](uint32_t at, K k[4]) {
      if (at < len) src.load(at + 4 * lane, k);
   };
   uint32_t b = static_cast<uint32_t>(wave) * 4 * kWave;
   load(b, k0), load(b + 4 * kRgBS, k1);
   for (; b < len; b += 4 * kRgBS) {
      K k[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) k[j] = k0[j], k0[j] = k1[j];
      load(b + 8 * kRgBS, k1);
#pragma unroll 1
      for (int j = 0; j < 4; ++j) {
         const uint32_t e = b + 4 * lane + j;
         K key = k[0];
         k[0] = k[1], k[1] = k[2], k[2] = k[3];
         uint32_t idx = src.index(e);
         bool on = src.valid(e);
         if (nreg > 1) {
            const bool in = on && (home_slot(key, sp) >> rlog) == r;
            const uint64_t m = __ballot(in);
            const uint32_t at = have + __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(m >> 32),
                                                                 __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(m), 0));
            if (in) {
               qk[at] = key;
               qi[at] = idx;
            }
            have += static_cast<uint32_t>(__popcll(m));
            if (have < static_cast<uint32_t>(kWave)) continue;
            wave_lds_sync(); // the first 64 out, the rest to the front
            key = qk[lane];
            idx = qi[lane];
            const K mk = qk[kWave + lane];
            const uint32_t mi = qi[kWave + lane];
            wave_lds_sync();
            have -= kWave;
            if (lane < have) {
               qk[lane] = mk;
               qi[lane] = mi;
            }
            on = true;
         }
         fn(on, idx, key);
      }
   }
   if (have) {
      wave_lds_sync();
      const bool on = lane < have;
      fn(on, on ? qi[lane] : 0, on ? qk[lane] : K(0));
   }
}

// Retrieve and erase on one region.  A query's key is the one that the plain
// probe finds: within the bound, and with no EMPTY slot between its home and
// its slot (a table with holes left by reset_to_empty may hold keys behind
// one).  A probe that runs past the held slots goes on in global memory, slot
// by slot.  A TOMBSTONE is stored to global memory slot by slot, never by
// writing the region back, so another region's probe into these slots sees a
// key or its TOMBSTONE, neither of which ends it; the keys of a region are
// retrieved and erased by its workgroup alone, in that order.
template <typename K>
__global__ __launch_bounds__(kRgBS) __attribute__((amdgpu_waves_per_eu(4))) void k_region_lookup(BatchArgs<K> a, BatchScratch* sc) {
   __shared__ IndexMem<K> L;
   constexpr K kEmpty = empty_key<K>();
   constexpr K kTomb = tomb_key<K>();
   constexpr int E = static_cast<int>((IndexMem<K>::kHeld + kRgBS - 1) / kRgBS); // held slots per thread
   const int lane = __lane_id(), wave = threadIdx.x / kWave;
   if (!(sc->any & kAnyLook)) return;
   uint64_t mi, r64, item = blockIdx.x;
   while (next_region(L, sc, a.n_maps, &item, &mi, &r64)) {
      const uint32_t ways = map_state(sc, a.n_maps)[mi].ways;
      if (!(ways & (kWayQry | kWayErs))) continue;
      const hn_batch_map M = a.maps[mi];
      const int sp = M.info->size_power;
      const uint32_t nq = (ways & kWayQry) ? static_cast<uint32_t>(M.qry_len) : 0;
      const uint32_t ne = (ways & kWayErs) ? static_cast<uint32_t>(M.ers_len) : 0;
      const int rlog = sp < kRegionLogB<K> ? sp : kRegionLogB<K>;
      const uint32_t r = static_cast<uint32_t>(r64), R = 1u << rlog, mask = slot_mask32(sp), first = r << rlog;
      const uint64_t nreg = 1ull << (sp - rlog);
      const uint64_t ovf = M.info->current_max_bucket_overflow, nsl = static_cast<uint64_t>(mask) + 1;
      const uint32_t bound = static_cast<uint32_t>(ovf < nsl ? ovf : nsl);
      const uint32_t held = nreg > 1 ? IndexMem<K>::kHeld : R;
      Slot<K>* const all = static_cast<Slot<K>*>(M.buckets);

      // the index
      const uint32_t words = R / 2 + 1; // of start
      for (uint32_t i = threadIdx.x; i < words; i += kRgBS) L.start[i] = 0;
      K key[E];
      uint32_t hs[E]; // home slot in the region << 16 | rank among its keys by arrival
      uint32_t clear_of = 0;
#pragma unroll
      for (int e = 0; e < E; ++e) {
         const uint32_t i = threadIdx.x + e * kRgBS;
         key[e] = kTomb;
         if (i < held) key[e] = all[(first + i) & mask].key;
      }
      __syncthreads();
#pragma unroll
      for (int e = 0; e < E; ++e) {
         const uint32_t i = threadIdx.x + e * kRgBS;
         hs[e] = 0xFFFFFFFFu;
         const uint64_t em = __ballot(key[e] == kEmpty);
         if (i < held) {
            if ((lane & 31) == 0) L.empty[i >> 5] = static_cast<uint32_t>(em >> (lane & 32));
            if (key[e] == kEmpty) clear_of = i + 1;
            if (key[e] != kEmpty && key[e] != kTomb) {
               const uint32_t home = home_slot(key[e], sp);
               if (home >> rlog == r) {
                  const uint32_t h = home & (R - 1), sh = (h & 1) * 16;
                  hs[e] = h << 16 | ((atomicAdd(&L.start[h >> 1], 1u << sh) >> sh) & 0xFFFFu);
               }
            }
         }
      }
      clear_of = wave_max(clear_of);
      if (lane == 0 && clear_of) atomicMax(&L.flag, clear_of);
      __syncthreads();
      { // exclusive scan of the 16-bit counts
         const uint32_t per = (words + kRgBS - 1) / kRgBS;
         const uint32_t c0 = std::min<uint32_t>(threadIdx.x * per, words), c1 = std::min<uint32_t>(c0 + per, words);
         uint32_t acc = 0;
         for (uint32_t i = c0; i < c1; ++i) acc += (L.start[i] & 0xFFFFu) + (L.start[i] >> 16);
         uint32_t inc = acc;
#pragma unroll
         for (int o = 1; o < kWave; o <<= 1) {
            const uint32_t y = __shfl_up(inc, o, kWave);
            if (lane >= o) inc += y;
         }
         if (lane == kWave - 1) L.wsum[wave] = inc;
         __syncthreads();
         uint32_t run = inc - acc;
         for (int w = 0; w < wave; ++w) run += L.wsum[w];
         for (uint32_t i = c0; i < c1; ++i) {
            const uint32_t c = L.start[i];
            L.start[i] = run | (run + (c & 0xFFFFu)) << 16;
            run += (c & 0xFFFFu) + (c >> 16);
         }
      }
      __syncthreads();
      auto start_of = [&](uint32_t h) { return (L.start[h >> 1] >> ((h & 1) * 16)) & 0xFFFFu; };
#pragma unroll
      for (int e = 0; e < E; ++e) {
         if (hs[e] != 0xFFFFFFFFu) {
            const uint32_t j = start_of(hs[e] >> 16) + (hs[e] & 0xFFFFu);
            L.key[j] = key[e];
            L.slot[j] = static_cast<uint16_t>(threadIdx.x + e * kRgBS);
         }
      }
      const uint32_t run_from = L.flag; // held slots from here on are occupied
      __syncthreads();

      // EMPTY slots in [h, s) of the held slots?
      auto gap = [&](uint32_t h, uint32_t s) {
         uint32_t any = 0;
         for (uint32_t w = h >> 5; w <= s >> 5 && h < s; ++w) {
            uint32_t v = L.empty[w];
            if (w == h >> 5) v &= ~0u << (h & 31);
            if (w == s >> 5) v &= (1u << (s & 31)) - 1u;
            any |= v;
            if (any) break;
         }
         return any != 0;
      };
      // Where a lookup of key finds it: its place in the index (below kHeld),
      // kHeld + its table slot, or kNone.
      constexpr uint32_t kNone = 0xFFFFFFFFu;
      auto walk = [&](K key, uint32_t off) -> uint32_t { // the probe in global memory from offset off on
         const uint32_t home = home_slot(key, sp);
         for (; off < bound; ++off) {
            const uint32_t p = (home + off) & mask;
            const K k = all[p].key;
            if (k == kEmpty) return kNone;
            if (k == key) return IndexMem<K>::kHeld + p;
         }
         return kNone;
      };
      auto find = [&](K key) -> uint32_t {
         if (key == kTomb) return walk(key, 0); // TOMBSTONEs are not in the index
         const uint32_t h = home_slot(key, sp) & (R - 1);
         uint32_t at = kNone, off = bound; // the nearest copy within the bound
         for (uint32_t j = start_of(h), j1 = start_of(h + 1); j < j1; ++j) {
            if (L.key[j] == key) {
               const uint32_t s = L.slot[j];
               // A slot before h: round the table's end in a one-region map; a key that went
               // round a larger one is left to the walk.
               const uint32_t o = s >= h ? s - h : nreg > 1 ? bound : s + R - h;
               if (o < off) {
                  off = o;
                  at = j;
               }
            }
         }
         if (at != kNone) {
            const uint32_t s = h + off;
            const bool g = s < R || nreg > 1 ? gap(h, s) : gap(h, R) || gap(0, s - R);
            return g ? kNone : at;
         }
         // not held: the probe leaves the held slots if none from home on is EMPTY
         if (nreg > 1 && h >= run_from) return walk(key, held - h);
         return kNone;
      };
      auto slot_of = [&](uint32_t at) -> uint32_t {
         return at < IndexMem<K>::kHeld ? (first + L.slot[at]) & mask : at - IndexMem<K>::kHeld;
      };
      if (nq) {
         K* const qv = a.qry_vals + M.qry_off;
         uint8_t* const qh = a.qry_hit ? a.qry_hit + M.qry_off : nullptr;
         region_keys<K>(L, KeyList<K>(a.qry_keys + M.qry_off, nq), sp, rlog, nreg, r,
                        [&](bool on, uint32_t idx, K k) {
                           if (!on) return;
                           const uint32_t at = find(k);
                           if (at != kNone) qv[idx] = all[slot_of(at)].val;
                           if (qh) qh[idx] = at != kNone ? 1 : 0;
                        });
      }
      if (ne) {
         if (nq) __syncthreads();
         uint32_t erased = 0;
         region_keys<K>(L, KeyList<K>(a.ers_keys + M.ers_off, ne), sp, rlog, nreg, r,
                        [&](bool on, uint32_t, K k) {
                           if (!on) return;
                           const uint32_t at = find(k);
                           if (at == kNone) return;
                           if (at >= IndexMem<K>::kHeld) {
                              if (atomic_cas(&all[slot_of(at)].key, k, kTomb) == k) ++erased;
                           } else if (lds_cas(&L.key[at], k, kTomb) == k) {
                              ++erased;
                              all[slot_of(at)].key = kTomb;
                           }
                        });
         erased = wave_sum(erased);
         if (lane == 0 && erased) atomicAdd(&L.n, static_cast<unsigned long long>(erased));
         __syncthreads();
         if (threadIdx.x == 0 && L.n) {
            atomic_add_relaxed(&M.info->tombstone_counter, static_cast<uint64_t>(L.n));
            __hip_atomic_fetch_sub(&M.info->fill, static_cast<uint64_t>(L.n), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
         }
      }
   }
}

// A cleaned map's Info, by one thread.
__device__ __forceinline__ void clean_info(hn_info* info, uint64_t placed, uint32_t max_probe, bool displaced,
                                           bool failed) {
   const uint64_t o = next_overflow(max_probe, kBucketOverflow);
   info->fill = placed;
   info->tombstone_counter = 0;
   info->current_max_bucket_overflow = o > kBucketOverflow ? o : kBucketOverflow;
   info->reserved1 = 0; // the keys are not placed in Robin Hood order
   if (displaced) info->err = failed ? HN_STATUS_FAIL : HN_STATUS_SUCCESS;
}

// Clean on one region: the live keys standing in it whose home lies in it are
// placed again in an LDS image that starts empty (read from the table, which
// does not change meanwhile), then the image is written over the region.  Of a
// key that stands there twice (inserted before an EMPTY slot that
// reset_to_empty has left on the way to its old copy) one copy is placed, as
// when the lifted keys are inserted again, so the keys placed are counted.
// Keys of other regions standing here, and keys that run past the region's
// end, go to the map's scratch slice (at most its live keys), from which
// k_boundary_insert and k_map_clean_end place them.  The Info of a map of
// several regions is not changed here.
template <typename K>
__global__ __launch_bounds__(kRgBS) void k_region_clean(BatchArgs<K> a, BatchScratch* sc) {
   __shared__ RegionMem<K> L;
   constexpr K kEmpty = empty_key<K>();
   constexpr int E = static_cast<int>(RegionMem<K>::kSlots / kRgBS); // slots per thread
   uint64_t mi, r, item = blockIdx.x;
   while (next_region(L, sc, a.n_maps, &item, &mi, &r)) {
      const hn_batch_map M = a.maps[mi];
      if (M.info->tombstone_counter == 0) continue;
      const int sp = M.info->size_power;
      if (M.info->fill > M.scratch_cap) { // not enough scratch: the map is left as it is
         if (sp <= kRegionLogB<K> && threadIdx.x == 0) M.info->err = HN_STATUS_FAIL;
         continue;
      }
      const int rlog = sp < kRegionLogB<K> ? sp : kRegionLogB<K>;
      const uint32_t R = 1u << rlog, W = R < kRgWin ? R : kRgWin, first = static_cast<uint32_t>(r << rlog);
      const uint64_t nreg = 1ull << (sp - rlog);
      Slot<K>* const b = static_cast<Slot<K>*>(M.buckets) + first;
      Slot<K>* const list = a.clean_scratch + M.scratch_off;
      MapState* const st = &map_state(sc, a.n_maps)[mi];
      for (uint32_t i = threadIdx.x; i < R; i += kRgBS) L.key[i] = kEmpty;
      __syncthreads();
      uint32_t max_probe = 0, placed = 0;
      bool displaced = false;
      lds_probe<K>(
          L, SlotKeys<K>{b, R}, sp,
          [&](uint32_t i, K key, uint32_t home) {
             if (key == kEmpty || key == tomb_key<K>()) return false;
             displaced = displaced || home != first + i;
             const bool own = (home >> rlog) == r;
             if (!own) list[atomic_add_relaxed(&st->listed, 1u)] = b[i];
             return own;
          },
          [&](uint32_t home) { return home & (R - 1); },
          [&](K key, uint32_t idx, uint32_t& pos, uint32_t& off) -> bool {
             uint32_t mm, em;
             window_bits<K>(L.key, pos, W, key, &mm, &em);
             const uint32_t w = pos & ~3u;
             if (mm) return true;
             if (em) {
                const uint32_t at = w + __ffs(em) - 1;
                if (lds_cas(&L.key[at], kEmpty, key) != kEmpty) return false; // look again
                L.val[at] = static_cast<K>(idx);
                const uint32_t pr = off + (at - pos) + 1;
                max_probe = pr > max_probe ? pr : max_probe;
                return true;
             }
             const uint32_t next = (pos & ~(W - 1)) + W;
             off += next - pos;
             pos = next;
             if (pos == R) {
                if (nreg > 1) {
                   list[atomic_add_relaxed(&st->listed, 1u)] = b[idx];
                   return true;
                }
                pos = 0;
             }
             return false; // the region's keys fit: they came from its slots
          });
      max_probe = wave_max(max_probe);
      const bool wd = __ballot(displaced) != 0;
      if (__lane_id() == 0) {
         if (max_probe) atomicMax(&L.max_probe, max_probe);
         if (wd) L.flag = 1;
      }
      __syncthreads();
      Slot<K> s[E];
#pragma unroll
      for (int e = 0; e < E; ++e) {
         const uint32_t i = threadIdx.x + e * kRgBS;
         s[e].key = kEmpty;
         s[e].val = 0;
         if (i < R) {
            s[e].key = L.key[i];
            if (s[e].key != kEmpty) s[e].val = b[static_cast<uint32_t>(L.val[i])].val;
            placed += s[e].key != kEmpty;
         }
      }
      placed = wave_sum(placed);
      if (__lane_id() == 0) atomicAdd(&L.n, static_cast<unsigned long long>(placed));
      __syncthreads(); // every value is read before the region is written
#pragma unroll
      for (int e = 0; e < E; ++e) {
         const uint32_t i = threadIdx.x + e * kRgBS;
         if (i < R) b[i] = s[e];
      }
      if (threadIdx.x == 0) {
         if (nreg == 1) {
            clean_info(M.info, L.n, L.max_probe, L.flag != 0, false);
         } else {
            if (L.n) atomic_add_relaxed(&st->placed, static_cast<uint32_t>(L.n));
            if (L.max_probe) atomic_max_relaxed(&st->max_probe, L.max_probe);
            if (L.flag) __hip_atomic_store(&st->displaced, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            // some key of the map has been listed by now, by this region or another
            if (__hip_atomic_load(&st->listed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) set_any(sc, kAnyListed);
         }
      }
   }
}

// After k_region_clean and k_boundary_insert, a workgroup per map of several
// regions: the listed keys, if some were left (those already placed find themselves),
// then the Info.
template <typename K>
__global__ __launch_bounds__(kRgBS) void k_map_clean_end(BatchArgs<K> a, BatchScratch* sc) {
   __shared__ uint32_t s_max, s_failed, s_placed;
   if (sc->several == 0) return;
   for (uint32_t m = blockIdx.x; m < a.n_maps; m += gridDim.x) {
      const hn_batch_map M = a.maps[m];
      hn_info* info = M.info;
      const int sp = info->size_power;
      const MapState st = map_state(sc, a.n_maps)[m];
      if (sp <= kRegionLogB<K> || !(st.ways & kWayClean) || info->tombstone_counter == 0) continue;
      if (info->fill > M.scratch_cap) { // not enough scratch: the map is left as it is
         if (threadIdx.x == 0) info->err = HN_STATUS_FAIL;
         continue;
      }
      if (threadIdx.x == 0) {
         s_max = st.max_probe;
         s_failed = 0;
         s_placed = st.placed;
      }
      __syncthreads();
      InsertCounters c;
      const Slot<K>* list = a.clean_scratch + M.scratch_off;
      for (uint32_t i = threadIdx.x; (st.spilled & 2u) && i < st.listed; i += kRgBS)
         insert_one<K>(static_cast<Slot<K>*>(M.buckets), sp, list[i].key, list[i].val, c);
      if (c.max_probe) atomicMax(&s_max, static_cast<uint32_t>(c.max_probe));
      if (c.failed) atomicOr(&s_failed, 1u);
      if (c.placed) atomicAdd(&s_placed, static_cast<uint32_t>(c.placed));
      __syncthreads();
      if (threadIdx.x == 0) clean_info(info, s_placed, s_max, st.displaced != 0, s_failed != 0);
      __syncthreads(); // s_max is rewritten for the next map
   }
}

// Fresh tables and Info(sp) for every map of a batch, one launch.
template <typename K>
__global__ __launch_bounds__(256) void k_batch_init(const hn_batch_map* maps, uint32_t n_maps, const int32_t* sps) {
   for (uint32_t m = blockIdx.x; m < n_maps; m += gridDim.x) {
      const hn_batch_map M = maps[m];
      const int sp = sps[m];
      Slot<K>* b = static_cast<Slot<K>*>(M.buckets);
      const uint64_t n = 1ull << sp;
      for (uint64_t i = threadIdx.x; i < n; i += blockDim.x) {
         Slot<K> s;
         s.key = empty_key<K>();
         s.val = 0;
         b[i] = s;
      }
      if (threadIdx.x == 0) {
         M.info->size_power = sp;
         M.info->reserved0 = 0;
         M.info->fill = 0;
         M.info->current_max_bucket_overflow = kBucketOverflow;
         M.info->tombstone_counter = 0;
         M.info->err = HN_STATUS_INVALID;
         M.info->reserved1 = 0;
      }
   }
}

template <typename K>
using BatchKernel = void (*)(BatchArgs<K>);

template <typename K>
BatchKernel<K> pick_batch(int G) {
   switch (G) {
   case 1: return k_batch<K, 1>;
   case 2: return k_batch<K, 2>;
   case 4: return k_batch<K, 4>;
   case 8: return k_batch<K, 8>;
   case 16: return k_batch<K, 16>;
   case 32: return k_batch<K, 32>;
   case 64: return k_batch<K, 64>;
   default: return nullptr;
   }
}

template <typename K>
int batch_run(const hn_batch_map* maps, uint32_t n_maps, uint32_t ops, const K* ik, const K* iv, const K* qk, K* qv,
              uint8_t* qh, const K* ek, void* clean_scratch, void* scratch, hipStream_t s, const hn_tune* t) {
   if (!maps || !scratch) return HN_EINVAL;
   if ((ops & HN_BATCH_INSERT) && (!ik || !iv)) return HN_EINVAL;
   if ((ops & HN_BATCH_RETRIEVE) && (!qk || !qv)) return HN_EINVAL;
   if ((ops & HN_BATCH_ERASE) && !ek) return HN_EINVAL;
   if ((ops & HN_BATCH_CLEAN) && !clean_scratch) return HN_EINVAL;
   if (n_maps == 0) return 0;
   const int G = (t && t->probe_width) ? t->probe_width : default_probe_width<K>(OP_INSERT);
   const int bs = (t && t->block_size) ? t->block_size : kRgBS;
   if (G < 1 || G > 64 || (G & (G - 1)) || bs < 64 || bs > 1024 || (bs % 64)) return HN_EINVAL;
   uint32_t blocks = (t && t->grid_blocks > 0) ? static_cast<uint32_t>(t->grid_blocks)
                                               : static_cast<uint32_t>(cu_count()) * (2048 / bs);
   if (blocks > n_maps) blocks = n_maps;
   BatchScratch* sc = static_cast<BatchScratch*>(scratch);
   BatchArgs<K> a{maps, n_maps, ops, ik, iv, qk, qv, qh, ek, static_cast<Slot<K>*>(clean_scratch), &sc->ticket, ops};
   auto retrieve_units = [&]() {
      static std::atomic<int> occ{0};
      const int per_cu = resident_blocks_per_cu(k_batch_retrieve_lane<K>, kWave, occ);
      hipLaunchKernelGGL(k_batch_retrieve_lane<K>, dim3(static_cast<uint32_t>(cu_count()) * per_cu), dim3(kWave), 0, s,
                         a, sc);
   };
   const uint32_t late = ops & (HN_BATCH_ERASE | HN_BATCH_CLEAN);
   if (t && (t->probe_width || t->block_size || t->grid_blocks)) {
      // Launch tuning asks for the one-workgroup-per-map kernel at that shape.
      BatchKernel<K> k = pick_batch<K>(G);
      auto group = [&](uint32_t phases) {
         a.ops = phases;
         hipLaunchKernelGGL(k_zero_u64, dim3(1), dim3(1), 0, s, &sc->ticket);
         hipLaunchKernelGGL(k, dim3(blocks), dim3(bs), 0, s, a);
      };
      if (ops & HN_BATCH_INSERT) group(HN_BATCH_INSERT);
      if (ops & HN_BATCH_RETRIEVE) {
         a.ops = 0;
         hipLaunchKernelGGL(k_batch_group<K>, dim3(1), dim3(kRgBS), 0, s, a, sc, 1, 0);
         retrieve_units();
      }
      if (late) group(late);
      return static_cast<int>(hipGetLastError());
   }
   const dim3 rg(static_cast<uint32_t>(cu_count()) * 2); // two regions' LDS per CU
   const dim3 per_map(std::min<uint32_t>(n_maps, rg.x)), bd(kRgBS);
   const uint32_t groups = std::min<uint32_t>(n_maps, 65535);
   // The set-up, and beside it the inserts that do not run by regions.
   a.ops = ops & HN_BATCH_INSERT;
   hipLaunchKernelGGL(k_batch_group<K>, dim3(1 + (a.ops ? groups : 0)), bd, 0, s, a, sc, 1, 1);
   if (ops & HN_BATCH_INSERT) {
      hipLaunchKernelGGL(k_region_insert<K>, rg, bd, 0, s, a, sc);
      hipLaunchKernelGGL((k_boundary_insert<K, false>), rg, bd, 0, s, a, sc);
      hipLaunchKernelGGL(k_map_insert_end<K>, per_map, bd, 0, s, a, sc);
   }
   if (ops & HN_BATCH_RETRIEVE) retrieve_units();
   if (ops & (HN_BATCH_RETRIEVE | HN_BATCH_ERASE)) hipLaunchKernelGGL(k_region_lookup<K>, rg, bd, 0, s, a, sc);
   if (late) {
      a.ops = late;
      hipLaunchKernelGGL(k_batch_group<K>, dim3(groups), bd, 0, s, a, sc, 0, 1);
   }
   if (ops & HN_BATCH_CLEAN) {
      hipLaunchKernelGGL(k_region_clean<K>, rg, bd, 0, s, a, sc);
      hipLaunchKernelGGL((k_boundary_insert<K, true>), rg, bd, 0, s, a, sc);
      hipLaunchKernelGGL(k_map_clean_end<K>, per_map, bd, 0, s, a, sc);
   }
   return static_cast<int>(hipGetLastError());
}

template <typename K>
int batch_init(const hn_batch_map* maps, uint32_t n_maps, const int32_t* sps, hipStream_t s) {
   if (!maps || !sps) return HN_EINVAL;
   if (n_maps == 0) return 0;
   const uint32_t blocks = n_maps < 65535u ? n_maps : 65535u;
   hipLaunchKernelGGL(k_batch_init<K>, dim3(blocks), dim3(256), 0, s, maps, n_maps, sps);
   return static_cast<int>(hipGetLastError());
}

} // namespace hn

using namespace hn;

extern "C" {

size_t hn_batch_scratch_bytes(uint32_t n_maps) { return batch_scratch_bytes(n_maps); }

int hn_batch_init_u32(const hn_batch_map* maps, uint32_t n, const int32_t* sps, hn_stream_t s) {
   return batch_init<uint32_t>(maps, n, sps, s);
}
int hn_batch_init_u64(const hn_batch_map* maps, uint32_t n, const int32_t* sps, hn_stream_t s) {
   return batch_init<uint64_t>(maps, n, sps, s);
}
int hn_batch_run_u32(const hn_batch_map* maps, uint32_t n, uint32_t ops, const uint32_t* ik, const uint32_t* iv,
                     const uint32_t* qk, uint32_t* qv, uint8_t* qh, const uint32_t* ek, void* cs, void* sc,
                     hn_stream_t s, const hn_tune* t) {
   return batch_run<uint32_t>(maps, n, ops, ik, iv, qk, qv, qh, ek, cs, sc, s, t);
}
int hn_batch_run_u64(const hn_batch_map* maps, uint32_t n, uint32_t ops, const uint64_t* ik, const uint64_t* iv,
                     const uint64_t* qk, uint64_t* qv, uint8_t* qh, const uint64_t* ek, void* cs, void* sc,
                     hn_stream_t s, const hn_tune* t) {
   return batch_run<uint64_t>(maps, n, ops, ik, iv, qk, qv, qh, ek, cs, sc, s, t);
}

} // extern "C"
