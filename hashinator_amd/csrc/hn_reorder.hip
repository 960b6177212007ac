// hn_reorder.hip -- Robin Hood reorder pass over a linear-probing table.
//
// The accelerated insert (kernels_AMD.h insert_kernel) leaves each cluster in
// the order the keys happened to arrive.  This pass rewrites every cluster (a
// maximal run of non-EMPTY slots) so that its elements stand in order of home
// slot, ties broken by key: the layout linear probing produces when the keys
// arrive in sorted-home order.  The live set, the occupancy of every slot,
// fill and tombstone count are unchanged; the longest probe cannot grow
// (within a run of fixed slots, home order minimises the largest
// displacement), and currentMaxBucketOverflow is recomputed from the new
// layout (at LF 0.9 it falls from ~700 to ~64).  In that order a lookup may stop at the first occupant whose
// own displacement is smaller than the probe offset: every slot after it holds
// keys whose home lies after the query's.  The lookup kernels do so when the
// table's Info carries the ordered bit, which this pass sets and every insert
// clears.
//
// Work split.  Tile t owns the segment [b_t, b_{t+1}) where b_t is the first
// EMPTY slot at or after t*T (positions unwrapped, b_{N/T} = b_0 + N), so
// segments are whole clusters and tile the table.  A workgroup stages its
// segment's keys in LDS, computes each element's rank from a packed
// histogram-and-occupancy scan, and writes only the elements that move.  A
// segment longer than the first pass's LDS capacity goes to a list that a
// second pass with 4x the capacity works through; one longer than that is
// left as it is and the table is then not marked ordered.
#include <algorithm>

#include "hn_device.hpp"
#include "hn_host.hpp"

namespace hn {

constexpr uint64_t kReorderTile = 1024;

struct ReorderHeader {
   uint32_t n_over;    // segments handed to the second pass
   uint32_t fail;      // a segment too long for the second pass
   uint32_t skip;      // tombstones present or no EMPTY slot: nothing is done
   uint32_t max_probe; // longest probe (displacement + 1) over the reordered segments
   uint32_t pad[60];
};
static_assert(sizeof(ReorderHeader) == 256, "header is one 256-byte line");

inline uint64_t reorder_tile(int sp) { return std::min<uint64_t>(kReorderTile, 1ull << sp); }

// `gate` (nullable): run only when *gate is nonzero (a flag another pass leaves).
__device__ __forceinline__ void reorder_begin(const hn_info* info, ReorderHeader* h, uint64_t n, const uint32_t* gate) {
   if (threadIdx.x == 0) {
      h->n_over = 0;
      h->fail = 0;
      h->max_probe = 0;
      h->skip = ((gate && *gate == 0) || info->tombstone_counter != 0 || info->fill >= n ||
                 (info->reserved1 & kInfoOrdered))
                    ? 1u
                    : 0u; // an ordered table is its own reorder
   }
}
__global__ void k_reorder_begin(const hn_info* info, ReorderHeader* h, uint64_t n, const uint32_t* gate) {
   reorder_begin(info, h, n, gate);
}

// Every segment reordered: the overflow is the new layout's own.  Otherwise
// the segments left as they were keep their probes, so it can only grow.
__device__ __forceinline__ void reorder_end(hn_info* info, const ReorderHeader* h) {
   if (threadIdx.x != 0 || h->skip) return;
   const uint64_t o = std::max<uint64_t>(kBucketOverflow, next_overflow(h->max_probe, kBucketOverflow));
   if (h->fail) {
      if (o > info->current_max_bucket_overflow) info->current_max_bucket_overflow = o;
   } else {
      info->current_max_bucket_overflow = o;
      info->reserved1 |= kInfoOrdered;
   }
}

// Unwrapped position of the first EMPTY slot in [from, from + limit), or kNoPos.
// Called by a whole wave.
constexpr uint64_t kNoPos = ~0ull;
template <typename K>
__device__ uint64_t first_empty(const Slot<K>* b, uint64_t mask, uint64_t from, uint64_t limit) {
   const int lane = __lane_id();
   for (uint64_t o = 0; o < limit; o += kWave) {
      const bool e = (o + lane < limit) && b[(from + o + lane) & mask].key == empty_key<K>();
      const uint64_t m = __ballot(e);
      if (m) return from + o + first_bit(m);
   }
   return kNoPos;
}

// One workgroup per segment.  LDS per slot of capacity: a key (in home
// order), a packed (histogram << 16 | occupied) scan word, and the slot of
// each occupied rank.  Bound by its LDS latencies, one after another, so the
// scan runs on DPP and the ranks of four keys side by side.  AHEAD (the first
// pass): the tile's keys are loaded at once and the segment's bounds found in
// them, instead of the bounds first; the values of the keys that move (few, in
// a sparse table) follow when that is known.  2^26 slots, before -> here: u64
// at load .36 686 -> 467 us, at .9 891 -> 586; u32 507 -> 448 and 630 -> 537.
// SOLO: the launch is one workgroup over the whole table, its begin and its
// end among the rest.
template <typename K, int BS, int E, bool AHEAD, bool SOLO = false>
__global__ __launch_bounds__(BS) void k_reorder(Slot<K>* b, int sp, hn_info* info, ReorderHeader* h,
                                                uint32_t* over, uint64_t tile, uint32_t n_tiles, int second,
                                                const uint32_t* gate) {
   constexpr uint32_t CAP = BS * E;
   static_assert(CAP < 65536, "16-bit LDS indices and packed scan halves");
   __shared__ K key_s[CAP];
   __shared__ uint32_t pre_s[CAP + 1];
   __shared__ uint16_t slot_of_s[CAP];
   __shared__ uint64_t bounds_s[2];
   __shared__ uint32_t rel_s[2];
   __shared__ uint32_t wsum_s[BS / kWave];
   __shared__ uint32_t probe_s;
   if constexpr (SOLO) {
      reorder_begin(info, h, 1ull << sp, gate);
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
      __syncthreads();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
   }
   if (h->skip) return;
   const uint64_t n = 1ull << sp, mask = n - 1;
   const int lane = __lane_id();
   const int wave = threadIdx.x / kWave;
   const uint32_t count = second ? h->n_over : n_tiles;
   if (threadIdx.x == 0) probe_s = 0;
   uint32_t max_probe = 0;
   for (uint32_t it = blockIdx.x; it < count; it += gridDim.x) {
      __syncthreads(); // LDS of the previous segment is no longer read
      const uint64_t t = second ? over[it] : it;
      const uint64_t lo = t * tile;
      K kk[E];
      uint64_t b0, b1;
      // the slot of a thread's element e, from b0
      auto at = [&](int e) -> uint32_t {
         const uint32_t x = threadIdx.x + e * BS;
         return AHEAD ? x - static_cast<uint32_t>(b0 - lo) : x; // before b0: past len
      };
      if constexpr (AHEAD) {
         if (threadIdx.x < 2) rel_s[threadIdx.x] = ~0u;
#pragma unroll
         for (int e = 0; e < E; ++e) {
            const uint32_t x = threadIdx.x + e * BS;
            if (x < tile) kk[e] = b[(lo + x) & mask].key;
         }
         K next = empty_key<K>(); // wave 0 looks behind the tile
         if (wave == 0) next = b[(lo + tile + lane) & mask].key;
         __syncthreads();
#pragma unroll
         for (int e = 0; e < E; ++e) {
            const uint32_t x = threadIdx.x + e * BS;
            const uint64_t m = __ballot(x < tile && kk[e] == empty_key<K>());
            if (m && lane == 0) atomicMin(&rel_s[0], x + static_cast<uint32_t>(first_bit(m)));
         }
         if (wave == 0) {
            const uint64_t m = __ballot(next == empty_key<K>());
            uint64_t r = m ? lo + tile + first_bit(m) : first_empty<K>(b, mask, lo + tile + kWave, CAP);
            if (lane == 0 && r != kNoPos) rel_s[1] = static_cast<uint32_t>(r - lo);
         }
         __syncthreads();
         b0 = rel_s[0] == ~0u ? kNoPos : lo + rel_s[0];
         b1 = rel_s[1] > CAP ? kNoPos : lo + rel_s[1];
      } else {
         if (wave < 2) {
            const uint64_t r = wave == 0 ? first_empty<K>(b, mask, lo, tile) : first_empty<K>(b, mask, lo + tile, CAP);
            if (lane == 0) bounds_s[wave] = r;
         }
         __syncthreads();
         b0 = bounds_s[0];
         b1 = bounds_s[1];
      }
      // No EMPTY slot in this tile: the segment is empty (b_t == b_{t+1}).
      if (b0 == kNoPos || b0 >= lo + tile) continue;
      if (b1 == kNoPos || b1 - b0 > CAP) {
         if (threadIdx.x == 0) {
            if (second) {
               __hip_atomic_store(&h->fail, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            } else {
               const uint32_t k = atomic_add_relaxed(&h->n_over, 1u);
               over[k] = static_cast<uint32_t>(t);
            }
         }
         continue;
      }
      const uint32_t len = static_cast<uint32_t>(b1 - b0);
      for (uint32_t i = threadIdx.x; i <= len; i += BS) pre_s[i] = 0;
#pragma unroll
      for (int e = 0; e < E; ++e)
         if (at(e) < len && (!AHEAD || threadIdx.x + e * BS >= tile)) kk[e] = b[(b0 + at(e)) & mask].key;
      __syncthreads();

      uint32_t rs[E]; // home from the segment's start << 16 | rank among its arrivals; 0: no key
#pragma unroll
      for (int e = 0; e < E; ++e) {
         const uint32_t i = at(e);
         rs[e] = 0;
         if (i < len && kk[e] != empty_key<K>()) {
            // A valid table has 1 <= r <= i.
            const uint32_t r = static_cast<uint32_t>(std::min<uint64_t>((fib_home(kk[e], sp) - b0) & mask, i));
            rs[e] = (r << 16) | (atomicAdd(&pre_s[r], 1u << 16) >> 16);
            atomicAdd(&pre_s[i], 1u);
         }
      }
      __syncthreads();

      // Exclusive scan of pre_s[0..len]: high half = elements with a smaller
      // relative home, low half = occupied slots before.
      {
         const uint32_t m = len + 1;
         const uint32_t per = (m + BS - 1) / BS;
         const uint32_t c0 = std::min<uint32_t>(threadIdx.x * per, m), c1 = std::min<uint32_t>(c0 + per, m);
         uint32_t acc = 0;
         for (uint32_t x = c0; x < c1; ++x) acc += pre_s[x];
         const uint32_t inc = wave_incl_add(acc);
         if (lane == kWave - 1) wsum_s[wave] = inc;
         __syncthreads();
         uint32_t run = inc - acc;
#pragma unroll
         for (int w = 0; w < BS / kWave; ++w) {
            const uint32_t c = wsum_s[w];
            run += w < wave ? c : 0u;
         }
         for (uint32_t x = c0; x < c1; ++x) {
            const uint32_t v = pre_s[x];
            pre_s[x] = run;
            run += v;
         }
      }
      __syncthreads();

      auto has = [&](int e) { return at(e) < len && kk[e] != empty_key<K>(); };
#pragma unroll
      for (int e = 0; e < E; ++e) {
         if (has(e)) {
            slot_of_s[pre_s[at(e)] & 0xFFFFu] = static_cast<uint16_t>(at(e));
            key_s[(pre_s[rs[e] >> 16] >> 16) + (rs[e] & 0xFFFFu)] = kk[e];
         }
      }
      __syncthreads();

      uint32_t dest[E];
      constexpr int SIDE = E < 4 ? E : 4;
#pragma unroll
      for (int b4 = 0; b4 < E; b4 += SIDE) {
         uint32_t s0[SIDE], sn[SIDE], tie[SIDE];
#pragma unroll
         for (int x = 0; x < SIDE; ++x) {
            const bool h4 = b4 + x < E && has(b4 + x);
            s0[x] = h4 ? pre_s[rs[b4 + x] >> 16] >> 16 : 0;
            sn[x] = h4 ? (pre_s[(rs[b4 + x] >> 16) + 1] >> 16) - s0[x] : 0;
            tie[x] = 0;
         }
         for (uint32_t r = 0;; ++r) {
            bool any = false;
#pragma unroll
            for (int x = 0; x < SIDE; ++x) any = any || r < sn[x];
            if (!__ballot(any)) break;
            K kj[SIDE];
#pragma unroll
            for (int x = 0; x < SIDE; ++x) kj[x] = key_s[s0[x] + (r < sn[x] ? r : 0)];
#pragma unroll
            for (int x = 0; x < SIDE; ++x)
               if (b4 + x < E) tie[x] += r < sn[x] && kj[x] < kk[b4 + x] ? 1u : 0u;
         }
#pragma unroll
         for (int x = 0; x < SIDE; ++x)
            if (b4 + x < E) dest[b4 + x] = sn[x] ? slot_of_s[s0[x] + tie[x]] : at(b4 + x);
      }
      // The values of the keys that move, all read before a slot is written.
      K vv[E];
#pragma unroll
      for (int e = 0; e < E; ++e) vv[e] = dest[e] != at(e) ? b[(b0 + at(e)) & mask].val : 0;
#pragma unroll
      for (int e = 0; e < E; ++e) asm volatile("" ::"v"(vv[e]) : "memory"); // they have arrived
      __syncthreads();
#pragma unroll
      for (int e = 0; e < E; ++e) {
         const uint32_t r = rs[e] >> 16;
         if (dest[e] != at(e)) {
            Slot<K> s;
            s.key = kk[e];
            s.val = vv[e];
            b[(b0 + dest[e]) & mask] = s;
         }
         if (has(e) && dest[e] >= r) max_probe = std::max<uint32_t>(max_probe, dest[e] - r + 1);
      }
   }
   // One atomic per block at most, and only while the running maximum grows.
   max_probe = wave_max(max_probe);
   __syncthreads();
   if (lane == 0 && max_probe) atomicMax(&probe_s, max_probe);
   __syncthreads();
   if constexpr (SOLO) {
      if (threadIdx.x == 0) h->max_probe = probe_s;
      reorder_end(info, h);
   } else if (threadIdx.x == 0 &&
              probe_s > __hip_atomic_load(&h->max_probe, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
      atomic_max_relaxed(&h->max_probe, probe_s);
   }
}

__global__ void k_reorder_end(hn_info* info, const ReorderHeader* h) { reorder_end(info, h); }

size_t reorder_scratch_bytes(int sp) {
   if (sp < 1 || sp > 63) return 0;
   const uint64_t tiles = (1ull << sp) / reorder_tile(sp);
   return sizeof(ReorderHeader) + tiles * sizeof(uint32_t);
}

constexpr int kReorderBS1 = 256, kReorderBS2 = 1024, kReorderE = 8;
// Tables up to 2^kReorderSolo slots fit one workgroup's segment whole: one
// launch instead of four (2^10 u64 slots: 17.2 -> 8.6 us, 2^12 18.0 -> 10.8).
constexpr int kReorderSolo = 12;

template <typename K>
int reorder(void* buckets, hn_info* info, int sp, void* scratch, size_t bytes, hipStream_t s,
            const uint32_t* gate = nullptr) {
   if (!buckets || !info || !scratch) return HN_EINVAL;
   if (sp < 1 || sp > max_size_power<K>()) return HN_EINVAL;
   if (bytes < reorder_scratch_bytes(sp)) return HN_ESCRATCH;
   const uint64_t n = 1ull << sp, tile = reorder_tile(sp), tiles = n / tile;
   if (tiles > 0xFFFFFFFFull) return HN_EINVAL;
   ReorderHeader* h = static_cast<ReorderHeader*>(scratch);
   uint32_t* over = reinterpret_cast<uint32_t*>(h + 1);
   Slot<K>* b = static_cast<Slot<K>*>(buckets);
   if (sp <= kReorderSolo) {
      hipLaunchKernelGGL((k_reorder<K, kReorderBS2, kReorderE, false, true>), dim3(1), dim3(kReorderBS2), 0, s, b, sp, info, h,
                         over, n, 1u, 0, gate);
      return static_cast<int>(hipGetLastError());
   }
   hipLaunchKernelGGL(k_reorder_begin, dim3(1), dim3(64), 0, s, info, h, n, gate);
   hipLaunchKernelGGL((k_reorder<K, kReorderBS1, kReorderE, true>), dim3(static_cast<uint32_t>(tiles)), dim3(kReorderBS1), 0,
                      s, b, sp, info, h, over, tile, static_cast<uint32_t>(tiles), 0, nullptr);
   const uint32_t grid2 = static_cast<uint32_t>(std::min<uint64_t>(tiles, static_cast<uint64_t>(cu_count())));
   hipLaunchKernelGGL((k_reorder<K, kReorderBS2, kReorderE, false>), dim3(grid2), dim3(kReorderBS2), 0, s, b, sp, info, h,
                      over, tile, static_cast<uint32_t>(tiles), 1, nullptr);
   hipLaunchKernelGGL(k_reorder_end, dim3(1), dim3(64), 0, s, info, h);
   return static_cast<int>(hipGetLastError());
}

// The reorder after the region clean of clean_tombstones, run only when the
// segment pass of hn_clean.hip left the table to that path.
template <typename K>
int reorder_gated(void* buckets, hn_info* info, int sp, void* scratch, size_t bytes, const uint32_t* gate,
                  hipStream_t s) {
   return reorder<K>(buckets, info, sp, scratch, bytes, s, gate);
}
template int reorder_gated<uint32_t>(void*, hn_info*, int, void*, size_t, const uint32_t*, hipStream_t);
template int reorder_gated<uint64_t>(void*, hn_info*, int, void*, size_t, const uint32_t*, hipStream_t);

} // namespace hn

using namespace hn;
extern "C" {
size_t hn_reorder_scratch_bytes(int sp) { return reorder_scratch_bytes(sp); }
int hn_reorder_u32(void* b, hn_info* i, int sp, void* sc, size_t sb, hn_stream_t s) {
   return reorder<uint32_t>(b, i, sp, sc, sb, s);
}
int hn_reorder_u64(void* b, hn_info* i, int sp, void* sc, size_t sb, hn_stream_t s) {
   return reorder<uint64_t>(b, i, sp, sc, sb, s);
}
} // extern "C"
