// hn_region.hpp -- probing a piece of a table in LDS, for the kernels that run
// on one (hn_batch.hip: regions of many maps; hn_map.hip: small tables).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "hn_device.hpp"
#include "hn_probe.hpp"

namespace hn {

// A region is 64 KiB of slots: two workgroups share a CU's LDS.  128 KiB
// regions (half the redundant key reads) would leave one.
template <typename K>
constexpr int kRegionLogB = sizeof(K) == 4 ? 13 : 12;

constexpr int kRgBS = 512; // threads per region; two regions share a CU
constexpr int kRgWaves = kRgBS / kWave;
constexpr uint32_t kRgQueue = 2 * kWave; // entries of a wave's queue
constexpr uint32_t kRgRefill = 16;       // idle lanes before a wave takes more keys

// Probe windows: four aligned slots, as the group insert's default
// (hn_probe.hpp), whose rule an insert keeps: a copy of the key anywhere in
// the window is updated before the window's EMPTY slots are looked at.
constexpr uint32_t kRgWin = 4;

template <typename K>
struct RegionMem {
   static constexpr uint32_t kSlots = 1u << kRegionLogB<K>;
   __align__(16) K key[kSlots];
   K val[kSlots]; // the value, or (insert, slots marked in `from`) its index in the list
   uint32_t from[kSlots / 32];
   K qkey[kRgWaves][kRgQueue];
   uint32_t qidx[kRgWaves][kRgQueue];
   unsigned long long n; // placed or erased
   uint32_t max_probe, flag;
};

template <typename K>
__device__ __forceinline__ K lds_cas(K* p, K expected, K desired) {
   __hip_atomic_compare_exchange_strong(p, &expected, desired, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                        __HIP_MEMORY_SCOPE_WORKGROUP);
   return expected;
}

// Match and EMPTY bits of the window that slot `pos` of an LDS key array lies
// in, from pos on.  W slots (a power of two of at most kRgWin) per window.
template <typename K>
__device__ __forceinline__ void window_bits(const K* key_s, uint32_t pos, uint32_t W, K key, uint32_t* mm,
                                            uint32_t* em) {
   const uint32_t w = pos & ~(W - 1);
   K k[kRgWin];
   if constexpr (sizeof(K) == 4) {
      // tiny regions (W < 4) start at slot 0 of the array: the load stays inside it
      const uint4 v = *reinterpret_cast<const uint4*>(key_s + (w & ~3u));
      k[0] = v.x, k[1] = v.y, k[2] = v.z, k[3] = v.w;
   } else {
      const ulonglong2 v0 = *reinterpret_cast<const ulonglong2*>(key_s + (w & ~3u));
      const ulonglong2 v1 = *reinterpret_cast<const ulonglong2*>(key_s + (w & ~3u) + 2);
      k[0] = v0.x, k[1] = v0.y, k[2] = v1.x, k[3] = v1.y;
   }
   uint32_t m = 0, e = 0;
#pragma unroll
   for (int j = 0; j < static_cast<int>(kRgWin); ++j) {
      m |= (k[j] == key ? 1u : 0u) << j;
      e |= (k[j] == empty_key<K>() ? 1u : 0u) << j;
   }
   const uint32_t valid = (W == kRgWin ? 15u : (1u << (w & 3u) << W) - 1u) & ~((1u << (pos & 3u)) - 1u);
   *mm = m & valid;
   *em = e & valid;
}

// The keys a workgroup runs through its LDS table: entries 4j..4j+3 in one
// step, 16-byte loads where a list of keys allows (a group that lies wholly
// inside [0, len) and starts on a 16-byte boundary).
template <typename K>
struct KeyList {
   const K* list;
   uint32_t len;
   uint32_t lead; // entries of group 0 that lie before list[0], so that groups start on 16-byte boundaries
   __device__ KeyList(const K* l, uint32_t n)
       : list(l), len(n), lead(static_cast<uint32_t>((reinterpret_cast<uintptr_t>(l) / sizeof(K)) & (16 / sizeof(K) - 1))) {
      if (reinterpret_cast<uintptr_t>(l) % sizeof(K)) lead = 0;
   }
   __device__ uint32_t entries() const { return len ? len + lead : 0; }
   __device__ bool valid(uint32_t e) const { return e >= lead && e - lead < len; }
   __device__ uint32_t index(uint32_t e) const { return e - lead; }
   __device__ void load(uint32_t e, K k[4]) const {
      if (e >= lead && e - lead + 4 <= len && (reinterpret_cast<uintptr_t>(list + (e - lead)) & 15u) == 0) {
         if constexpr (sizeof(K) == 4) {
            const uint4 v = *reinterpret_cast<const uint4*>(list + (e - lead));
            k[0] = v.x, k[1] = v.y, k[2] = v.z, k[3] = v.w;
         } else {
            const ulonglong2 v0 = *reinterpret_cast<const ulonglong2*>(list + (e - lead));
            const ulonglong2 v1 = *reinterpret_cast<const ulonglong2*>(list + (e - lead) + 2);
            k[0] = v0.x, k[1] = v0.y, k[2] = v1.x, k[3] = v1.y;
         }
      } else {
#pragma unroll
         for (int j = 0; j < 4; ++j) k[j] = valid(e + j) ? list[e + j - lead] : K(0);
      }
   }
};
// The same over some of a list's keys, by index.
template <typename K>
struct PickedKeys {
   const K* list;
   const uint32_t* pick;
   uint32_t len;
   __device__ uint32_t entries() const { return len; }
   __device__ bool valid(uint32_t e) const { return e < len; }
   __device__ uint32_t index(uint32_t e) const { return e < len ? pick[e] : 0; }
   __device__ void load(uint32_t e, K k[4]) const {
#pragma unroll
      for (int j = 0; j < 4; ++j) k[j] = e + j < len ? list[pick[e + j]] : K(0);
   }
};
// The same over the keys of a slot array.
template <typename K>
struct SlotKeys {
   const Slot<K>* slots;
   uint32_t len;
   __device__ uint32_t entries() const { return len; }
   __device__ bool valid(uint32_t e) const { return e < len; }
   __device__ uint32_t index(uint32_t e) const { return e; }
   __device__ void load(uint32_t e, K k[4]) const {
#pragma unroll
      for (int j = 0; j < 4; ++j) k[j] = e + j < len ? slots[e + j].key : K(0);
   }
};

// Runs the keys of `src` that `take` accepts through probes of the
// workgroup's LDS table.  Every lane probes a key of its own; `step` looks at
// one window (pos: the next slot to look at; off: its distance from the home
// slot) and returns whether the key is finished, and a lane that finishes
// takes the wave's next key, so a wave does not wait for its longest probe
// (velocity-grid ids at load factor 0.6 in 2^15 slots: mean probe of an
// absent key 54 slots, of the longest in 64 keys 198).  The waves take blocks
// of 256 entries in turn, four per lane, loaded two blocks ahead (a region of
// a map of eight reads eight times the keys it takes), and queue the ones
// they keep.  Every lane of the workgroup calls.
template <typename K, typename Src, typename Take, typename Home, typename Step>
__device__ __forceinline__ void lds_probe(RegionMem<K>& L, const Src src, int sp, Take take, Home home_pos, Step step) {
   const uint32_t lane = __lane_id();
   const int wave = threadIdx.x / kWave;
   K* const qk = L.qkey[wave];
   uint32_t* const qi = L.qidx[wave];
   const uint32_t len = src.entries();
   uint32_t b = static_cast<uint32_t>(wave) * 4 * kWave; // the block in k0, `sub` of its four parts taken
   uint32_t sub = 0;
   K k0[4], k1[4], k2[4]; // blocks b, b + 4 * BS, b + 8 * BS
   auto load = [&](uint32_t at, K k[4]) {
      if (at < len) src.load(at + 4 * lane, k);
   };
   load(b, k0), load(b + 4 * kRgBS, k1), load(b + 8 * kRgBS, k2);
   uint32_t head = 0, have = 0;
   bool active = false;
   K key = 0;
   uint32_t idx = 0, pos = 0, off = 0;
   for (;;) {
      const uint64_t idle = __ballot(!active);
      const uint32_t ni = static_cast<uint32_t>(__popcll(idle));
      if (ni == kWave && b >= len && have == 0) break;
      if (ni >= kRgRefill && (have || b < len)) {
         while (have < ni && have <= kRgQueue - kWave && b < len) {
            const uint32_t e = b + 4 * lane + sub;
            const K k = k0[0];
            const bool in = src.valid(e) && take(src.index(e), k, home_slot(k, sp));
            k0[0] = k0[1], k0[1] = k0[2], k0[2] = k0[3];
            if (++sub == 4) {
               sub = 0;
               b += 4 * kRgBS;
#pragma unroll
               for (int j = 0; j < 4; ++j) k0[j] = k1[j], k1[j] = k2[j];
               load(b + 8 * kRgBS, k2);
            }
            const uint64_t m = __ballot(in);
            const uint32_t rank = __builtin_amdgcn_mbcnt_hi(
                static_cast<uint32_t>(m >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(m), 0));
            if (in) {
               const uint32_t q = (head + have + rank) & (kRgQueue - 1);
               qk[q] = k;
               qi[q] = src.index(e);
            }
            have += static_cast<uint32_t>(__popcll(m));
         }
         wave_lds_sync();
         const uint32_t n = have < ni ? have : ni;
         const uint32_t rank = __builtin_amdgcn_mbcnt_hi(
             static_cast<uint32_t>(idle >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(idle), 0));
         if (!active && rank < n) {
            const uint32_t q = (head + rank) & (kRgQueue - 1);
            key = qk[q];
            idx = qi[q];
            pos = home_pos(home_slot(key, sp));
            off = 0;
            active = true;
         }
         wave_lds_sync(); // entries read before they are written again
         head += n;
         have -= n;
      }
      if (active) active = !step(key, idx, pos, off);
   }
}

// One window of an LDS insert of entry idx of the list: the key updated
// where a copy stands, or placed in the window's first EMPTY slot (*at, its
// probe off + (*at - pos) + 1 long); with neither, pos and off move on to the
// next window (STEP_NEXT; pos may now be R), and STEP_AGAIN says that another
// lane took the slot first: look at the window again.
enum InsertStep { STEP_DONE, STEP_PLACED, STEP_AGAIN, STEP_NEXT };
template <typename K>
__device__ __forceinline__ InsertStep lds_insert_step(RegionMem<K>& L, uint32_t R, uint32_t W, K key, uint32_t idx,
                                                      uint32_t& pos, uint32_t& off, uint32_t* at) {
   uint32_t mm, em;
   window_bits<K>(L.key, pos, W, key, &mm, &em);
   const uint32_t w = pos & ~3u; // bit 0's slot
   if (mm | em) {
      *at = w + __ffs(mm ? mm : em) - 1;
      bool placed = false;
      if (!mm) {
         const K old = lds_cas(&L.key[*at], empty_key<K>(), key);
         if (old != empty_key<K>() && old != key) return STEP_AGAIN;
         placed = old != key;
      }
      L.val[*at] = static_cast<K>(idx);
      atomicOr(&L.from[*at >> 5], 1u << (*at & 31));
      return placed ? STEP_PLACED : STEP_DONE;
   }
   const uint32_t next = (pos & ~(W - 1)) + W;
   off += next - pos;
   pos = next;
   return STEP_NEXT;
}

} // namespace hn
