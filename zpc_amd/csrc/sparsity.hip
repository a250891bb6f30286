// Block activation, neighbour enlargement and the particle -> block bucket
// sort on zpc's HashTable<i32,3,int> layout, for gfx950.
//
// zpc inserts keys with per-slot spin locks and an atomic block counter
// (container/HashTable.hpp:356-398), so under its parallel policies the block
// numbers and slot layout depend on timing. Here they are deterministic and
// equal to zpc's sequential semantics:
//   * numbering: a key gets the next block number in order of its first
//     occurrence (particle index for activation, (block, dx, dy, dz) loop
//     order for enlargement) -- found with a dedup hash holding the minimum
//     order per key; each new key's order sets one bit of a bitmap, and an
//     exclusive popcount scan of the bitmap ranks the new keys;
//   * slots: keys are placed by priority linear probing on the reference
//     probe sequence (home = (h % T + T) % T, step 127) with priority = block
//     number; the result equals inserting serially in block-number order
//     (Shun & Blelloch, "Phase-Concurrent Hash Tables for Determinism",
//     SPAA 2014), i.e. the layout zpc's seq_exec path produces.
// The bucket sort is stable by particle index (zpc's seq semantics of
// SpatiallyCount/SpatiallyDistribute): tiles of 1,024 particles are cut into
// segments of equal key; every segment takes a place in its bucket's list with
// the one atomic that also counts it, and a workgroup per bucket orders the
// list by first particle and writes the bucket's indices. No sort over the
// whole set: the counts give the buckets, and a list has ~2 entries when the
// particles are in bucket order (a few hundred when they are shuffled).
// The substep's own build (build_clear .. build_place) numbers, places and
// enlarges from one dedup hash and one clear, with no device-wide scan: 9
// launches where the stage-by-stage operators take about 35.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "zsmpm_device.hpp"
#include "zsmpm_internal.hpp"

namespace zsmpm {

namespace {

constexpr int kThreads = 256;

inline int groups_for(int64_t n, int threads) {
  int64_t g = (n + threads - 1) / threads;
  if (g < 1) g = 1;
  if (g > 65535 * 8) g = 65535 * 8;
  return (int)g;
}

// --------------------------------------------------------------- clearing
__global__ void clear_table_kernel(TableView t, uint64_t* skey, uint32_t* sorder, uint32_t* dmask, uint32_t ts,
                                   uint32_t* counters) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < (int64_t)((ts + 31u) >> 5); e += stride) dmask[e] = 0u;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < t.T; e += stride) {
    t.keys[3 * e] = kKeySentinel;
    t.keys[3 * e + 1] = kKeySentinel;
    t.keys[3 * e + 2] = kKeySentinel;
    t.indices[e] = -1;
    t.status[e] = -1;
  }
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < ts; e += stride) {
    skey[e] = kEmpty64;
    sorder[e] = 0xffffffffu;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    *t.cnt = 0;
    counters[kCtrList] = 0;
  }
}

__global__ void clear_scratch_kernel(uint64_t* skey, uint32_t* sorder, uint32_t* dmask, uint32_t ts,
                                     const int32_t* cnt, uint32_t* counters, uint32_t* bitmap, int64_t bm_n) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < (int64_t)((ts + 31u) >> 5); e += stride) dmask[e] = 0u;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < bm_n; e += stride) bitmap[e] = 0u;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < ts; e += stride) {
    skey[e] = kEmpty64;
    sorder[e] = 0xffffffffu;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    counters[kCtrList] = 0;
    counters[kCtrCnt0] = (uint32_t)*cnt;
  }
}

// ----------------------------------------------------------- dedup inserts
// The dedup scratch of one insertion pass: packed keys and minimum orders per
// slot, and one bit per slot the pass claimed, so the pass's keys are found
// by reading ts/32 words instead of all ts slots. (A list of claimed slots
// behind one atomic counter was slower: tens of thousands of same-address
// atomics serialize.)
struct Dedup {
  uint64_t* skey;
  uint32_t* sorder;
  uint32_t ts;
  uint32_t* err;
  uint32_t* dmask;  // [ts / 32]
};

__device__ __forceinline__ uint32_t dedup_home(uint64_t pk, uint32_t ts) { return (uint32_t)mix64(pk) & (ts - 1u); }

// Finishes an insert whose look at slot s showed cur: probes on until the slot
// is free or holds pk (ts probes in all); the insert that claims a free slot
// marks it in `mask`. Returns the slot holding pk, or ~0u when the scratch
// table is full. Plain loads come before the atomics: keys are only ever added,
// so a stale value costs an atomic that was not needed and nothing else.
__device__ __forceinline__ uint32_t dedup_finish(uint64_t pk, uint32_t s, uint64_t cur, const Dedup& d,
                                                 uint32_t* mask) {
  for (uint32_t probe = 1;; ++probe) {
    if (cur == pk) return s;
    if (cur == kEmpty64) {
      cur = atomicCAS((unsigned long long*)&d.skey[s], (unsigned long long)kEmpty64, (unsigned long long)pk);
      if (cur == kEmpty64) {
        atomicOr(&mask[s >> 5], 1u << (s & 31u));
        return s;
      }
      if (cur == pk) return s;
    }
    if (probe >= d.ts) {
      atomicOr(d.err, kErrTableFull);
      return ~0u;
    }
    s = (s + 1u) & (d.ts - 1u);
    cur = d.skey[s];
  }
}

// the slot's order lowered to `order` (orders are only lowered: a stale value
// is never too low)
__device__ __forceinline__ void dedup_order(uint32_t s, uint32_t order, const Dedup& d) {
  if (s != ~0u && d.sorder[s] > order) atomicMin(&d.sorder[s], order);
}

__device__ __forceinline__ uint32_t dedup_insert(uint64_t pk, uint32_t order, const Dedup& d) {
  uint32_t s = dedup_home(pk, d.ts);
  s = dedup_finish(pk, s, d.skey[s], d, d.dmask);
  dedup_order(s, order, d);
  return s;
}

// The particles are cut into tiles of consecutive ones, and a tile into
// segments of equal bucket. Per tile, the number of segments; per segment (the
// j-th of the tile at its first particle's index + j) the bucket it belongs to (a dedup slot or a
// block), its place in that bucket's list, from the atomic that counted it, and
// where it lies in the tile (first | length << 16). `place` holds segments << 32
// | particles per bucket. In bucket order a tile has ~3 segments and a bucket
// ~2; one wave's 64 particles per segment cost four times the atomics (the
// build's activation of 16M particles 136 us).
constexpr int kWideTile = 4;  // items per thread: tiles of 1,024, or
constexpr int kTightTile = 1; // of 256 below 2^21 particles, where workgroups are scarce
struct Segments {
  uint32_t* count = nullptr;  // [tiles]
  uint2* in = nullptr;        // [n, whole tiles]
  uint32_t* where = nullptr;  // [n, whole tiles]
  uint64_t* place = nullptr;
};

// The segments of a tile from its particles' keys (item r of thread i is
// particle r kThreads + i; `live` particles), listed in order: key and where
// (first | length << 16); returns their number. A particle without a key (live
// but out of range: kEmpty64) belongs to segments too.
template <int kTileItems>
struct TileLds {
  static constexpr int kTile = kThreads * kTileItems;
  uint64_t last[kTileItems][kThreads / kWave];
  uint64_t heads[kTile / kWave];
  uint64_t key[kTile];
  uint32_t where[kTile];
};
template <int kTileItems>
__device__ __forceinline__ uint32_t tile_segments(const uint64_t (&key)[kTileItems], int live,
                                                  TileLds<kTileItems>& lds) {
  const int lane = lane_id(), wave = uniform((int32_t)(threadIdx.x / kWave));
  constexpr int kW = kThreads / kWave;
#pragma unroll
  for (int r = 0; r < kTileItems; ++r)
    if (lane == kWave - 1) lds.last[r][wave] = key[r];
  __syncthreads();
  uint64_t heads[kTileItems];
#pragma unroll
  for (int r = 0; r < kTileItems; ++r) {
    uint64_t prev = __shfl_up(key[r], 1, kWave);
    const bool first = r == 0 && threadIdx.x == 0;
    if (lane == 0 && !first) prev = wave > 0 ? lds.last[r][wave - 1] : lds.last[r > 0 ? r - 1 : 0][kW - 1];
    heads[r] = ballot(r * kThreads + (int)threadIdx.x < live && (first || prev != key[r]));
    if (lane == 0) lds.heads[r * kW + wave] = heads[r];
  }
  __syncthreads();
  // lane q: heads before group q and the first head after it
  constexpr int kGroups = TileLds<kTileItems>::kTile / kWave;
  const uint64_t mq = lane < kGroups ? lds.heads[lane] : 0ull;
  int before = __popcll(mq), next = live;
  int first = mq ? lane * kWave + __ffsll((long long)mq) - 1 : live;
#pragma unroll
  for (int o = 1; o < kGroups; o <<= 1) {
    const int u = __shfl_up(before, o, kWave), f = __shfl_down(first, o, kWave);
    if (lane >= o) before += u;
    if (lane + o < kGroups) first = min(first, f);
  }
  const uint32_t count = (uint32_t)__builtin_amdgcn_readlane(before, kGroups - 1);
  before -= __popcll(mq);
  const int after = __shfl_down(first, 1, kWave);
  if (lane + 1 < kGroups) next = after;
#pragma unroll
  for (int r = 0; r < kTileItems; ++r) {
    if (heads[r] == 0) continue;  // most groups start no segment
    const int g = r * kW + wave, at = g * kWave + lane;
    const uint64_t above = lane == 63 ? 0ull : heads[r] >> (lane + 1);
    // read with the whole wave active: lane g holds group g's value
    const int later = __builtin_amdgcn_readlane(next, g);
    const int end = above ? at + __ffsll((long long)above) : later;
    const int rank = __builtin_amdgcn_readlane(before, g) + __popcll(heads[r] & lanemask_lt());
    if ((heads[r] >> lane) & 1ull) {
      lds.key[rank] = key[r];
      lds.where[rank] = (uint32_t)at | ((uint32_t)(end - at) << 16);
    }
  }
  __syncthreads();
  return count;
}

// ComputeSparsity candidates: one per segment of a tile, by its first particle
// (order = particle index). The kernel is bound by dependent round trips, not
// by bytes: a workgroup has its next tile's positions in flight while it
// inserts this one's segments, and the first probes are issued together. The dedup
// hash keeps the minimum order per key, so the result does not depend on the
// order of the inserts. kSegs: the segments are recorded for the bucket sort.
// kMulti (a batch, ss): particle p takes its scene's 1/dx, and its key is
// shifted by the scene's offset (a key outside the scene's own range
// [-512, 511) along axis 0 is a key-range error)
template <bool kMulti, bool kSegs, int kTileItems>
__global__ __launch_bounds__(kThreads) void activate_kernel(const float* __restrict__ x, int64_t n,
                                                            float dxinv, int blockLen, int offset,
                                                            float disp, Dedup dd, Segments sg, SceneSet ss) {
  constexpr int kTile = kThreads * kTileItems;
  uint32_t* err = dd.err;
  const int64_t ntiles = (n + kTile - 1) / kTile;
  __shared__ int64_t sfirst[kMulti ? kMaxScenes + 1 : 1];
  __shared__ TileLds<kTileItems> lds;
  if constexpr (kMulti) {
    for (int i = threadIdx.x; i <= ss.n; i += kThreads) sfirst[i] = ss.first[i];
    __syncthreads();
  }
  float nx[kTileItems], ny[kTileItems], nz[kTileItems];  // the next tile's positions, in flight
  auto load = [&](int64_t tile) {
#pragma unroll
    for (int r = 0; r < kTileItems; ++r) {
      const int64_t p = tile * kTile + (int64_t)r * kThreads + threadIdx.x;
      nx[r] = ny[r] = nz[r] = 0.f;
      if (p < n) {
        nx[r] = x[3 * p];
        ny[r] = x[3 * p + 1];
        nz[r] = x[3 * p + 2];
      }
    }
  };
  load(blockIdx.x);
  for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const int64_t base = tile * kTile;
    const int live = (int)min((int64_t)kTile, n - base);
    float cx[kTileItems], cy[kTileItems], cz[kTileItems];
#pragma unroll
    for (int r = 0; r < kTileItems; ++r) {
      cx[r] = nx[r];
      cy[r] = ny[r];
      cz[r] = nz[r];
    }
    load(tile + gridDim.x);
    uint64_t pk[kTileItems];
#pragma unroll
    for (int r = 0; r < kTileItems; ++r) {
      const int64_t p = base + (int64_t)r * kThreads + threadIdx.x;
      pk[r] = kEmpty64;
      if (p < n) {
        int32_t k0, k1, k2;
        bool in_range = true;
        if constexpr (kMulti) {
          const int32_t sc = scene_of_particle(sfirst, ss.n, p);
          block_key(cx[r], cy[r], cz[r], ss.p[sc].dx_inv, blockLen, offset, disp, k0, k1, k2);
          // below 511, so the enlargement's key + 1 stays in the scene's range
          in_range = k0 >= -kSceneKeyHalf && k0 < kSceneKeyHalf - 1;
          k0 += sc * kSceneKeyStride;
        } else {
          block_key(cx[r], cy[r], cz[r], dxinv, blockLen, offset, disp, k0, k1, k2);
        }
        if (in_range && key_packable(k0, k1, k2)) {
          pk[r] = pack_key(k0, k1, k2);
        } else {
          atomicOr(err, kErrKeyRange);
        }
      }
    }
    const uint32_t count = tile_segments(pk, live, lds);
    for (uint32_t j = threadIdx.x; j < count; j += kThreads) {
      const uint64_t key = lds.key[j];
      const uint32_t w = lds.where[j], order = (uint32_t)(base + (w & 0xffffu));
      uint32_t slot = ~0u, local = 0u;
      if (key != kEmpty64) {
        slot = dedup_home(key, dd.ts);
        slot = dedup_finish(key, slot, dd.skey[slot], dd, dd.dmask);
        dedup_order(slot, order, dd);
        if (kSegs && slot != ~0u)
          local = (uint32_t)(atomicAdd((unsigned long long*)&sg.place[slot],
                                       (1ull << 32) | (unsigned long long)(w >> 16)) >>
                             32);
      }
      if (kSegs) {
        sg.in[base + j] = make_uint2(slot, local);
        sg.where[base + j] = w;
      }
    }
    if (kSegs && threadIdx.x == 0) sg.count[tile] = count;
    __syncthreads();
  }
}

// EnlargeSparsity candidates: key_i + (dx, dy, dz) for i < n0 in loop order.
__global__ __launch_bounds__(kThreads) void enlarge_kernel(const int32_t* __restrict__ active,
                                                           const uint32_t* counters, int32_t lo0, int32_t lo1,
                                                           int32_t lo2, int32_t e0, int32_t e1, int32_t e2,
                                                           Dedup dd) {
  uint32_t* err = dd.err;
  const int64_t n0 = counters[kCtrCnt0];
  const int64_t nd = (int64_t)e0 * e1 * e2;
  const int64_t total = n0 * nd;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; c < total; c += stride) {
    const int64_t i = c / nd;
    const int32_t j = (int32_t)(c - i * nd);
    const int32_t dz = j % e2, dy = (j / e2) % e1, dx = j / (e1 * e2);
    const int32_t k0 = active[3 * i] + lo0 + dx, k1 = active[3 * i + 1] + lo1 + dy,
                  k2 = active[3 * i + 2] + lo2 + dz;
    if (!key_packable(k0, k1, k2)) {
      atomicOr(err, kErrKeyRange);
      continue;
    }
    (void)dedup_insert(pack_key(k0, k1, k2), (uint32_t)c, dd);
  }
}

constexpr int kCollectGroups = 1024;
constexpr int kCollectBuf = 2048;

__device__ __forceinline__ void list_put(uint32_t slot, uint32_t key, uint32_t val, uint32_t* lkey,
                                         uint32_t* lval, uint32_t list_cap, uint32_t* err) {
  if (slot < list_cap) {
    lkey[slot] = key;
    lval[slot] = val;
  } else {
    atomicOr(err, kErrCapacity);
  }
}

// Gather the dedup entries whose key is not in the table yet: (order, slot),
// and mark each one's order in the first-occurrence bitmap. Only the slots
// the pass claimed (set bits of dmask) are visited, not all ts. Each
// workgroup takes one contiguous range of dmask words, collects its entries in
// LDS and reserves list space with a single global atomic (entries beyond the
// LDS buffer go straight to the list). The list order is irrelevant: ranks
// come from the bitmap.
__global__ __launch_bounds__(kThreads) void collect_new_kernel(const uint64_t* __restrict__ skey,
                                                               const uint32_t* __restrict__ sorder,
                                                               const uint32_t* __restrict__ dmask,
                                                               uint32_t ts, TableView t, uint32_t* counters,
                                                               uint32_t* lkey, uint32_t* lval,
                                                               uint32_t list_cap, uint32_t* err,
                                                               uint32_t* bitmap, uint32_t bm_words) {
  __shared__ uint32_t bkey[kCollectBuf], bval[kCollectBuf];
  __shared__ uint32_t bcount, gbase;
  const bool table_empty = counters[kCtrCnt0] == 0;
  const int64_t nw = (int64_t)((ts + 31u) >> 5);
  const int64_t per = (nw + gridDim.x - 1) / gridDim.x;
  const int64_t lo = (int64_t)blockIdx.x * per;
  const int64_t hi = min(nw, lo + per);
  if (threadIdx.x == 0) bcount = 0;
  __syncthreads();
  const int lane = lane_id();
  for (int64_t base = lo; base < hi; base += blockDim.x) {  // uniform across the workgroup
    const int64_t j = base + threadIdx.x;
    uint32_t bits = j < hi ? dmask[j] : 0u;  // slots beyond ts are never marked
    while (ballot(bits != 0u) != 0) {  // one claimed slot per lane per step (wave-uniform loop)
      bool take = false;
      uint32_t s = 0;
      if (bits != 0u) {
        s = (uint32_t)(j * 32) + (uint32_t)(__ffs(bits) - 1);
        bits &= bits - 1u;
        const uint64_t pk = skey[s];
        if (pk != kEmpty64) {
          take = true;
          if (!table_empty) {
            int32_t k0, k1, k2;
            unpack_key(pk, k0, k1, k2);
            take = table_find(t, k0, k1, k2) < 0;
          }
        }
      }
      const uint64_t m = ballot(take);
      if (m == 0) continue;
      const int leader = __ffsll((long long)m) - 1;
      uint32_t wbase = 0;
      if (lane == leader) wbase = atomicAdd(&bcount, (uint32_t)__popcll(m));
      wbase = shfl(wbase, leader);
      if (take) {
        // mark the key's order: its rank among the new keys is the number of
        // marked orders below it (orders of distinct keys are distinct)
        const uint32_t o = sorder[s];
        if ((o >> 5) < bm_words) atomicOr(&bitmap[o >> 5], 1u << (o & 31u));
        const uint32_t slot = wbase + (uint32_t)__popcll(m & lanemask_lt());
        if (slot < (uint32_t)kCollectBuf) {
          bkey[slot] = sorder[s];
          bval[slot] = (uint32_t)s;
        } else {
          list_put(atomicAdd(&counters[kCtrList], 1u), sorder[s], (uint32_t)s, lkey, lval, list_cap, err);
        }
      }
    }
  }
  __syncthreads();
  const uint32_t nloc = min(bcount, (uint32_t)kCollectBuf);
  if (threadIdx.x == 0) gbase = nloc ? atomicAdd(&counters[kCtrList], nloc) : 0u;
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < nloc; i += blockDim.x)
    list_put(gbase + i, bkey[i], bval[i], lkey, lval, list_cap, err);
}

// block `rank` with the key k into zpc's table by priority linear probing on
// indices[] (the lower block number wins a slot)
__device__ __forceinline__ void place_block(const TableView& t, uint32_t rank, int32_t k0, int32_t k1, int32_t k2,
                                            uint32_t* err) {
  t.active[3 * (int64_t)rank] = k0;
  t.active[3 * (int64_t)rank + 1] = k1;
  t.active[3 * (int64_t)rank + 2] = k2;
  // carried element: starts as this key; a displaced lower-priority entry
  // continues from the slot after the one it lost
  uint32_t cur = rank;
  int32_t s = zpc_home(k0, k1, k2, t.T);
  int64_t steps = 0;
  const int64_t limit = 2ll * t.T + 64;
  while (true) {
    const uint32_t old = atomicMin((uint32_t*)&t.indices[s], cur);
    if (old == 0xffffffffu) break;
    if (old > cur) cur = old;
    s = probe_next(s, t.T);
    if (++steps > limit) {
      atomicOr(err, kErrTableFull);
      break;
    }
  }
}

// Number the new keys cnt0 + rank, record _activeKeys and place them by
// priority linear probing on indices[] (lower block number wins a slot).
__global__ __launch_bounds__(kThreads) void assign_kernel(const uint32_t* __restrict__ lorder,
                                                          const uint32_t* __restrict__ lslot,
                                                          const uint32_t* __restrict__ bitmap,
                                                          const uint32_t* __restrict__ bm_prefix, uint32_t bm_words,
                                                          const uint64_t* __restrict__ skey,
                                                          TableView t, const uint32_t* counters,
                                                          uint32_t list_cap, uint32_t* err) {
  const uint32_t nl = min(counters[kCtrList], list_cap);
  const uint32_t cnt0 = counters[kCtrCnt0];
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < nl; i += stride) {
    const uint32_t sl = lslot[i];
    const uint32_t o = lorder[i];
    if ((o >> 5) >= bm_words) {
      atomicOr(err, kErrCapacity);
      continue;
    }
    // first-occurrence rank: new keys with a smaller order
    const uint32_t below = bm_prefix[o >> 5] + (uint32_t)__popc(bitmap[o >> 5] & ((1u << (o & 31u)) - 1u));
    const uint64_t pk = skey[sl];
    int32_t k0, k1, k2;
    unpack_key(pk, k0, k1, k2);
    const uint32_t rank = cnt0 + below;
    if (rank >= (uint32_t)t.T) {
      atomicOr(err, kErrTableFull);
      continue;
    }
    place_block(t, rank, k0, k1, k2, err);
  }
}

// Write keys[] of every newly placed entry: block r probes from its home
// until it finds the slot holding r.
__global__ __launch_bounds__(kThreads) void fill_keys_kernel(TableView t, const uint32_t* counters,
                                                             uint32_t list_cap, uint32_t* err) {
  const uint32_t nl = min(counters[kCtrList], list_cap);
  const uint32_t cnt0 = counters[kCtrCnt0];
  if (blockIdx.x == 0 && threadIdx.x == 0) {  // nothing in this kernel reads the count
    const int64_t c = (int64_t)cnt0 + nl;
    *t.cnt = (int32_t)(c < t.T ? c : t.T);
  }
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < nl; i += stride) {
    const int32_t r = (int32_t)(cnt0 + (uint32_t)i);
    if (r >= t.T) continue;
    const int32_t k0 = t.active[3 * (int64_t)r], k1 = t.active[3 * (int64_t)r + 1],
                  k2 = t.active[3 * (int64_t)r + 2];
    int32_t s = zpc_home(k0, k1, k2, t.T);
    int32_t probe = 0;
    for (; probe < t.T; ++probe) {
      if (t.indices[s] == r) break;
      s = probe_next(s, t.T);
    }
    if (probe == t.T) {
      atomicOr(err, kErrTableFull);
      continue;
    }
    t.keys[3 * (int64_t)s] = k0;
    t.keys[3 * (int64_t)s + 1] = k1;
    t.keys[3 * (int64_t)s + 2] = k2;
  }
}

__global__ void query_kernel(TableView t, const int32_t* __restrict__ keys, int64_t n, int32_t* out) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += stride)
    out[i] = table_find(t, keys[3 * i], keys[3 * i + 1], keys[3 * i + 2]);
}

// ------------------------------------------------------- the substep's build
// Ranks among the set bits of a bitmap of orders: the bits are counted per
// 2^shift orders as they are set (c1, at most kRankGroups counts, whose prefix
// every workgroup of the numbering forms in LDS for itself: no scan launches),
// and 8 lanes per key add up the words before the order in its group (32 words
// up to 2^24 orders). Coarser counts set with the bits made the marking slow:
// 36K atomics on 128 adjacent counters take 40 us.
constexpr int kRankGroups = 12288;  // 48 KB of LDS
struct Ranks {
  uint32_t* bitmap = nullptr;
  uint32_t* c1 = nullptr;
  uint32_t words = 0;  // of the bitmap
  int32_t shift = 10;
  int32_t groups = 0;  // of c1
};

__device__ __forceinline__ void rank_mark(const Ranks& r, uint32_t o) {
  if ((o >> 5) >= r.words) return;  // reported where the rank is taken
  atomicOr(&r.bitmap[o >> 5], 1u << (o & 31u));
  atomicAdd(&r.c1[o >> r.shift], 1u);
}

// exclusive prefix of c1 into lds[0, groups)
__device__ __forceinline__ void rank_prefix(const Ranks& r, uint32_t* lds, uint32_t* wsum) {
  const int lane = lane_id(), wave = threadIdx.x / kWave;
  uint32_t carry = 0;
  for (int base = 0; base < r.groups; base += 4 * kThreads) {  // uniform across the workgroup
    const int i = base + 4 * threadIdx.x;
    uint4 q = make_uint4(0u, 0u, 0u, 0u);
    if (i < r.groups) q = *reinterpret_cast<const uint4*>(r.c1 + i);  // padded with zeros to a whole vector
    const uint32_t mine = q.x + q.y + q.z + q.w;
    uint32_t inc = mine;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const uint32_t u = __shfl_up(inc, o, kWave);
      if (lane >= o) inc += u;
    }
    if (lane == kWave - 1) wsum[wave] = inc;
    __syncthreads();
    uint32_t run = carry + inc - mine;
#pragma unroll
    for (int w = 0; w < kThreads / kWave; ++w) {
      run += w < wave ? wsum[w] : 0u;
      carry += wsum[w];
    }
    if (i < r.groups) *reinterpret_cast<uint4*>(lds + i) = make_uint4(run, run + q.x, run + q.x + q.y, run + q.x + q.y + q.z);
    __syncthreads();
  }
}

// set bits before order o; called by the 8 lanes of a key's group (j = lane & 7)
__device__ __forceinline__ uint32_t rank_below(const Ranks& r, const uint32_t* lds, uint32_t o, int j) {
  uint32_t s = 0;
  const uint32_t w0 = (o >> r.shift) << (r.shift - 5), w1 = o >> 5;
  for (uint32_t i = w0 + 4 * j; i <= w1; i += 32) {
    const uint4 q = *reinterpret_cast<const uint4*>(r.bitmap + i);  // padded to a whole vector
    const uint32_t v[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t w = i + k;
      s += (uint32_t)__popc(w < w1 ? v[k] : (w == w1 ? v[k] & ((1u << (o & 31u)) - 1u) : 0u));
    }
  }
#pragma unroll
  for (int d = 1; d < 8; d <<= 1) s += __shfl_xor(s, d, kWave);
  return lds[o >> r.shift] + s;
}

// Everything the build reads before it writes it, in one launch.
struct ClearList {
  static constexpr int kMax = 12;
  uint32_t* p[kMax];
  int64_t n[kMax];
  uint32_t v[kMax];
  int count = 0;
};

__global__ __launch_bounds__(kThreads) void build_clear_kernel(ClearList c, TableView t, uint32_t* counters) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const int64_t i0 = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  for (int k = 0; k < c.count; ++k) {
    const uint32_t v = c.v[k];
    uint32_t* p = c.p[k];
    const int64_t n = c.n[k];
    const int64_t mis = min(n, (int64_t)((4 - ((uintptr_t)p >> 2)) & 3));  // words before a 16-byte boundary
    const int64_t nv = (n - mis) / 4;
    for (int64_t i = i0; i < nv; i += stride) reinterpret_cast<uint4*>(p + mis)[i] = make_uint4(v, v, v, v);
    if (i0 < mis) p[i0] = v;
    if (i0 < n - mis - 4 * nv) p[mis + 4 * nv + i0] = v;
  }
  if (i0 == 0) {
    *t.cnt = 0;
    counters[kCtrList] = 0u;
    counters[kCtrBlocks] = 0u;
    counters[kCtrMaxVel] = 0u;
  }
}

// The slots a pass claimed (set bits of mask) as a list of (order, slot), their
// orders marked for ranking. A workgroup takes 64 mask words, lists their slots
// in LDS and reserves room with one atomic; the list's order is irrelevant.
__global__ __launch_bounds__(kThreads) void build_collect_kernel(const uint32_t* __restrict__ mask, uint32_t nw,
                                                                 const uint32_t* __restrict__ sorder, Ranks rk,
                                                                 uint32_t* count, uint32_t* __restrict__ lorder,
                                                                 uint32_t* __restrict__ lslot) {
  __shared__ uint32_t buf[kWave * 32];
  __shared__ uint32_t total, base;
  const uint32_t w = blockIdx.x * kWave + threadIdx.x;
  if (threadIdx.x < kWave) {
    uint32_t bits = w < nw ? mask[w] : 0u;
    const uint32_t c = (uint32_t)__popc(bits);
    uint32_t inc = c;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const uint32_t u = __shfl_up(inc, o, kWave);
      if (lane_id() >= o) inc += u;
    }
    uint32_t at = inc - c;
    while (bits) {
      buf[at++] = w * 32u + (uint32_t)(__ffs(bits) - 1);
      bits &= bits - 1u;
    }
    if (threadIdx.x == kWave - 1) {
      total = inc;
      base = inc ? atomicAdd(count, inc) : 0u;
    }
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < total; i += kThreads) {
    const uint32_t s = buf[i], o = sorder[s];
    rank_mark(rk, o);
    lorder[base + i] = o;
    lslot[base + i] = s;
  }
}

// Numbers the listed keys first + rank and places them, 8 lanes per key.
// kEnlarge (the particles' keys, first = 0): lane j also inserts the key's
// j-th neighbour key + (j>>2, j>>1&1, j&1) -- EnlargeSparsity's loop order --
// with order 8 b + j, and records its slot in nbr[8 b + j]: the 2^3 blocks the
// bucket's stencils cover need no table probe later. Only keys the particles
// did not have take an order (mask marks those). bcnt receives the bucket's
// segment and particle counts.
template <bool kEnlarge>
__global__ __launch_bounds__(kThreads) void build_number_kernel(const uint32_t* count, const uint32_t* first_count,
                                                                const uint32_t* __restrict__ lorder,
                                                                const uint32_t* __restrict__ lslot, Ranks rk,
                                                                TableView t, Dedup dd, uint32_t* mask2,
                                                                int32_t* slot_block, const uint64_t* scnt,
                                                                uint64_t* bcnt, int32_t* nbr) {
  extern __shared__ uint32_t prefix[];  // [rk.groups], whole vectors
  __shared__ uint32_t wsum[kThreads / kWave];
  const uint32_t nl = *count;
  if ((int64_t)blockIdx.x * blockDim.x >= 8ll * nl) return;
  rank_prefix(rk, prefix, wsum);
  const uint32_t first = kEnlarge ? 0u : *first_count;
  const int j = lane_id() & 7;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i8 = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i8 < 8ll * nl; i8 += stride) {
    const uint32_t o = lorder[i8 >> 3], sl = lslot[i8 >> 3];
    if ((o >> 5) >= rk.words) {
      if (j == 0) atomicOr(dd.err, kErrCapacity);
      continue;
    }
    int32_t k0, k1, k2;
    unpack_key(dd.skey[sl], k0, k1, k2);
    // the neighbour's first probe is in flight while the rank is taken
    uint64_t pk = kEmpty64, cur = kEmpty64;
    uint32_t s = ~0u;
    if (kEnlarge && j != 0) {
      const int32_t n0 = k0 + ((j >> 2) & 1), n1 = k1 + ((j >> 1) & 1), n2 = k2 + (j & 1);
      if (key_packable(n0, n1, n2)) {
        pk = pack_key(n0, n1, n2);
        s = dedup_home(pk, dd.ts);
        cur = dd.skey[s];
      } else {
        atomicOr(dd.err, kErrKeyRange);
      }
    }
    const uint32_t rank = first + rank_below(rk, prefix, o, j);
    if (rank >= (uint32_t)t.T) {
      if (j == 0) atomicOr(dd.err, kErrTableFull);
      continue;
    }
    if (j == 0) {
      slot_block[sl] = (int32_t)rank;
      if (kEnlarge) {
        bcnt[rank] = scnt[sl];
        nbr[8 * (int64_t)rank] = (int32_t)sl;
      }
      place_block(t, rank, k0, k1, k2, dd.err);
    } else if (kEnlarge) {
      if (s != ~0u) {
        s = dedup_finish(pk, s, cur, dd, mask2);
        if (s != ~0u && !((dd.dmask[s >> 5] >> (s & 31u)) & 1u)) dedup_order(s, 8u * rank + (uint32_t)j, dd);
      }
      nbr[8 * (int64_t)rank + j] = (int32_t)s;
    }
  }
}

// Bucket counts and offsets of the first nb blocks and the start of each
// bucket's segment list, from the counts per block (segments << 32 |
// particles): a workgroup adds up the counts before its 1,024 blocks and scans
// its own (nb counts are at most a few hundred KB, in L2). The entries past nb
// are filled by the emission.
__device__ __forceinline__ void counts_scan(const uint64_t* __restrict__ bcnt, int32_t nb, const SortView& sv,
                                            uint32_t* __restrict__ segoff, uint64_t* lds) {
  const int lane = lane_id(), wave = threadIdx.x / kWave;
  const int64_t nchunk = ((int64_t)nb + 1023) / 1024;
  for (int64_t c = blockIdx.x; c < nchunk; c += gridDim.x) {
    uint64_t before = 0;
#pragma unroll 4
    for (int64_t i = 2 * (int64_t)threadIdx.x; i < c * 1024; i += 2 * kThreads) {
      const ulonglong2 q = *reinterpret_cast<const ulonglong2*>(bcnt + i);
      before += q.x + q.y;
    }
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) before += __shfl_xor(before, o, kWave);
    uint64_t v[4], mine = 0;
    const int64_t b0 = c * 1024 + (int64_t)threadIdx.x * 4;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      v[k] = b0 + k < nb ? bcnt[b0 + k] : 0ull;
      mine += v[k];
    }
    uint64_t inc = mine;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const uint64_t u = __shfl_up(inc, o, kWave);
      if (lane >= o) inc += u;
    }
    if (lane == kWave - 1) lds[wave] = inc;
    if (lane == 0) lds[kThreads / kWave + wave] = before;
    __syncthreads();
    uint64_t run = inc - mine;
#pragma unroll
    for (int w = 0; w < kThreads / kWave; ++w) {
      run += w < wave ? lds[w] : 0ull;
      run += lds[kThreads / kWave + w];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (b0 + k < nb) {
        sv.counts[b0 + k] = (int32_t)(uint32_t)v[k];
        sv.offsets[b0 + k] = (int32_t)(uint32_t)run;
        segoff[b0 + k] = (uint32_t)(run >> 32);
      }
      run += v[k];
    }
    __syncthreads();
  }
}

// The last of the build's bookkeeping: the keys[] of every placed block (block
// r probes from its home until it finds the slot holding r), the block count,
// the neighbours' block numbers in place of their slots, the bucket offsets, and
// the grid channels of every block cleared: a launch of its own for that cost 2 us
// of a small substep (77.2 -> 74.8 at 4K particles) and 18 at 16M.
__global__ __launch_bounds__(kThreads) void build_finish_kernel(TableView t, uint32_t* counters, uint32_t* err,
                                                                const int32_t* __restrict__ slot_block, uint32_t ts,
                                                                int32_t* nbr, const uint64_t* __restrict__ bcnt,
                                                                SortView sv, uint32_t* segoff,
                                                                float4* __restrict__ grid, int32_t grid_cap) {
  __shared__ uint64_t lds[2 * (kThreads / kWave)];
  const int64_t na = min((int64_t)counters[kCtrBlocks], (int64_t)t.T);
  const int64_t nb = min((int64_t)counters[kCtrBlocks] + counters[kCtrList], (int64_t)t.T);
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const int64_t i0 = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i0 == 0) {  // nothing in this kernel reads the count
    *t.cnt = (int32_t)nb;
    if (na > sv.cap_blocks) atomicOr(err, kErrCapacity);
  }
  for (int64_t r = i0; r < nb; r += stride) {
    const int32_t k0 = t.active[3 * r], k1 = t.active[3 * r + 1], k2 = t.active[3 * r + 2];
    int32_t s = zpc_home(k0, k1, k2, t.T);
    int32_t probe = 0;
    for (; probe < t.T; ++probe) {
      if (t.indices[s] == (int32_t)r) break;
      s = probe_next(s, t.T);
    }
    if (probe == t.T) {
      atomicOr(err, kErrTableFull);
      continue;
    }
    t.keys[3 * (int64_t)s] = k0;
    t.keys[3 * (int64_t)s + 1] = k1;
    t.keys[3 * (int64_t)s + 2] = k2;
  }
  for (int64_t i = i0; i < 8 * na; i += stride) {
    const uint32_t sl = (uint32_t)nbr[i];
    nbr[i] = sl < ts ? slot_block[sl] : -1;
  }
  const int64_t quads = min(nb, (int64_t)grid_cap) * (kChannels * kBlockCells / 4);
  for (int64_t i = i0; i < quads; i += stride) grid[i] = make_float4(0.f, 0.f, 0.f, 0.f);
  counts_scan(bcnt, (int32_t)min(na, (int64_t)sv.cap_blocks), sv, segoff, lds);
}

// ------------------------------------------------------------ bucket sort
__global__ void zero_u32_kernel(uint32_t* p, int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += stride) p[i] = 0u;
}

// The stand-alone bucket sort's segments: the block each one's key maps to,
// from one table query per segment, counted per block.
template <int kTileItems>
__global__ __launch_bounds__(kThreads) void bucket_kernel(const float* __restrict__ x, int64_t n, float dxinv,
                                                          int blockLen, int offset, float disp, TableView t,
                                                          Segments sg, int32_t cap_blocks, uint32_t* err) {
  constexpr int kTile = kThreads * kTileItems;
  __shared__ TileLds<kTileItems> lds;
  const int64_t ntiles = (n + kTile - 1) / kTile;
  for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const int64_t base = tile * kTile;
    const int live = (int)min((int64_t)kTile, n - base);
    uint64_t pk[kTileItems];
#pragma unroll
    for (int r = 0; r < kTileItems; ++r) {
      const int64_t p = base + (int64_t)r * kThreads + threadIdx.x;
      int32_t k0 = 0, k1 = 0, k2 = 0;
      if (p < n) block_key(x[3 * p], x[3 * p + 1], x[3 * p + 2], dxinv, blockLen, offset, disp, k0, k1, k2);
      // no key the table can hold is out of the packed range
      pk[r] = p < n && key_packable(k0, k1, k2) ? pack_key(k0, k1, k2) : kEmpty64;
    }
    const uint32_t count = tile_segments(pk, live, lds);
    for (uint32_t j = threadIdx.x; j < count; j += kThreads) {
      const uint64_t key = lds.key[j];
      const uint32_t w = lds.where[j];
      int32_t b = -1;
      if (key != kEmpty64) {
        int32_t k0, k1, k2;
        unpack_key(key, k0, k1, k2);
        b = table_find(t, k0, k1, k2);
      }
      if (b < 0) atomicOr(err, kErrMissingBlock);
      if (b >= cap_blocks) {
        atomicOr(err, kErrCapacity);
        b = -1;
      }
      uint32_t local = 0;
      if (b >= 0)
        local = (uint32_t)(atomicAdd((unsigned long long*)&sg.place[b],
                                     (1ull << 32) | (unsigned long long)(w >> 16)) >>
                           32);
      sg.in[base + j] = make_uint2((uint32_t)b, local);
      sg.where[base + j] = w;
    }
    if (threadIdx.x == 0) sg.count[tile] = count;
    __syncthreads();
  }
}

__global__ __launch_bounds__(kThreads) void counts_scan_kernel(const uint64_t* __restrict__ bcnt,
                                                               const int32_t* nblocks, int32_t cap, SortView sv,
                                                               uint32_t* segoff) {
  __shared__ uint64_t lds[2 * (kThreads / kWave)];
  counts_scan(bcnt, min(min(*nblocks, cap), sv.cap_blocks), sv, segoff, lds);
}

// Every segment into its bucket's list: first particle | length << 32. A wave
// takes a tile, a lane a segment. slot_block: the segments name dedup slots;
// null: blocks. Also the counts and offsets past the counted blocks.
__global__ __launch_bounds__(kThreads) void segment_emit_kernel(Segments sg, int64_t n, int32_t tile_size,
                                                                const int32_t* __restrict__ slot_block, uint32_t ts,
                                                                const uint32_t* __restrict__ segoff,
                                                                const int32_t* nblocks, int32_t cap, SortView sv,
                                                                uint64_t* __restrict__ list, uint32_t* counters,
                                                                uint32_t* err) {
  const int lane = lane_id();
  const int64_t ntiles = (n + tile_size - 1) / tile_size;
  const int32_t nb = min(*nblocks, cap);
  {
    const int32_t total = nb > 0 ? sv.offsets[nb - 1] + sv.counts[nb - 1] : 0;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = nb + blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i <= sv.cap_blocks; i += stride) {
      sv.counts[i] = 0;
      sv.offsets[i] = total;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) counters[kCtrSorted] = (uint32_t)n;
  }
  const int64_t nwaves = (int64_t)gridDim.x * (kThreads / kWave);
  constexpr int kAhead = 4;
  for (int64_t tile = (int64_t)blockIdx.x * (kThreads / kWave) + threadIdx.x / kWave; tile < ntiles; tile += nwaves) {
    const int64_t base = tile * tile_size;
    const uint32_t count = min(sg.count[tile], (uint32_t)tile_size);
    for (uint32_t j0 = 0; j0 < count; j0 += kAhead * kWave) {
      uint2 e[kAhead];
      uint32_t w[kAhead], at[kAhead];
      int32_t b[kAhead];
#pragma unroll
      for (int k = 0; k < kAhead; ++k) {
        const uint32_t j = j0 + k * kWave + lane;
        e[k] = make_uint2(~0u, 0u);
        w[k] = 0u;
        if (j < count) {
          e[k] = sg.in[base + j];
          w[k] = sg.where[base + j];
        }
      }
#pragma unroll
      for (int k = 0; k < kAhead; ++k) {
        b[k] = (int32_t)e[k].x;
        if (slot_block) b[k] = e[k].x < ts ? slot_block[e[k].x] : -1;
      }
#pragma unroll
      for (int k = 0; k < kAhead; ++k) {
        const bool ok = b[k] >= 0 && b[k] < nb;
        at[k] = ok ? segoff[b[k]] + e[k].y : ~0u;
        if (slot_block && !ok && w[k] != 0u) atomicOr(err, b[k] < 0 ? kErrMissingBlock : kErrCapacity);
      }
#pragma unroll
      for (int k = 0; k < kAhead; ++k)
        if (at[k] != ~0u && (int64_t)at[k] < n)
          list[at[k]] = (uint64_t)(uint32_t)(base + (w[k] & 0xffffu)) | ((uint64_t)(w[k] >> 16) << 32);
    }
  }
}

// Runs of equal bucket in the last bucket sort (a diagnostic, formed when it is
// asked for): the segments, less those that continue the previous tile's last.
__global__ __launch_bounds__(1024) void count_runs_kernel(Segments sg, int64_t n, int32_t tile_size, uint32_t* runs) {
  __shared__ uint32_t wsum[1024 / kWave];
  const int64_t ntiles = (n + tile_size - 1) / tile_size;
  uint32_t sum = 0;
  for (int64_t tile = threadIdx.x; tile < ntiles; tile += blockDim.x) {
    const int64_t base = tile * tile_size;
    sum += sg.count[tile];
    if (tile > 0 && sg.in[base].x == sg.in[base - tile_size + sg.count[tile - 1] - 1].x) --sum;
  }
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) sum += __shfl_xor(sum, o, kWave);
  if (lane_id() == 0) wsum[threadIdx.x / kWave] = sum;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t total = 0;
    for (int w = 0; w < 1024 / kWave; ++w) total += wsum[w];
    *runs = total;
  }
}

// A bucket's particle indices in particle order, one workgroup per bucket: its
// segments ordered by first particle (they are disjoint), each written as a run.
// Up to 64 segments (particles in or near bucket order): a wave compares every
// segment with every other and needs only the summed lengths before each. Up to
// kPlaceLds: a bitonic sort in LDS and a scan of the lengths. Beyond (thousands
// of particles per bucket, interleaved): a radix sort of the list in global
// memory, 8 bits of the first particle at a time, `alt` the other buffer.
constexpr int kPlaceLds = 2048;  // 16 KB, eight workgroups per CU

// first, step: this thread's share of the segment
__device__ __forceinline__ void write_segment(int32_t* __restrict__ indices, int64_t n, int64_t at, uint32_t start,
                                              uint32_t len, uint32_t first, uint32_t step) {
  for (uint32_t q = first; q < len && at + q < n; q += step) indices[at + q] = (int32_t)(start + q);
}

// exclusive scan of one value per thread across the workgroup
__device__ __forceinline__ uint32_t group_scan(uint32_t v, uint32_t* lds, uint32_t& total) {
  const int lane = lane_id(), wave = threadIdx.x / kWave;
  uint32_t inc = v;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const uint32_t u = __shfl_up(inc, o, kWave);
    if (lane >= o) inc += u;
  }
  if (lane == kWave - 1) lds[wave] = inc;
  __syncthreads();
  uint32_t before = 0;
  total = 0;
#pragma unroll
  for (int w = 0; w < kThreads / kWave; ++w) {
    before += w < wave ? lds[w] : 0u;
    total += lds[w];
  }
  __syncthreads();
  return before + inc - v;
}

__global__ __launch_bounds__(kThreads) void segment_place_kernel(const uint64_t* __restrict__ bcnt,
                                                                 const uint32_t* __restrict__ segoff,
                                                                 const int32_t* nblocks, int32_t cap, SortView sv,
                                                                 int64_t n, int32_t bits, uint64_t* list,
                                                                 uint64_t* alt) {
  __shared__ uint64_t seg[kPlaceLds];
  __shared__ uint32_t hist[256], lds[kThreads / kWave];
  const int lane = lane_id(), wave = threadIdx.x / kWave;
  const int32_t nb = min(min(*nblocks, cap), sv.cap_blocks);
  for (int32_t b = blockIdx.x; b < nb; b += gridDim.x) {
    const uint64_t both = bcnt[b];
    const uint32_t R = (uint32_t)(both >> 32), cnt = (uint32_t)both;
    const int64_t off = sv.offsets[b];
    const uint32_t s0 = segoff[b];
    if (R == 0 || (int64_t)s0 + R > n) continue;
    if (R <= (uint32_t)kWave) {
      // every wave orders the list for itself; short segments go to one wave
      // each, long ones to the whole workgroup
      const uint64_t me = (uint32_t)lane < R ? list[s0 + lane] : ~0ull;
      const uint32_t start = (uint32_t)me, len = (uint32_t)lane < R ? (uint32_t)(me >> 32) : 0u;
      uint32_t before = 0;
      for (uint32_t k = 0; k < R; ++k) {
        const uint32_t ks = (uint32_t)__builtin_amdgcn_readlane((int)start, (int)k);
        const uint32_t kl = (uint32_t)__builtin_amdgcn_readlane((int)len, (int)k);
        before += ks < start ? kl : 0u;
      }
      const bool wide = cnt >= 64u * R;
      for (uint32_t k = wide ? 0 : wave; k < R; k += wide ? 1 : kThreads / kWave) {
        const uint32_t ks = (uint32_t)__builtin_amdgcn_readlane((int)start, (int)k);
        const uint32_t kl = (uint32_t)__builtin_amdgcn_readlane((int)len, (int)k);
        const uint32_t kb = (uint32_t)__builtin_amdgcn_readlane((int)before, (int)k);
        write_segment(sv.indices, n, off + kb, ks, kl, wide ? threadIdx.x : lane, wide ? kThreads : kWave);
      }
      continue;
    }
    if (R <= (uint32_t)kPlaceLds) {
      uint32_t P = 128;
      while (P < R) P <<= 1;
      // keyed by the first particle in the high word
      for (uint32_t i = threadIdx.x; i < P; i += kThreads) {
        const uint64_t v = i < R ? list[s0 + i] : ~0ull;
        seg[i] = (v << 32) | (v >> 32);
      }
      __syncthreads();
      for (uint32_t k = 2; k <= P; k <<= 1) {
        for (uint32_t j = k >> 1; j > 0; j >>= 1) {
          for (uint32_t i = threadIdx.x; i < P / 2; i += kThreads) {
            const uint32_t lo = 2 * i - (i & (j - 1)), hi = lo + j;
            const uint64_t a = seg[lo], c = seg[hi];
            if ((a > c) == ((lo & k) == 0)) {
              seg[lo] = c;
              seg[hi] = a;
            }
          }
          __syncthreads();
        }
      }
      uint32_t carry = 0;
      const bool runs = cnt >= 8u * R;  // long segments: a wave writes each
      for (uint32_t base = 0; base < R; base += kThreads) {  // uniform across the workgroup
        const uint32_t i = base + threadIdx.x;
        const uint64_t v = i < R ? seg[i] : 0ull;
        const uint32_t start = (uint32_t)(v >> 32), len = (uint32_t)v;
        uint32_t total;
        const uint32_t at = carry + group_scan(len, lds, total);
        if (runs) {
          for (int k = 0; k < kWave; ++k) {  // len 0 past the list
            const uint32_t kl = (uint32_t)__builtin_amdgcn_readlane((int)len, k);
            write_segment(sv.indices, n, off + (uint32_t)__builtin_amdgcn_readlane((int)at, k),
                          (uint32_t)__builtin_amdgcn_readlane((int)start, k), kl, lane, kWave);
          }
        } else {
          for (uint32_t q = 0; q < len && off + at + q < n; ++q) sv.indices[off + at + q] = (int32_t)(start + q);
        }
        carry += total;
      }
      __syncthreads();
      continue;
    }
    uint64_t *from = list + s0, *to = alt + s0;
    for (int shift = 0; shift < bits; shift += 8) {
      for (int i = threadIdx.x; i < 256; i += kThreads) hist[i] = 0u;
      __syncthreads();
      for (uint32_t i = threadIdx.x; i < R; i += kThreads) atomicAdd(&hist[((uint32_t)from[i] >> shift) & 255u], 1u);
      __syncthreads();
      uint32_t total;
      const uint32_t first = group_scan(hist[threadIdx.x], lds, total);
      hist[threadIdx.x] = first;
      __syncthreads();
      for (uint32_t base = 0; base < R; base += kWave) {  // one wave at a time keeps the pass stable
        if (wave == 0) {
          const uint32_t i = base + lane;
          const bool live = i < R;
          const uint64_t v = live ? from[i] : 0ull;
          const uint32_t d = ((uint32_t)v >> shift) & 255u;
          uint64_t peers = ballot(live);
#pragma unroll
          for (int bit = 0; bit < 8; ++bit) {
            const bool on = (d >> bit) & 1u;
            const uint64_t m = ballot(on);
            peers &= on ? m : ~m;
          }
          const uint32_t below = (uint32_t)__popcll(peers & lanemask_lt());
          const uint32_t at = live ? hist[d] + below : 0u;
          wave_lds_barrier();
          if (live && below == 0) hist[d] += (uint32_t)__popcll(peers);
          wave_lds_barrier();
          if (live) to[at] = v;
        }
      }
      __threadfence_block();
      __syncthreads();
      uint64_t* q = from;
      from = to;
      to = q;
    }
    uint32_t carry = 0;
    for (uint32_t base = 0; base < R; base += kThreads) {
      const uint32_t i = base + threadIdx.x;
      const uint64_t v = i < R ? from[i] : 0ull;
      const uint32_t start = (uint32_t)v, len = (uint32_t)(v >> 32);
      uint32_t total;
      const uint32_t at = carry + group_scan(len, lds, total);
      for (uint32_t q = 0; q < len && off + at + q < n; ++q) sv.indices[off + at + q] = (int32_t)(start + q);
      carry += total;
    }
    __syncthreads();
  }
}

// Neighbour blocks of every active block: nbr[8 b + d] = index of
// activeKeys[b] + (d>>2&1, d>>1&1, d&1), -1 where absent.
__global__ void neighbours_kernel(TableView t, int32_t* __restrict__ nbr, uint32_t cap) {
  const int64_t total = 8ll * (int64_t)min((uint32_t)*t.cnt, cap);
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total; i += stride) {
    const int64_t b = i >> 3;
    const int d = (int)(i & 7);
    nbr[i] = table_find(t, t.active[3 * b] + ((d >> 2) & 1), t.active[3 * b + 1] + ((d >> 1) & 1),
                        t.active[3 * b + 2] + (d & 1));
  }
}

int bits_for(uint64_t maxval) {
  int b = 0;
  while (b < 32 && (maxval >> b) != 0) ++b;
  return b;
}

Dedup dedup_of(const Workspace& ws) { return Dedup{ws.skey, ws.sorder, ws.ts_cap, ws.err, ws.dmask}; }

// words of the first-occurrence bitmap for orders below order_bound (orders
// beyond the bitmap are reported by assign)
uint64_t bitmap_words(const Workspace& ws, uint64_t order_bound) {
  const uint64_t words = order_bound / 32 + 1;
  return words > ws.bm_words ? ws.bm_words : words;
}

// dedup entries -> ranked, placed and keyed table entries (shared tail of
// activation and enlargement); the bitmap was cleared with the dedup scratch
hipError_t finish_insertion(const TableView& t, Workspace& ws, uint64_t order_bound, hipStream_t s) {
  const uint64_t words = bitmap_words(ws, order_bound);
  collect_new_kernel<<<kCollectGroups, kThreads, 0, s>>>(ws.skey, ws.sorder, ws.dmask, ws.ts_cap, t, ws.counters,
                                                         ws.la_key,
                                                         ws.la_val, ws.list_cap, ws.err, ws.bitmap, (uint32_t)words);
  hipError_t e = exclusive_scan_popc_u32(ws.bitmap, ws.bm_prefix, (uint32_t)words, ws.scan_tmp, s);
  if (e != hipSuccess) return e;
  const int gl = groups_for(ws.list_cap, kThreads);
  assign_kernel<<<gl, kThreads, 0, s>>>(ws.la_key, ws.la_val, ws.bitmap, ws.bm_prefix, (uint32_t)words, ws.skey, t,
                                        ws.counters, ws.list_cap, ws.err);
  fill_keys_kernel<<<gl, kThreads, 0, s>>>(t, ws.counters, ws.list_cap, ws.err);
  return hipGetLastError();
}

}  // namespace

hipError_t table_clear(const TableView& t, Workspace& ws, hipStream_t s) {
  const int64_t m = (int64_t)t.T > (int64_t)ws.ts_cap ? t.T : ws.ts_cap;
  clear_table_kernel<<<groups_for(m, kThreads), kThreads, 0, s>>>(t, ws.skey, ws.sorder, ws.dmask, ws.ts_cap,
                                                                   ws.counters);
  return hipGetLastError();
}

namespace {

bool wide_tiles(int64_t n) { return n >= (int64_t)1 << 21; }
int tile_size(int64_t n) { return kThreads * (wide_tiles(n) ? kWideTile : kTightTile); }
// workgroups of a kernel that strides over the tiles: at most eight per CU of the 256 over wide ones
int tile_groups(int64_t n) {
  const int g = groups_for(n, tile_size(n));
  return wide_tiles(n) && g > 2048 ? 2048 : g;
}

// the activation's insertion pass (a batch, ss, only in the substep's build, which records the segments)
template <bool kSegs>
void launch_activate(Workspace& ws, const float* x, int64_t n, float dx, int blockLen, int offset, float disp,
                     const Segments& sg, hipStream_t s, const SceneSet* ss) {
  const float dxinv = (float)1.0 / dx;
  const int g = tile_groups(n);
  const bool multi = ss && ss->n > 0;
  const SceneSet sset = multi ? *ss : SceneSet{};
  auto launch = [&](auto kernel) {
    kernel<<<g, kThreads, 0, s>>>(x, n, dxinv, blockLen, offset, disp, dedup_of(ws), sg, sset);
  };
  if constexpr (kSegs) {
    if (multi) {
      if (wide_tiles(n))
        launch(activate_kernel<true, true, kWideTile>);
      else
        launch(activate_kernel<true, true, kTightTile>);
      return;
    }
  }
  if (wide_tiles(n))
    launch(activate_kernel<false, kSegs, kWideTile>);
  else
    launch(activate_kernel<false, kSegs, kTightTile>);
}

Segments segments_of(const Workspace& ws, uint64_t* place) {
  Segments sg;
  sg.count = ws.seg_count;
  sg.in = ws.seg_in;
  sg.where = ws.seg_where;
  sg.place = place;
  return sg;
}

}  // namespace

hipError_t table_activate(const TableView& t, Workspace& ws, const float* x, int64_t n, float dx,
                          int blockLen, int offset, float disp, hipStream_t s) {
  if (blockLen <= 0) return hipErrorInvalidValue;
  const uint64_t order_bound = (uint64_t)(n > 0 ? n : 1);
  clear_scratch_kernel<<<groups_for(ws.ts_cap, kThreads), kThreads, 0, s>>>(
      ws.skey, ws.sorder, ws.dmask, ws.ts_cap, t.cnt, ws.counters, ws.bitmap, (int64_t)bitmap_words(ws, order_bound));
  if (n > 0) launch_activate<false>(ws, x, n, dx, blockLen, offset, disp, Segments{}, s, nullptr);
  return finish_insertion(t, ws, order_bound, s);
}

hipError_t table_enlarge(const TableView& t, Workspace& ws, const int32_t lo[3], const int32_t hi[3],
                         int32_t n0_cap, hipStream_t s) {
  const int32_t e0 = hi[0] - lo[0], e1 = hi[1] - lo[1], e2 = hi[2] - lo[2];
  if (e0 <= 0 || e1 <= 0 || e2 <= 0) return hipSuccess;
  const int64_t total_cap = (int64_t)n0_cap * e0 * e1 * e2;
  const uint64_t order_bound = (uint64_t)(total_cap > 0 ? total_cap : 1);
  clear_scratch_kernel<<<groups_for(ws.ts_cap, kThreads), kThreads, 0, s>>>(
      ws.skey, ws.sorder, ws.dmask, ws.ts_cap, t.cnt, ws.counters, ws.bitmap, (int64_t)bitmap_words(ws, order_bound));
  enlarge_kernel<<<groups_for(total_cap, kThreads), kThreads, 0, s>>>(t.active, ws.counters, lo[0], lo[1], lo[2],
                                                                       e0, e1, e2, dedup_of(ws));
  return finish_insertion(t, ws, order_bound, s);
}

hipError_t block_neighbours(const TableView& t, Workspace& ws, hipStream_t s) {
  const int g = groups_for(8ll * ws.ts_cap, kThreads);
  neighbours_kernel<<<g < 1024 ? g : 1024, kThreads, 0, s>>>(t, ws.nbr, ws.ts_cap);
  return hipGetLastError();
}

hipError_t table_query(const TableView& t, const int32_t* keys, int64_t n, int32_t* out, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  query_kernel<<<groups_for(n, kThreads), kThreads, 0, s>>>(t, keys, n, out);
  return hipGetLastError();
}

namespace {

// segments counted per block (bcnt) and scanned (offsets, segoff): the lists
// and the buckets' indices. slot_block as in segment_emit_kernel. *nblocks may
// exceed T where a larger scratch took more keys than the table (reported as
// full): only the first T blocks were numbered, counted and scanned.
hipError_t place_segments(const TableView& t, Workspace& ws, int64_t n, const int32_t* slot_block,
                          const int32_t* nblocks, const SortView& out, hipStream_t s) {
  const int64_t tiles = (n + tile_size(n) - 1) / tile_size(n);
  int32_t cap = out.cap_blocks < (int32_t)ws.ts_cap ? out.cap_blocks : (int32_t)ws.ts_cap;
  cap = cap < t.T ? cap : t.T;
  const int ge = groups_for(tiles * kWave, kThreads), gc = groups_for((int64_t)cap + 1, kThreads * 4);
  segment_emit_kernel<<<ge > gc ? ge : gc, kThreads, 0, s>>>(segments_of(ws, nullptr), n, tile_size(n), slot_block, ws.ts_cap,
                                                             ws.segoff, nblocks, cap, out, ws.seg_list,
                                                             ws.counters, ws.err);
  if (n <= 0) return hipGetLastError();
  const int g = cap < 32768 ? cap : 32768;
  segment_place_kernel<<<g, kThreads, 0, s>>>(ws.bcnt, ws.segoff, nblocks, cap, out, n, bits_for((uint64_t)n - 1),
                                              ws.seg_list, ws.seg_alt);
  return hipGetLastError();
}

}  // namespace

hipError_t count_runs(Workspace& ws, int64_t n, hipStream_t s) {
  count_runs_kernel<<<1, 1024, 0, s>>>(segments_of(ws, nullptr), n, tile_size(n), ws.counters + kCtrRuns);
  return hipGetLastError();
}

hipError_t bucket_sort(const TableView& t, Workspace& ws, const float* x, int64_t n, float dx, int blockLen,
                       int offset, float disp, const SortView& out, hipStream_t s) {
  if (n > (int64_t)ws.n_cap) return hipErrorInvalidValue;
  const float dxinv = (float)1.0 / dx;
  zero_u32_kernel<<<groups_for(2ll * ws.ts_cap, kThreads) < 2048 ? groups_for(2ll * ws.ts_cap, kThreads) : 2048,
                    kThreads, 0, s>>>((uint32_t*)ws.bcnt, 2ll * ws.ts_cap);
  const int32_t cap = out.cap_blocks < (int32_t)ws.ts_cap ? out.cap_blocks : (int32_t)ws.ts_cap;
  if (n > 0 && wide_tiles(n))
    bucket_kernel<kWideTile><<<tile_groups(n), kThreads, 0, s>>>(x, n, dxinv, blockLen, offset, disp, t,
                                                                 segments_of(ws, ws.bcnt), cap, ws.err);
  else if (n > 0)
    bucket_kernel<kTightTile><<<tile_groups(n), kThreads, 0, s>>>(x, n, dxinv, blockLen, offset, disp, t,
                                                                  segments_of(ws, ws.bcnt), cap, ws.err);
  const int gs = (cap + 1023) / 1024;
  counts_scan_kernel<<<gs < 1024 ? gs : 1024, kThreads, 0, s>>>(ws.bcnt, t.cnt, cap, out, ws.segoff);
  return place_segments(t, ws, n, nullptr, t.cnt, out, s);
}

// ------------------------------------------------------- the substep's build
namespace {

// orders of the particles' keys are particle indices, those of the enlargement
// candidates (8 b + j) lie below T while the particles' blocks fill at most T / 8
Ranks ranks_of(uint32_t* bitmap, uint32_t* c1, uint64_t orders) {
  Ranks r;
  r.bitmap = bitmap;
  r.c1 = c1;
  r.words = (uint32_t)(orders / 32 + 1);
  while ((((uint64_t)r.words * 32) >> r.shift) + 1 > (uint64_t)kRankGroups) ++r.shift;
  r.groups = (int32_t)((((uint64_t)r.words * 32) >> r.shift) + 1);
  return r;
}
Ranks ranks_a(const Workspace& ws, int64_t n) { return ranks_of(ws.bitmap, ws.rank_a, (uint64_t)(n > 0 ? n : 1)); }
Ranks ranks_b(const Workspace& ws, const TableView& t) {
  return ranks_of(ws.bitmap_b, ws.rank_b, 8ull * (uint64_t)(t.T / 8 > 0 ? t.T / 8 : 1));
}
int64_t padded(int64_t groups) { return (groups + 3) & ~(int64_t)3; }
// a workgroup of the numbering reads all of c1: few of them where there is much
// of it (the LDS it fills also bounds them to two per CU then)
int number_groups(const Ranks& r, uint32_t ts, int64_t most) {
  const int g = groups_for(8ll * ts, kThreads);
  const int cap = (int)(r.groups > 4096 ? 512 : most);
  return g < cap ? g : cap;
}
int few(int64_t n, int most) {
  const int g = groups_for(n, kThreads);
  return g < most ? g : most;
}

}  // namespace

size_t rank_scratch_words() { return kRankGroups + 4; }

hipError_t build_clear(const TableView& t, Workspace& ws, int64_t n, hipStream_t s) {
  ClearList c;
  int64_t most = 0;
  auto add = [&](void* p, int64_t words, uint32_t v) {
    c.p[c.count] = (uint32_t*)p;
    c.n[c.count] = words;
    c.v[c.count++] = v;
    most = words > most ? words : most;
  };
  const int64_t ts = ws.ts_cap;
  add(t.keys, 3ll * t.T, (uint32_t)kKeySentinel);
  add(t.indices, t.T, 0xffffffffu);
  add(t.status, t.T, 0xffffffffu);
  add(ws.skey, 2 * ts, 0xffffffffu);
  add(ws.sorder, ts, 0xffffffffu);
  add(ws.scnt, 2 * ts, 0u);
  add(ws.dmask, 2 * (ts / 32 + 1), 0u);  // both masks
  add(ws.bitmap, ranks_a(ws, n).words, 0u);
  add(ws.rank_a, padded(ranks_a(ws, n).groups), 0u);
  add(ws.bitmap_b, ranks_b(ws, t).words, 0u);
  add(ws.rank_b, padded(ranks_b(ws, t).groups), 0u);
  build_clear_kernel<<<few(most / 4 + 1, 4096), kThreads, 0, s>>>(c, t, ws.counters);
  return hipGetLastError();
}

hipError_t build_activate(const TableView& t, Workspace& ws, const float* x, int64_t n, float dx, hipStream_t s,
                          const SceneSet* ss) {
  if (n > (int64_t)ws.n_cap) return hipErrorInvalidValue;
  if (n > 0) launch_activate<true>(ws, x, n, dx, 4, -2, 0.5f, segments_of(ws, ws.scnt), s, ss);
  const uint32_t nw = (ws.ts_cap + 31u) / 32u;
  build_collect_kernel<<<(int)((nw + kWave - 1) / kWave), kThreads, 0, s>>>(
      ws.dmask, nw, ws.sorder, ranks_a(ws, n), ws.counters + kCtrBlocks, ws.la_key, ws.la_val);
  return hipGetLastError();
}

hipError_t build_enlarge(const TableView& t, Workspace& ws, int64_t n, const SortView& sv, float* grid,
                         int32_t grid_cap, hipStream_t s) {
  uint32_t* mask2 = ws.dmask + (ws.ts_cap / 32 + 1);
  const Ranks ra = ranks_a(ws, n), rb = ranks_b(ws, t);
  build_number_kernel<true><<<number_groups(ra, ws.ts_cap, 1024), kThreads, 4 * padded(ra.groups), s>>>(
      ws.counters + kCtrBlocks, nullptr, ws.la_key, ws.la_val, ra, t, dedup_of(ws), mask2, ws.slot_block, ws.scnt,
      ws.bcnt, ws.nbr);
  const uint32_t nw = (ws.ts_cap + 31u) / 32u;
  build_collect_kernel<<<(int)((nw + kWave - 1) / kWave), kThreads, 0, s>>>(
      mask2, nw, ws.sorder, rb, ws.counters + kCtrList, ws.lb_key, ws.lb_val);
  build_number_kernel<false><<<number_groups(rb, ws.ts_cap, 256), kThreads, 4 * padded(rb.groups), s>>>(
      ws.counters + kCtrList, ws.counters + kCtrBlocks, ws.lb_key, ws.lb_val, rb, t, dedup_of(ws), mask2,
      ws.slot_block, ws.scnt, ws.bcnt, ws.nbr);
  build_finish_kernel<<<few(ws.ts_cap, 2048), kThreads, 0, s>>>(t, ws.counters, ws.err, ws.slot_block, ws.ts_cap,
                                                                ws.nbr, ws.bcnt, sv, ws.segoff,
                                                                reinterpret_cast<float4*>(grid), grid_cap);
  return hipGetLastError();
}

hipError_t build_place(const TableView& t, Workspace& ws, int64_t n, const SortView& out, hipStream_t s) {
  return place_segments(t, ws, n, ws.slot_block, reinterpret_cast<const int32_t*>(ws.counters + kCtrBlocks), out, s);
}

}  // namespace zsmpm
