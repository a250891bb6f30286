// P2G, grid update and G2P for the gfx950 MLS-MPM substep.
//
// Work is organised per particle bucket: the 4^3 block a particle's key maps
// to (SparsityOp.hpp:72-77 with blockLen 4, offset -2, displacement 0.5). A
// particle with key cell c has its quadratic stencil base at c+1 (c or c+2
// only at rounding ties), so the stencils of a bucket whose key block starts
// at cell 4b lie in nodes [4b, 4b+8)^3, all inside the 2x2x2 blocks
// b + {0,1}^3 that EnlargeSparsity{0..2} activates.
//
// P2G. On gfx950 LDS float atomics (ds_add_f32) retire about one lane every
// three clocks, roughly 30x slower than a plain LDS read-modify-write, so the
// scatter avoids them:
//   A  every lane takes one particle (full occupancy): stress (3x3 SVD and
//      the constitutive model), then an affine record -- mass, B and dx*A with
//      node value(o) = W(o) (B + dx A o) -- kept in LDS, and a base-cell id
//      (one of the 64 main cells [4b+1, 4b+5)^3, or "overflow");
//   B  a counting sort of the chunk by base cell (LDS integer atomics);
//   C  lane l of a wave sums its share of main cell l's particles in
//      registers, one x-slab of the 27-node stencil at a time, and adds the
//      node sums to the wave's own 6^3 node arena with plain float4
//      read-modify-writes (the 64 lanes address 64 different nodes);
//      overflow particles scatter with global atomics;
//   then the four wave arenas are summed and flushed with one global float
//   atomic per touched node and channel (zpc's CUDA P2G issues 189 global
//   atomics per particle, cuda/simulation/transfer/P2G.hpp:98-115).
// The substep's P2G adds the force term to the momentum channels (the
// explicit driver's v = (mv + rhs)/m convention) and the grid carries
// {m, mv + rhs}; the stage-wise P2G keeps the rhs channels 4..6 as zpc lays
// them out, from two launches: momentum only, then the force only.
//
// G2P stages the 8^3 node velocities of a bucket in LDS (float4 per node) and
// gathers from there.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "zsmpm_device.hpp"
#include "zsmpm_internal.hpp"

namespace zsmpm {

namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWave;
constexpr int kMainCells = 64;    // base cells [4b+1, 4b+5)^3
constexpr int kArena6 = 216;      // nodes [4b+1, 4b+7)^3
constexpr int kArena8 = 512;      // nodes [4b, 4b+8)^3
// G2P velocity stage: node (r0, r1, r2) at r0*73 + r1*9 + r2, so a float4
// node's LDS bank group is (r0 + r1 + r2) mod 8 rather than r2 alone
constexpr int kVelSY = 9, kVelSX = 73, kVelNodes = 7 * kVelSX + 7 * kVelSY + 8;
__device__ __forceinline__ int vel_at(int r0, int r1, int r2) { return r0 * kVelSX + r1 * kVelSY + r2; }
// one workgroup per bucket. Two waves: a bucket's 8 staged velocity blocks
// serve ~3 rounds of 64 particles per wave, and eight such workgroups per CU
// (the register limit, 4 waves per SIMD) keep more buckets' loads in flight
// than four workgroups of four waves (0.82 -> 0.79 ms at 16M particles)
constexpr int kG2PThreads = 128;
// G2P of a small scene: as many waves as a full bucket has rounds of rows. With
// two, a bucket's rounds ran one after another while most CUs idled: substep
// 77.2 -> 68.8 us at 64K particles of 8 per cell, 91.0 -> 87.0 at 262K (729
// buckets). Sparse buckets leave the extra waves idle and many buckets fill the
// card with two: 115 -> 124 at 250K of 2 per cell (2,200 buckets), 81.5 -> 89.8
// at 64K of 1 (1,331). The line is on the buckets' capacity (wide_buckets); below
// it bodies of 1 particle per cell lose most, 69.8 -> 72.9 at 27K, and dense ones
// gain most, 241 -> 176 at 512K of 64.
constexpr int kG2PWide = 512;
constexpr int kG2PWideBuckets = 2048;
constexpr int kP2GThreads = 256;  // one workgroup per bucket
constexpr int kP2GWaves = kP2GThreads / kWave;
// Launch tiles the autotuner chooses between. P2G tile 0: four waves and
// chunks of Rec::kChunk particles (a whole bucket of up to 576, three
// workgroups per CU); tile 1: two waves and chunks of 256 (six workgroups per
// CU, for sparser buckets). G2P: 128 or 256 threads per bucket.
//
// kWideTile, P2G of a small scene: eight waves per bucket (records and scatter
// in about one round each, no serial chain of three). At 128 registers two such
// workgroups fit a CU, so it pays while every bucket is resident at once, up to
// 512: substep 67.1 -> 64.7 us at 4K particles, 70.9 -> 68.9 at 64K, 88.3 -> 82.3
// at 128K of 16 per cell, 224 -> 170 at 262K of 64 (73.8 -> 74.0 at 97K and 74.2 ->
// 75.0 at 120K of 8, some 350 buckets); past the line 89.4 -> 101 at 64K of 1 per
// cell (1,331 buckets). Nine waves at 144 registers, one workgroup
// per CU, cost more from 256 buckets on (72.5 -> 76.2 at 72K). Splitting a bucket
// over four workgroups instead gained 3 us at 4K and lost 15 at 64K.
constexpr int kP2GWideBuckets = 1024;
constexpr int kWideTile = 2, kWideP2GThreads = 512;
constexpr int p2g_threads(int tile) { return tile == kWideTile ? kWideP2GThreads : tile == 1 ? 128 : kP2GThreads; }
constexpr int p2g_chunk(int tile, int fold_chunk) { return tile == 1 ? 256 : fold_chunk; }

inline int groups_for(int64_t n, int threads) {
  int64_t g = (n + threads - 1) / threads;
  if (g < 1) g = 1;
  if (g > 65535 * 8) g = 65535 * 8;
  return (int)g;
}

__device__ __forceinline__ int64_t grid_at(int32_t b, int ch, int cell) {
  return ((int64_t)b * kChannels + ch) * kBlockCells + cell;
}

// node r in [0, 8)^3 relative to 4b -> (neighbour block of b + {0,1}^3, cell)
__device__ __forceinline__ void node_home(int r0, int r1, int r2, int& nb, int& cell) {
  nb = ((r0 >> 2) << 2) | ((r1 >> 2) << 1) | (r2 >> 2);
  cell = ((r0 & 3) << 4) | ((r1 & 3) << 2) | (r2 & 3);
}

__global__ void grid_clear_kernel(float* grid, const int32_t* nblocks, int32_t cap) {
  const int32_t nb = min(*nblocks, cap);
  const int64_t total = (int64_t)nb * kChannels * kBlockCells / 4;
  float4* g4 = reinterpret_cast<float4*>(grid);
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total; i += stride)
    g4[i] = make_float4(0.f, 0.f, 0.f, 0.f);
}

// active block count, clipped to what the grid and bucket arrays hold
__device__ __forceinline__ int32_t bounded_blocks(const TableView& t, const SortView& sv, int32_t grid_cap,
                                                  uint32_t* err) {
  const int32_t nb = *t.cnt;
  const int32_t cap = min(grid_cap, sv.cap_blocks);
  if (nb > cap) {
    if (blockIdx.x == 0 && threadIdx.x == 0) atomicOr(err, kErrCapacity);
    return cap;
  }
  return nb;
}

// neighbour blocks key + (d>>2&1, d>>1&1, d&1) of bucket b, from the
// per-substep neighbour table
__device__ __forceinline__ void load_neighbours(const int32_t* __restrict__ nbr_tab, int32_t b, int32_t* nbr,
                                                uint32_t* err) {
  if (threadIdx.x < 8) {
    const int32_t r = nbr_tab[8 * (int64_t)b + threadIdx.x];
    nbr[threadIdx.x] = r;
    if (r < 0) atomicOr(err, kErrMissingBlock);
  }
}

// Main base cell (i, j, k) in [0,4)^3 <-> lane of the scatter rounds. Lane
// bits are (k0, k1, i0, j0, i1, j1): the 8 consecutive lanes one LDS b128
// access serves together cover 4 values of k and 2 of i, 36 nodes apart in
// the 6^3 arena (36 = 4 mod 8), so they fall in 8 distinct bank groups.
__device__ __forceinline__ int cell_lane(int i, int j, int k) {
  return k | ((i & 1) << 2) | ((j & 1) << 3) | ((i >> 1) << 4) | ((j >> 1) << 5);
}
__device__ __forceinline__ void lane_cell(int l, int& i, int& j, int& k) {
  k = l & 3;
  i = ((l >> 2) & 1) | (((l >> 4) & 1) << 1);
  j = ((l >> 3) & 1) | (((l >> 5) & 1) << 1);
}

// The quadratic B-spline's argument (quadratic_bspline_weights,
// math/curve/InterpolationKernel.hpp:95-130): the local position l = X -
// floor(X - 0.5) less floor(l - 0.5). That floor is 0 for X >= 0.5, where l is
// exact; at negative X the rounding of X - 0.5 can leave l just below 0.5 (X =
// -127.50001 has base -128) and the floor is -1, as in make_arena. It is taken
// once per record, not in the scatter's three passes.
__device__ __forceinline__ float bspline_arg(float l) {
#pragma clang fp contract(off)
  return l - (float)(int32_t)floorf(l - 0.5f);
}

// its weights on the nodes base .. base + 2
__device__ __forceinline__ void bspline_w(float d0, float (&w)[3]) {
#pragma clang fp contract(off)
  w[0] = 0.5f * (1.5f - d0) * (1.5f - d0);
  const float d1 = d0 - 1.0f;
  w[1] = 0.75f - d1 * d1;
  const float zz = 0.5f + d1;
  w[2] = 0.5f * zz * zz;
}

// Node weights of the particle -> cell -> node kernel (P2C2GTransfer,
// simulation/transfer/P2C2G.hpp:143-147 and the 1/8 of :164; G2C2PTransfer,
// G2C2P.hpp:81-84, :112-119): the tent weights 1 - t and t to the two cell
// centres within reach (t = l - 0.5 from the local position l in [0.5, 1.5)),
// each spread evenly over its cell's corners, per axis (1 - t) / 2, 1 / 2 and
// t / 2 on the nodes base .. base + 2.
__device__ __forceinline__ void cell_w(float l, float (&w)[3]) {
#pragma clang fp contract(off)
  const float t = l - 0.5f;
  w[0] = (1.f - t) * 0.5f;
  w[1] = 0.5f;
  w[2] = t * 0.5f;
}

// weights from a record's l: the local position (cell kernel) or bspline_arg of it
template <bool kCell>
__device__ __forceinline__ void stencil_w(float l, float (&w)[3]) {
  if constexpr (kCell)
    cell_w(l, w);
  else
    bspline_w(l, w);
}

// Per-axis factor of the cell kernel (P2C2G.hpp:86-90, G2C2P.hpp:235-238):
// Dinv = 2 / (dx^2 - 2 Xrel^2), Xrel = x - floor(x dx_inv + 0.5) dx the offset
// from the nearest node; 1 / Dinv is the kernel's second moment on that axis.
__device__ __forceinline__ void cell_dinv(const float (&x)[3], float dx, float dx_inv, float (&Dinv)[3]) {
#pragma clang fp contract(off)
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const float xr = x[d] - (float)(int32_t)floorf(x[d] * dx_inv + 0.5f) * dx;
    Dinv[d] = 2.f / (dx * dx - 2.f * xr * xr);
  }
}

// Record layout (float4 units): q0 = (m, B0, B1, B2), q1 = (l0, l1, l2, A8),
// q2 = A0..A3, q3 = A4..A7 with A column-major (A[d + 3e]) already times dx; l
// is the argument of stencil_w.
struct Rec {
  static constexpr int kQuads = 4;
  // particles staged per pass. 576 (nine waves) holds a whole bucket at 8
  // particles per cell (up to 562 in the 16M sand column; 39% of its buckets
  // exceed 512 and took a nearly empty second pass, 0.80 -> 0.765 ms) and
  // keeps the workgroup at 53 KB of LDS, three per CU
  static constexpr int kChunk = 576;
};

// Per-particle constitutive part of P2G (P2G.hpp:57-100): vol P F^T from the
// stored F (fixed-corotated or the Drucker-Prager return mapping, which
// writes logJp back). Particles in array order, 64 consecutive per wave, so
// the results leave as 16-byte vectors.
// kKind: 0 fixed-corotated, 1 Drucker-Prager, 2 each particle its scene's
// model (a batch, ss; only where some scene has the FP64 SVD on). kGap: the
// model has the FP64 SVD on; its code stays out of the other instances, which
// it held to three waves per SIMD
template <int kKind, bool kGap>
__global__ __launch_bounds__(kThreads) void stress_kernel(Model m, ParticlesView ps, float* __restrict__ contrib,
                                                          uint32_t* counters, SceneSet ss) {
  __shared__ float4 stage4[kWaves][stage_floats(9) / 4];
  __shared__ int64_t sfirst[kKind == 2 ? kMaxScenes + 1 : 1];
  const int wave = uniform((int32_t)(threadIdx.x / kWave)), lane = lane_id();
  float* stage = reinterpret_cast<float*>(stage4[wave]);
  const int64_t nwaves = (int64_t)gridDim.x * kWaves;
  uint32_t fp64_used = 0;
  if constexpr (kKind == 2) {
    for (int i = threadIdx.x; i <= ss.n; i += kThreads) sfirst[i] = ss.first[i];
    __syncthreads();
  }
  // The next group's F row and logJp are in flight while this group's SVD runs
  // (stress pass 0.70 -> 0.67 ms beside the sparsity stages at 16M particles).
  // Two groups ahead made the pass faster still (0.61 ms) but took enough of the
  // machine to slow the bucket sort beside it by more. Each lane loads its own
  // row (through LDS 125 -> 128 us for 4.2M strained particles with the FP64 SVD
  // on: vector instructions bound it); past the end row 0, which nobody uses.
  float Fn[9], lj_next = 0.f;
  int64_t w = (int64_t)blockIdx.x * kWaves + wave;
  auto load = [&](int64_t group) {
    int64_t q = group * kWave + lane;
    if (q >= ps.n) q = 0;
    load_row(ps.F, q, Fn);
    if (kKind == 1) lj_next = ps.logJp[q];
  };
  if (w * kWave < ps.n) load(w);
  for (; w * kWave < ps.n; w += nwaves) {
    const int64_t p0 = w * kWave;
    const int32_t cw = (int32_t)min((int64_t)kWave, ps.n - p0);
    const int64_t p = p0 + lane;
    float F[9], PF[9];
    float lj = lj_next;
#pragma unroll
    for (int k = 0; k < 9; ++k) F[k] = Fn[k];
    if ((w + nwaves) * kWave < ps.n) load(w + nwaves);
    if (lane < cw) {
      bool f64 = false;
      if constexpr (kKind != 2) {
        if constexpr (kGap)
          stress_gap(m, F, lj, PF, f64);
        else
          stress_plain(m, F, lj, PF);
        if (kKind == 1) ps.logJp[p] = lj;
      } else {
        const Model ms = ss.p[scene_of_particle(sfirst, ss.n, p)].model;
        if (ms.kind != 0) lj = ps.logJp[p];
        stress_any(ms, F, lj, PF, f64);
        if (ms.kind != 0) ps.logJp[p] = lj;
      }
      fp64_used += f64 ? 1u : 0u;
    }
    wave_store_rows<9>(contrib, p0, cw, stage, PF);
  }
  if (fp64_used) atomicAdd(&counters[kCtrFp64], fp64_used);
}

// kMode 0: mass and momentum with the force folded in (channels 0..3);
// 1: mass and momentum only (the stress is not read); 2: the force only, as
// if every particle were massless (v, C and m are not read), into channels
// fch .. fch + 2. kMulti (a batch, ss): each bucket's dx and dt are its
// scene's. kTile: the launch tile (p2g_threads, p2g_chunk).
// The stress is either read (st.F == nullptr: contrib, an earlier pass's vol P
// F^T) or formed here from st.F, particle by particle, before the record: a
// pass of its own wrote and re-read 36 bytes per particle and read F itself
// (72 of the substep's 370 bytes per particle).
// kCell (mode 0, one scene): P2C2GTransfer's particle -> cell -> node kernel
// (cell_w) in place of the quadratic B-spline, with C and the stress scaled
// per column by the cell kernel's Dinv.
template <int kMode, bool kMulti, bool kCell = false, int kTile = 0>
__global__ __launch_bounds__(p2g_threads(kTile),
                             kTile == kWideTile ? 4 : 3) void p2g_kernel(ParticlesView ps,
                                                       const float* __restrict__ contrib, StressFrom st,
                                                       TableView t, SortView sv, const int32_t* __restrict__ nbr_tab,
                                                       float* __restrict__ grid, int32_t grid_cap, float dt,
                                                       float dx, uint32_t* err, SceneSet ss, int32_t fch) {
  static_assert(kMode >= 0 && kMode <= 2 && (!kCell || kMode == 0), "P2G modes");
  constexpr bool kMom = kMode != 2;     // mass, v and C are read
  constexpr bool kStress = kMode != 1;  // the stress is read
  constexpr int kQ = Rec::kQuads;
  constexpr int kT = p2g_threads(kTile);
  constexpr int kWv = kT / kWave;
  constexpr int kChunk = p2g_chunk(kTile, Rec::kChunk);
  static_assert(kT % kWave == 0 && kChunk % kWave == 0,
                "whole waves; a chunk is a whole number of waves");
  __shared__ float4 arena[kWv][kArena6];
  // records in component-major order: component k of record i at
  // rec[k * kChunk + i], so consecutive records are consecutive float4 (no
  // LDS bank conflicts when lanes write consecutive records)
  __shared__ float4 rec[kChunk * kQ];
  __shared__ uint16_t list[kChunk];
  __shared__ uint8_t cellof[kChunk];
  __shared__ int32_t ccount[kMainCells + 1], cstart[kMainCells + 1], cfill[kMainCells + 1];
  __shared__ int32_t nbr[8];

  const float* __restrict__ stress_rows = st.F ? st.F : contrib;
  const int32_t nb = bounded_blocks(t, sv, grid_cap, err);
  const float dx_inv = (float)1.0 / dx;
  const float D_inv = 4.f * dx_inv * dx_inv;
  const float scale = -dt * D_inv;
  const int wave = uniform((int32_t)(threadIdx.x / kWave)), lane = lane_id();
  // Workgroup i takes the buckets i, i + grid, ... (a queue in their place cost
  // an atomic and two round trips per bucket and balanced no better: a workgroup
  // has ~50 buckets at 16M particles) in items of up to kChunk particles, and
  // keeps the next item's loads in flight: its bucket's count, offset and key
  // during phase A, its particle indices from the counting sort on, its first
  // 64 rows per wave during phase C and the flush; within phase A, the next
  // round's rows while this round's records are formed. With each lane loading
  // its own rows (load_row) and the divisions, zero fills and scale products
  // gone from phase A, 1.03 -> 0.81 ms at 16M particles; what bounds it now is
  // the arithmetic (0.59 ms of vector issue; 2.2 GB of traffic are 0.46 ms).
  constexpr int kPre = (kChunk + kT - 1) / kT;  // rounds of 64 rows per wave
  const int32_t nscenes = kMulti ? ss.n : 0;
  auto in_range = [&](int32_t cnt, int32_t off) { return cnt > 0 && off >= 0 && (int64_t)off + cnt <= ps.n; };
  int32_t b = blockIdx.x, cnt = 0, off = 0, c0 = 0;
  for (; b < nb; b += gridDim.x) {  // the first bucket with particles
    cnt = uniform(sv.counts[b]);
    off = uniform(sv.offsets[b]);
    if (in_range(cnt, off)) break;
  }
  if (b >= nb) return;
  int32_t key[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) key[d] = uniform(t.active[3 * (int64_t)b + d]);
  for (int c = threadIdx.x; c <= kMainCells; c += kT) {
    ccount[c] = 0;
    cfill[c] = 0;
  }
  struct Rows {
    float x[3], v[3], P[9], C[9], m, lj;
  };
  Rows ahead;  // rows in flight
  ahead.m = ahead.lj = 0.f;
  if (!kMom)
    for (int d = 0; d < 3; ++d) ahead.v[d] = 0.f;
  // an index out of range loads row 0, which nobody uses
  auto load_rows = [&](int32_t q) {
    if (q < 0 || q >= ps.n) q = 0;
    // a wave issues its loads ahead of other waves' scatter arithmetic
    __builtin_amdgcn_s_setprio(2);
    load_row(ps.x, q, ahead.x);
    if (kMom) load_row(ps.v, q, ahead.v);
    if (kStress) load_row(stress_rows, q, ahead.P);
    if (kMom) load_row(ps.C, q, ahead.C);
    if (kMom) ahead.m = ps.m[q];
    if (kStress && st.F && ps.logJp) ahead.lj = ps.logJp[q];
    __builtin_amdgcn_s_setprio(0);
  };
  int32_t pre[kPre];
  auto load_indices = [&](int32_t icnt, int32_t ioff, int32_t ic0) {
    const int32_t lim = min(icnt - ic0, kChunk);
#pragma unroll
    for (int k = 0; k < kPre; ++k) {
      const int32_t i = threadIdx.x + k * kT;
      pre[k] = i < lim ? sv.indices[ioff + ic0 + i] : -1;
    }
  };
  load_indices(cnt, off, 0);
  load_rows(pre[0]);
  __syncthreads();

  for (;;) {
    const int32_t nch = min(kChunk, cnt - c0);
    const bool last = c0 + kChunk >= cnt;
    // the next bucket's count, offset and key, in flight during phase A
    int32_t nx_b = last ? b + (int32_t)gridDim.x : b;
    int32_t nx_cnt = 0, nx_off = 0, nx_key[3] = {0, 0, 0};
    if (last && nx_b < nb) {
      nx_cnt = sv.counts[nx_b];
      nx_off = sv.offsets[nx_b];
#pragma unroll
      for (int d = 0; d < 3; ++d) nx_key[d] = t.active[3 * (int64_t)nx_b + d];
    }
    int32_t nbr_r = 0;
    if (c0 == 0 && threadIdx.x < 8) nbr_r = nbr_tab[8 * (int64_t)b + threadIdx.x];
    int32_t k0 = key[0];
    // the bucket's grid spacing and force scale (its scene's, in a batch)
    float bdx = dx, bscale = scale;
    const Model* bmodel = &st.m;
    if constexpr (kMulti) {
      const int32_t sc = scene_of_key(k0, nscenes);
      k0 -= sc * kSceneKeyStride;
      const SceneParams& sp = ss.p[sc];
      bdx = sp.dx;
      const float bdx_inv = (float)1.0 / bdx;
      bscale = -sp.dt * (4.f * bdx_inv * bdx_inv);
      bmodel = &sp.model;
    }
    const int32_t o0 = k0 * 4, o1 = key[1] * 4, o2 = key[2] * 4;
    {
      // ---- A: stress + affine record per particle. Each wave takes 64
      // consecutive chunk slots (i = threadIdx.x + k * kT, as phase B expects).
      // Not unrolled: the loop body with both stress paths is 3,000
      // instructions, and three copies of it (110 KB with the rest) overflow the
      // 64 KB instruction cache two CUs share.
#pragma clang loop unroll(disable)
      for (int kk = 0; kk < kPre; ++kk) {
        const int32_t i0 = wave * kWave + kk * kT;
        if (i0 >= nch) break;
        int32_t p = pre[0], pnext = -1;
#pragma unroll
        for (int q = 1; q < kPre; ++q) {
          p = kk == q ? pre[q] : p;
          pnext = kk == q - 1 ? pre[q] : pnext;
        }
        const int32_t i = i0 + lane;
        const bool valid = i < nch;
        const bool live = valid && p >= 0 && p < ps.n;
        if (valid && !live) {
          atomicOr(err, kErrCapacity);
          cellof[i] = 255;
          list[i] = 0;
        }
        const Rows row = ahead;
        if (i0 + kT < nch) load_rows(pnext);
        if (!live) continue;
        const float (&xv)[3] = row.x;
        const float (&vv)[3] = row.v;
        const float (&C)[9] = row.C;
        const float mass = row.m;
        float PF[9];
#pragma unroll
        for (int k = 0; k < 9; ++k) PF[k] = row.P[k];
        if (kStress && st.F) {
          float lj = row.lj;
          stress_plain(*bmodel, row.P, lj, PF);
          if (bmodel->kind != 0 && st.store_lj) ps.logJp[p] = lj;
        }
        const float x0 = xv[0], x1 = xv[1], x2 = xv[2];
        const float v0 = vv[0], v1 = vv[1], v2 = vv[2];
        // base node and local position in grid units (LocalArena::init, Utils.hpp:51-70)
        float l[3];
        int32_t base[3];
        {
#pragma clang fp contract(off)
          const float xs[3] = {x0, x1, x2};
          const bool pow2 = is_pow2(bdx);
          const float bdx_inv = 1.f / bdx;
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            const float X = pow2 ? xs[d] * bdx_inv : xs[d] / bdx;
            base[d] = (int32_t)floorf(X - 0.5f);
            l[d] = X - (float)base[d];
          }
        }
        const int r0 = base[0] - o0, r1 = base[1] - o1, r2 = base[2] - o2;  // in [0, 6)
        int cell;
        if (r0 >= 1 && r0 <= 4 && r1 >= 1 && r1 <= 4 && r2 >= 1 && r2 <= 4) {
          cell = cell_lane(r0 - 1, r1 - 1, r2 - 1);
        } else if (r0 >= 0 && r0 <= 5 && r1 >= 0 && r1 <= 5 && r2 >= 0 && r2 <= 5) {
          cell = kMainCells;  // overflow: scattered with global atomics
        } else {
          atomicOr(err, kErrArena);
          cell = 255;
        }
        // affine record: m v + (m C + contrib') (o - l) dx
        float A[9], Bv[3];
        const float mv[3] = {mass * v0, mass * v1, mass * v2};
        if constexpr (kCell) {
          // P2C2G.hpp:86-96, 138-140: C and vol P F^T scaled per column by
          // Dinv, the stress by -dt, summed with m C
#pragma clang fp contract(off)
          float Dinv[3];
          cell_dinv(xv, bdx, dx_inv, Dinv);
#pragma unroll
          for (int k = 0; k < 9; ++k) A[k] = (PF[k] * (Dinv[k / 3] * -dt) + (C[k] * Dinv[k / 3]) * mass) * bdx;
        } else {
#pragma unroll
          for (int k = 0; k < 9; ++k) {
            if (kMode == 0) A[k] = (mass * bdx) * C[k] + PF[k] * (bscale * bdx);
            if (kMode == 1) A[k] = (mass * bdx) * C[k];
            if (kMode == 2) A[k] = PF[k] * (bscale * bdx);
          }
        }
#pragma unroll
        for (int d = 0; d < 3; ++d) Bv[d] = mv[d] - (A[d] * l[0] + A[d + 3] * l[1] + A[d + 6] * l[2]);
        rec[0 * kChunk + i] = make_float4(mass, Bv[0], Bv[1], Bv[2]);
        if constexpr (!kCell)
#pragma unroll
          for (int d = 0; d < 3; ++d) l[d] = bspline_arg(l[d]);
        rec[1 * kChunk + i] = make_float4(l[0], l[1], l[2], A[8]);
        rec[2 * kChunk + i] = make_float4(A[0], A[1], A[2], A[3]);
        rec[3 * kChunk + i] = make_float4(A[4], A[5], A[6], A[7]);
        cellof[i] = (uint8_t)cell;
        if (cell <= kMainCells) atomicAdd(&ccount[cell], 1);
        list[i] = (uint16_t)((r0 << 6) | (r1 << 3) | r2);  // base offsets; the list is rebuilt in B
      }
      if (c0 == 0) {
        if (threadIdx.x < 8) {
          nbr[threadIdx.x] = nbr_r;
          if (nbr_r < 0) atomicOr(err, kErrMissingBlock);
        }
        for (int k = lane; k < kArena6; k += kWave) arena[wave][k] = make_float4(0.f, 0.f, 0.f, 0.f);
      }
      __syncthreads();
      // ---- B: counting sort of the chunk by base cell
      if (threadIdx.x < kWave) {
        const int32_t c = (threadIdx.x < kMainCells) ? ccount[threadIdx.x] : 0;
        int32_t inc = c;
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) {
          const int32_t u = __shfl_up(inc, o, kWave);
          if (lane >= o) inc += u;
        }
        cstart[threadIdx.x] = inc - c;
        if (threadIdx.x == kWave - 1) cstart[kMainCells] = inc;  // overflow particles follow the main cells
      }
      // each thread keeps the base offsets and cells of its own particles
      // across the rebuild of list[]
      uint16_t keep[kPre];
      uint8_t keepc[kPre];
#pragma unroll
      for (int k = 0; k < kPre; ++k) {
        const int32_t i = threadIdx.x + k * kT;
        keep[k] = i < nch ? list[i] : (uint16_t)0;
        keepc[k] = i < nch ? cellof[i] : (uint8_t)255;
      }
      __syncthreads();
#pragma unroll
      for (int k = 0; k < kPre; ++k) {
        const int32_t i = threadIdx.x + k * kT;
        if (i < nch && keepc[k] <= kMainCells) {
          const int32_t slot = atomicAdd(&cfill[keepc[k]], 1);
          list[cstart[keepc[k]] + slot] = (uint16_t)i;
        }
      }
      __syncthreads();
      // the next item; its indices load during the first slab
      int32_t nx_c0 = 0;
      if (last) {
        nx_cnt = uniform(nx_cnt);
        nx_off = uniform(nx_off);
#pragma unroll
        for (int d = 0; d < 3; ++d) nx_key[d] = uniform(nx_key[d]);
        while (nx_b < nb && !in_range(nx_cnt, nx_off)) {  // an empty (enlarged-only) block
          nx_b += gridDim.x;
          if (nx_b >= nb) break;
          nx_cnt = uniform(sv.counts[nx_b]);
          nx_off = uniform(sv.offsets[nx_b]);
#pragma unroll
          for (int d = 0; d < 3; ++d) nx_key[d] = uniform(t.active[3 * (int64_t)nx_b + d]);
        }
      } else {
        nx_cnt = cnt;
        nx_off = off;
#pragma unroll
        for (int d = 0; d < 3; ++d) nx_key[d] = key[d];
        nx_c0 = c0 + kChunk;
      }
      const bool more = nx_b < nb;
      if (more) load_indices(nx_cnt, nx_off, nx_c0);
      // ---- C: rounds, lane = main cell
      {
        const int32_t lcount = ccount[lane];
        const int32_t lstart = cstart[lane];
        int lr0, lr1, lr2;  // base - (4b+1) of the lane's main cell
        lane_cell(lane, lr0, lr1, lr2);
        float4* ar = arena[wave];
        // All particles of one base cell touch the same 27 nodes: the lane
        // sums its share of its cell's particles (every kWv-th, starting
        // at the wave index) in registers and adds the node sums to the
        // wave's arena once per cell, instead of 27 LDS read-modify-writes
        // per particle. One pass per x-slab of the stencil keeps the
        // accumulators at 9 nodes x 4 channels.
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          float acc[9][4];
#pragma unroll
          for (int k = 0; k < 9; ++k) acc[k][0] = acc[k][1] = acc[k][2] = acc[k][3] = 0.f;
          for (int32_t r = wave; r < lcount; r += kWv) {
            const int32_t i = list[lstart + r];
            const float4 q0 = rec[i], q1 = rec[kChunk + i], q2 = rec[2 * kChunk + i], q3 = rec[3 * kChunk + i];
            float w0[3], w1[3], w2[3];
            stencil_w<kCell>(q1.x, w0);
            stencil_w<kCell>(q1.y, w1);
            stencil_w<kCell>(q1.z, w2);
            const float fa = (float)a;
#pragma unroll
            for (int bb = 0; bb < 3; ++bb) {
              const float w01 = w0[a] * w1[bb];
              const float fb = (float)bb;
              // offset 0 adds nothing (the compiler keeps x * 0)
              float s0 = q0.y, s1 = q0.z, s2 = q0.w;
              if (a > 0) {
                s0 += q2.x * fa;
                s1 += q2.y * fa;
                s2 += q2.z * fa;
              }
              if (bb > 0) {
                s0 += q2.w * fb;
                s1 += q3.x * fb;
                s2 += q3.y * fb;
              }
#pragma unroll
              for (int c = 0; c < 3; ++c) {
                const float W = w01 * w2[c];
                const float fc = (float)c;
                float* e = acc[bb * 3 + c];
                if (kMom) e[0] += q0.x * W;
                e[1] += W * (c > 0 ? s0 + q3.z * fc : s0);
                e[2] += W * (c > 0 ? s1 + q3.w * fc : s1);
                e[3] += W * (c > 0 ? s2 + q1.w * fc : s2);
              }
            }
          }
          if (wave < lcount) {
#pragma unroll
            for (int bb = 0; bb < 3; ++bb)
#pragma unroll
              for (int c = 0; c < 3; ++c) {
                const int n = (lr0 + a) * 36 + (lr1 + bb) * 6 + (lr2 + c);
                const float* e = acc[bb * 3 + c];
                // Lanes of one step touch distinct nodes, but a node a lane
                // updates in this step may be one another lane updated in an
                // earlier step. The LDS unit serves a wave's accesses in issue
                // order; this barrier keeps the compiler from hoisting this
                // step's read above earlier steps' writes.
                asm volatile("" ::: "memory");
                float4 v = ar[n];
                v.x += e[0];
                v.y += e[1];
                v.z += e[2];
                v.w += e[3];
                ar[n] = v;
              }
          }
          if (a == 0 && more) load_rows(pre[0]);  // in flight across the other slabs and the flush
        }
      }
      // ---- overflow particles (rare): global atomics straight into the grid
      if (ccount[kMainCells] > 0) {
#pragma clang loop unroll(disable)
        for (int k = 0; k < kPre; ++k) {
          const int32_t i = threadIdx.x + k * kT;
          uint32_t base = keep[0], home = keepc[0];
#pragma unroll
          for (int q = 1; q < kPre; ++q) {
            base = k == q ? keep[q] : base;
            home = k == q ? keepc[q] : home;
          }
          if (i >= nch || home != (uint32_t)kMainCells) continue;
          const int r0 = (base >> 6) & 7, r1 = (base >> 3) & 7, r2 = base & 7;
          const float4 q0 = rec[i], q1 = rec[kChunk + i], q2 = rec[2 * kChunk + i], q3 = rec[3 * kChunk + i];
          float w0[3], w1[3], w2[3];
          stencil_w<kCell>(q1.x, w0);
          stencil_w<kCell>(q1.y, w1);
          stencil_w<kCell>(q1.z, w2);
#pragma clang loop unroll(disable)
          for (int o = 0; o < 27; ++o) {
            const int a = o / 9, bb = o / 3 % 3, c = o % 3;
            const float W = (a == 0 ? w0[0] : a == 1 ? w0[1] : w0[2]) *
                            (bb == 0 ? w1[0] : bb == 1 ? w1[1] : w1[2]) * (c == 0 ? w2[0] : c == 1 ? w2[1] : w2[2]);
            int nbi, cell;
            node_home(r0 + a, r1 + bb, r2 + c, nbi, cell);
            const int32_t gb = nbr[nbi];
            if (gb < 0 || gb >= grid_cap) continue;
            float* gp = grid + grid_at(gb, 0, cell);
            const float fa = (float)a, fb = (float)bb, fc = (float)c;
            float* gv = kMom ? gp + kBlockCells : gp + fch * kBlockCells;  // momentum or force channels
            if (kMom) unsafeAtomicAdd(gp, q0.x * W);
            unsafeAtomicAdd(gv, W * (q0.y + q2.x * fa + q2.w * fb + q3.z * fc));
            unsafeAtomicAdd(gv + kBlockCells, W * (q0.z + q2.y * fa + q3.x * fb + q3.w * fc));
            unsafeAtomicAdd(gv + 2 * kBlockCells, W * (q0.w + q2.z * fa + q3.y * fb + q1.w * fc));
          }
        }
      }
      __syncthreads();
      // the next item finds its cell counters cleared (they are not read from
      // here on; the barrier after the flush orders the clear)
      for (int c = threadIdx.x; c <= kMainCells; c += kT) {
        ccount[c] = 0;
        cfill[c] = 0;
      }
      b = nx_b;
      cnt = nx_cnt;
      off = nx_off;
      c0 = nx_c0;
#pragma unroll
      for (int d = 0; d < 3; ++d) key[d] = nx_key[d];
      if (!last) {  // the bucket's next chunk adds to the same arenas
        __syncthreads();
        continue;
      }
    }
    // ---- flush: sum the wave arenas, one global atomic per touched node/channel
    for (int n = threadIdx.x; n < kArena6; n += kT) {
      float4 s = arena[0][n];
#pragma unroll
      for (int w = 1; w < kWv; ++w) {
        const float4 u = arena[w][n];
        s.x += u.x;
        s.y += u.y;
        s.z += u.z;
        s.w += u.w;
      }
      // every node a particle touched, massless particles included (zpc adds
      // all 27 nodes, P2G.hpp:114-123); untouched nodes hold exact zeros
      const bool touched = s.x != 0.f || s.y != 0.f || s.z != 0.f || s.w != 0.f;
      if (touched) {
        int nbi, cell;
        node_home(n / 36 + 1, (n / 6) % 6 + 1, n % 6 + 1, nbi, cell);
        const int32_t gb = nbr[nbi];
        if (gb >= 0 && gb < grid_cap) {
          float* gp = grid + grid_at(gb, 0, cell);
          float* gv = kMom ? gp + kBlockCells : gp + fch * kBlockCells;  // momentum or force channels
          if (kMom) unsafeAtomicAdd(gp, s.x);
          unsafeAtomicAdd(gv, s.y);
          unsafeAtomicAdd(gv + kBlockCells, s.z);
          unsafeAtomicAdd(gv + 2 * kBlockCells, s.w);
        }
      }
    }
    if (b >= nb) break;
    __syncthreads();
  }
}

// v = (mv [+ rhs]) / m + extf dt where m != 0 (GridOp.hpp:71-110), max |v|^2,
// then the colliders in order on nodes with m > 0 (GridOp.hpp:112-164,
// Collider.h:80-107). fold adds the rhs channels first (the explicit
// driver's convention when P2G kept them separate).
// Signed distance of a general collider's level set at the material-space
// point X (AnalyticLevelSet.h: Plane :26-29, Cuboid :81-88, Sphere :142-145,
// Cylinder :180-207), rounded as written.
__device__ __forceinline__ float level_set_sdf(const GeneralCollider& c, const float (&X)[3]) {
#pragma clang fp contract(off)
  if (c.geometry == 0) {
    return c.p1[0] * (X[0] - c.p0[0]) + c.p1[1] * (X[1] - c.p0[1]) + c.p1[2] * (X[2] - c.p0[2]);
  }
  if (c.geometry == 1) {
    float point[3], mx = 0.f;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const float center = (c.p0[d] + c.p1[d]) / 2.f;
      point[d] = fabsf(X[d] - center) - (c.p1[d] - c.p0[d]) / 2.f;
      mx = d == 0 ? point[d] : fmaxf(mx, point[d]);
    }
#pragma unroll
    for (int d = 0; d < 3; ++d)
      if (point[d] < 0.f) point[d] = 0.f;
    const float len = sqrtf(point[0] * point[0] + point[1] * point[1] + point[2] * point[2]);
    return (mx < 0.f ? mx : 0.f) + len;
  }
  if (c.geometry == 2) {
    const float o0 = X[0] - c.p0[0], o1 = X[1] - c.p0[1], o2 = X[2] - c.p0[2];
    return sqrtf(o0 * o0 + o1 * o1 + o2 * o2) - c.p1[0];
  }
  const int ax = c.axis;
  const float dr0 = X[ax == 0 ? 1 : 0] - c.p0[ax == 0 ? 1 : 0];
  const float dr1 = X[ax == 2 ? 1 : 2] - c.p0[ax == 2 ? 1 : 2];
  const float disR = sqrtf(dr0 * dr0 + dr1 * dr1);
  const float r = c.p1[0], len = c.p1[1];
  const bool outside = disR > r;
  if (X[ax] < c.p0[ax]) {
    const float disL = c.p0[ax] - X[ax];
    return outside ? sqrtf((disR - r) * (disR - r) + disL * disL) : disL;
  }
  if (X[ax] > c.p0[ax] + len) {
    const float disL = X[ax] - (c.p0[ax] + len);
    return outside ? sqrtf((disR - r) * (disR - r) + disL * disL) : disL;
  }
  if (outside) return disR - r;
  const float disL = fminf(c.p0[ax] + len - X[ax], X[ax] - c.p0[ax]);
  return -fminf(disL, r - disR);
}

// Material-space normal (AnalyticLevelSet.h :30-33, :89-103, :146-150,
// :208-222): the plane's normal as given, the sphere's outward direction
// (zero within 1e-7 squared of the center), normalised central differences
// of step 1e-6 for the cuboid and the cylinder.
__device__ __forceinline__ void level_set_normal(const GeneralCollider& c, const float (&X)[3], float (&n)[3]) {
#pragma clang fp contract(off)
  if (c.geometry == 0) {
    n[0] = c.p1[0];
    n[1] = c.p1[1];
    n[2] = c.p1[2];
    return;
  }
  if (c.geometry == 2) {
    const float o[3] = {X[0] - c.p0[0], X[1] - c.p0[1], X[2] - c.p0[2]};
    const float l2 = o[0] * o[0] + o[1] * o[1] + o[2] * o[2];
    if (l2 < 1e-7f) {
      n[0] = n[1] = n[2] = 0.f;
      return;
    }
    const float l = sqrtf(l2);
    n[0] = o[0] / l;
    n[1] = o[1] / l;
    n[2] = o[2] / l;
    return;
  }
  const float eps = 1e-6f;
  float diff[3];
  for (int i = 0; i < 3; ++i) {
    float v1[3] = {X[0], X[1], X[2]}, v2[3] = {X[0], X[1], X[2]};
    v1[i] = X[i] + eps;
    v2[i] = X[i] - eps;
    diff[i] = (level_set_sdf(c, v1) - level_set_sdf(c, v2)) / (eps + eps);
  }
  const float l = sqrtf(diff[0] * diff[0] + diff[1] * diff[1] + diff[2] * diff[2]);
  n[0] = diff[0] / l;
  n[1] = diff[1] / l;
  n[2] = diff[2] / l;
}

// Collider::resolveCollision (Collider.h:81-107) with erosion 0 and the
// analytic level sets' zero material velocity.
__device__ __forceinline__ void resolve_general(const GeneralCollider& c, const float (&x)[3], float (&v)[3]) {
#pragma clang fp contract(off)
  const float xmb[3] = {x[0] - c.b[0], x[1] - c.b[1], x[2] - c.b[2]};
  const float inv_s = 1.f / c.s;
  float X[3];
#pragma unroll
  for (int i = 0; i < 3; ++i)
    X[i] = (c.R[0 + 3 * i] * xmb[0] + c.R[1 + 3 * i] * xmb[1] + c.R[2 + 3 * i] * xmb[2]) * inv_s;
  if (!(level_set_sdf(c, X) < 0.f)) return;
  const float rate = c.dsdt * inv_s;
  const float wx[3] = {c.omega[1] * xmb[2] - c.omega[2] * xmb[1], c.omega[2] * xmb[0] - c.omega[0] * xmb[2],
                       c.omega[0] * xmb[1] - c.omega[1] * xmb[0]};
  float vo[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) vo[d] = wx[d] + rate * xmb[d] + c.dbdt[d];
  if (c.type == 0) {
#pragma unroll
    for (int d = 0; d < 3; ++d) v[d] = vo[d];
    return;
  }
#pragma unroll
  for (int d = 0; d < 3; ++d) v[d] -= vo[d];
  float nm[3], n[3];
  level_set_normal(c, X, nm);
#pragma unroll
  for (int r = 0; r < 3; ++r) n[r] = c.R[r] * nm[0] + c.R[r + 3] * nm[1] + c.R[r + 6] * nm[2];
  const float proj = n[0] * v[0] + n[1] * v[1] + n[2] * v[2];
  if ((c.type == 2 && proj < 0.f) || c.type == 1) {
#pragma unroll
    for (int d = 0; d < 3; ++d) v[d] -= proj * n[d];
  }
#pragma unroll
  for (int d = 0; d < 3; ++d) v[d] += vo[d];
}

// Node velocity and colliders of one node (mass != 0) of the block with key
// k; cols is the kernel argument or a scene's colliders in a batch.
// kLocal: k0_local is the key's first component with a batch's scene offset
// removed; otherwise the table's own key is read.
// kGen: general colliders or a level-set boundary are set.
template <bool kLocal, bool kGen, typename Cols, typename Gen>
__device__ __forceinline__ void node_velocity(float* gp, float mass, int fold, float e0, float e1, float e2,
                                              const Cols& cols, const Gen& gen, const TableView& t,
                                              int32_t b, int32_t k0_local, int cell, float dx, float& vmax) {
  // rounded as written (no FMA contraction): a node on a collider plane has
  // phi = 0 in exact arithmetic, and the sign of the rounded phi must be the
  // one the host path computes
#pragma clang fp contract(off)
  const float inv = 1.f / mass;
  float mv0 = gp[1 * kBlockCells], mv1 = gp[2 * kBlockCells], mv2 = gp[3 * kBlockCells];
  if (fold) {
    mv0 = mv0 + gp[4 * kBlockCells];
    mv1 = mv1 + gp[5 * kBlockCells];
    mv2 = mv2 + gp[6 * kBlockCells];
  }
  float v[3] = {mv0 * inv + e0, mv1 * inv + e1, mv2 * inv + e2};
  vmax = fmaxf(vmax, v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
  if (mass > 0.f && (cols.n > 0 || kGen)) {
    const int32_t k0 = kLocal ? k0_local : t.active[3 * (int64_t)b];
    const int32_t k1 = t.active[3 * (int64_t)b + 1], k2 = t.active[3 * (int64_t)b + 2];
    const float pos[3] = {((float)k0 * 4.f + (float)((cell >> 4) & 3)) * dx,
                          ((float)k1 * 4.f + (float)((cell >> 2) & 3)) * dx,
                          ((float)k2 * 4.f + (float)(cell & 3)) * dx};
    for (int c = 0; c < cols.n; ++c) {
      const PlaneCollider& pc = cols.c[c];
      const float phi = pc.normal[0] * (pos[0] - pc.origin[0]) + pc.normal[1] * (pos[1] - pc.origin[1]) +
                        pc.normal[2] * (pos[2] - pc.origin[2]);
      if (phi < 0.f) {
        if (pc.type == 0) {
          v[0] = v[1] = v[2] = 0.f;
        } else {
          const float proj = pc.normal[0] * v[0] + pc.normal[1] * v[1] + pc.normal[2] * v[2];
          if ((pc.type == 2 && proj < 0.f) || pc.type == 1) {
            v[0] -= proj * pc.normal[0];
            v[1] -= proj * pc.normal[1];
            v[2] -= proj * pc.normal[2];
          }
        }
      }
    }
    if constexpr (kGen) {
      for (int c = 0; c < gen.n; ++c) resolve_general(gen.c[c], pos, v);
      if (gen.ls.on) levelset_resolve(gen.ls, pos, v);
    }
  }
  gp[1 * kBlockCells] = v[0];
  gp[2 * kBlockCells] = v[1];
  gp[3 * kBlockCells] = v[2];
}

// Gen: GeneralColliders, or NoColliders where none are set: the general
// colliders' code (180 KB with the level set) and arguments stay out of the
// ordinary update.
struct NoColliders {};
template <bool kMulti, typename Gen>
__global__ __launch_bounds__(kThreads) void grid_update_kernel(float* __restrict__ grid, int32_t grid_cap,
                                                               TableView t, float dt, float g0, float g1,
                                                               float g2, Colliders cols, float dx, int fold,
                                                               uint32_t* counters, uint32_t* err, SceneSet ss,
                                                               Gen gen) {
  constexpr bool kGen = std::is_same<Gen, GeneralColliders>::value;
  int32_t nb = *t.cnt;
  if (nb > grid_cap) {
    if (blockIdx.x == 0 && threadIdx.x == 0) atomicOr(err, kErrCapacity);
    nb = grid_cap;
  }
  const int64_t nodes = (int64_t)nb * kBlockCells;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  float vmax = 0.f;
  const float e0 = g0 * dt, e1 = g1 * dt, e2 = g2 * dt;
  for (int64_t base = (int64_t)blockIdx.x * blockDim.x; base < nodes; base += stride) {
    const int64_t i = base + threadIdx.x;
    if (i < nodes) {
      const int32_t b = (int32_t)(i >> 6);
      const int cell = (int)(i & 63);
      float* gp = grid + grid_at(b, 0, cell);
      const float mass = gp[0];
      if (mass != 0.f) {
        if constexpr (kMulti) {
          // the node's scene (from its block key): its dt, gravity, dx and colliders
          int32_t k0 = t.active[3 * (int64_t)b];
          const int32_t sc = scene_of_key(k0, ss.n);
          const SceneParams& sp = ss.p[sc];
          k0 -= sc * kSceneKeyStride;
          node_velocity<true, kGen>(gp, mass, fold, sp.g[0] * sp.dt, sp.g[1] * sp.dt, sp.g[2] * sp.dt, sp.cols, gen, t, b,
                              k0, cell, sp.dx, vmax);
        } else {
          node_velocity<false, kGen>(gp, mass, fold, e0, e1, e2, cols, gen, t, b, 0, cell, dx, vmax);
        }
      } else if (fold) {
        // the fold covers every node, massless ones included (their
        // momentum channels then hold mv + rhs, as after a separate fold)
#pragma unroll
        for (int d = 1; d <= 3; ++d) gp[d * kBlockCells] = gp[d * kBlockCells] + gp[(d + 3) * kBlockCells];
      }
    }
  }
  // max |v|^2: wave, then workgroup, then one atomic per workgroup -- and only
  // when it raises the running maximum (same-address atomics serialise)
  __shared__ float wmax[kWaves];
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) vmax = fmaxf(vmax, __shfl_xor(vmax, o, kWave));
  if (lane_id() == 0) wmax[threadIdx.x / kWave] = vmax;
  __syncthreads();
  if (threadIdx.x == 0) {
    float g = wmax[0];
    for (int w = 1; w < kWaves; ++w) g = fmaxf(g, wmax[w]);
    const uint32_t bits = __float_as_uint(g);
    if (g > 0.f && bits > __atomic_load_n(&counters[kCtrMaxVel], __ATOMIC_RELAXED))
      atomicMax(&counters[kCtrMaxVel], bits);
  }
}

// GridAngularMomentum (GridOp.hpp:216-259): for every node with m != 0,
// x = (blockkey * 4 + coord(cell)) * dx; sum[0..2] += (double)(x cross mv)
// formed in float, sum[3..5] += (double)mv. Per-thread double partials, a
// wave and workgroup reduction, six double atomics per workgroup.
__global__ __launch_bounds__(kThreads) void angular_momentum_kernel(const float* __restrict__ grid, int32_t grid_cap,
                                                                    TableView t, float dx, int mchn, int mvchn,
                                                                    double* sum, uint32_t* err) {
#pragma clang fp contract(off)
  int32_t nb = *t.cnt;
  if (nb > grid_cap) {
    if (blockIdx.x == 0 && threadIdx.x == 0) atomicOr(err, kErrCapacity);
    nb = grid_cap;
  }
  const int64_t nodes = (int64_t)nb * kBlockCells;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  double acc[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < nodes; i += stride) {
    const int32_t b = (int32_t)(i >> 6);
    const int cell = (int)(i & 63);
    const float mass = grid[grid_at(b, mchn, cell)];
    if (mass == 0.f) continue;
    const float x0 = ((float)t.active[3 * (int64_t)b] * 4.f + (float)((cell >> 4) & 3)) * dx;
    const float x1 = ((float)t.active[3 * (int64_t)b + 1] * 4.f + (float)((cell >> 2) & 3)) * dx;
    const float x2 = ((float)t.active[3 * (int64_t)b + 2] * 4.f + (float)(cell & 3)) * dx;
    const float m0 = grid[grid_at(b, mvchn, cell)], m1 = grid[grid_at(b, mvchn + 1, cell)],
                m2 = grid[grid_at(b, mvchn + 2, cell)];
    acc[0] += (double)(x1 * m2 - x2 * m1);
    acc[1] += (double)(x2 * m0 - x0 * m2);
    acc[2] += (double)(x0 * m1 - x1 * m0);
    acc[3] += (double)m0;
    acc[4] += (double)m1;
    acc[5] += (double)m2;
  }
  __shared__ double part[kWaves][6];
#pragma unroll
  for (int k = 0; k < 6; ++k) {
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) acc[k] += __shfl_xor(acc[k], o, kWave);
  }
  const int wave = threadIdx.x / kWave;
  if (lane_id() == 0)
    for (int k = 0; k < 6; ++k) part[wave][k] = acc[k];
  __syncthreads();
  if (threadIdx.x < 6) {
    double s = 0.0;
    for (int w = 0; w < kWaves; ++w) s += part[w][threadIdx.x];
    if (s != 0.0) atomicAdd(&sum[threadIdx.x], s);
  }
}

// v += sum W v_i and B += sum W v_i (x_i - x)^T (column-major) over the 27
// staged nodes. The weights are products over the axes, so the sums are taken
// axis by axis: 279 multiply-adds per particle against 513 node by node (substep
// at 16M particles 1638 -> 1613 us, implicit product at 1M 127 -> 123.5).
__device__ __forceinline__ void gather_nodes(const float4* vel, int b0, int b1, int b2, const Arena& ar, float dx,
                                             float (&v)[3], float (&B)[9]) {
  float wx1[3], wx2[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    wx1[k] = ar.w[1][k] * ((float)k * dx - ar.lp[1]);
    wx2[k] = ar.w[2][k] * ((float)k * dx - ar.lp[2]);
  }
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    float T[3] = {0.f, 0.f, 0.f}, Y[3] = {0.f, 0.f, 0.f}, Z[3] = {0.f, 0.f, 0.f};
#pragma unroll
    for (int bb = 0; bb < 3; ++bb) {
      float t[3] = {0.f, 0.f, 0.f}, z[3] = {0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const float4 q = vel[vel_at(b0 + a, b1 + bb, b2 + c)];
        const float vi[3] = {q.x, q.y, q.z};
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          t[d] += ar.w[2][c] * vi[d];
          z[d] += wx2[c] * vi[d];
        }
      }
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        T[d] += ar.w[1][bb] * t[d];
        Y[d] += wx1[bb] * t[d];
        Z[d] += ar.w[1][bb] * z[d];
      }
    }
    const float w0 = ar.w[0][a], wx0 = w0 * ((float)a * dx - ar.lp[0]);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      v[d] += w0 * T[d];
      B[d] += wx0 * T[d];
      B[d + 3] += w0 * Y[d];
      B[d + 6] += w0 * Z[d];
    }
  }
}

// kNext: -1 plain G2P; 0 / 1 (reorder only): also the next substep's
// fixed-corotated / Drucker-Prager stress from the updated F (NextStress).
// kCell (in place, one scene): G2C2PTransfer with its pre and post passes
// (G2C2P.hpp:58-151, 197-271): the cell kernel's weights (cell_w), B =
// sum W v_i (x_i - x_p)^T stored as C, and F updated with B scaled per column
// by Dinv at the old position.
template <bool kReorder, int kNext, bool kMulti = false, bool kCell = false, int kT = kG2PThreads>
__global__ __launch_bounds__(kT) void g2p_kernel(ParticlesView ps, ParticlesView out, TableView t,
                                                          SortView sv, const int32_t* __restrict__ nbr_tab,
                                                          const float* __restrict__ grid, int32_t grid_cap,
                                                          float dt_arg, float dx_arg, NextStress ns, uint32_t* err,
                                                          uint32_t* counters, SceneSet ss) {
  static_assert(kNext < 0 || kReorder, "the fused stress writes in output slot order");
  uint32_t fp64_used = 0;
  __shared__ float4 vel[kVelNodes];
  __shared__ int32_t nbr[8];
  __shared__ float4 stage4[kT / kWave][stage_floats(9) / 4];
  const int32_t nb = bounded_blocks(t, sv, grid_cap, err);
  const float dx_inv_arg = (float)1 / dx_arg;
  const float D_inv_arg = 4.f * dx_inv_arg * dx_inv_arg;
  const int wave = uniform((int32_t)(threadIdx.x / kWave)), lane = lane_id();
  float* stage = reinterpret_cast<float*>(stage4[wave]);
  for (int32_t b = blockIdx.x; b < nb; b += gridDim.x) {
    const int32_t cnt = sv.counts[b];
    const int32_t off = sv.offsets[b];
    if (cnt <= 0 || off < 0 || (int64_t)off + cnt > ps.n) continue;
    // the wave's first 64 particles: indices, then rows, load while the
    // velocities are staged
    int32_t pnext = -1;
    if (wave * kWave + lane < cnt) pnext = sv.indices[off + wave * kWave + lane];
    load_neighbours(nbr_tab, b, nbr, err);
    int32_t k0 = t.active[3 * (int64_t)b];
    // the bucket's grid spacing and time step (its scene's, in a batch)
    float dx = dx_arg, dt = dt_arg, D_inv = D_inv_arg;
    if constexpr (kMulti) {
      const int32_t sc = scene_of_key(k0, ss.n);
      k0 -= sc * kSceneKeyStride;
      dx = ss.p[sc].dx;
      dt = ss.p[sc].dt;
      const float dx_inv = (float)1 / dx;
      D_inv = 4.f * dx_inv * dx_inv;
    }
    const int32_t o0 = k0 * 4, o1 = t.active[3 * (int64_t)b + 1] * 4, o2 = t.active[3 * (int64_t)b + 2] * 4;
    __syncthreads();
    // x, F and the attributes the reorder only moves, of the next round; an
    // index out of range loads row 0, which nobody uses
    float xr[3], Fr[9], mr = 0.f, ljr = 0.f;
    int32_t idr = 0;
    auto load_ahead = [&](int32_t q) {
      if (q < 0 || q >= ps.n) q = 0;
      load_row(ps.x, q, xr);
      load_row(ps.F, q, Fr);
      if (kReorder) {
        mr = ps.m[q];
        if (ps.logJp) ljr = ns.lj_src ? ns.lj_src[q] : ps.logJp[q];
        idr = ps.id ? ps.id[q] : q;
      }
    };
    load_ahead(pnext);
    // stage node velocities: slot s -> (neighbour block s>>6, cell s&63), stored at vel_at(r0, r1, r2)
    for (int s = threadIdx.x; s < kArena8; s += kT) {
      const int nbi = s >> 6, cell = s & 63;
      const int r0 = ((nbi >> 2) & 1) * 4 + ((cell >> 4) & 3);
      const int r1 = ((nbi >> 1) & 1) * 4 + ((cell >> 2) & 3);
      const int r2 = (nbi & 1) * 4 + (cell & 3);
      const int32_t gb = nbr[nbi];
      float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
      if (gb >= 0 && gb < grid_cap) {
        const float* gp = grid + grid_at(gb, 1, cell);
        v = make_float4(gp[0], gp[kBlockCells], gp[2 * kBlockCells], 0.f);
      }
      vel[vel_at(r0, r1, r2)] = v;
    }
    __syncthreads();
    // each wave takes 64 consecutive bucket slots at a time (wave-uniform loop)
    for (int32_t i0 = wave * kWave; i0 < cnt; i0 += kT) {
      const int32_t cw = min(kWave, cnt - i0);
      const bool valid = lane < cw;
      const int64_t p = pnext;
      const bool more = i0 + kT < cnt;  // uniform across the wave
      if (more) pnext = i0 + kT + lane < cnt ? sv.indices[off + i0 + kT + lane] : -1;
      const bool bad = valid && (p < 0 || p >= ps.n);
      if (bad) atomicOr(err, kErrCapacity);
      const bool live = valid && !bad;
      int64_t p0;
      const bool contig = wave_contiguous(p, live, p0) && ballot(bad) == 0;
      float x[3], F[9];
#pragma unroll
      for (int d = 0; d < 3; ++d) x[d] = xr[d];
#pragma unroll
      for (int k = 0; k < 9; ++k) F[k] = Fr[k];
      const float mcopy = mr, ljcopy = ljr;
      const int32_t idcopy = idr;
      Arena ar;
      make_arena(x[0], x[1], x[2], dx, ar);
      if constexpr (kCell) {
#pragma clang fp contract(off)
#pragma unroll
        for (int d = 0; d < 3; ++d) cell_w(x[d] / dx - (float)ar.base[d], ar.w[d]);
      }
      const int lb0 = ar.base[0] - o0, lb1 = ar.base[1] - o1, lb2 = ar.base[2] - o2;
      const bool outside = live && (lb0 < 0 || lb0 > 5 || lb1 < 0 || lb1 > 5 || lb2 < 0 || lb2 > 5);
      if (outside) atomicOr(err, kErrArena);
      const bool ok = live && !outside;
      float v[3] = {0.f, 0.f, 0.f};
      float C[9] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      float xn[3], Fn[9];
      if (ok) {
        gather_nodes(vel, lb0, lb1, lb2, ar, dx, v, C);
        if constexpr (!kCell)  // the cell kernel keeps B (no D_inv): C = B Dinv is formed below
#pragma unroll
          for (int k = 0; k < 9; ++k) C[k] *= D_inv;
        // F <- (I + dt C) F, column-major (G2P.hpp:75-78); the cell kernel's
        // C is B scaled per column by Dinv (G2C2P.hpp:231-253)
        float Cs[9];
        if constexpr (kCell) {
#pragma clang fp contract(off)
          float Dinv[3];
          cell_dinv(x, dx, (float)1 / dx, Dinv);
#pragma unroll
          for (int k = 0; k < 9; ++k) Cs[k] = C[k] * Dinv[k / 3];
        } else {
#pragma unroll
          for (int k = 0; k < 9; ++k) Cs[k] = C[k];
        }
#pragma unroll
        for (int j = 0; j < 3; ++j)
#pragma unroll
          for (int r = 0; r < 3; ++r) {
            const float a0 = Cs[r] * dt + (r == 0 ? 1.f : 0.f);
            const float a1 = Cs[r + 3] * dt + (r == 1 ? 1.f : 0.f);
            const float a2 = Cs[r + 6] * dt + (r == 2 ? 1.f : 0.f);
            Fn[r + 3 * j] = a0 * F[3 * j] + a1 * F[3 * j + 1] + a2 * F[3 * j + 2];
          }
#pragma unroll
        for (int d = 0; d < 3; ++d) xn[d] = x[d] + v[d] * dt;
      } else {
        // a particle outside its bucket's arena keeps its state (the error is
        // reported at the next sync)
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          xn[d] = x[d];
          v[d] = outside ? ps.v[3 * p + d] : 0.f;
        }
#pragma unroll
        for (int k = 0; k < 9; ++k) {
          Fn[k] = F[k];
          C[k] = outside ? ps.C[9 * p + k] : 0.f;
        }
      }
      if (more) load_ahead(pnext);
      if (kReorder) {
        // destination slots off + i0 + lane are contiguous by construction
        const int64_t q = (int64_t)off + i0 + lane;
        if (live) {
          out.m[q] = mcopy;
          if (ps.logJp) out.logJp[q] = ljcopy;
          if (out.id) out.id[q] = idcopy;
        }
        wave_store_rows<3>(out.x, (int64_t)off + i0, cw, stage, xn);
        wave_store_rows<3>(out.v, (int64_t)off + i0, cw, stage, v);
        wave_store_rows<9>(out.C, (int64_t)off + i0, cw, stage, C);
        wave_store_rows<9>(out.F, (int64_t)off + i0, cw, stage, Fn);
        if constexpr (kNext >= 0) {
          // the next substep's P2G stress from F_new and the logJp this
          // substep leaves (P2G.hpp:57-100 on the stored F)
          float PF[9] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
          if (live) {
            bool f64 = false;
            float lj = ljcopy;
            stress_any(ns.m, Fn, lj, PF, f64);
            if (kNext == 1) ns.lj_next[q] = lj;
            fp64_used += f64 ? 1u : 0u;
          }
          wave_store_rows<9>(ns.contrib, (int64_t)off + i0, cw, stage, PF);
        }
      } else if (contig && ballot(outside) == 0) {
        wave_store_rows<3>(ps.x, p0, cw, stage, xn);
        wave_store_rows<3>(ps.v, p0, cw, stage, v);
        wave_store_rows<9>(ps.C, p0, cw, stage, C);
        wave_store_rows<9>(ps.F, p0, cw, stage, Fn);
      } else if (ok) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          ps.x[3 * p + d] = xn[d];
          ps.v[3 * p + d] = v[d];
        }
#pragma unroll
        for (int k = 0; k < 9; ++k) {
          ps.C[9 * p + k] = C[k];
          ps.F[9 * p + k] = Fn[k];
        }
      }
    }
    __syncthreads();
  }
  if (kNext >= 0 && fp64_used) atomicAdd(&counters[kCtrFp64], fp64_used);
}

// The gather half of G2PTransfer's implicit twin, G2P2GTransfer::operator()
// (simulation/transfer/G2P2G.hpp:49-84), per bucket as G2P: the bucket's
// 8^3 node velocities from the vector v (3 floats per node, node = block * 64
// + cell) are staged in LDS, and each particle takes C from its 27 staged
// nodes and writes F = (I + dt C) F_old to Fout[9 p]. The model's stress of
// that F is the ordinary stress pass (full occupancy; the SVD inside this
// kernel held it to three waves per SIMD), the force scatter P2G's.
__global__ __launch_bounds__(kG2PThreads) void g2p2g_gather_kernel(ParticlesView ps, TableView t, SortView sv,
                                                                   const int32_t* __restrict__ nbr_tab,
                                                                   const float* __restrict__ v, int32_t grid_cap,
                                                                   float dt, float dx, float* __restrict__ Fout,
                                                                   uint32_t* err) {
  __shared__ float4 vel[kVelNodes];
  __shared__ int32_t nbr[8];
  __shared__ float4 stage4[kG2PThreads / kWave][stage_floats(9) / 4];
  const int32_t nb = bounded_blocks(t, sv, grid_cap, err);
  const float dx_inv = (float)1 / dx;
  const float D_inv = 4.f * dx_inv * dx_inv;
  const int wave = uniform((int32_t)(threadIdx.x / kWave)), lane = lane_id();
  float* stage = reinterpret_cast<float*>(stage4[wave]);
  for (int32_t b = blockIdx.x; b < nb; b += gridDim.x) {
    const int32_t cnt = sv.counts[b];
    const int32_t off = sv.offsets[b];
    if (cnt <= 0 || off < 0 || (int64_t)off + cnt > ps.n) continue;
    if (threadIdx.x < 8) {
      const int32_t r = nbr_tab[8 * (int64_t)b + threadIdx.x];
      nbr[threadIdx.x] = r;
      if (r < 0) atomicOr(err, kErrMissingBlock);
    }
    const int32_t o0 = t.active[3 * (int64_t)b] * 4, o1 = t.active[3 * (int64_t)b + 1] * 4,
                  o2 = t.active[3 * (int64_t)b + 2] * 4;
    int32_t first = -1;
    if (wave * kWave + lane < cnt) first = sv.indices[off + wave * kWave + lane];
    __syncthreads();
    for (int s = threadIdx.x; s < kArena8; s += kG2PThreads) {
      const int nbi = s >> 6, cell = s & 63;
      const int r0 = ((nbi >> 2) & 1) * 4 + ((cell >> 4) & 3);
      const int r1 = ((nbi >> 1) & 1) * 4 + ((cell >> 2) & 3);
      const int r2 = (nbi & 1) * 4 + (cell & 3);
      const int32_t gb = nbr[nbi];
      float4 w = make_float4(0.f, 0.f, 0.f, 0.f);
      if (gb >= 0 && gb < grid_cap) {
        const float* vp = v + 3 * ((int64_t)gb * kBlockCells + cell);
        w = make_float4(vp[0], vp[1], vp[2], 0.f);
      }
      vel[vel_at(r0, r1, r2)] = w;
    }
    __syncthreads();
    for (int32_t i0 = wave * kWave; i0 < cnt; i0 += kG2PThreads) {
      const int32_t cw = min(kWave, cnt - i0);
      const bool valid = lane < cw;
      const int64_t p = valid ? (int64_t)(i0 == wave * kWave ? first : sv.indices[off + i0 + lane]) : -1;
      const bool bad = valid && (p < 0 || p >= ps.n);
      if (bad) atomicOr(err, kErrCapacity);
      const bool live = valid && !bad;
      int64_t p0;
      const bool contig = wave_contiguous(p, live, p0) && ballot(bad) == 0;
      float x[3], F[9];
      const int64_t row = live ? p : 0;
      load_row(ps.x, row, x);
      load_row(ps.F, row, F);
      Arena ar;
      make_arena(x[0], x[1], x[2], dx, ar);
      const int lb0 = ar.base[0] - o0, lb1 = ar.base[1] - o1, lb2 = ar.base[2] - o2;
      const bool outside = live && (lb0 < 0 || lb0 > 5 || lb1 < 0 || lb1 > 5 || lb2 < 0 || lb2 > 5);
      if (outside) atomicOr(err, kErrArena);
      const bool ok = live && !outside;
      float Fn[9];
#pragma unroll
      for (int k = 0; k < 9; ++k) Fn[k] = F[k];
      if (ok) {
        float v[3] = {0.f, 0.f, 0.f}, C[9] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        gather_nodes(vel, lb0, lb1, lb2, ar, dx, v, C);
#pragma unroll
        for (int k = 0; k < 9; ++k) C[k] *= D_inv;
        // F = (I + dt C) F_old, column-major (G2P2G.hpp:81-84)
#pragma unroll
        for (int j = 0; j < 3; ++j)
#pragma unroll
          for (int r = 0; r < 3; ++r) {
            const float a0 = C[r] * dt + (r == 0 ? 1.f : 0.f);
            const float a1 = C[r + 3] * dt + (r == 1 ? 1.f : 0.f);
            const float a2 = C[r + 6] * dt + (r == 2 ? 1.f : 0.f);
            Fn[r + 3 * j] = a0 * F[3 * j] + a1 * F[3 * j + 1] + a2 * F[3 * j + 2];
          }
      }
      if (contig && ballot(outside) == 0) {
        wave_store_rows<9>(Fout, p0, cw, stage, Fn);
      } else if (live) {
#pragma unroll
        for (int k = 0; k < 9; ++k) Fout[9 * p + k] = Fn[k];
      }
    }
    __syncthreads();
  }
}

// Vector::reorder gather (container/Vector.hpp:617-646) of every attribute
__global__ __launch_bounds__(kThreads) void reorder_kernel(ParticlesView in, ParticlesView out,
                                                           const int32_t* __restrict__ map, uint32_t* err) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < out.n; i += stride) {
    const int64_t p = map[i];
    if (p < 0 || p >= in.n) {
      atomicOr(err, kErrCapacity);
      continue;
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      out.x[3 * i + d] = in.x[3 * p + d];
      out.v[3 * i + d] = in.v[3 * p + d];
    }
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      out.C[9 * i + k] = in.C[9 * p + k];
      out.F[9 * i + k] = in.F[9 * p + k];
    }
    out.m[i] = in.m[p];
    if (in.logJp) out.logJp[i] = in.logJp[p];
    if (out.id) out.id[i] = in.id ? in.id[p] : (int32_t)p;
  }
}

// ImplicitMPMSystem::Projector (simulation/mpm/ImplicitMPM.hpp:65-101) for
// every boundary at once: a node with mass resolves its vector against the
// plane colliders, the general colliders and the level-set boundary in that
// order; a node without mass is cleared.
__global__ __launch_bounds__(kThreads) void implicit_project_kernel(const float* __restrict__ grid, int32_t grid_cap,
                                                                    TableView t, float dx, Colliders cols,
                                                                    GeneralColliders gen, float* dof) {
#pragma clang fp contract(off)
  int32_t nb = *t.cnt;
  if (nb > grid_cap) nb = grid_cap;
  const int64_t nodes = (int64_t)nb * kBlockCells;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < nodes; i += stride) {
    const int32_t b = (int32_t)(i >> 6);
    const int cell = (int)(i & 63);
    float* dv = dof + 3 * i;
    if (!(grid[grid_at(b, 0, cell)] > 0.f)) {
      dv[0] = dv[1] = dv[2] = 0.f;
      continue;
    }
    const int32_t k0 = t.active[3 * (int64_t)b], k1 = t.active[3 * (int64_t)b + 1], k2 = t.active[3 * (int64_t)b + 2];
    const float pos[3] = {((float)k0 * 4.f + (float)((cell >> 4) & 3)) * dx,
                          ((float)k1 * 4.f + (float)((cell >> 2) & 3)) * dx,
                          ((float)k2 * 4.f + (float)(cell & 3)) * dx};
    float v[3] = {dv[0], dv[1], dv[2]};
    for (int c = 0; c < cols.n; ++c) {
      const PlaneCollider& pc = cols.c[c];
      const float phi = pc.normal[0] * (pos[0] - pc.origin[0]) + pc.normal[1] * (pos[1] - pc.origin[1]) +
                        pc.normal[2] * (pos[2] - pc.origin[2]);
      if (phi < 0.f) {
        if (pc.type == 0) {
          v[0] = v[1] = v[2] = 0.f;
        } else {
          const float proj = pc.normal[0] * v[0] + pc.normal[1] * v[1] + pc.normal[2] * v[2];
          if ((pc.type == 2 && proj < 0.f) || pc.type == 1) {
            v[0] -= proj * pc.normal[0];
            v[1] -= proj * pc.normal[1];
            v[2] -= proj * pc.normal[2];
          }
        }
      }
    }
    for (int c = 0; c < gen.n; ++c) resolve_general(gen.c[c], pos, v);
    if (gen.ls.on) levelset_resolve(gen.ls, pos, v);
    dv[0] = v[0];
    dv[1] = v[1];
    dv[2] = v[2];
  }
}

}  // namespace

hipError_t implicit_project(const float* grid, int32_t grid_cap, const TableView& t, float dx, const Colliders& cols,
                            const GeneralColliders& gen, float* dof, hipStream_t s) {
  if (cols.n == 0 && gen.n == 0 && !gen.ls.on) return hipSuccess;  // no boundary: nothing changes
  implicit_project_kernel<<<persistent_groups(), kThreads, 0, s>>>(grid, grid_cap, t, dx, cols, gen, dof);
  return hipGetLastError();
}

// Dynamic LDS the stress pass reserves (and does not use) when it runs beside
// the sparsity stages: with its 9,280 bytes of static LDS, three workgroups
// fit in a CU's 160 KiB and a fourth does not. Uncapped, its workgroups (120
// VGPRs, four waves per SIMD) fill the register files and the sparsity
// kernels wait for CUs; capped, both finish earlier (measured on the 16M
// sand column: 2.52 -> 2.46 ms per substep; a cap of two is slower again).
constexpr size_t kStressLdsReserve = 40960;

hipError_t check_launch_limits(int device) {
  int max_lds = 0;
  hipError_t e = hipDeviceGetAttribute(&max_lds, hipDeviceAttributeMaxSharedMemoryPerBlock, device);
  if (e != hipSuccess) return e;
  const void* kernels[] = {
      reinterpret_cast<const void*>(&stress_kernel<0, false>), reinterpret_cast<const void*>(&stress_kernel<1, false>),
      reinterpret_cast<const void*>(&stress_kernel<0, true>), reinterpret_cast<const void*>(&stress_kernel<1, true>),
      reinterpret_cast<const void*>(&stress_kernel<2, true>), reinterpret_cast<const void*>(&p2g_kernel<0, false>),
      reinterpret_cast<const void*>(&p2g_kernel<1, false>), reinterpret_cast<const void*>(&p2g_kernel<0, true>),
      reinterpret_cast<const void*>(&p2g_kernel<1, true>),
      reinterpret_cast<const void*>(&g2p_kernel<false, -1>), reinterpret_cast<const void*>(&g2p_kernel<true, -1>),
      reinterpret_cast<const void*>(&g2p_kernel<true, 0>), reinterpret_cast<const void*>(&g2p_kernel<true, 1>),
      reinterpret_cast<const void*>(&g2p_kernel<true, -1, true>),
      reinterpret_cast<const void*>(&g2p_kernel<false, -1, true>),
      reinterpret_cast<const void*>(&p2g_kernel<0, false, true>),
      reinterpret_cast<const void*>(&g2p_kernel<false, -1, false, true>),
      reinterpret_cast<const void*>(&p2g_kernel<0, false, false, 1>),
      reinterpret_cast<const void*>(&p2g_kernel<0, true, false, 1>),
      reinterpret_cast<const void*>(&p2g_kernel<0, false, false, kWideTile>),
      reinterpret_cast<const void*>(&g2p_kernel<true, -1, false, false, kG2PWide>),
      reinterpret_cast<const void*>(&g2p_kernel<false, -1, false, false, kG2PWide>),
      reinterpret_cast<const void*>(&g2p_kernel<true, -1, false, false, 256>),
      reinterpret_cast<const void*>(&g2p_kernel<true, -1, true, false, 256>),
      reinterpret_cast<const void*>(&g2p2g_gather_kernel),
      reinterpret_cast<const void*>(&p2g_kernel<2, false>),
      reinterpret_cast<const void*>(&p2g_kernel<2, true>),
      reinterpret_cast<const void*>(&g2p_kernel<true, -1, false, true>)};
  for (int i = 0; i < (int)(sizeof(kernels) / sizeof(kernels[0])); ++i) {
    hipFuncAttributes attr;
    e = hipFuncGetAttributes(&attr, kernels[i]);
    if (e != hipSuccess) return e;
    const size_t extra = i < 5 ? kStressLdsReserve : 0;  // the stress kernels' reserve
    if (attr.sharedSizeBytes + extra > (size_t)max_lds) return hipErrorInvalidConfiguration;
  }
  return closure_launch_limits();
}

hipError_t grid_clear(float* grid, const int32_t* nblocks_dev, int32_t cap_blocks, hipStream_t s) {
  const int64_t total = (int64_t)cap_blocks * kChannels * kBlockCells / 4;
  grid_clear_kernel<<<groups_for(total, kThreads), kThreads, 0, s>>>(grid, nblocks_dev, cap_blocks);
  return hipGetLastError();
}

hipError_t stress(const Model& m, const ParticlesView& ps, Workspace& ws, hipStream_t s, const ClosureView* closure,
                  float* contrib, bool beside_sparsity, const SceneSet* ss) {
  if (ps.n <= 0) return hipSuccess;
  float* out = contrib ? contrib : ws.contrib;
  const int64_t waves = (ps.n + kWave - 1) / kWave;
  const int g = groups_for(waves * kWave, kThreads);
  const size_t lds = beside_sparsity ? kStressLdsReserve : 0;
  const bool multi = ss && ss->n > 0;
  const SceneSet sset = multi ? *ss : SceneSet{};
  auto launch = [&](auto kernel) {
    kernel<<<g, kThreads, lds, s>>>(m, ps, out, ws.counters, sset);
    return hipGetLastError();
  };
  if (multi) {  // a batch without the FP64 SVD has no stress pass
    if (closure) return hipErrorNotSupported;
    return launch(stress_kernel<2, true>);
  }
  if (closure && m.kind == 1 && m.mu != 0.f) return stress_closure(m, *closure, ps, out, ws, s);
  const bool gap = m.fp64_gap > 0.f;
  if (m.kind == 0) return gap ? launch(stress_kernel<0, true>) : launch(stress_kernel<0, false>);
  return gap ? launch(stress_kernel<1, true>) : launch(stress_kernel<1, false>);
}

namespace {

// Workgroups of the per-bucket kernels: the policy's counts, else P2G as many
// as are resident and G2P one per bucket up to 32,768; no more than there can
// be buckets.
int bucket_bound(const SortView& sv, int32_t grid_cap) {
  const int32_t cap = grid_cap < sv.cap_blocks ? grid_cap : sv.cap_blocks;
  return cap > 1 ? cap : 1;
}
// The caller's capacity for blocks is at most `line`. The launch cannot know how
// many buckets there will be, but grids are sized for a table of at least twice
// the blocks with their enlargement, so at most half the capacity is in use.
bool wide_buckets(const SortView& sv, int32_t grid_cap, int line) { return bucket_bound(sv, grid_cap) <= line; }
int p2g_groups(const Workspace& ws, const SortView& sv, int32_t grid_cap) {
  const int g = ws.grid_p2g > 0 ? ws.grid_p2g : default_p2g_groups(ws.p2g_chunk);
  const int cap = bucket_bound(sv, grid_cap);
  return g < cap ? g : cap;
}
int g2p_groups(const Workspace& ws, const SortView& sv, int32_t grid_cap) {
  const int g = ws.grid_g2p > 0 ? ws.grid_g2p : default_g2p_groups();
  const int cap = bucket_bound(sv, grid_cap);
  return g < cap ? g : cap;
}

}  // namespace

hipError_t p2g_scatter(const ParticlesView& ps, const TableView& t, const SortView& sv, float* grid,
                       int32_t grid_cap, float dt, float dx, bool fold, Workspace& ws, hipStream_t s,
                       const SceneSet* ss, const StressFrom& st) {
  const int g = p2g_groups(ws, sv, grid_cap);
  const bool multi = ss && ss->n > 0;
  const SceneSet sset = multi ? *ss : SceneSet{};
  const bool tile1 = ws.p2g_chunk == 256;  // the folded launches take the tuned tile
  if (fold && ws.cell && !multi)  // the substep's P2C2G (one tile)
    p2g_kernel<0, false, true><<<g, kP2GThreads, 0, s>>>(ps, ws.contrib, st, t, sv, ws.nbr, grid, grid_cap, dt, dx,
                                                         ws.err, sset, 1);
  else if (fold && multi && tile1)
    p2g_kernel<0, true, false, 1><<<g, p2g_threads(1), 0, s>>>(ps, ws.contrib, st, t, sv, ws.nbr, grid, grid_cap, dt, dx,
                                                               ws.err, sset, 1);
  else if (fold && multi)
    p2g_kernel<0, true><<<g, kP2GThreads, 0, s>>>(ps, ws.contrib, st, t, sv, ws.nbr, grid, grid_cap, dt, dx, ws.err, sset, 1);
  else if (fold && tile1)
    p2g_kernel<0, false, false, 1><<<g, p2g_threads(1), 0, s>>>(ps, ws.contrib, st, t, sv, ws.nbr, grid, grid_cap, dt,
                                                                dx, ws.err, sset, 1);
  else if (fold && ws.p2g_chunk == 0 && wide_buckets(sv, grid_cap, kP2GWideBuckets))
    p2g_kernel<0, false, false, kWideTile><<<g, p2g_threads(kWideTile), 0, s>>>(ps, ws.contrib, st, t, sv, ws.nbr, grid,
                                                                               grid_cap, dt, dx, ws.err, sset, 1);
  else if (fold)
    p2g_kernel<0, false><<<g, kP2GThreads, 0, s>>>(ps, ws.contrib, st, t, sv, ws.nbr, grid, grid_cap, dt, dx, ws.err, sset, 1);
  else if (multi) {
    // the force kept in channels 4..6: momentum, then the force
    p2g_kernel<1, true><<<g, kP2GThreads, 0, s>>>(ps, ws.contrib, st, t, sv, ws.nbr, grid, grid_cap, dt, dx, ws.err, sset, 1);
    p2g_kernel<2, true><<<g, kP2GThreads, 0, s>>>(ps, ws.contrib, st, t, sv, ws.nbr, grid, grid_cap, dt, dx, ws.err, sset, 4);
  } else {
    p2g_kernel<1, false><<<g, kP2GThreads, 0, s>>>(ps, ws.contrib, st, t, sv, ws.nbr, grid, grid_cap, dt, dx, ws.err, sset, 1);
    p2g_kernel<2, false><<<g, kP2GThreads, 0, s>>>(ps, ws.contrib, st, t, sv, ws.nbr, grid, grid_cap, dt, dx, ws.err, sset, 4);
  }
  return hipGetLastError();
}

hipError_t p2c2g_scatter(const ParticlesView& ps, const TableView& t, const SortView& sv, float* grid,
                         int32_t grid_cap, float dt, float dx, Workspace& ws, hipStream_t s, const StressFrom& st) {
  const int g = p2g_groups(ws, sv, grid_cap);
  p2g_kernel<0, false, true><<<g, kP2GThreads, 0, s>>>(ps, ws.contrib, st, t, sv, ws.nbr, grid, grid_cap, dt, dx,
                                                       ws.err, SceneSet{}, 1);
  return hipGetLastError();
}

hipError_t p2g_force_scatter(const ParticlesView& ps, const TableView& t, const SortView& sv, float* grid,
                             int32_t grid_cap, float dt, float dx, Workspace& ws, hipStream_t s,
                             const StressFrom& st) {
  const int g = p2g_groups(ws, sv, grid_cap);
  p2g_kernel<2, false><<<g, kP2GThreads, 0, s>>>(ps, ws.contrib, st, t, sv, ws.nbr, grid, grid_cap, dt, dx, ws.err, SceneSet{}, 1);
  return hipGetLastError();
}

hipError_t g2p2g_gather(const ParticlesView& ps, const TableView& t, const SortView& sv, const float* v,
                        int32_t grid_cap, float dt, float dx, float* Fout, Workspace& ws, hipStream_t s) {
  if (ps.n == 0) return hipSuccess;
  const int g = g2p_groups(ws, sv, grid_cap);
  g2p2g_gather_kernel<<<g, kG2PThreads, 0, s>>>(ps, t, sv, ws.nbr, v, grid_cap, dt, dx, Fout, ws.err);
  return hipGetLastError();
}

hipError_t g2c2p(const ParticlesView& ps, const TableView& t, const SortView& sv, const float* grid, int32_t grid_cap,
                 float dt, float dx, Workspace& ws, hipStream_t s) {
  const int g = g2p_groups(ws, sv, grid_cap);
  g2p_kernel<false, -1, false, true><<<g, kG2PThreads, 0, s>>>(ps, ps, t, sv, ws.nbr, grid, grid_cap, dt, dx,
                                                               NextStress{}, ws.err, ws.counters, SceneSet{});
  return hipGetLastError();
}

hipError_t grid_update(float* grid, int32_t grid_cap, const TableView& t, float dt, const float extf[3],
                       const Colliders& cols, float dx, int fold_rhs, Workspace& ws, hipStream_t s,
                       const SceneSet* ss, const GeneralColliders* gen) {
  const bool multi = ss && ss->n > 0;
  const SceneSet sset = multi ? *ss : SceneSet{};
  auto launch = [&](auto kernel, auto g) {
    kernel<<<persistent_groups(), kThreads, 0, s>>>(grid, grid_cap, t, dt, extf[0], extf[1], extf[2], cols, dx,
                                                    fold_rhs, ws.counters, ws.err, sset, g);
  };
  if (gen && (gen->n > 0 || gen->ls.on)) {
    if (multi)
      launch(grid_update_kernel<true, GeneralColliders>, *gen);
    else
      launch(grid_update_kernel<false, GeneralColliders>, *gen);
  } else if (multi) {
    launch(grid_update_kernel<true, NoColliders>, NoColliders{});
  } else {
    launch(grid_update_kernel<false, NoColliders>, NoColliders{});
  }
  return hipGetLastError();
}

hipError_t grid_angular_momentum(const float* grid, int32_t grid_cap, const TableView& t, float dx, int mchn,
                                 int mvchn, double* sum, Workspace& ws, hipStream_t s) {
  angular_momentum_kernel<<<1024, kThreads, 0, s>>>(grid, grid_cap, t, dx, mchn, mvchn, sum, ws.err);
  return hipGetLastError();
}

hipError_t g2p(const ParticlesView& ps, const ParticlesView* out, const TableView& t, const SortView& sv,
               const float* grid, int32_t grid_cap, float dt, float dx, Workspace& ws, hipStream_t s,
               const NextStress* next, const SceneSet* ss) {
  const int g = g2p_groups(ws, sv, grid_cap);
  NextStress ns{};
  if (next) ns = *next;
  const SceneSet sset = ss ? *ss : SceneSet{};
  if (ws.cell) {  // the substep's G2C2P (no batch, no fused stress; one tile)
    if ((next && next->contrib) || sset.n > 0) return hipErrorInvalidValue;
    if (out)
      g2p_kernel<true, -1, false, true><<<g, kG2PThreads, 0, s>>>(ps, *out, t, sv, ws.nbr, grid, grid_cap, dt, dx,
                                                                  ns, ws.err, ws.counters, sset);
    else
      g2p_kernel<false, -1, false, true><<<g, kG2PThreads, 0, s>>>(ps, ps, t, sv, ws.nbr, grid, grid_cap, dt, dx,
                                                                   ns, ws.err, ws.counters, sset);
  } else if (next && next->contrib) {
    if (!out || sset.n > 0) return hipErrorInvalidValue;
    if (ns.m.kind == 0)
      g2p_kernel<true, 0><<<g, kG2PThreads, 0, s>>>(ps, *out, t, sv, ws.nbr, grid, grid_cap, dt, dx, ns, ws.err,
                                                    ws.counters, sset);
    else
      g2p_kernel<true, 1><<<g, kG2PThreads, 0, s>>>(ps, *out, t, sv, ws.nbr, grid, grid_cap, dt, dx, ns, ws.err,
                                                    ws.counters, sset);
  } else if (out && sset.n > 0 && ws.g2p_threads == 256) {
    g2p_kernel<true, -1, true, false, 256><<<g, 256, 0, s>>>(ps, *out, t, sv, ws.nbr, grid, grid_cap, dt, dx, ns,
                                                             ws.err, ws.counters, sset);
  } else if (out && sset.n > 0) {
    g2p_kernel<true, -1, true><<<g, kG2PThreads, 0, s>>>(ps, *out, t, sv, ws.nbr, grid, grid_cap, dt, dx, ns, ws.err,
                                                         ws.counters, sset);
  } else if (out && ws.g2p_threads == 256) {
    g2p_kernel<true, -1, false, false, 256><<<g, 256, 0, s>>>(ps, *out, t, sv, ws.nbr, grid, grid_cap, dt, dx, ns,
                                                              ws.err, ws.counters, sset);
  } else if (sset.n == 0 && ws.g2p_threads == 0 && wide_buckets(sv, grid_cap, kG2PWideBuckets)) {
    if (out)
      g2p_kernel<true, -1, false, false, kG2PWide><<<g, kG2PWide, 0, s>>>(ps, *out, t, sv, ws.nbr, grid, grid_cap, dt,
                                                                          dx, ns, ws.err, ws.counters, sset);
    else
      g2p_kernel<false, -1, false, false, kG2PWide><<<g, kG2PWide, 0, s>>>(ps, ps, t, sv, ws.nbr, grid, grid_cap, dt,
                                                                           dx, ns, ws.err, ws.counters, sset);
  } else if (out) {
    g2p_kernel<true, -1><<<g, kG2PThreads, 0, s>>>(ps, *out, t, sv, ws.nbr, grid, grid_cap, dt, dx, ns, ws.err,
                                                   ws.counters, sset);
  } else if (sset.n > 0) {
    g2p_kernel<false, -1, true><<<g, kG2PThreads, 0, s>>>(ps, ps, t, sv, ws.nbr, grid, grid_cap, dt, dx, ns, ws.err,
                                                          ws.counters, sset);
  } else {
    g2p_kernel<false, -1><<<g, kG2PThreads, 0, s>>>(ps, ps, t, sv, ws.nbr, grid, grid_cap, dt, dx, ns, ws.err,
                                                    ws.counters, sset);
  }
  return hipGetLastError();
}

hipError_t reorder_particles(const ParticlesView& in, const ParticlesView& out, const int32_t* map,
                             Workspace& ws, hipStream_t s) {
  if (out.n <= 0) return hipSuccess;
  reorder_kernel<<<groups_for(out.n, kThreads), kThreads, 0, s>>>(in, out, map, ws.err);
  return hipGetLastError();
}

}  // namespace zsmpm
