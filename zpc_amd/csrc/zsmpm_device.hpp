// Device-side building blocks of the gfx950 MLS-MPM substep: block keys and
// the zpc table hash, 64-lane wavefront helpers, the 3x3 SVD and the two
// constitutive models. Everything here is __device__ code for CDNA4 (wave64).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "rowspan.hpp"

namespace zsmpm {

constexpr int kWave = 64;
constexpr int kChannels = 7;        // m, v(3), rhs(3): Grids{{m,1},{v,3},{rhs,3}}
constexpr int kBlockCells = 64;     // 4^3 cells per block
constexpr int32_t kKeySentinel = 0x7fffffff;
constexpr int32_t kProbeStep = 127;
constexpr uint64_t kEmpty64 = ~0ull;
constexpr int32_t kPackBias = 1 << 20;  // packed keys hold components in [-2^20, 2^20)

// error bits raised by kernels, read back by the host at synchronisation points
enum : uint32_t {
  kErrTableFull = 1u << 0,    // a probe walked the whole table
  kErrKeyRange = 1u << 1,     // a block key does not fit the 21-bit packing
  kErrArena = 1u << 2,        // a stencil fell outside its block's 8^3 arena
  kErrCapacity = 1u << 3,     // more blocks / runs than the buffers hold
  kErrMissingBlock = 1u << 4  // a neighbour block was not active (table not enlarged)
};

// ---------------------------------------------------------------------------
// zpc's table hash (container/HashTable.hpp:496-500 + math/Hash.hpp:17-27):
// 64-bit hash_combine seeded by the sign-extended first component, truncated
// to i32, reduced with (h % T + T) % T (:359).
// ---------------------------------------------------------------------------
__device__ __forceinline__ int32_t zpc_hash(int32_t k0, int32_t k1, int32_t k2) {
  uint64_t r = (uint64_t)(int64_t)k0;
  r ^= (uint64_t)(int64_t)k1 + 0x9e3779b97f4a7c15ull + (r << 12) + (r >> 4);
  r ^= (uint64_t)(int64_t)k2 + 0x9e3779b97f4a7c15ull + (r << 12) + (r >> 4);
  return (int32_t)(uint32_t)r;
}
__device__ __forceinline__ int32_t zpc_home(int32_t k0, int32_t k1, int32_t k2, int32_t T) {
  const int32_t h = zpc_hash(k0, k1, k2);
  return (h % T + T) % T;
}

// Block key of a position (SparsityOp.hpp:72-77): c = floor(x*dxinv + disp) + offset,
// key = floor(c / blockLen). Rounded exactly as written (no contraction), so the
// integer result matches the host path bit for bit.
__device__ __forceinline__ void block_key(float x0, float x1, float x2, float dxinv, int blockLen,
                                          int offset, float disp, int32_t& k0, int32_t& k1,
                                          int32_t& k2) {
#pragma clang fp contract(off)
  const float xs[3] = {x0, x1, x2};
  int32_t out[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const float t = xs[d] * dxinv;
    const int32_t c = (int32_t)floorf(t + disp) + offset;
    if ((blockLen & (blockLen - 1)) == 0) {
      out[d] = c >> (__ffs(blockLen) - 1);  // floor division by a power of two
    } else {
      const int32_t b = c + (c < 0 ? -blockLen + 1 : 0);
      out[d] = b / blockLen;
    }
  }
  k0 = out[0];
  k1 = out[1];
  k2 = out[2];
}

__device__ __forceinline__ bool key_packable(int32_t k0, int32_t k1, int32_t k2) {
  return k0 >= -kPackBias && k0 < kPackBias && k1 >= -kPackBias && k1 < kPackBias &&
         k2 >= -kPackBias && k2 < kPackBias;
}
__device__ __forceinline__ uint64_t pack_key(int32_t k0, int32_t k1, int32_t k2) {
  return ((uint64_t)(uint32_t)(k0 + kPackBias) << 42) | ((uint64_t)(uint32_t)(k1 + kPackBias) << 21) |
         (uint64_t)(uint32_t)(k2 + kPackBias);
}
__device__ __forceinline__ void unpack_key(uint64_t p, int32_t& k0, int32_t& k1, int32_t& k2) {
  k0 = (int32_t)((p >> 42) & 0x1fffff) - kPackBias;
  k1 = (int32_t)((p >> 21) & 0x1fffff) - kPackBias;
  k2 = (int32_t)(p & 0x1fffff) - kPackBias;
}
// murmur3 finaliser: slot hash of the scratch (dedup) table
__device__ __forceinline__ uint64_t mix64(uint64_t z) {
  z ^= z >> 33;
  z *= 0xff51afd7ed558ccdull;
  z ^= z >> 33;
  z *= 0xc4ceb9fe1a85ec53ull;
  z ^= z >> 33;
  return z;
}

// a positive normal power of two: x / d and x * (1 / d) round alike
__device__ __forceinline__ bool is_pow2(float d) {
  const uint32_t u = __float_as_uint(d);
  return (u & 0x7fffffu) == 0u && u > 0x00800000u && u < 0x7e800000u;
}

// ---------------------------------------------------------------------------
// wavefront helpers (wave64)
// ---------------------------------------------------------------------------
__device__ __forceinline__ int lane_id() { return (int)__lane_id(); }
__device__ __forceinline__ uint64_t lanemask_lt() { return (1ull << lane_id()) - 1ull; }
__device__ __forceinline__ uint64_t ballot(bool p) { return __ballot(p); }

template <typename T>
__device__ __forceinline__ T shfl(T v, int src) {
  return __shfl(v, src, kWave);
}

// Value of the first active lane as a wave-uniform (scalar) value. Called
// with the whole wave active, that is lane 0.
__device__ __forceinline__ int32_t uniform(int32_t v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ int64_t uniform(int64_t v) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int32_t)(uint32_t)v);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int32_t)(uint32_t)((uint64_t)v >> 32));
  return (int64_t)(((uint64_t)hi << 32) | lo);
}

// Wave-uniform, called with the whole wave active: do the valid lanes hold
// one contiguous run p0 + lane (lane 0 valid)? p0 receives lane 0's index.
__device__ __forceinline__ bool wave_contiguous(int64_t p, bool valid, int64_t& p0) {
  p0 = uniform(p);
  const uint64_t vm = ballot(valid);
  return (vm & 1ull) != 0 && ballot(valid && p == p0 + lane_id()) == vm;
}

// Orders a wave's own LDS writes before its later LDS reads by other lanes
// (the LDS serves one wave's instructions in issue order; this keeps the
// compiler from moving accesses across the point).
__device__ __forceinline__ void wave_lds_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_wave_barrier();
  asm volatile("" ::: "memory");
}

// Particle rows are streamed: every kernel reads a row once and writes it
// once, and the next reader is a later kernel. Their 16-byte vector loads and
// stores are non-temporal, so the streams do not evict what is re-used from
// L2 (staged grid velocities, table and bucket arrays). On the 16M sand
// column this took the substep from 2.46 to 2.36 ms (G2P 0.86 -> 0.82 ms).
typedef float zs_f4 __attribute__((ext_vector_type(4)));

// Split-phase load of rows q0 .. q0+cnt-1 (cnt <= 64) of W floats: issue()
// puts the wave's global vector loads in flight (no LDS, no wait), finish()
// transposes them through the wave's LDS stage so lane l < cnt receives row
// q0 + l. Several RowLoads issued back to back cost one memory round trip.
// Both calls are made by the whole wave with wave-uniform q0, cnt.
template <int W>
struct RowLoad {
  static constexpr int kVec = (W * kWave / 4 + kWave - 1) / kWave;  // float4 per lane
  RowSpan r;
  float4 v[kVec];
  float head, tail;
  __device__ __forceinline__ void issue(const float* __restrict__ base, int64_t q0, int32_t cnt) {
    const int lane = lane_id();
    r = row_span((uint64_t)(uintptr_t)base, q0, cnt, W);
    const int64_t hn = r.a4 - r.a;
    const int64_t t0 = r.a4 + 4 * r.nvec;
    head = lane < hn ? base[r.a + lane] : 0.f;
    tail = lane < r.b - t0 ? base[t0 + lane] : 0.f;
#pragma unroll
    for (int k = 0; k < kVec; ++k) {
      const int64_t j = lane + (int64_t)k * kWave;
      if (j < r.nvec) {
        const zs_f4 t = __builtin_nontemporal_load(reinterpret_cast<const zs_f4*>(base + r.a4 + 4 * j));
        v[k] = make_float4(t.x, t.y, t.z, t.w);
      } else {
        v[k] = make_float4(0.f, 0.f, 0.f, 0.f);
      }
    }
  }
  __device__ __forceinline__ void finish(float* stage, int32_t cnt, float (&out)[W]) {
    const int lane = lane_id();
    const int64_t hn = r.a4 - r.a;
    const int64_t t0 = r.a4 + 4 * r.nvec;
    if (lane < hn) stage[r.shift + lane] = head;
#pragma unroll
    for (int k = 0; k < kVec; ++k) {
      const int64_t j = lane + (int64_t)k * kWave;
      if (j < r.nvec) *reinterpret_cast<float4*>(stage + r.shift + hn + 4 * j) = v[k];
    }
    if (lane < r.b - t0) stage[r.shift + (t0 - r.a) + lane] = tail;
    wave_lds_barrier();
    if (lane < cnt) {
#pragma unroll
      for (int k = 0; k < W; ++k) out[k] = stage[r.shift + lane * W + k];
    }
    wave_lds_barrier();
  }
};

// Row p of W floats (W a multiple of 3) by one lane, in 12-byte loads (rows are
// 4-byte aligned). Consecutive lanes read consecutive rows: the three loads of
// a 9-float row touch the same lines one after another.
typedef float zs_f3 __attribute__((ext_vector_type(3), aligned(4)));
template <int W>
__device__ __forceinline__ void load_row(const float* __restrict__ base, int64_t p, float (&out)[W]) {
  static_assert(W % 3 == 0, "rows of 3-vectors");
  const float* r = base + (int64_t)W * p;
#pragma unroll
  for (int k = 0; k < W; k += 3) {
    const zs_f3 t = *reinterpret_cast<const zs_f3*>(r + k);
    out[k] = t.x;
    out[k + 1] = t.y;
    out[k + 2] = t.z;
  }
}

// One-shot form: issue and finish.
template <int W>
__device__ __forceinline__ void wave_load_rows(const float* __restrict__ base, int64_t q0, int32_t cnt,
                                               float* stage, float (&out)[W]) {
  RowLoad<W> ld;
  ld.issue(base, q0, cnt);
  ld.finish(stage, cnt, out);
}

// The store counterpart: lane l < cnt provides row q0 + l.
template <int W>
__device__ __forceinline__ void wave_store_rows(float* __restrict__ base, int64_t q0, int32_t cnt, float* stage,
                                                const float (&in)[W]) {
  const int lane = lane_id();
  const RowSpan r = row_span((uint64_t)(uintptr_t)base, q0, cnt, W);
  if (lane < cnt) {
#pragma unroll
    for (int k = 0; k < W; ++k) stage[r.shift + lane * W + k] = in[k];
  }
  wave_lds_barrier();
  const int64_t head = r.a4 - r.a;
  if (lane < head) base[r.a + lane] = stage[r.shift + lane];
  for (int64_t j = lane; j < r.nvec; j += kWave)
    __builtin_nontemporal_store(*reinterpret_cast<const zs_f4*>(stage + r.shift + head + 4 * j),
                                reinterpret_cast<zs_f4*>(base + r.a4 + 4 * j));
  const int64_t t0 = r.a4 + 4 * r.nvec;
  if (lane < r.b - t0) base[t0 + lane] = stage[r.shift + (t0 - r.a) + lane];
  wave_lds_barrier();
}

// The SVD and the stress up to the arena below: products are fused with sums
// within an expression (decided once, here), not across statements by each
// kernel's own schedule, so that instances agree bit by bit.
#pragma clang fp contract(on)

// ---------------------------------------------------------------------------
// 3x3 SVD: McAdams et al. 2011 ("Computing the SVD of 3x3 matrices with
// minimal branching and elementary floating point operations"), the method
// zpc uses (math/matrix/SVD.hpp). Four sweeps of approximate Jacobi
// conjugations on A^T A accumulate V as a quaternion; B = A V is column-sorted
// by norm (V kept a rotation by sign flips) and Givens QR gives U and the
// singular values (sigma_3 carries the sign of det A). Matrices are row-major
// a[r][c] here.
// ---------------------------------------------------------------------------
struct Svd3 {
  static constexpr float kFourGammaSq = 5.8284273147583007813f;  // 4 (3 + 2 sqrt 2) in float
  static constexpr float kSinPi8 = 0.3826834261417388916f;       // sin(pi/8) rounded to float
  static constexpr float kCosPi8 = 0.9238795042037963867f;       // cos(pi/8) rounded to float
  static constexpr float kTiny = 1.e-20f;
  static constexpr float kSmall = 1.e-12f;

  // hardware reciprocal square root (v_rsq_f32, about 1 ulp): zpc's SVD calls
  // zs::rsqrt (math/matrix/SVD.hpp:113), which is ::rsqrtf on its CUDA backend
  // and 1/sqrtf on the host (ZpcMathUtils.hpp:805-846)
  __device__ static __forceinline__ float rsq(float v) { return __builtin_amdgcn_rsqf(v); }

  // approximate Jacobi conjugation for pivot (P, Q), third index R (quaternion axis)
  template <int P, int Q, int R>
  __device__ static __forceinline__ void conjugate(float (&s)[3][3], float& qs, float (&qv)[3]) {
    float sh = s[Q][P] * 0.5f;
    float t5 = s[P][P] - s[Q][Q];
    const bool big = sh * sh >= kTiny;
    sh = big ? sh : 0.0f;
    float ch = big ? t5 : 1.0f;
    float t1 = sh * sh;
    float t2 = ch * ch;
    const float w = rsq(t1 + t2);
    sh = w * sh;
    ch = w * ch;
    const bool pi8 = t2 <= kFourGammaSq * t1;
    sh = pi8 ? kSinPi8 : sh;
    ch = pi8 ? kCosPi8 : ch;
    t1 = sh * sh;
    t2 = ch * ch;
    const float c = t2 - t1;
    float sn = ch * sh;
    sn = sn + sn;
    const float sc = t1 + t2;
    s[R][R] = s[R][R] * sc * sc;
    float rp = s[R][P] * sc, rq = s[R][Q] * sc;
    const float a1 = sn * rp, a2 = sn * rq;
    rp = c * rp + a2;
    rq = c * rq - a1;
    const float ss = sn * sn;
    const float cc = c * c;
    const float pp = s[P][P], qq = s[Q][Q], qp = s[Q][P];
    const float cs = c * sn;
    const float two_qp_cs = (qp + qp) * cs;
    s[P][P] = pp * cc + qq * ss + two_qp_cs;
    s[Q][Q] = qq * cc + pp * ss - two_qp_cs;
    s[Q][P] = qp * (cc - ss) - t5 * cs;
    s[P][Q] = s[Q][P];
    s[R][P] = rp;
    s[P][R] = rp;
    s[R][Q] = rq;
    s[Q][R] = rq;
    constexpr int A = R, B = (R + 1) % 3, Cc = (R + 2) % 3;
    const float u1 = sh * qv[B], u2 = sh * qv[Cc], u3 = sh * qv[A], shs = sh * qs;
    qs = ch * qs - u3;
    const float na = ch * qv[A] + shs;
    const float nb = ch * qv[B] + u2;
    const float nc = ch * qv[Cc] - u1;
    qv[A] = na;
    qv[B] = nb;
    qv[Cc] = nc;
  }

  template <int I, int J, int NEG>
  __device__ static __forceinline__ void sort_step(float (&b)[3][3], float (&v)[3][3], float (&n)[3]) {
    const bool sw = n[I] < n[J];
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      const float bi = b[r][I], bj = b[r][J], vi = v[r][I], vj = v[r][J];
      b[r][I] = sw ? bj : bi;
      b[r][J] = sw ? bi : bj;
      v[r][I] = sw ? vj : vi;
      v[r][J] = sw ? vi : vj;
    }
    const float ni = n[I], nj = n[J];
    n[I] = sw ? nj : ni;
    n[J] = sw ? ni : nj;
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      b[r][NEG] = sw ? -b[r][NEG] : b[r][NEG];
      v[r][NEG] = sw ? -v[r][NEG] : v[r][NEG];
    }
  }

  // one Newton step on rsqrt: r (1.5 - 0.5 x r^2), written as the method does
  __device__ static __forceinline__ float newton_rsq(float x) {
    const float r = rsq(x);
    const float h = r * 0.5f;
    return (r + h) - x * (r * (r * h));
  }

  template <int P, int Q>
  __device__ static __forceinline__ void givens_qr(float (&b)[3][3], float (&u)[3][3]) {
    const float a_qp = b[Q][P], a_pp = b[P][P];
    float sh = (a_qp * a_qp >= kSmall) ? a_qp : 0.0f;
    float ch = fmaxf(fmaxf(-a_pp, a_pp), kSmall);
    const bool nonneg = a_pp >= 0.f;
    const float rr = ch * ch + sh * sh;
    ch = ch + newton_rsq(rr) * rr;
    const float tch = nonneg ? ch : sh;
    const float tsh = nonneg ? sh : ch;
    const float w = newton_rsq(tch * tch + tsh * tsh);
    ch = tch * w;
    sh = tsh * w;
    const float c = ch * ch - sh * sh;
    float sn = sh * ch;
    sn = sn + sn;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const float bp = b[P][j], bq = b[Q][j];
      b[P][j] = c * bp + sn * bq;
      b[Q][j] = c * bq - sn * bp;
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const float up = u[i][P], uq = u[i][Q];
      u[i][P] = c * up + sn * uq;
      u[i][Q] = c * uq - sn * up;
    }
  }

  __device__ static __forceinline__ void svd(const float (&a)[3][3], float (&U)[3][3], float (&S)[3],
                                             float (&V)[3][3]) {
    float s[3][3];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = 0; j <= i; ++j) {
        const float t = a[0][i] * a[0][j] + a[1][i] * a[1][j] + a[2][i] * a[2][j];
        s[i][j] = t;
        s[j][i] = t;
      }
    float qs = 1.f, qv[3] = {0.f, 0.f, 0.f};
#pragma unroll
    for (int sweep = 0; sweep < 4; ++sweep) {
      conjugate<0, 1, 2>(s, qs, qv);
      conjugate<1, 2, 0>(s, qs, qv);
      conjugate<2, 0, 1>(s, qs, qv);
    }
    const float qn = newton_rsq(qs * qs + qv[0] * qv[0] + qv[1] * qv[1] + qv[2] * qv[2]);
    qs *= qn;
    qv[0] *= qn;
    qv[1] *= qn;
    qv[2] *= qn;
    const float xx = qv[0] * qv[0], yy = qv[1] * qv[1], zz = qv[2] * qv[2], ww = qs * qs;
    float v[3][3];
    v[0][0] = ww + xx - yy - zz;
    v[1][1] = ww - xx + yy - zz;
    v[2][2] = ww - xx - yy + zz;
    const float tx = qv[0] + qv[0], ty = qv[1] + qv[1], tz = qv[2] + qv[2];
    const float sx = qs * tx, sy = qs * ty, sz = qs * tz;
    const float xy = qv[1] * tx, yz = qv[2] * ty, xz = qv[0] * tz;
    v[0][1] = xy - sz;
    v[1][0] = xy + sz;
    v[1][2] = yz - sx;
    v[2][1] = yz + sx;
    v[2][0] = xz - sy;
    v[0][2] = xz + sy;
    float b[3][3];
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int c = 0; c < 3; ++c) b[r][c] = a[r][0] * v[0][c] + a[r][1] * v[1][c] + a[r][2] * v[2][c];
    float n[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) n[c] = b[0][c] * b[0][c] + b[1][c] * b[1][c] + b[2][c] * b[2][c];
    sort_step<0, 1, 1>(b, v, n);
    sort_step<0, 2, 0>(b, v, n);
    sort_step<1, 2, 2>(b, v, n);
    float u[3][3] = {{1.f, 0.f, 0.f}, {0.f, 1.f, 0.f}, {0.f, 0.f, 1.f}};
    givens_qr<0, 1>(b, u);
    givens_qr<0, 2>(b, u);
    givens_qr<1, 2>(b, u);
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        U[i][j] = u[i][j];
        V[i][j] = v[i][j];
      }
    S[0] = b[0][0];
    S[1] = b[1][1];
    S[2] = b[2][2];
  }
};

// FP64 SVD for nearly repeated singular values: cyclic Jacobi with exact
// rotations on A^T A until the off-diagonal mass is below 1e-34 of the
// diagonal, then the same column sort and Givens QR conventions.
__device__ inline void svd3_fp64(const float (&af)[3][3], float (&U)[3][3], float (&S)[3],
                                 float (&V)[3][3]) {
  double a[3][3];
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) a[i][j] = (double)af[i][j];
  double s[3][3];
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) s[i][j] = a[0][i] * a[0][j] + a[1][i] * a[1][j] + a[2][i] * a[2][j];
  double v[3][3] = {{1, 0, 0}, {0, 1, 0}, {0, 0, 1}};
  for (int sweep = 0; sweep < 12; ++sweep) {
    const double off = s[0][1] * s[0][1] + s[0][2] * s[0][2] + s[1][2] * s[1][2];
    const double dia = s[0][0] * s[0][0] + s[1][1] * s[1][1] + s[2][2] * s[2][2];
    if (off <= 1e-34 * dia) break;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const int p = (k == 2) ? 0 : k, q = (k == 0) ? 1 : 2;
      const double spq = s[p][q];
      if (spq == 0.0) continue;
      const double theta = (s[q][q] - s[p][p]) / (2.0 * spq);
      const double t = (theta >= 0 ? 1.0 : -1.0) / (fabs(theta) + sqrt(theta * theta + 1.0));
      const double c = 1.0 / sqrt(t * t + 1.0), sn = t * c;
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        const double srp = s[r][p], srq = s[r][q];
        s[r][p] = c * srp - sn * srq;
        s[r][q] = sn * srp + c * srq;
      }
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        const double spr = s[p][r], sqr = s[q][r];
        s[p][r] = c * spr - sn * sqr;
        s[q][r] = sn * spr + c * sqr;
      }
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        const double vp = v[r][p], vq = v[r][q];
        v[r][p] = c * vp - sn * vq;
        v[r][q] = sn * vp + c * vq;
      }
    }
  }
  double b[3][3];
#pragma unroll
  for (int r = 0; r < 3; ++r)
#pragma unroll
    for (int c = 0; c < 3; ++c) b[r][c] = a[r][0] * v[0][c] + a[r][1] * v[1][c] + a[r][2] * v[2][c];
  double n[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) n[c] = b[0][c] * b[0][c] + b[1][c] * b[1][c] + b[2][c] * b[2][c];
  auto sort_step = [&](int i, int j, int neg) {
    if (n[i] < n[j]) {
      for (int r = 0; r < 3; ++r) {
        double t = b[r][i]; b[r][i] = b[r][j]; b[r][j] = t;
        t = v[r][i]; v[r][i] = v[r][j]; v[r][j] = t;
      }
      double t = n[i]; n[i] = n[j]; n[j] = t;
      for (int r = 0; r < 3; ++r) { b[r][neg] = -b[r][neg]; v[r][neg] = -v[r][neg]; }
    }
  };
  sort_step(0, 1, 1);
  sort_step(0, 2, 0);
  sort_step(1, 2, 2);
  double u[3][3] = {{1, 0, 0}, {0, 1, 0}, {0, 0, 1}};
  auto givens = [&](int p, int q) {
    const double x = b[p][p], y = b[q][p];
    const double r = sqrt(x * x + y * y);
    double c = 1.0, sn = 0.0;  // c = x / r, s = y / r leaves the pivot at r >= 0
    if (r != 0.0) {
      c = x / r;
      sn = y / r;
    }
    for (int j = 0; j < 3; ++j) {
      const double bp = b[p][j], bq = b[q][j];
      b[p][j] = c * bp + sn * bq;
      b[q][j] = -sn * bp + c * bq;
    }
    for (int i = 0; i < 3; ++i) {
      const double up = u[i][p], uq = u[i][q];
      u[i][p] = c * up + sn * uq;
      u[i][q] = -sn * up + c * uq;
    }
  };
  givens(0, 1);
  givens(0, 2);
  givens(1, 2);
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      U[i][j] = (float)u[i][j];
      V[i][j] = (float)v[i][j];
    }
  S[0] = (float)b[0][0];
  S[1] = (float)b[1][1];
  S[2] = (float)b[2][2];
}

// SVD of a column-major F (F[i + 3j] = F_ij) with the FP64 path for nearly
// repeated singular values: when min_i |sigma_i - sigma_{i+1}| < gap * |sigma_1|
// (gap > 0) the FP32 result is replaced by the FP64 one.
__device__ __forceinline__ void svd_colmajor(const float* F, float (&U)[3][3], float (&S)[3],
                                             float (&V)[3][3], float fp64_gap, bool& used_fp64) {
  float a[3][3];
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) a[i][j] = F[i + 3 * j];
  Svd3::svd(a, U, S, V);
  used_fp64 = false;
  if (fp64_gap > 0.f) {
    const float g = fminf(fabsf(S[0] - S[1]), fabsf(S[1] - S[2]));
    if (g < fp64_gap * fabsf(S[0])) {
      svd3_fp64(a, U, S, V);
      used_fp64 = true;
    }
  }
}

// ---------------------------------------------------------------------------
// constitutive models (physics/ConstitutiveModel_Vol_dP.hpp:10-46, 241-325)
// ---------------------------------------------------------------------------
struct Model {
  int32_t kind;  // 0 fixed-corotated, 1 Drucker-Prager sand
  float volume, mu, lambda, cohesion, beta, yield_surface;
  int32_t volume_correction;
  float fp64_gap;
};

// Both models need only functions of b = F F^T, isotropic in it: with the
// Hencky strain E = 1/2 log b = U diag(log sigma) U^T sand's Kirchhoff stress is
// linear in E and I, and fixed-corotated's is 2 mu (b - sqrt b) + lambda (J - 1)
// J I (det F > 0; V never enters). Near b = I both come without a
// decomposition from Z = (b - I)(b + I)^-1, b = (I + Z)(I - Z)^-1:
//   1/2 log b    = atanh Z = sum z^(2k+1) / (2k+1)
//   sqrt b - I   = (I + Z)(I - Z^2)^(-1/2) - I = z + z^2/2 + z^3/2 + ...
// as polynomials of degree 13 reduced with Cayley-Hamilton (Z^3 = i1 Z^2 - i2 Z
// + i3 I), three multiply-adds per degree. b - I = G + G^T + G G^T, G = F - I,
// has no cancellation, so small strains keep their relative accuracy (the SVD
// forms log sigma from sigma ~ 1: an absolute 1e-7). About 170 operations
// against 1,240 with the four-sweep SVD; the range is ||Z||_F <= 0.3 (sigma
// in [0.734, 1.363]), where the first omitted terms are 1e-8.
struct NearB {
  float A[6], Z[6], Y[6];  // b - I, Z, Z^2 as (xx, yy, zz, xy, xz, yz)
  float i1, i2, i3;        // invariants of Z
};
constexpr float kNearZ2 = 0.09f;  // largest ||Z||_F^2 of the series
// No ||A||_F^2 above this is near: A's eigenvalues are a = 2 z / (1 - z), so |z| <=
// 0.3 gives |a| <= |z| 2 / 0.7 and the sum of a^2 at most 0.09 (2 / 0.7)^2 = 0.7347.
// It is looked at before det(b + I), which overflows its reciprocal for stretches
// beyond 2e6 (Z would come out 0), and ends a far wave's attempt early.
constexpr float kNearA2 = 0.74f;

__device__ __forceinline__ void sym_mul(const float (&a)[6], const float (&b)[6], float (&c)[6]) {
  // product of two symmetric matrices that commute (so it is symmetric)
  c[0] = a[0] * b[0] + a[3] * b[3] + a[4] * b[4];
  c[1] = a[3] * b[3] + a[1] * b[1] + a[5] * b[5];
  c[2] = a[4] * b[4] + a[5] * b[5] + a[2] * b[2];
  c[3] = a[0] * b[3] + a[3] * b[1] + a[4] * b[5];
  c[4] = a[0] * b[4] + a[3] * b[5] + a[4] * b[2];
  c[5] = a[3] * b[4] + a[1] * b[5] + a[5] * b[2];
}

// F column-major; false (also for NaN) when the series does not apply
__device__ __forceinline__ bool near_identity(const float* F, NearB& n) {
  float G[9];
#pragma unroll
  for (int k = 0; k < 9; ++k) G[k] = (k & 3) == 0 ? F[k] - 1.f : F[k];
  constexpr int I[6] = {0, 1, 2, 0, 0, 1}, J[6] = {0, 1, 2, 1, 2, 2};
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    const int i = I[k], j = J[k];
    n.A[k] = (G[i + 3 * j] + G[j + 3 * i]) + (G[i] * G[j] + G[i + 3] * G[j + 3] + G[i + 6] * G[j + 6]);
  }
  const float (&A)[6] = n.A;
  if (!(A[0] * A[0] + A[1] * A[1] + A[2] * A[2] + 2.f * (A[3] * A[3] + A[4] * A[4] + A[5] * A[5]) <= kNearA2))
    return false;
  // (b + I)^-1 from the adjugate; b + I >= I, so the determinant is >= 1
  const float m0 = 2.f + A[0], m1 = 2.f + A[1], m2 = 2.f + A[2];
  float adj[6];
  adj[0] = m1 * m2 - A[5] * A[5];
  adj[1] = m0 * m2 - A[4] * A[4];
  adj[2] = m0 * m1 - A[3] * A[3];
  adj[3] = A[4] * A[5] - A[3] * m2;
  adj[4] = A[3] * A[5] - A[4] * m1;
  adj[5] = A[3] * A[4] - m0 * A[5];
  const float det = m0 * adj[0] + A[3] * adj[3] + A[4] * adj[4];
  float r = __builtin_amdgcn_rcpf(det);
  r = r * (2.f - det * r);
  sym_mul(A, adj, n.Z);
#pragma unroll
  for (int k = 0; k < 6; ++k) n.Z[k] *= r;
  sym_mul(n.Z, n.Z, n.Y);
  const float (&Z)[6] = n.Z;
  const float t2 = n.Y[0] + n.Y[1] + n.Y[2];
  n.i1 = Z[0] + Z[1] + Z[2];
  n.i2 = 0.5f * (n.i1 * n.i1 - t2);
  n.i3 = Z[0] * (Z[1] * Z[2] - Z[5] * Z[5]) - Z[3] * (Z[3] * Z[2] - Z[5] * Z[4]) + Z[4] * (Z[3] * Z[5] - Z[1] * Z[4]);
  return t2 <= kNearZ2;
}

// sum_k p[k] Z^k = a I + b Z + c Z^2 (Horner with Cayley-Hamilton)
template <int N>
__device__ __forceinline__ void near_poly(const NearB& n, const float (&p)[N], float& a, float& b, float& c) {
  a = b = c = 0.f;
#pragma unroll
  for (int k = N - 1; k >= 0; --k) {
    const float na = c * n.i3 + p[k], nb = a - c * n.i2, nc = b + c * n.i1;
    a = na;
    b = nb;
    c = nc;
  }
}

// P F^T = U diag(tau) U^T of an isotropic model, tau the principal Kirchhoff
// stresses (times the volume): with F = U diag(s) V^T and P = U diag(Ph) V^T,
// tau_i = Ph_i s_i and V^T V = I drops out. Symmetric: 6 entries, and V is not
// needed past A V. Against 64 bits it is closer than P F^T multiplied out,
// which keeps the four-sweep SVD's residual (strains of 0.3 to 1: 2.4e-5, 2.1e-5
// and 2.3e-5 of the 2-norm against 2.5e-5, 3.9e-5 and 5.7e-5).
__device__ __forceinline__ void kirchhoff(const float (&U)[3][3], const float (&tau)[3], float* PF) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = i; j < 3; ++j) {
      const float e = U[i][0] * tau[0] * U[j][0] + U[i][1] * tau[1] * U[j][1] + U[i][2] * tau[2] * U[j][2];
      PF[i + 3 * j] = e;
      PF[j + 3 * i] = e;
    }
}

// Fixed-corotated near the identity; false: out of the series' range (nothing written).
__device__ __forceinline__ bool series_fixedcorotated(const Model& m, const float* F, float* PF) {
  NearB nb;
  if (!near_identity(F, nb)) return false;
  // J - 1 = tr G + (second invariant of G) + det G, G = F - I; a reflection
  // (J < 0) has b near I too and takes the SVD
  const float g0 = F[0] - 1.f, g4 = F[4] - 1.f, g8 = F[8] - 1.f;
  const float q0 = g4 * g8 - F[5] * F[7];
  const float Jm1 = (g0 + g4 + g8) + (g0 * (g4 + g8) + q0 - F[3] * F[1] - F[6] * F[2]) +
                    (g0 * q0 - F[3] * (F[1] * g8 - F[2] * F[7]) + F[6] * (F[1] * F[5] - F[2] * g4));
  if (!(Jm1 > -1.f)) return false;
  constexpr float p[14] = {0.f,       1.f,        0.5f,       0.5f,        0.375f,      0.375f,        0.3125f,
                           0.3125f,   0.2734375f, 0.2734375f, 0.24609375f, 0.24609375f, 0.2255859375f, 0.2255859375f};
  float a, b, c;
  near_poly(nb, p, a, b, c);
  const float smu = 2.f * m.mu * m.volume;
  const float iso = m.lambda * Jm1 * (Jm1 + 1.f) * m.volume;
  float T[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    // b - sqrt b = A - X
    const float X = b * nb.Z[k] + c * nb.Y[k] + (k < 3 ? a : 0.f);
    T[k] = smu * (nb.A[k] - X) + (k < 3 ? iso : 0.f);
  }
  PF[0] = T[0];
  PF[4] = T[1];
  PF[8] = T[2];
  PF[1] = PF[3] = T[3];
  PF[2] = PF[6] = T[4];
  PF[5] = PF[7] = T[5];
  return true;
}

// Fixed-corotated from the SVD: Ph_i = 2 mu (s_i - 1) + lambda (J - 1) prod_{j!=i} s_j.
__device__ __forceinline__ void svd_fixedcorotated(const Model& m, const float (&U)[3][3], const float (&S)[3],
                                                   float* PF) {
  const float J = S[0] * S[1] * S[2];
  const float smu = 2.f * m.mu;
  const float slam = m.lambda * (J - 1.f);
  const float tau[3] = {(smu * (S[0] - 1.f) + slam * (S[1] * S[2])) * S[0] * m.volume,
                        (smu * (S[1] - 1.f) + slam * (S[0] * S[2])) * S[1] * m.volume,
                        (smu * (S[2] - 1.f) + slam * (S[0] * S[1])) * S[2] * m.volume};
  kirchhoff(U, tau, PF);
}

// Sand near the identity: the return mapping of stress_sand on the tensor E.
// Returns its case, or -1 out of the series' range (nothing written).
__device__ __forceinline__ int series_sand(const Model& m, const float* F, float& logJp, float* PF) {
  NearB nb;
  if (m.mu == 0.f || !near_identity(F, nb)) return -1;
  // the return mapping on the tensor E: eps_i are the eigenvalues of E -
  // cohesion I, and every case leaves H (the projected log sigma_i) linear in
  // E and I
  constexpr float p[14] = {0.f,       1.f, 0.f,       1.f / 3.f,  0.f, 1.f / 5.f,  0.f,
                           1.f / 7.f, 0.f, 1.f / 9.f, 0.f,        1.f / 11.f, 0.f, 1.f / 13.f};
  float a, b, c;
  near_poly(nb, p, a, b, c);
  float E[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) E[k] = b * nb.Z[k] + c * nb.Y[k] + (k < 3 ? a : 0.f);
  const float trE = E[0] + E[1] + E[2];
  const float sum_eps = trE - 3.f * m.cohesion;
  const float tr = sum_eps + logJp;
  const float shift = m.cohesion + tr * (1.f / 3.f);  // eps - tr/3: the deviator zpc projects (logJp included)
  const float d0 = E[0] - shift, d1 = E[1] - shift, d2 = E[2] - shift;
  // its norm and inverse norm from one reciprocal root and a Newton step (0 and
  // a huge number at a zero deviator, which is never projected)
  const float eh2 = d0 * d0 + d1 * d1 + d2 * d2 + 2.f * (E[3] * E[3] + E[4] * E[4] + E[5] * E[5]);
  float inv = __builtin_amdgcn_rsqf(fmaxf(eh2, 1e-37f));
  inv = inv * (1.5f - 0.5f * eh2 * inv * inv);
  const float ehn = eh2 * inv;
  const float smu = 2.f * m.mu;
  int which = 1;
  float keep = 1.f, add = 0.f;  // H = keep E + add I
  if (tr >= 0.f) {
    which = 2;
    keep = 0.f;
    add = m.cohesion;
    if (m.volume_correction) logJp = m.beta * sum_eps + logJp;
  } else {
    logJp = 0.f;
    const float kt = (3.f * m.lambda + smu) / smu * tr * m.yield_surface;
    const float dg = ehn + kt;
    if (!(dg <= 0.f)) {
      which = 3;  // E - dg / ehn (E - shift I)
      keep = -kt * inv;
      add = dg * inv * shift;
    }
  }
  const float iso = (m.lambda * (keep * trE + 3.f * add) + smu * add) * m.volume;
  const float dev = smu * keep * m.volume;
  PF[0] = dev * E[0] + iso;
  PF[4] = dev * E[1] + iso;
  PF[8] = dev * E[2] + iso;
  PF[1] = PF[3] = dev * E[3];
  PF[2] = PF[6] = dev * E[4];
  PF[5] = PF[7] = dev * E[5];
  return which;
}

// Drucker-Prager with volume correction, from the SVD; logJp is updated. tau_i =
// Ph_i ns_i = 2 mu ln ns_i + lambda sum_j ln ns_j of the projected F = U diag(ns)
// V^T: ln ns_i = H_i is the exponent the projection chose (no exp / log round
// trip, no division). Returns the case: 1 inside the cone, 2 cone tip, 3
// projected to the cone surface, 0 otherwise (mu = 0 under compression: zpc
// leaves ns at 0 there, and log 0 over 0 makes every entry NaN).
__device__ __forceinline__ int svd_sand(const Model& m, const float (&U)[3][3], const float (&S)[3], float& logJp,
                                        float* PF) {
  const float smu = 2.f * m.mu;
  float eps[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const float a = fmaxf(fabsf(S[i]), 1e-4f);
    eps[i] = logf(a) - m.cohesion;
  }
  const float sum_eps = eps[0] + eps[1] + eps[2];
  const float tr = sum_eps + logJp;
  const float third = tr / 3.f;
  const float eh[3] = {eps[0] - third, eps[1] - third, eps[2] - third};
  const float ehn = sqrtf(eh[0] * eh[0] + eh[1] * eh[1] + eh[2] * eh[2]);
  const float nan = __builtin_nanf("");
  float H[3] = {nan, nan, nan};
  int which = 0;
  if (tr >= 0.f) {
    H[0] = H[1] = H[2] = m.cohesion;
    if (m.volume_correction) logJp = m.beta * sum_eps + logJp;
    which = 2;
  } else if (m.mu != 0.f) {
    logJp = 0.f;
    const float dg = ehn + (3.f * m.lambda + smu) / smu * tr * m.yield_surface;
    if (dg <= 0.f) {
#pragma unroll
      for (int i = 0; i < 3; ++i) H[i] = eps[i] + m.cohesion;
      which = 1;
    } else {
      const float r = dg / ehn;
#pragma unroll
      for (int i = 0; i < 3; ++i) H[i] = eps[i] - r * eh[i] + m.cohesion;
      which = 3;
    }
  }
  const float trl = H[0] + H[1] + H[2];
  const float tau[3] = {(smu * H[0] + m.lambda * trl) * m.volume, (smu * H[1] + m.lambda * trl) * m.volume,
                        (smu * H[2] + m.lambda * trl) * m.volume};
  kirchhoff(U, tau, PF);
  return which;
}

// vol P F^T of a model with its FP64 SVD off (fp64_gap = 0): the series where
// it applies, else the float SVD; sand updates logJp
__device__ __forceinline__ void stress_plain(const Model& m, const float* F, float& logJp, float* PF) {
  if (m.kind == 0) {
    if (series_fixedcorotated(m, F, PF)) return;
  } else {
    if (series_sand(m, F, logJp, PF) >= 0) return;
  }
  float U[3][3], S[3], V[3][3];
  bool fp64;
  svd_colmajor(F, U, S, V, 0.f, fp64);
  if (m.kind == 0)
    svd_fixedcorotated(m, U, S, PF);
  else
    (void)svd_sand(m, U, S, logJp, PF);
}

// The same of a model with the FP64 SVD on (fp64_gap > 0): a particle with nearly
// repeated singular values takes that (and sets fp64), every other one what it
// gets with it off. One float SVD serves the look at the singular values and
// the particles out of the series' range.
__device__ __forceinline__ void stress_gap(const Model& m, const float* F, float& logJp, float* PF, bool& fp64) {
  float U[3][3], S[3], V[3][3];
  svd_colmajor(F, U, S, V, m.fp64_gap, fp64);
  if (m.kind == 0) {
    if (!fp64 && series_fixedcorotated(m, F, PF)) return;
    svd_fixedcorotated(m, U, S, PF);
  } else {
    if (!fp64 && series_sand(m, F, logJp, PF) >= 0) return;
    (void)svd_sand(m, U, S, logJp, PF);
  }
}

__device__ __forceinline__ void stress_any(const Model& m, const float* F, float& logJp, float* PF, bool& fp64) {
  fp64 = false;
  if (m.fp64_gap > 0.f)
    stress_gap(m, F, logJp, PF, fp64);
  else
    stress_plain(m, F, logJp, PF);
}

#pragma clang fp contract(fast)

// ---------------------------------------------------------------------------
// quadratic B-spline arena (simulation/Utils.hpp:51-70): X = x / dx,
// base = floor(X - 0.5), local = X - base, weights per axis, local *= dx.
// ---------------------------------------------------------------------------
struct Arena {
  int32_t base[3];
  float lp[3];   // local position * dx
  float w[3][3]; // w[axis][node]
};

__device__ __forceinline__ void make_arena(float x0, float x1, float x2, float dx, Arena& ar) {
#pragma clang fp contract(off)
  const float xs[3] = {x0, x1, x2};
  const bool pow2 = is_pow2(dx);
  const float dx_inv = 1.f / dx;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const float X = pow2 ? xs[d] * dx_inv : xs[d] / dx;
    const int32_t b = (int32_t)floorf(X - 0.5f);
    const float l = X - (float)b;
    const float d0 = l - (float)(int32_t)floorf(l - 0.5f);
    ar.base[d] = b;
    ar.w[d][0] = 0.5f * (1.5f - d0) * (1.5f - d0);
    const float d1 = d0 - 1.0f;
    ar.w[d][1] = 0.75f - d1 * d1;
    const float zz = 0.5f + d1;
    ar.w[d][2] = 0.5f * zz * zz;
    ar.lp[d] = l * dx;
  }
}

}  // namespace zsmpm
