// Softened direct-N gravity (sph_grav_kernel.cu:14-195).
//
// Layout: one lane per i-particle, 256 i per block.  The block stages j
// records in LDS tiles of 512 with coalesced loads; all lanes of a wave then
// read the same j from LDS (a broadcast), so the loop body is VALU work plus
// one LDS read per j per wave.  (Reading j through scalar loads instead was
// measured ~4% slower at N = 2^20: the scalar cache misses once the j array
// outgrows L2.)  j runs in ascending order over all records, the reference's
// summation order.  The mixed and FP64 forms have no such order to keep and take
// each pair of particles once for both where that pays (k_gravity_mixed_pairs,
// pairs64.h).
//
// Variants (template parameters):
//   SOFT  0: M4 spline at the SPH range, half from each side (reference)
//         1: Plummer eps
//   ACC   0: per-pair double-float (dreal) accumulation (reference, dreal.h)
//         1: blocked compensation -- a plain FP32 partial over each tile of
//            kTile j, folded into a two-sum (hi,lo) total (mixed form)
//         2: plain accumulation in T (FP64 form)
//   EXACT 1: 1/sqrt correctly rounded (bit-exact with the CPU restatement);
//         0: hardware reciprocal square root (the reference uses rsqrtf)
//   HILO  positions carry low words (mixed form): r_ij = (hi_i-hi_j)+(lo_i-lo_j)
#include <algorithm>
#include <type_traits>

#include "kernels.h"
#include "pairs64.h"
#include "sph_math.h"

namespace cudasph {

struct DR {
  float hi, lo;
};
// two-sum subtraction with renormalisation (Knuth; the reference's dsub,
// dreal.h:43-52)
__device__ __forceinline__ void dr_sub(DR& x, float y) {
  const float t1 = x.hi - y;
  const float e = t1 - x.hi;
  const float t2 = ((-y - e) + (x.hi - (t1 - e))) + x.lo;
  const float s = t1 + t2;
  x.lo = t2 - (s - t1);
  x.hi = s;
}
__device__ __forceinline__ void dr_add(DR& x, float y) { dr_sub(x, -y); }

// A dreal sum with its last step's low word still to be formed: hi, and
// lo = t2 - (hi - t1).  sub is dr_sub.  The fast ones are dr_sub where
// |hi| >= |y|: the rounding error of hi - y is then exact in two operations
// (Dekker's fast two-sum) instead of five, so they return dr_sub's bits with
// 7 operations instead of 10.
struct Chain {
  float hi = 0.f, t1 = 0.f, t2 = 0.f;
  __device__ __forceinline__ void sub(float y) {
    DR v{hi, t2 - (hi - t1)};
    const float d1 = v.hi - y;
    const float e = d1 - v.hi;
    const float d2 = ((-y - e) + (v.hi - (d1 - e))) + v.lo;
    hi = d1 + d2;
    t1 = d1;
    t2 = d2;
  }
  __device__ __forceinline__ void sub_fast(float y) {
    const float lo = t2 - (hi - t1), d1 = hi - y;
    t2 = ((hi - d1) - y) + lo;
    hi = d1 + t2;
    t1 = d1;
  }
  // ... for a wavefront that has only this chain to issue: a step depends on
  // the one before through 5 operations, and the two that form the previous
  // low word go between them (left to itself the compiler puts all 7 in a row)
  __device__ __forceinline__ void sub_fast_alone(float y) {
    float n1, q, d;
    asm("v_sub_f32 %[n1], %[hi], %[y]\n\t"     // n1 = hi - y
        "v_sub_f32 %[q], %[hi], %[t1]\n\t"
        "v_sub_f32 %[d], %[hi], %[n1]\n\t"
        "v_sub_f32 %[q], %[t2], %[q]\n\t"      // q = the low word
        "v_sub_f32 %[d], %[d], %[y]\n\t"       // d = the rounding error
        "v_add_f32 %[t2], %[d], %[q]\n\t"
        "v_add_f32 %[hi], %[n1], %[t2]"
        : [n1] "=&v"(n1), [q] "=&v"(q), [d] "=&v"(d), [hi] "+&v"(hi), [t2] "+&v"(t2)
        : [t1] "v"(t1), [y] "v"(y));
    t1 = n1;
  }
};
// the four sums of one particle
struct Chains4 {
  Chain a0, a1, a2, a3;
};

template <class T, int ACC>
struct GAcc;
template <>
struct GAcc<float, 1> {                      // blocked compensation
  DR v{0.f, 0.f};
  float part = 0.f;
  __device__ __forceinline__ void sub(float y) { part -= y; }
  __device__ __forceinline__ void fsub(float a, float b) { part = __builtin_fmaf(-a, b, part); }
  // fold the block's partial into (hi, lo): Knuth's two-sum of hi and the
  // partial, its exact error added to lo (lo stays a small FP32 sum of the
  // rounding errors; no renormalisation is needed until get())
  __device__ __forceinline__ void tile_end() {
    const float s = v.hi + part;
    const float bp = s - v.hi;
    v.lo += (v.hi - (s - bp)) + (part - bp);
    v.hi = s;
    part = 0.f;
  }
  __device__ __forceinline__ float get() const { return v.hi + v.lo; }
};
template <>
struct GAcc<double, 2> {
  double v = 0.0;
  __device__ __forceinline__ void sub(double y) { v -= y; }
  __device__ __forceinline__ void tile_end() {}
  __device__ __forceinline__ double get() const { return v; }
};

// v_rsq_f32 between scalar instructions.  A wavefront whose next vector
// operation follows a transcendental one directly holds up the SIMD's vector
// issue for the other wavefronts too: 11 multiplies and a v_rsq_f32 take 54
// cycles of a SIMD with 4 or 8 wavefronts, 40 with a scalar instruction after
// the v_rsq_f32 (the wait state its use needs anyway) and 33 with one on
// either side, the sum of their issue times.  Raising the issue priority for
// the v_rsq_f32 is the scalar instruction that helped the gravity kernels
// most: mixed gravity at 2^20 particles 284 -> 275 ms in the same process (in
// cycles 7 %; the clock falls from 2.24 to 2.14 GHz as the SIMDs fill), s_nop
// on both sides 290-292 against 293.  Not for k_gravity_lane's pipelined loop,
// whose order it breaks (100 003 particles 11.4 -> 13.2 ms), nor where the
// caller has raised its own priority (it returns to 0).
__device__ __forceinline__ float rsq_spaced(float x) {
  float r;
  asm("s_setprio 1\n\tv_rsq_f32 %0, %1\n\ts_setprio 0" : "=v"(r) : "v"(x));
  return r;
}

template <bool EXACT>
__device__ __forceinline__ float inv_sqrt(float x) {
  if constexpr (EXACT) return 1.0f / __builtin_sqrtf(x);
  else return __builtin_amdgcn_rsqf(x);
}
template <bool EXACT>
// FP64: hardware reciprocal square root refined by two Newton steps (each
// squares the relative error; the result is within a few ulp of 1/sqrt(x)),
// in place of the long correctly rounded sqrt + divide sequences
__device__ __forceinline__ double inv_sqrt(double x) {
  double y = __builtin_amdgcn_rsq(x);
  y = y * (1.5 - 0.5 * x * y * y);
  return y * (1.5 - 0.5 * x * y * y);
}

// sum C of an accumulator set
template <int C, class T, int ACC>
__device__ __forceinline__ GAcc<T, ACC>& acc(GAcc<T, ACC> (&a)[4]) { return a[C]; }
template <int C, class S>
__device__ __forceinline__ auto& acc(S& a) {
  if constexpr (C == 0) return a.a0;
  else if constexpr (C == 1) return a.a1;
  else if constexpr (C == 2) return a.a2;
  else return a.a3;
}

// spline-softened pair (sph_grav_kernel.cu:14-111); pj = (x,y,z,m),
// vi.w / vj.w = range^2
template <class T, bool EXACT, class A>
__device__ __forceinline__ void pair_spline(A&& a, T rx, T ry, T rz, T ri2, T mj, T rj2) {
  const T d2 = rx * rx + ry * ry + rz * rz;
  const T inv = inv_sqrt<EXACT>(d2);
  const T inv3 = inv * inv * inv;
  T s3 = mj * inv3;
  if (d2 >= ri2 && d2 >= rj2) {
    acc<0>(a).sub(rx * s3);
    acc<1>(a).sub(ry * s3);
    acc<2>(a).sub(rz * s3);
    acc<3>(a).sub(mj * inv);
    return;
  }
  s3 = T(0.5f) * s3;
  if (d2 < ri2) {
    const T u2 = d2 / ri2, h = dsqrt(ri2), u = dsqrt(u2), u3 = u2 * u;
    T gacc, gpot;
    if (u < T(0.5)) {
      gacc = T(32.0 / 3.0) + u2 * (T(32) * u - T(38.4));
      gpot = T(-2.8) + u2 * (T(16.0 / 3.0) + u2 * (T(6.4) * u - T(9.6)));
    } else {
      gacc = T(64.0 / 3.0) - T(48) * u + T(38.4) * u2 - T(32.0 / 3.0) * u3 - T(1.0 / 15.0) / u3;
      gpot = T(-3.2) + T(1.0 / 15.0) / u + u2 * (T(32.0 / 3.0) + u * (T(-16) + u * (T(9.6) - T(32.0 / 15.0) * u)));
    }
    gacc = T(0.5 * (double)mj * (double)gacc / (double)(ri2 * h));
    gpot = -gpot;
    acc<0>(a).sub(rx * gacc);
    acc<1>(a).sub(ry * gacc);
    acc<2>(a).sub(rz * gacc);
    acc<3>(a).sub(mj * gpot / h);
  } else {
    acc<0>(a).sub(rx * s3);
    acc<1>(a).sub(ry * s3);
    acc<2>(a).sub(rz * s3);
    acc<3>(a).sub(mj * inv);
  }
  if (d2 < rj2) {
    const T u2 = d2 / rj2, h = dsqrt(rj2), u = dsqrt(u2), u3 = u2 * u;
    T gacc;
    if (u < T(0.5)) gacc = T(32.0 / 3.0) + u2 * (T(32) * u - T(38.4));
    else gacc = T(64.0 / 3.0) - T(48) * u + T(38.4) * u2 - T(32.0 / 3.0) * u3 - T(1.0 / 15.0) / u3;
    gacc = T(0.5 * (double)mj * (double)gacc / (double)(rj2 * h));
    acc<0>(a).sub(rx * gacc);
    acc<1>(a).sub(ry * gacc);
    acc<2>(a).sub(rz * gacc);
  } else {
    acc<0>(a).sub(rx * s3);
    acc<1>(a).sub(ry * s3);
    acc<2>(a).sub(rz * s3);
  }
}

// Plummer pair: a -= m r (r^2+eps^2)^-3/2, phi -= m (r^2+eps^2)^-1/2
template <class T, bool EXACT, class A>
__device__ __forceinline__ void pair_plummer(A&& a, T rx, T ry, T rz, T mj, T eps2) {
  const T d2 = rx * rx + ry * ry + rz * rz + eps2;
  const T inv = inv_sqrt<EXACT>(d2);
  const T inv3 = inv * inv * inv;
  const T s3 = mj * inv3;
  acc<0>(a).sub(rx * s3);
  acc<1>(a).sub(ry * s3);
  acc<2>(a).sub(rz * s3);
  acc<3>(a).sub(mj * inv);
}

constexpr int kGravBlock = 256;
constexpr int kTile = 64;        // j per blocked-compensation partial (mixed form)
constexpr int kJTile = 512;      // j records staged in LDS per block iteration (reference-layout kernels)
// j records per LDS tile of the mixed Plummer kernel: one 64-record sub-tile
// per wavefront.  Its 12 KB of LDS lets 8 blocks share a CU (the kernel's 63
// VGPRs allow 8 waves per SIMD), so the 4096 x 8 blocks at N = 2^20 run in
// exactly 16 rounds; 512-record tiles (24 KB) fit 6 blocks and left the last
// of 21 1/3 rounds a third full (measured 2 % slower)
constexpr int kJTileMixed = kGravBlock;

// Block-cooperative staging of j records into LDS.  Every lane of a wave then
// reads the same LDS address (a broadcast read), so one j record serves the
// whole wave, and the block's 256 lanes share one coalesced global read of
// the tile.
template <class R>
__device__ __forceinline__ int stage_tile(R* __restrict__ s, const R* __restrict__ g, int t0, int n_j) {
  const int cnt = min(kJTile, n_j - t0);
  __syncthreads();
  for (int q = threadIdx.x; q < cnt; q += kGravBlock) s[q] = g[t0 + q];
  __syncthreads();
  return cnt;
}

// reference-layout kernel of the FP64 form (spline softening, and Plummer's
// reference arithmetic): gpos = (x,y,z,m), gvel.w = range^2
template <class T, int SOFT, int ACC, bool EXACT>
__global__ __launch_bounds__(kGravBlock) void k_gravity(const V4<T>* __restrict__ gpos,
                                                        const V4<T>* __restrict__ gvel, V4<T>* __restrict__ out,
                                                        int n_i, int n_j, T eps2) {
  __shared__ V4<T> s_pos[kJTile];
  __shared__ T s_r2[SOFT == 0 ? kJTile : 1];
  const int i = blockIdx.x * kGravBlock + threadIdx.x;
  const int ii = i < n_i ? i : n_i - 1;
  const V4<T> pi = gpos[ii];
  const T ri2 = SOFT == 0 ? gvel[ii].w : T(0);
  GAcc<T, ACC> a[4];
  for (int t0 = 0; t0 < n_j; t0 += kJTile) {
    const int cnt = stage_tile(s_pos, gpos, t0, n_j);
    if constexpr (SOFT == 0) {
      for (int q = threadIdx.x; q < cnt; q += kGravBlock) s_r2[q] = gvel[t0 + q].w;
      __syncthreads();
    }
    auto body = [&](int j) {
      const V4<T> pj = s_pos[j];
      const T rx = pi.x - pj.x, ry = pi.y - pj.y, rz = pi.z - pj.z;
      if constexpr (SOFT == 0) pair_spline<T, EXACT>(a, rx, ry, rz, ri2, pj.w, s_r2[j]);
      else pair_plummer<T, EXACT>(a, rx, ry, rz, pj.w, eps2);
    };
    // j in ascending order (the reference's summation order).  The loop is
    // left rolled: unrolling it measured slower for these longer pair bodies
    for (int j = 0; j < cnt; ++j) body(j);
  }
  if (i < n_i) out[i] = {a[0].get(), a[1].get(), a[2].get(), a[3].get()};
}

// ---------------------------------------------------------------------------
// Plain form: the reference's per-pair dreal sums.  A particle's four sums
// (ax, ay, az, potential) are serial chains from record to record, in
// ascending j, and each term is pair_plummer's (pair_spline's) expression, so
// the results are the reference's bits.
//
// FP32 VALU issue bounds it: 17 operations and an rsq for a pair's terms, and
// 4 two-sums of 10 operations; with few particles the latency of the chains
// (a dependent operation takes about 9 cycles in a lone wavefront, and a SIMD
// issues at its full rate only from 4 wavefronts on).
//
// k_gravity_chains (up to kChainsMaxN particles): a block takes 64 particles.
// Its first four wavefronts keep one sum each; the other four compute the
// terms, each of a quarter of a batch of records, and hand them over through
// LDS, double buffered, with one barrier per batch.  So a pair's distance
// and rsq are computed once, and every SIMD has an independent stream of
// terms beside its dependent chain.
//  * A chain takes its terms 8 at a time.  The fast two-sum is right where the
//    sum is at least as large as the term; for 8 terms that holds if |sum| >= 9
//    times the largest (7 of them lower |sum| by 7 times that at most).  Sums
//    over many records exceed their next terms by far: 87 % of the groups take
//    it at 16 384 particles, 98 % at 131 072.  The wavefront decides by one ballot,
//    and a group that fails takes dr_sub.
//  * Terms past the last record are zero: a two-sum with zero changes nothing.
//  * Spline softening: a record beyond both ranges has the Newtonian term.
//    One inside them has a term for each range; 4 records of which some lane
//    has one inside carry the second terms (zero for the others) in a buffer
//    of their own.
// Measured alone, one lane per particle (four wavefronts with a sum each up to
// 16 384, two with two each up to 65 536) -> this kernel, ms: Plummer 1 000
// particles 0.057 -> 0.044, 16 384: 0.88 -> 0.51, 32 768: 2.48 -> 1.42, 65 536:
// 5.9 -> 4.6, 100 003: 11.4 -> 11.3, 131 072: 15.0 -> 16.1; spline 16 384: 3.9 ->
// 0.82, 65 536: 13.9 -> 6.8, 100 003: 20.9 -> 17.0.  Plain Plummer step, beside
// the SPH passes, one lane / this kernel: 65 536: 7.6 / 5.3, 81 920: 10.1 / 8.6,
// 90 112: 11.0 / 10.2, 100 003: 12.1 / 12.5, 131 072: 15.7 / 16.3.  (32 records per batch: 16 384 particles 0.49, but 1 045
// against 914 ms at 2^20, where fewer blocks fit; two sums per wavefront:
// 16 384: 0.79, 65 536: 5.3.)
constexpr int kChainParticles = 64;   // particles per block

// the terms of one pair: y[0..2], y[3] and, with the spline softening, the
// second acceleration terms z[0..2]
struct PairTerms {
  float y[4], z[3];
};
// pair_spline's accumulator that takes its terms apart: the first sub of a
// component is its first term
struct TermSink {
  float first = 0.f, second = 0.f;
  bool have = false;
  __device__ __forceinline__ void sub(float y) {
    if (have) second = y;
    else first = y;
    have = true;
  }
};
struct TermSinks {
  TermSink a0, a1, a2, a3;
};

template <int SOFT, bool EXACT>
__device__ __forceinline__ bool pair_terms(PairTerms& t, const F4& pj, float rj2, const F4& pi, float ri2,
                                           float eps2) {
  const float rx = pi.x - pj.x, ry = pi.y - pj.y, rz = pi.z - pj.z;
  float d2 = rx * rx + ry * ry + rz * rz;
  if constexpr (SOFT == 1) d2 = d2 + eps2;
  const float inv = inv_sqrt<EXACT>(d2);
  const float s3 = pj.w * (inv * inv * inv);
  t.y[0] = rx * s3;
  t.y[1] = ry * s3;
  t.y[2] = rz * s3;
  t.y[3] = pj.w * inv;
  return SOFT == 0 && !(d2 >= ri2 && d2 >= rj2);
}
template <bool EXACT>
__device__ __forceinline__ void pair_terms_near(PairTerms& t, const F4& pj, float rj2, const F4& pi, float ri2) {
  TermSinks k;
  pair_spline<float, EXACT>(k, pi.x - pj.x, pi.y - pj.y, pi.z - pj.z, ri2, pj.w, rj2);
  t.y[0] = k.a0.first;
  t.y[1] = k.a1.first;
  t.y[2] = k.a2.first;
  t.y[3] = k.a3.first;
  t.z[0] = k.a0.second;
  t.z[1] = k.a1.second;
  t.z[2] = k.a2.second;
}

__device__ __forceinline__ float max_abs8(const float* y) {
  const float m = fmaxf(fmaxf(fabsf(y[0]), fabsf(y[1])), fabsf(y[2]));
  const float n = fmaxf(fmaxf(fabsf(y[3]), fabsf(y[4])), fabsf(y[5]));
  return fmaxf(fmaxf(m, n), fmaxf(fabsf(y[6]), fabsf(y[7])));
}
// 4 records (wavefront-uniform: scalar loads)
template <int SOFT>
struct Quad {
  F4 p[4];
  float r2[4];
  __device__ __forceinline__ void load(const F4* __restrict__ gpos, const F4* __restrict__ gvel, int j0, int n_j) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int j = min(j0 + k, n_j - 1);
      p[k] = gpos[j];
      r2[k] = SOFT == 0 ? gvel[j].w : 0.f;
    }
  }
};

// the terms of a quad at records j0 .. j0 + 3 for the lane's particle; returns
// whether some lane needs the second terms
template <int SOFT, bool EXACT>
__device__ __forceinline__ bool quad_terms(PairTerms (&t)[4], const Quad<SOFT>& r, int j0, int n_j, const F4& pi,
                                           float ri2, float eps2) {
  bool near = false;
#pragma unroll
  for (int k = 0; k < 4; ++k) near |= pair_terms<SOFT, EXACT>(t[k], r.p[k], r.r2[k], pi, ri2, eps2);
  bool any = false;
  if constexpr (SOFT == 0) {
    any = __any(near);
    if (any) {
#pragma unroll
      for (int k = 0; k < 4; ++k) pair_terms_near<EXACT>(t[k], r.p[k], r.r2[k], pi, ri2);
    }
  }
  if (j0 + 4 > n_j) {   // past the last record
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (j0 + k >= n_j) {
        t[k].y[0] = t[k].y[1] = t[k].y[2] = t[k].y[3] = 0.f;
        t[k].z[0] = t[k].z[1] = t[k].z[2] = 0.f;
      }
  }
  return any;
}

constexpr int kChainBlock = 512;
template <int SOFT, bool EXACT>
__global__ __launch_bounds__(kChainBlock) void k_gravity_chains(const F4* __restrict__ gpos,
                                                             const F4* __restrict__ gvel, F4* __restrict__ out,
                                                             int n_i, int n_j, float eps2) {
  constexpr int B = 16, Q = B / 4;   // records and quads per batch, one quad per wavefront of terms
  __shared__ float4 s_y[2][4][Q][64];
  __shared__ float4 s_z[SOFT == 0 ? 2 : 1][SOFT == 0 ? 3 : 1][SOFT == 0 ? Q : 1][SOFT == 0 ? 64 : 1];
  __shared__ int s_near[2][Q];
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int i = blockIdx.x * kChainParticles + lane;
  const int ii = i < n_i ? i : n_i - 1;
  const int batches = (n_j + B - 1) / B;
  if (w >= 4) {   // terms
    const F4 pi = gpos[ii];
    const float ri2 = SOFT == 0 ? gvel[ii].w : 0.f;
    const int quad = w - 4;
    Quad<SOFT> r;
    r.load(gpos, gvel, quad * 4, n_j);
    for (int b = 0; b < batches; ++b) {
      Quad<SOFT> next;   // (past the last batch: the last record once more, unused)
      next.load(gpos, gvel, (b + 1) * B + quad * 4, n_j);
      PairTerms t[4];
      const bool any = quad_terms<SOFT, EXACT>(t, r, b * B + quad * 4, n_j, pi, ri2, eps2);
#pragma unroll
      for (int c = 0; c < 4; ++c)
        s_y[b & 1][c][quad][lane] = make_float4(t[0].y[c], t[1].y[c], t[2].y[c], t[3].y[c]);
      if constexpr (SOFT == 0) {
        if (any) {
#pragma unroll
          for (int c = 0; c < 3; ++c)
            s_z[b & 1][c][quad][lane] = make_float4(t[0].z[c], t[1].z[c], t[2].z[c], t[3].z[c]);
        }
        if (lane == 0) s_near[b & 1][quad] = any;
      }
      r = next;
      __syncthreads();
    }
  } else {   // chains: batch b while the next one's terms are computed
    Chain a;
    for (int b = 0; b < batches; ++b) {
      __syncthreads();
      float y[B];
#pragma unroll
      for (int k = 0; k < Q; ++k) {
        const float4 v = s_y[b & 1][w][k][lane];
        y[4 * k] = v.x, y[4 * k + 1] = v.y, y[4 * k + 2] = v.z, y[4 * k + 3] = v.w;
      }
      unsigned second = 0;   // quads with second terms (the potential has none)
      if (SOFT == 0 && w < 3) {
#pragma unroll
        for (int k = 0; k < Q; ++k)
          second |= (unsigned)__builtin_amdgcn_readfirstlane(s_near[b & 1][k]) << k;
      }
      float m = max_abs8(y);
      bool fast = __all(fabsf(a.hi) >= 9.f * m);
#pragma unroll
      for (int g = 0; g < B; g += 8) {
        const float mn = g + 8 < B ? max_abs8(y + g + 8) : 0.f;
        if (SOFT == 0 && ((second >> (g / 4)) & 3u)) {
#pragma unroll
          for (int h = g / 4; h < g / 4 + 2; ++h) {
            const float4 e = (second >> h) & 1u ? s_z[b & 1][w % 3][h][lane] : make_float4(0.f, 0.f, 0.f, 0.f);
            a.sub(y[4 * h]);
            a.sub(e.x);
            a.sub(y[4 * h + 1]);
            a.sub(e.y);
            a.sub(y[4 * h + 2]);
            a.sub(e.z);
            a.sub(y[4 * h + 3]);
            a.sub(e.w);
          }
          fast = __all(fabsf(a.hi) >= 9.f * mn);
        } else {
          // the next 8 are judged by the sum before these 8, which lower it
          // by 8 times their largest at most: the verdict is there in time
          const bool next = __all(fabsf(a.hi) >= 9.5f * (m + mn));
          if (fast) {
#pragma unroll
            for (int k = 0; k < 8; ++k) a.sub_fast_alone(y[g + k]);
          } else {
#pragma unroll
            for (int k = 0; k < 8; ++k) a.sub(y[g + k]);
          }
          fast = next;
        }
        m = mn;
      }
    }
    if (i < n_i) reinterpret_cast<float*>(out + i)[w] = a.hi;
  }
}

// Many particles: a lane keeps all four chains of its particle, 256 particles
// per block, the records in LDS tiles, software-pipelined (the next record's
// terms are computed in the same block as the current one's chain steps).
template <bool EXACT>
__global__ __launch_bounds__(kGravBlock) void k_gravity_lane(const F4* __restrict__ gpos, F4* __restrict__ out,
                                                             int n_i, int n_j, float eps2) {
  __shared__ F4 s_pos[kJTile];
  const int i = blockIdx.x * kGravBlock + threadIdx.x;
  const F4 pi = gpos[i < n_i ? i : n_i - 1];
  DR a0{0.f, 0.f}, a1{0.f, 0.f}, a2{0.f, 0.f}, a3{0.f, 0.f};
  for (int t0 = 0; t0 < n_j; t0 += kJTile) {
    const int cnt = stage_tile(s_pos, gpos, t0, n_j);
    auto terms = [&](int j) {
      PairTerms t;
      pair_terms<1, EXACT>(t, s_pos[j], 0.f, pi, 0.f, eps2);
      return F4{t.y[0], t.y[1], t.y[2], t.y[3]};
    };
    auto chain = [&](const F4& y) {
      dr_sub(a0, y.x);
      dr_sub(a1, y.y);
      dr_sub(a2, y.z);
      dr_sub(a3, y.w);
    };
    F4 y = terms(0);
    for (int j = 1; j < cnt; ++j) {
      const F4 yn = terms(j);
      chain(y);
      y = yn;
    }
    chain(y);
  }
  if (i < n_i) out[i] = {a0.hi, a1.hi, a2.hi, a3.hi};
}

// The same with the shortened two-sum, the records judged 16 at a time by a
// bound of their terms that needs only the group's place: M / d^2 for an
// acceleration and M / d for the potential, M the group's largest mass and d
// its distance (from a record of the group, less the group's radius about it).
// A group that fails, or one that comes within the spline's ranges, takes its
// records one by one.  Measured, Plummer, this kernel against k_gravity_lane:
// 131 072 particles 18.9 / 15.0 ms, 262 144: 64.3 / 58.9 (2 and 4 wavefronts per
// SIMD, where the longer block issues worse), 2^20: 848 / 946.  Spline, against
// the one-record loop it replaces: 100 003: 15.5 / 20.9, 131 072: 19.4 / 26.9,
// 262 144: 65.6 / 85.2.
constexpr int kLaneGroup = 16;
struct LaneGroup {
  float x, y, z, radius;
  float m, r2;   // 17.5 times the largest |mass|; the largest range^2
};

template <int SOFT, bool EXACT>
__global__ __launch_bounds__(kGravBlock) void k_gravity_lane_fast(const F4* __restrict__ gpos,
                                                                  const F4* __restrict__ gvel, F4* __restrict__ out,
                                                                  int n_i, int n_j, float eps2) {
  __shared__ F4 s_pos[kJTile + 1];   // (the last one is read ahead, unused)
  __shared__ float s_r2[SOFT == 0 ? kJTile : 1];
  __shared__ LaneGroup s_group[kJTile / kLaneGroup];
  const int i = blockIdx.x * kGravBlock + threadIdx.x;
  const int ii = i < n_i ? i : n_i - 1;
  const F4 pi = gpos[ii];
  const float ri2 = SOFT == 0 ? gvel[ii].w : 0.f;
  Chains4 a;
  for (int t0 = 0; t0 < n_j; t0 += kJTile) {
    const int cnt = min(kJTile, n_j - t0);
    __syncthreads();
    for (int q = threadIdx.x; q < kJTile; q += kGravBlock) {
      const int j = min(t0 + q, n_j - 1);   // (past the end: the last record again, outside every whole group)
      const F4 p = gpos[j];
      s_pos[q] = p;
      float r2 = 0.f;
      if constexpr (SOFT == 0) {
        r2 = gvel[j].w;
        s_r2[q] = r2;
      }
      const float cx = __shfl(p.x, kLaneGroup / 2, kLaneGroup), cy = __shfl(p.y, kLaneGroup / 2, kLaneGroup),
                  cz = __shfl(p.z, kLaneGroup / 2, kLaneGroup);
      const float dx = p.x - cx, dy = p.y - cy, dz = p.z - cz;
      float d2 = dx * dx + dy * dy + dz * dz, m = fabsf(p.w);
      for (int o = 1; o < kLaneGroup; o <<= 1) {
        d2 = fmaxf(d2, __shfl_xor(d2, o));
        m = fmaxf(m, __shfl_xor(m, o));
        if constexpr (SOFT == 0) r2 = fmaxf(r2, __shfl_xor(r2, o));
      }
      if (q % kLaneGroup == 0)
        s_group[q / kLaneGroup] = {cx, cy, cz, 1.00001f * __builtin_sqrtf(d2), 17.5f * m, r2};
    }
    __syncthreads();
    auto terms = [&](int j) {
      PairTerms t;
      pair_terms<SOFT, EXACT>(t, s_pos[j], 0.f, pi, ri2, eps2);
      return F4{t.y[0], t.y[1], t.y[2], t.y[3]};
    };
    auto one = [&](int j) {
      const F4 pj = s_pos[j];
      const float rx = pi.x - pj.x, ry = pi.y - pj.y, rz = pi.z - pj.z;
      if constexpr (SOFT == 0) pair_spline<float, EXACT>(a, rx, ry, rz, ri2, pj.w, s_r2[j]);
      else pair_plummer<float, EXACT>(a, rx, ry, rz, pj.w, eps2);
    };
    auto chain = [&](const F4& y) {
      a.a0.sub(y.x);
      a.a1.sub(y.y);
      a.a2.sub(y.z);
      a.a3.sub(y.w);
    };
    int g = 0;
    F4 y = terms(0);
    for (; (g + 1) * kLaneGroup <= cnt; ++g) {
      const LaneGroup b = s_group[g];
      const float dx = pi.x - b.x, dy = pi.y - b.y, dz = pi.z - b.z;
      const float d = fmaxf(__builtin_amdgcn_sqrtf(dx * dx + dy * dy + dz * dz) - b.radius, 0.f);
      const float d2 = SOFT == 1 ? d * d + eps2 : d * d;
      const int j0 = g * kLaneGroup;
      if (SOFT == 0 && !__all(0.99999f * d2 >= fmaxf(ri2, b.r2))) {
        for (int k = 0; k < kLaneGroup; ++k) one(j0 + k);
        y = terms(j0 + kLaneGroup);
        continue;
      }
      const float inv = __builtin_amdgcn_rsqf(d2), pot = b.m * inv, acc = pot * inv;
      const bool fast = fminf(fminf(fabsf(a.a0.hi), fabsf(a.a1.hi)), fabsf(a.a2.hi)) >= acc && fabsf(a.a3.hi) >= pot;
      if (__all(fast)) {
#pragma unroll 2
        for (int k = 1; k <= kLaneGroup; ++k) {
          const F4 n = terms(j0 + k);
          a.a0.sub_fast(y.x);
          a.a1.sub_fast(y.y);
          a.a2.sub_fast(y.z);
          a.a3.sub_fast(y.w);
          y = n;
        }
      } else {
#pragma unroll 1
        for (int k = 1; k <= kLaneGroup; ++k) {
          const F4 n = terms(j0 + k);
          chain(y);
          y = n;
        }
      }
    }
    for (int j = g * kLaneGroup; j < cnt; ++j) one(j);
  }
  if (i < n_i) out[i] = {a.a0.hi, a.a1.hi, a.a2.hi, a.a3.hi};
}

// ---------------------------------------------------------------------------
// Multipole far field of the mixed Plummer kernel (optional, flags bit 4).
//
// Each 64-record sub-tile of the j-set (records [64 s, 64 s + 64), the
// sub-tiles the kernel below stages) gets its moments up to order 4 about its
// centre of mass, for the softened kernel phi(y) = (|y|^2 + eps^2)^(-1/2):
//   sum_j m_j phi(y - e_j) = sum_n (-1)^n / n! M^(n) . D^(n)(y),
//   M^(n) = sum_j m_j e_j^(x n),  D^(n) = grad^n phi,  e_j = x_j - COM.
// phi depends on u = |y|^2 / 2 only, so D^(n) is a sum over pairings of its
// indices: g_{n-m} times y^(n-2m) and m Kronecker deltas, with
// g_k = d^k phi / du^k = (-1)^k (2k-1)!! s^-(2k+1), s^2 = |y|^2 + eps^2.
// Contracted with the (not traceless: phi is not harmonic under softening)
// moments this needs M2, M3, M4, their traces tr M2, t3 = tr M3 and
// Q = tr M4, tr Q.  M^(1) = 0 about the centre of mass.  Truncation after
// order 4 leaves a relative error ~ (R / |y|)^5 of the sub-tile's force
// (R = max |e_j|): the far field is used for a (wavefront, sub-tile) only
// when every lane has |y| >= q R.  The default q = 8 (the engine's
// grav_far_ratio) bounds that error near 1e-6 of one sub-tile's force, below
// the FP32 pair arithmetic's: measured against FP64 at N = 2^20 the median
// per-particle error rises by 5 % over the pairwise kernel's, the maximum
// not at all; at q = 5 the maximum passes 1e-5.
constexpr int kMomWords = 52;     // floats per sub-tile record, see k_subtile_moments

__device__ __forceinline__ float wave_sum(float v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// the factors of the stored moments (far_field)
constexpr float kTrM2 = 0.5f, kTrQ = 0.375f, kM2 = 3.f, kT3 = -1.5f, kQ = 7.5f, kM3 = -7.5f, kM4 = 17.5f;

// record of sub-tile s: [0..2] centre-of-mass offset from the origin record
// (the middle real record; its coordinates in [48..50]), [3] R^2, [4] M0
// (0: no real record, the sub-tile is skipped), [5] tr M2,
// [6] tr Q, [8..13] M2 (xx xy xz yy yz zz), [14..16] t3, [17..22] Q,
// [23..32] M3 (xxx xxy xxz xyy xyz xzz yyy yyz yzz zzz), [33..47] M4
// (xxxx xxxy xxxz xxyy xxyz xxzz xyyy xyyz xyzz xzzz yyyy yyyz yyzz yzzz
// zzzz), [5..47] times their factors.  Masses as the kernel uses them (1 when every mass is equal);
// padding records (j >= n_real) are left out.  One wavefront per sub-tile.
__global__ __launch_bounds__(kGravBlock) void k_subtile_moments(const F4* __restrict__ hi, const F4* __restrict__ lo,
                                                                float* __restrict__ mom, int n_j, int n_real,
                                                                int n_sub, int G, int flags,
                                                                const float* __restrict__ mass_range) {
  const bool uniform = (flags & 2) == 0 && mass_range[0] == mass_range[1];
  const int s = blockIdx.x * (kGravBlock / 64) + (int)(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (s >= n_sub) return;   // whole wavefronts
  // a group of G <= 64 records; lanes past it add nothing (a group past
  // n_j, possible for G < 64, is empty: M0 = 0, skipped where it is read)
  const int j0 = s * G, nj = min(G, n_j - j0);
  // origin: the middle real record (a padding record sits at 1e30)
  const int nr = max(0, min(nj, n_real - j0));
  const F4 c = hi[min(j0 + nr / 2, n_j - 1)];
  const int j = j0 + lane;
  const bool valid = lane < nj && j < n_real;
  float dx = 0.f, dy = 0.f, dz = 0.f, m = 0.f;
  if (valid) {
    const F4 h = hi[j], l = lo[j];
    dx = (h.x - c.x) + l.x;
    dy = (h.y - c.y) + l.y;
    dz = (h.z - c.z) + l.z;
    m = uniform ? 1.f : h.w;
  }
  const float M0 = wave_sum(m);
  const float sx = wave_sum(m * dx), sy = wave_sum(m * dy), sz = wave_sum(m * dz);
  const float mx = M0 > 0.f ? sx / M0 : 0.f, my = M0 > 0.f ? sy / M0 : 0.f, mz = M0 > 0.f ? sz / M0 : 0.f;
  const float ex = valid ? dx - mx : 0.f, ey = valid ? dy - my : 0.f, ez = valid ? dz - mz : 0.f;
  float r2 = __builtin_fmaf(ex, ex, __builtin_fmaf(ey, ey, ez * ez));
  for (int o = 32; o > 0; o >>= 1) r2 = fmaxf(r2, __shfl_xor(r2, o));
  const float mex = m * ex, mey = m * ey, mez = m * ez;
  const float xx = mex * ex, xy = mex * ey, xz = mex * ez, yy = mey * ey, yz = mey * ez, zz = mez * ez;
  const float xxx = xx * ex, xxy = xx * ey, xxz = xx * ez, xyy = xy * ey, xyz = xy * ez, xzz = xz * ez,
              yyy = yy * ey, yyz = yy * ez, yzz = yz * ez, zzz = zz * ez;
  const float p4[15] = {xxx * ex, xxx * ey, xxx * ez, xxy * ey, xxy * ez, xxz * ez, xyy * ey, xyy * ez,
                        xyz * ez, xzz * ez, yyy * ey, yyy * ez, yyz * ez, yzz * ez, zzz * ez};
  const float p2[6] = {xx, xy, xz, yy, yz, zz};
  const float p3[10] = {xxx, xxy, xxz, xyy, xyz, xzz, yyy, yyz, yzz, zzz};
  float M2[6], M3[10], M4[15];
#pragma unroll
  for (int k = 0; k < 6; ++k) M2[k] = wave_sum(p2[k]);
#pragma unroll
  for (int k = 0; k < 10; ++k) M3[k] = wave_sum(p3[k]);
#pragma unroll
  for (int k = 0; k < 15; ++k) M4[k] = wave_sum(p4[k]);
  if (lane == 0) {
    float* r = mom + (size_t)s * kMomWords;
    const float Q[6] = {M4[0] + M4[3] + M4[5], M4[1] + M4[6] + M4[8], M4[2] + M4[7] + M4[9],
                        M4[3] + M4[10] + M4[12], M4[4] + M4[11] + M4[13], M4[5] + M4[12] + M4[14]};
    r[0] = mx;
    r[1] = my;
    r[2] = mz;
    r[3] = r2;
    r[4] = M0;
    r[5] = kTrM2 * (M2[0] + M2[3] + M2[5]);
    r[6] = kTrQ * (Q[0] + Q[3] + Q[5]);
    r[7] = 0.f;
#pragma unroll
    for (int k = 0; k < 6; ++k) r[8 + k] = kM2 * M2[k];
    r[14] = kT3 * (M3[0] + M3[3] + M3[5]);
    r[15] = kT3 * (M3[1] + M3[6] + M3[8]);
    r[16] = kT3 * (M3[2] + M3[7] + M3[9]);
#pragma unroll
    for (int k = 0; k < 6; ++k) r[17 + k] = kQ * Q[k];
#pragma unroll
    for (int k = 0; k < 10; ++k) r[23 + k] = kM3 * M3[k];
#pragma unroll
    for (int k = 0; k < 15; ++k) r[33 + k] = kM4 * M4[k];
    r[48] = c.x;
    r[49] = c.y;
    r[50] = c.z;
    r[51] = 0.f;
  }
}

// Cells of C = 256, 1024, 4096 and 16384 records (the hierarchy above the
// sub-tiles): one block per cell, the same record layout.  Sums in FP64, the
// whole cell at once: a cell holds up to 16384 records, whose FP32 sums
// would round at ~1e-5.
constexpr int kFarLevels = 4;
constexpr int kCellSize[kFarLevels] = {16384, 4096, 1024, 256};   // coarse to fine
// squared acceptance ratios: [L] for the cell level L, [kFarLevels] for
// the 64-record sub-tiles, [kFarLevels + 1] for their 32-record halves
struct FarRatios {
  float q2[kFarLevels + 2];
};

__device__ __forceinline__ double block_sum(double v, double* s_red) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = v;
  __syncthreads();
  double t = 0.0;
  for (int w = 0; w < kGravBlock / 64; ++w) t += s_red[w];   // fixed order, every thread the same
  return t;
}

__global__ __launch_bounds__(kGravBlock) void k_cell_moments(const F4* __restrict__ hi, const F4* __restrict__ lo,
                                                             float* __restrict__ mom, int n_j, int n_real, int C,
                                                             int flags, const float* __restrict__ mass_range) {
  __shared__ double s_red[kGravBlock / 64];
  const bool uniform = (flags & 2) == 0 && mass_range[0] == mass_range[1];
  const int cell = blockIdx.x;
  const int j0 = cell * C, nj = min(C, n_j - j0);
  // origin: the middle real record (a padding record sits at 1e30)
  const int nr = max(0, min(nj, n_real - j0));
  const F4 c = hi[j0 + nr / 2];
  // pass 1: mass and centre of mass
  double m0 = 0.0, sx = 0.0, sy = 0.0, sz = 0.0;
  for (int q = threadIdx.x; q < nj; q += kGravBlock) {
    const int j = j0 + q;
    if (j >= n_real) continue;
    const F4 h = hi[j], l = lo[j];
    const double m = uniform ? 1.0 : (double)h.w;
    m0 += m;
    sx += m * (double)((h.x - c.x) + l.x);
    sy += m * (double)((h.y - c.y) + l.y);
    sz += m * (double)((h.z - c.z) + l.z);
  }
  m0 = block_sum(m0, s_red);
  sx = block_sum(sx, s_red);
  sy = block_sum(sy, s_red);
  sz = block_sum(sz, s_red);
  const double mx = m0 > 0.0 ? sx / m0 : 0.0, my = m0 > 0.0 ? sy / m0 : 0.0, mz = m0 > 0.0 ? sz / m0 : 0.0;
  // pass 2: radius and central moments
  double acc[31];
  for (int k = 0; k < 31; ++k) acc[k] = 0.0;
  float r2 = 0.f;
  for (int q = threadIdx.x; q < nj; q += kGravBlock) {
    const int j = j0 + q;
    if (j >= n_real) continue;
    const F4 h = hi[j], l = lo[j];
    const double m = uniform ? 1.0 : (double)h.w;
    const double ex = (double)((h.x - c.x) + l.x) - mx, ey = (double)((h.y - c.y) + l.y) - my,
                 ez = (double)((h.z - c.z) + l.z) - mz;
    r2 = fmaxf(r2, (float)(ex * ex + ey * ey + ez * ez));
    const double xx = m * ex * ex, xy = m * ex * ey, xz = m * ex * ez, yy = m * ey * ey, yz = m * ey * ez,
                 zz = m * ez * ez;
    const double xxx = xx * ex, xxy = xx * ey, xxz = xx * ez, xyy = xy * ey, xyz = xy * ez, xzz = xz * ez,
                 yyy = yy * ey, yyz = yy * ez, yzz = yz * ez, zzz = zz * ez;
    const double t[31] = {xx, xy, xz, yy, yz, zz, xxx, xxy, xxz, xyy, xyz, xzz, yyy, yyz, yzz, zzz,
                          xxx * ex, xxx * ey, xxx * ez, xxy * ey, xxy * ez, xxz * ez, xyy * ey, xyy * ez,
                          xyz * ez, xzz * ez, yyy * ey, yyy * ez, yyz * ez, yzz * ez, zzz * ez};
    for (int k = 0; k < 31; ++k) acc[k] += t[k];
  }
  for (int k = 0; k < 31; ++k) acc[k] = block_sum(acc[k], s_red);
  for (int o = 32; o > 0; o >>= 1) r2 = fmaxf(r2, __shfl_xor(r2, o));
  __syncthreads();
  float* s_r2 = reinterpret_cast<float*>(s_red);
  if ((threadIdx.x & 63) == 0) s_r2[threadIdx.x >> 6] = r2;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kGravBlock / 64; ++w) r2 = fmaxf(r2, s_r2[w]);
    const double* M2 = acc;
    const double* M3 = acc + 6;
    const double* M4 = acc + 16;
    const double Q[6] = {M4[0] + M4[3] + M4[5], M4[1] + M4[6] + M4[8], M4[2] + M4[7] + M4[9],
                         M4[3] + M4[10] + M4[12], M4[4] + M4[11] + M4[13], M4[5] + M4[12] + M4[14]};
    float* r = mom + (size_t)cell * kMomWords;
    r[0] = (float)mx;
    r[1] = (float)my;
    r[2] = (float)mz;
    r[3] = r2;
    r[4] = (float)m0;
    r[5] = (float)(kTrM2 * (M2[0] + M2[3] + M2[5]));
    r[6] = (float)(kTrQ * (Q[0] + Q[3] + Q[5]));
    r[7] = 0.f;
    for (int k = 0; k < 6; ++k) r[8 + k] = (float)(kM2 * M2[k]);
    r[14] = (float)(kT3 * (M3[0] + M3[3] + M3[5]));
    r[15] = (float)(kT3 * (M3[1] + M3[6] + M3[8]));
    r[16] = (float)(kT3 * (M3[2] + M3[7] + M3[9]));
    for (int k = 0; k < 6; ++k) r[17 + k] = (float)(kQ * Q[k]);
    for (int k = 0; k < 10; ++k) r[23 + k] = (float)(kM3 * M3[k]);
    for (int k = 0; k < 15; ++k) r[33 + k] = (float)(kM4 * M4[k]);
    r[48] = c.x;
    r[49] = c.y;
    r[50] = c.z;
    r[51] = 0.f;
  }
}

// acceleration G = sum_j m_j (x_j - x_i) s^-3 and potential -sum_j m_j / s of
// one sub-tile from its record M, at y = x_i - COM (order-4 expansion):
//   sum m_j / s = sum_k g_k B_k and G = y sum_k g_(k+1) B_k + sum_k g_k V_k with
//   V_2 = M2.y - t3 / 2, V_3 = (Q.y - M3.yy) / 2, V_4 = M4.yyy / 6,
//   B_0 = M0, B_1 = tr M2 / 2, B_2 = y.M2.y / 2 - t3.y / 2 + tr Q / 8,
//   B_3 = y.Q.y / 4 - M3.yyy / 6, B_4 = M4.yyyy / 24,
// that is B_3 = y.(V_3 + Q.y / 4) / 3 and B_4 = y.V_4 / 4.  The kernel with the far
// field is bound by VALU issue, these operations about half of it: counted at
// 2^20 particles, a wavefront takes 6 500 expansions and 84 000 pairs (polytropes:
// 1.0e6 and 1.1e6 operations), 8 300 and 68 000 (turbulent sphere: 1.3e6, 0.9e6).
// The moments are stored with the factors (2 k - 1)!! of g_k, so that the G_k are
// plain powers, and every line is a chain of multiply-adds: 141 operations
// and a v_rsq_f32 (196 term by term).
__device__ __forceinline__ void far_field(const float* __restrict__ M, float yx, float yy, float yz, float eps2,
                                          float& gx, float& gy, float& gz, float& pot) {
  const auto fma = [](float a, float b, float c) { return __builtin_fmaf(a, b, c); };
  const float s2 = fma(yx, yx, fma(yy, yy, fma(yz, yz, eps2)));
  const float G0 = rsq_spaced(s2), h = -G0 * G0;
  const float G1 = G0 * h, G2 = G1 * h, G3 = G2 * h, G4 = G3 * h, G5 = G4 * h;
  const float* m2 = M + 8;
  const float* t3 = M + 14;
  const float* Q = M + 17;
  const float* m3 = M + 23;
  const float* m4 = M + 33;
  const float V2x = fma(m2[0], yx, fma(m2[1], yy, fma(m2[2], yz, t3[0])));
  const float V2y = fma(m2[1], yx, fma(m2[3], yy, fma(m2[4], yz, t3[1])));
  const float V2z = fma(m2[2], yx, fma(m2[4], yy, fma(m2[5], yz, t3[2])));
  const float B2 = fma(0.5f, fma(V2x + t3[0], yx, fma(V2y + t3[1], yy, (V2z + t3[2]) * yz)), M[6]);
  // quadratic monomials, off-diagonal ones doubled: (M3 . y y)_k
  const float yx2 = 2.f * yx, yy2 = 2.f * yy;
  const float qxx = yx * yx, qxy = yx2 * yy, qxz = yx2 * yz, qyy = yy * yy, qyz = yy2 * yz, qzz = yz * yz;
  const float Qx = fma(Q[0], yx, fma(Q[1], yy, Q[2] * yz));
  const float Qy = fma(Q[1], yx, fma(Q[3], yy, Q[4] * yz));
  const float Qz = fma(Q[2], yx, fma(Q[4], yy, Q[5] * yz));
  const auto dot6 = [&](float a, float b, float c, float d, float e, float f, float to) {
    return fma(qxx, a, fma(qxy, b, fma(qxz, c, fma(qyy, d, fma(qyz, e, fma(qzz, f, to))))));
  };
  const float V3x = dot6(m3[0], m3[1], m3[2], m3[3], m3[4], m3[5], Qx);
  const float V3y = dot6(m3[1], m3[3], m3[4], m3[6], m3[7], m3[8], Qy);
  const float V3z = dot6(m3[2], m3[4], m3[5], m3[7], m3[8], m3[9], Qz);
  const float B3 = (1.f / 3.f) * fma(fma(0.5f, Qx, V3x), yx, fma(fma(0.5f, Qy, V3y), yy, fma(0.5f, Qz, V3z) * yz));
  // cubic monomials with their multinomial weights: (M4 . y y y)_k
  const float qxx3 = 3.f * qxx, qyy3 = 3.f * qyy, qzz3 = 3.f * qzz;
  const float cxxx = qxx * yx, cxxy = qxx3 * yy, cxxz = qxx3 * yz, cxyy = qyy3 * yx, cxyz = 3.f * qxy * yz,
              cxzz = qzz3 * yx, cyyy = qyy * yy, cyyz = qyy3 * yz, cyzz = qzz3 * yy, czzz = qzz * yz;
  const auto dot10 = [&](int a, int b, int c, int d, int e, int f, int g, int k, int l, int m) {
    return fma(cxxx, m4[a], fma(cxxy, m4[b], fma(cxxz, m4[c], fma(cxyy, m4[d], fma(cxyz, m4[e],
           fma(cxzz, m4[f], fma(cyyy, m4[g], fma(cyyz, m4[k], fma(cyzz, m4[l], czzz * m4[m])))))))));
  };
  const float V4x = dot10(0, 1, 2, 3, 4, 5, 6, 7, 8, 9);
  const float V4y = dot10(1, 3, 4, 6, 7, 8, 10, 11, 12, 13);
  const float V4z = dot10(2, 4, 5, 7, 8, 9, 11, 12, 13, 14);
  const float B4 = 0.25f * fma(V4x, yx, fma(V4y, yy, V4z * yz));
  const float A = fma(M[4], G1, fma(3.f * M[5], G2, fma(5.f * B2, G3, fma(7.f * B3, G4, 9.f * B4 * G5))));
  pot = -fma(M[4], G0, fma(M[5], G1, fma(B2, G2, fma(B3, G3, B4 * G4))));
  gx = fma(A, yx, fma(G2, V2x, fma(G3, V3x, G4 * V4x)));
  gy = fma(A, yy, fma(G2, V2y, fma(G3, V3y, G4 * V4y)));
  gz = fma(A, yz, fma(G2, V2z, fma(G3, V3z, G4 * V4z)));
}

// mixed form, Plummer: split positions, FMA pair arithmetic, blocked
// compensated sums.  hi = (x,y,z,m) rounded, lo = (x-hi, y-hi, z-hi, 0).
//
// Two ways to form r = x_i - x_j, chosen per (wavefront, sub-tile of 64 j):
//  split:  r = (hi_i - hi_j) + (lo_i - lo_j), 9 operations per pair, relative
//          error ~2^-24 for every pair;
//  tile:   the sub-tile is expressed relative to its middle record c,
//          d_j = (hi_j - c) + lo_j (staged in LDS) and d_i = (hi_i - c) + lo_i
//          (once per sub-tile per lane), r = d_i - d_j: 3 operations per pair,
//          absolute error <= 2^-24 (|d_i| + |d_j|) + rounding of r.
// The tile form is used only when every lane of the wavefront has
// |d_i| >= 3 R, R = max_j |d_j| over the sub-tile: then |r| >= |d_i| - R >= 2 R
// and (|d_i| + |d_j|) / |r| <= (|d_i| + R) / (|d_i| - R) <= 2, so r keeps a
// relative error of a few 2^-24 -- the accuracy of the split form.
// Wavefronts near a sub-tile (the pairs whose separation the split
// coordinates exist for) use the split form.  With particles in
// Peano-Hilbert order 64 consecutive records are compact and most
// (wavefront, sub-tile) combinations are far apart; with an unordered input
// every sub-tile is as large as the system and every wavefront uses the split
// form.  split_only bit 0 forces the split form everywhere; bit 1 disables
// the unit-mass body; bit 2 the expanded unit-mass tile body (measurement
// switches).
// After r: 3 FMAs for r^2 + eps^2, one rsq, 3 multiplies, 3 FMAs into the
// partial acceleration, 1 subtraction for the potential.  With every mass
// equal, tile-form sub-tiles skip r altogether (the expanded body below).
//
// This kernel evaluates every ordered pair: with the far field, with a
// measurement switch, and below kMixedPairsMinN particles
// (k_gravity_mixed_pairs otherwise).
// Grid: `parts` j-parts per i-block, block b = i_block * parts + part.  Part p
// takes the units p, p + parts, ... of j_unit records: tiles of 256, so that
// the sub-tiles near an i-block, which are slower, fall to its parts evenly
// (one contiguous unit per part below two tiles each, and for the far field,
// whose cells must lie inside a part).  Workgroups are dispatched round-robin
// over the 8 XCDs, so with 8 parts part p runs on XCD p and each XCD streams
// only its 1/8 of the j-set (4 MiB of hi+lo records at N = 2^20), which its L2
// holds; without the split every XCD streams the whole j-set and re-fetches it
// from HBM.  Each block writes its compensated (hi, lo) partial sums;
// k_gravity_combine adds the parts in order.
// The far-field instantiation holds the 48 moment words of an expansion in
// VGPRs next to the pairwise state: left alone the compiler takes 127
// registers (4 wavefronts per SIMD); capped at 5 wavefronts it fits 96
// registers without spilling (at 6 it spills 15 registers and runs 4-8 %
// slower).  The pairwise instantiation is held to 8 wavefronts (60 registers;
// left alone it took 125, and 65 536 particles 2.2 in place of 1.9 ms).
template <int JT, bool FAR>
__global__ __launch_bounds__(kGravBlock) __attribute__((amdgpu_waves_per_eu(FAR ? 5 : 8)))
void k_gravity_mixed_plummer(const F4* __restrict__ hi, const F4* __restrict__ lo, F4* __restrict__ part_hi,
                             F4* __restrict__ part_lo, int n_i, int n_j, int j_unit, float eps2, int split_only,
                             const float* __restrict__ mass_range, const float* __restrict__ mom,
                             FarRatios far_q2, const float* __restrict__ cells,
                             const float* __restrict__ halves, int n_real, int parts) {
  // every mass equal (mass_range = {min, max} over the real particles): the
  // pair body drops its mass factor and k_gravity_combine scales by m once;
  // padding records sit at 1e30, where r^2 overflows and rsq returns 0, so
  // they add exactly nothing without their zero mass
  const bool uniform = (split_only & 2) == 0 && mass_range[0] == mass_range[1];
  const bool expand = uniform && (split_only & 4) == 0;
  // a separate instantiation: the far-field code raises the VGPR count, which
  // would lower the occupancy of the pairwise kernel
  const bool far_on = FAR && (split_only & 1) == 0;
  // split_only bit 6: 32-record halves of a sub-tile not taken whole
  const bool half_on = far_on && (split_only & 64) != 0 && halves != nullptr;
  split_only &= 1;
  constexpr int kSub = JT / kTile;   // sub-tiles of kTile records, each with its own origin
  __shared__ F4 s_hi[JT], s_lo[JT], s_rel[JT];
  __shared__ F4 s_c[kSub];
  __shared__ float s_r2[kSub];
  __shared__ __align__(16) float s_mom[kSub][FAR ? kMomWords : 1];
  static_assert(kTile == 64 && JT % kGravBlock == 0, "each wavefront stages whole sub-tiles");
  const int part = blockIdx.x % parts;
  const int i = (blockIdx.x / parts) * kGravBlock + threadIdx.x;
  const int ii = i < n_i ? i : n_i - 1;
  const int lane = threadIdx.x & 63;
  const F4 pi = hi[ii], li = lo[ii];
  // padding lanes (records at 1e30) take no far-field term: its products
  // would overflow there; they pass every acceptance test
  const bool real_i = !FAR || i < n_real;
  GAcc<float, 1> a[4];
  auto add_far = [&](const float* M, float yx, float yy, float yz) {
    float gx, gy, gz, pt;
    far_field(M, yx, yy, yz, eps2, gx, gy, gz, pt);
    if (real_i) {
      a[0].part += gx;
      a[1].part += gy;
      a[2].part += gz;
      a[3].part += pt;
    }
  };
  int j_begin = part * j_unit, j_end = min(j_begin + j_unit, n_j);
  auto next_tile = [&](int t) {
    t += JT;
    if (t < j_end) return t;
    j_begin += parts * j_unit;
    j_end = min(j_begin + j_unit, n_j);
    return j_begin;
  };
  int skip_end = j_begin;   // this wavefront is done with the records below (FAR: one unit per part)
  for (int t0 = j_begin; t0 < j_end; t0 = next_tile(t0)) {
    const int cnt = min(JT, j_end - t0);
    bool need = true;
    if constexpr (FAR) {
      // the coarsest cell starting here, inside this part (or the array's
      // last, partial cell), that every lane sees from beyond q cell radii:
      // one expansion for all of it
      if (far_on) {
        need = t0 >= skip_end;
        const float* Mc = nullptr;
        int Cc = 0;
        size_t off = 0;
        for (int L = 0; L < kFarLevels; ++L) {
          const int C = kCellSize[L];
          if (need && !Mc && t0 % C == 0 && (t0 + C <= j_end || j_end == n_j)) {
            const float* M = cells + off + (size_t)(t0 / C) * kMomWords;
            const float yx = ((pi.x - M[48]) + li.x) - M[0], yy = ((pi.y - M[49]) + li.y) - M[1],
                        yz = ((pi.z - M[50]) + li.z) - M[2];
            const float y2 = __builtin_fmaf(yx, yx, __builtin_fmaf(yy, yy, yz * yz));
            if (M[4] == 0.f || __all(!real_i || y2 >= far_q2.q2[L] * M[3])) {
              Mc = M;
              Cc = C;
            }
          }
          off += (size_t)((n_j + C - 1) / C) * kMomWords;
        }
        if (Mc) {   // one expansion, whichever level accepted (none for an empty cell)
          if (Mc[4] != 0.f)
            add_far(Mc, ((pi.x - Mc[48]) + li.x) - Mc[0], ((pi.y - Mc[49]) + li.y) - Mc[1],
                    ((pi.z - Mc[50]) + li.z) - Mc[2]);
          for (int k = 0; k < 4; ++k) a[k].tile_end();
          skip_end = min(t0 + Cc, j_end);
          need = false;
        }
      }
      // the barrier that orders the previous tile's LDS reads before this
      // tile's staging also tells whether any wavefront needs the records
      if (!__syncthreads_or(need)) continue;
    } else {
      __syncthreads();
    }
    // stage: this wavefront's sub-tiles, each relative to its middle real
    // record, and each sub-tile's squared radius about that record.  A
    // padding record (at 1e30) as origin would collapse every real offset
    // to -1e30 and make its squared radius infinite; the tile test would
    // then pass for every wavefront and the real records would add nothing.
    // A sub-tile of padding only keeps its middle record.
    for (int q = threadIdx.x; q < JT; q += kGravBlock) {
      const int sub = q / kTile, sub0 = sub * kTile;
      float r2 = 0.f;
      if (sub0 < cnt) {
        const int nj = min(kTile, cnt - sub0), nr = max(0, min(nj, n_real - (t0 + sub0)));
        const F4 c = hi[t0 + sub0 + (nr > 0 ? nr : nj) / 2];
        if (q < cnt) {
          const F4 h = hi[t0 + q], l = lo[t0 + q];
          F4 d{(h.x - c.x) + l.x, (h.y - c.y) + l.y, (h.z - c.z) + l.z, h.w};
          r2 = __builtin_fmaf(d.x, d.x, __builtin_fmaf(d.y, d.y, d.z * d.z));
          if (expand) d.w = r2;   // the expanded body needs |d_j|^2, not m
          s_hi[q] = h;
          s_lo[q] = l;
          s_rel[q] = d;
        }
        for (int o = 32; o > 0; o >>= 1) r2 = fmaxf(r2, __shfl_xor(r2, o));
        if (lane == 0) {
          s_c[sub] = c;
          s_r2[sub] = r2;
        }
      }
    }
    if constexpr (FAR) {   // the tile's sub-tile records (t0 is a multiple of kTile)
      for (int q = threadIdx.x; q < kSub * kMomWords; q += kGravBlock) {
        const int sub = q / kMomWords, w = q % kMomWords;
        if (sub * kTile < cnt) s_mom[sub][w] = mom[(size_t)(t0 / kTile + sub) * kMomWords + w];
      }
    }
    __syncthreads();
    if (FAR && !need) continue;   // a cell covered this tile for this wavefront
    auto pair = [&](float rx, float ry, float rz, float mj) {
      const float d2 = __builtin_fmaf(rx, rx, __builtin_fmaf(ry, ry, __builtin_fmaf(rz, rz, eps2)));
      const float inv = rsq_spaced(d2);
      const float mi = mj * inv;
      const float s3 = mi * (inv * inv);
      a[0].fsub(rx, s3);
      a[1].fsub(ry, s3);
      a[2].fsub(rz, s3);
      a[3].sub(mi);
    };
    auto pair_unit = [&](float rx, float ry, float rz) {   // unit mass: 12 VALU + rsq
      const float d2 = __builtin_fmaf(rx, rx, __builtin_fmaf(ry, ry, __builtin_fmaf(rz, rz, eps2)));
      const float inv = rsq_spaced(d2);
      const float s3 = inv * (inv * inv);
      a[0].fsub(rx, s3);
      a[1].fsub(ry, s3);
      a[2].fsub(rz, s3);
      a[3].sub(inv);
    };
    for (int sub = 0; sub * kTile < cnt; ++sub) {
      const int j0 = sub * kTile, nj = min(kTile, cnt - j0);
      int jb = j0, je = j0 + nj;   // the records taken pair by pair
      const F4 c = s_c[sub];
      const float dx = (pi.x - c.x) + li.x, dy = (pi.y - c.y) + li.y, dz = (pi.z - c.z) + li.z;
      // tile form only if every lane of the wavefront has |d_i| >= 3 R_sub
      // (uniform per wavefront: no divergence); the squared test carries a
      // margin of 1.1 for the rounding of the squares
      if (FAR && far_on) {
        // multipole far field when every lane is q sub-tile radii from its
        // centre of mass (far_q2 = q^2; uniform per wavefront)
        const float* M = &s_mom[sub][0];
        const float yx = ((pi.x - M[48]) + li.x) - M[0], yy = ((pi.y - M[49]) + li.y) - M[1],
                    yz = ((pi.z - M[50]) + li.z) - M[2];
        const float y2 = __builtin_fmaf(yx, yx, __builtin_fmaf(yy, yy, yz * yz));
        if (M[4] == 0.f || __all(!real_i || y2 >= far_q2.q2[kFarLevels] * M[3])) {
          if (M[4] != 0.f) add_far(M, yx, yy, yz);
          if ((sub & 1) || j0 + kTile >= cnt)
            for (int k = 0; k < 4; ++k) a[k].tile_end();
          continue;
        }
        if (half_on && nj == kTile) {
          // each 32-record half the wavefront sees from beyond q of its radii
          // takes its expansion; the pairs run over the rest
          bool took[2];
          for (int h = 0; h < 2; ++h) {
            const float* H = halves + ((size_t)(t0 / kTile + sub) * 2 + h) * kMomWords;
            const float hx = ((pi.x - H[48]) + li.x) - H[0], hy = ((pi.y - H[49]) + li.y) - H[1],
                        hz = ((pi.z - H[50]) + li.z) - H[2];
            const float h2 = __builtin_fmaf(hx, hx, __builtin_fmaf(hy, hy, hz * hz));
            took[h] = H[4] == 0.f || __all(!real_i || h2 >= far_q2.q2[kFarLevels + 1] * H[3]);
            if (took[h] && H[4] != 0.f) add_far(H, hx, hy, hz);
          }
          if (took[0] && took[1]) {
            if ((sub & 1) || j0 + kTile >= cnt)
              for (int k = 0; k < 4; ++k) a[k].tile_end();
            continue;
          }
          if (took[0]) jb = j0 + kTile / 2;
          if (took[1]) je = j0 + kTile / 2;
        }
      }
      const bool far = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz)) >= 9.9f * s_r2[sub];
      const bool tile_form = !split_only && __all(far);
      auto pair_tile = [&](int j) {
        const F4 pj = s_rel[j];
        pair(dx - pj.x, dy - pj.y, dz - pj.z, pj.w);
      };
      auto pair_split = [&](int j) {
        const F4 pj = s_hi[j], lj = s_lo[j];
        pair((pi.x - pj.x) + (li.x - lj.x), (pi.y - pj.y) + (li.y - lj.y), (pi.z - pj.z) + (li.z - lj.z), pj.w);
      };
      auto unit_tile = [&](int j) {
        const F4 pj = s_rel[j];
        pair_unit(dx - pj.x, dy - pj.y, dz - pj.z);
      };
      auto unit_split = [&](int j) {
        const F4 pj = s_hi[j], lj = s_lo[j];
        pair_unit((pi.x - pj.x) + (li.x - lj.x), (pi.y - pj.y) + (li.y - lj.y), (pi.z - pj.z) + (li.z - lj.z));
      };
      // full sub-tiles (all of them when n_j is a multiple of kTile) have a
      // fixed trip count, unrolled so LDS reads are issued ahead of their use;
      // the branches are uniform per wavefront
      // the pairs of `len` consecutive staged records from `base`: a whole
      // sub-tile (len 64) or, in the far-field kernel, the half the
      // wavefront did not take by its expansion (len 32); fixed trip counts,
      // unrolled so LDS reads are issued ahead of their use
      auto run = [&](int base, auto len_c) {
        constexpr int len = decltype(len_c)::value;
        if (uniform) {
          if (tile_form && expand) {
            // expanded equal-mass body: r^2 + eps^2 = (|d_i|^2 + eps^2 + |d_j|^2)
            // - 2 d_i.d_j and sum_j s3 (d_j - d_i) = M - d_i S over the
            // records, 11 VALU + rsq per pair.  With |d_j| <= |d_i| / 3 the
            // expansion loses at most a factor (4/2)^2 of relative accuracy
            // in r^2 to cancellation, and M - d_i S none (|M| <= |d_i| S / 3).
            const float ci = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, __builtin_fmaf(dz, dz, eps2)));
            const float bx = -2.f * dx, by = -2.f * dy, bz = -2.f * dz;
            float sa = 0.f, mx = 0.f, my = 0.f, mz = 0.f;
#pragma unroll 16
            for (int j = 0; j < len; ++j) {
              const F4 pj = s_rel[base + j];
              const float d2 =
                  __builtin_fmaf(pj.x, bx, __builtin_fmaf(pj.y, by, __builtin_fmaf(pj.z, bz, ci + pj.w)));
              const float inv = rsq_spaced(d2);
              const float s3 = inv * (inv * inv);
              sa += s3;
              mx = __builtin_fmaf(pj.x, s3, mx);
              my = __builtin_fmaf(pj.y, s3, my);
              mz = __builtin_fmaf(pj.z, s3, mz);
              a[3].sub(inv);
            }
            a[0].part += __builtin_fmaf(-dx, sa, mx);
            a[1].part += __builtin_fmaf(-dy, sa, my);
            a[2].part += __builtin_fmaf(-dz, sa, mz);
          } else if (tile_form) {
#pragma unroll 16
            for (int j = 0; j < len; ++j) unit_tile(base + j);
          } else {
#pragma unroll 16
            for (int j = 0; j < len; ++j) unit_split(base + j);
          }
        } else if (tile_form) {
#pragma unroll 16
          for (int j = 0; j < len; ++j) pair_tile(base + j);
        } else {
#pragma unroll 16
          for (int j = 0; j < len; ++j) pair_split(base + j);
        }
      };
      // full sub-tiles (all of them when n_j is a multiple of kTile); the
      // branches are uniform per wavefront
      if (nj == kTile) {
        bool whole = true;
        if constexpr (FAR) {
          if (je - jb != kTile) {
            run(jb, std::integral_constant<int, kTile / 2>{});
            whole = false;
          }
        }
        if (whole) run(j0, std::integral_constant<int, kTile>{});
      } else {
        for (int j = j0; j < j0 + nj; ++j) {
          if (uniform) {
            if (tile_form) unit_tile(j);
            else unit_split(j);
          } else if (tile_form) {
            pair_tile(j);
          } else {
            pair_split(j);
          }
        }
      }
      // fold the FP32 partials every two sub-tiles (128 pairs) and at the end
      if ((sub & 1) || j0 + kTile >= cnt)
        for (int k = 0; k < 4; ++k) a[k].tile_end();
    }
  }
  if (i < n_i) {
    const size_t o = (size_t)part * n_i + i;
    part_hi[o] = {a[0].v.hi, a[1].v.hi, a[2].v.hi, a[3].v.hi};
    part_lo[o] = {a[0].v.lo, a[1].v.lo, a[2].v.lo, a[3].v.lo};
  }
}

// The mixed form with each pair of particles evaluated once for both: tiles of
// 512 meet each other once, as the tiles of pairs64.h do (order of tiles and
// rows, rotation of the reactions, slots).  A lane keeps two particles, so the
// rotation of a record's reactions, one move per component, serves two pairs; a
// wavefront's 128 particles choose the body per sub-tile as above:
//  expanded: s3 (d_j, 1) for i and s3 (d_i, 1) for j, 16 VALU and a rsq for the
//            two interactions in place of 22 and 2; the reaction on j is
//            sum s3 d_i - d_j sum s3, |d_i| >= 3 |d_j|;
//  split:    r once, 3 FMAs for each.
// A move between lanes takes 4.2 cycles of a SIMD and, like a transcendental
// operation, holds up the other wavefronts where vector operations directly
// follow it (3 multiplies and a move: 16.4 cycles against 4 x 2.1), so the moves
// of a step stand together between scalar instructions, and so do its two
// v_rsq_f32.
// A wavefront's reaction on a sub-tile is a plain FP32 sum of 4 sums of 32 terms
// (one sum of 128 had twice the rounding error of a particle's own sums of 64);
// the four wavefronts' are added and written, and
// k_gravity_mixed_pairs_sum adds a particle's own (hi, lo) sums and its
// reactions in two-sums, in a fixed order.
struct Reaction {
  float x = 0.f, y = 0.f, z = 0.f, w = 0.f, s = 0.f;
  // to the previous lane of the row of 16 (cyclic), with the record it is for
  __device__ __forceinline__ void turn() {
    asm("s_nop 1\n\t"
        "v_mov_b32_dpp %0, %0 row_ror:15 row_mask:0xf bank_mask:0xf\n\t"
        "v_mov_b32_dpp %1, %1 row_ror:15 row_mask:0xf bank_mask:0xf\n\t"
        "v_mov_b32_dpp %2, %2 row_ror:15 row_mask:0xf bank_mask:0xf\n\t"
        "v_mov_b32_dpp %3, %3 row_ror:15 row_mask:0xf bank_mask:0xf\n\t"
        "v_mov_b32_dpp %4, %4 row_ror:15 row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 0"
        : "+v"(x), "+v"(y), "+v"(z), "+v"(w), "+v"(s));
  }
  __device__ __forceinline__ void add(const Reaction& r) {
    x += r.x;
    y += r.y;
    z += r.z;
    w += r.w;
    s += r.s;
  }
  __device__ __forceinline__ void next_row(int from) {
    x = __shfl(x, from);
    y = __shfl(y, from);
    z = __shfl(z, from);
    w = __shfl(w, from);
    s = __shfl(s, from);
  }
};

// two rsq_spaced in one
__device__ __forceinline__ void rsq_spaced(float (&v)[2]) {
  float a, b;
  asm("s_setprio 1\n\tv_rsq_f32 %0, %2\n\tv_rsq_f32 %1, %3\n\ts_setprio 0" : "=&v"(a), "=v"(b) : "v"(v[0]), "v"(v[1]));
  v[0] = a;
  v[1] = b;
}

// 4 wavefronts per SIMD (120 VGPRs, nothing in scratch).  The two forms of r for
// unequal masses stand in loops of their own: with the choice inside one loop
// the kernel kept 596 bytes per lane in scratch, which this body reloaded in every
// step (65 536 particles of unequal masses, the pass alone: 8.4 ms, 1.58 with loops
// of their own; every ordered pair 2.24; equal masses 1.47 -> 1.42).
constexpr int kMixTile = 512, kMixHalf = 256;
__global__ __launch_bounds__(kMixHalf) __attribute__((amdgpu_waves_per_eu(4)))
void k_gravity_mixed_pairs(const F4* __restrict__ hi, const F4* __restrict__ lo, F4* __restrict__ own_hi,
                           F4* __restrict__ own_lo, F4* __restrict__ react, int n, int n_real, int tiles, int parts,
                           int d0, int d1, float eps2, const float* __restrict__ mass_range) {
  static_assert(kMixHalf == 4 * kTile, "a wavefront stages a sub-tile");
  const bool uniform = mass_range[0] == mass_range[1];
  // records relative to their sub-tile's origin: -2 d_j, |d_j|^2 (equal masses)
  // or d_j, m; twice in a row of 16, whose place 31 stays free and holds the
  // sub-tile's origin and squared radius (so 5 blocks share a CU's LDS)
  __shared__ F4 s_rel[kMixHalf / 16][32], s_hi[kMixHalf], s_lo[kMixHalf], s_acc[4][kMixHalf];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c16 = lane & 15, row = lane >> 4;
  const int tile = (int)blockIdx.x / parts, part = (int)blockIdx.x % parts;
  const int np = tiles * kMixTile;
  const auto load = [&](int i, F4& h, F4& l) {
    if (i < n) {
      h = hi[i];
      l = lo[i];
    } else {   // as the padding records: r^2 overflows and rsq returns 0
      h = {1e30f, 1e30f, 1e30f, 0.f};
      l = {0.f, 0.f, 0.f, 0.f};
    }
  };
  const int i0 = tile * kMixTile + 2 * kTile * wave + lane;
  F4 pi[2], li[2];
  GAcc<float, 1> a[2][4];
  for (int p = 0; p < 2; ++p) load(i0 + kTile * p, pi[p], li[p]);
  for (int d = d0 + part; d < d1; d += parts) {
    if (2 * d == tiles && tile >= d) break;   // the opposite tile's block has this pair of tiles
    const int other = tile + d < tiles ? tile + d : tile + d - tiles;
    for (int j_half = other * kMixTile; j_half < (other + 1) * kMixTile; j_half += kMixHalf) {
      __syncthreads();
      {
        const int sub0 = j_half + wave * kTile, nr = min(kTile, n_real - sub0);
        F4 h, l;
        load(sub0 + lane, h, l);
        if (nr > 0) {
          const F4 c = hi[sub0 + nr / 2];
          F4 dj{(h.x - c.x) + l.x, (h.y - c.y) + l.y, (h.z - c.z) + l.z, h.w};
          float r2 = __builtin_fmaf(dj.x, dj.x, __builtin_fmaf(dj.y, dj.y, dj.z * dj.z));
          if (uniform) dj = {-2.f * dj.x, -2.f * dj.y, -2.f * dj.z, r2};
          s_rel[tid >> 4][c16] = dj;
          if (c16 < 15) s_rel[tid >> 4][c16 + 16] = dj;
          s_hi[tid] = h;
          s_lo[tid] = l;
          for (int o = 32; o > 0; o >>= 1) r2 = fmaxf(r2, __shfl_xor(r2, o));
          if (lane == 0) s_rel[4 * wave][31] = {c.x, c.y, c.z, r2};
        } else if (lane == 0) {
          s_rel[4 * wave][31].w = -1.f;   // only padding
        }
      }
      __syncthreads();
      for (int sub = 0; sub < 4; ++sub) {
        Reaction R, total;   // of 16 records' steps, of all
        const F4 c = s_rel[4 * sub][31];
        if (!(c.w < 0.f)) {   // (a NaN place gives a NaN radius, and its NaN must reach the sums)
          float dx[2], dy[2], dz[2], di2[2];
          for (int p = 0; p < 2; ++p) {
            dx[p] = (pi[p].x - c.x) + li[p].x;
            dy[p] = (pi[p].y - c.y) + li[p].y;
            dz[p] = (pi[p].z - c.z) + li[p].z;
            di2[p] = __builtin_fmaf(dx[p], dx[p], __builtin_fmaf(dy[p], dy[p], dz[p] * dz[p]));
          }
          const bool tile_form = d > 0 && __all(fminf(di2[0], di2[1]) >= 9.9f * c.w);
          // body(group, step) over the 64 records, the reactions moving with them
          const auto sweep = [&](auto&& body) {
            for (int q = 0; q < 4; ++q) {
              const int grp = sub * 4 + ((row + q) & 3);
#pragma unroll
              for (int s = 0; s < 16; ++s) {
                body(grp, s);
                R.turn();
              }
              total.add(R);
              R = Reaction{};
              total.next_row((lane + 16) & 63);
            }
            R = total;
          };
          const auto split = [&](int j, float (&rx)[2], float (&ry)[2], float (&rz)[2], float (&inv)[2]) {
            const F4 pj = s_hi[j], lj = s_lo[j];
            for (int p = 0; p < 2; ++p) {
              rx[p] = (pi[p].x - pj.x) + (li[p].x - lj.x);
              ry[p] = (pi[p].y - pj.y) + (li[p].y - lj.y);
              rz[p] = (pi[p].z - pj.z) + (li[p].z - lj.z);
              inv[p] = __builtin_fmaf(rx[p], rx[p], __builtin_fmaf(ry[p], ry[p], __builtin_fmaf(rz[p], rz[p], eps2)));
            }
            rsq_spaced(inv);
            return pj.w;
          };
          if (d == 0) {   // all ordered pairs of the tile, without reactions
            for (int j = sub * kTile; j < sub * kTile + kTile; ++j) {
              float rx[2], ry[2], rz[2], inv[2];
              const float mj = split(j, rx, ry, rz, inv);
              for (int p = 0; p < 2; ++p) {
                const float m = uniform ? inv[p] : mj * inv[p], s3 = m * (inv[p] * inv[p]);
                a[p][0].fsub(rx[p], s3);
                a[p][1].fsub(ry[p], s3);
                a[p][2].fsub(rz[p], s3);
                a[p][3].sub(m);
              }
            }
          } else if (uniform && tile_form) {
            float sa[2] = {}, mx[2] = {}, my[2] = {}, mz[2] = {};   // of -2 d_j
            for (int p = 0; p < 2; ++p) di2[p] += eps2;
            sweep([&](int grp, int s) {
              const F4 pj = s_rel[grp][c16 + s];
              float inv[2];
              for (int p = 0; p < 2; ++p)
                inv[p] = __builtin_fmaf(pj.x, dx[p], __builtin_fmaf(pj.y, dy[p], __builtin_fmaf(pj.z, dz[p], di2[p] + pj.w)));
              rsq_spaced(inv);
              for (int p = 0; p < 2; ++p) {
                const float s3 = inv[p] * (inv[p] * inv[p]);
                sa[p] += s3;
                mx[p] = __builtin_fmaf(pj.x, s3, mx[p]);
                my[p] = __builtin_fmaf(pj.y, s3, my[p]);
                mz[p] = __builtin_fmaf(pj.z, s3, mz[p]);
                a[p][3].sub(inv[p]);
                R.s += s3;
                R.x = __builtin_fmaf(dx[p], s3, R.x);
                R.y = __builtin_fmaf(dy[p], s3, R.y);
                R.z = __builtin_fmaf(dz[p], s3, R.z);
                R.w -= inv[p];
              }
            });
            for (int p = 0; p < 2; ++p) {
              a[p][0].part += __builtin_fmaf(-dx[p], sa[p], -0.5f * mx[p]);
              a[p][1].part += __builtin_fmaf(-dy[p], sa[p], -0.5f * my[p]);
              a[p][2].part += __builtin_fmaf(-dz[p], sa[p], -0.5f * mz[p]);
            }
            const F4 dj = s_rel[sub * 4 + row][c16];
            R.x = __builtin_fmaf(0.5f * dj.x, R.s, R.x);
            R.y = __builtin_fmaf(0.5f * dj.y, R.s, R.y);
            R.z = __builtin_fmaf(0.5f * dj.z, R.s, R.z);
          } else if (uniform) {
            sweep([&](int grp, int s) {
              float rx[2], ry[2], rz[2], inv[2];
              split(grp * 16 + ((c16 + s) & 15), rx, ry, rz, inv);
              for (int p = 0; p < 2; ++p) {
                const float s3 = inv[p] * (inv[p] * inv[p]);
                a[p][0].fsub(rx[p], s3);
                a[p][1].fsub(ry[p], s3);
                a[p][2].fsub(rz[p], s3);
                a[p][3].sub(inv[p]);
                R.x = __builtin_fmaf(rx[p], s3, R.x);
                R.y = __builtin_fmaf(ry[p], s3, R.y);
                R.z = __builtin_fmaf(rz[p], s3, R.z);
                R.w -= inv[p];
              }
            });
          } else {
            const auto both = [&](const float (&rx)[2], const float (&ry)[2], const float (&rz)[2],
                                  const float (&inv)[2], float mj) {
              for (int p = 0; p < 2; ++p) {
                const float i2 = inv[p] * inv[p], wj = mj * inv[p], wi = pi[p].w * inv[p], sj = wj * i2, si = wi * i2;
                a[p][0].fsub(rx[p], sj);
                a[p][1].fsub(ry[p], sj);
                a[p][2].fsub(rz[p], sj);
                a[p][3].sub(wj);
                R.x = __builtin_fmaf(rx[p], si, R.x);
                R.y = __builtin_fmaf(ry[p], si, R.y);
                R.z = __builtin_fmaf(rz[p], si, R.z);
                R.w -= wi;
              }
            };
            if (tile_form)
              sweep([&](int grp, int s) {
                const F4 pj = s_rel[grp][c16 + s];
                float rx[2], ry[2], rz[2], inv[2];
                for (int p = 0; p < 2; ++p) {
                  rx[p] = dx[p] - pj.x;
                  ry[p] = dy[p] - pj.y;
                  rz[p] = dz[p] - pj.z;
                  inv[p] =
                      __builtin_fmaf(rx[p], rx[p], __builtin_fmaf(ry[p], ry[p], __builtin_fmaf(rz[p], rz[p], eps2)));
                }
                rsq_spaced(inv);
                both(rx, ry, rz, inv, pj.w);
              });
            else
              sweep([&](int grp, int s) {
                float rx[2], ry[2], rz[2], inv[2];
                const float mj = split(grp * 16 + ((c16 + s) & 15), rx, ry, rz, inv);
                both(rx, ry, rz, inv, mj);
              });
          }
        }
        if (sub & 1)
          for (int p = 0; p < 2; ++p)
            for (int k = 0; k < 4; ++k) a[p][k].tile_end();
        s_acc[wave][sub * kTile + lane] = {R.x, R.y, R.z, R.w};
      }
      if (d == 0) continue;
      __syncthreads();
      const F4 r0 = s_acc[0][tid], r1 = s_acc[1][tid], r2 = s_acc[2][tid], r3 = s_acc[3][tid];
      react[(size_t)(d - d0) * np + j_half + tid] = {(r0.x + r1.x) + (r2.x + r3.x), (r0.y + r1.y) + (r2.y + r3.y),
                                                     (r0.z + r1.z) + (r2.z + r3.z), (r0.w + r1.w) + (r2.w + r3.w)};
    }
  }
  for (int p = 0; p < 2; ++p) {
    const size_t o = (size_t)part * np + i0 + kTile * p;
    own_hi[o] = {a[p][0].v.hi, a[p][1].v.hi, a[p][2].v.hi, a[p][3].v.hi};
    own_lo[o] = {a[p][0].v.lo, a[p][1].v.lo, a[p][2].v.lo, a[p][3].v.lo};
  }
}

// The offsets [d0, d1) of a particle: own sums and reactions, added to what the
// offsets before left in acc (hi, then lo); the last call writes the result.
__global__ __launch_bounds__(kBlock) void k_gravity_mixed_pairs_sum(const F4* __restrict__ own_hi,
                                                                    const F4* __restrict__ own_lo,
                                                                    const F4* __restrict__ react,
                                                                    F4* __restrict__ acc, F4* __restrict__ out, int n,
                                                                    int tiles, int parts, int d0, int d1, int last,
                                                                    const float* __restrict__ mass_range) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const int np = tiles * kMixTile;
  DR a[4] = {{0.f, 0.f}, {0.f, 0.f}, {0.f, 0.f}, {0.f, 0.f}};
  const auto add = [&](const F4& v) {
    dr_add(a[0], v.x);
    dr_add(a[1], v.y);
    dr_add(a[2], v.z);
    dr_add(a[3], v.w);
  };
  if (d0 > 0) {
    add(acc[i]);
    add(acc[np + i]);
  }
  for (int p = 0; p < parts; ++p) {
    add(own_hi[(size_t)p * np + i]);
    add(own_lo[(size_t)p * np + i]);
  }
  int d_end = d1;
  if (2 * (d1 - 1) == tiles && i / kMixTile < tiles / 2) --d_end;   // met by the opposite tile's block
#pragma unroll 4
  for (int d = max(d0, 1); d < d_end; ++d) add(react[(size_t)(d - d0) * np + i]);
  if (!last) {
    acc[i] = {a[0].hi, a[1].hi, a[2].hi, a[3].hi};
    acc[np + i] = {a[0].lo, a[1].lo, a[2].lo, a[3].lo};
    return;
  }
  const float m = mass_range[0] == mass_range[1] ? mass_range[0] : 1.f;
  out[i] = {m * (a[0].hi + a[0].lo), m * (a[1].hi + a[1].lo), m * (a[2].hi + a[2].lo), m * (a[3].hi + a[3].lo)};
}

// sum of the `parts` compensated partials of each i, in part order, times
// the common mass when every mass is equal
__global__ __launch_bounds__(kBlock) void k_gravity_combine(const F4* __restrict__ part_hi,
                                                            const F4* __restrict__ part_lo, F4* __restrict__ out,
                                                            int n_i, const float* __restrict__ mass_range,
                                                            int flags, int parts) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n_i) return;
  const float m = (flags & 2) == 0 && mass_range[0] == mass_range[1] ? mass_range[0] : 1.f;
  DR a[4] = {{0.f, 0.f}, {0.f, 0.f}, {0.f, 0.f}, {0.f, 0.f}};
  for (int p = 0; p < parts; ++p) {
    const F4 h = part_hi[(size_t)p * n_i + i], l = part_lo[(size_t)p * n_i + i];
    dr_add(a[0], h.x);
    dr_add(a[0], l.x);
    dr_add(a[1], h.y);
    dr_add(a[1], l.y);
    dr_add(a[2], h.z);
    dr_add(a[2], l.z);
    dr_add(a[3], h.w);
    dr_add(a[3], l.w);
  }
  out[i] = {m * (a[0].hi + a[0].lo), m * (a[1].hi + a[1].lo), m * (a[2].hi + a[2].lo), m * (a[3].hi + a[3].lo)};
}

// {min, max} of the masses of the real particles: per-block partials, then
// one block (fixed tree order, no atomics)
__global__ __launch_bounds__(kBlock) void k_mass_range_partials(const F4* __restrict__ hi, int n,
                                                                float* __restrict__ partial) {
  __shared__ float smin[kBlock], smax[kBlock];
  const int i = blockIdx.x * kBlock + threadIdx.x;
  const float m = i < n ? hi[i].w : hi[0].w;
  smin[threadIdx.x] = m;
  smax[threadIdx.x] = m;
  __syncthreads();
  for (int k = kBlock / 2; k > 0; k >>= 1) {
    if ((int)threadIdx.x < k) {
      smin[threadIdx.x] = fminf(smin[threadIdx.x], smin[threadIdx.x + k]);
      smax[threadIdx.x] = fmaxf(smax[threadIdx.x], smax[threadIdx.x + k]);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    partial[2 * blockIdx.x] = smin[0];
    partial[2 * blockIdx.x + 1] = smax[0];
  }
}
__global__ __launch_bounds__(kBlock) void k_mass_range_final(const float* __restrict__ partial, int nb,
                                                             float* __restrict__ out) {
  __shared__ float smin[kBlock], smax[kBlock];
  float lo = partial[0], hi = partial[1];
  for (int b = threadIdx.x; b < nb; b += kBlock) {
    lo = fminf(lo, partial[2 * b]);
    hi = fmaxf(hi, partial[2 * b + 1]);
  }
  smin[threadIdx.x] = lo;
  smax[threadIdx.x] = hi;
  __syncthreads();
  for (int k = kBlock / 2; k > 0; k >>= 1) {
    if ((int)threadIdx.x < k) {
      smin[threadIdx.x] = fminf(smin[threadIdx.x], smin[threadIdx.x + k]);
      smax[threadIdx.x] = fmaxf(smax[threadIdx.x], smax[threadIdx.x + k]);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    out[0] = smin[0];
    out[1] = smax[0];
  }
}

// mixed form, spline softening: same accumulation and split positions
__global__ __launch_bounds__(kGravBlock) void k_gravity_mixed_spline(const F4* __restrict__ hi,
                                                                      const F4* __restrict__ lo,
                                                                      const F4* __restrict__ gvel,
                                                                      F4* __restrict__ out, int n_i, int n_j) {
  __shared__ F4 s_hi[kJTile], s_lo[kJTile];
  __shared__ float s_r2[kJTile];
  const int i = blockIdx.x * kGravBlock + threadIdx.x;
  const int ii = i < n_i ? i : n_i - 1;
  const F4 pi = hi[ii], li = lo[ii];
  const float ri2 = gvel[ii].w;
  GAcc<float, 1> a[4];
  for (int t0 = 0; t0 < n_j; t0 += kJTile) {
    const int cnt = stage_tile(s_hi, hi, t0, n_j);
    for (int q = threadIdx.x; q < cnt; q += kGravBlock) {
      s_lo[q] = lo[t0 + q];
      s_r2[q] = gvel[t0 + q].w;
    }
    __syncthreads();
    for (int j0 = 0; j0 < cnt; j0 += kTile) {
      const int j1 = min(j0 + kTile, cnt);
      for (int j = j0; j < j1; ++j) {
        const F4 pj = s_hi[j], lj = s_lo[j];
        const float rx = (pi.x - pj.x) + (li.x - lj.x);
        const float ry = (pi.y - pj.y) + (li.y - lj.y);
        const float rz = (pi.z - pj.z) + (li.z - lj.z);
        pair_spline<float, false>(a, rx, ry, rz, ri2, pj.w, s_r2[j]);
      }
      for (int k = 0; k < 4; ++k) a[k].tile_end();
    }
  }
  if (i < n_i) out[i] = {a[0].get(), a[1].get(), a[2].get(), a[3].get()};
}

// ---------------------------------------------------------------------------
// FP64 form, Plummer softening.  The pair body in fused multiply-adds (the
// FP64 form has no bit contract with the reference's FP32 arithmetic):
// 3 sub, 3 FMA for s^2 = r^2 + eps^2, v_rsq_f64 refined by one third-order
// step (y0 (1 + e (1/2 + 3/8 e)), e = 1 - s^2 y0^2: 5 operations, its remainder
// 5/16 e^3 below one rounding), 3 for m/s^3, 3 FMA into the acceleration and one
// into the potential.  Here every ordered pair is evaluated: below kPairs64MinN
// and above kPairs64MaxN particles, or with other j than i (pairs64.h between).
// With few i-blocks (N below 2^19) the j-range is split
// into parts, one block per (i-block, part), so that the GPU holds enough
// wavefronts to hide the FP64 latencies; the parts' sums are added in part
// order (deterministic).
constexpr int kG64Tile = kGravBlock;
__global__ __launch_bounds__(kGravBlock) void k_gravity64_plummer(const D4* __restrict__ gpos, D4* __restrict__ out,
                                                                   int n_i, int n_j, int parts, int chunk,
                                                                   double eps2) {
  __shared__ D4 s_pos[kG64Tile];
  const int part = (int)blockIdx.x % parts, ib = (int)blockIdx.x / parts;
  const int i = ib * kGravBlock + threadIdx.x;
  const D4 pi = gpos[i < n_i ? i : n_i - 1];
  const int j_begin = part * chunk, j_end = min(n_j, j_begin + chunk);
  double ax = 0.0, ay = 0.0, az = 0.0, ph = 0.0;
  for (int t0 = j_begin; t0 < j_end; t0 += kG64Tile) {
    const int cnt = min(kG64Tile, j_end - t0);
    __syncthreads();
    if ((int)threadIdx.x < cnt) s_pos[threadIdx.x] = gpos[t0 + threadIdx.x];
    __syncthreads();
    for (int j = 0; j < cnt; ++j) {
      const D4 pj = s_pos[j];
      const double rx = pi.x - pj.x, ry = pi.y - pj.y, rz = pi.z - pj.z;
      const double d2 = __builtin_fma(rx, rx, __builtin_fma(ry, ry, __builtin_fma(rz, rz, eps2)));
      const double y0 = __builtin_amdgcn_rsq(d2);
      const double e = __builtin_fma(-(d2 * y0), y0, 1.0);
      const double y = __builtin_fma(__builtin_fma(e, 0.375, 0.5), y0 * e, y0);
      const double my = pj.w * y;
      const double s3 = my * (y * y);
      ax = __builtin_fma(-rx, s3, ax);
      ay = __builtin_fma(-ry, s3, ay);
      az = __builtin_fma(-rz, s3, az);
      ph -= my;
    }
  }
  if (i < n_i) out[(size_t)part * n_i + i] = {ax, ay, az, ph};
}

// the parts' sums, in part order
__global__ __launch_bounds__(kBlock) void k_gravity64_combine(const D4* __restrict__ part, D4* __restrict__ out,
                                                               int n_i, int parts) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n_i) return;
  D4 a = part[i];
  for (int p = 1; p < parts; ++p) {
    const D4 b = part[(size_t)p * n_i + i];
    a = {a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w};
  }
  out[i] = a;
}

static int gpu_cus() {
  int dev = 0, cus = 0;
  CS_HIP(hipGetDevice(&dev));
  CS_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  return cus;
}

// Parts for the passes of the FP64 form: of 2 .. 8 (1 from 2^19 particles on)
// the count whose blocks fill the CUs most evenly, the larger of equals.
// Where every block is resident at once (pairs: 4 blocks a CU, so tiles * parts up
// to 1 024 on 256 CUs) and takes the same time, a pass lasts as long as its fullest
// CU; with more blocks it is a guide only, and matters less.  Pairs taken once,
// gravity alone, 8 / 5 parts, ms: 50 021 particles (98 tiles on 256 CUs) 1.59 / 1.34,
// 65 536 (128): 2.06 / 2.36, 100 003 (196): 5.42 / 5.09, 131 072 (256): 7.9 / 8.2.
int gravity64_parts(int n_i) {
  const bool pairs = pairs64_fits(n_i);
  const int blocks = pairs ? pairs64_tiles(n_i) : ceil_div(n_i, kGravBlock);
  if (blocks >= 2048) return 1;
  const int cus = gpu_cus();
  int best = 8;
  for (int p = 7; p >= 2 && (pairs || (long)p * blocks >= 4l * cus); --p)   // fewer: too few wavefronts per SIMD
    // fullest CU's blocks per unit of work: ceil(p blocks / cus) / p
    if ((long)ceil_div((long)p * blocks, cus) * best < (long)ceil_div((long)best * blocks, cus) * p) best = p;
  return best;
}

// the pair body above, for both particles
struct GravityPairs {
  static constexpr int kRec = 2, kAcc = 4;
  const D4* gpos;
  double eps2;
  __device__ __forceinline__ D4 load(int i, int n) const {
    if (i < n) return gpos[i];
    return {1e30, 1e30, 1e30, 0.0};   // no mass: its partners get exactly nothing
  }
  template <class S>
  __device__ __forceinline__ void stage(S&& put, int j, int n) const {
    const D4 p = load(j, n);
    put(0, make_double2(p.x, p.y));
    put(1, make_double2(p.z, p.w));
  }
  template <bool REACT>
  __device__ __forceinline__ void pair(const D4& pi, const double2 (&r)[2], double (&g)[4], double (&a)[4]) const {
    const double rx = pi.x - r[0].x, ry = pi.y - r[0].y, rz = pi.z - r[1].x;
    const double d2 = __builtin_fma(rx, rx, __builtin_fma(ry, ry, __builtin_fma(rz, rz, eps2)));
    const double y0 = __builtin_amdgcn_rsq(d2);
    const double e = __builtin_fma(-(d2 * y0), y0, 1.0);
    const double y = __builtin_fma(__builtin_fma(e, 0.375, 0.5), y0 * e, y0);
    const double y3 = y * (y * y), mj = r[1].y * y3;
    g[0] = __builtin_fma(-rx, mj, g[0]);
    g[1] = __builtin_fma(-ry, mj, g[1]);
    g[2] = __builtin_fma(-rz, mj, g[2]);
    g[3] = __builtin_fma(-r[1].y, y, g[3]);
    if constexpr (REACT) {
      const double mi = pi.w * y3;
      a[0] = __builtin_fma(rx, mi, a[0]);
      a[1] = __builtin_fma(ry, mi, a[1]);
      a[2] = __builtin_fma(rz, mi, a[2]);
      a[3] = __builtin_fma(-pi.w, y, a[3]);
    }
  }
};

__global__ __launch_bounds__(kBlock) void k_gravity64_pairs_sum(const double* __restrict__ own,
                                                                const double* __restrict__ react,
                                                                double* __restrict__ out, int n, int tiles,
                                                                int parts) {
  const int i = blockIdx.x * kBlock + threadIdx.x, k = blockIdx.y;
  if (i < n) out[4 * (size_t)i + k] = pairs64_sum<4>(own, react, i, k, tiles, parts);
}

void launch_gravity64_plummer(const D4* gpos, D4* out, D4* part, int n_i, int n_j, double eps, hipStream_t s,
                              int parts) {
  if (parts <= 0) parts = gravity64_parts(n_i);
  if (parts > 8) throw std::invalid_argument("gravity: at most 8 j-parts");
  if (n_i == n_j && pairs64_fits(n_i)) {
    double* ws = (double*)part;
    launch_pairs64(GravityPairs{gpos, eps * eps}, n_i, parts, ws, s);
    hipLaunchKernelGGL(k_gravity64_pairs_sum, dim3(ceil_div(n_i, kBlock), 4), dim3(kBlock), 0, s, ws,
                       ws + pairs64_own(n_i, parts), (double*)out, n_i, pairs64_tiles(n_i), pairs64_parts(n_i, parts));
    CS_CHECK_LAUNCH();
    return;
  }
  const int chunk = ceil_div(ceil_div(n_j, parts), kG64Tile) * kG64Tile;
  hipLaunchKernelGGL(k_gravity64_plummer, dim3(ceil_div(n_i, kGravBlock) * parts), dim3(kGravBlock), 0, s, gpos,
                     parts > 1 ? part : out, n_i, n_j, parts, chunk, eps * eps);
  CS_CHECK_LAUNCH();
  if (parts > 1) {
    hipLaunchKernelGGL(k_gravity64_combine, dim3(ceil_div(n_i, kBlock)), dim3(kBlock), 0, s, part, out, n_i, parts);
    CS_CHECK_LAUNCH();
  }
}

static bool gravity_by_chains(int n_i, int soft, int sums) {
  if (sums >= 0) return sums != 0;
  return n_i <= (soft == 1 ? kChainsMaxN : kChainsMaxNSpline);
}

template <class T>
void launch_gravity(const V4<T>* gpos, const V4<T>* gvel, V4<T>* out, int n_i, int n_j, int soft, T eps,
                    int exact, hipStream_t s, int sums) {
  const dim3 grid(ceil_div(n_i, kGravBlock)), block(kGravBlock);
  const T eps2 = eps * eps;
  if constexpr (sizeof(T) == 4) {
    const bool chains = gravity_by_chains(n_i, soft, sums);
    const auto pick = [&](auto soft_c, auto exact_c) {
      constexpr int S = decltype(soft_c)::value;
      constexpr bool E = decltype(exact_c)::value;
      if (chains)
        hipLaunchKernelGGL((k_gravity_chains<S, E>), dim3(ceil_div(n_i, kChainParticles)), dim3(kChainBlock), 0, s,
                           gpos, gvel, out, n_i, n_j, eps2);
      else if (S == 0 || n_i >= kFastLaneMinN)
        hipLaunchKernelGGL((k_gravity_lane_fast<S, E>), grid, block, 0, s, gpos, gvel, out, n_i, n_j, eps2);
      else
        hipLaunchKernelGGL(k_gravity_lane<E>, grid, block, 0, s, gpos, out, n_i, n_j, eps2);
    };
    using Spline = std::integral_constant<int, 0>;
    using Plummer = std::integral_constant<int, 1>;
    if (soft == 1 && exact) pick(Plummer{}, std::true_type{});
    else if (soft == 1) pick(Plummer{}, std::false_type{});
    else if (exact) pick(Spline{}, std::true_type{});
    else pick(Spline{}, std::false_type{});
  } else {
    if (soft == 0) hipLaunchKernelGGL((k_gravity<double, 0, 2, true>), grid, block, 0, s, gpos, gvel, out, n_i, n_j, eps2);
    else hipLaunchKernelGGL((k_gravity<double, 1, 2, true>), grid, block, 0, s, gpos, gvel, out, n_i, n_j, eps2);
  }
  CS_CHECK_LAUNCH();
}

int mixed_pairs_chunk(int n) {
  const int tiles = ceil_div(n, kMixTile);
  const size_t slot = sizeof(F4) * kMixTile * (size_t)tiles;
  return (int)std::min<size_t>(tiles / 2 + 1, std::max<size_t>(1, ((size_t)2 << 30) / slot));
}
size_t mixed_part_words(int n, bool pairs) {
  const size_t items = 2 * kGravMixedParts * (size_t)n;
  if (!pairs || !mixed_pairs_fit(n)) return items;
  const size_t np = (size_t)ceil_div(n, kMixTile) * kMixTile;
  return std::max(items, (2 * kGravMixedParts + 2 + mixed_pairs_chunk(n)) * np);
}

void launch_gravity_mixed(const F4* hi, const F4* lo, const F4* gvel, F4* out, F4* part, float* mass_range,
                          float* moments, float far_ratio, float far_grade, int n_i, int n_j, int n_real,
                          int soft, float eps, int split_only, hipStream_t s, int parts) {
  const dim3 grid(ceil_div(n_i, kGravBlock)), block(kGravBlock);
  if (soft == 0) {
    hipLaunchKernelGGL(k_gravity_mixed_spline, grid, block, 0, s, hi, lo, gvel, out, n_i, n_j);
  } else {
    // mass_range: 2 floats of result followed by 2 per block of n_real
    const int nb = ceil_div(n_real, kBlock);
    hipLaunchKernelGGL(k_mass_range_partials, dim3(nb), dim3(kBlock), 0, s, hi, n_real, mass_range + 2);
    CS_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_mass_range_final, dim3(1), dim3(kBlock), 0, s, mass_range + 2, nb, mass_range);
    CS_CHECK_LAUNCH();
    if (n_i == n_j && split_only == 0 && mixed_pairs_fit(n_j)) {
      if (parts <= 0) parts = kGravMixedParts;
      if (parts > kGravMixedParts) throw std::invalid_argument("gravity: at most 8 j-parts");
      const int tiles = ceil_div(n_j, kMixTile), np = tiles * kMixTile, d_end = tiles / 2 + 1,
                chunk = mixed_pairs_chunk(n_j);
      F4 *own_hi = part, *own_lo = own_hi + (size_t)parts * np, *acc = own_lo + (size_t)parts * np,
         *react = acc + 2 * (size_t)np;
      for (int d0 = 0; d0 < d_end; d0 += chunk) {
        const int d1 = min(d_end, d0 + chunk);
        hipLaunchKernelGGL(k_gravity_mixed_pairs, dim3(tiles * parts), dim3(kMixHalf), 0, s, hi, lo, own_hi, own_lo,
                           react, n_j, n_real, tiles, parts, d0, d1, eps * eps, mass_range);
        CS_CHECK_LAUNCH();
        hipLaunchKernelGGL(k_gravity_mixed_pairs_sum, dim3(ceil_div(n_i, kBlock)), dim3(kBlock), 0, s, own_hi, own_lo,
                           react, acc, out, n_i, tiles, parts, d0, d1, (int)(d1 == d_end), mass_range);
        CS_CHECK_LAUNCH();
      }
      return;
    }
    const bool far = (split_only & 16) && moments;
    if (parts <= 0 || far) parts = kGravMixedParts;
    if (parts > kGravMixedParts) throw std::invalid_argument("gravity: at most 8 j-parts");
    int unit = ceil_div(ceil_div(n_j, parts), kTile) * kTile;
    if (!far && unit >= 2 * kJTileMixed) unit = kJTileMixed;
    F4* part_hi = part;
    F4* part_lo = part + (size_t)parts * n_i;
    float* cells = nullptr;
    float* halves = nullptr;
    if ((split_only & 16) && moments) {
      const int n_sub = ceil_div(n_j, kTile);
      hipLaunchKernelGGL(k_subtile_moments, dim3(ceil_div(n_sub, kGravBlock / 64)), block, 0, s, hi, lo, moments,
                         n_j, n_real, n_sub, kTile, split_only, mass_range);
      CS_CHECK_LAUNCH();
      // the cell levels follow the sub-tile records in the same buffer
      cells = moments + (size_t)n_sub * kMomWords;
      size_t off = 0;
      for (int L = 0; L < kFarLevels; ++L) {
        const int n_cells = ceil_div(n_j, kCellSize[L]);
        hipLaunchKernelGGL(k_cell_moments, dim3(n_cells), block, 0, s, hi, lo, cells + off, n_j, n_real,
                           kCellSize[L], split_only, mass_range);
        CS_CHECK_LAUNCH();
        off += (size_t)n_cells * kMomWords;
      }
      if (split_only & 64) {   // the 32-record halves of the sub-tiles, after the cells
        halves = cells + off;
        const int n_half = 2 * n_sub;
        hipLaunchKernelGGL(k_subtile_moments, dim3(ceil_div(n_half, kGravBlock / 64)), block, 0, s, hi, lo, halves,
                           n_j, n_real, n_half, kTile / 2, split_only, mass_range);
        CS_CHECK_LAUNCH();
      }
    }
    // ratio q at the coarsest level, graded by (C / C_coarsest)^far_grade:
    // an order-4 group's truncation error goes as M R^5 / y^7, and with
    // equal masses M grows with the record count C while R grows as
    // C^(1/3), so a grade near 1/15 asks every level for the same bound
    FarRatios fq{};
    for (int L = 0; L <= kFarLevels + 1; ++L) {
      const float c = (float)(L < kFarLevels ? kCellSize[L] : (L == kFarLevels ? kTile : kTile / 2)) /
                      (float)kCellSize[0];
      const float q = far_ratio * powf(c, far_grade);
      fq.q2[L] = q * q;
    }
    const int n_items = ceil_div(n_i, kGravBlock) * parts;
    if (far)
      hipLaunchKernelGGL((k_gravity_mixed_plummer<kJTileMixed, true>), dim3(n_items), block, 0, s, hi, lo, part_hi,
                         part_lo, n_i, n_j, unit, eps * eps, split_only, mass_range, moments, fq, cells, halves,
                         n_real, parts);
    else
      hipLaunchKernelGGL((k_gravity_mixed_plummer<kJTileMixed, false>), dim3(n_items), block, 0, s, hi, lo, part_hi,
                         part_lo, n_i, n_j, unit, eps * eps, split_only, mass_range, nullptr, fq, nullptr, nullptr,
                         n_real, parts);
    CS_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_gravity_combine, dim3(ceil_div(n_i, kBlock)), dim3(kBlock), 0, s, part_hi, part_lo, out,
                       n_i, mass_range, split_only, parts);
  }
  CS_CHECK_LAUNCH();
}

template void launch_gravity<float>(const F4*, const F4*, F4*, int, int, int, float, int, hipStream_t, int);
template void launch_gravity<double>(const D4*, const D4*, D4*, int, int, int, double, int, hipStream_t, int);

}  // namespace cudasph
