// SPH passes on the GPU: density, EOS and hydro accelerations (the tree walks
// are in walks.hip).
//
// Lanes take particles in the order of the hash array (thread t ->
// bodies_hash[t].value, as in the reference).  The engine fills it with
// kd-tree heap order, or with memory order when the particles are already in
// Peano-Hilbert order; either way a wavefront holds spatially adjacent
// particles and their neighbour gathers hit the same cache lines.  Plain and
// FP64 forms: 16 lanes per particle, its sums in list order, so in the plain
// form each particle's result is the same bit pattern as the CPU
// restatement's.  The mixed form has its own density and hydro kernels (FP32
// pair arithmetic, compensated sums).
#include "kernels.h"
#include "sph_math.h"

namespace cudasph {

// ---------------------------------------------------------------------------
// compensated (two-sum) accumulator for the mixed form
struct KSum {
  float s = 0.f, c = 0.f;   // the compensated value is s - c
  __device__ __forceinline__ void add(float x) {
    const float y = x - c;
    const float t = s + y;
    c = (t - s) - y;
    s = t;
  }
  __device__ __forceinline__ float get() const { return s; }
  __device__ __forceinline__ float value() const { return s - c; }
};

// lanes per particle in the cooperative mixed-form kernels
constexpr int kGroup = 8;

// sum of the group's KSums into every lane of the group: a butterfly over
// the kGroup lanes, each step an exact two-sum of the partial values with the
// rounding error carried into the compensation
__device__ __forceinline__ void group_sum(KSum& a) {
  for (int o = kGroup / 2; o > 0; o >>= 1) {
    const float s2 = __shfl_xor(a.s, o, kGroup), c2 = __shfl_xor(a.c, o, kGroup);
    const float t = a.s + s2;
    const float bp = t - a.s;
    const float err = (a.s - (t - bp)) + (s2 - bp);   // a.s + s2 = t + err exactly
    a.c = (a.c + c2) - err;
    a.s = t;
  }
}
__device__ __forceinline__ float group_max(float v) {
  for (int o = kGroup / 2; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, kGroup));
  return v;
}
// density, grad-h terms, div v and |curl v| (dev_density_loop.cu:29-111);
// plain and FP64 forms.  A group of 16 lanes per particle, its sums in list
// order (OrderedSums).  One lane per particle waited for one neighbour's records
// after another.  Density / hydro, one lane -> this, us: plain 1 000 particles 110 ->
// 13 / 141 -> 16, 16 384: 80 -> 16 / 97 -> 20, 131 072: 90 -> 63 / 241 -> 97, 600 000:
// 649 -> 280 / 1278 -> 443; FP64 65 536: 76 -> 48 / 116 -> 68.
template <class T>
__global__ __launch_bounds__(kBlock) void k_density(const V4<T>* __restrict__ pos, const V4<T>* __restrict__ vel,
                                                     V4<T>* __restrict__ hydro,
                                                     V4<T>* __restrict__ dots, const KV* __restrict__ hash,
                                                     const int* __restrict__ offset, const int* __restrict__ count,
                                                     const int* __restrict__ list, int n_dev) {
  chain_priority();
  using Sums = OrderedSums<T, 8>;   // rho, omega, psi, -den, div v, curl v
  __shared__ __align__(16) T s_rows[kBlock / 16][Sums::kRow];
  const int t = (xcd_block(blockIdx.x, gridDim.x) * kBlock + (int)threadIdx.x) / 16, l = threadIdx.x % 16;
  if (t >= n_dev) return;   // whole groups leave together
  const int i = (int)hash[t].value;
  const V4<T> bp = pos[i], bv = vel[i];
  Sums sums{T(0), s_rows[threadIdx.x / 16], l};
  const int off = offset[i], n = count[i];
  for (int k = l; k - l < n; k += 16) {
    T a[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) a[c] = Sums::none();
    if (k < n) {
      const int j = list[off + k];
      const V4<T> pj = pos[j], vj = vel[j];
      const T dx = bp.x - pj.x, dy = bp.y - pj.y, dz = bp.z - pj.z;
      const T u = T(2) * dsqrt(dx * dx + dy * dy + dz * dz) / bp.w;
      a[0] = vj.w * kern_w<T>(u);
      a[1] = vj.w * kern_dwdh<T>(u);
      a[2] = vj.w * kern_dphidh<T>(u);
      a[3] = -kern_digdh<T>(u);
      const T dvx = bv.x - vj.x, dvy = bv.y - vj.y, dvz = bv.z - vj.z;
      const T mdw = bv.w * kern_dw<T>(u);
      a[4] = mdw * (dx * dvx + dy * dvy + dz * dvz);
      a[5] = mdw * (dy * dvz - dz * dvy);
      a[6] = mdw * (dz * dvx - dx * dvz);
      a[7] = mdw * (dx * dvy - dy * dvx);
    }
    sums.add(a);
  }
  const T rho = sums.get(0), om = sums.get(1), psi = sums.get(2), d = sums.get(3), divv = sums.get(4),
          x = sums.get(5), y = sums.get(6), z = sums.get(7);
  if (l != 0) return;
  const T h = T(0.5 * (double)bp.w);
  const T h3 = h * h * h, h5 = h * h * h * h * h;
  T o, p;
  if (d != T(0)) {
    o = T((double)om * (1.0 / (double)h3 / (double)d));
    p = T((double)psi * (1.0 / (double)h / (double)d));
  } else {
    o = p = T(0);
  }
  const T r = T((double)rho * (1.0 / (double)h3));
  const T dv = T((double)divv * (1.0 / (double)r / (double)h5));
  const T curl = dsqrt(x * x + y * y + z * z) / r / h5;
  hydro[i].x = r;
  dots[i] = {dv, curl, o, p};
}

// dev_compute_pressure.cu:99-111 (every record, no hash, as the reference)
template <class T>
__global__ __launch_bounds__(kBlock) void k_eos(V4<T>* __restrict__ hydro, int n_dev, EosConst c) {
  chain_priority();
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n_dev) return;
  hydro[i].y = eos_record<T>(hydro[i], c);
}

// mixed form: P from the FP64 internal energy with the FP64 Newton root, and
// the per-particle factors the viscosity needs (dev_art_visc.cu:12-26), once
// per particle instead of once per pair: hydro2 = {v_sig (hydro pass),
// sound speed c = sqrt(5/3 P/rho), P/rho^2, Balsara |div v| / (|div v| +
// |curl v| + 1e-4 c/h)}
__global__ __launch_bounds__(kBlock) void k_eos_mixed(F4* __restrict__ hydro, const double* __restrict__ u64,
                                                       const F4* __restrict__ pos, const F4* __restrict__ dots,
                                                       F4* __restrict__ hydro2, int n, EosConst c) {
  chain_priority();
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const F4 hd = hydro[i];
  const double P = eos_pressure_fp64((double)hd.x, u64[i], (double)hd.w, c);
  hydro[i].y = (float)P;
  const double rho = hd.x;
  const double cs = sqrt(5.0 / 3.0 * P / rho);
  const F4 dd = dots[i];
  const double ad = fabs((double)dd.x);
  const double bal = ad / ((ad + (double)dd.y) + 0.0001 * cs / (0.5 * (double)pos[i].w));
  F4 h2 = hydro2[i];
  h2.y = (float)cs;
  h2.z = (float)(P / (rho * rho));
  h2.w = (float)bal;
  hydro2[i] = h2;
}

// hydro accelerations, du/dt and max signal speed (dev_hydro_dots.cu:25-113);
// writes the per-pair reaction coefficient m_i*acc to ngb_acc[k]; plain and
// FP64 forms, 16 lanes per particle as k_density
template <class T>
__global__ __launch_bounds__(kBlock) void k_hydro(const V4<T>* __restrict__ pos, const V4<T>* __restrict__ vel,
                                                   const V4<T>* __restrict__ hydro,
                                                   const V4<T>* __restrict__ dots, V4<T>* __restrict__ bdots,
                                                   V4<T>* __restrict__ hydro2, T* __restrict__ ngb_acc,
                                                   const KV* __restrict__ hash, const int* __restrict__ offset,
                                                   const int* __restrict__ count, const int* __restrict__ list,
                                                   int n_dev, T alpha, T beta) {
  chain_priority();
  using Sums = OrderedSums<T, 4>;   // acceleration, du/dt
  __shared__ __align__(16) T s_rows[kBlock / 16][Sums::kRow];
  const int t = (xcd_block(blockIdx.x, gridDim.x) * kBlock + (int)threadIdx.x) / 16, l = threadIdx.x % 16;
  if (t >= n_dev) return;   // whole groups leave together
  const int i = (int)hash[t].value;
  const V4<T> bp = pos[i], bv = vel[i], hd = hydro[i], dd = dots[i];
  const T prho2 = hd.y / (hd.x * hd.x);
  const double hw = 0.5 * (double)bp.w;
  // POW5(0.5*range) and POW2(0.5*range) expand left to right in the reference
  const double pow5 = hw * 0.5 * (double)bp.w * 0.5 * (double)bp.w * 0.5 * (double)bp.w * 0.5 * (double)bp.w;
  const double pow2 = hw * 0.5 * (double)bp.w;
  Sums sums{T(0), s_rows[threadIdx.x / 16], l};
  T vsig = T(0);
  const int off = offset[i], n = count[i];
  for (int k = l; k - l < n; k += 16) {
    T a[4] = {Sums::none(), Sums::none(), Sums::none(), Sums::none()};
    if (k < n) {
      const int j = list[off + k];
      const V4<T> pj = pos[j], vj = vel[j], hj = hydro[j], dj = dots[j];
      const T dx = bp.x - pj.x, dy = bp.y - pj.y, dz = bp.z - pj.z;
      const T dvx = bv.x - vj.x, dvy = bv.y - vj.y, dvz = bv.z - vj.z;
      const T ds = dsqrt(dx * dx + dy * dy + dz * dz);
      const T u = T((double)ds / hw);
      const T drdv = dx * dvx + dy * dvy + dz * dvz;
      const Visc<T> av = art_visc<T>(bp.w, pj.w, ds, drdv, hd, dd, hj, dj, alpha, beta);
      vsig = dmax(vsig, av.vsig);
      const double w1 = (double)kern_dw<T>(u);
      const T g = kern_dig<T>(u);
      const double pv = (double)prho2 + 0.5 * (double)av.pi;
      T acc = T(pv * w1 / pow5);
      acc = T((double)acc - ((double)(prho2 * dd.z) + 0.5 * (double)dd.w) / (double)vj.w * (double)g / pow2);
      a[0] = -(vj.w * acc * dx);
      a[1] = -(vj.w * acc * dy);
      a[2] = -(vj.w * acc * dz);
      ngb_acc[off + k] = bv.w * acc;
      T udot = T((double)vj.w * pv * w1 / pow5);
      udot = T((double)udot - (double)(prho2 * dd.z * g) / pow2);
      a[3] = udot * drdv;
    }
    sums.add(a);
  }
  for (int o = 8; o > 0; o >>= 1) vsig = dmax(vsig, __shfl_xor(vsig, o, 16));
  const V4<T> b{sums.get(0), sums.get(1), sums.get(2), sums.get(3)};
  if (l != 0) return;
  bdots[i] = b;
  hydro2[i].x = vsig;
}

// ---------------------------------------------------------------------------
// Mixed form: FP32 pair arithmetic with FMA polynomials (f32k), hardware
// square root and reciprocals, split hi/lo position differences and Kahan
// sums.  The per-particle quantities of the viscosity come precomputed from
// k_eos_mixed.  Same sums as k_density / k_hydro, same list order.

// density, grad-h terms, div v, |curl v| (dev_density_loop.cu:29-111); a
// group of kGroup lanes per particle, each lane taking every kGroup-th
// neighbour, partial sums combined by group_sum
__global__ __launch_bounds__(kBlock) void k_density_mixed(const F4* __restrict__ pos, const F4* __restrict__ vel,
                                                          const F4* __restrict__ pos_lo, F4* __restrict__ hydro,
                                                          F4* __restrict__ dots, const KV* __restrict__ hash,
                                                          const int* __restrict__ offset,
                                                          const int* __restrict__ count,
                                                          const int* __restrict__ list, int n_dev) {
  chain_priority();
  const int g = xcd_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
  const int t = g / kGroup, lane = g % kGroup;
  if (t >= n_dev) return;   // whole groups leave together
  const int i = (int)hash[t].value;
  const F4 bp = pos[i], bv = vel[i], loi = pos_lo[i];
  const int off = offset[i], n = count[i];
  const float two_over_r = n > 0 ? 2.f / bp.w : 0.f;
  KSum rho, om, psi, den, divv, cx, cy, cz;
  for (int k = off + lane; k < off + n; k += kGroup) {
    const int j = list[k];
    const F4 pj = pos[j], vj = vel[j], lj = pos_lo[j];
    const float dx = (bp.x - pj.x) + (loi.x - lj.x);
    const float dy = (bp.y - pj.y) + (loi.y - lj.y);
    const float dz = (bp.z - pj.z) + (loi.z - lj.z);
    const float d2 = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz));
    const float u = __builtin_amdgcn_sqrtf(d2) * two_over_r;
    const float iu = __builtin_amdgcn_rcpf(u);
    rho.add(vj.w * f32k::w(u));
    om.add(vj.w * f32k::dwdh(u));
    psi.add(vj.w * f32k::dphidh(u));
    den.add(-f32k::digdh(u));
    const float dvx = bv.x - vj.x, dvy = bv.y - vj.y, dvz = bv.z - vj.z;
    const float mdw = bv.w * f32k::dw(u, iu);
    divv.add(mdw * __builtin_fmaf(dx, dvx, __builtin_fmaf(dy, dvy, dz * dvz)));
    cx.add(mdw * __builtin_fmaf(dy, dvz, -dz * dvy));
    cy.add(mdw * __builtin_fmaf(dz, dvx, -dx * dvz));
    cz.add(mdw * __builtin_fmaf(dx, dvy, -dy * dvx));
  }
  group_sum(rho);
  group_sum(om);
  group_sum(psi);
  group_sum(den);
  group_sum(divv);
  group_sum(cx);
  group_sum(cy);
  group_sum(cz);
  if (lane != 0) return;
  if (n == 0) {
    hydro[i].x = 0.f;
    dots[i] = {0.f, 0.f, 0.f, 0.f};
    return;
  }
  const double h = 0.5 * (double)bp.w, h3 = h * h * h, h5 = h3 * h * h;
  const double d = den.value();
  double o = 0.0, ps = 0.0;
  if (d != 0.0) {
    o = om.value() / (h3 * d);
    ps = psi.value() / (h * d);
  }
  const double r = rho.value() / h3;
  const double x = cx.value(), y = cy.value(), z = cz.value();
  hydro[i].x = (float)r;
  dots[i] = {(float)(divv.value() / (r * h5)), (float)(sqrt(x * x + y * y + z * z) / (r * h5)), (float)o,
             (float)ps};
}

// hydro accelerations, du/dt, v_sig and the reaction coefficients
// (dev_hydro_dots.cu:25-113, dev_art_visc.cu:8-32); a group of kGroup lanes
// per particle, as in k_density_mixed
__global__ __launch_bounds__(kBlock) void k_hydro_mixed(const F4* __restrict__ pos, const F4* __restrict__ vel,
                                                        const F4* __restrict__ pos_lo, const F4* __restrict__ hydro,
                                                        const F4* __restrict__ dots, F4* __restrict__ bdots,
                                                        F4* __restrict__ hydro2, float* __restrict__ ngb_acc,
                                                        const KV* __restrict__ hash, const int* __restrict__ offset,
                                                        const int* __restrict__ count, const int* __restrict__ list,
                                                        int n_dev, float alpha, float beta) {
  chain_priority();
  const int gl = xcd_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
  const int t = gl / kGroup, lane = gl % kGroup;
  if (t >= n_dev) return;   // whole groups leave together
  const int i = (int)hash[t].value;
  const int off = offset[i], n = count[i];
  const F4 bp = pos[i], bv = vel[i], loi = pos_lo[i], dd = dots[i], qi = hydro2[i];
  const float ci = qi.y, prho2 = qi.z, bal_i = qi.w;
  const float inv_h = n > 0 ? 2.f / bp.w : 0.f, inv_h2 = inv_h * inv_h, inv_h5 = inv_h2 * inv_h2 * inv_h;
  const float k1 = (prho2 * dd.z + 0.5f * dd.w) * inv_h2;   // (P/rho^2 Omega + Psi/2) / h^2
  const float k2 = prho2 * dd.z * inv_h2;                   // P/rho^2 Omega / h^2
  KSum ax, ay, az, ud;
  float vsig = 0.f;
  for (int k = off + lane; k < off + n; k += kGroup) {
    const int j = list[k];
    const F4 pj = pos[j], vj = vel[j], lj = pos_lo[j], qj = hydro2[j];
    const float dx = (bp.x - pj.x) + (loi.x - lj.x);
    const float dy = (bp.y - pj.y) + (loi.y - lj.y);
    const float dz = (bp.z - pj.z) + (loi.z - lj.z);
    const float dvx = bv.x - vj.x, dvy = bv.y - vj.y, dvz = bv.z - vj.z;
    const float d2 = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz));
    const float ds = __builtin_amdgcn_sqrtf(d2);
    const float u = ds * inv_h;
    const float iu = __builtin_amdgcn_rcpf(u);
    const float drdv = __builtin_fmaf(dx, dvx, __builtin_fmaf(dy, dvy, dz * dvz));
    const float cs = ci + qj.y;
    float pi_ = 0.f, vs = cs;
    if (drdv < 0.f) {
      const float r_ds = __builtin_amdgcn_rcpf(ds);
      vs = __builtin_fmaf(-beta * drdv, r_ds, cs);
      const float mu = drdv * r_ds * __builtin_amdgcn_rcpf(cs) * (bal_i + qj.w);
      pi_ = (prho2 + qj.z) * mu * __builtin_fmaf(beta, mu, -alpha);
    }
    vsig = fmaxf(vsig, vs);
    const float w1 = f32k::dw(u, iu), gk = f32k::dig(u, iu);
    const float t1 = __builtin_fmaf(0.5f, pi_, prho2) * w1 * inv_h5;
    const float mjA = __builtin_fmaf(vj.w, t1, -k1 * gk);      // m_j * acc
    ax.add(-mjA * dx);
    ay.add(-mjA * dy);
    az.add(-mjA * dz);
    ngb_acc[k] = bv.w * mjA * __builtin_amdgcn_rcpf(vj.w);   // m_i * acc
    ud.add(__builtin_fmaf(vj.w, t1, -k2 * gk) * drdv);
  }
  group_sum(ax);
  group_sum(ay);
  group_sum(az);
  group_sum(ud);
  vsig = group_max(vsig);
  if (lane != 0) return;
  bdots[i] = {ax.value(), ay.value(), az.value(), ud.value()};
  hydro2[i].x = vsig;
}

// ---------------------------------------------------------------------------
// launchers

template <class T>
void launch_density(const V4<T>* pos, const V4<T>* vel, V4<T>* hydro, V4<T>* dots, const KV* hash,
                    const int* offset, const int* count, const int* list, int n_dev, hipStream_t s) {
  hipLaunchKernelGGL(k_density<T>, dim3(ceil_div(n_dev, kBlock / 16)), dim3(kBlock), 0, s, pos, vel, hydro, dots, hash,
                     offset, count, list, n_dev);
  CS_CHECK_LAUNCH();
}

template <class T>
void launch_eos(V4<T>* hydro, int n_dev, const EosConst& c, hipStream_t s) {
  hipLaunchKernelGGL(k_eos<T>, dim3(ceil_div(n_dev, kBlock)), dim3(kBlock), 0, s, hydro, n_dev, c);
  CS_CHECK_LAUNCH();
}

void launch_eos_mixed(F4* hydro, const double* u64, const F4* pos, const F4* dots, F4* hydro2, int n,
                      const EosConst& c, hipStream_t s) {
  hipLaunchKernelGGL(k_eos_mixed, dim3(ceil_div(n, kBlock)), dim3(kBlock), 0, s, hydro, u64, pos, dots, hydro2, n, c);
  CS_CHECK_LAUNCH();
}

void launch_density_mixed(const F4* pos, const F4* vel, const F4* pos_lo, F4* hydro, F4* dots, const KV* hash,
                          const int* offset, const int* count, const int* list, int n_dev, hipStream_t s) {
  hipLaunchKernelGGL(k_density_mixed, dim3(ceil_div(n_dev * kGroup, kBlock)), dim3(kBlock), 0, s, pos, vel, pos_lo,
                     hydro, dots, hash, offset, count, list, n_dev);
  CS_CHECK_LAUNCH();
}

void launch_hydro_mixed(const F4* pos, const F4* vel, const F4* pos_lo, const F4* hydro, const F4* dots, F4* bdots,
                        F4* hydro2, float* ngb_acc, const KV* hash, const int* offset, const int* count,
                        const int* list, int n_dev, float alpha, float beta, hipStream_t s) {
  hipLaunchKernelGGL(k_hydro_mixed, dim3(ceil_div(n_dev * kGroup, kBlock)), dim3(kBlock), 0, s, pos, vel, pos_lo,
                     hydro, dots, bdots, hydro2, ngb_acc, hash, offset, count, list, n_dev, alpha, beta);
  CS_CHECK_LAUNCH();
}

template <class T>
void launch_hydro(const V4<T>* pos, const V4<T>* vel, const V4<T>* hydro, const V4<T>* dots, V4<T>* bdots,
                  V4<T>* hydro2, T* ngb_acc, const KV* hash, const int* offset, const int* count, const int* list,
                  int n_dev, T alpha, T beta, hipStream_t s) {
  hipLaunchKernelGGL(k_hydro<T>, dim3(ceil_div(n_dev, kBlock / 16)), dim3(kBlock), 0, s, pos, vel, hydro, dots, bdots,
                     hydro2, ngb_acc, hash, offset, count, list, n_dev, alpha, beta);
  CS_CHECK_LAUNCH();
}

template void launch_eos<float>(F4*, int, const EosConst&, hipStream_t);
template void launch_eos<double>(D4*, int, const EosConst&, hipStream_t);
template void launch_density<float>(const F4*, const F4*, F4*, F4*, const KV*, const int*, const int*, const int*,
                                    int, hipStream_t);
template void launch_density<double>(const D4*, const D4*, D4*, D4*, const KV*, const int*, const int*, const int*,
                                     int, hipStream_t);
template void launch_hydro<float>(const F4*, const F4*, const F4*, const F4*, F4*, F4*, float*, const KV*, const int*,
                                  const int*, const int*, int, float, float, hipStream_t);
template void launch_hydro<double>(const D4*, const D4*, const D4*, const D4*, D4*, D4*, double*, const KV*,
                                   const int*, const int*, const int*, int, double, double, hipStream_t);

}  // namespace cudasph
