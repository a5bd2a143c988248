// Host-side declarations of the kernel launchers (implemented in the .hip
// files).  Every launcher enqueues on the given stream and checks the launch.
#pragma once

#include "common.h"

namespace cudasph {

// The SPH passes are short and latency-bound: a wavefront waits on a fetch or
// a launch and then needs only a few instructions.  Beside gravity, whose
// wavefronts always have VALU work ready, they would wait for issue behind
// them too.  Their wavefronts take the highest issue priority instead, so they
// issue as soon as their data is back and gravity fills the remaining cycles.
__device__ __forceinline__ void chain_priority() { __builtin_amdgcn_s_setprio(3); }

// orders this wavefront's LDS writes before its later LDS reads (the LDS
// serves one wavefront's accesses in order; this holds the compiler to it)
__device__ __forceinline__ void lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Sums of NC terms over a list by a group of 16 lanes, in list order (so with
// the bits of one lane's running sums): each lane computes the terms of one
// entry, the group hands them over through its LDS row, and lane c adds component
// c % NC of the 16 one after another.  Lanes past the end of the list hand over
// none(), which changes no sum.
template <class T, int NC>
struct OrderedSums {
  static constexpr int kRow = NC * 16 + 16;   // LDS of a group (16 more, so that the groups' banks differ)
  T s;
  T* row;
  int l;
  static __device__ __forceinline__ T none() { return T(-0.0); }
  __device__ __forceinline__ void add(const T (&t)[NC]) {
#pragma unroll
    for (int c = 0; c < NC; ++c) row[c * 16 + l] = t[c];
    lds_order();
    const T* r = row + (l % NC) * 16;
    T v[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) v[k] = r[k];
#pragma unroll
    for (int k = 0; k < 16; ++k) s += v[k];
    lds_order();
  }
  __device__ __forceinline__ T get(int c) const { return __shfl(s, c, 16); }
};

struct WalkParams {
  int n_nodes;        // real particles (the reference passes n_bodies, CUDA_calls.cpp:5)
  int fix_phantom;
  float rel_err;
  float desired_ngb;
  int max_iter;
  // subtree bounding boxes (launch_tree_boxes), or null: with them the walk
  // also skips a child whose subtree box lies beyond the range.  The same
  // neighbours in the same order; fewer nodes visited (the walk length)
  const F4* boxes = nullptr;
  // the h-solve keeps the distances of its first walk and filters them at its
  // later ranges (0: it walks at every range); the same bits either way
  int solve_cache = 1;
};

struct EosConst;  // sph_math.h

// ---- walks.hip ----
template <class T>
void launch_solve_range(V4<T>* pos, int* n_ngb, const KV* hash, const V4<T>* tree, int n_dev,
                        const WalkParams& wp, hipStream_t s);
// list_cap >= 0: the slots of list; the total offset[n_dev] goes to flags[3],
// and nothing is written if it exceeds them (or is negative)
template <class T>
void launch_find_ngb(const V4<T>* pos, const V4<T>* tree, KV* hash, const int* offset, const int* cap_count,
                     int* count_out, int* list, int* flags, int n_dev, const WalkParams& wp, int clamp, int list_cap,
                     hipStream_t s);
// ---- sph_passes.hip ----
// plain and FP64 forms
template <class T>
void launch_density(const V4<T>* pos, const V4<T>* vel, V4<T>* hydro, V4<T>* dots, const KV* hash,
                    const int* offset, const int* count, const int* list, int n_dev, hipStream_t s);
template <class T>
void launch_eos(V4<T>* hydro, int n_dev, const EosConst& c, hipStream_t s);
// mixed form: FP64 pressure and the per-particle viscosity factors into hydro2.yzw
void launch_eos_mixed(F4* hydro, const double* u64, const F4* pos, const F4* dots, F4* hydro2, int n,
                      const EosConst& c, hipStream_t s);
// mixed form: FP32 pair arithmetic (f32k), Kahan sums, split positions
void launch_density_mixed(const F4* pos, const F4* vel, const F4* pos_lo, F4* hydro, F4* dots, const KV* hash,
                          const int* offset, const int* count, const int* list, int n_dev, hipStream_t s);
void launch_hydro_mixed(const F4* pos, const F4* vel, const F4* pos_lo, const F4* hydro, const F4* dots, F4* bdots,
                        F4* hydro2, float* ngb_acc, const KV* hash, const int* offset, const int* count,
                        const int* list, int n_dev, float alpha, float beta, hipStream_t s);
template <class T>
void launch_hydro(const V4<T>* pos, const V4<T>* vel, const V4<T>* hydro, const V4<T>* dots, V4<T>* bdots,
                  V4<T>* hydro2, T* ngb_acc, const KV* hash, const int* offset, const int* count, const int* list,
                  int n_dev, T alpha, T beta, hipStream_t s);

// ---- gravity.hip ----
// sums (FP32): 0 keeps a particle's four sums in one lane (k_gravity_lane), 1
// and 2 one per wavefront (k_gravity_chains), -1 (auto) the latter up to
// kChainsMaxN particles (kChainsMaxNSpline with the spline softening); the
// same bits either way.  kFastLaneMinN: see k_gravity_lane.
constexpr int kChainsMaxN = 94208;
constexpr int kChainsMaxNSpline = 81920;
constexpr int kFastLaneMinN = 1 << 19;
template <class T>
void launch_gravity(const V4<T>* gpos, const V4<T>* gvel, V4<T>* out, int n_i, int n_j, int soft, T eps,
                    int exact, hipStream_t s, int sums = -1);
// FP64 form, Plummer softening (fused pair body; the j-range split into
// `parts` parts, 0 for gravity64_parts(n_i), `part` then holding parts * n_i
// records when parts > 1).  gravity64_parts: also the reverse pass's split.
int gravity64_parts(int n_i);
void launch_gravity64_plummer(const D4* gpos, D4* out, D4* part, int n_i, int n_j, double eps, hipStream_t s,
                              int parts = 0);
// part: scratch of mixed_part_words(n_j, pairs) records (Plummer only): the
// parts' sums, and where pairs are taken once (never with the far field) running
// sums and a chunk of reactions (at most 2 GiB); mass_range: scratch of 2 + 2 * ceil(n_real / 256) floats ({min, max}
// of the real particles' masses, then per-block partials)
// moments: scratch of 52 floats per 64-record j sub-tile followed by 52 per
// cell of 16384, 4096, 1024 and 256 records and, with split_only bit 6, 52
// per 32-record half sub-tile (the optional multipole far
// field, split_only bit 4, taken where every lane of a wavefront is
// far_ratio radii away, the ratio at a level of C records scaled by
// (C / 16384)^far_grade; may be null otherwise)
// parts: the number of j-parts, 1 .. kGravMixedParts; 0 for the most.
constexpr int kGravMixedParts = 8;   // one per XCD
// Pairs taken once (k_gravity_mixed_pairs).  Steps / the pass alone, ms, every
// ordered pair against once: 8 192 particles 0.378 / 0.103 against 0.377 / 0.143,
// 12 288: 0.425 / 0.152, 0.421 / 0.159, 14 336: 0.432 / 0.176, 0.427 / 0.161, 18 432:
// 0.478 / 0.244, 0.468 / 0.271, 24 576: 0.522 / 0.327, 0.521 / 0.299, 32 768: 0.671,
// 0.595, 65 536: 2.00, 1.64, 131 072: 6.17, 4.78, 250 007: 19.0, 15.7, 2^20: 272.7,
// 231.6; unequal masses 65 536: 2.01, 1.75, 2^20: 300, 254.  (Few tiles: 16 at 8 192,
// whose 128 blocks leave half of the CUs to the SPH passes, and idle without them.)
constexpr int kMixedPairsMinN = 12288;
inline bool mixed_pairs_fit(int n) { return n >= kMixedPairsMinN; }
int mixed_pairs_chunk(int n);
size_t mixed_part_words(int n, bool pairs);   // F4s of `part`
void launch_gravity_mixed(const F4* hi, const F4* lo, const F4* gvel, F4* out, F4* part, float* mass_range,
                          float* moments, float far_ratio, float far_grade, int n_i, int n_j, int n_real,
                          int soft, float eps, int split_only, hipStream_t s, int parts = 0);

// ---- sort.hip ----
// exclusive scan of in[0..n) into out[0..n]; out[n] = total.  mode 1 scans
// n_norm(in[i], 4) (the neighbour-list slot layout).  scratch holds
// scan_scratch_ints(n) ints.
long scan_scratch_ints(long n);
void launch_exclusive_scan(const int* in, int* out, long n, int mode, int* scratch, hipStream_t s);
// stable LSD radix sort of KV records by key bits [0, bits); the result is
// left in `data` (alt is scratch of the same length).  scratch holds
// radix_scratch_ints(n) ints.  max_polls: a tile's looks at the table of the
// earlier ones' counts before it counts their records itself (negative: some
// seconds of them)
long radix_scratch_ints(long n);
void launch_radix_sort(KV* data, KV* alt, long n, int bits, int* scratch, hipStream_t s, int max_polls = -1);
constexpr long radix_header_ints = 8 * 257 + 8;
// ints of a sort's scratch to be zero before launch_axis_sorts
long radix_clear_ints(long n);
// for each axis a the ids 0 .. n-1 in ascending order of (pos[id]'s coordinate
// a, id), in lists + a * list_stride.  kv and alt hold 3 n records; scratch
// 3 radix_scratch_ints(n) ints, the first radix_clear_ints(n) of each third
// zero
template <class T>
void launch_axis_sorts(const V4<T>* pos, int n, KV* kv, KV* alt, int* lists, long list_stride, int* scratch,
                       hipStream_t s);
// the reaction lists: for each of the n particles j, the list slots k
// naming j in ascending k, as pairs {key = owner i, value = k} in
// pairs[start[j], start[j + 1]).  tcnt holds n ints, zero on entry and again
// on return, alt as many pairs as pairs, scan_scratch scan_scratch_ints(n)
// ints.
void launch_reaction_transpose(const int* offset, const int* count, const int* list, int n, int* tcnt,
                               int* start, KV* pairs, KV* alt, int* scan_scratch, hipStream_t s);
// kv[t].key = keys[t]
void launch_set_keys(KV* kv, const uint32_t* keys, int n, hipStream_t s);
// bdots[j].xyz += ngb_acc[k] (r_i - r_j) over the reaction pairs of j, in
// ascending k (sph_accelerations.cpp:104-115)
template <class T>
void launch_reaction(const V4<T>* pos, V4<T>* bdots, const T* ngb_acc, const KV* pairs, const int* start,
                     int n, hipStream_t s);
void launch_reaction_mixed(const F4* pos, const F4* pos_lo, F4* bdots, const float* ngb_acc, const KV* pairs,
                           const int* start, int n, hipStream_t s);
// Peano-Hilbert keys on the bounding cube (sort_bodies.cpp:121-163); keys
// are 3*bits wide, written as (hi,lo) 32-bit halves; scratch holds
// 6 * (ceil(n / 256) + 1) reals of type T
template <class T>
void launch_ph_keys(const V4<T>* pos, int n, int bits, uint32_t* key_hi, uint32_t* key_lo, int* scratch,
                    hipStream_t s);

// ---- tree.hip ----
// The kd-tree of the first n positions (kd_tree.cpp:39-128) built on the
// device: tree[0..n_dev+1] and hash[0..n_dev) as the host builder writes them
// (heap_order 1: hash in the nodes' heap order, 0: identity).  work holds
// tree_work_ints(n) ints; kv and kv_alt 3 n records each; sort_scratch
// 3 radix_scratch_ints(n) ints.
long tree_work_ints(long n);
// ties (may be null): cleared, and set to 1 when some node's particle shares its split
// coordinate with another particle of its subtree -- the one case in which
// the reference's quicksort may have picked the other particle as the node;
// otherwise the tree is the reference's, bit for bit.
template <class T>
void launch_tree_build(const V4<T>* pos, int n, int n_dev, V4<T>* tree, KV* hash, int heap_order, int* work,
                       KV* kv, KV* kv_alt, int* sort_scratch, hipStream_t s, int* ties = nullptr);
// Subtree bounding boxes of a kd-tree over n_nodes particles: box[2k] (low
// corner) and box[2k+1] (high corner) of node k's subtree, for k up to
// n_nodes+1; FP32, rounded outward.  Two launches: one block per subtree
// below level 10, then one block for the levels above.
template <class T>
void launch_tree_boxes(const V4<T>* tree, F4* box, int n_nodes, int fix_phantom, hipStream_t s);

// ---- integrate.hip ----
template <class T>
void launch_gravity_pack(const V4<T>* pos, const V4<T>* vel, V4<T>* gpos, V4<T>* gvel, int n, int n_dev,
                         hipStream_t s);
void launch_gravity_pack_mixed(const D4* pos64, const F4* pos, const F4* vel, F4* hi, F4* lo, F4* gvel, int n,
                               int n_dev, hipStream_t s);
template <class T>
void launch_predict(V4<T>* pos, V4<T>* vel, V4<T>* hydro, V4<T>* bdots, V4<T>* grav, V4<T>* old_vu,
                    const double* dt, int n, hipStream_t s);
template <class T>
void launch_correct(V4<T>* vel, V4<T>* hydro, const V4<T>* bdots, const V4<T>* old_vu, const double* dt_new,
                    const double* dt_old, int n, hipStream_t s);
void launch_predict_mixed(D4* pos64, D4* vel64, double* u64, D4* old64, F4* pos, F4* pos_lo, F4* vel, F4* hydro,
                          F4* bdots, F4* grav, const double* dt, int n, hipStream_t s);
void launch_correct_mixed(D4* vel64, double* u64, const D4* old64, F4* vel, F4* hydro, const F4* bdots,
                          const double* dt_new, const double* dt_old, int n, hipStream_t s);
void launch_refresh_mixed(const D4* pos64, const D4* vel64, const double* u64, F4* pos, F4* pos_lo, F4* vel,
                          F4* hydro, int n, hipStream_t s);
// The end of a step over the n real particles, `what` a sum of:
enum {
  kAddGravity = 1,   // bdots += grav; force6: the force and torque sums
  kStatistics = 2,   // stats6: T U W Jx Jy Jz; diag: bounding box, mass and mass-weighted position and velocity
                     // sums, the h-solve counts n_ngb (min, max, sum, sum of squares), the number whose list
                     // length ngb_count differs, the longest list (19 doubles; layout: integrate.hip, kDg*)
  kTimestep = 4      // dt = min_i 1/(1/dt_vel + 1/dt_eth) (compute_timestep.cpp:3-25); round_float stores the
                     // float-rounded value as the reference returns float
};
template <class T>
struct StepEnd {
  V4<T>* bdots;
  const V4<T>*grav, *pos, *vel, *hydro, *hydro2;
  const D4 *pos64, *vel64;   // the mixed form's state, else null
  const double* u64;
  const int *n_ngb, *ngb_count;
  int n;
  float cn_vel, cn_eth;
  double* partials;          // reduce_partials(n)
};
long reduce_partials(int n);
template <class T>
void launch_step_end(const StepEnd<T>& e, int what, int round_float, double* force6, double* stats6, double* diag,
                     double* dt_out, hipStream_t s);
// permutation gather of a 4-record array: dst[t] = src[perm[t]]
template <class R>
void launch_gather(const R* src, R* dst, const KV* perm, int n, hipStream_t s);
void launch_iota_kv(KV* kv, int n, hipStream_t s);
// pos[i].w <-> range[i]
template <class T>
void launch_set_range(V4<T>* pos, const double* range, int n, hipStream_t s);
template <class T>
void launch_get_range(const V4<T>* pos, double* range, int n, hipStream_t s);
void launch_copy16(const F4* src, F4* dst, long n, hipStream_t s);
// FP32 FMA probe: blocks x kBlock lanes, 8 * iters FMAs per lane (form 0:
// 8 chains of v_fma_f32 with scalar coefficients; form 1: 16 chains of the
// accumulate form v_fmac_f32 with vector operands); out holds blocks * kBlock
// floats
void launch_fma_peak(float* out, int blocks, int iters, int form, hipStream_t s);
// the expanded gravity pair body alone: blocks x kBlock lanes, 16 * rounds
// pairs per lane (variant 1: the rsq replaced by a multiply)
void launch_pair_body(float* out, int blocks, int rounds, int variant, hipStream_t s);

}  // namespace cudasph
