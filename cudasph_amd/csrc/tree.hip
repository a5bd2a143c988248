// Device build of the reference's kd-tree (kd_tree.cpp:39-128, packing
// sph_accelerations.cpp:21-33).
//
// The tree is the left-balanced implicit tree: node p holds one particle, its
// children are 2p and 2p+1, the split axis of depth d is d % 3, and the node's
// particle is the one at rank size(2p) (the size of its left subtree) of its
// subtree's particles along that axis.  Every node of the nodes 1..n exists,
// so the tree's shape, every subtree's size and where it starts among the
// nodes of a level are closed forms of n (subtree_size, subtree_start).
//
// The build is level by level, on three lists of particle ids, one per axis,
// each sorted once by (coordinate, id) (launch_axis_sorts) and kept grouped by
// subtree: at level L each list holds the particles not yet placed subtree by
// subtree (t ascending), each subtree's run still in its axis's order.  A
// place in a list tells its subtree (subtree_at), all in closed form.  One
// level, two launches:
//  * the list of the split axis L % 3 holds each subtree's particles in split
//    order, so the particle at rank size(2t) of the run becomes node t, the
//    ones before go to subtree 2t and the ones after to 2t+1 -- both runs stay
//    contiguous and in order, shifted by the closed-form count of nodes placed
//    before them;
//  * the other two lists are partitioned stably.  A particle's side follows
//    from (its coordinate, its id) against the node's particle's -- the order
//    of the split axis's list.  k_tree_count finds the sides and counts them
//    per tile of 1024 places; k_tree_move adds the tiles before, and places each
//    particle after the earlier ones of its side: those of its own run are the
//    counted ones less the closed-form total of the runs before.
// Levels: floor(log2 n) + 1.  Work per level is O(n); nothing is sorted after
// the first three sorts.
//
// Bound: the latency of its dependent launches (few particles) and of their
// gathers.  Five launches of presorts, two per level and the LDS finish, in
// place of 22, six per level and the finish; every closed form is a handful of
// operations (they had been loops over the levels).
//
// Ties in a coordinate: the reference's first-element-pivot quicksort decides
// which of two equal-coordinate particles becomes the node; here the order of
// the first sort (ascending particle id) does.  Either way every particle of a
// left subtree has coordinate <= the node's and every one of a right subtree
// >= it, which is all the walks' pruning (dev_solve_range.cu:48-61) uses, so
// the neighbour sets are the same; without ties the two trees are identical.
#include "common.h"
#include "kernels.h"

namespace cudasph {
namespace {

// The complete tree of n nodes: levels 0 .. D, all full but the last, which
// holds heap nodes 2^D .. n.  A node k levels above the last has 2^k places in
// it, filled from the left.
__host__ __device__ __forceinline__ int floor_log2(int x) {
#ifdef __HIP_DEVICE_COMPILE__
  return 31 - __clz(x);
#else
  return 31 - __builtin_clz((unsigned)x);
#endif
}

// nodes in the subtree of heap node t (0 if t > n)
__host__ __device__ __forceinline__ int subtree_size(int t, int n) {
  if (t > n) return 0;
  const int k = floor_log2(n) - floor_log2(t);
  const int first = t << k, last = n - first + 1;   // (places of the last level: below 2^24)
  return (1 << k) - 1 + (last < 0 ? 0 : last < (1 << k) ? last : 1 << k);
}

// among the nodes of levels >= L, laid out subtree by subtree, the offset of
// the subtree of level-L node t (2^L <= t <= 2^(L+1)): the nodes below the
// level-L nodes left of t
__host__ __device__ __forceinline__ int subtree_start(int t, int L, int n) {
  const int k = floor_log2(n) - L;
  if (k < 0) return 0;
  const int m = t - (1 << L), fill = n + 1 - (1 << (k + L)), slots = m << k;
  return m * ((1 << k) - 1) + (slots < fill ? slots : fill);
}

// of those, the ones below left children
__host__ __device__ __forceinline__ int lefts_before(int t, int L, int n) {
  const int k = floor_log2(n) - L - 1;   // of the level-(L+1) children
  if (k < 0) return 0;
  const int m = t - (1 << L), fill = n + 1 - (1 << (k + 1 + L)), slots = m << (k + 1);
  const int filled = slots < fill ? slots : fill;
  const int part = filled & ((2 << k) - 1);
  return m * ((1 << k) - 1) + ((filled >> (k + 1)) << k) + (part < (1 << k) ? part : 1 << k);
}

// the level-L node whose run holds place idx of the level's layout
__host__ __device__ __forceinline__ int subtree_at(int idx, int L, int n) {
  const int k = floor_log2(n) - L;
  const int fill = n + 1 - (1 << (k + L)), full = fill >> k, part = fill & ((1 << k) - 1);
  const int large = (2 << k) - 1, small = (1 << k) - 1;   // a subtree's nodes with and without its last level
  if (idx < full * large) return (1 << L) + idx / large;
  idx -= full * large;
  return (1 << L) + full + (idx < small + part ? 0 : 1 + (idx - small - part) / small);
}

template <class T>
__device__ __forceinline__ T coord(const V4<T>& p, int axis) {
  return axis == 0 ? p.x : (axis == 1 ? p.y : p.z);
}

__device__ __forceinline__ float node_word(float, int bits) { return __int_as_float(bits); }
__device__ __forceinline__ double node_word(double, int bits) { return (double)bits; }

// fixed slots (sph_accelerations.cpp:21-33, read_state.cpp:85-88): slot 0 and
// slot n_dev+1 zero, slots n+1..n_dev far sentinels with split 3; the
// identity hash, or the padding part of the heap-order hash
// and the zeros that the presorts start from
template <class T>
__global__ __launch_bounds__(kBlock) void k_tree_fixed(V4<T>* __restrict__ tree, KV* __restrict__ hash, int n,
                                                        int n_dev, int heap_order, int* __restrict__ scratch,
                                                        int clear, long stride, int* __restrict__ ties) {
  chain_priority();
  const int t = blockIdx.x * kBlock + threadIdx.x;
  if (t < clear)
    for (int a = 0; a < 3; ++a) scratch[a * stride + t] = 0;
  if (ties && t == 0) *ties = 0;
  if (t >= n_dev + 2) return;
  if (t == 0 || t == n_dev + 1) tree[t] = {T(0), T(0), T(0), T(0)};
  else if (t > n) tree[t] = {T(1e10), T(1e10), T(1e10), node_word(T(0), -1)};
  if (t < n_dev) {
    if (!heap_order) hash[t] = {(uint32_t)t, (uint32_t)t};
    else if (t >= n) hash[t] = {1u << 24, (uint32_t)t};
  }
}

// order of the split axis's list: (coordinate image, id)
__device__ __forceinline__ bool before(float a, int ia, float b, int ib) {
  const uint32_t x = __float_as_uint(a), y = __float_as_uint(b);
  const uint32_t ox = (x & 0x80000000u) ? ~x : (x | 0x80000000u), oy = (y & 0x80000000u) ? ~y : (y | 0x80000000u);
  return ox < oy || (ox == oy && ia < ib);
}
__device__ __forceinline__ bool before(double a, int ia, double b, int ib) {
  const uint64_t x = (uint64_t)__double_as_longlong(a), y = (uint64_t)__double_as_longlong(b), top = 1ull << 63;
  const uint64_t ox = (x & top) ? ~x : (x | top), oy = (y & top) ? ~y : (y | top);
  return ox < oy || (ox == oy && ia < ib);
}

constexpr int kLevelRounds = 4;
constexpr int kLevelTile = kBlock * kLevelRounds;   // places per block
enum { kPlaced = 0, kLeft = 1, kRight = 2 };

// place of round r of this thread in its tile: each wavefront takes 256
// consecutive places
__device__ __forceinline__ int level_place(int r) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  return blockIdx.x * kLevelTile + wave * (kLevelTile / 4) + r * 64 + lane;
}

// level L: the side of every place of the two lists not split (blockIdx.y 0,
// 1), and each tile's {left, right} counts
template <class T>
__global__ __launch_bounds__(kBlock) void k_tree_count(const int* __restrict__ la, const int* __restrict__ lb,
                                                        const int* __restrict__ lc, const V4<T>* __restrict__ pos,
                                                        uint8_t* __restrict__ side, int2* __restrict__ tile_counts,
                                                        int m, int L, int n, int axis) {
  chain_priority();
  __shared__ int2 s_wave[kBlock / 64];
  const int* l = blockIdx.y ? lc : lb;
  side += (size_t)blockIdx.y * n;
  int nl = 0, nr = 0;
#pragma unroll
  for (int r = 0; r < kLevelRounds; ++r) {
    const int idx = level_place(r);
    int f = kPlaced;
    if (idx < m) {
      const int id = l[idx];
      const int t = subtree_at(idx, L, n);
      const int node = la[subtree_start(t, L, n) + subtree_size(2 * t, n)];   // becomes node t
      if (id != node)
        f = before(coord(pos[id], axis), id, coord(pos[node], axis), node) ? kLeft : kRight;
      side[idx] = (uint8_t)f;
    }
    nl += __popcll(__ballot(f == kLeft));
    nr += __popcll(__ballot(f == kRight));
  }
  if ((threadIdx.x & 63) == 0) s_wave[threadIdx.x >> 6] = make_int2(nl, nr);
  __syncthreads();
  if (threadIdx.x == 0) {
    int2 c = s_wave[0];
    for (int w = 1; w < kBlock / 64; ++w) {
      c.x += s_wave[w].x;
      c.y += s_wave[w].y;
    }
    tile_counts[(size_t)blockIdx.y * gridDim.x + blockIdx.x] = c;
  }
}

// level L: the three lists into the next level's layout (blockIdx.y 0: the
// split axis's, 1, 2: the others), the nodes placed
template <class T>
__global__ __launch_bounds__(kBlock) void k_tree_move(const int* __restrict__ la, const int* __restrict__ lb,
                                                       const int* __restrict__ lc, int* __restrict__ la_next,
                                                       int* __restrict__ lb_next, int* __restrict__ lc_next,
                                                       const uint8_t* __restrict__ side,
                                                       const int2* __restrict__ tile_counts,
                                                       const V4<T>* __restrict__ pos, V4<T>* __restrict__ tree,
                                                       KV* __restrict__ hash, int m, int L, int n, int axis,
                                                       int heap_order, int* __restrict__ ties) {
  chain_priority();
  if (blockIdx.y == 0) {
#pragma unroll
    for (int r = 0; r < kLevelRounds; ++r) {
      const int idx = level_place(r);
      if (idx >= m) continue;
      const int id = la[idx];
      const int t = subtree_at(idx, L, n);
      const int p = idx - subtree_start(t, L, n), lt = subtree_size(2 * t, n);
      const int placed_before = t - (1 << L);   // level-L nodes left of t
      if (p < lt) {
        la_next[idx - placed_before] = id;
      } else if (p > lt) {
        la_next[idx - placed_before - 1] = id;
      } else {
        const V4<T> q = pos[id];
        tree[t] = {q.x, q.y, q.z, node_word(T(0), id | (axis << 24))};
        if (heap_order) hash[t - 1] = {(uint32_t)(t - 1), (uint32_t)id};
        // a run neighbour with the node's coordinate: which of the two becomes
        // the node is the presort's choice, not necessarily the reference's
        if (ties) {
          const T c = coord(q, axis);
          if ((p > 0 && coord(pos[la[idx - 1]], axis) == c) ||
              (p + 1 < subtree_size(t, n) && coord(pos[la[idx + 1]], axis) == c))
            atomicOr(ties, 1);
        }
      }
    }
    return;
  }
  const int which = blockIdx.y - 1;
  const int* l = which ? lc : lb;
  int* next = which ? lc_next : lb_next;
  side += (size_t)which * n;
  tile_counts += (size_t)which * gridDim.x;
  __shared__ int2 s_before[kBlock / 64], s_wave[kBlock / 64];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  // the tiles before
  int2 sum = make_int2(0, 0);
  for (int b = threadIdx.x; b < (int)blockIdx.x; b += kBlock) {
    const int2 c = tile_counts[b];
    sum.x += c.x;
    sum.y += c.y;
  }
  for (int o = 32; o > 0; o >>= 1) {
    sum.x += __shfl_xor(sum.x, o);
    sum.y += __shfl_xor(sum.y, o);
  }
  int f[kLevelRounds], lefts[kLevelRounds], rights[kLevelRounds], nl = 0, nr = 0;
  const unsigned long long below = (1ull << lane) - 1ull;
#pragma unroll
  for (int r = 0; r < kLevelRounds; ++r) {
    const int idx = level_place(r);
    f[r] = idx < m ? side[idx] : (int)kPlaced;
    const unsigned long long ml = __ballot(f[r] == kLeft), mr = __ballot(f[r] == kRight);
    lefts[r] = nl + __popcll(ml & below);
    rights[r] = nr + __popcll(mr & below);
    nl += __popcll(ml);
    nr += __popcll(mr);
  }
  if (lane == 0) {
    s_before[wave] = sum;
    s_wave[wave] = make_int2(nl, nr);
  }
  __syncthreads();
  int bl = 0, br = 0;
  for (int w = 0; w < kBlock / 64; ++w) {
    bl += s_before[w].x + (w < wave ? s_wave[w].x : 0);
    br += s_before[w].y + (w < wave ? s_wave[w].y : 0);
  }
#pragma unroll
  for (int r = 0; r < kLevelRounds; ++r) {
    if (f[r] == kPlaced) continue;
    const int idx = level_place(r);
    const int t = subtree_at(idx, L, n);
    const int start = subtree_start(t, L, n), run = t - (1 << L);   // placed before this run: one per run
    const int base = start - run;                                    // where subtree 2t starts in the next layout
    const int lb0 = lefts_before(t, L, n);
    if (f[r] == kLeft) next[base + bl + lefts[r] - lb0] = l[idx];
    else next[base + subtree_size(2 * t, n) + br + rights[r] - (base - lb0)] = l[idx];
  }
}

// ---------------------------------------------------------------------------
// The last levels in LDS.  Once every subtree of level L0 holds at most
// kLdsMax particles, one block per subtree builds the rest of it in its own
// LDS: the block reads its three runs (particle ids, in the level-L0 layout),
// names each particle by its rank in the first run (a slot), and runs the
// split / flags / scans / regroup of the level kernels above on slots, with
// per-level positions taken relative to where the subtree's runs start in
// that level's layout.  The level kernels' dependent global-memory passes
// (the build's cost at small N) become LDS passes; the results are the same
// nodes in the same places.
constexpr int kLdsMax = 1024;
// threads of a finishing block: few blocks run (one per subtree), so each
// takes a whole CU's worth of wavefronts to keep its passes short
constexpr int kLdsThreads = 512;

struct LocalLevel {
  int L, r0, r1, r0n;        // level, the runs' range in its layout, and their start at level L+1
  int t_base;                // first level-L node of the subtree
};

// exclusive scans of two values per thread (kLdsThreads threads) at once: within
// each wavefront by shuffles, then across the block's wavefronts through
// LDS (one barrier)
__device__ __forceinline__ void block_excl_scan2(int& x, int& y, int* s_tot) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int ix = x, iy = y;
  for (int o = 1; o < 64; o <<= 1) {
    const int ux = __shfl_up(ix, o), uy = __shfl_up(iy, o);
    if (lane >= o) {
      ix += ux;
      iy += uy;
    }
  }
  if (lane == 63) {
    s_tot[wave] = ix;
    s_tot[kLdsThreads / 64 + wave] = iy;
  }
  __syncthreads();
  int bx = 0, by = 0;
  for (int w = 0; w < wave; ++w) {
    bx += s_tot[w];
    by += s_tot[kLdsThreads / 64 + w];
  }
  x = bx + ix - x;
  y = by + iy - y;
}

template <class T>
__global__ __launch_bounds__(kLdsThreads) void k_tree_lds(const int* __restrict__ work, int* __restrict__ slot_of, int n,
                                                      int L0, int cur0, int cur1, int cur2,
                                                      const V4<T>* __restrict__ pos, V4<T>* __restrict__ tree,
                                                      KV* __restrict__ hash, int heap_order, int* __restrict__ ties) {
  chain_priority();
  __shared__ uint16_t s_list[3][2][kLdsMax];   // slots, per axis, double-buffered
  __shared__ int s_tag[kLdsMax];               // the heap node each slot's particle belongs to
  __shared__ uint8_t s_fb[kLdsMax], s_fc[kLdsMax];
  __shared__ uint16_t s_sb[kLdsMax], s_sc[kLdsMax];
  __shared__ uint16_t s_at_b[kLdsMax], s_at_c[kLdsMax];   // local position of each node's placed particle
  __shared__ int s_tot[2 * kLdsThreads / 64];
  const int tid = threadIdx.x;
  const int T0 = (1 << L0) + (int)blockIdx.x;
  if (T0 > n) return;
  const int base0 = subtree_start(T0, L0, n);
  const int m0 = subtree_size(T0, n);
  const int* gl[3];
  const int curs[3] = {cur0, cur1, cur2};
  for (int a = 0; a < 3; ++a) gl[a] = work + (size_t)(2 * a + curs[a]) * n + base0;
  // slots: rank in the first run; slot_of (indexed by particle) carries
  // the names to the other two runs
  for (int k = tid; k < m0; k += kLdsThreads) {
    const int id = gl[0][k];
    s_tag[k] = T0;
    s_list[0][0][k] = (uint16_t)k;
    slot_of[id] = k;
  }
  __syncthreads();
  for (int k = tid; k < m0; k += kLdsThreads) {
    s_list[1][0][k] = (uint16_t)slot_of[gl[1][k]];
    s_list[2][0][k] = (uint16_t)slot_of[gl[2][k]];
  }
  __syncthreads();
  int cur[3] = {0, 0, 0};
  for (int L = L0; L < 31; ++L) {
    const long long d0 = (long long)T0 << (L - L0), d1 = (long long)(T0 + 1) << (L - L0);
    if (d0 > n) break;
    const int r0 = subtree_start((int)d0, L, n);
    const int r1 = subtree_start((int)min(d1, (long long)n + 1), L, n);
    if (r0 >= r1) break;
    const long long e0 = d0 << 1;
    const int r0n = subtree_start((int)min(e0, (long long)n + 1), L + 1, n);
    const int a = L % 3, b = (L + 1) % 3, c = (L + 2) % 3;
    const int next_level = 2 << L;
    const int t_base = (int)d0;
    // split on axis a
    for (int i = tid; i < r1 - r0; i += kLdsThreads) {
      const int g = r0 + i;
      const int slot = s_list[a][cur[a]][i];
      const int t = s_tag[slot];
      const int p = g - subtree_start(t, L, n);
      const int lt = subtree_size(2 * t, n);
      const int pb = t - (1 << L);
      if (p < lt) {
        s_tag[slot] = 2 * t;
        s_list[a][cur[a] ^ 1][g - pb - r0n] = (uint16_t)slot;
      } else if (p == lt) {
        const int id = gl[0][slot];   // the slot is the particle's rank in the first run
        const V4<T> q = pos[id];
        tree[t] = {q.x, q.y, q.z, node_word(T(0), id | (a << 24))};
        if (heap_order) hash[t - 1] = {(uint32_t)(t - 1), (uint32_t)id};
        if (ties) {   // as in k_tree_move
          const T cq = coord(q, a);
          if ((p > 0 && coord(pos[gl[0][s_list[a][cur[a]][i - 1]]], a) == cq) ||
              (p + 1 < subtree_size(t, n) && coord(pos[gl[0][s_list[a][cur[a]][i + 1]]], a) == cq))
            atomicOr(ties, 1);
        }
      } else {
        s_tag[slot] = 2 * t + 1;
        s_list[a][cur[a] ^ 1][g - pb - 1 - r0n] = (uint16_t)slot;
      }
    }
    __syncthreads();
    // flags of the other two lists, and where each node's placed particle sits in them
    for (int i = tid; i < r1 - r0; i += kLdsThreads) {
      const int tb = s_tag[s_list[b][cur[b]][i]], tc = s_tag[s_list[c][cur[c]][i]];
      s_fb[i] = tb >= next_level && !(tb & 1);
      s_fc[i] = tc >= next_level && !(tc & 1);
      if (tb < next_level) s_at_b[tb - t_base] = (uint16_t)i;
      if (tc < next_level) s_at_c[tc - t_base] = (uint16_t)i;
    }
    __syncthreads();
    // exclusive scans of the flags over the runs (chunks of ceil(R / kLdsThreads) per thread)
    {
      const int R = r1 - r0;
      const int chunk = (R + kLdsThreads - 1) / kLdsThreads;
      const int i0 = min(R, tid * chunk), i1 = min(R, i0 + chunk);
      int cb = 0, cc = 0;
      for (int i = i0; i < i1; ++i) {
        cb += s_fb[i];
        cc += s_fc[i];
      }
      int ob = cb, oc = cc;
      block_excl_scan2(ob, oc, s_tot);
      for (int i = i0; i < i1; ++i) {
        s_sb[i] = (uint16_t)ob;
        s_sc[i] = (uint16_t)oc;
        ob += s_fb[i];
        oc += s_fc[i];
      }
    }
    __syncthreads();
    // regroup the other two lists into the next level's runs
    for (int i = tid; i < r1 - r0; i += kLdsThreads) {
      const int g = r0 + i;
      for (int k = 0; k < 2; ++k) {
        const int ax = k ? c : b;
        const int slot = s_list[ax][cur[ax]][i];
        const int nt = s_tag[slot];
        if (nt < next_level) continue;   // placed at this level
        const int t = nt >> 1;
        const int s = subtree_start(t, L, n);
        const int base = s - (t - (1 << L));
        const uint16_t* scn = k ? s_sc : s_sb;
        const int lefts = scn[i] - scn[s - r0];
        int dst;
        if (!(nt & 1)) {
          dst = base + lefts;
        } else {
          const int at = (k ? s_at_c : s_at_b)[t - t_base];
          dst = base + subtree_size(2 * t, n) + (g - s) - lefts - (at < i ? 1 : 0);
        }
        s_list[ax][cur[ax] ^ 1][dst - r0n] = (uint16_t)slot;
      }
    }
    __syncthreads();
    for (int k = 0; k < 3; ++k) cur[k] ^= 1;
  }
}

}  // namespace

// three lists and their next-level copies, the sides (bytes) and tile counts
// of two, the slot names of the LDS finish
static long level_tiles(long n) { return (n + kLevelTile - 1) / kLevelTile; }
long tree_work_ints(long n) { return 8 * n + 4 * level_tiles(n) + 16; }

template <class T>
void launch_tree_build(const V4<T>* pos, int n, int n_dev, V4<T>* tree, KV* hash, int heap_order, int* work,
                       KV* kv, KV* kv_alt, int* sort_scratch, hipStream_t s, int* ties) {
  if (n <= 0 || n > n_dev) throw std::invalid_argument("tree build: need 0 < n <= n_dev");
  const long clear = radix_clear_ints(n);
  hipLaunchKernelGGL((k_tree_fixed<T>), dim3(ceil_div(std::max<long>(n_dev + 2, clear), kBlock)), dim3(kBlock), 0, s,
                     tree, hash, n, n_dev, heap_order, sort_scratch, (int)clear, radix_scratch_ints(n), ties);
  CS_CHECK_LAUNCH();
  int* list[3][2];
  for (int a = 0; a < 3; ++a)
    for (int k = 0; k < 2; ++k) list[a][k] = work + (size_t)(2 * a + k) * n;
  int* slot_of = work + 6 * (size_t)n;
  // (16-byte steps: int2 counts, then the bytes)
  int2* tile_counts = reinterpret_cast<int2*>(work + ((7 * (size_t)n + 3) & ~(size_t)3));
  uint8_t* side = reinterpret_cast<uint8_t*>(tile_counts + 2 * level_tiles(n));
  launch_axis_sorts<T>(pos, n, kv, kv_alt, list[0][0], 2l * n, sort_scratch, s);
  int cur[3] = {0, 0, 0};
  int m = n;
  // level kernels while the level's subtrees hold more than kLdsMax
  // particles (the leftmost is the largest), then one launch in LDS
  int L_lds = 0;
  while (subtree_size(1 << L_lds, n) > kLdsMax) ++L_lds;
  for (int L = 0; m > 0 && L < L_lds; ++L) {
    const int a = L % 3, b = (L + 1) % 3, c = (L + 2) % 3, tiles = (int)level_tiles(m);
    hipLaunchKernelGGL((k_tree_count<T>), dim3(tiles, 2), dim3(kBlock), 0, s, list[a][cur[a]], list[b][cur[b]],
                       list[c][cur[c]], pos, side, tile_counts, m, L, n, a);
    CS_CHECK_LAUNCH();
    hipLaunchKernelGGL((k_tree_move<T>), dim3(tiles, 3), dim3(kBlock), 0, s, list[a][cur[a]], list[b][cur[b]],
                       list[c][cur[c]], list[a][cur[a] ^ 1], list[b][cur[b] ^ 1], list[c][cur[c] ^ 1], side,
                       tile_counts, pos, tree, hash, m, L, n, a, heap_order, ties);
    CS_CHECK_LAUNCH();
    for (int k = 0; k < 3; ++k) cur[k] ^= 1;
    m -= (int)std::min<long>(1l << L, (long)n - ((1l << L) - 1));
  }
  if (m > 0) {
    const int roots = (int)std::min<long>(1l << L_lds, (long)n - (1l << L_lds) + 1);
    hipLaunchKernelGGL((k_tree_lds<T>), dim3(roots), dim3(kLdsThreads), 0, s, work, slot_of, n, L_lds, cur[0], cur[1],
                       cur[2], pos, tree, hash, heap_order, ties);
    CS_CHECK_LAUNCH();
  }
}

namespace {

// a coordinate as a float bound: rounded down (lo) or up (hi) when it is not
// a float already
__device__ __forceinline__ float lo_bound(float x) { return x; }
__device__ __forceinline__ float hi_bound(float x) { return x; }
// the neighbouring float below / above a finite f (its bit pattern moved by
// one unit away from or towards zero)
__device__ __forceinline__ float float_below(float f) {
  const int b = __float_as_int(f);
  return f > 0.f ? __int_as_float(b - 1) : (f < 0.f ? __int_as_float(b + 1) : -__int_as_float(1));
}
__device__ __forceinline__ float float_above(float f) {
  const int b = __float_as_int(f);
  return f > 0.f ? __int_as_float(b + 1) : (f < 0.f ? __int_as_float(b - 1) : __int_as_float(1));
}
__device__ __forceinline__ float lo_bound(double x) {
  const float f = (float)x;
  return (double)f > x ? float_below(f) : f;
}
__device__ __forceinline__ float hi_bound(double x) {
  const float f = (float)x;
  return (double)f < x ? float_above(f) : f;
}

// box of node k: the node's own particle and the boxes of the children a
// walk can enter from it (their boxes written before)
template <class T>
__device__ __forceinline__ void box_node(const V4<T>* __restrict__ tree, F4* box, int n_nodes, int fix_phantom,
                                         int k) {
  const V4<T> nd = tree[k];
  F4 lo = {lo_bound(nd.x), lo_bound(nd.y), lo_bound(nd.z), 0.f};
  F4 hi = {hi_bound(nd.x), hi_bound(nd.y), hi_bound(nd.z), 0.f};
  const int c = 2 * k;
  for (int ch = c; ch <= c + 1; ++ch) {
    // children 2k, 2k+1 <= n_nodes; node n_nodes+1 (the phantom) is entered
    // from 2k = n_nodes unless fix_phantom
    if (ch > n_nodes && !(ch == n_nodes + 1 && c == n_nodes && !fix_phantom)) continue;
    const F4 a = box[2 * ch], b = box[2 * ch + 1];
    lo = {fminf(lo.x, a.x), fminf(lo.y, a.y), fminf(lo.z, a.z), 0.f};
    hi = {fmaxf(hi.x, b.x), fmaxf(hi.y, b.y), fmaxf(hi.z, b.z), 0.f};
  }
  box[2 * k] = lo;
  box[2 * k + 1] = hi;
}

// One block per subtree rooted at level S (node 2^S + blockIdx.x): its levels
// deepest first, with a barrier between levels, so that a node's children
// were written by the same block before it reads them.
template <class T>
__global__ __launch_bounds__(kBlock) void k_tree_boxes_sub(const V4<T>* __restrict__ tree, F4* box, int n_nodes,
                                                            int fix_phantom, int S, int levels, int last_node) {
  chain_priority();
  const long r = (1l << S) + blockIdx.x;
  for (int L = levels; L >= S; --L) {
    const long first = r << (L - S), cnt = 1l << (L - S);
    for (long q = threadIdx.x; q < cnt; q += kBlock)
      if (first + q <= last_node) box_node<T>(tree, box, n_nodes, fix_phantom, (int)(first + q));
    __syncthreads();
  }
}

// the levels above S, in one block
template <class T>
__global__ __launch_bounds__(kBlock) void k_tree_boxes_top(const V4<T>* __restrict__ tree, F4* box, int n_nodes,
                                                            int fix_phantom, int S, int last_node) {
  chain_priority();
  for (int L = S - 1; L >= 0; --L) {
    const int last = (int)std::min<long>((2l << L) - 1, (long)last_node);
    for (int k = (1 << L) + (int)threadIdx.x; k <= last; k += kBlock) box_node<T>(tree, box, n_nodes, fix_phantom, k);
    __syncthreads();
  }
}

}  // namespace

constexpr int kBoxSubtreeLevel = 10;

template <class T>
void launch_tree_boxes(const V4<T>* tree, F4* box, int n_nodes, int fix_phantom, hipStream_t s) {
  const int last_node = n_nodes + 1;   // the phantom's box is its record's point
  int levels = 0;
  while ((2l << levels) <= (long)last_node) ++levels;   // deepest level: floor(log2(last_node))
  // subtrees rooted at level S, up to 2^10 of them, then the levels above
  const int S = std::min(levels, kBoxSubtreeLevel);
  hipLaunchKernelGGL(k_tree_boxes_sub<T>, dim3(1 << S), dim3(kBlock), 0, s, tree, box, n_nodes, fix_phantom, S, levels,
                     last_node);
  CS_CHECK_LAUNCH();
  if (S > 0) {
    hipLaunchKernelGGL(k_tree_boxes_top<T>, dim3(1), dim3(kBlock), 0, s, tree, box, n_nodes, fix_phantom, S,
                       last_node);
    CS_CHECK_LAUNCH();
  }
}

template void launch_tree_build<float>(const F4*, int, int, F4*, KV*, int, int*, KV*, KV*, int*, hipStream_t, int*);
template void launch_tree_build<double>(const D4*, int, int, D4*, KV*, int, int*, KV*, KV*, int*, hipStream_t, int*);
template void launch_tree_boxes<float>(const F4*, F4*, int, int, hipStream_t);
template void launch_tree_boxes<double>(const D4*, F4*, int, int, hipStream_t);

}  // namespace cudasph
