// Tree walks on the GPU: smoothing-length solve and neighbour lists.
//
// A walk (dev_solve_range.cu:17-75, dev_find_ngb.cu:13-73) pops a node, pushes
// its left child if the query sphere reaches below the split plane and its
// right child if it reaches above (so the right subtree is visited first),
// then tests the node's own particle.  Children are pushed for every node
// with 2p <= n_nodes, which for even n_nodes includes the nonexistent node
// n+1; the tree buffer holds a zero record there, which is what the
// reference's out-of-range texture fetch returns.  fix_phantom drops that push
// instead.
//
// With `boxes` (subtree bounding boxes, launch_tree_boxes) a child is pushed
// only if its box also comes within the range: a subtree whose box lies
// beyond it holds no neighbour, so the neighbours, their order and every sum
// over them stay the same, and only the walk length shrinks.  The test keeps
// a margin of 2^-16 of r^2 over the rounding of the box distance and of d^2.
//
// One walk is a chain of dependent tree fetches, and a lane that walks alone
// takes as long as its particle's walk: with a lane per particle both kernels
// lasted as long as their slowest lanes (a halo particle's large sphere in
// sparse space, solved by several walks).  Here 16 lanes share a particle.
// Each turn they take the top 16 nodes of the particle's stack together, so a
// walk of V nodes is about V / 16 + log2 n turns instead of V, and a wavefront
// holds 4 particles.  The order of the visits does not decide anything but the
// order of the accepted particles, and that order is the depth-first walk's
// preorder, which is a closed form of the node's heap index (walk_rank); the
// accepted records are sorted by it afterwards.  So every list, count and
// sum is that of the reference's walk, term by term in its order.
//
// Measured (solve / lists alone, ms, a lane per particle -> 16 lanes):
// 16 384 particles 0.72 / 0.24 -> 0.07 / 0.04 (plain form, no boxes: 3.9 /
// 0.71 -> 0.20 / 0.16), 65 536: 0.66 / 0.38 -> 0.17 / 0.12, 100 003 plain 2.4 /
// 1.7 -> 0.46 / 0.37, 262 144: 0.96 / 0.64 -> 0.59 / 0.42.  What bounds it
// then is VALU issue: a turn is about 125 instructions for 4 particles, of whose
// 64 lanes a part is idle.  At 2^20 particles, where a lane per particle
// fills the GPU for many rounds and its slow lanes no longer show, the shared
// walk does more work in all (2.2 / 1.3 -> 3.3 / 1.6), so there a lane walks
// alone (walk_alone).
#include "kernels.h"
#include "sph_math.h"

namespace cudasph {

template <class T>
__device__ __forceinline__ T box_dist2(const F4 lo, const F4 hi, T qx, T qy, T qz) {
  const T dx = fmax(fmax(T(lo.x) - qx, qx - T(hi.x)), T(0));
  const T dy = fmax(fmax(T(lo.y) - qy, qy - T(hi.y)), T(0));
  const T dz = fmax(fmax(T(lo.z) - qz, qz - T(hi.z)), T(0));
  return dx * dx + dy * dy + dz * dz;
}
template <class T>
__device__ __forceinline__ T range2_margin(T r2) {   // the box test's r^2 with its margin
  return r2 * T(1.0 + 1.0 / 65536.0);
}

// ---------------------------------------------------------------------------
// groups of 16 lanes: one row of the DPP network
constexpr int kWalkGroup = 16;
constexpr int kWalkCap = 96;     // records one pass of a walk may accept
constexpr int kWalkStack = 96;   // pending nodes of one pass
constexpr int kWalkRoots = 32;   // pending subtrees of a walk taken in several passes (a tree has at most 24 levels)

struct Lane {
  int l;       // lane within its group
  int shift;   // the group's first lane within the wavefront
  __device__ Lane() : l((int)threadIdx.x & 15), shift((int)threadIdx.x & 48) {}
  __device__ __forceinline__ unsigned ballot(bool p) const { return (unsigned)(__ballot(p) >> shift) & 0xffffu; }
  __device__ __forceinline__ int before(unsigned mask) const { return __popc(mask & ((1u << l) - 1u)); }
};

// lane S of the row, in every lane of the row
template <int S>
__device__ __forceinline__ int row_bcast(int v) {
  return __builtin_amdgcn_update_dpp(0, v, 0x150 + S, 0xf, 0xf, true);
}
template <int S>
__device__ __forceinline__ float row_bcast(float v) {
  return __int_as_float(row_bcast<S>(__float_as_int(v)));
}
template <int S>
__device__ __forceinline__ double row_bcast(double v) {
  return __hiloint2double(row_bcast<S>(__double2hiint(v)), row_bcast<S>(__double2loint(v)));
}

// lane l ^ X of the row
template <int X>
__device__ __forceinline__ unsigned row_xor(unsigned v) {
  const int x = (int)v;
  if constexpr (X == 1) return (unsigned)__builtin_amdgcn_update_dpp(0, x, 0xB1, 0xf, 0xf, true);
  else if constexpr (X == 2) return (unsigned)__builtin_amdgcn_update_dpp(0, x, 0x4E, 0xf, 0xf, true);
  else if constexpr (X == 4) {   // mirrored within 8 (xor 7), then within 4 (xor 3)
    const int h = __builtin_amdgcn_update_dpp(0, x, 0x141, 0xf, 0xf, true);
    return (unsigned)__builtin_amdgcn_update_dpp(0, h, 0x1B, 0xf, 0xf, true);
  } else {
    static_assert(X == 8, "");
    return (unsigned)__builtin_amdgcn_update_dpp(0, x, 0x128, 0xf, 0xf, true);   // rotated by 8
  }
}

// place of heap node id among the nodes of a perfect tree of `levels` levels
// in the walk's order (a node, its right subtree, its left subtree): each step
// to a right child passes 1 node, each step to a left child at depth j also
// the 2^(levels - j) - 1 nodes of its sibling
__device__ __forceinline__ unsigned walk_rank(unsigned id, int levels) {
  const int d = 31 - __clz((int)id);
  return ((~id & ((1u << d) - 1u)) << (levels - d)) + (unsigned)__popc(id) - 1u;
}
// levels of the heap nodes 1 .. n+1
__device__ __forceinline__ int walk_levels(int n_nodes) { return 32 - __clz(n_nodes + 1); }

// a group's share of LDS
template <class V, bool REACH>
struct WalkLds {
  V val[kWalkCap];             // the accepted records' values; in walk order once sorted
  unsigned key[kWalkCap];      // their rank in the walk's order, and the slot of val
  int stk[kWalkStack];         // pending nodes
  float reach[REACH ? kWalkStack : 1];   // ... and the path bound of each
  int roots[kWalkRoots];
};

// ascending sort of the N = 16 P keys k[r] = element l * P + r of the group
template <int P>
__device__ __forceinline__ void sort_keys(unsigned (&k)[P], int l) {
  constexpr int N = kWalkGroup * P;
#pragma unroll
  for (int size = 2; size <= N; size <<= 1) {
    // descending runs are sorted as ascending runs of the complement
    if (size >= P) {
      const unsigned flip = (l * P) & size ? ~0u : 0u;
#pragma unroll
      for (int r = 0; r < P; ++r) k[r] ^= flip;
#pragma unroll
      for (int j = size >> 1; j > 0; j >>= 1) {
        if (j >= P) {
          const bool low = (l & (j / P)) == 0;
#pragma unroll
          for (int r = 0; r < P; ++r) {
            unsigned o;
            if (j / P == 1) o = row_xor<1>(k[r]);
            else if (j / P == 2) o = row_xor<2>(k[r]);
            else if (j / P == 4) o = row_xor<4>(k[r]);
            else o = row_xor<8>(k[r]);
            k[r] = low ? min(k[r], o) : max(k[r], o);
          }
        } else {
#pragma unroll
          for (int r = 0; r < P; ++r)
            if ((r & j) == 0) {
              const unsigned a = k[r], b = k[r | j];
              k[r] = min(a, b);
              k[r | j] = max(a, b);
            }
        }
      }
#pragma unroll
      for (int r = 0; r < P; ++r) k[r] ^= flip;
    } else {
#pragma unroll
      for (int j = size >> 1; j > 0; j >>= 1)
#pragma unroll
        for (int r = 0; r < P; ++r)
          if ((r & j) == 0) {
            const unsigned a = k[r], b = k[r | j];
            const bool up = (r & size) == 0;
            k[r] = up ? min(a, b) : max(a, b);
            k[r | j] = up ? max(a, b) : min(a, b);
          }
    }
  }
}

// the n accepted records' values into walk order
template <int P, class S>
__device__ __forceinline__ void order_records_p(const Lane& g, S& s, int n) {
  unsigned k[P];
#pragma unroll
  for (int r = 0; r < P; ++r) k[r] = r * kWalkGroup + g.l < n ? s.key[r * kWalkGroup + g.l] : ~0u;
  sort_keys<P>(k, g.l);
  decltype(+s.val[0]) v[P];
#pragma unroll
  for (int r = 0; r < P; ++r) v[r] = s.val[k[r] == ~0u ? 0u : k[r] & 127u];
  lds_order();
#pragma unroll
  for (int r = 0; r < P; ++r)
    if (g.l * P + r < n) s.val[g.l * P + r] = v[r];
  lds_order();
}
template <class S>
__device__ __forceinline__ void order_records(const Lane& g, S& s, int n) {
  if (n <= 32) order_records_p<2>(g, s, n);
  else if (n <= 64) order_records_p<4>(g, s, n);
  else order_records_p<8>(g, s, n);
}

template <class T>
struct Tree {
  const V4<T>* __restrict__ node;
  const F4* __restrict__ boxes;   // or null
  int n, fix_phantom, levels;
  __device__ Tree(const V4<T>* t, const WalkParams& wp)
      : node(t), boxes(wp.boxes), n(wp.n_nodes), fix_phantom(wp.fix_phantom), levels(walk_levels(wp.n_nodes)) {}
};

template <class T>
struct Visit {
  bool left, right, in;   // push a child; accept the node's particle
  T ds2;
  int particle;
  float margin_l, margin_r;   // (REACH) distance to the split plane a push to that child crosses
};

// the tests of one node at range q.w
template <bool REACH, class T>
__device__ __forceinline__ Visit<T> visit_node(const V4<T>& q, const Tree<T>& tr, int id) {
  Visit<T> v;
  const V4<T> node = tr.node[id];
  F4 b0, b1, b2, b3;
  if (tr.boxes) {   // the children's boxes, beside the node (a leaf fetches the root's: unused)
    const int cb = 2 * id <= tr.n ? 4 * id : 4;
    b0 = tr.boxes[cb];
    b1 = tr.boxes[cb + 1];
    b2 = tr.boxes[cb + 2];
    b3 = tr.boxes[cb + 3];
  }
  const T r2 = q.w * q.w, r2m = range2_margin(r2);
  const int bits = node_bits(node.w);
  const int split = (bits >> 24) & 3;
  const int c = 2 * id;
  v.left = v.right = false;
  v.margin_l = v.margin_r = 0.f;
  if (c <= tr.n && split < 3) {
    const T qc = (split & 2) ? q.z : ((split & 1) ? q.y : q.x);
    const T nc = (split & 2) ? node.z : ((split & 1) ? node.y : node.x);
    T bl = T(0), br = T(0);
    if (tr.boxes) {
      bl = box_dist2<T>(b0, b1, q.x, q.y, q.z);
      br = box_dist2<T>(b2, b3, q.x, q.y, q.z);
    }
    v.left = qc - q.w < nc && bl <= r2m;
    v.right = qc + q.w > nc && (!tr.fix_phantom || c < tr.n) && br <= r2m;
    if constexpr (REACH) {
      v.margin_l = (float)fmax(qc - nc, T(0));
      v.margin_r = (float)fmax(nc - qc, T(0));
    }
  }
  const T dx = q.x - node.x, dy = q.y - node.y, dz = q.z - node.z;
  v.ds2 = dx * dx + dy * dy + dz * dz;
  v.in = v.ds2 < r2;
  v.particle = bits & ~(3 << 24);
  return v;
}

// One pass: the walk of the subtree of `root` at range q.w, its accepted
// records unsorted in s.key and s.val (make(visit) gives a record's value).
// Returns their number, or -1 when they or the pending nodes outgrow the
// group's LDS (nothing counted then).  n_walk grows by the nodes visited;
// phantom gets bit 0 when the walk reads node n+1 and bit 1 when it takes it.
// With REACH, reach_ok is cleared when some accepted record's path bound (the
// largest distance to a split plane that the path's pushes crossed) is not
// below its distance: the phantom, whose place is not its particle's; a tree
// whose nodes do not respect its own split planes.  (A box holds its
// subtree's particles, so the box distances on the path are below it too.)
// The bound is squared in T, where the distance is: squares of FP64 distances
// have no place in a float.  Squares so small that they lose digits decide
// nothing.
template <bool REACH, class T, class S, class Make>
__device__ __forceinline__ int walk_pass(const Lane& g, const V4<T>& q, const Tree<T>& tr, int root, S& s,
                                         int& n_walk, int& phantom, bool& reach_ok, Make&& make) {
  if (g.l == 0) {
    s.stk[0] = root;
    if (REACH) s.reach[0] = 0.f;
  }
  lds_order();
  int top = 1, n = 0, nw = 0;
  while (top > 0) {
    const int m = min(top, kWalkGroup);
    top -= m;
    nw += m;
    Visit<T> v;
    v.left = v.right = v.in = false;
    int id = 0;
    float path = 0.f;
    bool odd = false;
    if (g.l < m) {
      id = s.stk[top + m - 1 - g.l];
      if (REACH) path = s.reach[top + m - 1 - g.l];
      v = visit_node<REACH, T>(q, tr, id);
      if (id == tr.n + 1) phantom |= v.in ? 3 : 1;
      // rounding of the margins and of ds2: below 2^-18
      constexpr T kTiny = sizeof(T) == 4 ? T(1e-30) : T(1e-60);
      if (REACH)
        odd = v.in && path > 0.f && !((T)path * (T)path <= v.ds2 * T(1.00001) && v.ds2 >= kTiny);
    }
    if (REACH && g.ballot(odd)) reach_ok = false;
    const unsigned bl = g.ballot(v.left), br = g.ballot(v.right), ba = g.ballot(v.in);
    if (v.left) {
      const int p = top + g.before(bl);
      s.stk[p] = 2 * id;
      if (REACH) s.reach[p] = fmaxf(path, v.margin_l);
    }
    top += __popc(bl);
    if (v.right) {
      const int p = top + g.before(br);
      s.stk[p] = 2 * id + 1;
      if (REACH) s.reach[p] = fmaxf(path, v.margin_r);
    }
    top += __popc(br);
    const int na = __popc(ba);
    if (n + na > kWalkCap || top > kWalkStack - kWalkGroup) return -1;
    if (v.in) {
      const int p = n + g.before(ba);
      s.key[p] = (walk_rank((unsigned)id, tr.levels) << 7) | (unsigned)p;
      s.val[p] = make(v);
    }
    n += na;
    lds_order();
  }
  n_walk += nw;
  return n;
}
static_assert(kWalkCap <= 1 << 7, "the slot's bits in a key");
static_assert(kWalkStack >= 3 * kWalkGroup, "a turn takes 16 nodes and pushes up to 32");

// The whole walk at range q.w: take(n) is called with the next n records in
// walk order in s.val, one or more times.  A subtree that outgrows a pass is
// split: its root is taken alone, then its right subtree, then its left one.
template <class T, class S, class Make, class Take>
__device__ __forceinline__ int walk_all(const Lane& g, const V4<T>& q, const Tree<T>& tr, S& s, int& phantom,
                                        Make&& make, Take&& take) {
  int n_walk = 0, roots = 0, root = 1;
  bool unused = true;
  for (;;) {
    const int n = walk_pass<false, T>(g, q, tr, root, s, n_walk, phantom, unused, make);
    if (n >= 0) {
      order_records(g, s, n);
      take(n);
    } else {   // every lane of the group the same node
      const Visit<T> v = visit_node<false, T>(q, tr, root);
      ++n_walk;
      if (root == tr.n + 1) phantom |= v.in ? 3 : 1;
      lds_order();
      if (g.l == 0) {
        if (v.left) s.roots[roots] = 2 * root;
        if (v.right) s.roots[roots + (v.left ? 1 : 0)] = 2 * root + 1;
        s.val[0] = make(v);
      }
      roots += (v.left ? 1 : 0) + (v.right ? 1 : 0);
      lds_order();
      if (v.in) take(1);
    }
    if (roots == 0) return n_walk;
    lds_order();
    root = s.roots[--roots];
    lds_order();
  }
}

// ---------------------------------------------------------------------------
// smoothed count minus target, Newton step and integer count of one
// evaluation (dev_solve_range.cu:17-89), its terms added in walk order
template <class T>
struct NgbEval {
  T f, step, count;
};

template <class T>
struct NgbSum {
  T f = T(0), df = T(0);
  int count = 0;
  // one record inside the range
  __device__ __forceinline__ void one(T ds2, T r) {
    const T u = T(2) * dsqrt(ds2) / r;
    f += kern_ig<T>(u);
    df -= kern_digdh<T>(u);
    ++count;
  }
  // records val[0 .. n), those with ds2 < r2; returns whether one of them
  // lies at or beyond sure2.  16 terms at a time are computed side by side and
  // then added one after another; a record outside adds zero, which changes
  // no bit of the sums
  __device__ __forceinline__ bool add(const Lane& g, const T* val, int n, T r, T r2, T sure2) {
    bool close = false;
    for (int e0 = 0; e0 < n; e0 += kWalkGroup) {
      T ig = T(0), dg = T(0);
      bool in = false;
      if (e0 + g.l < n) {
        const T ds2 = val[e0 + g.l];
        in = ds2 < r2;
        if (in) {
          const T u = T(2) * dsqrt(ds2) / r;
          ig = kern_ig<T>(u);
          dg = kern_digdh<T>(u);
          close |= !(ds2 < sure2);
        }
      }
      count += __popc(g.ballot(in));
      serial<0>(ig, dg);
    }
    return g.ballot(close) != 0;
  }
  template <int S>
  __device__ __forceinline__ void serial(T ig, T dg) {
    if constexpr (S < kWalkGroup) {
      f += row_bcast<S>(ig);
      df -= row_bcast<S>(dg);
      serial<S + 1>(ig, dg);
    }
  }
  __device__ __forceinline__ NgbEval<T> finish(T range, float desired_ngb) {
    f -= T(desired_ngb);
    df = T((double)df * (1.0 / (double)range));
    if (df != T(0)) df = f / df;
    else df = f < T(0) ? -range : range;
    return {f, df, T(count)};
  }
};

// The evaluations of one particle's solve.  The first walks at 17/16 of its
// range and keeps the distances accepted there, in walk order; a later one at
// r <= that range takes the kept distances below r.  That is the walk at r
// if every one of them is reached by it.  A record's path bound (the
// largest margin by which the path's pushes needed the range) is below its
// distance (checked when it was kept, reach_ok), so a walk at r reaches it
// when r exceeds its distance by more than the rounding of the push tests,
// fl(qc -+ r) against nc: at most 2^-24 (|qc| + r) (2^-53 in FP64), taken 32 times over.  If
// a distance lies closer to r than that, the evaluation walks at r instead.
constexpr double kWide = 1.0625;
template <class T>
struct Solver {
  const Lane g;
  const Tree<T> tr;
  const WalkParams& wp;
  WalkLds<T, true>& s;
  T pad;               // the rounding allowance at r = 0
  int n = -1;          // records kept, -1: none
  T radius = T(0);     // ... of a walk at this range
  bool full = false;   // the records of a walk at kWide full_at outgrew the group's share
  T full_at = T(0);
  __device__ Solver(const V4<T>& q, const V4<T>* tree, const WalkParams& w, WalkLds<T, true>& lds)
      : tr(tree, w), wp(w), s(lds) {
    constexpr T eps = sizeof(T) == 4 ? T(1.0 / 16777216.0) : T(1.0 / 9007199254740992.0);
    pad = T(32) * eps * fmax(fmax(dabs(q.x), dabs(q.y)), dabs(q.z));
  }
  __device__ __forceinline__ NgbEval<T> eval(const V4<T>& q) {
    constexpr T eps = sizeof(T) == 4 ? T(1.0 / 16777216.0) : T(1.0 / 9007199254740992.0);
    const T r = q.w, r2 = r * r;
    int nw = 0, ph = 0;
    const auto make = [](const Visit<T>& v) { return v.ds2; };
    if (wp.solve_cache && (n < 0 || r > radius) && !(full && r >= full_at)) {
      V4<T> wide = q;
      wide.w = r * T(kWide);
      bool ok = true;
      n = walk_pass<true, T>(g, wide, tr, 1, s, nw, ph, ok, make);
      radius = wide.w;
      if (n < 0) {
        full = true;
        full_at = r;
      }
      if (n >= 0 && ok) order_records(g, s, n);
      else n = -1;
    }
    if (n >= 0) {
      // 2^-15: the slack of the path bound against the distance
      const T sure = (r - (pad + T(32) * eps * r)) * T(1.0 - 1.0 / 32768.0);
      NgbSum<T> sum;
      if (!sum.add(g, s.val, n, r, r2, sure > T(0) ? sure * sure : T(0))) return sum.finish(r, wp.desired_ngb);
      n = -1;
    }
    NgbSum<T> sum;
    walk_all<T>(g, q, tr, s, ph, make, [&](int m) { sum.add(g, s.val, m, r, r2, r2); });
    return sum.finish(r, wp.desired_ngb);
  }
};

template <class T>
__device__ __forceinline__ T clamp_step(T dx, T range) {   // f_scale = 0.1, dev_solve_range.cu:92,100-103
  if ((double)dabs(dx) > 0.1 * (double)range) dx = T((dx < T(0) ? -0.1 : 0.1) * (double)range);
  return dx;
}

// bracket [lo, hi] around the target (dev_solve_range.cu:93-135); z = count
template <class T, class S>
__device__ __forceinline__ V4<T> bracket(V4<T> q, S& s) {
  const T rel = T(s.wp.rel_err);
  NgbEval<T> f = s.eval(q);
  T dx = f.step;
  if (dabs(dx) < rel * q.w)
    return {T((double)q.w - 0.5 * (double)dabs(dx)), T((double)q.w + 0.5 * (double)dabs(dx)), f.count, T(0)};
  dx = clamp_step<T>(dx, q.w);
  T x_prev = q.w, f_prev = f.f;
  int iter = 0;
  while ((f_prev * f.f >= T(0)) && (iter++ < s.wp.max_iter)) {
    x_prev = q.w;
    f_prev = f.f;
    q.w -= dx;
    f = s.eval(q);
    dx = f.step;
    if (dabs(dx) < rel * q.w)
      return {T((double)q.w - 0.5 * (double)dabs(dx)), T((double)q.w + 0.5 * (double)dabs(dx)), f.count, T(0)};
    dx = clamp_step<T>(dx, q.w);
  }
  if (x_prev < q.w) return {x_prev, q.w, f.count, T(0)};
  return {q.w, x_prev, f.count, T(0)};
}

// safeguarded Newton inside the bracket (dev_solve_range.cu:137-172)
template <class T, class S>
__device__ __forceinline__ void solve_range(V4<T> q, S& s, T& range, T& count) {
  const T rel = T(s.wp.rel_err);
  const V4<T> br = bracket<T, S>(q, s);
  T lo = br.x, hi = br.y;
  count = br.z;
  q.w = T(0.5 * (double)(lo + hi));
  T dx = T(0);
  if (dabs(lo - hi) > rel * q.w) {
    bool keep = true;
    int iter = 0;
    while (keep && (iter++ < s.wp.max_iter)) {
      q.w -= dx;
      if ((q.w - hi) * (q.w - lo) >= T(0)) {          // left the bracket: bisect
        dx = T(0.5 * (double)(hi - lo));
        q.w = T(0.5 * (double)(lo + hi));
      }
      const NgbEval<T> f = s.eval(q);
      count = f.count;
      if (f.f < T(0)) lo = q.w;
      else hi = q.w;
      dx = f.step;
      keep = dabs(dx) > rel * q.w;
    }
  }
  range = q.w;
}

// dev_solve_range.cu:174-189
template <class T>
__global__ __launch_bounds__(kBlock) void k_solve_range(V4<T>* __restrict__ pos, int* __restrict__ n_ngb,
                                                         const KV* __restrict__ hash,
                                                         const V4<T>* __restrict__ tree, int n_dev,
                                                         WalkParams wp) {
  chain_priority();
  extern __shared__ __align__(16) char s_mem[];   // WalkLds<T, true> per group
  WalkLds<T, true>& s = reinterpret_cast<WalkLds<T, true>*>(s_mem)[threadIdx.x / kWalkGroup];
  const int t = (xcd_block(blockIdx.x, gridDim.x) * (int)blockDim.x + (int)threadIdx.x) / kWalkGroup;
  if (t >= n_dev) return;   // whole groups leave together
  const int i = (int)hash[t].value;
  const V4<T> q = pos[i];
  T range = T(0), count = T(0);
  if (q.w > T(0)) {
    Solver<T> solver(q, tree, wp, s);
    solve_range<T, Solver<T>>(q, solver, range, count);
  }
  if (threadIdx.x % kWalkGroup == 0) {
    pos[i].w = range;
    n_ngb[i] = (int)count;
  }
}

// Whether the lists' total, offset[n_dev], exceeds their allocation of list_cap
// slots (list_cap < 0: not asked, offset then has no such entry).  The launch
// reports the total in flags[3] and then writes nothing, so the walk can be
// queued before the host has seen the total.
__device__ __forceinline__ bool list_overflow(const int* __restrict__ offset, int n_dev, int list_cap,
                                              int* __restrict__ flags) {
  if (list_cap < 0) return false;
  const int total = offset[n_dev];
  if (blockIdx.x == 0 && threadIdx.x == 0) flags[3] = total;
  return total < 0 || total > list_cap;
}

// dev_find_ngb.cu:75-87.  Capacity of particle i's slot is
// n_norm(cap_count[i], 4) (the layout of sph_accelerations.cpp:58-64); at most
// that many ids are written, the true count goes to count_out[i], and
// flags[0] is raised when a count exceeds its slot; flags[1] and flags[2]
// count the walks that read node n+1 and that took it as a neighbour.  With
// clamp set, count_out is clamped to the slot (for callers that own the
// offsets).  flags holds at least 3 ints, zeroed by the caller.
template <class T>
__global__ __launch_bounds__(kBlock) void k_find_ngb(const V4<T>* __restrict__ pos, const V4<T>* __restrict__ tree,
                                                      KV* __restrict__ hash, const int* __restrict__ offset,
                                                      const int* cap_count, int* count_out,
                                                      int* __restrict__ list, int* __restrict__ flags,
                                                      int n_dev, WalkParams wp, int clamp, int list_cap) {
  chain_priority();
  if (list_overflow(offset, n_dev, list_cap, flags)) return;
  extern __shared__ __align__(16) char s_mem[];   // WalkLds<int, false> per group
  WalkLds<int, false>& s = reinterpret_cast<WalkLds<int, false>*>(s_mem)[threadIdx.x / kWalkGroup];
  const int t = (xcd_block(blockIdx.x, gridDim.x) * (int)blockDim.x + (int)threadIdx.x) / kWalkGroup;
  if (t >= n_dev) return;   // whole groups leave together
  const Lane g;
  const int i = (int)hash[t].value;
  const V4<T> q = pos[i];
  const int off = offset[i];
  const int cap = n_norm(cap_count[i], 4);
  const Tree<T> tr(tree, wp);
  int c = 0, ph = 0;
  const int nw = walk_all<T>(
      g, q, tr, s, ph, [](const Visit<T>& v) { return v.particle; },
      [&](int n) {
        for (int e = g.l; e < n; e += kWalkGroup)
          if (c + e < cap) list[off + c + e] = s.val[e];
        c += n;
      });
  const unsigned read = g.ballot(ph & 1), taken = g.ballot(ph & 2);
  if (g.l != 0) return;
  hash[t].key = (uint32_t)nw;
  if (read) atomicAdd(flags + 1, 1);    // walks that read node n+1 (rare: a few per tree)
  if (taken) atomicAdd(flags + 2, 1);   // ... and took it as a neighbour
  if (c > cap) {
    atomicOr(flags, 1);
    if (clamp) c = cap;
  }
  count_out[i] = c;
}

// ---------------------------------------------------------------------------
// a lane per particle

// the walk at range q.w, its stack in LDS, one column per lane of the block;
// visit(v) for each accepted node.  Returns the number of nodes visited.
template <class T, class F>
__device__ __forceinline__ int lane_walk(const V4<T>& q, const Tree<T>& tr, int* __restrict__ stk, int& phantom,
                                         F&& visit) {
  const int stride = (int)blockDim.x;
  int top = 0, n_walk = 0;
  stk[0] = 1;
  while (top >= 0) {
    ++n_walk;
    const int id = stk[top * stride];
    const Visit<T> v = visit_node<false, T>(q, tr, id);
    if (v.left) stk[(top++) * stride] = 2 * id;
    if (v.right) stk[(top++) * stride] = 2 * id + 1;
    --top;
    if (v.in) visit(v);
    if (id == tr.n + 1) phantom |= v.in ? 3 : 1;
  }
  return n_walk;
}

template <class T>
struct LaneSolver {
  const Tree<T> tr;
  const WalkParams& wp;
  int* stk;
  __device__ __forceinline__ NgbEval<T> eval(const V4<T>& q) {
    NgbSum<T> sum;
    int ph = 0;
    lane_walk<T>(q, tr, stk, ph, [&](const Visit<T>& v) { sum.one(v.ds2, q.w); });
    return sum.finish(q.w, wp.desired_ngb);
  }
};

template <class T>
__global__ __launch_bounds__(kBlock) void k_solve_range_lane(V4<T>* __restrict__ pos, int* __restrict__ n_ngb,
                                                              const KV* __restrict__ hash,
                                                              const V4<T>* __restrict__ tree, int n_dev,
                                                              WalkParams wp) {
  chain_priority();
  extern __shared__ int s_stack[];   // walk_stack_depth(n_nodes) entries per lane
  const int t = xcd_block(blockIdx.x, gridDim.x) * (int)blockDim.x + threadIdx.x;
  if (t >= n_dev) return;
  const int i = (int)hash[t].value;
  const V4<T> q = pos[i];
  T range = T(0), count = T(0);
  if (q.w > T(0)) {
    LaneSolver<T> solver{Tree<T>(tree, wp), wp, s_stack + threadIdx.x};
    solve_range<T, LaneSolver<T>>(q, solver, range, count);
  }
  pos[i].w = range;
  n_ngb[i] = (int)count;
}

// as k_find_ngb
template <class T>
__global__ __launch_bounds__(kBlock) void k_find_ngb_lane(const V4<T>* __restrict__ pos,
                                                           const V4<T>* __restrict__ tree, KV* __restrict__ hash,
                                                           const int* __restrict__ offset, const int* cap_count,
                                                           int* count_out, int* __restrict__ list,
                                                           int* __restrict__ flags, int n_dev, WalkParams wp,
                                                           int clamp, int list_cap) {
  chain_priority();
  if (list_overflow(offset, n_dev, list_cap, flags)) return;
  extern __shared__ int s_stack[];   // walk_stack_depth(n_nodes) entries per lane
  const int t = xcd_block(blockIdx.x, gridDim.x) * (int)blockDim.x + threadIdx.x;
  if (t >= n_dev) return;
  const int i = (int)hash[t].value;
  const V4<T> q = pos[i];
  const int off = offset[i];
  const int cap = n_norm(cap_count[i], 4);
  // ids go out four at a time as one 16-byte store when the slot run is
  // 16-byte aligned (offsets are multiples of 4 in the reference layout): a
  // wavefront's lanes write 64 different lists, so a 4-byte store per id
  // would dirty a cache line per lane per id
  const bool vec = (off & 3) == 0 && (reinterpret_cast<uintptr_t>(list) & 15) == 0;
  int c = 0, ph = 0;
  int b0 = 0, b1 = 0, b2 = 0;   // the current group's first three ids
  const int nw = lane_walk<T>(q, Tree<T>(tree, wp), s_stack + threadIdx.x, ph, [&](const Visit<T>& v) {
    const int id = v.particle, r = c & 3;
    if (vec) {
      if (r == 3) {
        if (c < cap) *reinterpret_cast<int4*>(list + off + c - 3) = make_int4(b0, b1, b2, id);
      } else {
        b0 = r == 0 ? id : b0;
        b1 = r == 1 ? id : b1;
        b2 = r == 2 ? id : b2;
      }
    } else if (c < cap) {
      list[off + c] = id;
    }
    ++c;
  });
  if (vec) {   // the last, partial group (slots past the count stay untouched)
    const int g = c & ~3, r = c & 3;
    if (r > 0 && g < cap) {
      list[off + g] = b0;
      if (r > 1) list[off + g + 1] = b1;
      if (r > 2) list[off + g + 2] = b2;
    }
  }
  hash[t].key = (uint32_t)nw;
  if (ph & 1) atomicAdd(flags + 1, 1);
  if (ph & 2) atomicAdd(flags + 2, 1);
  if (c > cap) {
    atomicOr(flags, 1);
    if (clamp) c = cap;
  }
  count_out[i] = c;
}

// A lane walks alone where its longer chain is hidden by many rounds of
// others: from 2^19 particles on, and for long lists earlier.  A walk of more
// than kWalkCap records takes several passes, parts of which are walked twice:
// the first walk of an h-solve takes 1.2 times the list, so from a target of 42
// (lists of 59) on a growing part of them do.  Solve + lists, ms, 16 lanes / one lane:
//   target, particles        turbulent sphere   polytropes FP64   Plummer sphere
//   45.2 (64)   131 072       0.80 / 1.13        1.30 / 1.74       1.00 / 2.80
//               262 144       1.51 / 1.61        2.46 / 2.66       1.80 / 4.15
//               327 680       1.88 / 1.88        2.93 / 2.95       2.14 / 4.25
//   50 (72)      98 304       0.81 / 1.16        1.35 / 1.83       1.10 / 2.81
//               131 072       1.15 / 1.21        2.02 / 1.88       1.38 / 2.99
//               262 144       2.35 / 1.68        3.73 / 2.69       2.66 / 4.11
//   57 (82)      65 536       1.11 / 1.27        1.47 / 1.50       1.31 / 2.64
//                98 304       1.50 / 1.25        2.14 / 1.90       1.72 / 2.81
//   62 (89)      65 536       1.49 / 1.30        2.29 / 1.60       1.86 / 2.66
//               262 144       6.48 / 1.91       10.5  / 2.86       7.17 / 4.37
// so the two are even where particles * (target - 42) is about 2^20, but for the
// Plummer sphere, whose halo keeps single lanes long.  (A solve started far
// from its range, with some thousand records in its first walks, is not
// foreseen by this: 3 times off at 262 144 particles, 97 / 21 ms in the sphere,
// 168 / 277 in the Plummer sphere, once in a run.)
static bool walk_alone(int n_dev, const WalkParams& wp) {
  constexpr int kMin = 1 << 16, kAlways = 1 << 19;
  return n_dev >= kAlways || (n_dev >= kMin && n_dev * ((double)wp.desired_ngb - 42.0) >= 1 << 20);
}

// threads per block of the walks: one wavefront while there are few
// particles, so that they spread over every CU
static int walk_block(int n_dev) { return n_dev < 512 * kBlock ? 64 : kBlock; }

template <class T>
void launch_solve_range(V4<T>* pos, int* n_ngb, const KV* hash, const V4<T>* tree, int n_dev,
                        const WalkParams& wp, hipStream_t s) {
  const int bs = walk_block(n_dev);
  if (walk_alone(n_dev, wp)) {
    const size_t lds = (size_t)walk_stack_depth(wp.n_nodes) * bs * sizeof(int);
    hipLaunchKernelGGL(k_solve_range_lane<T>, dim3(ceil_div(n_dev, bs)), dim3(bs), lds, s, pos, n_ngb, hash, tree,
                       n_dev, wp);
  } else {
    const int per = bs / kWalkGroup;
    hipLaunchKernelGGL(k_solve_range<T>, dim3(ceil_div(n_dev, per)), dim3(bs), per * sizeof(WalkLds<T, true>), s, pos,
                       n_ngb, hash, tree, n_dev, wp);
  }
  CS_CHECK_LAUNCH();
}

template <class T>
void launch_find_ngb(const V4<T>* pos, const V4<T>* tree, KV* hash, const int* offset, const int* cap_count,
                     int* count_out, int* list, int* flags, int n_dev, const WalkParams& wp, int clamp, int list_cap,
                     hipStream_t s) {
  const int bs = walk_block(n_dev);
  if (walk_alone(n_dev, wp)) {
    const size_t lds = (size_t)walk_stack_depth(wp.n_nodes) * bs * sizeof(int);
    hipLaunchKernelGGL(k_find_ngb_lane<T>, dim3(ceil_div(n_dev, bs)), dim3(bs), lds, s, pos, tree, hash, offset,
                       cap_count, count_out, list, flags, n_dev, wp, clamp, list_cap);
  } else {
    const int per = bs / kWalkGroup;
    hipLaunchKernelGGL(k_find_ngb<T>, dim3(ceil_div(n_dev, per)), dim3(bs), per * sizeof(WalkLds<int, false>), s, pos,
                       tree, hash, offset, cap_count, count_out, list, flags, n_dev, wp, clamp, list_cap);
  }
  CS_CHECK_LAUNCH();
}

#define CS_INST(T)                                                                                        \
  template void launch_solve_range<T>(V4<T>*, int*, const KV*, const V4<T>*, int, const WalkParams&,      \
                                      hipStream_t);                                                       \
  template void launch_find_ngb<T>(const V4<T>*, const V4<T>*, KV*, const int*, const int*, int*, int*,   \
                                   int*, int, const WalkParams&, int, int, hipStream_t);
CS_INST(float)
CS_INST(double)
#undef CS_INST

}  // namespace cudasph
