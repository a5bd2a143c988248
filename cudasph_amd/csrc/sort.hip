// Device-wide primitives: exclusive scan, stable LSD radix sort of
// (key,value) records, the counting-sort transpose that turns the i-side
// neighbour lists into j-side reaction lists, and Peano-Hilbert keys.
#include <algorithm>

#include "kernels.h"

namespace cudasph {

constexpr int kScanBlock = 256;
constexpr int kScanItems = 8;
constexpr int kScanTile = kScanBlock * kScanItems;   // 2048

__device__ __forceinline__ int scan_load(const int* in, long idx, long n, int mode) {
  if (idx >= n) return 0;
  const int v = in[idx];
  return mode == 1 ? n_norm(v, 4) : v;
}

// block-wide exclusive scan of one value per thread; returns the block total
__device__ __forceinline__ int block_exclusive_scan(int v, int* s_tmp, int& total) {
  const int tid = threadIdx.x;
  s_tmp[tid] = v;
  __syncthreads();
  for (int off = 1; off < kScanBlock; off <<= 1) {
    const int add = tid >= off ? s_tmp[tid - off] : 0;
    __syncthreads();
    s_tmp[tid] += add;
    __syncthreads();
  }
  const int incl = s_tmp[tid];
  total = s_tmp[kScanBlock - 1];
  __syncthreads();
  return incl - v;
}

__global__ __launch_bounds__(kScanBlock) void k_scan_reduce(const int* __restrict__ in, long n, int mode,
                                                             int* __restrict__ partial) {
  chain_priority();
  __shared__ int s_tmp[kScanBlock];
  const long base = (long)blockIdx.x * kScanTile + (long)threadIdx.x * kScanItems;
  int sum = 0;
  for (int k = 0; k < kScanItems; ++k) sum += scan_load(in, base + k, n, mode);
  int total;
  block_exclusive_scan(sum, s_tmp, total);
  if (threadIdx.x == 0) partial[blockIdx.x] = total;
}

// each block adds the tiles before its own itself (a few loads per lane; a
// launch of one block in between cost more)
__global__ __launch_bounds__(kScanBlock) void k_scan_down(const int* __restrict__ in, long n, int mode,
                                                           const int* __restrict__ partial, int* __restrict__ out) {
  chain_priority();
  __shared__ int s_tmp[kScanBlock], s_before[kScanBlock / 64];
  const long base = (long)blockIdx.x * kScanTile + (long)threadIdx.x * kScanItems;
  int v[kScanItems];
  int sum = 0, before = 0;
  for (int t = threadIdx.x; t < (int)blockIdx.x; t += kScanBlock) before += partial[t];
  for (int o = 32; o > 0; o >>= 1) before += __shfl_xor(before, o);
  if ((threadIdx.x & 63) == 0) s_before[threadIdx.x >> 6] = before;
  for (int k = 0; k < kScanItems; ++k) {
    v[k] = scan_load(in, base + k, n, mode);
    sum += v[k];
  }
  int total;
  int run = block_exclusive_scan(sum, s_tmp, total);   // (its barriers publish s_before)
  for (int w = 0; w < kScanBlock / 64; ++w) {
    run += s_before[w];
    total += s_before[w];
  }
  for (int k = 0; k < kScanItems; ++k) {
    if (base + k < n) out[base + k] = run;
    run += v[k];
  }
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) out[n] = total;
}

long scan_scratch_ints(long n) { return (n + kScanTile - 1) / kScanTile + 1; }

void launch_exclusive_scan(const int* in, int* out, long n, int mode, int* scratch, hipStream_t s) {
  const int n_part = (int)((n + kScanTile - 1) / kScanTile);
  if (n_part == 0) {
    CS_HIP(hipMemsetAsync(out, 0, sizeof(int), s));
    return;
  }
  hipLaunchKernelGGL(k_scan_reduce, dim3(n_part), dim3(kScanBlock), 0, s, in, n, mode, scratch);
  CS_CHECK_LAUNCH();
  hipLaunchKernelGGL(k_scan_down, dim3(n_part), dim3(kScanBlock), 0, s, in, n, mode, scratch, out);
  CS_CHECK_LAUNCH();
}

// ---------------------------------------------------------------------------
// Radix sort (replaces the reference's RadixSort, radixsort.cu:50-77): stable,
// least significant digit first, 8 bits a pass, one launch and one reading
// and writing of the records per pass.
//
// The digit counts of all passes are taken in one reading of the keys (they
// do not depend on the order).  In a pass a block sorts a tile of 4096
// records by its digit: each wavefront ranks its 256 records by matching
// digits with ballots, the block's digit counts come from the wavefronts'
// in order, and the tile goes out through LDS in runs of equal digits.
// Where a tile's run of digit d starts is the count of smaller digits plus
// that of d in earlier tiles.  For the latter the tiles publish their digit
// counts in a table and look back over it (decoupled look-back, Merrill and
// Garland): an entry says whether it holds the tile's own count or already
// the sum over all tiles up to it, and a tile adds earlier ones' counts until
// it meets a sum.  An entry is 0 until it is published, then the count + 1 (at
// most 4097) or the sum + 4098: 32 bits hold sums up to 2^31 - 1.  Tiles take their number from a counter as they start, so a
// tile waits only for ones that are running, and those publish before they
// wait.  A pass uses one of two tables and clears its part of the other for
// the next.  The wait is bounded all the same: a thread that has looked often
// enough counts the digits of the missing tile in its records.
//
// Bound: the records in and out (16 B a pass and record) for many records,
// the chain of launches for few.  1 000 003 records, 4 passes: 137 us with a
// histogram, a scan of 3 launches and a scatter per pass -> 79 us, of which the
// four passes take about 17 each: 245 tiles on 256 CUs are one chain of loads,
// ranks, look-back and stores.
constexpr int kRadixBlock = 1024;
constexpr int kRadixItems = 4;
constexpr int kRadixTile = kRadixBlock * kRadixItems;   // records per block
constexpr int kRadixMaxPasses = 8;
constexpr unsigned kCountBase = 1, kSumBase = kRadixTile + 2;   // what an entry's count, or sum, is above
// looks at the table before a thread counts an earlier tile's records itself
// (seconds; an earlier tile that never publishes can only mean that another
// sort uses the same scratch)
constexpr int kRadixMaxPolls = 1 << 22;

// scratch of one sort: digit counts of each pass, the tile counter of each
// pass, two tables of 256 entries per tile
__host__ __device__ __forceinline__ long radix_tiles(long n) { return (n + kRadixTile - 1) / kRadixTile; }
long radix_scratch_ints(long n) { return radix_header_ints + 2 * 256 * radix_tiles(n); }
static_assert(radix_header_ints >= kRadixMaxPasses * 257, "counts and counters");

// zero the header and the first table
__global__ __launch_bounds__(kBlock) void k_radix_clear(int* __restrict__ scratch, long count, long stride) {
  const long t = (long)blockIdx.x * kBlock + threadIdx.x;
  if (t < count) scratch[blockIdx.y * stride + t] = 0;
}
long radix_clear_ints(long n) { return radix_header_ints + 256 * radix_tiles(n); }

// adds the digit counts of 4 keys' worth of passes for one record
__device__ __forceinline__ void count_digits(int (*s_hist)[256], uint32_t key, int first, int passes) {
  for (int p = 0; p < passes; ++p) atomicAdd(&s_hist[first + p][(key >> (8 * p)) & 255], 1);
}

__global__ __launch_bounds__(kRadixBlock) void k_radix_count(const KV* __restrict__ in, long n, int passes,
                                                              int* __restrict__ scratch) {
  __shared__ int s_hist[4][256];
  (&s_hist[0][0])[threadIdx.x] = 0;
  __syncthreads();
  for (int r = 0; r < kRadixItems; ++r) {
    const long p = (long)blockIdx.x * kRadixTile + r * kRadixBlock + threadIdx.x;
    if (p < n) count_digits(s_hist, in[p].key, 0, passes);
  }
  __syncthreads();
  const int c = (&s_hist[0][0])[threadIdx.x];
  if (c && (int)threadIdx.x < passes * 256) atomicAdd(&scratch[threadIdx.x], c);
}

// records of digit d in the tiles 0 .. t, those of an unpublished tile counted
// one by one (an earlier tile is full)
template <class Rekey>
__device__ __forceinline__ unsigned count_earlier(const KV* in, long t, int shift, int d, const unsigned* table,
                                               Rekey rekey) {
  unsigned sum = 0;
  for (; t >= 0; --t) {
    const unsigned v = __hip_atomic_load(&table[t * 256 + d], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (v >= kSumBase) return sum + v - kSumBase;
    if (v >= kCountBase) {
      sum += v - kCountBase;
      continue;
    }
    for (long q = t * kRadixTile; q < (t + 1) * kRadixTile; ++q) sum += (int)((rekey(in[q]).key >> shift) & 255) == d;
  }
  return sum;
}

// rekey(record) may replace a record's key as it is read; out_ids, if given,
// receives the values alone
template <class Rekey>
__device__ __forceinline__ void radix_pass(const KV* __restrict__ in, KV* __restrict__ out, int* __restrict__ out_ids,
                                           long n, int shift, int pass, int* __restrict__ scratch, int max_polls,
                                           Rekey&& rekey) {
  __shared__ int s_cnt[kRadixBlock / 64][256];   // per wavefront and digit: count, then first place
  __shared__ KV s_rec[kRadixTile];
  __shared__ int s_local[256], s_out[256];       // a digit's first place in the tile; its run's place in `out`, less that
  __shared__ int s_tot[2][4];
  __shared__ int s_tile;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const long tiles = radix_tiles(n);
  int* hist = scratch + pass * 256;
  int* counter = scratch + kRadixMaxPasses * 256 + pass;
  unsigned* table = reinterpret_cast<unsigned*>(scratch + radix_header_ints) + (pass & 1) * 256 * tiles;
  unsigned* other = reinterpret_cast<unsigned*>(scratch + radix_header_ints) + ((pass & 1) ^ 1) * 256 * tiles;
  if (tid == 0) s_tile = atomicAdd(counter, 1);
  for (int q = tid; q < kRadixBlock / 64 * 256; q += kRadixBlock) (&s_cnt[0][0])[q] = 0;
  __syncthreads();
  const long tile = s_tile, base = tile * kRadixTile;
  if (tile >= tiles) return;   // (a counter shared with another sort)
  const int cnt = (int)(n - base < kRadixTile ? n - base : kRadixTile);
  KV rec[kRadixItems];
  int rank[kRadixItems];
#pragma unroll
  for (int r = 0; r < kRadixItems; ++r) {
    const int q = wave * 64 * kRadixItems + r * 64 + lane;
    rec[r] = q < cnt ? rekey(in[base + q]) : KV{0u, 0u};
  }
#pragma unroll
  for (int r = 0; r < kRadixItems; ++r) {
    const bool valid = wave * 64 * kRadixItems + r * 64 + lane < cnt;
    const int d = (int)((rec[r].key >> shift) & 255);
    unsigned long long same = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const bool bit = (d >> b) & 1;
      const unsigned long long m = __ballot(valid && bit);
      same &= bit ? m : ~m;
    }
    const int below = __popcll(same & ((1ull << lane) - 1ull));
    const int before = s_cnt[wave][d];
    rank[r] = before + below;
    __builtin_amdgcn_wave_barrier();
    if (valid && below == 0) s_cnt[wave][d] = before + __popcll(same);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }
  __syncthreads();
  int total = 0, excl = 0, smaller = 0;
  if (tid < 256) {   // digit tid
    for (int w = 0; w < kRadixBlock / 64; ++w) {
      const int c = s_cnt[w][tid];
      s_cnt[w][tid] = total;
      total += c;
    }
    __hip_atomic_store(&table[tile * 256 + tid], (tile == 0 ? kSumBase : kCountBase) + (unsigned)total,
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    other[tile * 256 + tid] = 0;
    // exclusive sums over the digits: of the tile's counts, of all records'
    int x = total, y = hist[tid];
    const int y0 = y;
    for (int o = 1; o < 64; o <<= 1) {
      const int ux = __shfl_up(x, o), uy = __shfl_up(y, o);
      if (lane >= o) {
        x += ux;
        y += uy;
      }
    }
    if (lane == 63) {
      s_tot[0][wave] = x;
      s_tot[1][wave] = y;
    }
    excl = x - total;
    smaller = y - y0;
  }
  __syncthreads();
  if (tid < 256) {
    for (int w = 0; w < wave; ++w) {
      excl += s_tot[0][w];
      smaller += s_tot[1][w];
    }
    s_local[tid] = excl;
    unsigned earlier = 0;
    int polls = 0;
    long t = tile - 1;
    while (t >= 0) {
      constexpr int kAhead = 4;   // entries read together
      unsigned v[kAhead];
#pragma unroll
      for (int k = 0; k < kAhead; ++k)
        v[k] = t - k >= 0 ? __hip_atomic_load(&table[(t - k) * 256 + tid], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                          : kSumBase;
      bool done = false;
#pragma unroll
      for (int k = 0; k < kAhead; ++k) {
        if (done || v[k] < kCountBase) break;   // not published: read again from here
        earlier += v[k] - kCountBase;
        done = v[k] >= kSumBase;
        --t;
      }
      if (done) earlier -= kSumBase - kCountBase;
      if (done || ++polls > max_polls) break;
    }
    if (polls > max_polls) earlier += count_earlier(in, t, shift, tid, table, rekey);
    if (tile > 0)
      __hip_atomic_store(&table[tile * 256 + tid], kSumBase + earlier + (unsigned)total, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    s_out[tid] = smaller + (int)earlier - excl;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kRadixItems; ++r) {
    const int d = (int)((rec[r].key >> shift) & 255);
    if (wave * 64 * kRadixItems + r * 64 + lane < cnt) s_rec[s_local[d] + s_cnt[wave][d] + rank[r]] = rec[r];
  }
  __syncthreads();
  for (int q = tid; q < cnt; q += kRadixBlock) {
    const KV e = s_rec[q];
    const long to = (long)s_out[(e.key >> shift) & 255] + q;
    if (to < 0 || to >= n) continue;   // (only where the table was not this sort's alone)
    if (out_ids) out_ids[to] = (int)e.value;
    else out[to] = e;
  }
}

__global__ __launch_bounds__(kRadixBlock) void k_radix_pass(const KV* __restrict__ in, KV* __restrict__ out, long n,
                                                             int shift, int pass, int* __restrict__ scratch,
                                                             int max_polls) {
  radix_pass(in, out, nullptr, n, shift, pass, scratch, max_polls, [](const KV& e) { return e; });
}

void launch_radix_sort(KV* data, KV* alt, long n, int bits, int* scratch, hipStream_t s, int max_polls) {
  if (max_polls < 0) max_polls = kRadixMaxPolls;
  if (n <= 1 || bits <= 0) return;
  const int passes = std::min(4, (bits + 7) / 8), nb = (int)radix_tiles(n);
  const long clear = radix_clear_ints(n);
  hipLaunchKernelGGL(k_radix_clear, dim3(ceil_div(clear, kBlock)), dim3(kBlock), 0, s, scratch, clear, 0l);
  CS_CHECK_LAUNCH();
  hipLaunchKernelGGL(k_radix_count, dim3(nb), dim3(kRadixBlock), 0, s, data, n, passes, scratch);
  CS_CHECK_LAUNCH();
  KV* src = data;
  KV* dst = alt;
  for (int p = 0; p < passes; ++p) {
    hipLaunchKernelGGL(k_radix_pass, dim3(nb), dim3(kRadixBlock), 0, s, src, dst, n, 8 * p, p, scratch, max_polls);
    CS_CHECK_LAUNCH();
    std::swap(src, dst);
  }
  if (passes & 1) CS_HIP(hipMemcpyAsync(data, alt, n * sizeof(KV), hipMemcpyDeviceToDevice, s));
}

// The three axes' presorts of the tree build (blockIdx.y = axis): ids in
// ascending order of (coordinate image, id).
//
// order-preserving unsigned images of a coordinate (IEEE: flip all bits of a
// negative value, the sign bit of a positive one)
__device__ __forceinline__ uint32_t ordered_bits(float x) {
  const uint32_t u = __float_as_uint(x);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ uint64_t ordered_bits(double x) {
  const uint64_t u = (uint64_t)__double_as_longlong(x);
  return (u & 0x8000000000000000ull) ? ~u : (u | 0x8000000000000000ull);
}
template <class T>
__device__ __forceinline__ T coordinate(const V4<T>& p, int axis) {
  return axis == 0 ? p.x : (axis == 1 ? p.y : p.z);
}

// records {low key word, id} and the digit counts of every pass
template <class T>
__global__ __launch_bounds__(kRadixBlock) void k_axis_keys(const V4<T>* __restrict__ pos, KV* __restrict__ kv, int n,
                                                            int* __restrict__ scratch, long stride) {
  chain_priority();
  constexpr int P = (int)sizeof(T);   // passes
  __shared__ int s_hist[P][256];
  const int axis = blockIdx.y;
  for (int q = threadIdx.x; q < P * 256; q += kRadixBlock) (&s_hist[0][0])[q] = 0;
  __syncthreads();
  for (int r = 0; r < kRadixItems; ++r) {
    const int i = blockIdx.x * kRadixTile + r * kRadixBlock + threadIdx.x;
    if (i >= n) continue;
    const auto b = ordered_bits(coordinate(pos[i], axis));
    kv[(size_t)axis * n + i] = {(uint32_t)b, (uint32_t)i};
    count_digits(s_hist, (uint32_t)b, 0, 4);
    if constexpr (P == 8) count_digits(s_hist, (uint32_t)(b >> 32), 4, 4);
  }
  __syncthreads();
  for (int q = threadIdx.x; q < P * 256; q += kRadixBlock) {
    const int c = (&s_hist[0][0])[q];
    if (c) atomicAdd(&scratch[axis * stride + q], c);
  }
}

// pass p; the pass that starts the high key words (FP64) takes them from the
// coordinates; the last one writes the ids to the axis's list
template <class T>
__global__ __launch_bounds__(kRadixBlock) void k_axis_pass(const KV* __restrict__ in, KV* __restrict__ out,
                                                            int* __restrict__ lists, long list_stride, int n, int pass,
                                                            int* __restrict__ scratch, long stride,
                                                            const V4<T>* __restrict__ pos) {
  chain_priority();
  const int axis = blockIdx.y;
  radix_pass(in + (size_t)axis * n, out + (size_t)axis * n,
             pass == (int)sizeof(T) - 1 ? lists + axis * list_stride : nullptr, n, 8 * (pass & 3), pass,
             scratch + axis * stride, kRadixMaxPolls, [&](const KV& e) {
               if (sizeof(T) == 8 && pass == 4)
                 return KV{(uint32_t)((uint64_t)ordered_bits(coordinate(pos[e.value], axis)) >> (sizeof(T) * 4)),
                           e.value};
               return e;
             });
}

template <class T>
void launch_axis_sorts(const V4<T>* pos, int n, KV* kv, KV* alt, int* lists, long list_stride, int* scratch,
                       hipStream_t s) {
  const int nb = (int)radix_tiles(n);
  const long stride = radix_scratch_ints(n);
  hipLaunchKernelGGL(k_axis_keys<T>, dim3(nb, 3), dim3(kRadixBlock), 0, s, pos, kv, n, scratch, stride);
  CS_CHECK_LAUNCH();
  for (int p = 0; p < (int)sizeof(T); ++p) {
    hipLaunchKernelGGL(k_axis_pass<T>, dim3(nb, 3), dim3(kRadixBlock), 0, s, (p & 1) ? alt : kv, (p & 1) ? kv : alt,
                       lists, list_stride, n, p, scratch, stride, pos);
    CS_CHECK_LAUNCH();
  }
}
template void launch_axis_sorts<float>(const F4*, int, KV*, KV*, int*, long, int*, hipStream_t);
template void launch_axis_sorts<double>(const D4*, int, KV*, KV*, int*, long, int*, hipStream_t);

// ---------------------------------------------------------------------------
// reaction transpose: for every j, the list slots k that name j, in
// ascending k (ascending owner i: the slots of i are contiguous and the
// offsets ascend with i), as pairs {key = owner i, value = k} in
// pairs[start[j], start[j + 1]).  A counting sort: per-j counts, their
// exclusive scan, a scatter that places each slot in its j's bucket (in
// whatever order the atomics resolve), and a sort of each bucket by k.

// one wavefront per particle i (measured faster than 16 lanes per particle:
// 0.69 against 1.28 ms for the count at N = 2^20): each real slot adds one to
// its j's count
__global__ __launch_bounds__(kBlock) void k_tr_count(const int* __restrict__ offset, const int* __restrict__ count,
                                                      const int* __restrict__ list, int* __restrict__ tcnt, int n) {
  chain_priority();
  const int i = blockIdx.x * (kBlock / 64) + (int)(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (i >= n) return;
  const int off = offset[i], c = count[i];
  for (int k = off + lane; k < off + c; k += 64) atomicAdd(&tcnt[list[k]], 1);
}

// each real slot takes a place in its j's bucket; tcnt counts down to zero,
// which is what the next transpose starts from
__global__ __launch_bounds__(kBlock) void k_tr_fill(const int* __restrict__ offset, const int* __restrict__ count,
                                                     const int* __restrict__ list, const int* __restrict__ start,
                                                     int* __restrict__ tcnt, KV* __restrict__ pairs, int n) {
  chain_priority();
  const int i = blockIdx.x * (kBlock / 64) + (int)(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (i >= n) return;
  const int off = offset[i], c = count[i];
  for (int k = off + lane; k < off + c; k += 64) {
    const int j = list[k];
    const int p = atomicSub(&tcnt[j], 1) - 1;
    pairs[start[j] + p] = KV{(uint32_t)i, (uint32_t)k};
  }
}

// bitonic sort of the m <= kTrSortMax pairs at p by k (value), ascending, in
// the one-wavefront block's LDS array s
__device__ __forceinline__ void bucket_sort(KV* __restrict__ p, int m, unsigned long long* s, int lane) {
  int P = 2;
  while (P < m) P <<= 1;
  for (int t = lane; t < P; t += 64) {
    if (t < m) {
      const KV e = p[t];
      s[t] = ((unsigned long long)e.value << 32) | e.key;
    } else {
      s[t] = ~0ull;
    }
  }
  __syncthreads();
  for (int k = 2; k <= P; k <<= 1)
    for (int h = k >> 1; h > 0; h >>= 1) {
      for (int t = lane; t < P / 2; t += 64) {
        const int x = ((t & ~(h - 1)) << 1) | (t & (h - 1)), y = x + h;
        const unsigned long long u = s[x], v = s[y];
        const bool up = (x & k) == 0;
        if ((u > v) == up) {
          s[x] = v;
          s[y] = u;
        }
      }
      __syncthreads();
    }
  for (int t = lane; t < m; t += 64) p[t] = KV{(uint32_t)(s[t] & 0xffffffffu), (uint32_t)(s[t] >> 32)};
}

// one one-wavefront block per bucket (measured faster than blocks that loop
// over buckets: 1.0 against 1.17 ms at N = 2^20): a bitonic sort by k in LDS
// (the k are distinct) for buckets of up to kTrSortMax slots; a larger bucket
// is ranked instead (each slot's place is the number of smaller k), through
// `alt`
constexpr int kTrSortMax = 512;
__global__ __launch_bounds__(64) void k_tr_sort(KV* __restrict__ pairs, KV* __restrict__ alt,
                                                 const int* __restrict__ start, int n) {
  chain_priority();
  __shared__ unsigned long long s[kTrSortMax];
  const int j = blockIdx.x, lane = threadIdx.x;
  if (j >= n) return;
  const int b = start[j], m = start[j + 1] - b;
  if (m <= 1) return;
  if (m > kTrSortMax) {
    for (int t = lane; t < m; t += 64) {
      const KV e = pairs[b + t];
      int r = 0;
      for (int q = 0; q < m; ++q) r += pairs[b + q].value < e.value;
      alt[b + r] = e;
    }
    __syncthreads();
    for (int t = lane; t < m; t += 64) pairs[b + t] = alt[b + t];
    return;
  }
  bucket_sort(pairs + b, m, s, lane);
}

void launch_reaction_transpose(const int* offset, const int* count, const int* list, int n, int* tcnt,
                               int* start, KV* pairs, KV* alt, int* scan_scratch, hipStream_t s) {
  const dim3 waves(ceil_div(n, kBlock / 64));
  hipLaunchKernelGGL(k_tr_count, waves, dim3(kBlock), 0, s, offset, count, list, tcnt, n);
  CS_CHECK_LAUNCH();
  launch_exclusive_scan(tcnt, start, n, 0, scan_scratch, s);
  hipLaunchKernelGGL(k_tr_fill, waves, dim3(kBlock), 0, s, offset, count, list, start, tcnt, pairs, n);
  CS_CHECK_LAUNCH();
  hipLaunchKernelGGL(k_tr_sort, dim3(n), dim3(64), 0, s, pairs, alt, start, n);
  CS_CHECK_LAUNCH();
}

__global__ __launch_bounds__(kBlock) void k_set_keys(KV* __restrict__ kv, const uint32_t* __restrict__ keys, int n) {
  const int t = blockIdx.x * kBlock + threadIdx.x;
  if (t < n) kv[t].key = keys[t];
}
void launch_set_keys(KV* kv, const uint32_t* keys, int n, hipStream_t s) {
  hipLaunchKernelGGL(k_set_keys, dim3(ceil_div(n, kBlock)), dim3(kBlock), 0, s, kv, keys, n);
  CS_CHECK_LAUNCH();
}

// plain and FP64 forms: a group of 16 lanes per particle, its sums in slot order
// (OrderedSums).  One lane per particle -> this, with the lists, us: plain
// 1 000 particles 73 -> 33, 16 384: 99 -> 66, 131 072: 377 -> 310, 600 000: 2198 -> 1423;
// FP64 65 536: 205 -> 178.
template <class T>
__global__ __launch_bounds__(kBlock) void k_reaction(const V4<T>* __restrict__ pos, V4<T>* __restrict__ bdots,
                                                      const T* __restrict__ ngb_acc, const KV* __restrict__ pairs,
                                                      const int* __restrict__ start, int n) {
  chain_priority();
  using Sums = OrderedSums<T, 4>;
  __shared__ __align__(16) T s_rows[kBlock / 16][Sums::kRow];
  const int j = (xcd_block(blockIdx.x, gridDim.x) * kBlock + (int)threadIdx.x) / 16, l = threadIdx.x % 16;
  if (j >= n) return;   // whole groups leave together
  const V4<T> pj = pos[j], d = bdots[j];
  Sums sums{l % 4 == 0 ? d.x : l % 4 == 1 ? d.y : l % 4 == 2 ? d.z : d.w, s_rows[threadIdx.x / 16], l};
  const int p0 = start[j], p1 = start[j + 1];
  for (int p = p0 + l; p - l < p1; p += 16) {
    T a[4] = {Sums::none(), Sums::none(), Sums::none(), Sums::none()};
    if (p < p1) {
      const KV e = pairs[p];
      const T acc = ngb_acc[e.value];
      const V4<T> pi = pos[e.key];
      a[0] = acc * (pi.x - pj.x);
      a[1] = acc * (pi.y - pj.y);
      a[2] = acc * (pi.z - pj.z);
    }
    sums.add(a);
  }
  const V4<T> b{sums.get(0), sums.get(1), sums.get(2), sums.get(3)};
  if (l == 0) bdots[j] = b;
}

template <class T>
void launch_reaction(const V4<T>* pos, V4<T>* bdots, const T* ngb_acc, const KV* pairs, const int* start,
                     int n, hipStream_t s) {
  hipLaunchKernelGGL(k_reaction<T>, dim3(ceil_div(n, kBlock / 16)), dim3(kBlock), 0, s, pos, bdots, ngb_acc, pairs,
                     start, n);
  CS_CHECK_LAUNCH();
}
template void launch_reaction<float>(const F4*, F4*, const float*, const KV*, const int*, int, hipStream_t);
template void launch_reaction<double>(const D4*, D4*, const double*, const KV*, const int*, int, hipStream_t);

// mixed form: the same gather with split positions and compensated sums; a
// group of 8 lanes per j, each lane taking every 8th of j's slots, partial
// sums combined with exact two-sums
__global__ __launch_bounds__(kBlock) void k_reaction_mixed(const F4* __restrict__ pos, const F4* __restrict__ lo,
                                                            F4* __restrict__ bdots, const float* __restrict__ ngb_acc,
                                                            const KV* __restrict__ pairs,
                                                            const int* __restrict__ start, int n) {
  chain_priority();
  constexpr int kG = 8;
  const int g = xcd_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
  const int j = g / kG, lane = g % kG;
  if (j >= n) return;   // whole groups leave together
  const F4 pj = pos[j], lj = lo[j];
  float s[3] = {0.f, 0.f, 0.f}, c[3] = {0.f, 0.f, 0.f};
  auto kadd = [&](int q, float x) {
    const float y = x - c[q];
    const float t = s[q] + y;
    c[q] = (t - s[q]) - y;
    s[q] = t;
  };
  for (int p = start[j] + lane, p1 = start[j + 1]; p < p1; p += kG) {
    const KV e = pairs[p];
    const int i = (int)e.key;
    const float acc = ngb_acc[e.value];
    const F4 pi = pos[i], li = lo[i];
    kadd(0, acc * ((pi.x - pj.x) + (li.x - lj.x)));
    kadd(1, acc * ((pi.y - pj.y) + (li.y - lj.y)));
    kadd(2, acc * ((pi.z - pj.z) + (li.z - lj.z)));
  }
  for (int q = 0; q < 3; ++q)
    for (int o = kG / 2; o > 0; o >>= 1) {
      const float s2 = __shfl_xor(s[q], o, kG), c2 = __shfl_xor(c[q], o, kG);
      const float t = s[q] + s2;
      const float bp = t - s[q];
      const float err = (s[q] - (t - bp)) + (s2 - bp);
      c[q] = (c[q] + c2) - err;
      s[q] = t;
    }
  if (lane != 0) return;
  F4 d = bdots[j];
  d.x += s[0] - c[0];
  d.y += s[1] - c[1];
  d.z += s[2] - c[2];
  bdots[j] = d;
}

void launch_reaction_mixed(const F4* pos, const F4* pos_lo, F4* bdots, const float* ngb_acc, const KV* pairs,
                           const int* start, int n, hipStream_t s) {
  hipLaunchKernelGGL(k_reaction_mixed, dim3(ceil_div(n * 8, kBlock)), dim3(kBlock), 0, s, pos, pos_lo, bdots, ngb_acc,
                     pairs, start, n);
  CS_CHECK_LAUNCH();
}

// ---------------------------------------------------------------------------
// Peano-Hilbert keys (sort_bodies.cpp:11-105, 119-163).  The state tables are
// Gadget-2's; they fix the curve and therefore the particle order.
__constant__ int c_ph_quad[24 * 8] = {
    0, 7, 1, 6, 3, 4, 2, 5,  7, 4, 6, 5, 0, 3, 1, 2,  4, 3, 5, 2, 7, 0, 6, 1,  3, 0, 2, 1, 4, 7, 5, 6,
    1, 0, 6, 7, 2, 3, 5, 4,  0, 3, 7, 4, 1, 2, 6, 5,  3, 2, 4, 5, 0, 1, 7, 6,  2, 1, 5, 6, 3, 0, 4, 7,
    6, 1, 7, 0, 5, 2, 4, 3,  1, 2, 0, 3, 6, 5, 7, 4,  2, 5, 3, 4, 1, 6, 0, 7,  5, 6, 4, 7, 2, 1, 3, 0,
    7, 6, 0, 1, 4, 5, 3, 2,  6, 5, 1, 2, 7, 4, 0, 3,  5, 4, 2, 3, 6, 7, 1, 0,  4, 7, 3, 0, 5, 6, 2, 1,
    6, 7, 5, 4, 1, 0, 2, 3,  7, 0, 4, 3, 6, 1, 5, 2,  0, 1, 3, 2, 7, 6, 4, 5,  1, 6, 2, 5, 0, 7, 3, 4,
    2, 3, 1, 0, 5, 4, 6, 7,  3, 4, 0, 7, 2, 5, 1, 6,  4, 5, 7, 6, 3, 2, 0, 1,  5, 2, 6, 1, 4, 3, 7, 0};
__constant__ int c_ph_rotx[24] = {4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 0, 1, 2, 3, 17, 18, 19, 16, 23, 20, 21, 22};
__constant__ int c_ph_roty[24] = {1, 2, 3, 0, 16, 17, 18, 19, 11, 8, 9, 10, 22, 23, 20, 21, 14, 15, 12, 13, 4, 5, 6, 7};
__constant__ int c_ph_nx[8] = {3, 0, 0, 2, 2, 0, 0, 1};
__constant__ int c_ph_ny[8] = {0, 1, 1, 2, 2, 3, 3, 0};
__constant__ int c_ph_sense[8] = {-1, -1, -1, +1, +1, -1, -1, -1};

__device__ unsigned long long ph_key_dev(int x, int y, int z, int bits) {
  unsigned long long key = 0;
  int rot = 0, sense = 1;
  for (int b = bits - 1; b >= 0; --b) {
    const int q = c_ph_quad[rot * 8 + (((x >> b) & 1) << 2) + (((y >> b) & 1) << 1) + ((z >> b) & 1)];
    key = (key << 3) + (unsigned long long)(sense == 1 ? q : 7 - q);
    for (int k = 0; k < c_ph_nx[q]; ++k) rot = c_ph_rotx[rot];
    for (int k = 0; k < c_ph_ny[q]; ++k) rot = c_ph_roty[rot];
    sense *= c_ph_sense[q];
  }
  return key;
}

// bounding box (sort_bodies.cpp:121-134): per-block min/max of x,y,z, then
// one block folds the block results into box[6 nb .. 6 nb + 5] (min and max
// are exact in any order)
template <class T>
__global__ __launch_bounds__(kBlock) void k_bbox(const V4<T>* __restrict__ pos, int n, T* __restrict__ out) {
  __shared__ T s[6][kBlock];
  const int i = blockIdx.x * kBlock + threadIdx.x;
  const V4<T> p = pos[i < n ? i : 0];
  s[0][threadIdx.x] = p.x; s[1][threadIdx.x] = p.y; s[2][threadIdx.x] = p.z;
  s[3][threadIdx.x] = p.x; s[4][threadIdx.x] = p.y; s[5][threadIdx.x] = p.z;
  __syncthreads();
  for (int off = kBlock / 2; off > 0; off >>= 1) {
    if (threadIdx.x < off) {
      for (int c = 0; c < 3; ++c) s[c][threadIdx.x] = fmin(s[c][threadIdx.x], s[c][threadIdx.x + off]);
      for (int c = 3; c < 6; ++c) s[c][threadIdx.x] = fmax(s[c][threadIdx.x], s[c][threadIdx.x + off]);
    }
    __syncthreads();
  }
  if (threadIdx.x < 6) out[blockIdx.x * 6 + threadIdx.x] = s[threadIdx.x][0];
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_bbox_fold(T* __restrict__ box, int nb) {
  __shared__ T s[6][kBlock];
  T v[6];
  for (int c = 0; c < 6; ++c) v[c] = box[c];   // block 0 always exists
  for (int b = threadIdx.x; b < nb; b += kBlock) {
    for (int c = 0; c < 3; ++c) v[c] = fmin(v[c], box[6 * b + c]);
    for (int c = 3; c < 6; ++c) v[c] = fmax(v[c], box[6 * b + c]);
  }
  for (int c = 0; c < 6; ++c) s[c][threadIdx.x] = v[c];
  __syncthreads();
  for (int off = kBlock / 2; off > 0; off >>= 1) {
    if (threadIdx.x < off) {
      for (int c = 0; c < 3; ++c) s[c][threadIdx.x] = fmin(s[c][threadIdx.x], s[c][threadIdx.x + off]);
      for (int c = 3; c < 6; ++c) s[c][threadIdx.x] = fmax(s[c][threadIdx.x], s[c][threadIdx.x + off]);
    }
    __syncthreads();
  }
  if (threadIdx.x < 6) box[6 * nb + threadIdx.x] = s[threadIdx.x][0];
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_ph_keys(const V4<T>* __restrict__ pos, int n, int bits,
                                                     const T* __restrict__ box, uint32_t* key_hi,
                                                     uint32_t* key_lo) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  T lo[3], hi[3];
  for (int c = 0; c < 3; ++c) { lo[c] = box[c]; hi[c] = box[3 + c]; }
  const T size = fmax(hi[2] - lo[2], fmax(hi[1] - lo[1], hi[0] - lo[0]));
  const T fac = T(1.0 / (double)size * (double)(1LL << bits));
  const V4<T> p = pos[i];
  const int x = (int)((p.x - lo[0]) * fac), y = (int)((p.y - lo[1]) * fac), z = (int)((p.z - lo[2]) * fac);
  const unsigned long long key = ph_key_dev(x, y, z, bits);
  key_hi[i] = (uint32_t)(key >> 32);
  key_lo[i] = (uint32_t)key;
}

template <class T>
void launch_ph_keys(const V4<T>* pos, int n, int bits, uint32_t* key_hi, uint32_t* key_lo, int* scratch,
                    hipStream_t s) {
  const int nb = ceil_div(n, kBlock);
  T* box = reinterpret_cast<T*>(scratch);
  hipLaunchKernelGGL(k_bbox<T>, dim3(nb), dim3(kBlock), 0, s, pos, n, box);
  CS_CHECK_LAUNCH();
  hipLaunchKernelGGL(k_bbox_fold<T>, dim3(1), dim3(kBlock), 0, s, box, nb);
  CS_CHECK_LAUNCH();
  hipLaunchKernelGGL(k_ph_keys<T>, dim3(nb), dim3(kBlock), 0, s, pos, n, bits, box + 6 * (size_t)nb, key_hi,
                     key_lo);
  CS_CHECK_LAUNCH();
}
template void launch_ph_keys<float>(const F4*, int, int, uint32_t*, uint32_t*, int*, hipStream_t);
template void launch_ph_keys<double>(const D4*, int, int, uint32_t*, uint32_t*, int*, hipStream_t);

}  // namespace cudasph
