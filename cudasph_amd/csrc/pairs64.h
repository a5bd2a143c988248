// FP64 N^2 sums over pairs whose two contributions come from one evaluation.
#pragma once

#include "common.h"

namespace cudasph {

// Particles in tiles of 512.  A block keeps tile I's particles, two per lane, and
// meets the tiles J = I + d (mod tiles), in halves, that its part takes in turn:
// each pair of tiles is met once, by the tile that is at most half way round
// behind the other (at exactly half way by the lower one), and each pair of
// particles is evaluated once for both.  The FP64 pair body is VALU-bound (22 to
// 36 operations of 4.4 to 5.4 cycles and a v_rsq_f64 of 16), so halving the
// evaluations is worth the bookkeeping: the sums of J's particles (the
// reactions) move with the records instead of staying in a lane.  In a row of 16
// lanes, lane c meets record (c + s) % 16 of 16 at step s, and the reactions
// rotate by one lane per step (2 moves each, 4.2 cycles a move: shared by the
// lane's two particles); after 16 steps the four rows exchange their 16 records.
// After 64 records the four wavefronts' reactions are added in order and
// written, (d - 1, J) is the slot of a block of its own, and pairs64_sum adds own
// sums and reactions of a particle in a fixed order: no atomics, the same bits
// each time.  Tile d = 0 is I itself: all ordered pairs, without reactions.
// The records are staged twice in a row of 16, so that record c + s needs no
// wrap: the loop reads at constant offsets.
//
// Body: kRec (records' double2s), kAcc (sums), I load(i, n), stage(dst, i, n)
// with dst(k) the place of double2 k, and pair<REACT>(I, record, own, react).
// Gravity alone, ms, every ordered pair / this kernel: 8 192 particles 0.092 /
// 0.082, 16 384: 0.254 / 0.239, 32 768: 0.88 / 0.62, 50 021: 1.92 / 1.34, 65 536: 2.94 /
// 2.06, 131 072: 11.4 / 7.9 (one particle per lane: 0.66, 1.41, 2.25, 8.6 at the last
// four).  So from 8 192 on; to 2^18, where the reactions take 2 GiB (n^2 / 32 bytes;
// written and read once, 2 % of the time).
constexpr int kPairTile = 512, kPairHalf = 256;
constexpr int kPairs64MinN = 8192, kPairs64MaxN = 1 << 18;
inline bool pairs64_fits(int n) { return n >= kPairs64MinN && n <= kPairs64MaxN; }
inline int pairs64_tiles(int n) { return (n + kPairTile - 1) / kPairTile; }
// few tiles: more parts than asked for, so that the GPU has blocks enough (8 192
// particles 0.145 -> 0.082 ms; at 16 384, 0.239 -> 0.174 alone, they hold up the SPH
// passes of a step, 0.71 -> 0.76)
inline int pairs64_parts(int n, int parts) { return n < 12288 ? 3 * parts : parts; }
// doubles: own sums of the parts, then the reactions
inline size_t pairs64_own(int n, int parts) {
  return (size_t)pairs64_parts(n, parts) * 4 * pairs64_tiles(n) * kPairTile;
}
inline size_t pairs64_words(int n, int parts) {
  return pairs64_own(n, parts) + (size_t)(pairs64_tiles(n) / 2) * 4 * pairs64_tiles(n) * kPairTile;
}

__device__ __forceinline__ double from_next_lane16(double v) {   // of the row of 16, cyclic
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x12f, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x12f, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

template <class B>
__global__ __launch_bounds__(kPairHalf) __attribute__((amdgpu_waves_per_eu(4)))
void k_pairs64(B b, int n, int tiles, int parts, double* __restrict__ own, double* __restrict__ react) {
  __shared__ double2 s_rec[B::kRec][kPairHalf / 16][32];
  __shared__ double s_acc[4][B::kAcc][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane & 15, row = lane >> 4;
  const int tile = (int)blockIdx.x / parts, part = (int)blockIdx.x % parts, half = tiles / 2;
  const size_t np = (size_t)tiles * kPairTile;
  const int i0 = tile * kPairTile + 128 * wave + lane;   // and i0 + 64
  const auto p0 = b.load(i0, n), p1 = b.load(i0 + 64, n);
  double g0[B::kAcc] = {}, g1[B::kAcc] = {};
  for (int u = part; u < 2 * (half + 1); u += parts) {   // half tiles
    const int d = u >> 1;
    if (2 * d == tiles && tile >= half) break;   // the opposite tile's block has this pair of tiles
    const int j_half = (tile + d < tiles ? tile + d : tile + d - tiles) * kPairTile + (u & 1) * kPairHalf;
    __syncthreads();
    b.stage([&](int k, double2 v) {
      s_rec[k][tid >> 4][tid & 15] = v;
      s_rec[k][tid >> 4][(tid & 15) + 16] = v;
    }, j_half + tid, n);
    __syncthreads();
    if (d == 0) {
      for (int j = 0; j < kPairHalf; ++j) {
        double2 r[B::kRec];
        for (int k = 0; k < B::kRec; ++k) r[k] = s_rec[k][j >> 4][j & 15];
        b.template pair<false>(p0, r, g0, g0);
        b.template pair<false>(p1, r, g1, g1);
      }
      continue;
    }
    for (int j0 = 0; j0 < kPairHalf / 16; j0 += 4) {
      double a[B::kAcc] = {};
      for (int q = 0; q < 4; ++q) {
        const int grp = j0 + ((row + q) & 3);
#pragma unroll
        for (int s = 0; s < 16; ++s) {
          double2 r[B::kRec];
          for (int k = 0; k < B::kRec; ++k) r[k] = s_rec[k][grp][c + s];
          b.template pair<true>(p0, r, g0, a);
          b.template pair<true>(p1, r, g1, a);
          for (int k = 0; k < B::kAcc; ++k) a[k] = from_next_lane16(a[k]);
        }
        for (int k = 0; k < B::kAcc; ++k) a[k] = __shfl(a[k], (lane + 16) & 63);
      }
      for (int k = 0; k < B::kAcc; ++k) s_acc[wave][k][lane] = a[k];
      __syncthreads();
      if (wave < B::kAcc)
        react[((size_t)(d - 1) * B::kAcc + wave) * np + j_half + j0 * 16 + lane] =
            (s_acc[0][wave][lane] + s_acc[1][wave][lane]) + (s_acc[2][wave][lane] + s_acc[3][wave][lane]);
      __syncthreads();
    }
  }
  for (int k = 0; k < B::kAcc; ++k) {
    own[((size_t)part * B::kAcc + k) * np + i0] = g0[k];
    own[((size_t)part * B::kAcc + k) * np + i0 + 64] = g1[k];
  }
}

// the sum of component blockIdx.y of a particle: own parts, then reactions
template <int ACC>
__device__ __forceinline__ double pairs64_sum(const double* __restrict__ own, const double* __restrict__ react,
                                              int i, int k, int tiles, int parts) {
  const size_t np = (size_t)tiles * kPairTile;
  const int half = tiles / 2, last = 2 * half == tiles && i / kPairTile < half ? half - 1 : half;
  double s = 0.0;
  for (int p = 0; p < parts; ++p) s += own[((size_t)p * ACC + k) * np + i];
#pragma unroll 8
  for (int d = 0; d < last; ++d) s += react[((size_t)d * ACC + k) * np + i];
  return s;
}

template <class B>
void launch_pairs64(const B& b, int n, int parts, double* ws, hipStream_t s) {
  const int tiles = pairs64_tiles(n), np = pairs64_parts(n, parts);
  hipLaunchKernelGGL(k_pairs64<B>, dim3(tiles * np), dim3(kPairHalf), 0, s, b, n, tiles, np, ws,
                     ws + pairs64_own(n, parts));
  CS_CHECK_LAUNCH();
}

}  // namespace cudasph
