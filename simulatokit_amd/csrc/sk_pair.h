// sk_pair.h — two-stage row and column passes for lines of M = RA RB points (RA >= RB, both at most 48 with prime
// factors up to 13): the passes of every smooth grid length without a pass of its own, and of every full-width 2-D
// transform (potentials, probes, the lens).
//
// A line's transform is one DFT of RA points per lane, one exchange through LDS, and one DFT of RB points per lane:
//   layout I: lane i < RB holds the elements i + RB r (r < RA);  layout Q: lane q < RA holds q + RA p (p < RB).
//   from I to Q: DFT_RA over r, LDS [q][i], the root w_M^{i q}, DFT_RB over i      (either sign)
//   from Q to I: DFT_RB over p, the root w_M^{q q'}, LDS [q][q'], DFT_RA over q, both DFTs by the transposed flow
//                graph: the whole is the transpose of the way from I to Q, so that in a pass (one way with one sign,
//                back with the other) the rounding of the constants enters as F F^H, whose phase errors cancel
// A row pass of the slice loop (inverse, times t, forward) goes I -> Q -> I and a column pass (forward, times P,
// inverse) the same way with the signs exchanged, so a pass costs two exchanges and two products with the roots per
// point, where a Stockham transform with radices up to 13 in LDS costs as many exchanges per transform as it has stages.
// The roots come from two tables [p][q] in LDS that the block's units share (read through the L1 cache instead, 600^2
// ran at 0.159 against 0.129 ms a row pass). Lane q reads and writes only the LDS row [q][.] and lane i only the column
// [.][i], so nothing but the two hand-overs of a pass needs a barrier; the next unit's first write needs none where a pass goes both
// ways.
//
// Bounds at 600^2 (128 positions, waves in the last-level cache): the row pass issues about 76 vector instructions per
// point, 0.10 ms at 2.2 GHz of the 0.129 ms it takes; the column pass moves its 0.49 GB at 4.0 TB/s. The Stockham
// passes it replaces took 0.70 and 0.47 ms. A scan of 256 positions and 20 slices: 92 k -> 469 k position-slices/s.
//
// A unit of a row pass is one row x of one position; consecutive lines of a block take consecutive units, positions
// fastest, so they share the row t(x, .) and a small batch still fills the block. A column pass takes TC compact
// columns (row segments of 8 TC bytes) of NP positions.
#pragma once

#include <atomic>

#include "sk_rdft.h"

namespace sk {

constexpr int kPairMax = 48;  // the largest radix
constexpr bool pair_radix(int r) {
  if (r < 2 || r > kPairMax) return false;
  for (int p : {2, 3, 5, 7, 11, 13})
    while (r % p == 0) r /= p;
  return r == 1;
}
// RA of a line length: the smallest radix at or above sqrt(M) whose cofactor is a radix too (0: none)
constexpr int pair_ra(int m) {
  for (int a = 2; a <= kPairMax; ++a)
    if (a * a >= m && m % a == 0 && pair_radix(a) && pair_radix(m / a)) return a;
  return 0;
}

template <int M>
struct PairShape {
  static constexpr int RA = pair_ra(M), RB = M / RA;
  static constexpr int S1 = RB | 1;  // LDS row stride: odd, so that lanes q reading column i fall on distinct banks
  static constexpr int LS = RA * S1;
  // wavefronts per SIMD the registers are held to, by the larger radix. At three, the columns of 360 and 400 points and
  // the row passes of 546, 572, 576, 624, 648, 650, 675, 676, 702 and 729 spill 12 to 84 bytes a lane; at two, the columns
  // of 819 points and more spill up to 128. Where the LDS holds fewer wavefronts than that, the compiler takes the
  // registers that they leave (600: row pass 177 VGPRs, two). 600's column pass: 0.123 ms per 128 positions at two, 0.387
  // at three, where P's values spill.
  static constexpr int ROW_WAVES = RA <= 28 ? 3 : 2, COL_WAVES = RA <= 20 ? 3 : 2;
  // The wavefronts of blocks of `threads` threads that a CU holds (160 KB of LDS with the roots' tables, `waves` per
  // SIMD).
  static constexpr int held(int threads, int lines, int waves) {
    const int lds = lines * LS * 8 + 2 * M * 8, per_block = (threads + 63) / 64;
    const int blocks = 160 * 1024 / lds, limit = 4 * waves / per_block;
    return lines < 1 ? 0 : (blocks < limit ? blocks : limit) * per_block;
  }
  // row pass: blocks of 64 .. 256 threads, by the share of threads that have a lane and the root of the wavefronts held
  // (an idle thread costs in full, each further wavefront hides less). Bluestein's 900 points for 509^2: 0.394, 0.344
  // and 0.285 ms per 119 positions with 64, 128 and 256 threads (5, 6 and 8 wavefronts a CU, no idle thread more); 600
  // points: 0.129 ms with 128 threads (8 wavefronts, 98 % of the threads), 0.167 with 192 (9, 91 %).
  static constexpr double row_score(int nt) {
    const double share = double(nt / RA * RA) / nt;
    return share * share * held(nt, nt / RA, ROW_WAVES);
  }
  static constexpr int row_threads() {
    int best = 64;
    for (int nt = 128; nt <= 256; nt += 64)
      if (row_score(nt) > 1.04 * row_score(best)) best = nt;
    return best;
  }
  static constexpr int NT = row_threads(), L = NT / RA;
  // column pass: TC columns (8, row segments of 64 bytes, whose neighbour runs on the same XCD, or 16) of NP positions,
  // by the wavefronts held and the share of their threads. 360 points (211^2): 0.160 ms with 8 columns, 0.252 with 16;
  // 1024 points (613^2): 0.396 ms with two positions, 0.583 with one.
  struct ColShape {
    int tc, np;
  };
  static constexpr double col_score(ColShape c) {
    const int threads = c.tc * c.np * RA, waves = (threads + 63) / 64;
    return threads > 512 ? 0.0 : double(held(threads, c.tc * c.np, COL_WAVES)) * threads / (waves * 64);
  }
  static constexpr ColShape col_shape() {
    ColShape best{8, 1};
    for (int tc = 8; tc <= 16; tc += 8)
      for (int np = 1; np <= 4; ++np)
        if (col_score({tc, np}) > 1.02 * col_score(best)) best = ColShape{tc, np};
    return best;
  }
  static constexpr int TC = col_shape().tc, NP = col_shape().np;
  static constexpr int CT = (TC * RA * NP + 63) / 64 * 64;  // threads of a column block
};

// Where the elements i + RB r (every lane i) of a line of M points stand in the compact form: the kept columns
// satisfy |k| <= M / 3 on every grid, so a whole group r lies among the low frequencies (compact column e, kept when
// e <= kept_hi), among the high ones (column e - kept_shift, kept when e >= kept_lo) or in the band between, which no
// grid keeps and whose values are zeros at compile time.
enum PairGroup : int { PAIR_LOW, PAIR_HIGH, PAIR_BAND };
template <int M>
__host__ __device__ constexpr int pair_group(int r) {
  constexpr int RB = PairShape<M>::RB, K = M / 3;
  return RB * r <= K ? PAIR_LOW : RB * (r + 1) - 1 >= M - K ? PAIR_HIGH : PAIR_BAND;
}

template <int M>
__global__ void __launch_bounds__(PairShape<M>::NT, PairShape<M>::ROW_WAVES) row_pair_kernel(RowArgs a, int batch, int rounds) {
  using S = PairShape<M>;
  constexpr int RA = S::RA, RB = S::RB, S1 = S::S1, L = S::L;
  __shared__ float2 lds[L * S::LS];
  const int tid = threadIdx.x;
  __shared__ float2 tab[2 * M];  // the plan's two tables of roots
  for (int e = tid; e < 2 * M; e += S::NT) tab[e] = a.fy.pair[e];
  __syncthreads();
  // the thread's line and lane in the two layouts; threads past the last line's lanes take part in the barriers only
  const int li = tid / RB, i = tid - li * RB;
  const int lq = tid / RA, q = tid - lq * RA;
  const bool on_i = li < L, on_q = lq < L;
  float2* bi = lds + (on_i ? li : 0) * S::LS + i;
  float2* bq = lds + (on_q ? lq : 0) * S::LS + q * S1;
  const int f = a.flags;
  const long long gw = (long long)a.nx * a.nc;
  const long long units = (long long)a.nx * batch;
#pragma unroll 1
  for (int round = 0; round < rounds; ++round) {
    const long long u0 = ((long long)blockIdx.x * rounds + round) * L;
    if (u0 >= units) break;  // uniform over the block
    const long long ui = u0 + li, uq = u0 + lq;
    const bool live_i = on_i && ui < units, live_q = on_q && uq < units;
    // unit -> (row x, position b), positions fastest
    const int xi = live_i ? int((unsigned)ui / (unsigned)batch) : 0, bbi = live_i ? int(ui - (long long)xi * batch) : 0;
    const int xq = live_q ? int((unsigned)uq / (unsigned)batch) : 0, bbq = live_q ? int(uq - (long long)xq * batch) : 0;
    // the lane indices as values the compiler cannot follow across rounds: element offsets and masks are recomputed
    // here rather than held in registers (one or two each) over the loop
    int il = i, ql = q;
    asm volatile("" : "+v"(il), "+v"(ql));
    const float2* w = tab + ql;
    float2 v[RB];  // layout Q
    if (f & ROW_INV) {
      float2 u[RA];  // layout I
      if (f & ROW_IN_COMPACT) {
        // unmasked loads (a group's address is clamped to the row's kept columns), then zeros where not kept
        const float2* g = a.G + bbi * gw + (long long)xi * a.nc;
        const float2* lo = g + il;
        const float2* hi = g + il - a.kept_shift;
#pragma unroll
        for (int r = 0; r < RA; ++r) {
          const int group = pair_group<M>(r);
          u[r] = make_float2(0.f, 0.f);
          if (group == PAIR_LOW) {
            const int over = il + RB * r - a.kept_hi;
            const float2 t = lo[over > 0 ? -il : RB * r];
            if (over <= 0) u[r] = t;
          } else if (group == PAIR_HIGH) {
            const int under = a.kept_lo - (il + RB * r);
            const float2 t = hi[under > 0 ? a.kept_shift - il : RB * r];
            if (under <= 0) u[r] = t;
          }
        }
      } else {
        const float2* g = a.in_full + bbi * a.in_full_stride + (long long)xi * M + il;
#pragma unroll
        for (int r = 0; r < RA; ++r) u[r] = g[RB * r];
      }
      rdft<RA, +1>(u);
      if (on_i) {
#pragma unroll
        for (int r = 0; r < RA; ++r) bi[r * S1] = u[r];
      }
      __syncthreads();
#pragma unroll
      for (int p = 0; p < RB; ++p) v[p] = cmulc(bq[p], w[RA * p]);
      rdft<RB, +1>(v);
    } else {
      const float2* g = a.in_full + bbq * a.in_full_stride + (long long)xq * M + ql;
#pragma unroll
      for (int p = 0; p < RB; ++p) v[p] = g[RA * p];
    }
    if ((f & ROW_WRITE_PLANE) && live_q) {
      float2* pl = a.plane + bbq * a.plane_stride + (long long)xq * M + ql;
#pragma unroll
      for (int p = 0; p < RB; ++p) pl[RA * p] = cscale(v[p], a.out_scale);
    }
    if (f & ROW_FWD) {
      if (f & ROW_MUL_T) {
        const float2* t = a.t + (long long)xq * M + ql;
#pragma unroll
        for (int p = 0; p < RB; ++p) v[p] = cmul(v[p], t[RA * p]);
      }
      rdft<RB, -1, true>(v);
      if (on_q) {
#pragma unroll
        for (int p = 0; p < RB; ++p) bq[p] = cmul(v[p], w[M + RA * p]);
      }
      __syncthreads();
      float2 u[RA];
#pragma unroll
      for (int r = 0; r < RA; ++r) u[r] = bi[r * S1];
      rdft<RA, -1, true>(u);
      if ((f & ROW_OUT_COMPACT) && live_i) {
        float2* g = a.G + bbi * gw + (long long)xi * a.nc;
        float2* lo = g + il;
        float2* hi = g + il - a.kept_shift;
#pragma unroll
        for (int r = 0; r < RA; ++r) {
          const int group = pair_group<M>(r);
          if (group == PAIR_LOW) {
            if (il + RB * r <= a.kept_hi) lo[RB * r] = u[r];
          } else if (group == PAIR_HIGH) {
            if (il + RB * r >= a.kept_lo) hi[RB * r] = u[r];
          }
        }
      } else if (live_i) {
        float2* g = a.out_full + bbi * a.out_full_stride + (long long)xi * M + il;
#pragma unroll
        for (int r = 0; r < RA; ++r) g[RB * r] = cscale(u[r], a.out_scale);
      }
    } else if ((f & ROW_OUT_FULL) && live_q) {
      float2* g = a.out_full + bbq * a.out_full_stride + (long long)xq * M + ql;
#pragma unroll
      for (int p = 0; p < RB; ++p) g[RA * p] = cscale(v[p], a.out_scale);
    }
    // one transform alone begins the next round in the layout that it does not end in: its first write waits for this
    // round's reads
    if ((f & (ROW_INV | ROW_FWD)) != (ROW_INV | ROW_FWD)) __syncthreads();
  }
}

// Column pass. Threads: (lane, column) with the column fastest, so that a row segment of TC values is one access;
// the LDS slot of (row, lane) of column cb is [row][lane][cb]. Global addresses are a block-uniform start per row
// group (scalar registers) plus one 32-bit byte offset per lane.
template <int M>
__global__ void __launch_bounds__(PairShape<M>::CT, PairShape<M>::COL_WAVES) col_pair_kernel(ColArgs a, int batch, int rounds,
                                                                                                  int tiles) {
  using S = PairShape<M>;
  constexpr int RA = S::RA, RB = S::RB, S1 = S::S1, TC = S::TC, NP = S::NP;
  __shared__ float2 lds[NP * TC * S::LS];
  const int tid = threadIdx.x;
  __shared__ float2 tab[2 * M];  // the plan's two tables of roots
  for (int e = tid; e < 2 * M; e += S::CT) tab[e] = a.fx.pair[e];
  __syncthreads();
  const int cb = tid % TC, lane = tid / TC;
  const int ni = lane / RB, i = lane - ni * RB;
  const int nq = lane / RA, q = lane - nq * RA;
  const bool on_i = ni < NP, on_q = nq < NP;
  float2* bi = lds + (on_i ? ni : 0) * TC * S::LS + i * TC + cb;
  float2* bq = lds + (on_q ? nq : 0) * TC * S::LS + q * S1 * TC + cb;
  // The device deals blocks round-robin over its 8 XCDs: each XCD takes consecutive units (tile fastest), so that
  // neighbouring 64-byte tiles read their shared 128-byte lines through one L2 (the grid is padded to whole rounds).
  const int per_xcd = gridDim.x / 8, u = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
  const int2 unit = make_int2(u % tiles, u / tiles);
  const int c = unit.x * TC + cb;
  const int iy = c < a.nc ? a.keep[c] : -1;
  const bool kept = iy >= 0;  // padding columns: read as zeros, never stored
  const int f = a.flags;
  const long long gw = (long long)a.nx * a.nc;
#pragma unroll 1
  for (int round = 0; round < rounds; ++round) {
    const long long p0 = ((long long)unit.y * rounds + round) * NP;
    if (p0 >= batch) break;  // uniform over the block
    const bool live_i = on_i && kept && p0 + ni < batch, live_q = on_q && kept && p0 + nq < batch;
    const char* base = reinterpret_cast<const char*>(a.G + p0 * gw + unit.x * TC);
    // byte offsets of (position, row, column) from the unit's first value; a lane without a value reads the first
    int ie = i, qe = q;
    asm volatile("" : "+v"(ie), "+v"(qe));  // as in the row pass
    const float2* w = tab + qe;
    const unsigned oi = live_i ? unsigned(ni * gw + (long long)ie * a.nc + cb) * 8u : 0u;
    const unsigned oq = live_q ? unsigned(nq * gw + (long long)qe * a.nc + cb) * 8u : 0u;
    const long long si = 8LL * RB * a.nc, sq = 8LL * RA * a.nc;  // bytes from one row group to the next
    float2 v[RB];  // layout Q
    if (f & COL_FWD) {
      float2 u[RA];  // layout I
#pragma unroll
      for (int r = 0; r < RA; ++r) u[r] = *reinterpret_cast<const float2*>(base + r * si + oi);
      if (!live_i) {
#pragma unroll
        for (int r = 0; r < RA; ++r) u[r] = make_float2(0.f, 0.f);
      }
      rdft<RA, -1>(u);
      if (on_i) {
#pragma unroll
        for (int r = 0; r < RA; ++r) bi[r * S1 * TC] = u[r];
      }
      float2 pv[RB];
      if (f & COL_MUL_P) {
        const char* pb = reinterpret_cast<const char*>(a.P + unit.x * TC);
        const unsigned op = live_q ? unsigned((long long)qe * a.nc + cb) * 8u : 0u;
#pragma unroll
        for (int p = 0; p < RB; ++p) pv[p] = *reinterpret_cast<const float2*>(pb + p * sq + op);
      }
      __syncthreads();
#pragma unroll
      for (int p = 0; p < RB; ++p) v[p] = cmul(bq[p * TC], w[RA * p]);
      rdft<RB, -1>(v);
      if (f & COL_MUL_P) {
#pragma unroll
        for (int p = 0; p < RB; ++p) v[p] = cmul(v[p], pv[p]);
      }
    } else if (f & COL_GENERATE) {
      const long long b = p0 + nq;
#pragma unroll
      for (int p = 0; p < RB; ++p) {
        const int x = qe + RA * p;
        v[p] = live_q ? cmul(cmul(a.spec[(long long)x * a.ny + iy], a.rx[b * M + x]), a.ry[b * a.ny + iy])
                      : make_float2(0.f, 0.f);
      }
    } else {
#pragma unroll
      for (int p = 0; p < RB; ++p) v[p] = *reinterpret_cast<const float2*>(base + p * sq + oq);
    }
    if (f & COL_INV) {
      rdft<RB, +1, true>(v);
      if (on_q) {
#pragma unroll
        for (int p = 0; p < RB; ++p) bq[p * TC] = cmulc(v[p], w[M + RA * p]);
      }
      __syncthreads();
      float2 u[RA];
#pragma unroll
      for (int r = 0; r < RA; ++r) u[r] = bi[r * S1 * TC];
      rdft<RA, +1, true>(u);
      if (live_i) {
        char* out = const_cast<char*>(base);
#pragma unroll
        for (int r = 0; r < RA; ++r) *reinterpret_cast<float2*>(out + r * si + oi) = u[r];
      }
    } else {
      if (live_q) {
        char* out = const_cast<char*>(base);
#pragma unroll
        for (int p = 0; p < RB; ++p) *reinterpret_cast<float2*>(out + p * sq + oq) = v[p];
      }
    }
    if ((f & (COL_FWD | COL_INV)) != (COL_FWD | COL_INV)) __syncthreads();  // as in the row pass
  }
}

// The kernels of one length and what their launches need.
struct PairKernels {
  int m = 0;
  void (*row)(RowArgs, int, int) = nullptr;
  void (*col)(ColArgs, int, int, int) = nullptr;
  int row_threads = 0, row_lines = 0, col_threads = 0, col_tile = 0, col_positions = 0;
  std::atomic<int> row_per_cu{0}, col_per_cu{0};  // blocks a CU holds at once (0: not asked yet)
};

template <int M>
void pair_kernels(PairKernels& k) {
  using S = PairShape<M>;
  k.m = M;
  k.row = &row_pair_kernel<M>;
  k.col = &col_pair_kernel<M>;
  k.row_threads = S::NT;
  k.row_lines = S::L;
  k.col_threads = S::CT;
  k.col_tile = S::TC;
  k.col_positions = S::NP;
}

}  // namespace sk
