// sk_blue.h — Bluestein's algorithm on the two-stage transforms (sk_pair.h): row and column passes for grid lengths n
// with a prime factor above 13.
//
// Bluestein (1970): X_k = c_k sum_j (x_j c_j) conj(c_{k-j}), c_l = e^{-i pi l^2 / n} (conjugated for the inverse), the
// sum done as a cyclic convolution of M points: forward transform (layout I to Q), the product with the kernel's
// transform in layout Q, inverse transform (Q to I). Both ends of a convolution are in layout I, so a pass of the slice
// loop is two convolutions with one product (t or P) between them, in registers; the chirps that meet there cancel.
//
// The convolution only has to separate the outputs that are used. In the slice loop one side of every transform is the
// band that the antialias aperture keeps, at most 2 floor(n / 3) + 1 frequencies: a spectrum is held centred, frequency k
// in slot k mod M, and M >= n + 2 floor(n / 3) suffices (5 n / 3) where a transform of every frequency takes 2 n - 1. The
// slots past the input are zeros: for every n that takes M, n <= 3 M / 5 + 1, so most of them are known at compile time
// and the first radix folds them away, as the last one drops the outputs that no n uses.
//
//   n = 509: M = 900 where a power of two took 1024; n = 257: 440 (1024); n = 601: 1024 (2048)
//
// Bound by vector arithmetic and LDS, four M-point transforms a pass (509: two wavefronts a SIMD, issuing vector
// instructions about 80 % of the row pass's time). A unit's loads are issued together, before any is used: where each
// was used under its slot's condition the compiler waited for one before it issued the next, 2.44 / 1.97 us a position at
// 509^2 against 2.09 / 1.62, and 2.80 / 2.21 against 2.06 / 1.52 where the waves come from HBM (4,096 positions a launch).
// Milliseconds per launch on an MI355X, row / column pass, against the passes on power-of-two convolutions that were
// here before (register-resident for 257..512, else in LDS):
//   131^2 (512 positions)  0.066 / 0.049   0.336 / 0.235     613^2 (123)   0.379 / 0.316   2.04 / 1.46
//   211^2 (512)            0.164 / 0.138   0.564 / 0.371     863^2 (123)   1.02 / 0.96     3.24 / 2.28
//   347^2 (256)            0.297 / 0.234   0.422 / 0.335     1021^2 (88)   1.47 / 1.12     2.80 / 2.03
//   509^2 (119)            0.249 / 0.193   0.300 / 0.300     509^2 (4096)  8.4 / 6.2       8.8 / 7.3
#pragma once

#include "sk_pair.h"

namespace sk {

// The convolution lengths. A length n takes the first that fits; steps of about a tenth keep the padding small.
constexpr int kBlueLengths[] = {112, 128, 144, 160, 180, 200, 224, 252, 280, 320, 360, 400, 440, 480, 528, 576, 624,
                                672, 720, 784, 840, 900, 960, 1024, 1152, 1280, 1440, 1536, 1728};
constexpr int kBlueCount = sizeof(kBlueLengths) / sizeof(int);

// the largest grid length that takes M points: n + 2 floor(n / 3) <= M, and 2 n - 1 <= M
template <int M>
struct BlueReach {
  static constexpr int band_n() {
    int n = 1;
    while (n + 1 + 2 * ((n + 1) / 3) <= M) ++n;
    return n;
  }
  static constexpr int N = band_n(), H = N / 3;  // the largest n, and the largest kept |k|
  static constexpr int FULL_N = (M + 1) / 2;
};

// The convolution of a line in layout I (u, on return too) with the kernel whose transform is kh. ST: slots from one LDS
// position to the next (columns side by side). It begins with writes to the slots that the same lane reads at its end,
// so convolutions follow one another without a barrier between them.
template <int M, int ST>
__device__ __forceinline__ void blue_convolve(float2 (&u)[PairShape<M>::RA], float2* bi, float2* bq, bool on_i,
                                              bool on_q, const float2* w, const float2* __restrict__ kh) {
  using S = PairShape<M>;
  constexpr int RA = S::RA, RB = S::RB, S1 = S::S1;
  rdft<RA, -1>(u);
  if (on_i) {
#pragma unroll
    for (int r = 0; r < RA; ++r) bi[r * S1 * ST] = u[r];
  }
  __syncthreads();
  float2 v[RB];
#pragma unroll
  for (int p = 0; p < RB; ++p) v[p] = cmul(bq[p * ST], w[RA * p]);
  rdft<RB, -1>(v);
#pragma unroll
  for (int p = 0; p < RB; ++p) v[p] = cmul(v[p], kh[RA * p]);
  rdft<RB, +1, true>(v);
  if (on_q) {
#pragma unroll
    for (int p = 0; p < RB; ++p) bq[p * ST] = cmulc(v[p], w[M + RA * p]);
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < RA; ++r) u[r] = bi[r * S1 * ST];
  rdft<RA, +1, true>(u);
}

// Groups of slots i + RB r (every lane i) of a centred spectrum: low frequencies k = slot <= H, high ones k = slot - M
// >= -H, or slots between, zero for every n.
template <int M>
__host__ __device__ constexpr int blue_group(int r) {
  constexpr int RB = PairShape<M>::RB, H = BlueReach<M>::H;
  return RB * r <= H ? PAIR_LOW : RB * (r + 1) - 1 >= M - H ? PAIR_HIGH : PAIR_BAND;
}

// Row pass: compact line -> inverse [-> exit plane] [-> * t -> forward -> compact line], or a full-width wave -> * t ->
// forward -> compact line. Only the band of that forward transform is used, so the band's convolution does: one wave of
// 509^2 enters in 11.7 us, against 26.9 through the 1024 points that every frequency takes.
template <int M>
__global__ void __launch_bounds__(PairShape<M>::NT, PairShape<M>::ROW_WAVES) row_blue_kernel(RowArgs a, BlueLine f,
                                                                                           int batch, int rounds) {
  using S = PairShape<M>;
  constexpr int RA = S::RA, RB = S::RB, S1 = S::S1, L = S::L, NMAX = BlueReach<M>::N;
  __shared__ float2 lds[L * S::LS];
  __shared__ float2 tab[2 * M];
  const int tid = threadIdx.x;
  for (int e = tid; e < 2 * M; e += S::NT) tab[e] = f.pair[e];
  __syncthreads();
  const int li = tid / RB, i = tid - li * RB;
  const int lq = tid / RA, q = tid - lq * RA;
  const bool on_i = li < L, on_q = lq < L;
  float2* bi = lds + (on_i ? li : 0) * S::LS + i;
  float2* bq = lds + (on_q ? lq : 0) * S::LS + q * S1;
  const int n = a.ny;
  const long long gw = (long long)a.nx * a.nc, units = (long long)a.nx * batch;
#pragma unroll 1
  for (int round = 0; round < rounds; ++round) {
    const long long u0 = ((long long)blockIdx.x * rounds + round) * L;
    if (u0 >= units) break;  // uniform over the block
    const long long ui = u0 + li;
    const bool live = on_i && ui < units;
    const int x = live ? int((unsigned)ui / (unsigned)batch) : 0, b = live ? int(ui - (long long)x * batch) : 0;
    int il = i, ql = q;
    asm volatile("" : "+v"(il), "+v"(ql));  // as in row_pair_kernel
    float2* g = a.G + b * gw + (long long)x * a.nc;
    float2 u[RA];
    const int high = M - n + a.kept_shift;  // compact column of a high slot: slot - high
    const float2* t = a.t + (long long)x * n;
    if (a.flags & ROW_INV) {
      // every load first (a slot without a value reads the line's first), then the chirp and the zeros
#pragma unroll
      for (int r = 0; r < RA; ++r) {
        const int group = blue_group<M>(r), s = il + RB * r;
        if (group == PAIR_LOW) u[r] = g[s <= a.kept_hi ? s : 0];
        if (group == PAIR_HIGH) u[r] = g[s >= M - n + a.kept_lo ? s - high : 0];
      }
#pragma unroll
      for (int r = 0; r < RA; ++r) {
        const int group = blue_group<M>(r), s = il + RB * r;
        if (group == PAIR_BAND) {
          u[r] = make_float2(0.f, 0.f);
        } else {
          const bool in = group == PAIR_LOW ? s <= a.kept_hi : s >= M - n + a.kept_lo;
          const float2 z = cmulc(u[r], f.chirp[in ? (group == PAIR_LOW ? s : M - s) : 0]);
          u[r] = in ? z : make_float2(0.f, 0.f);
        }
      }
      blue_convolve<M, 1>(u, bi, bq, on_i, on_q, tab + ql, f.inverse + ql);
      if ((a.flags & ROW_WRITE_PLANE) && live) {
        float2* pl = a.plane + b * a.plane_stride + (long long)x * n;
#pragma unroll
        for (int r = 0; r < RA; ++r) {
          const int s = il + RB * r;
          if (RB * r < NMAX && s < n) pl[s] = cscale(cmulc(u[r], f.chirp[s]), a.out_scale);
        }
      }
      if (!(a.flags & ROW_FWD)) continue;
      // the inverse's closing chirp and the forward's opening one cancel; t is taken as zero past n
#pragma unroll
      for (int r = 0; r < RA; ++r) {
        const int s = il + RB * r;
        if (RB * r >= NMAX) {
          u[r] = make_float2(0.f, 0.f);
        } else {
          const float2 p = cmul(u[r], t[s < n ? s : 0]);
          u[r] = s < n ? p : make_float2(0.f, 0.f);
        }
      }
    } else {  // a full-width wave in real space
      const float2* in = a.in_full + b * a.in_full_stride + (long long)x * n;
#pragma unroll
      for (int r = 0; r < RA; ++r)
        if (RB * r < NMAX) u[r] = in[il + RB * r < n ? il + RB * r : 0];
#pragma unroll
      for (int r = 0; r < RA; ++r) {
        const int s = il + RB * r, sx = s < n ? s : 0;
        if (RB * r >= NMAX) {
          u[r] = make_float2(0.f, 0.f);
        } else {
          const float2 p = cmul(cmul(u[r], t[sx]), f.chirp[sx]);
          u[r] = s < n ? p : make_float2(0.f, 0.f);
        }
      }
    }
    blue_convolve<M, 1>(u, bi, bq, on_i, on_q, tab + ql, f.forward + ql);
    if (live) {
#pragma unroll
      for (int r = 0; r < RA; ++r) {
        const int group = blue_group<M>(r), s = il + RB * r;
        if (group == PAIR_LOW) {
          if (s <= a.kept_hi) g[s] = cmul(u[r], f.chirp[s]);
        } else if (group == PAIR_HIGH) {
          if (s >= M - n + a.kept_lo) g[s - high] = cmul(u[r], f.chirp[M - s]);
        }
      }
    }
  }
}

// Column pass: forward, * P, then inverse and store (a middle slice), or the spectra stored (the last slice: the
// detectors read them).
template <int M>
__global__ void __launch_bounds__(PairShape<M>::CT, PairShape<M>::COL_WAVES) col_blue_kernel(ColArgs a, BlueLine f,
                                                                                           int batch, int rounds,
                                                                                           int tiles) {
  using S = PairShape<M>;
  constexpr int RA = S::RA, RB = S::RB, S1 = S::S1, TC = S::TC, NP = S::NP, NMAX = BlueReach<M>::N;
  __shared__ float2 lds[NP * TC * S::LS];
  __shared__ float2 tab[2 * M];
  const int tid = threadIdx.x;
  for (int e = tid; e < 2 * M; e += S::CT) tab[e] = f.pair[e];
  __syncthreads();
  const int cb = tid % TC, lane = tid / TC;
  const int ni = lane / RB, i = lane - ni * RB;
  const int nq = lane / RA, q = lane - nq * RA;
  const bool on_i = ni < NP, on_q = nq < NP;
  float2* bi = lds + (on_i ? ni : 0) * TC * S::LS + i * TC + cb;
  float2* bq = lds + (on_q ? nq : 0) * TC * S::LS + q * S1 * TC + cb;
  const int per_xcd = gridDim.x / 8, un = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;  // as in col_pair_kernel
  const int2 unit = make_int2(un % tiles, un / tiles);
  const int c = unit.x * TC + cb;
  const bool kept = c < a.nc && a.keep[c] >= 0;
  const int n = a.nx;
  const long long gw = (long long)a.nx * a.nc;
#pragma unroll 1
  for (int round = 0; round < rounds; ++round) {
    const long long p0 = ((long long)unit.y * rounds + round) * NP;
    if (p0 >= batch) break;  // uniform over the block
    const bool live = on_i && kept && p0 + ni < batch;
    char* base = reinterpret_cast<char*>(a.G + p0 * gw + unit.x * TC);
    int il = i, ql = q;
    asm volatile("" : "+v"(il), "+v"(ql));
    const unsigned start = live ? unsigned(ni * gw + cb) * 8u : 0u, row = unsigned(a.nc) * 8u;
    auto at = [&](int x) -> float2& { return *reinterpret_cast<float2*>(base + (start + unsigned(x) * row)); };
    float2 u[RA];
    // as in the row pass: every load first, then the chirp and the zeros
#pragma unroll
    for (int r = 0; r < RA; ++r)
      if (RB * r < NMAX) u[r] = at(live && il + RB * r < n ? il + RB * r : 0);
#pragma unroll
    for (int r = 0; r < RA; ++r) {
      const int s = il + RB * r;
      if (RB * r < NMAX) {
        const float2 z = cmul(u[r], f.chirp[s < n ? s : 0]);
        u[r] = live && s < n ? z : make_float2(0.f, 0.f);
      } else {
        u[r] = make_float2(0.f, 0.f);
      }
    }
    blue_convolve<M, TC>(u, bi, bq, on_i, on_q, tab + ql, f.forward + ql);
    const char* pb = reinterpret_cast<const char*>(a.P + unit.x * TC);
    const unsigned cbo = kept ? unsigned(cb) * 8u : 0u;
    const bool back = (a.flags & COL_INV) != 0;
#pragma unroll
    for (int r = 0; r < RA; ++r) {
      const int group = blue_group<M>(r), s = il + RB * r;
      const bool low = group == PAIR_LOW;
      if (group == PAIR_BAND) {
        u[r] = make_float2(0.f, 0.f);
      } else {
        const bool in = low ? s <= f.hi : s >= M - f.lo;  // kx = s, or s - M + n
        const int kx = in ? (low ? s : s - M + n) : 0;
        const float2 p = cmul(u[r], *reinterpret_cast<const float2*>(pb + (cbo + unsigned(kx) * row)));
        u[r] = in ? p : make_float2(0.f, 0.f);
      }
    }
    if (!back) {
      // the spectra in the grid's own order, the band that P prunes as zeros (the closing chirp is left out: only
      // intensities are read)
      if (live) {
#pragma unroll
        for (int r = 0; r < RA; ++r) {
          const int group = blue_group<M>(r), s = il + RB * r;
          if (group == PAIR_HIGH && s >= M - f.lo) at(s - M + n) = u[r];
          else if (s < n - f.lo) at(s) = (group == PAIR_LOW && s <= f.hi) ? u[r] : make_float2(0.f, 0.f);
        }
      }
      continue;
    }
    blue_convolve<M, TC>(u, bi, bq, on_i, on_q, tab + ql, f.inverse + ql);
    if (live) {
#pragma unroll
      for (int r = 0; r < RA; ++r) {
        const int s = il + RB * r;
        if (RB * r < NMAX && s < n) at(s) = cmulc(u[r], f.chirp[s]);
      }
    }
  }
}

// Full-width row pass (every frequency, natural order, M >= 2 n - 1): in_full -> one transform -> out_full, or in_full
// -> [inverse] -> * t -> forward -> compact line (the first slice, from a wave that is not compact).
template <int M>
__global__ void __launch_bounds__(PairShape<M>::NT, PairShape<M>::ROW_WAVES) row_blue_full_kernel(RowArgs a, BlueLine f,
                                                                                                int batch, int rounds) {
  using S = PairShape<M>;
  constexpr int RA = S::RA, RB = S::RB, S1 = S::S1, L = S::L, NMAX = BlueReach<M>::FULL_N;
  __shared__ float2 lds[L * S::LS];
  __shared__ float2 tab[2 * M];
  const int tid = threadIdx.x;
  for (int e = tid; e < 2 * M; e += S::NT) tab[e] = f.pair[e];
  __syncthreads();
  const int li = tid / RB, i = tid - li * RB;
  const int lq = tid / RA, q = tid - lq * RA;
  const bool on_i = li < L, on_q = lq < L;
  float2* bi = lds + (on_i ? li : 0) * S::LS + i;
  float2* bq = lds + (on_q ? lq : 0) * S::LS + q * S1;
  const int n = a.ny;
  const long long units = (long long)a.nx * batch;
  const bool mul = (a.flags & ROW_MUL_T) != 0;
#pragma unroll 1
  for (int round = 0; round < rounds; ++round) {
    const long long u0 = ((long long)blockIdx.x * rounds + round) * L;
    if (u0 >= units) break;  // uniform over the block
    const long long ui = u0 + li;
    const bool live = on_i && ui < units;
    const int x = live ? int((unsigned)ui / (unsigned)batch) : 0, b = live ? int(ui - (long long)x * batch) : 0;
    int il = i, ql = q;
    asm volatile("" : "+v"(il), "+v"(ql));
    const float2* in = a.in_full + b * a.in_full_stride + (long long)x * n;
    const float2* t = a.t + (long long)x * n;
    float sign = (a.flags & ROW_INV) ? -1.f : 1.f;  // the inverse: conjugate in and out
    float2 u[RA];
#pragma unroll
    for (int r = 0; r < RA; ++r) {
      const int s = il + RB * r, sx = s < n ? s : 0;
      u[r] = make_float2(0.f, 0.f);
      if (RB * r < NMAX) {
        float2 z = in[sx];
        if (mul && sign > 0) z = cmul(z, t[sx]);
        z = cmul(make_float2(z.x, sign * z.y), f.chirp[sx]);
        if (s < n) u[r] = z;
      }
    }
#pragma unroll 1
    for (;;) {
      blue_convolve<M, 1>(u, bi, bq, on_i, on_q, tab + ql, f.full + ql);
      if (sign > 0 || !mul) break;
      // after the inverse: conjugated back, * t, then the forward's opening chirp, which its closing one cancels
      sign = 1.f;
#pragma unroll
      for (int r = 0; r < RA; ++r) {
        const int s = il + RB * r;
        const float2 z = cmul(make_float2(u[r].x, -u[r].y), t[s < n ? s : 0]);
        u[r] = RB * r < NMAX && s < n ? z : make_float2(0.f, 0.f);
      }
    }
    if (live && (a.flags & ROW_OUT_COMPACT)) {
      float2* g = a.G + b * ((long long)a.nx * a.nc) + (long long)x * a.nc;
#pragma unroll
      for (int r = 0; r < RA; ++r) {
        const int s = il + RB * r;
        if (RB * r < NMAX && s < n && (s <= a.kept_hi || s >= a.kept_lo))
          g[s <= a.kept_hi ? s : s - a.kept_shift] = cmul(u[r], f.chirp[s]);
      }
    } else if (live) {
      float2* out = a.out_full + b * a.out_full_stride + (long long)x * n;
#pragma unroll
      for (int r = 0; r < RA; ++r) {
        const int s = il + RB * r;
        if (RB * r < NMAX && s < n) {
          const float2 z = cmul(u[r], f.chirp[s]);
          out[s] = make_float2(z.x * a.out_scale, sign * a.out_scale * z.y);
        }
      }
    }
  }
}

// Full-width column pass: G -> [forward, * P] -> [inverse] -> G, or (GENERATE, a scan's first pass) the generated probe ->
// inverse -> G, which is one convolution and held apart for its registers: with the other modes around it the 1024 points
// of 509^2 spilled 196 bytes a lane, 3.77 ms a launch of 2,048 positions against 2.46 without.
template <int M, bool GENERATE>
__global__ void __launch_bounds__(PairShape<M>::CT, PairShape<M>::COL_WAVES) col_blue_full_kernel(ColArgs a, BlueLine f,
                                                                                                int batch, int rounds,
                                                                                                int tiles) {
  using S = PairShape<M>;
  constexpr int RA = S::RA, RB = S::RB, S1 = S::S1, TC = S::TC, NP = S::NP, NMAX = BlueReach<M>::FULL_N;
  __shared__ float2 lds[NP * TC * S::LS];
  __shared__ float2 tab[2 * M];
  const int tid = threadIdx.x;
  for (int e = tid; e < 2 * M; e += S::CT) tab[e] = f.pair[e];
  __syncthreads();
  const int cb = tid % TC, lane = tid / TC;
  const int ni = lane / RB, i = lane - ni * RB;
  const int nq = lane / RA, q = lane - nq * RA;
  const bool on_i = ni < NP, on_q = nq < NP;
  float2* bi = lds + (on_i ? ni : 0) * TC * S::LS + i * TC + cb;
  float2* bq = lds + (on_q ? nq : 0) * TC * S::LS + q * S1 * TC + cb;
  const int per_xcd = gridDim.x / 8, un = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
  const int2 unit = make_int2(un % tiles, un / tiles);
  const int c = unit.x * TC + cb;
  const int iy = c < a.nc ? a.keep[c] : -1;
  const bool kept = iy >= 0;
  const int n = a.nx, fl = GENERATE ? COL_GENERATE | COL_INV | COL_OUT : a.flags & ~COL_GENERATE;
  const long long gw = (long long)a.nx * a.nc;
#pragma unroll 1
  for (int round = 0; round < rounds; ++round) {
    const long long p0 = ((long long)unit.y * rounds + round) * NP, b = p0 + ni;
    if (p0 >= batch) break;
    const bool live = on_i && kept && b < batch;
    char* base = reinterpret_cast<char*>(a.G + p0 * gw + unit.x * TC);
    int il = i, ql = q;
    asm volatile("" : "+v"(il), "+v"(ql));
    const unsigned start = live ? unsigned(ni * gw + cb) * 8u : 0u, row = unsigned(a.nc) * 8u;
    auto at = [&](int x) -> float2& { return *reinterpret_cast<float2*>(base + (start + unsigned(x) * row)); };
    float sign = (fl & COL_FWD) ? 1.f : -1.f;  // the inverse: conjugate in and out
    float2 u[RA];
    if constexpr (GENERATE) {  // spectrum times ramps; a lane without a value reads element 0
      const float2* spec = a.spec + (live ? iy : 0);
      const float2* rx = a.rx + (live ? b * n : 0);
      const float2 ry = a.ry[live ? b * a.ny + iy : 0];
#pragma unroll
      for (int r = 0; r < RA; ++r) {
        if (RB * r < NMAX) {
          const int s = il + RB * r, sx = live && s < n ? s : 0;
          u[r] = cmul(cmul(spec[(long long)sx * a.ny], rx[sx]), ry);
        }
      }
    } else {
#pragma unroll
      for (int r = 0; r < RA; ++r)
        if (RB * r < NMAX) u[r] = at(live && il + RB * r < n ? il + RB * r : 0);
    }
#pragma unroll
    for (int r = 0; r < RA; ++r) {
      const int s = il + RB * r;
      if (RB * r < NMAX) {
        const float2 t = cmul(make_float2(u[r].x, sign * u[r].y), f.chirp[s < n ? s : 0]);
        u[r] = live && s < n ? t : make_float2(0.f, 0.f);
      } else {
        u[r] = make_float2(0.f, 0.f);
      }
    }
#pragma unroll 1
    for (;;) {
      blue_convolve<M, TC>(u, bi, bq, on_i, on_q, tab + ql, f.full + ql);
      if (sign < 0 || !(fl & COL_INV)) break;
      // after the forward transform: its closing chirp, * P, then the inverse's opening one (conjugated)
      sign = -1.f;
#pragma unroll
      for (int r = 0; r < RA; ++r) {
        const int s = il + RB * r;
        float2 z = make_float2(0.f, 0.f);
        if (RB * r < NMAX && live && s < n) {
          z = cmul(u[r], f.chirp[s]);
          if (fl & COL_MUL_P) z = cmul(z, a.P[(long long)s * a.nc + c]);
          z = cmul(make_float2(z.x, -z.y), f.chirp[s]);
        }
        u[r] = z;
      }
    }
    if (live) {
#pragma unroll
      for (int r = 0; r < RA; ++r) {
        const int s = il + RB * r;
        if (RB * r < NMAX && s < n) {
          float2 z = cmul(u[r], f.chirp[s]);
          if ((fl & COL_FWD) && !(fl & COL_INV) && (fl & COL_MUL_P)) z = cmul(z, a.P[(long long)s * a.nc + c]);
          at(s) = make_float2(z.x, sign * z.y);
        }
      }
    }
  }
}

}  // namespace sk
