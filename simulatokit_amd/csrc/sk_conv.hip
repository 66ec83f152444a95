// sk_conv.hip — the layers of the HAADF surrogate (build-only; the reference has no learned part): 5 x 5
// convolutions with circular padding (the cells are periodic), bfloat16 weights and float32 activations and
// accumulation, their two backward passes, the fixed separable resampling of the output to the scan grid, the squared
// error's gradient and an Adam step that keeps float32 master weights and publishes their bfloat16 rounding.
// Every reduction runs in a fixed order, so a training run is reproducible bit for bit.

#include <hip/hip_runtime.h>

#include <cstdint>

#include "sk_internal.h"
#include "sk_mfma.h"
#include "../../include/simulato_surrogate.h"

namespace sk {
namespace {

constexpr int kTile = 16;  // output tile edge
constexpr int kCo = 8;     // output channels per block
constexpr int kCi = 8;     // input channels per LDS chunk
constexpr int kHalo = kTile + 4;

__device__ __forceinline__ float bf16_to_f32(uint16_t b) { return __uint_as_float(uint32_t(b) << 16); }

__device__ __forceinline__ uint16_t f32_to_bf16(float f) {
  uint32_t u = __float_as_uint(f);
  u += 0x7fffu + ((u >> 16) & 1u);
  return uint16_t(u >> 16);
}

__device__ __forceinline__ int wrap(int i, int n) { return i < 0 ? i + n : (i >= n ? i - n : i); }

// y[b][co][p] = bias[co] + sum_{ci, ky, kx} w[co][ci][ky][kx] x[b][ci][p + (ky - 2, kx - 2) mod (h, w)], then ReLU if
// asked. Block: a 16 x 16 tile of one image and 8 output channels; the input tile with its 2-pixel halo and the
// weights (as [ci][k][co], so one read serves eight output channels) go through LDS in chunks of 8 input channels.
__global__ void __launch_bounds__(256) conv5_forward_kernel(const float* __restrict__ x, const uint16_t* __restrict__ wt,
                                                            const float* __restrict__ bias, int cin, int cout, int h,
                                                            int w, int relu, float* __restrict__ y) {
  __shared__ float tile[kCi][kHalo][kHalo + 1];
  __shared__ float4 wsh[kCi][25][kCo / 4];
  const int tx = threadIdx.x % kTile, ty = threadIdx.x / kTile;
  const int tiles_x = w / kTile;
  const int x0 = (blockIdx.x % tiles_x) * kTile, y0 = (blockIdx.x / tiles_x) * kTile;
  const int co0 = blockIdx.y * kCo;
  const long long b = blockIdx.z;
  float acc[kCo];
#pragma unroll
  for (int c = 0; c < kCo; ++c) acc[c] = (bias && co0 + c < cout) ? bias[co0 + c] : 0.f;
  for (int ci0 = 0; ci0 < cin; ci0 += kCi) {
    for (int idx = threadIdx.x; idx < kCi * kHalo * kHalo; idx += 256) {
      const int c = idx / (kHalo * kHalo), r = idx % (kHalo * kHalo), yy = r / kHalo, xx = r % kHalo;
      float v = 0.f;
      if (ci0 + c < cin)
        v = x[((b * cin + ci0 + c) * h + wrap(y0 + yy - 2, h)) * (long long)w + wrap(x0 + xx - 2, w)];
      tile[c][yy][xx] = v;
    }
    for (int idx = threadIdx.x; idx < kCi * 25 * kCo; idx += 256) {
      const int c = idx / (25 * kCo), r = idx % (25 * kCo), k = r / kCo, o = r % kCo;
      float v = 0.f;
      if (ci0 + c < cin && co0 + o < cout) v = bf16_to_f32(wt[((size_t)(co0 + o) * cin + ci0 + c) * 25 + k]);
      reinterpret_cast<float*>(&wsh[c][k][0])[o] = v;
    }
    __syncthreads();
    for (int c = 0; c < kCi; ++c)
#pragma unroll
      for (int ky = 0; ky < 5; ++ky)
#pragma unroll
        for (int kx = 0; kx < 5; ++kx) {
          const float v = tile[c][ty + ky][tx + kx];
          const float4 wa = wsh[c][ky * 5 + kx][0], wb = wsh[c][ky * 5 + kx][1];
          acc[0] += wa.x * v;
          acc[1] += wa.y * v;
          acc[2] += wa.z * v;
          acc[3] += wa.w * v;
          acc[4] += wb.x * v;
          acc[5] += wb.y * v;
          acc[6] += wb.z * v;
          acc[7] += wb.w * v;
        }
    __syncthreads();
  }
#pragma unroll
  for (int c = 0; c < kCo; ++c) {
    if (co0 + c >= cout) break;
    float v = acc[c];
    if (relu) v = v > 0.f ? v : 0.f;
    y[((b * cout + co0 + c) * h + y0 + ty) * (long long)w + x0 + tx] = v;
  }
}

// Matrix-core forward convolution for up to 32 input and 32 output channels (every layer of the surrogate, and the
// backward pass over the data of each): an implicit GEMM, y[co][p] = sum over k = (tap, ci) of W[co][k] x[ci][p + tap],
// on v_mfma_f32_32x32x16_bf16 (A = the weights, 32 output channels x 16 k; B = 16 k x 32 pixels of one output row).
// The weights are bfloat16 already, so A is exact; each activation enters as a bfloat16 pair x = hi + lo (lo =
// bf16(x - hi), leaving a relative 2^-18), two products accumulated in float32. Block: W wavefronts, each R output
// rows of 32 pixels (R 32 x 32 tiles); the input rows with their circular halo (W R + 4 rows x 36 columns x CINP
// channels, the channels past cin zero) sit in LDS as the hi and lo halves, [row][column][channel] with the channels
// padded to CINP + 8 (a 16-byte read per lane; the padding spreads a row's 32 pixels over all 64 banks). The weights
// come as wtm[tap][32][CINP] (sk_conv5_weights_tap_major: the rows past cout and the columns past cin zero), 8
// consecutive channels per lane and k-step; only the cout real output channels are stored. `mask` (may be null): a
// ReLU layer's output of y's shape, y is zero where it is not positive.
// Bound by the read of the tiles and the matrix cores in turn (a CU's two blocks load and multiply in step): 32 to 32
// channels at 128 x 128, 1 image 16.8 -> 9.7 us, 4: 23.6 -> 17.1, 16: 59.2 -> 51.6 (matrix cores busy a quarter of it),
// against one load in flight per thread, weights loaded tap by tap and every LDS row read once per output row.
constexpr int kMfCols = 32, kMfHC = kMfCols + 4;

typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));  // four floats at any float's address

template <int CINP, int R, int W>
__global__ void __launch_bounds__(64 * W, 2) conv5_forward_mfma_kernel(const float* __restrict__ x,
                                                                       const __bf16* __restrict__ wtm,
                                                                       const float* __restrict__ bias, int cin,
                                                                       int cout, int h, int w, int relu,
                                                                       const float* __restrict__ mask,
                                                                       float* __restrict__ y) {
  constexpr int CP = CINP + 8, HR = W * R + 4, STEPS = CINP / 16;
  __shared__ __align__(16) __bf16 xhi[HR * kMfHC * CP];
  __shared__ __align__(16) __bf16 xlo[HR * kMfHC * CP];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int tiles_x = w / kMfCols;
  const int x0 = (blockIdx.x % tiles_x) * kMfCols, y0 = (blockIdx.x / tiles_x) * (W * R);
  const long long b = blockIdx.y;
  const int n = lane & 31, half = lane >> 5;
  // A[m = output channel n][k = 8 half + j] of every kx and k-step of tap row ky, loaded one tap row ahead
  const __bf16* wl = wtm + n * CINP + 8 * half;
  bf16x8 a[5][5 * STEPS];
#pragma unroll
  for (int q = 0; q < 5 * STEPS; ++q)
    a[0][q] = *reinterpret_cast<const bf16x8*>(wl + (q / STEPS) * 32 * CINP + 16 * (q % STEPS));
  // The input rows y0 - 2 .. y0 + W R + 1 (circular), every channel. A task is 8 channels of 4 pixels, columns x0 - 4 +
  // 4 g .. (the tile takes x0 - 2 .. x0 + 33; w is a multiple of 4, so a group wraps as a whole), written to LDS as one
  // 16-byte hi and lo per pixel. Every task of a thread is loaded before the first is used.
  constexpr int GROUPS = kMfCols / 4 + 2, TASKS = (CINP / 8) * HR * GROUPS, PER = (TASKS + 64 * W - 1) / (64 * W);
  f32x4u v[PER][8];
#pragma unroll
  for (int e = 0; e < PER; ++e) {
    const int task = tid + 64 * W * e, g = task % GROUPS, r = task / GROUPS, rr = r % HR, c8 = 8 * (r / HR);
    const long long pix = (long long)wrap(y0 + rr - 2, h) * w + wrap(x0 - 4 + 4 * g, w);
#pragma unroll
    for (int j = 0; j < 8; ++j)
      v[e][j] = c8 + j < cin ? *reinterpret_cast<const f32x4u*>(x + (b * cin + c8 + j) * (long long)h * w + pix)
                             : f32x4u{0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int e = 0; e < PER; ++e) {
    const int task = tid + 64 * W * e, g = task % GROUPS, r = task / GROUPS, rr = r % HR, c8 = 8 * (r / HR);
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int cc = 4 * g + p - 2;
      float u[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) u[j] = v[e][j][p];
      bf16x8 hi, lo;
      split_bf16(u, hi, lo);
      if (cc >= 0 && cc < kMfHC && task < TASKS) {
        *reinterpret_cast<bf16x8*>(xhi + (rr * kMfHC + cc) * CP + c8) = hi;
        *reinterpret_cast<bf16x8*>(xlo + (rr * kMfHC + cc) * CP + c8) = lo;
      }
    }
  }
  __syncthreads();
  f32x16 acc[R][2];
#pragma unroll
  for (int t = 0; t < R; ++t)
#pragma unroll
    for (int q = 0; q < 16; ++q) acc[t][0][q] = acc[t][1][q] = 0.f;
  // Halo row rr serves every output row t of the wavefront with tap row ky = rr - t: its values are read once, and each
  // output's products keep the order (tap row, tap column, channels).
#pragma unroll
  for (int rr = 0; rr < R + 4; ++rr) {
    if (rr < 4) {
#pragma unroll
      for (int q = 0; q < 5 * STEPS; ++q)
        a[rr + 1][q] = *reinterpret_cast<const bf16x8*>(wl + ((rr + 1) * 5 + q / STEPS) * 32 * CINP + 16 * (q % STEPS));
    }
#pragma unroll
    for (int q = 0; q < 5 * STEPS; ++q) {
      const int slot = ((wv * R + rr) * kMfHC + n + q / STEPS) * CP + 16 * (q % STEPS) + 8 * half;
      const bf16x8 bh = *reinterpret_cast<const bf16x8*>(xhi + slot);
      const bf16x8 bl = *reinterpret_cast<const bf16x8*>(xlo + slot);
#pragma unroll
      for (int t = 0; t < R; ++t) {
        if (rr - t < 0 || rr - t > 4) continue;
        acc[t][1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[rr - t][q], bl, acc[t][1], 0, 0, 0);
        acc[t][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[rr - t][q], bh, acc[t][0], 0, 0, 0);
      }
    }
  }
  // D register q of lane l: D[8 (q / 4) + 4 (l / 32) + q % 4][l % 32]: output channel, pixel n
#pragma unroll
  for (int t = 0; t < R; ++t) {
    const int oy = y0 + wv * R + t;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int co = 8 * (q / 4) + 4 * half + (q % 4);
      if (co >= cout) continue;
      const long long at = ((b * cout + co) * h + oy) * (long long)w + x0 + n;
      float o = acc[t][1][q] + acc[t][0][q] + (bias ? bias[co] : 0.f);
      if (relu) o = o > 0.f ? o : 0.f;
      if (mask && !(mask[at] > 0.f)) o = 0.f;
      y[at] = o;
    }
  }
}

// The tap-major bfloat16 layout the matrix-core kernel reads, wtm[tap][32][kp] with kp = 16 for up to 16 input
// channels of the convolution it serves and 32 above: wtm[tap][co][ci] = w[co][ci][tap] (flip = 0; rows = cout,
// columns = cin), or the flipped, transposed kernel of the backward pass over the data, wtm[tap][ci][co] =
// w[co][ci][24 - tap] (flip = 1; rows = cin, columns = cout); the rows and columns past those zero.
__global__ void weights_tap_major_kernel(const uint16_t* __restrict__ wt, int cin, int cout, int flip, int kp,
                                         uint16_t* __restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= 25 * 32 * kp) return;
  const int col = i % kp, row = (i / kp) % 32, tap = i / (32 * kp);
  const int co = flip ? col : row, ci = flip ? row : col, src_tap = flip ? 24 - tap : tap;
  out[i] = (co < cout && ci < cin) ? wt[((size_t)co * cin + ci) * 25 + src_tap] : uint16_t(0);
}

// Matrix-core gradient of the weights for up to 32 input and 32 output channels: dw[co][ci][tap] = sum over the
// pixels p of every image of dy[co][p] x[ci][p + tap], a GEMM of M = 32 output channels by N = 32 input channels per
// tap with the pixels as K, on v_mfma_f32_32x32x16_bf16 with both operands as bfloat16 hi + lo pairs and three
// products (lo hi, hi lo, hi hi; the dropped lo lo is a relative 2^-18). Work unit: a strip of 4 rows x 32 columns
// of one image; at most kWgBlocks blocks take equal runs of them, down the columns of strips, each keeping its sums in
// registers and writes them to its own slice of `partial`; a second kernel adds the slices in block order, so the
// result does not depend on the device or on timing. Block: 5 wavefronts, wavefront ky the five taps (ky, 0..4).
// LDS: x rows y0 - 2 .. y0 + 5, columns x0 - 8 .. x0 + 39 (circular; groups of 8 columns keep every 16-byte read
// aligned), [row][channel][column] with a 56-column stride, and dy rows y0 .. y0 + 3, columns x0 .. x0 + 31 with a
// 40-column stride (112- and 80-byte strides put 16 lanes' 16-byte reads on distinct banks); both as hi and lo.
// The x rows are a ring: the next strip down needs four new ones. Bound by the loads and the split into hi and lo, which
// the CU's other block covers in part: 16 images of 32 to 32 channels at 128 x 128 take 78 -> 60 us (matrix cores busy
// 18 us of them) with every load of a strip in flight and half the rows, against eight rows a strip, one load a
// thread at a time, and registers (177) for one block a CU.
// For output row r and k-step t (16 pixels from column 16 t), lane half h reads the 24 staged x columns 16 t + 8 h ..
// + 23 of its channel once; tap kx takes elements 6 + kx .. 13 + kx of them (odd kx by a 16-bit funnel shift).
constexpr int kWgWaves = 5, kWgRows = 4, kWgCols = 32, kWgXRows = kWgRows + 4;
constexpr int kWgXStride = 56, kWgDStride = 40, kWgXGroups = (kWgCols + 16) / 8, kWgDGroups = kWgCols / 8;
constexpr int kWgXPer = (4 * 32 * kWgXGroups + 64 * kWgWaves - 1) / (64 * kWgWaves);  // groups of 8 values a thread
constexpr int kWgDPer = (kWgRows * 32 * kWgDGroups + 64 * kWgWaves - 1) / (64 * kWgWaves);
constexpr int kWgBlocks = 512, kWgOut = 25 * 32 * 32;
static_assert(kWgBlocks * kWgOut + 2 * 32 * 64 == SK_CONV5_MFMA_WORKSPACE_FLOATS, "workspace size");

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void load8(const float* __restrict__ src, bool valid, float4 (&v)[2]) {
  v[0] = valid ? reinterpret_cast<const float4*>(src)[0] : make_float4(0.f, 0.f, 0.f, 0.f);
  v[1] = valid ? reinterpret_cast<const float4*>(src)[1] : make_float4(0.f, 0.f, 0.f, 0.f);
}
__device__ __forceinline__ void store8(const float4 (&v)[2], uint16_t* hi_at, uint16_t* lo_at, int slot) {
  const float u[8] = {v[0].x, v[0].y, v[0].z, v[0].w, v[1].x, v[1].y, v[1].z, v[1].w};
  bf16x8 h, l;
  split_bf16(u, h, l);
  *reinterpret_cast<u32x4*>(hi_at + slot) = __builtin_bit_cast(u32x4, h);
  *reinterpret_cast<u32x4*>(lo_at + slot) = __builtin_bit_cast(u32x4, l);
}

// elements o .. o + 7 of the 24-element window held as 12 packed pairs
template <int O>
__device__ __forceinline__ bf16x8 window8(const uint32_t (&wv)[12]) {
  u32x4 r;
  if constexpr (O % 2 == 0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = wv[O / 2 + i];
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = (wv[O / 2 + i] >> 16) | (wv[O / 2 + i + 1] << 16);
  }
  return __builtin_bit_cast(bf16x8, r);
}

__global__ void __launch_bounds__(64 * kWgWaves, 3) conv5_wgrad_mfma_kernel(const float* __restrict__ x,
                                                                            const float* __restrict__ dy, int cin,
                                                                            int cout, int h, int w, long long strips,
                                                                            float* __restrict__ partial) {
  __shared__ __align__(16) uint16_t xs[2][kWgXRows * 32 * kWgXStride];
  __shared__ __align__(16) uint16_t ds[2][kWgRows * 32 * kWgDStride];
  const int tid = threadIdx.x, lane = tid & 63, ky = tid >> 6;
  const int n = lane & 31, half = lane >> 5;
  f32x16 acc[5];
#pragma unroll
  for (int k = 0; k < 5; ++k)
#pragma unroll
    for (int q = 0; q < 16; ++q) acc[k][q] = 0.f;
  const int sy = h / kWgRows, sx = w / kWgCols;
  const long long s0 = blockIdx.x * strips / gridDim.x, s1 = (blockIdx.x + 1) * strips / gridDim.x;
  auto x_rows = [&](const float* xb, int y0, int x0, float4 (&v)[kWgXPer][2]) {  // halo rows y0 .. y0 + 3 of an image
#pragma unroll
    for (int k = 0; k < kWgXPer; ++k) {
      const int e = tid + 64 * kWgWaves * k, g = e % kWgXGroups, rc = e / kWgXGroups, ci = rc % 32, rr = (rc / 32) % 4;
      load8(xb + (long long)((ci < cin ? ci : 0) * h + wrap(y0 + rr, h)) * w + wrap(x0 - 8 + 8 * g, w), ci < cin, v[k]);
    }
  };
  auto x_store = [&](int y0, const float4 (&v)[kWgXPer][2]) {  // row y in slot (y + 2) mod 8
#pragma unroll
    for (int k = 0; k < kWgXPer; ++k) {
      const int e = tid + 64 * kWgWaves * k, g = e % kWgXGroups, rc = e / kWgXGroups, ci = rc % 32, rr = rc / 32;
      if (rr < 4) store8(v[k], xs[0], xs[1], (((y0 + 2 + rr) & 7) * 32 + ci) * kWgXStride + 8 * g);
    }
  };
#pragma unroll 1
  for (long long s = s0; s < s1; ++s) {
    // strip s: rows 4 (s mod sy) .. of columns 32 ((s / sy) mod sx) .. of image s / (sx sy)
    const int per_image = sx * sy, b = int(s / per_image), r0 = int(s - (long long)b * per_image);
    const int y0 = (r0 % sy) * kWgRows, x0 = (r0 / sy) * kWgCols;
    const float* xb = x + (long long)b * cin * h * w;
    const float* dyb = dy + (long long)b * cout * h * w;
    float4 xv[kWgXPer][2], dv[kWgDPer][2];
    x_rows(xb, y0 + 2, x0, xv);  // the lower four halo rows: the upper four are the strip before's
#pragma unroll
    for (int k = 0; k < kWgDPer; ++k) {
      const int e = tid + 64 * kWgWaves * k, g = e % kWgDGroups, rc = e / kWgDGroups, co = rc % 32, rr = (rc / 32) % 4;
      load8(dyb + (long long)((co < cout ? co : 0) * h + y0 + rr) * w + x0 + 8 * g, co < cout, dv[k]);
    }
    __syncthreads();  // the previous strip's reads are done
    if (s == s0 || y0 == 0) {  // the top of a column of strips: its upper halo rows too
      float4 uv[kWgXPer][2];
      x_rows(xb, y0 - 2, x0, uv);
      x_store(y0 - 2, uv);
    }
    x_store(y0 + 2, xv);
#pragma unroll
    for (int k = 0; k < kWgDPer; ++k) {
      const int e = tid + 64 * kWgWaves * k, g = e % kWgDGroups, rc = e / kWgDGroups;
      if (rc < kWgRows * 32) store8(dv[k], ds[0], ds[1], rc * kWgDStride + 8 * g);
    }
    __syncthreads();
#pragma unroll 1
    for (int r = 0; r < kWgRows; ++r) {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int da = (r * 32 + n) * kWgDStride + 16 * t + 8 * half;
        const bf16x8 ah = *reinterpret_cast<const bf16x8*>(ds[0] + da);
        const bf16x8 al = *reinterpret_cast<const bf16x8*>(ds[1] + da);
        const int xa = (((y0 + r + ky) & 7) * 32 + n) * kWgXStride + 16 * t + 8 * half;
        uint32_t wh[12], wl[12];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          const u32x4 vh = *reinterpret_cast<const u32x4*>(xs[0] + xa + 8 * i);
          const u32x4 vl = *reinterpret_cast<const u32x4*>(xs[1] + xa + 8 * i);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            wh[4 * i + j] = vh[j];
            wl[4 * i + j] = vl[j];
          }
        }
        acc[0] = mfma3(ah, al, window8<6>(wh), window8<6>(wl), acc[0]);
        acc[1] = mfma3(ah, al, window8<7>(wh), window8<7>(wl), acc[1]);
        acc[2] = mfma3(ah, al, window8<8>(wh), window8<8>(wl), acc[2]);
        acc[3] = mfma3(ah, al, window8<9>(wh), window8<9>(wl), acc[3]);
        acc[4] = mfma3(ah, al, window8<10>(wh), window8<10>(wl), acc[4]);
      }
    }
  }
  // D register q of lane l: D[co = 8 (q / 4) + 4 (l / 32) + q % 4][ci = l % 32]
  float* out = partial + (size_t)blockIdx.x * kWgOut;
#pragma unroll
  for (int kx = 0; kx < 5; ++kx)
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int co = 8 * (q / 4) + 4 * half + (q % 4);
      out[((ky * 5 + kx) * 32 + co) * 32 + n] = acc[kx][q];
    }
}

// dw[co][ci][tap] = the sum of the blocks' slices in a fixed order, for the real channels: a block takes 64
// consecutive outputs, its four wavefronts a quarter of the slices each (in block order, float64), and the quarters
// are added in order. The block after the outputs' (launched with db) adds the bias gradient's chunks.
constexpr int kBgChunks = 64;
__global__ void __launch_bounds__(256) wgrad_reduce_kernel(const float* __restrict__ partial, int blocks, int cin,
                                                           int cout, float* __restrict__ dw,
                                                           const double* __restrict__ bias_partial,
                                                           float* __restrict__ db) {
  __shared__ double part[4][64];
  if (blockIdx.x == kWgOut / 64) {
    const int co = threadIdx.x;
    if (co >= cout) return;
    double s = 0.0;
#pragma unroll 8
    for (int c = 0; c < kBgChunks; ++c) s += bias_partial[co * kBgChunks + c];
    db[co] = float(s);
    return;
  }
  const int o = threadIdx.x & 63, quarter = threadIdx.x >> 6;
  const int i = blockIdx.x * 64 + o;  // [tap][co][ci]
  const int per = (blocks + 3) / 4, g0 = quarter * per, g1 = g0 + per < blocks ? g0 + per : blocks;
  double s = 0.0;
#pragma unroll 8
  for (int g = g0; g < g1; ++g) s += partial[(size_t)g * kWgOut + i];
  part[quarter][o] = s;
  __syncthreads();
  if (quarter) return;
  const int ci = i % 32, co = (i / 32) % 32, tap = i / 1024;
  if (ci < cin && co < cout)
    dw[((size_t)co * cin + ci) * 25 + tap] = float(((part[0][o] + part[1][o]) + part[2][o]) + part[3][o]);
}

// db[co] = sum over images and pixels of dy[b][co][p], in a fixed order: block (co, chunk) sums one of kBgChunks
// contiguous ranges of the batch's pixels into partial[co][chunk] (float64), four pixels a load; wgrad_reduce_kernel's
// last block adds the chunks in order. Bound by the read of dy: 16 images of 32 x 128 x 128 (34 MB) took 12.4 us with a
// division per pixel.
__global__ void __launch_bounds__(256) bias_partial_kernel(const float* __restrict__ dy, int batch, int cout,
                                                           long long hw, double* __restrict__ partial) {
  __shared__ double red[256];
  const int co = blockIdx.x, chunk = blockIdx.y;
  const long long quads = hw / 4, total = batch * quads, len = (total + kBgChunks - 1) / kBgChunks;
  const long long i0 = chunk * len, i1 = i0 + len < total ? i0 + len : total;
  long long i = i0 + threadIdx.x, b = i / quads, at = i - b * quads;  // image b, its quad `at`
  double s = 0.0;
  for (; i < i1; i += 256, at += 256) {
    while (at >= quads) {
      at -= quads;
      ++b;
    }
    const float4 v = reinterpret_cast<const float4*>(dy + (b * cout + co) * hw)[at];
    s += ((double)v.x + v.y) + ((double)v.z + v.w);
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if ((int)threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[co * kBgChunks + chunk] = red[0];
}

// w'[ci][co][ky][kx] = w[co][ci][4 - ky][4 - kx]: the backward pass over the data is the forward convolution of dy
// with the flipped, transposed kernel.
__global__ void flip_transpose_kernel(const uint16_t* __restrict__ wt, int cin, int cout, uint16_t* __restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= cin * cout * 25) return;
  const int k = i % 25, r = i / 25, co = r % cout, ci = r / cout;
  out[i] = wt[((size_t)co * cin + ci) * 25 + (24 - k)];
}

// dw[co][ci][ky][kx] = sum_{b, p} dy[b][co][p] x[b][ci][p + (ky - 2, kx - 2)]: one block per (co, ci), a fixed-order
// reduction (each thread's strided partials, then a tree over the block); db[co] the same over dy alone.
__global__ void __launch_bounds__(256) conv5_backward_weights_kernel(const float* __restrict__ x,
                                                                     const float* __restrict__ dy, int batch, int cin,
                                                                     int cout, int h, int w, float* __restrict__ dw,
                                                                     float* __restrict__ db) {
  __shared__ float red[256];
  const int co = blockIdx.x / cin, ci = blockIdx.x % cin;
  float acc[25];
#pragma unroll
  for (int k = 0; k < 25; ++k) acc[k] = 0.f;
  float accb = 0.f;
  const long long hw = (long long)h * w;
  for (long long idx = threadIdx.x; idx < batch * hw; idx += 256) {
    const long long b = idx / hw, p = idx % hw;
    const int py = int(p / w), px = int(p % w);
    const float g = dy[(b * cout + co) * hw + p];
    accb += g;
    const float* xs = x + (b * cin + ci) * hw;
#pragma unroll
    for (int ky = 0; ky < 5; ++ky) {
      const float* row = xs + (long long)wrap(py + ky - 2, h) * w;
#pragma unroll
      for (int kx = 0; kx < 5; ++kx) acc[ky * 5 + kx] += g * row[wrap(px + kx - 2, w)];
    }
  }
  for (int k = 0; k <= 25; ++k) {
    red[threadIdx.x] = k < 25 ? acc[k] : accb;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
      if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
      __syncthreads();
    }
    if (threadIdx.x == 0) {
      if (k < 25) dw[(size_t)blockIdx.x * 25 + k] = red[0];
      else if (ci == 0 && db) db[co] = red[0];
    }
    __syncthreads();
  }
}

// dy *= (y > 0): the ReLU's backward pass, y the layer's output after the ReLU
__global__ void relu_mask_kernel(float* dy, const float* y, long long n) {
  const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i < n && !(y[i] > 0.f)) dy[i] = 0.f;
}

// y[b][q][p] = sum_k x[b][p][k] A[q][k], p < rows, q < m, k < n: one half of the separable map, its result transposed so
// that the same kernel is the other half. A block takes 16 x 16 outputs and stages 64 k of their rows in LDS (rows 68
// floats apart: 16 lanes' 16-byte reads on distinct banks); every sum runs over k in order. Bound by its launches:
// 128 x 128 to 96 x 96, both halves, 48.0 -> 7.6 us for 1 image and 79.8 -> 10.6 us for 16, against each thread
// reading its rows from global memory.
constexpr int kSepK = 64, kSepTile = 16;
__global__ void __launch_bounds__(256) sep_half_kernel(const float* __restrict__ x, const float* __restrict__ A,
                                                       int rows, int n, int m, float* __restrict__ y) {
  __shared__ __align__(16) float xs[kSepTile][kSepK + 4], as[kSepTile][kSepK + 4];
  const int tid = threadIdx.x, pi = tid % kSepTile, qi = tid / kSepTile;
  const int p0 = blockIdx.x * kSepTile, q0 = blockIdx.y * kSepTile;
  const float* xb = x + (size_t)blockIdx.z * rows * n;
  const int lr = tid / (kSepK / 4), lk = 4 * (tid % (kSepK / 4));  // the staged row and the first of 4 k
  float s = 0.f;
  for (int k0 = 0; k0 < n; k0 += kSepK) {
    float u[4], v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int k = k0 + lk + j;
      u[j] = k < n && p0 + lr < rows ? xb[(size_t)(p0 + lr) * n + k] : 0.f;
      v[j] = k < n && q0 + lr < m ? A[(size_t)(q0 + lr) * n + k] : 0.f;
    }
    __syncthreads();  // the previous chunk's reads are done
    *reinterpret_cast<float4*>(&xs[lr][lk]) = make_float4(u[0], u[1], u[2], u[3]);
    *reinterpret_cast<float4*>(&as[lr][lk]) = make_float4(v[0], v[1], v[2], v[3]);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kSepK; k += 4) {
      const float4 a = *reinterpret_cast<const float4*>(&as[qi][k]), b = *reinterpret_cast<const float4*>(&xs[pi][k]);
      s = fmaf(a.x, b.x, s);
      s = fmaf(a.y, b.y, s);
      s = fmaf(a.z, b.z, s);
      s = fmaf(a.w, b.w, s);
    }
  }
  if (p0 + pi < rows && q0 + qi < m) y[((size_t)blockIdx.z * m + q0 + qi) * rows + p0 + pi] = s;
}

// g = 2 (pred - label) / count; loss partials per block (fixed-order sums)
// g = 2 w (pred - label) / n and the block's sum of w (pred - label)^2, w = weights[i / per] (1 when weights is null)
__global__ void mse_grad_kernel(const float* pred, const float* label, long long n, const float* weights,
                                long long per, float* g, double* partial) {
  __shared__ double red[256];
  const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  double e = 0;
  if (i < n) {
    const float d = pred[i] - label[i];
    const float wt = weights ? weights[i / per] : 1.f;
    g[i] = 2.f * wt * d / float(n);
    e = (double)wt * d * d;
  }
  red[threadIdx.x] = e;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

__global__ void adam_kernel(float* p, const float* g, float* m, float* v, uint16_t* p_bf16, long long n, float lr,
                            float b1, float b2, float eps, float c1, float c2) {
  const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi, vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float pi = p[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  p[i] = pi;
  if (p_bf16) p_bf16[i] = f32_to_bf16(pi);
}

__global__ void to_bf16_kernel(const float* in, uint16_t* out, long long n) {
  const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i < n) out[i] = f32_to_bf16(in[i]);
}

unsigned blocks_for(long long n) { return (unsigned)((n + 255) / 256); }

hipStream_t pick(void* stream) { return stream ? static_cast<hipStream_t>(stream) : nullptr; }

void check_conv(int batch, int cin, int cout, int h, int w) {
  if (sk_hip_available() != 1) fail(SK_ERR_UNAVAILABLE, std::string("conv5: ") + sk_hip_last_error());
  if (batch < 1 || cin < 1 || cout < 1) fail(SK_ERR_INVALID, "conv5: empty shape");
  if (h % kTile || w % kTile || h < kTile || w < kTile) fail(SK_ERR_INVALID, "conv5: h and w must be multiples of 16");
  if (batch > 65535) fail(SK_ERR_INVALID, "conv5: batch above 65535");
}

template <int R, int W>
void go_conv5_mfma(const float* x, int batch, int cin, int h, int w, const uint16_t* wtm, const float* bias, int cout,
                   int relu, const float* mask, float* y, hipStream_t s) {
  const dim3 grid((h / (R * W)) * (w / kMfCols), batch);
  const __bf16* wm = reinterpret_cast<const __bf16*>(wtm);
  if (cin <= 16)
    hipLaunchKernelGGL((conv5_forward_mfma_kernel<16, R, W>), grid, dim3(64 * W), 0, s, x, wm, bias, cin, cout, h, w,
                       relu, mask, y);
  else
    hipLaunchKernelGGL((conv5_forward_mfma_kernel<32, R, W>), grid, dim3(64 * W), 0, s, x, wm, bias, cin, cout, h, w,
                       relu, mask, y);
}

void launch_conv5_mfma(const float* x, int batch, int cin, int h, int w, const uint16_t* wtm, const float* bias,
                       int cout, int relu, const float* mask, float* y, hipStream_t s) {
  // Four-row blocks while the chip holds them at one a CU (2 images of 128 x 128: 10.8 us against 13.4 for 32 to 32
  // channels; 1 image: 9.7 against 12.7), above that eight rows, which read less halo and share each row's LDS reads
  // between two output rows (4 images: 17.1 us against 19.4; 16: 51.6 against 59.0).
  if ((long long)batch * (h / 4) * (w / kMfCols) <= 256)
    go_conv5_mfma<1, 4>(x, batch, cin, h, w, wtm, bias, cout, relu, mask, y, s);
  else
    go_conv5_mfma<2, 4>(x, batch, cin, h, w, wtm, bias, cout, relu, mask, y, s);
}

}  // namespace
}  // namespace sk

extern "C" {

int sk_conv5_forward(const float* x, int batch, int cin, int h, int w, const uint16_t* wt, const float* bias, int cout,
                     int relu, float* y, void* stream) {
  using namespace sk;
  return guarded_call([&] {
    if (!x || !wt || !y) fail(SK_ERR_INVALID, "conv5_forward: null pointer");
    check_conv(batch, cin, cout, h, w);
    dim3 grid((h / kTile) * (w / kTile), (cout + kCo - 1) / kCo, batch);
    hipLaunchKernelGGL(conv5_forward_kernel, grid, dim3(256), 0, pick(stream), x, wt, bias, cin, cout, h, w, relu, y);
    SK_HIP(hipGetLastError());
  });
}

int sk_conv5_weights_tap_major(const uint16_t* wt, int cin, int cout, int flip, uint16_t* out, void* stream) {
  using namespace sk;
  return guarded_call([&] {
    if (!wt || !out || cin < 1 || cout < 1 || cin > 32 || cout > 32)
      fail(SK_ERR_INVALID, "conv5_weights_tap_major: null pointer, or channels outside 1 .. 32");
    if (sk_hip_available() != 1) fail(SK_ERR_UNAVAILABLE, sk_hip_last_error());
    const int kp = (flip ? cout : cin) <= 16 ? 16 : 32;
    hipLaunchKernelGGL(weights_tap_major_kernel, dim3(blocks_for(25LL * 32 * kp)), dim3(256), 0, pick(stream), wt, cin,
                       cout, flip ? 1 : 0, kp, out);
    SK_HIP(hipGetLastError());
  });
}

int sk_conv5_forward_tap_major(const float* x, int batch, int cin, int h, int w, const uint16_t* wtm,
                               const float* bias, int cout, int relu, float* y, void* stream) {
  using namespace sk;
  return guarded_call([&] {
    if (!x || !wtm || !y) fail(SK_ERR_INVALID, "conv5_forward_tap_major: null pointer");
    check_conv(batch, cin, cout, h, w);
    if (cin > 32 || cout > 32 || w % kMfCols || h % 8)
      fail(SK_ERR_INVALID, "conv5_forward_tap_major: at most 32 input and 32 output channels, w a multiple of 32 "
                           "and h of 8");
    launch_conv5_mfma(x, batch, cin, h, w, wtm, bias, cout, relu, nullptr, y, pick(stream));
    SK_HIP(hipGetLastError());
  });
}

int sk_conv5_backward_data_tap_major(const float* dy, int batch, int cin, int h, int w, const uint16_t* wtm, int cout,
                                     const float* act, float* dx, void* stream) {
  using namespace sk;
  return guarded_call([&] {
    if (!dy || !wtm || !dx) fail(SK_ERR_INVALID, "conv5_backward_data_tap_major: null pointer");
    check_conv(batch, cin, cout, h, w);
    if (cin > 32 || cout > 32 || w % kMfCols)
      fail(SK_ERR_INVALID, "conv5_backward_data_tap_major: at most 32 input and 32 output channels, w a multiple of 32");
    launch_conv5_mfma(dy, batch, cout, h, w, wtm, nullptr, cin, 0, act, dx, pick(stream));
    SK_HIP(hipGetLastError());
  });
}

int sk_conv5_backward_weights_mfma(const float* x, const float* dy, int batch, int cin, int h, int w, int cout,
                                   float* dw, float* db, float* workspace, void* stream) {
  using namespace sk;
  return guarded_call([&] {
    if (!x || !dy || !dw || !workspace) fail(SK_ERR_INVALID, "conv5_backward_weights_mfma: null pointer");
    check_conv(batch, cin, cout, h, w);
    if (cin > 32 || cout > 32 || w % kWgCols || h % kWgRows)
      fail(SK_ERR_INVALID, "conv5_backward_weights_mfma: at most 32 input and 32 output channels, w a multiple of 32");
    hipStream_t s = pick(stream);
    const long long strips = (long long)batch * (h / kWgRows) * (w / kWgCols);
    const int blocks = (int)(strips < kWgBlocks ? strips : kWgBlocks);
    hipLaunchKernelGGL(conv5_wgrad_mfma_kernel, dim3(blocks), dim3(64 * kWgWaves), 0, s, x, dy, cin, cout, h, w,
                       strips, workspace);
    double* bias = reinterpret_cast<double*>(workspace + (size_t)kWgBlocks * kWgOut);
    if (db)
      hipLaunchKernelGGL(bias_partial_kernel, dim3(cout, kBgChunks), dim3(256), 0, s, dy, batch, cout,
                         (long long)h * w, bias);
    hipLaunchKernelGGL(wgrad_reduce_kernel, dim3(kWgOut / 64 + (db ? 1 : 0)), dim3(256), 0, s, workspace, blocks, cin,
                       cout, dw, bias, db);
    SK_HIP(hipGetLastError());
  });
}

int sk_conv5_backward_data(const float* dy, int batch, int cin, int h, int w, const uint16_t* wt, int cout, float* dx,
                           uint16_t* wt_scratch, void* stream) {
  using namespace sk;
  return guarded_call([&] {
    if (!dy || !wt || !dx || !wt_scratch) fail(SK_ERR_INVALID, "conv5_backward_data: null pointer");
    check_conv(batch, cin, cout, h, w);
    hipStream_t s = pick(stream);
    hipLaunchKernelGGL(flip_transpose_kernel, dim3(blocks_for((long long)cin * cout * 25)), dim3(256), 0, s, wt, cin,
                       cout, wt_scratch);
    dim3 grid((h / kTile) * (w / kTile), (cin + kCo - 1) / kCo, batch);
    hipLaunchKernelGGL(conv5_forward_kernel, grid, dim3(256), 0, s, dy, wt_scratch, nullptr, cout, cin, h, w, 0, dx);
    SK_HIP(hipGetLastError());
  });
}

int sk_conv5_backward_weights(const float* x, const float* dy, int batch, int cin, int h, int w, int cout, float* dw,
                              float* db, void* stream) {
  using namespace sk;
  return guarded_call([&] {
    if (!x || !dy || !dw) fail(SK_ERR_INVALID, "conv5_backward_weights: null pointer");
    check_conv(batch, cin, cout, h, w);
    hipLaunchKernelGGL(conv5_backward_weights_kernel, dim3(cin * cout), dim3(256), 0, pick(stream), x, dy, batch, cin,
                       cout, h, w, dw, db);
    SK_HIP(hipGetLastError());
  });
}

int sk_relu_backward(float* dy, const float* y, long long n, void* stream) {
  using namespace sk;
  return guarded_call([&] {
    if (!dy || !y || n < 0) fail(SK_ERR_INVALID, "relu_backward: invalid arguments");
    if (sk_hip_available() != 1) fail(SK_ERR_UNAVAILABLE, sk_hip_last_error());
    if (n == 0) return;
    hipLaunchKernelGGL(relu_mask_kernel, dim3(blocks_for(n)), dim3(256), 0, pick(stream), dy, y, n);
    SK_HIP(hipGetLastError());
  });
}

int sk_separable_map(const float* in, int batch, int n, const float* A, int m, float* tmp, float* out, void* stream) {
  using namespace sk;
  return guarded_call([&] {
    if (!in || !A || !tmp || !out || batch < 1 || n < 1 || m < 1) fail(SK_ERR_INVALID, "separable_map: invalid");
    if (sk_hip_available() != 1) fail(SK_ERR_UNAVAILABLE, sk_hip_last_error());
    hipStream_t s = pick(stream);
    // tmp[b][v][i] = sum_j in[b][i][j] A[v][j], then out[b][u][v] = sum_i tmp[b][v][i] A[u][i]
    const unsigned tn = (n + kSepTile - 1) / kSepTile, tm = (m + kSepTile - 1) / kSepTile;
    for (long long b0 = 0; b0 < batch; b0 += 65535) {  // the grid's limit of images
      const unsigned nb = unsigned(batch - b0 < 65535 ? batch - b0 : 65535);
      hipLaunchKernelGGL(sep_half_kernel, dim3(tn, tm, nb), dim3(256), 0, s, in + (size_t)b0 * n * n, A, n, n, m,
                         tmp + (size_t)b0 * n * m);
      hipLaunchKernelGGL(sep_half_kernel, dim3(tm, tm, nb), dim3(256), 0, s, tmp + (size_t)b0 * n * m, A, m, n, m,
                         out + (size_t)b0 * m * m);
    }
    SK_HIP(hipGetLastError());
  });
}

int sk_mse_grad(const float* pred, const float* label, long long n, float* grad, double* partials, void* stream) {
  using namespace sk;
  return guarded_call([&] {
    if (!pred || !label || !grad || !partials || n < 1) fail(SK_ERR_INVALID, "mse_grad: invalid");
    if (sk_hip_available() != 1) fail(SK_ERR_UNAVAILABLE, sk_hip_last_error());
    hipLaunchKernelGGL(mse_grad_kernel, dim3(blocks_for(n)), dim3(256), 0, pick(stream), pred, label, n,
                       (const float*)nullptr, 1LL, grad, partials);
    SK_HIP(hipGetLastError());
  });
}

int sk_weighted_mse_grad(const float* pred, const float* label, const float* weights, long long per, long long n,
                         float* grad, double* partials, void* stream) {
  using namespace sk;
  return guarded_call([&] {
    if (!pred || !label || !weights || !grad || !partials || n < 1 || per < 1 || n % per)
      fail(SK_ERR_INVALID, "weighted_mse_grad: invalid");
    if (sk_hip_available() != 1) fail(SK_ERR_UNAVAILABLE, sk_hip_last_error());
    hipLaunchKernelGGL(mse_grad_kernel, dim3(blocks_for(n)), dim3(256), 0, pick(stream), pred, label, n, weights,
                       per, grad, partials);
    SK_HIP(hipGetLastError());
  });
}

int sk_adam_step(float* p, const float* g, float* m, float* v, uint16_t* p_bf16, long long n, float lr, float b1,
                 float b2, float eps, int step, void* stream) {
  using namespace sk;
  return guarded_call([&] {
    if (!p || !g || !m || !v || n < 1 || step < 1) fail(SK_ERR_INVALID, "adam_step: invalid");
    if (sk_hip_available() != 1) fail(SK_ERR_UNAVAILABLE, sk_hip_last_error());
    const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
    hipLaunchKernelGGL(adam_kernel, dim3(blocks_for(n)), dim3(256), 0, pick(stream), p, g, m, v, p_bf16, n, lr, b1,
                       b2, eps, c1, c2);
    SK_HIP(hipGetLastError());
  });
}

int sk_to_bf16(const float* in, uint16_t* out, long long n, void* stream) {
  using namespace sk;
  return guarded_call([&] {
    if (!in || !out || n < 1) fail(SK_ERR_INVALID, "to_bf16: invalid");
    if (sk_hip_available() != 1) fail(SK_ERR_UNAVAILABLE, sk_hip_last_error());
    hipLaunchKernelGGL(to_bf16_kernel, dim3(blocks_for(n)), dim3(256), 0, pick(stream), in, out, n);
    SK_HIP(hipGetLastError());
  });
}

}  // extern "C"
