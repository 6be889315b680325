// FDK kernels for gfx950: fused cosine weight + ramp filter + transpose,
// voxel-driven backprojection, and their exact transposes (the matched
// projector and the transposed filter) for the adjoint.
//
// Reference: recon/bp3d20_325.cpp:39-175 (weight :39-46, filter :51-81,
// backprojection :91-175).  The reference runs these as scalar FP64 loops; here
// each is one kernel:
//   filter:  a pair of detector rows is one complex transform, held by 8 to 32
//            lanes; the weighted [u][v] tile is transposed through LDS.
//   backprojection: one thread per voxel column (x,y), or per orbit of columns
//            that a part of a turn maps onto each other, and ZC voxels along z.
//            Along a column u, the distance weight and the v-slope are constant,
//            so per voxel-update only v moves (one integer add) before the four
//            bilinear taps are read from the view's patch in LDS.  Tiles are
//            ordered so each XCD owns a contiguous z-slab (its L2 then holds
//            only the detector rows that slab projects to).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "internal.h"

namespace monte {

// ------------------------------------------------------------------- fill
// 16-byte stores of the aligned part, one a thread: 67 MB in 10.6 us and 2.3 GB in 0.32 ms
// (7.1 TB/s), 18.6 us and 0.38 ms in stores of 4 bytes by 65536 blocks, and 0.46 ms in stores
// of 16 by 8192.
__global__ __launch_bounds__(256) void fill_kernel(float* __restrict__ p, float v, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (size_t)gridDim.x * blockDim.x;
  const size_t head = min(n, ((16 - ((uintptr_t)p & 15)) & 15) / 4), quads = (n - head) / 4;
  float4* q = (float4*)(p + head);
  for (size_t k = i; k < quads; k += stride) q[k] = make_float4(v, v, v, v);
  if (i < head) p[i] = v;
  if (i < n - head - 4 * quads) p[head + 4 * quads + i] = v;
}

hipError_t launch_fill(float* p, float v, size_t n, hipStream_t s) {
  if (n == 0) return hipSuccess;
  const size_t blocks = std::min<size_t>((n + 1023) / 1024, max_blocks(256));  // (the rest by looping)
  hipLaunchKernelGGL(fill_kernel, dim3((unsigned)blocks), dim3(256), 0, s, p, v, n);
  return hipGetLastError();
}

// Maps a hardware block index to a logical tile so that the blocks the
// dispatcher sends to XCD x (blocks x, x+8, x+16, ...) cover one contiguous
// range of logical tiles.  Tiles are numbered z-chunk slowest.
__device__ inline int xcd_tile(int b, int nblocks) {
  const int q = nblocks >> 3, r = nblocks & 7;
  const int xcd = b & 7, j = b >> 3;
  return xcd * q + (xcd < r ? xcd : r) + j;
}

// ---------------------------------------------------------------- filter
__device__ inline float cos_weight(const FilterParams& fp, int r, int c) {
  const float a = fmaf(fp.b_u, (float)r, fp.a_u);
  const float b = fmaf(fp.b_v, (float)c, fp.a_v);
  return fp.D / sqrtf(fmaf(fp.D, fp.D, fmaf(a, a, b * b)));
}

// The ramp filter of one view is a product with a Toeplitz matrix:
//   out[v][b] = cs sum_c A[v][c] H[c][b],  H[c][b] = h[c - b + nu - 1],
// with A the cosine-weighted projection.  Long rows are filtered so (launch_fdk_filter has
// the rule).  Each block computes a
// 64 (v) x 64 kFnt (b) tile with v_mfma_f32_32x32x2_f32: wave w owns rows
// 32 (w & 1) and the kFnt 32-column tiles at 32 kFnt (w >> 1).  A is staged in LDS
// 32 columns of c at a time as As[c][v]; H is read straight from the taps in
// LDS, shifted by kFbn so every index of the tile stays inside the array.
// Operand layouts (one wave, 32 x 32 x 2): A from lane l is A[l % 32][l / 32],
// B from lane l is B[l / 32][l % 32], and accumulator i of lane l is
// D[8 (i / 4) + 4 (l / 32) + i % 4][l % 32].
constexpr int kFnt = 4;  // 32-column product tiles per wave
constexpr int kFbm = 64, kFbn = 64 * kFnt, kFkc = 32;
constexpr int kFas = kFbm + 1;  // LDS row pitch of As

typedef float floatx16 __attribute__((ext_vector_type(16)));

// Taps into LDS: Ht[i + kFbn] = h[i], zero elsewhere (2 nu + kFkc + 2 kFbn floats).
__device__ inline void stage_taps(float* __restrict__ Ht, const float* __restrict__ taps, int nu) {
  const int n = 2 * nu + kFkc + 2 * kFbn;
  for (int i = threadIdx.x; i < n; i += 256) {
    const int j = i - kFbn;
    Ht[i] = (j >= 0 && j < 2 * nu - 1) ? taps[j] : 0.f;
  }
}

// acc[t] += A[rows][c0 .. c0 + kFkc) x H[c0 .. c0 + kFkc)[cols of tile t]
__device__ inline void mfma_chunk(const float* __restrict__ As, const float* __restrict__ Ht, int c0, int b0, int nu,
                                  floatx16 (&acc)[kFnt]) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int r = (w & 1) * 32 + (lane & 31), kl = lane >> 5;
  const int col = b0 + (w >> 1) * (32 * kFnt) + (lane & 31);
  // H index of (c0 + kk + kl, col + 32 t) is c - b + nu - 1 + kFbn
  const int h0 = c0 + kl - col + nu - 1 + kFbn;
#pragma unroll
  for (int kk = 0; kk < kFkc; kk += 2) {
    const float a = As[(kk + kl) * kFas + r];
    float bv[kFnt];
#pragma unroll
    for (int t = 0; t < kFnt; ++t) bv[t] = Ht[h0 + kk - 32 * t];
#pragma unroll
    for (int t = 0; t < kFnt; ++t) acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, bv[t], acc[t], 0, 0, 0);
  }
}

// proj [view][nu][nv] -> filt_pad [view][rows][pitch] (interior at +kPadLo).
// Thread (tc, tv) stages A[c0 + tc + 4 j][v0 + tv], j < 8; the next chunk's
// loads are issued before the current chunk's products, so their latency
// hides behind the MFMAs.
__global__ __launch_bounds__(256) void filter_fwd_mfma_kernel(const float* __restrict__ proj,
                                                              float* __restrict__ out,
                                                              const float* __restrict__ taps, FilterParams fp) {
  extern __shared__ float sm[];
  float* const A0 = sm;  // double-buffered [kFkc][kFas]
  float* const A1 = sm + kFkc * kFas;
  float* Ht = sm + 2 * kFkc * kFas;
  const int nu = fp.nu, nv = fp.nv;
  const int v0 = blockIdx.x * kFbm, b0 = blockIdx.y * kFbn, view = blockIdx.z;
  stage_taps(Ht, taps, nu);
  const float* src = proj + (size_t)view * nu * nv;
  const int tv = threadIdx.x & 63, tc = threadIdx.x >> 6;
  const int v = v0 + tv, vc = v < nv ? v : nv - 1;
  float pre[kFkc / 4];
  auto load = [&](int c0) {
#pragma unroll
    for (int j = 0; j < kFkc / 4; ++j) {
      const int c = c0 + tc + 4 * j;
      pre[j] = src[(size_t)(c < nu ? c : nu - 1) * nv + vc];
    }
  };
  auto stage = [&](float* A, int c0) {
#pragma unroll
    for (int j = 0; j < kFkc / 4; ++j) {
      const int kc = tc + 4 * j, c = c0 + kc;
      A[kc * kFas + tv] = (c < nu && v < nv) ? pre[j] * cos_weight(fp, c, v) : 0.f;
    }
  };
  load(0);
  stage(A0, 0);
  __syncthreads();
  floatx16 acc[kFnt] = {};
  // chunk k is multiplied from one buffer while chunk k + 1 is loaded and
  // staged into the other; one barrier per chunk
  int buf = 0;
  for (int c0 = 0; c0 < nu; c0 += kFkc) {
    const bool more = c0 + kFkc < nu;
    if (more) load(c0 + kFkc);
    mfma_chunk(buf ? A1 : A0, Ht, c0, b0, nu, acc);
    if (more) stage(buf ? A0 : A1, c0 + kFkc);
    __syncthreads();
    buf ^= 1;
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  float* dst = out + (size_t)view * fp.rows * fp.pitch;
#pragma unroll
  for (int t = 0; t < kFnt; ++t) {
    const int b = b0 + (w >> 1) * (32 * kFnt) + 32 * t + (lane & 31);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int vo = v0 + (w & 1) * 32 + 8 * (i / 4) + 4 * (lane >> 5) + (i & 3);
      if (vo < nv && b < nu) dst[(size_t)(vo + kPadLo) * fp.pitch + b + kPadLo] = fp.cs * acc[t][i];
    }
  }
}

// The ramp filter by FFT.  With N >= 2 nu points a row's circular convolution is the
// linear one.  Rows v and v + 1 are the real and imaginary
// parts of one transform (the taps are real).
//   What is transformed is the row's difference x[n] - x[n - 1], against the taps' running
// sum: a ramp filter takes most of a smooth row's size away, and rounding errors that a
// transform of x itself spreads over all frequencies would stay (rel. errors of smooth
// rows of 512: 7e-6 by x, 2e-6 by the sums of products, 1.3e-7 by differences).  The
// running sum closes the circle with a tap in the unused lag N / 2 that makes the taps' sum
// zero; the spectrum, scaled and with the running sum in it, is made in FP64 (spec).
//   N = R1 M: M lanes hold a pair of rows, lane m the samples m + M n1.  R1 points in
// registers, a twiddle, an exchange through LDS (a wave's own, real and imaginary parts
// in turn), M points in registers, the spectrum, and the same way back.
//   A transform's rounding errors are shared by the two rows of a pair, in proportion to the root of
// both rows' summed squares.  So each row is scaled by the power of two that brings its own sum of
// squares of differences to [1/4, 1), unless both have the same: its errors are then of its own
// size, whatever its neighbour holds: 1.1e-7 to 1.8e-7 rms.  (Scaled only where the largest samples
// differed by 16, a row of 512 beside one 15 times as large had 1.1e-6, and a smooth row beside
// noise, whose differences are far larger, 2.5e-5, for 2.7e-7 and 2e-6 by sums of products.)
// Rows that are not finite are summed directly.
//   Bound by VALU instructions: 1600 of a wave's 2750 (two pairs of 512) are the four
// transforms, 400 twiddles and spectrum, 450 the weighted tile.  360 views of 512^2 take
// 0.287 ms and 0.265 transposed, for 0.94 and 0.87 as products with the taps' Toeplitz matrix
// (103 TFLOP/s of fp32 matrix instructions, of 147 in a large product); 325^2 takes 0.17 ms
// for 0.50, 1024 x 768 transposed 1.4 for 4.6.  Rows that just miss a power of two gain
// least: 180 views of 600 x 512 transposed, with the copy in, 0.52 ms for 0.85.
// y = DFT of x[OFF + STRIDE i], i < LEN, in order.  HALF: of x, only the first half and
// x[R / 2] are not zero.
template <int R, int LEN, int STRIDE, int OFF, bool INV, bool HALF>
__device__ __forceinline__ void fft_regs(const float (&xr)[R], const float (&xi)[R], float (&yr)[LEN],
                                         float (&yi)[LEN]) {
  if constexpr (LEN == 2) {
    const float ar = xr[OFF], ai = xi[OFF];
    if constexpr (HALF && OFF != 0) {
      yr[0] = yr[1] = ar;
      yi[0] = yi[1] = ai;
    } else {
      const float br = xr[OFF + STRIDE], bi = xi[OFF + STRIDE];
      yr[0] = ar + br;
      yi[0] = ai + bi;
      yr[1] = ar - br;
      yi[1] = ai - bi;
    }
  } else {
    constexpr int H = LEN / 2;
    float er[H], ei[H], dr[H], di[H];
    fft_regs<R, H, 2 * STRIDE, OFF, INV, HALF>(xr, xi, er, ei);
    fft_regs<R, H, 2 * STRIDE, OFF + STRIDE, INV, HALF>(xr, xi, dr, di);
#pragma unroll
    for (int k = 0; k < H; ++k) {
      if (k == 0) {
        yr[0] = er[0] + dr[0];
        yi[0] = ei[0] + di[0];
        yr[H] = er[0] - dr[0];
        yi[H] = ei[0] - di[0];
      } else if (4 * k == LEN) {  // times -i, or i
        const float tr = INV ? -di[k] : di[k], ti = INV ? dr[k] : -dr[k];
        yr[k] = er[k] + tr;
        yi[k] = ei[k] + ti;
        yr[k + H] = er[k] - tr;
        yi[k + H] = ei[k] - ti;
      } else {
        const float c = cos64(k * (64 / LEN)), sn = INV ? cos64(k * (64 / LEN) - 16) : -cos64(k * (64 / LEN) - 16);
        yr[k] = fmaf(c, dr[k], fmaf(-sn, di[k], er[k]));
        yi[k] = fmaf(c, di[k], fmaf(sn, dr[k], ei[k]));
        yr[k + H] = fmaf(2.0f, er[k], -yr[k]);
        yi[k + H] = fmaf(2.0f, ei[k], -yi[k]);
      }
    }
  }
}

__device__ inline void wave_lds_sync() {  // between a wave's own writes and reads of LDS
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// LDS words of a pair of rows: R1 rows of M + 1, padded so that the pairs of a wave
// take different banks in the exchanges and in the staging of tiles.
constexpr int fft_stride(int r1, int m) {
  const int base = r1 * (m + 1);
  return base + (((m % 32 + 2 - base) % 32 + 32) % 32);
}

// The cosine weight D / sqrt(s) to about an ulp: an estimate and a Newton step (the
// divisions and roots above are four fifths of a transform's instructions).
__device__ inline float cos_weight_of(float D, float s) {
  const float y = __builtin_amdgcn_rsqf(s);
  const float dy = D * y;
  return fmaf(0.5f * dy, fmaf(-s * y, y, 1.0f), dy);
}

// TRANS false: proj [view][nu][nv], weighted, -> out [view][rows][pitch] with its guard
// cells (wrap: of the bp3d20 preset, see fill_pads_kernel); true: the transpose (guard cells
// not read).  A block takes 128 / M rows per wave.
template <int R1, int M, bool TRANS>
__global__ __launch_bounds__(R1 == 64 ? 512 : 256, R1 == 64 ? 2 : (R1 == 32 ? 3 : 4)) void filter_fft_kernel(
    const float* __restrict__ in, float* __restrict__ out, const float* __restrict__ taps,
    const float2* __restrict__ twid, const float2* __restrict__ spec, FilterParams fp, int tiles, int wrap) {
  constexpr int N = R1 * M, P = 64 / M, S = R1 / M, kHalf = N / 2, kStride = fft_stride(R1, M);
  // tables in LDS (from L1, a block's twiddles and spectrum took as long as its transforms:
  // 0.45 ms where it is 0.29), without the spectrum where 8 waves would not fit (transposed rows
  // of more than 512)
  constexpr bool kSpLds = N <= 1024;
  // the transpose's blocks take tiles in turn, loading the next one's samples while they write: 0.40 -> 0.27 ms
  // for the transpose at 360 x 512^2; forward, 0.29 -> 0.44 (more waits at barriers)
  constexpr bool kAhead = TRANS && R1 <= 32;
  extern __shared__ float sm[];
  const int waves = blockDim.x >> 6, rows_b = 2 * P * waves, rshift = 31 - __builtin_clz(rows_b);
  float2* const twl = (float2*)sm;
  float2* const spl = twl + N;
  float* const bufs = sm + (kSpLds ? 4 : 2) * N;
  const float2* const sp = kSpLds ? spl : spec;
  const int nu = fp.nu, nv = fp.nv;
  const int lane0 = threadIdx.x & 63, wave0 = threadIdx.x >> 6;
  auto tables = [&] {
    for (int i = threadIdx.x; i < N; i += blockDim.x) {
      twl[i] = twid[i];
      if (kSpLds) spl[i] = spec[i];
    }
  };
  if (TRANS) {
    tables();
    __syncthreads();
  }
  // XCD x takes an eighth of the tiles, as xcd_tile deals them: a view's lines meet in one L2
  const int xcd = blockIdx.x & 7, q8 = (tiles * fp.n_views) >> 3, r8 = (tiles * fp.n_views) & 7;
  const int tile0 = xcd * q8 + min(xcd, r8), tile_end = tile0 + q8 + (xcd < r8 ? 1 : 0);
  const int step = (gridDim.x + 7 - xcd) >> 3;
  int tile = tile0 + (blockIdx.x >> 3);
  if (tile >= tile_end) return;
  // a tile's samples: of [nu][nv], thread t has sample t mod rows_b of the lines t / rows_b +
  // j M / 2; of [v][u], a lane has its two rows
  float nx[R1];
  auto load = [&](int tl, int lane, int wave) {
    const int view = tl / tiles, v0 = (tl - view * tiles) * rows_b;
    if (TRANS) {
      const int m = lane & (M - 1), v = v0 + 2 * (wave * P + lane / M);
      const float* pad = in + (size_t)view * fp.rows * fp.pitch + kPadLo;
      const float* row = pad + (size_t)(min(v, nv - 1) + kPadLo) * fp.pitch;
      const float* row2 = pad + (size_t)(min(v + 1, nv - 1) + kPadLo) * fp.pitch;
#pragma unroll
      for (int j = 0; j < R1 / 2; ++j) {
        const int uc = min(m + M * j, nu - 1);
        nx[2 * j] = row[uc];
        nx[2 * j + 1] = row2[uc];
      }
    } else {
      const int t = wave * 64 + lane, tu = t >> rshift;
      const float* src = in + (size_t)view * nu * nv + min(v0 + (t & (rows_b - 1)), nv - 1);
#pragma unroll
      for (int j = 0; j < R1; ++j) nx[j] = src[(size_t)min(tu + j * (M / 2), nu - 1) * nv];
    }
  };
  if (kAhead) load(tile, lane0, wave0);
  for (;;) {
    int lane = lane0, wave = wave0;
    if (TRANS) {  // opaque, or the loop's addresses and weights are kept in registers, and spilt
      asm volatile("" : "+v"(lane));
      asm volatile("" : "+v"(wave));
    }
    const int m = lane & (M - 1), pair = wave * P + lane / M;
    float* const buf = bufs + pair * kStride;
    float* const buf2 = buf + kHalf + 1;  // the second row when staging
    const int view = tile / tiles, v0 = (tile - view * tiles) * rows_b, v = v0 + 2 * pair;
    const float* proj = in + (size_t)view * nu * nv;                     // !TRANS
    const float* pad = in + (size_t)view * fp.rows * fp.pitch + kPadLo;  // TRANS
    const int t = wave * 64 + lane, tr = t & (rows_b - 1), tu = t >> rshift;
    float* const tbuf = bufs + (tr >> 1) * kStride + (tr & 1) * (kHalf + 1) + tu;
    const bool tin = v0 + tr < nv;
    const float bv = fmaf(fp.b_v, (float)(v0 + tr), fp.a_v), bb = fmaf(fp.D, fp.D, bv * bv);
    if (!kAhead) load(tile, lane, wave);
    if (!TRANS) {
#pragma unroll
      for (int j = 0; j < R1; ++j) {
        const int u = tu + j * (M / 2);
        const float au = fmaf(fp.b_u, (float)u, fp.a_u);
        const float w = cos_weight_of(fp.D, fmaf(au, au, bb));
        tbuf[j * (M / 2)] = u < nu && tin ? nx[j] * w : 0.f;
      }
    } else {
#pragma unroll
      for (int j = 0; j < R1 / 2; ++j) {
        const int u = m + M * j;
        buf[u] = u < nu && v < nv ? nx[2 * j] : 0.f;
        buf2[u] = u < nu && v + 1 < nv ? nx[2 * j + 1] : 0.f;
      }
      wave_lds_sync();
    }
    if (!TRANS) {
      tables();
      __syncthreads();
    }

    float yr[R1], yi[R1];  // at the end, filtered samples m + M n1 in the first half
    if (v < nv) {
      float xr[R1], xi[R1];
      float n1 = 0.f, n2 = 0.f;  // sums of squares of each row's differences
      auto sum_squares = [&] {
        n1 = n2 = 0.f;
#pragma unroll
        for (int j = 0; j <= R1 / 2; ++j) {
          n1 = fmaf(xr[j], xr[j], n1);
          n2 = fmaf(xi[j], xi[j], n2);
        }
#pragma unroll
        for (int d = 1; d < M; d *= 2) {
          n1 += __shfl_xor(n1, d);
          n2 += __shfl_xor(n2, d);
        }
      };
      auto scale = [&](int a1, int a2) {
#pragma unroll
        for (int j = 0; j <= R1 / 2; ++j) {
          xr[j] = ldexpf(xr[j], a1);
          xi[j] = ldexpf(xi[j], a2);
        }
      };
#pragma unroll
      for (int j = 0; j < R1 / 2; ++j) {
        const int u = m + M * j;
        const float a = buf[u], b = buf2[u];
        float a0 = buf[j == 0 ? max(u - 1, 0) : u - 1], b0 = buf2[j == 0 ? max(u - 1, 0) : u - 1];
        if (j == 0 && m == 0) a0 = b0 = 0.f;
        xr[j] = a - a0;
        xi[j] = b - b0;
        xr[R1 / 2 + j] = xi[R1 / 2 + j] = 0.f;
      }
      if (m == 0) {
        xr[R1 / 2] = -buf[kHalf - 1];
        xi[R1 / 2] = -buf2[kHalf - 1];
      }
      sum_squares();
      int e1 = 0, e2 = 0;  // the rows' scales
      const bool plain = fminf(n1, n2) > 1e-25f && fmaxf(n1, n2) < 1e35f;
      if (!plain) {  // by their largest differences first, so that no square leaves the range (or a row is zero)
        float big1 = 0.f, big2 = 0.f;  // (a NaN is left out)
#pragma unroll
        for (int j = 0; j <= R1 / 2; ++j) {
          big1 = fmaxf(big1, fabsf(xr[j]));
          big2 = fmaxf(big2, fabsf(xi[j]));
        }
#pragma unroll
        for (int d = 1; d < M; d *= 2) {
          big1 = fmaxf(big1, __shfl_xor(big1, d));
          big2 = fmaxf(big2, __shfl_xor(big2, d));
        }
        e1 = __builtin_amdgcn_frexp_expf(big1);
        e2 = __builtin_amdgcn_frexp_expf(big2);
        scale(-e1, -e2);
        sum_squares();
      }
      const bool zero1 = n1 == 0.f, zero2 = n2 == 0.f;
      const int h1 = (__builtin_amdgcn_frexp_expf(n1) + 1) >> 1, h2 = (__builtin_amdgcn_frexp_expf(n2) + 1) >> 1;
      const bool balance = h1 != h2 && !zero1 && !zero2;
      if (balance) {
        scale(-h1, -h2);
        e1 += h1;
        e2 += h2;
      }
      const bool scaled = balance || !plain;
      fft_regs<R1, R1, 1, 0, false, true>(xr, xi, yr, yi);
      // the lane's sums of differences, or NaN or infinity with one of them
      float odd = fmaf(0.f, yr[0], 0.f * yi[0]);
#pragma unroll
      for (int d = 1; d < M; d *= 2) odd += __shfl_xor(odd, d);
      const bool direct = !(odd == 0.f);
      if (direct) {
#pragma unroll
        for (int j = 0; j < R1; ++j) yr[j] = yi[j] = 0.f;
#pragma unroll 1
        for (int c = 0; c < nu; ++c) {
          float a, b;
          if (TRANS) {
            a = pad[(size_t)(v + kPadLo) * fp.pitch + c];
            b = v + 1 < nv ? pad[(size_t)(v + 1 + kPadLo) * fp.pitch + c] : 0.f;
          } else {
            a = proj[(size_t)c * nv + v] * cos_weight(fp, c, v);
            b = v + 1 < nv ? proj[(size_t)c * nv + v + 1] * cos_weight(fp, c, v + 1) : 0.f;
          }
#pragma unroll
          for (int j = 0; j < R1 / 2; ++j) {
            const int u = m + M * j;
            const float h = taps[u < nu ? c - u + nu - 1 : 0];
            yr[j] = fmaf(a, h, yr[j]);
            yi[j] = fmaf(b, h, yi[j]);
          }
        }
#pragma unroll
        for (int j = 0; j < R1 / 2; ++j) {
          yr[j] *= fp.cs;
          yi[j] *= fp.cs;
        }
      } else {
#pragma unroll
        for (int k = 1; k < R1; ++k) {
          const float2 t = twl[k * M + m];
          const float a = yr[k];
          yr[k] = fmaf(a, t.x, -yi[k] * t.y);
          yi[k] = fmaf(a, t.y, yi[k] * t.x);
        }
        wave_lds_sync();
#pragma unroll
        for (int k = 0; k < R1; ++k) buf[k * (M + 1) + m] = yr[k];
        wave_lds_sync();
        float zr[S][M], zi[S][M];
#pragma unroll
        for (int q = 0; q < S; ++q)
#pragma unroll
          for (int j = 0; j < M; ++j) zr[q][j] = buf[(m + M * q) * (M + 1) + j];
        wave_lds_sync();
#pragma unroll
        for (int k = 0; k < R1; ++k) buf[k * (M + 1) + m] = yi[k];
        wave_lds_sync();
#pragma unroll
        for (int q = 0; q < S; ++q)
#pragma unroll
          for (int j = 0; j < M; ++j) zi[q][j] = buf[(m + M * q) * (M + 1) + j];
#pragma unroll
        for (int q = 0; q < S; ++q) {
          float fr[M], fi[M];
          fft_regs<M, M, 1, 0, false, false>(zr[q], zi[q], fr, fi);
#pragma unroll
          for (int k = 0; k < M; ++k) {
            const float2 t = sp[k * R1 + m + M * q];
            const float a = fr[k];
            fr[k] = fmaf(a, t.x, -fi[k] * t.y);
            fi[k] = fmaf(a, t.y, fi[k] * t.x);
          }
          fft_regs<M, M, 1, 0, true, false>(fr, fi, zr[q], zi[q]);
        }
        wave_lds_sync();
#pragma unroll
        for (int q = 0; q < S; ++q)
#pragma unroll
          for (int j = 0; j < M; ++j) buf[(m + M * q) * (M + 1) + j] = zr[q][j];
        wave_lds_sync();
#pragma unroll
        for (int k = 0; k < R1; ++k) xr[k] = buf[k * (M + 1) + m];
        wave_lds_sync();
#pragma unroll
        for (int q = 0; q < S; ++q)
#pragma unroll
          for (int j = 0; j < M; ++j) buf[(m + M * q) * (M + 1) + j] = zi[q][j];
        wave_lds_sync();
#pragma unroll
        for (int k = 0; k < R1; ++k) xi[k] = buf[k * (M + 1) + m];
#pragma unroll
        for (int k = 1; k < R1; ++k) {
          const float2 t = twl[k * M + m];
          const float a = xr[k];
          xr[k] = fmaf(a, t.x, xi[k] * t.y);
          xi[k] = fmaf(-a, t.y, xi[k] * t.x);
        }
        fft_regs<R1, R1, 1, 0, true, false>(xr, xi, yr, yi);
        if (scaled)
#pragma unroll
          for (int j = 0; j < R1 / 2; ++j) {
            yr[j] = ldexpf(yr[j], e1);
            yi[j] = ldexpf(yi[j], e2);
          }
        if (zero1)  // (its partner's rounding errors)
#pragma unroll
          for (int j = 0; j < R1 / 2; ++j) yr[j] = 0.f;
        if (zero2)
#pragma unroll
          for (int j = 0; j < R1 / 2; ++j) yi[j] = 0.f;
      }
    }

    if (TRANS) {
      wave_lds_sync();
      if (v < nv) {
#pragma unroll
        for (int j = 0; j < R1 / 2; ++j) {
          buf[m + M * j] = yr[j];
          buf2[m + M * j] = yi[j];
        }
      }
      if (kAhead && tile + step < tile_end) load(tile + step, lane, wave);
      __syncthreads();
      float* dst = out + (size_t)view * nu * nv + v0 + tr;
#pragma unroll 16
      for (int j = 0; j < R1; ++j) {
        const int u = tu + j * (M / 2);
        const float au = fmaf(fp.b_u, (float)u, fp.a_u);
        if (u < nu && tin) dst[(size_t)u * nv] = tbuf[j * (M / 2)] * cos_weight_of(fp.D, fmaf(au, au, bb));
      }
      if ((tile += step) >= tile_end) return;
      __syncthreads();
      continue;
    }

    float* const dst = out + (size_t)view * fp.rows * fp.pitch + kPadLo * fp.pitch + kPadLo;
    const size_t plane = (size_t)fp.rows * fp.pitch;
    if (v < nv) {
      float* row = dst + (size_t)v * fp.pitch;
#pragma unroll
      for (int j = 0; j < R1 / 2; ++j) {
        const int u = m + M * j;
        if (u < nu) row[u] = yr[j];
      }
      if (v + 1 < nv) {
        row += fp.pitch;
#pragma unroll
        for (int j = 0; j < R1 / 2; ++j) {
          const int u = m + M * j;
          if (u < nu) row[u] = yi[j];
        }
      }
      // guard cells before and after these rows
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int r = v + h;
        if (r >= nv) break;
        if (m < 1 + kPadHi && (!wrap || m == 0 || (r == nv - 1 && view == fp.n_views - 1)))
          dst[(size_t)r * fp.pitch + (m == 0 ? -1 : nu + m - 1)] = 0.f;
        if (!wrap) continue;
        // the guard cells that alias sample (view, r, u), see fold_pads_kernel
        if (m < kPadHi) {
          const float y = h == 0 ? yr[0] : yi[0];
          if (r >= 1) dst[(size_t)(r - 1) * fp.pitch + nu + m] = y;
          if (view >= 1 && r <= kPadHi) (dst - plane)[(size_t)(nv + r - 1) * fp.pitch + nu + m] = y;
        }
        if (view >= 1 && r < kPadHi) {
          float* above = dst - plane + (size_t)(nv + r) * fp.pitch;
#pragma unroll
          for (int j = 0; j < R1 / 2; ++j) {
            const int u = m + M * j;
            if (u < nu) above[u] = h == 0 ? yr[j] : yi[j];
          }
        }
      }
    }
    // guard rows
    if (v0 == 0)
      for (int i = threadIdx.x; i < fp.pitch; i += blockDim.x) dst[i - fp.pitch - kPadLo] = 0.f;
    if (v0 + rows_b >= nv)
      for (int i = threadIdx.x; i < kPadHi * fp.pitch; i += blockDim.x) {
        const int c = i % fp.pitch;
        if (!wrap || c < kPadLo || view == fp.n_views - 1) dst[(size_t)nv * fp.pitch - kPadLo + i] = 0.f;
      }
    return;
  }
}

// Points of the row transforms, and lanes that hold a pair of rows.
int filter_fft_points(int nu) {
  int n = 128;
  while (n < 2 * nu) n *= 2;
  return n;
}
int filter_fft_lanes(int n) { return n >= 1024 ? 32 : (n == 128 ? 8 : 16); }

template <bool TRANS>
static hipError_t launch_filter_fft(const float* in, float* out, const float* taps, const float2* tables,
                                    const FilterParams& fp, int wrap, hipStream_t s) {
  if (fp.nu > 1024) return hipErrorInvalidValue;  // (check_geom)
  const int n = filter_fft_points(fp.nu), m = filter_fft_lanes(n), per_wave = 128 / m;
  int waves = n <= 1024 ? 4 : 8;
  while (waves > 1 && (long)fp.n_views * ((fp.nv + per_wave * waves - 1) / (per_wave * waves)) < 512) waves /= 2;
  const int rows_b = per_wave * waves, tiles = (fp.nv + rows_b - 1) / rows_b;
  if ((long)tiles * fp.n_views > 0x3fffffffL) return hipErrorInvalidValue;
  const size_t lds = sizeof(float) * ((n <= 1024 ? 4 : 2) * n + (size_t)(64 / m) * waves * fft_stride(n / m, m));
  long blocks = (long)tiles * fp.n_views;
  if (!TRANS && blocks > (long)max_blocks(64 * waves)) return hipErrorInvalidValue;
  if (TRANS) blocks = std::min<long>(blocks, 256 * std::min<long>(160 * 1024 / lds, 16 / waves));
#define MONTE_FFT(R, L)                                                                                        \
  hipLaunchKernelGGL((filter_fft_kernel<R, L, TRANS>), dim3((unsigned)blocks), dim3(64 * waves), lds, s, in,   \
                     out, taps, tables, tables + n, fp, tiles, wrap)
  switch (n) {
    case 128: MONTE_FFT(16, 8); break;
    case 256: MONTE_FFT(16, 16); break;
    case 512: MONTE_FFT(32, 16); break;
    case 1024: MONTE_FFT(32, 32); break;
    default:
      if constexpr (TRANS) MONTE_FFT(64, 32);
  }
#undef MONTE_FFT
  return hipGetLastError();
}

// Forward, rows of more than 512 samples stay products, at 5.2 ms for 1.5 (360 x 1024 x
// 768): the filter's gain at a row's lowest frequencies, each of which has one factor in
// FP32, is 1e-8 off by FFT, and sums over a volume, as the FP64 loss of a reconstruction's
// residual, show it.  Products keep such a loss to 1e-9 (512^3 from 1024 x 768; 3e-8 by FFT);
// up to 512 samples the scale's and the taps' rounding is as large.
hipError_t launch_fdk_filter(const float* proj, float* filt_pad, const float* taps, const float2* tables,
                             const FilterParams& fp, int wrap, hipStream_t s) {
  if (fp.nu <= 512 && (!wrap || (fp.nu >= kPadHi && fp.nv > kPadHi)))
    return launch_filter_fft<false>(proj, filt_pad, taps, tables, fp, wrap, s);
  if (fp.nu <= 512) {  // guard cells past the next row or view
    const hipError_t e = launch_filter_fft<false>(proj, filt_pad, taps, tables, fp, 0, s);
    if (e != hipSuccess) return e;
  } else {
    const size_t lds = sizeof(float) * (2 * (size_t)kFkc * kFas + 2 * (size_t)fp.nu + kFkc + 2 * kFbn);
    if (lds > 64 * 1024) return hipErrorInvalidValue;
    const dim3 grid((fp.nv + kFbm - 1) / kFbm, (fp.nu + kFbn - 1) / kFbn, fp.n_views);
    hipLaunchKernelGGL(filter_fwd_mfma_kernel, grid, dim3(256), lds, s, proj, filt_pad, taps, fp);
  }
  return launch_fill_pads(filt_pad, fp.n_views, fp.nu, fp.nv, fp.pitch, fp.rows, wrap, s);
}

hipError_t launch_fdk_filter_T(const float* filt_pad, float* proj, const float* taps, const float2* tables,
                               const FilterParams& fp, hipStream_t s) {
  return launch_filter_fft<true>(filt_pad, proj, taps, tables, fp, 0, s);
}

// -------------------------------------------------------------- pad copies
__global__ void pad_copy_kernel(const float* __restrict__ src, float* __restrict__ dst, int n_views, int nu, int nv,
                                int pitch, int rows, int to_padded) {
  const size_t n = (size_t)n_views * rows * pitch;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    const size_t k = i / ((size_t)rows * pitch);
    const int rem = (int)(i - k * rows * pitch);
    const int r = rem / pitch - kPadLo, c = rem % pitch - kPadLo;
    const bool inside = r >= 0 && r < nv && c >= 0 && c < nu;
    const size_t si = (k * nv + (inside ? r : 0)) * nu + (inside ? c : 0);
    if (to_padded)
      dst[i] = inside ? src[si] : 0.f;
    else if (inside)
      dst[si] = src[i];
  }
}

hipError_t launch_pad_copy(const float* filt, float* filt_pad, int n_views, int nu, int nv, int pitch, int rows,
                           hipStream_t s) {
  const size_t n = (size_t)n_views * rows * pitch;
  size_t blocks = (n + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(pad_copy_kernel, dim3((unsigned)blocks), dim3(256), 0, s, filt, filt_pad, n_views, nu, nv,
                     pitch, rows, 1);
  return hipGetLastError();
}

// Guard cells of a padded stack.  Standard preset: zeros (the bilinear
// interpolant's zero extension).  bp3d20 preset (wrap != 0): the value the
// reference reads there.  recon/bp3d20_325.cpp:163-166 index the flat array
// map_out[view*H*W + row*H + col], so a tap at col == H lands on the next
// row's first elements and a tap at row == H on the next view's first row;
// cells past the last view read as zero.  Cells before the interior are never
// sampled in that preset and are zeroed.
__device__ inline bool wrap_source(int k, int r, int c, int n_views, int nu, int nv, int& kk, int& rr, int& cc) {
  if (r < 0 || c < 0) return false;
  const long flat = (long)r * nu + c;
  const long plane = (long)nu * nv;
  kk = k + (int)(flat / plane);
  const long w = flat % plane;
  rr = (int)(w / nu);
  cc = (int)(w % nu);
  return kk < n_views;
}

// One thread per guard cell (the interior is left alone): per view, the guard
// rows above the detector, the guard columns of its nv rows, the guard rows below.
__global__ void fill_pads_kernel(float* __restrict__ buf, int n_views, int nu, int nv, int pitch, int rows,
                                 int wrap) {
  const int top = kPadLo * pitch, side = pitch - nu, mid = nv * side;
  const int per_view = rows * pitch - nu * nv;
  const size_t n = (size_t)n_views * per_view;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    const int k = (int)(i / per_view);
    int j = (int)(i - (size_t)k * per_view);
    int r, c;  // detector coordinates of the guard cell
    if (j < top) {
      r = j / pitch - kPadLo;
      c = j % pitch - kPadLo;
    } else if ((j -= top) < mid) {
      r = j / side;
      const int q = j - r * side;
      c = q < kPadLo ? q - kPadLo : nu + (q - kPadLo);
    } else {
      j -= mid;
      r = nv + j / pitch;
      c = j % pitch - kPadLo;
    }
    float v = 0.f;
    int kk, rr, cc;
    if (wrap && wrap_source(k, r, c, n_views, nu, nv, kk, rr, cc))
      v = buf[((size_t)kk * rows + rr + kPadLo) * pitch + cc + kPadLo];
    buf[((size_t)k * rows + r + kPadLo) * pitch + c + kPadLo] = v;
  }
}

hipError_t launch_fill_pads(float* buf, int n_views, int nu, int nv, int pitch, int rows, int wrap, hipStream_t s) {
  const size_t n = (size_t)n_views * ((size_t)rows * pitch - (size_t)nu * nv);
  size_t blocks = (n + 255) / 256;
  if (blocks > 16384) blocks = 16384;
  hipLaunchKernelGGL(fill_pads_kernel, dim3((unsigned)blocks), dim3(256), 0, s, buf, n_views, nu, nv, pitch, rows,
                     wrap);
  return hipGetLastError();
}

// Transpose of the bp3d20 guard-cell wrap: what the matched projector
// deposited on a guard cell belongs to the interior cell it aliases.  An
// interior cell (k, r, c) is aliased by at most three guard cells (for
// nu >= kPadHi and nv > kPadHi):
//   (k, r - 1, nu + c)        when c < kPadHi and r >= 1,
//   (k - 1, nv + r - 1, nu + c) when c < kPadHi and r <= kPadHi,
//   (k - 1, nv + r, c)        when r < kPadHi,
// the inverse of wrap_source.  Each interior cell gathers them in that fixed
// order, so the sum does not depend on scheduling.
__global__ void fold_pads_kernel(float* __restrict__ buf, int n_views, int nu, int nv, int pitch, int rows) {
  const size_t n = (size_t)n_views * nv * nu;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    const int k = (int)(i / ((size_t)nv * nu));
    const int rem = (int)(i - (size_t)k * nv * nu);
    const int r = rem / nu, c = rem - r * nu;
    if (c >= kPadHi && r > kPadHi) continue;
    auto at = [&](int kk, int rr, int cc) -> float& {
      return buf[((size_t)kk * rows + rr + kPadLo) * pitch + cc + kPadLo];
    };
    float v = at(k, r, c);
    if (c < kPadHi && r >= 1) v += at(k, r - 1, nu + c);
    if (k >= 1 && c < kPadHi && r <= kPadHi) v += at(k - 1, nv + r - 1, nu + c);
    if (k >= 1 && r < kPadHi) v += at(k - 1, nv + r, c);
    at(k, r, c) = v;
  }
}

hipError_t launch_fold_pads(float* buf, int n_views, int nu, int nv, int pitch, int rows, hipStream_t s) {
  if (nu < kPadHi || nv <= kPadHi) return hipErrorInvalidValue;
  const size_t n = (size_t)n_views * nv * nu;
  size_t blocks = (n + 255) / 256;
  if (blocks > 16384) blocks = 16384;
  hipLaunchKernelGGL(fold_pads_kernel, dim3((unsigned)blocks), dim3(256), 0, s, buf, n_views, nu, nv, pitch, rows);
  return hipGetLastError();
}

hipError_t launch_unpad_copy(const float* filt_pad, float* filt, int n_views, int nu, int nv, int pitch, int rows,
                             hipStream_t s) {
  const size_t n = (size_t)n_views * rows * pitch;
  size_t blocks = (n + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(pad_copy_kernel, dim3((unsigned)blocks), dim3(256), 0, s, filt_pad, filt, n_views, nu, nv,
                     pitch, rows, 0);
  return hipGetLastError();
}

// ------------------------------------------------------- backprojection

// 1 / U and wn / dd rounded as the divisions are (for normal numbers, and all but one in 2^40): a
// hardware estimate and Newton steps, a third of the divisions' instructions.
__device__ inline double recip64(double u) {
  double y = __builtin_amdgcn_rcp(u);
  y = fma(y, fma(-u, y, 1.0), y);
  return fma(y, fma(-u, y, 1.0), y);
}

// floor as an integer in one instruction (v_floor + v_cvt otherwise)
__device__ inline int floor_i(float f) {
  int r;
  asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(r) : "v"(f));
  return r;
}

// Per-column quantities of one view, shared by the backprojector and its
// transpose so both evaluate bit-identical weights.
struct ColumnCore {
  int iu;       // u pixel index of the left tap (sample window clamped)
  float fu;     // u fraction
  float w;      // distance weight x angular factor
  bool ok;      // su inside the window
  double kv;    // d(sv)/dZ = svk / U
  float dsv;    // sv increment per voxel step along z
};

// STANDARD: the view's distance weight has no signed term (BpView's g and h are 0).
template <bool STANDARD = false>
__device__ inline ColumnCore column_core(const BpView& c, double X, double Y, float Xf, float Yf, const BpGrid& g) {
  ColumnCore r;
  const double U = fma(c.cx, X, fma(c.cy, Y, c.c0));
  const double inv = recip64(U);
  double su = fma(c.suk * fma(c.ax, X, c.ay * Y), inv, c.su0);
  r.ok = su >= g.lo_u && su <= g.hi_u;
  su = fmin(fmax(su, g.lo_u), g.hi_u);
  const double fu0 = floor(su);
  r.iu = (int)fu0;
  r.fu = (float)(su - fu0);
  r.kv = c.svk * inv;
  r.dsv = (float)(r.kv * g.gsz);
  // sign test in unfused FP64 (as recon/bp3d20_325.cpp:145,151 evaluates it)
  float dd = fmaf(c.dx, Xf, fmaf(c.dy, Yf, c.d0));
  if (!STANDARD) {
    const double gp = xadd(xmul(X, c.gx), xmul(Y, c.gy));
    const float hp = fabsf(fmaf(c.hx, Xf, c.hy * Yf));
    dd -= gp < 0.0 ? -hp : hp;
  }
  float rd = __builtin_amdgcn_rcpf(dd);
  rd = fmaf(rd, fmaf(-dd, rd, 1.0f), rd);
  float q = c.wn * rd;
  q = fmaf(fmaf(-dd, q, c.wn), rd, q);  // (rounded as the division is)
  r.w = c.fac * q * q;
  return r;
}

// The v coordinate of voxel z is formed from a base taken in the middle of its
// 16-aligned group, whatever the thread's z-chunk, so every tuned z-chunk and tile
// shape evaluates the same floating-point expression for each voxel and the
// volume is bitwise independent of them.  (Launches of part of the views add the
// same terms in another order, and take orbits apart.)
constexpr int kZBase = 16;
constexpr int kZMid = kZBase / 2;  // the base voxel of a group of 16: dsv's rounding is multiplied by 8 at most

__device__ inline double base_z(const BpGrid& g, int zb) {
  // recon/bp3d20_325.cpp:109 forms the coordinate as start - index * step, unfused
  return xadd(g.gz0, xmul((double)zb, g.gsz));
}

// The v coordinates of a group's voxels in the column's view: row ivb of the
// base voxel, and in fixed point of kVBits fraction bits, relative to that row,
// the base voxel's coordinate, the step per voxel and the window.  Integers add
// without rounding, so a coordinate is within 2^-(kVBits + 1) rows x 9 of the
// FP64 line; as FP32 multiply-adds of the step they were 2^-21 off (|f| up to 16).
// The tiled kernel takes steps of up to 4.5 rows per voxel, so a group stays
// within +-37 rows of its base.
constexpr int kVBits = 25;
struct GroupV {
  int ivb;
  int f, d;        // base coordinate and step
  int flo, fhi;    // window, clamped to +-63 rows
};

__device__ inline GroupV group_v(const ColumnCore& cc, const BpView& c, double Zb, const BpGrid& g) {
  constexpr double one = (double)(1 << kVBits);
  GroupV b;
  double sv = fma(cc.kv, Zb, c.sv0);
  // (a group whose base lies 40 rows outside the window lies outside as a whole)
  sv = fmin(fmax(sv, g.lo_v - 40.0), g.hi_v + 40.0);
  const double fv0 = floor(sv);
  b.ivb = (int)fv0;
  b.f = (int)rint((sv - fv0) * one);
  b.d = (int)rint(cc.kv * g.gsz * one);
  b.flo = (int)(fmin(fmax(g.lo_v - fv0, -63.0), 63.0) * one);
  b.fhi = (int)(fmin(fmax(g.hi_v - fv0, -63.0), 63.0) * one);
  return b;
}

// Whether voxel z's sample lies in the v window, edges included.  Decided on the
// FP64 line: in the bp3d20 preset samples fall on an edge exactly (rational
// geometry), and the reference's FP64 comparison decides whether they count.
__device__ inline bool in_window(const ColumnCore& cc, const BpView& c, const BpGrid& g, int z) {
  const double sv = fma(cc.kv, base_z(g, z), c.sv0);
  return sv >= g.lo_v && sv <= g.hi_v;
}

__device__ inline bool in_mask(const BpGrid& g, int x, int y, int z) {
  if (!g.mask) return true;
  const int dz = z - g.mcz, dy = y - g.mcy, dx = x - g.mcx;
  return (float)(dz * dz + dy * dy + dx * dx) <= g.mask_r2;
}

// recon/bp3d20_325.cpp:107-108 form X and Y as start + index * step, unfused
__device__ inline double voxel_x(const BpGrid& g, int x) { return xadd(g.gx0, xmul((double)x, g.gsx)); }
__device__ inline double voxel_y(const BpGrid& g, int y) { return xadd(g.gy0, xmul((double)y, g.gsy)); }

// The backprojector reads its bilinear taps from LDS.  A block owns a tile of
// 256 voxel columns over ZC voxels of z; in one view that tile projects to a
// small patch of the detector (25 x 22 cells at 325^3 / 512^2), which the block
// copies into LDS with coalesced loads while it works on the view before.
// What bounds it: taps gathered from global memory cost 16.4 clocks per wave and
// load whatever lies in cache (8- and 16-byte gathers alike, 5.4 for 4 bytes),
// against 3.3 for a pair of words from LDS, so the gathers were the floor of the
// kernel this one replaced (6.83 ms at 325^3 / 512^2 / 360 views, 21.7 clocks
// per wave update, and 0.36 ms to write the four taps of every cell side by side,
// 1.5 GB; 3.8 ms now: the VALU issues 89% of the time and LDS reads take 83%).
//
// NQ > 1: a scan of a full turn in V views, of a volume that 1/NQ of a turn maps
// onto itself, sees voxel column c in view k exactly as it sees c turned by q/NQ
// in view k + q V / NQ: NQ = 4 for square volumes and V a multiple of 4, NQ = 2
// for any volume about the axis and V even.  A thread then owns the NQ columns of
// one orbit: it forms the sample coordinates and weights of its first column once
// per view and applies them to the patches of NQ views, one per column.  VALU
// instructions per update: 10 / NQ of geometry and 5 of taps (NQ = 1: 13 in all,
// by interpolating u, v in turn), and about 70 per column and view.
//
// ZEROS: the guard cells around the views are zeros (standard preset), so a
// sample clamped to the window's edge reads zeros and needs no mask.
//
// LDS cell (r, q, c) of a patch is at r kRS + q kCols + c: a wave's copy
// instruction fills 64 words in a row (straight from memory to LDS), one row of
// one view (of two views for NQ = 4); the row pitch kRS spreads neighbouring rows
// over different banks (16 mod 64), and keeps every tap of the four patches
// within one instruction's offsets of a single address (144 + 3 * 32 + 1 < 256).
template <int NQ>
struct PatchLayout {
  static constexpr int kCols = NQ == 4 ? 32 : 64;
  static constexpr int kRS = NQ == 1 ? 80 : 144;
  static constexpr int kMaxRows = NQ == 4 ? 34 : (NQ == 2 ? 45 : 62);  // two patches in 39 to 52 KB of LDS
};

// One dword per lane from `row` + off (bytes) to 64 consecutive words of LDS, all
// three wave-uniform but off.  Written as an instruction because the compiler
// cannot tell the two patches apart and would wait for the copies of one
// before it reads the other; there is no result register, and the caller waits
// (vmcnt) and meets the other waves before anything reads the words.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"  // (that M0 is a reserved register)
__device__ inline void copy_to_lds(const char* row, uint32_t off, float* dst) {
  const uint32_t at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) float*)dst;
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
               :
               : "s"(__builtin_amdgcn_readfirstlane((int)at)), "v"(off), "s"(row)
               : "memory", "m0");
}
#pragma clang diagnostic pop

// min(max(x, lo), hi) in one instruction
__device__ inline int clamp_i(int x, int lo, int hi) {
  int r;
  asm("v_med3_i32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "v"(lo), "v"(hi));
  return r;
}

constexpr float kFracUnit = 2.3283064365386963e-10f;  // 2^-32
// A voxel's bilinear taps in the patches of its orbit.
template <int NQ>
struct Taps {
  float p[NQ][4];
  float fv;   // row fraction
  bool live;  // inside the v window and the mask
};

constexpr int kRegionViews = 32;  // views whose patch origins are found at a time

template <int ZC, int NQ, bool ZEROS>
__global__ __launch_bounds__(1024) void backproject_kernel(const float* __restrict__ pad,
                                                             const BpView* __restrict__ views, int view0,
                                                             int nviews, BpGrid g, float* __restrict__ vol,
                                                             int accumulate, int tile_x, int tiles_x, int tiles_y,
                                                             int patch_rows, int turn, int stack) {
  using L = PatchLayout<NQ>;
  // per group of 4 waves, two patches of patch_rows rows, one read while the other is filled
  extern __shared__ float patches[];
  __shared__ int2 regions[4][2][kRegionViews];
  const int t = xcd_tile(blockIdx.x, gridDim.x);
  const int per_z = tiles_x * tiles_y;
  const int zc = t / per_z;
  const int rem = t - zc * per_z;
  const int ty_t = rem / tiles_x, tx_t = rem - ty_t * tiles_x;
  const int tile_y = 256 / (tile_x * stack);
  // The block's groups of 256 threads share its views out (one group when there are
  // tiles enough); their sums are added in order at the end.
  const int tid = threadIdx.x & 255, group = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8), groups = blockDim.x >> 8;
  const int first_view = view0 + (int)((long)group * nviews / groups);
  const int my_views = view0 + (int)((long)(group + 1) * nviews / groups) - first_view;
  const int loop_views = (nviews + groups - 1) / groups;
  // columns up to (xb, yb) are owned: all of them, or the first quadrant or half of the orbits
  const int xb = NQ == 4 ? (g.nx + 1) / 2 : g.x1, yb = NQ > 1 ? (g.ny + 1) / 2 : g.ny;
  const int tx0 = (NQ > 1 ? 0 : g.x0) + tx_t * tile_x, ty0 = ty_t * tile_y;
  // a wave takes 8 x 8 columns of the tile: the smallest patch, so its taps share
  // words and fewer rows of them meet in one bank
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wx = tile_x / 8;
  const int wz = stack == 1 ? 0 : wave, wt = stack == 1 ? wave : 0;  // (its place along z and in the tile)
  const int xw = tx0 + wt % wx * 8, yw = ty0 + wt / wx * 8;
  const bool idle = xw >= xb || yw >= yb;  // (a wave past the edge only copies)
  // (past the end: repeats a column, never stored)
  const int x = min(xw + lane % 8, xb - 1), y = min(yw + lane / 8, yb - 1);
  const int zt = zc * ZC * stack, z0 = zt + wz * ZC;  // the tile's first voxel and the wave's
  // its groups of 16 start at zb; its first voxel's place from the middle of its group
  const int zb = ZC % kZBase == 0 ? z0 : (z0 / kZBase) * kZBase, joff = ZC % kZBase == 0 ? -kZMid : z0 - zb - kZMid;
  const int patch_words = patch_rows * L::kRS;
  float* const patch = patches + group * 2 * patch_words;
  int2 (*const region)[kRegionViews] = regions[group];
  const int part = g.n_views / NQ;  // views of 1/NQ of a turn

  // Patch origin (row, column of the padded view) of views [first, first + 32):
  // the sample coordinates are monotonic along any line of the tile, so their
  // minima lie at its corners.  8 lanes per view evaluate the 8 corners.
  auto find_regions = [&](int first) {
    int tid = threadIdx.x & 255;
    asm volatile("" : "+v"(tid));  // (opaque: the corners are formed here, not kept in registers over the views)
    const int k = min(first + (tid >> 3), first_view + my_views - 1);
    const BpView& c = views[k];
    const double Xc = voxel_x(g, (tid & 1) ? min(tx0 + tile_x, xb) - 1 : tx0);
    const double Yc = voxel_y(g, (tid & 2) ? min(ty0 + tile_y, yb) - 1 : ty0);
    const double Zc = base_z(g, (tid & 4) ? zt + ZC * stack - 1 : zt);
    const double inv = recip64(fma(c.cx, Xc, fma(c.cy, Yc, c.c0)));
    const double su = fma(c.suk * fma(c.ax, Xc, c.ay * Yc), inv, c.su0), sv = fma(c.svk * inv, Zc, c.sv0);
    float u = (float)fmin(fmax(su, g.lo_u), g.hi_u), v = (float)fmin(fmax(sv, g.lo_v), g.hi_v);
#pragma unroll
    for (int o = 1; o < 8; o <<= 1) {
      u = fminf(u, __shfl_xor(u, o, 64));
      v = fminf(v, __shfl_xor(v, o, 64));
    }
    // (0.01: the voxels' own coordinates round differently)
    if ((tid & 7) == 0)
      region[((first - first_view) / kRegionViews) & 1][tid >> 3] =
          make_int2(max(floor_i(v - 0.01f) + kPadLo, 0), max(floor_i(u - 0.01f) + kPadLo, 0));
  };

  // Copies view k's patch, or the patches of views k + q V / NQ mod V: wave w
  // takes rows w, w + 4, ...; lane l column l % kCols.  Rows and columns past the
  // padded view repeat its last ones; no tap reads them.
  const uint32_t view_bytes = (uint32_t)g.rows * (uint32_t)g.pitch * 4u;
  auto copy = [&](int k, float* buf) {
    const int2 o = region[((k - first_view) / kRegionViews) & 1][(k - first_view) % kRegionViews];
    const int r0 = __builtin_amdgcn_readfirstlane(o.x), c0 = __builtin_amdgcn_readfirstlane(o.y);
    const uint32_t col = (uint32_t)min(c0 + lane % L::kCols, g.pitch - 1) * 4u;
    const int kq = NQ > 1 ? k % part : k, turned = NQ > 1 ? k / part : 0;
    const char* src = (const char*)pad + (size_t)kq * view_bytes;
#pragma unroll
    for (int h = 0; h < (NQ > 1 ? 2 : 1); ++h) {
      // patch q holds view (k + q part) mod V = k mod part + ((q + turned) mod NQ) part
      const uint32_t q = (uint32_t)(h * (64 / L::kCols) + lane / L::kCols);
      const uint32_t off = col + (NQ > 1 ? ((q + turned) & (NQ - 1u)) * (uint32_t)part * view_bytes : 0u);
      for (int r = wave; r < patch_rows; r += 4) {
        const char* row = src + (uint32_t)min(r0 + r, g.rows - 1) * (uint32_t)g.pitch * 4u;
        copy_to_lds(row, off, buf + r * L::kRS + h * 64);
      }
    }
  };

  float acc[NQ][ZC];
#pragma unroll
  for (int q = 0; q < NQ; ++q)
#pragma unroll
    for (int j = 0; j < ZC; ++j) acc[q][j] = 0.f;

  if (my_views > 0) find_regions(first_view);
  __syncthreads();
  if (my_views > 0) copy(first_view, patch);
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): the copies are in LDS
  __syncthreads();
  for (int i = 0; i < loop_views; ++i) {
    const int k = first_view + i;
    const bool more = i + 1 < my_views;
    if (more) copy(k + 1, patch + ((i + 1) & 1) * patch_words);
    // the next batch of origins, half a batch ahead of its first use
    if (i % kRegionViews == kRegionViews / 2 && i + kRegionViews / 2 < my_views)
      find_regions(k + kRegionViews / 2);
    if (!idle && i < my_views) {
      const BpView& c = views[k];
      int xc = x, yc = y;
      asm volatile("" : "+v"(xc), "+v"(yc));  // (two registers kept over the views instead of four)
      const double X = voxel_x(g, xc), Y = voxel_y(g, yc);
      const ColumnCore cc = column_core<ZEROS>(c, X, Y, (float)X, (float)Y, g);
      const int2 o = region[(i / kRegionViews) & 1][i % kRegionViews];
      const float wu = ZEROS || cc.ok ? cc.w : 0.f;
      const float w1 = wu * cc.fu, w0 = wu - w1;
      // The reads of one voxel are issued before the sums of the voxel before it
      // (left to itself the compiler saves registers and waits for each pair of
      // words: 6.6 against 4.8 ms for the FDK at 325^3 / 512^2 / 360 views).
      GroupV cb;
      int base = 0;
      auto taps_of = [&](int j) {
        if (j % kZBase == 0) {
          cb = group_v(cc, c, base_z(g, zb + j + kZMid), g);
          base = (group * 2 + (i & 1)) * patch_words + (cb.ivb + kPadLo - o.x) * L::kRS + (cc.iu + kPadLo - o.y);
          asm volatile("" : "+v"(base));  // (keeps the constants out of the reads' offsets, which the taps need)
        }
        const int f = cb.f + (joff + j % kZBase) * cb.d;
        const int fc = clamp_i(f, cb.flo, cb.fhi);
        const float* s = patches + (base + __mul24(fc >> kVBits, L::kRS));
        Taps<NQ> t;
        t.fv = kFracUnit * (float)((uint32_t)fc << (32 - kVBits));
        t.live = ZEROS || (in_window(cc, c, g, z0 + j) && in_mask(g, x, y, z0 + j));
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
          const float* sq = s + q * L::kCols;
          t.p[q][0] = sq[0];
          t.p[q][1] = sq[1];
          t.p[q][2] = sq[L::kRS];
          t.p[q][3] = sq[L::kRS + 1];
        }
        return t;
      };
      Taps<NQ> cur = taps_of(0);
#pragma unroll
      for (int j = 0; j < ZC; ++j) {
        const Taps<NQ> t = cur;
        if (j + 1 < ZC) cur = taps_of(j + 1);
        __builtin_amdgcn_sched_barrier(0);
        if (NQ == 1) {
          const float a = fmaf(cc.fu, t.p[0][1] - t.p[0][0], t.p[0][0]);
          const float b = fmaf(cc.fu, t.p[0][3] - t.p[0][2], t.p[0][2]);
          acc[0][j] = fmaf(t.live ? wu : 0.f, fmaf(t.fv, b - a, a), acc[0][j]);
        } else {
          const float b0 = w0 * t.fv, b1 = w1 * t.fv, a0 = w0 - b0, a1 = w1 - b1;
#pragma unroll
          for (int q = 0; q < NQ; ++q) {
            float val = a0 * t.p[q][0];
            val = fmaf(a1, t.p[q][1], val);
            val = fmaf(b0, t.p[q][2], val);
            val = fmaf(b1, t.p[q][3], val);
            acc[q][j] += val;
          }
        }
      }
    }
    __builtin_amdgcn_s_waitcnt(0x0f70);
    __syncthreads();
  }
  if (groups > 1) {  // group g hands its sums to group 0 through LDS, in order
    for (int g1 = 1; g1 < groups; ++g1) {
#pragma unroll
      for (int q = 0; q < NQ; ++q)
#pragma unroll
        for (int j = 0; j < ZC; ++j)
          if (group == g1) patches[(q * ZC + j) * 256 + tid] = acc[q][j];
      __syncthreads();
#pragma unroll
      for (int q = 0; q < NQ; ++q)
#pragma unroll
        for (int j = 0; j < ZC; ++j)
          if (group == 0) acc[q][j] += patches[(q * ZC + j) * 256 + tid];
      __syncthreads();
    }
    if (group != 0) return;
  }
  // (the lane's column again: kept over the views it would cost registers)
  int tl = threadIdx.x;  // (below 256: group 0)
  asm volatile("" : "+v"(tl));
  const int xs = xw + tl % 8, ys = yw + (tl & 63) / 8;
  if (xs >= xb || ys >= yb) return;
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    int xq = xs, yq = ys;
    // an odd volume's middle row holds whole orbits (half turns), or turned middle
    // columns and the centre (quarter turns): each voxel is stored once
    if (NQ > 1 && 2 * ys + 1 == g.ny && (q > 0 || (NQ == 4 && 2 * xs + 1 != g.nx))) continue;
    if (NQ > 1) {
      const int m = NQ == 2 ? 2 * q : (turn > 0 ? q : (4 - q) & 3);  // quarter turns (x, y) -> (n - 1 - y, x)
      xq = m == 0 ? xs : (m == 1 ? g.nx - 1 - ys : (m == 2 ? g.nx - 1 - xs : ys));
      yq = m == 0 ? ys : (m == 1 ? xs : (m == 2 ? g.ny - 1 - ys : g.nx - 1 - xs));
    }
#pragma unroll
    for (int j = 0; j < ZC; ++j) {
      if (z0 + j >= g.nz) break;
      float* o = vol + ((size_t)(z0 + j) * g.ny + yq) * g.nx + xq;
      *o = accumulate ? *o + acc[q][j] : acc[q][j];
    }
  }
}

// Volumes too small to fill the chip with tiles, and voxels so coarse on the
// detector that a tile's patch does not fit in LDS: taps straight from the
// padded views, in two 8-byte gathers a voxel: a gather costs by the lines its lanes
// reach, and four of 4 bytes took 443 us for 378 in the reference geometry's FDK, and
// twice as long in volumes of 34^3 to 60^3 (158 : 73 us for 35 x 28 x 34 from 322 views).
// A wave takes 64 columns in a row (x fastest) over ZC voxels, and
// the block's waves share the views out, so a small volume's chain of views is
// short (one voxel takes the latency of a view's set-up and gathers after
// another); their sums are added in wave order, so the volume does not depend
// on scheduling.
typedef float Pair4 __attribute__((ext_vector_type(2), aligned(4)));  // two floats at any 4-byte address

template <int ZC, bool ZEROS>
__global__ __launch_bounds__(1024) void backproject_direct_kernel(const float* __restrict__ pad,
                                                                  const BpView* __restrict__ views, int view0,
                                                                  int nviews, BpGrid g, float* __restrict__ vol,
                                                                  int accumulate, int col_blocks, int zc0) {
  extern __shared__ float part[];  // [waves][ZC][64]
  const int cb_i = blockIdx.x % col_blocks, zc = zc0 + blockIdx.x / col_blocks;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  const int ncx = g.x1 - g.x0, ncol = ncx * g.ny;
  const int col = min(cb_i * 64 + lane, ncol - 1);
  const int y = col / ncx, x = g.x0 + col - y * ncx;
  const int z0 = zc * ZC;
  const int zb = (z0 / kZBase) * kZBase, joff = z0 - zb - kZMid;
  const double X = voxel_x(g, x), Y = voxel_y(g, y), Zb = base_z(g, zb + kZMid);
  const float Xf = (float)X, Yf = (float)Y;
  const size_t view_stride = (size_t)g.rows * g.pitch;
  float acc[ZC];
#pragma unroll
  for (int j = 0; j < ZC; ++j) acc[j] = 0.f;
  const int ka = view0 + (int)((long)wave * nviews / waves), kb = view0 + (int)((long)(wave + 1) * nviews / waves);
  for (int k = ka; k < kb; ++k) {
    const BpView& c = views[k];
    const ColumnCore cc = column_core<ZEROS>(c, X, Y, Xf, Yf, g);
    // v in 32.32 fixed point: any step per voxel
    long long sv = __double2ll_rn(fmin(fmax(fma(cc.kv, Zb, c.sv0), -1.0e6), 1.0e6) * 4294967296.0);
    const long long dv = __double2ll_rn(cc.kv * g.gsz * 4294967296.0);
    const long long lo = (long long)g.lo_v << 32, hi = (long long)g.hi_v << 32;
    const float* src = pad + (size_t)k * view_stride;
    const uint32_t off0 = (uint32_t)(kPadLo * g.pitch + cc.iu + kPadLo);
    sv += joff * dv;
    int zo = z0, xm = x;  // (opaque: voxel coordinates and mask squares are formed where they are used)
    asm volatile("" : "+s"(zo), "+v"(xm));
    // whether a lane's voxels come within a row of the window's edge
    const long long sl = sv + (ZC - 1) * dv, one = 1LL << 32;
    const bool edge = __any(min(sv, sl) < lo + one || max(sv, sl) > hi - one);
    const float wu = ZEROS || cc.ok ? cc.w : 0.f;
    const float w1 = wu * cc.fu, w0 = wu - w1;
#pragma unroll
    for (int j = 0; j < ZC; ++j) {
      bool live = ZEROS || in_mask(g, xm, y, zo + j);
      long long sc = sv;
      if (edge) {
        if (!ZEROS) live = live && in_window(cc, c, g, zo + j);
        sc = sv < lo ? lo : (sv > hi ? hi : sv);
      }
      const float fv = (float)(uint32_t)sc * 2.3283064365386963e-10f;  // 2^-32
      const float m0 = live ? w0 : 0.f, m1 = live ? w1 : 0.f;
      const float b0 = m0 * fv, b1 = m1 * fv;
      const uint32_t at = off0 + (uint32_t)__mul24((int)(sc >> 32), g.pitch);
      sv += dv;
      const Pair4 ta = *(const Pair4*)(src + at), tb = *(const Pair4*)(src + at + (uint32_t)g.pitch);
      float val = (m0 - b0) * ta.x;
      val = fmaf(m1 - b1, ta.y, val);
      val = fmaf(b0, tb.x, val);
      val = fmaf(b1, tb.y, val);
      acc[j] += val;
    }
  }
#pragma unroll
  for (int j = 0; j < ZC; ++j) part[(wave * ZC + j) * 64 + lane] = acc[j];
  __syncthreads();
  const int own = cb_i * 64 + lane;
  const int oy = own / ncx, ox = g.x0 + own - oy * ncx;
  if (own >= ncol) return;
  for (int j = wave; j < ZC; j += waves) {
    if (z0 + j >= g.nz) break;
    float sum = 0.f;
    for (int w = 0; w < waves; ++w) sum += part[(w * ZC + j) * 64 + lane];
    float* o = vol + ((size_t)(z0 + j) * g.ny + oy) * g.nx + ox;
    *o = accumulate ? *o + sum : sum;
  }
}

// Bounds on the patch of a tile of tile_x x tile_y columns and zc voxels: rows
// and columns of the detector it can touch in any view, taps included.  su and
// sv move by at most |suk| s and |svk| s per unit of length across the tile,
// s = sqrt(U^2 + y'^2) / U^2 for su (largest on the circle through the volume's
// farthest corner), 1 / U along z and |Z| / U^2 across for sv.
static void patch_bounds(const BpGrid& g, const BpReach& r, int tile_x, int tile_y, int zc, int& rows, int& cols) {
  const double dx = (tile_x - 1) * std::fabs(g.gsx), dy = (tile_y - 1) * std::fabs(g.gsy);
  const double diag = std::sqrt(dx * dx + dy * dy);
  double c = -(r.sod * r.sod + 2.0 * r.rad * r.rad) / (3.0 * r.sod * std::max(r.rad, 1e-30));
  c = std::min(1.0, std::max(-1.0, c));
  const double U = r.sod + r.rad * c, s = std::sqrt(r.sod * r.sod + 2.0 * r.sod * r.rad * c + r.rad * r.rad) / (U * U);
  const double um = r.sod - r.rad;
  const double zs = std::fabs(g.gsz);
  const double zmax = std::max(std::fabs(g.gz0), std::fabs(g.gz0 + (g.nz + zc) * g.gsz));
  const double wu = r.suk * s * diag, wv = r.svk * ((zc - 1) * zs / um + zmax * diag / (um * um));
  // floor of the two ends' difference, the 0.01 margin of the origin, and the tap above
  cols = wu < 1e6 ? (int)std::floor(wu + 0.03) + 3 : 1 << 20;
  rows = wv < 1e6 ? (int)std::floor(wv + 0.03) + 3 : 1 << 20;
}

// Whether the patches of an orbit fit, two for each of `groups` in a CU's 160 KB of LDS.
template <int NQ>
static bool patch_fits(int rows, int cols, int groups) {
  using L = PatchLayout<NQ>;
  return cols <= L::kCols && rows <= L::kMaxRows && 2 * sizeof(float) * rows * L::kRS * groups <= 156 * 1024;
}
static bool patch_fits(int orbit, int rows, int cols, int groups) {
  return orbit == 4 ? patch_fits<4>(rows, cols, groups)
                    : (orbit == 2 ? patch_fits<2>(rows, cols, groups) : patch_fits<1>(rows, cols, groups));
}

// Which kernel takes a backprojection: a property of the scan alone (sizes of
// the default tiling), so the volume does not depend on the tuned tile shape.
struct BpPlan {
  int orbit;   // columns a thread owns: 4 or 2 where 1/4 or 1/2 of a turn maps the scan onto itself, 1,
               // or 0: straight from memory
  int groups;  // groups of 4 waves that share a tile's views out
  int zc;      // voxels per thread at most
  int stack;   // 1: a block's 4 waves lie side by side over its columns; 4: one above the other
};

// The tiled kernel runs where the patches fit and there are 512 groups of 4 waves
// (2 per CU) at least: tiles of 16 voxels of z (32 for single columns, which
// halves what the set-up costs a voxel), else of 8 or 4, whose views up to 4 groups
// share; where 16 x 16 columns are too wide a patch, 8 x 8 of 4 times the
// depth.
//   These stay while 16 voxels deep, or 8 with 2048 tiles: 61 views of 161^3, 3.4 columns a
// voxel, take 381 us (487 straight from memory) at 0.9 rows a voxel, 432 (493) at 1.2; of
// 113^3 in 900 tiles of 8 172 (152) at 1.6 rows, and in tiles of 4 243 (167) at 2.4.
//   Orbits share a set-up and halve or quarter the tiles; shallow tiles pay more set-up
// than they share: below 16 voxels (8 for quarter turns), single columns are taken, from
// 40 views of 65^3 in 35 us for 45 and 193^3 in 216 for 263, from 122 views of 65^3 in
// 72 for 97 and 241^3, 2.4 pixels a voxel, in 1.72 ms for 1.85 (but of 113^3, in 252 us
// for 234).  Volumes that make fewer than 640 groups in tiles of 8 go straight from memory:
// 57^3 from 61 views in 37 us for 42, 65^3 (900 groups) in 45 for 44.
//
// A region of fewer than 8 columns along x (the reference's 5 of 256) goes straight
// from memory, whose waves take columns in a row: tiles of 8 x 8 would idle 24 lanes
// of 64 (the reference geometry's FDK took 0.83 ms so, 0.76 straight from memory with
// the filter and the gathers of then, and 0.38 now).
static BpPlan bp_plan(const BpGrid& g, const BpReach& r) {
  // a group of 16 voxels has to stay within the 40 rows of group_v's clamp
  if (g.x1 - g.x0 < 8 || !(r.svk * std::fabs(g.gsz) / (r.sod - r.rad) <= 4.5)) return {0, 1, 8, 1};
  // (the views' offsets from the first are 32-bit)
  const bool near = (double)g.n_views * g.rows * g.pitch * 4.0 < 4294967296.0;
  const int hx = (g.nx + 1) / 2, hy = (g.ny + 1) / 2;
  for (int orbit : {4, 2, 1}) {
    if (orbit > 1 && !(near && (orbit == 4 ? r.turn != 0 : r.half))) continue;
    for (int stack : {1, 4})
      for (int zc : {32, 16, 8, 4}) {
        if (zc == 32 && (orbit > 1 || stack > 1 || !r.zeros)) continue;
        if (orbit > 1 && (stack > 1 || zc < (orbit == 4 ? 8 : 16))) continue;
        const int nx = orbit == 4 ? hx : g.x1 - g.x0, ny = orbit > 1 ? hy : g.ny;
        const int tx = stack == 1 ? 16 : 8, ty = 256 / (tx * stack);
        int rows, cols;
        patch_bounds(g, r, tx, ty, zc * stack, rows, cols);
        const long tiles = (long)((nx + tx - 1) / tx) * ((ny + ty - 1) / ty) * ((g.nz + zc * stack - 1) / (zc * stack));
        if (stack > 1 && zc < 16 && (zc < 8 || tiles < 2048)) continue;
        for (int groups : {1, 2, 4})
          if (tiles * groups >= (zc < 16 && orbit == 1 ? 640 : 512) && g.n_views >= 4 * groups &&
              patch_fits(orbit, rows, cols, groups))
            return {orbit, groups, zc, stack};
      }
  }
  return {0, 1, 8, 1};
}

// The kernel and tile shape of one launch of a backprojection; false: the call cannot run.
struct BpLaunch {
  BpPlan plan;
  int zc, tile_x, tiles_x, tiles_y;
  int rows, cols;  // of a patch
  long blocks;     // (0: straight from memory)
};
static bool bp_launch(const BpGrid& grid, const BpReach& reach, int nviews_chunk, const monte_tuning& t, BpLaunch& L) {
  // taps are addressed by 32-bit offsets with a 24-bit row multiply
  if (grid.pitch >= (1 << 23) || (long long)grid.rows * grid.pitch * 4 >= (1LL << 32)) return false;
  if (t.bp_tile_x > 0 && 256 % t.bp_tile_x) return false;
  int zc = t.bp_zchunk > 0 ? t.bp_zchunk : 16;
  if (zc != 4 && zc != 8 && zc != 16) return false;
  L = BpLaunch{};
  BpPlan& plan = L.plan;
  plan = bp_plan(grid, reach);
  if (plan.orbit > 1 && nviews_chunk != grid.n_views) {  // orbits need the whole turn
    int rows, cols;
    patch_bounds(grid, reach, 16, 16, plan.zc, rows, cols);
    plan = {patch_fits<1>(rows, cols, 1) ? 1 : 0, 1, plan.zc, 1};
  }
  if (plan.orbit == 0) return true;
  const int nq = plan.orbit, groups = plan.groups, stack = plan.stack;
  zc = zc == 16 ? std::min(32, plan.zc) : std::min(zc, plan.zc);  // (the largest tuned chunk stands for 32 too)
  const int nx = nq == 4 ? (grid.nx + 1) / 2 : grid.x1 - grid.x0, ny = nq > 1 ? (grid.ny + 1) / 2 : grid.ny;
  // whole 8 x 8 sub-tiles, one per wave
  int tile_x = stack == 1 ? std::min(32, std::max(8, (int)t.bp_tile_x)) : 8;
  auto blocks_of = [&](int tx, int z) {
    const int ty = 256 / (tx * stack);
    return (long)((nx + tx - 1) / tx) * ((ny + ty - 1) / ty) * ((grid.nz + z * stack - 1) / (z * stack));
  };
  patch_bounds(grid, reach, tile_x, 256 / (tile_x * stack), zc * stack, L.rows, L.cols);
  const long most_blocks = (long)max_blocks(256 * groups);
  if (!patch_fits(nq, L.rows, L.cols, groups) || blocks_of(tile_x, zc) > most_blocks) {  // not the tuned shape: the default
    tile_x = stack == 1 ? 16 : 8;
    zc = plan.zc;
    patch_bounds(grid, reach, tile_x, 256 / (tile_x * stack), zc * stack, L.rows, L.cols);
  }
  L.zc = zc;
  L.tile_x = tile_x;
  const int tile_y = 256 / (tile_x * stack);
  L.tiles_x = (nx + tile_x - 1) / tile_x;
  L.tiles_y = (ny + tile_y - 1) / tile_y;
  L.blocks = blocks_of(tile_x, zc);
  return L.blocks <= most_blocks;
}

hipError_t launch_backproject(const float* filt_pad, const BpView* views, int view0, int nviews_chunk,
                              const BpGrid& grid, const BpReach& reach, float* vol, int accumulate,
                              const monte_tuning& t, hipStream_t s) {
  BpLaunch L;
  if (!bp_launch(grid, reach, nviews_chunk, t, L)) return hipErrorInvalidValue;
  const int ncx = grid.x1 - grid.x0;
  if (ncx <= 0 || grid.ny <= 0 || grid.nz <= 0 || nviews_chunk <= 0) return hipSuccess;
  const int nq = L.plan.orbit, groups = L.plan.groups, stack = L.plan.stack, zc = L.zc, rows = L.rows;
  if (nq == 0) {
    // 8 voxels a lane (16 spill registers in the bp3d20 preset), and waves per block
    // until about 4 per SIMD are in flight
    constexpr int zd = 8;
    const long ncol = (long)ncx * grid.ny, cb = (ncol + 63) / 64;
    const int most = std::min(16, std::max(1, nviews_chunk / 2));
    const int zchunks = (grid.nz + zd - 1) / zd;
    int waves = 1;
    while (2 * waves <= most && cb * zchunks * waves < 4096) waves *= 2;
    const int step = (int)std::min<long>(zchunks, max_blocks(64 * waves) / cb);  // chunks of z of a launch
    if (step == 0) return hipErrorInvalidValue;
#define MONTE_BP(ZEROS)                                                                                        \
  hipLaunchKernelGGL((backproject_direct_kernel<zd, ZEROS>), dim3((unsigned)(cb * n)), dim3(64 * waves),       \
                     sizeof(float) * waves * zd * 64, s, filt_pad, views, view0, nviews_chunk, grid, vol,      \
                     accumulate, (int)cb, z)
    for (int z = 0; z < zchunks; z += step) {
      const int n = std::min(step, zchunks - z);
      if (reach.zeros) MONTE_BP(true); else MONTE_BP(false);
    }
#undef MONTE_BP
    return hipGetLastError();
  }
  // the groups' patches, which the sums of a group go through at the end
  auto lds_of = [&](int row_words, int sums) {
    const size_t patch = (size_t)2 * rows * row_words * groups;
    return sizeof(float) * (groups > 1 ? std::max(patch, (size_t)sums * 256) : patch);
  };
#define MONTE_BP(ZC, NQ, ZEROS)                                                                                \
  hipLaunchKernelGGL((backproject_kernel<ZC, NQ, ZEROS>), dim3((unsigned)L.blocks), dim3(256 * groups), \
                     lds_of(PatchLayout<NQ>::kRS, NQ * ZC), s, filt_pad, views, view0, nviews_chunk,          \
                     grid, vol, accumulate, L.tile_x, L.tiles_x, L.tiles_y, rows, reach.turn, stack)
#define MONTE_BP_Z(NQ, ZEROS)                                                                                    \
  switch (zc) {                                                                                                \
    case 4: MONTE_BP(4, NQ, ZEROS); break;                                                                            \
    case 8: MONTE_BP(8, NQ, ZEROS); break;                                                                            \
    default: MONTE_BP(16, NQ, ZEROS); break;                                                                   \
  }
  if (nq == 4) { MONTE_BP_Z(4, true) }
  else if (nq == 2) { MONTE_BP_Z(2, true) }
  else if (zc == 32) MONTE_BP(32, 1, true);
  else if (reach.zeros) { MONTE_BP_Z(1, true) }
  else { MONTE_BP_Z(1, false) }
#undef MONTE_BP_Z
#undef MONTE_BP
  return hipGetLastError();
}

// ------------------------------------------- transposed backprojection
// The matched projector, written as a gather so no atomics are needed.
// One wave owns a strip of kStripW padded detector columns (all rows) of one
// view, held in its own LDS.  It walks the voxel columns whose left tap
// lands in the strip (each voxel column of the view belongs to exactly one
// strip; its right tap may spill into the next strip's first column), from a
// list enumerated once per geometry: for each slab of the volume across the view's rays
// (x-slabs when |cos b| >= |sin b|, y-slabs otherwise) the projective map
// su(X,Y) is inverted at the strip's two edges, giving a range of columns on
// that slab (widened by one voxel each side).  The lanes evaluate the
// candidate columns of a range in parallel with the backprojector's own
// column arithmetic and keep those whose taps fall in the strip.  Each kept
// column is then walked along z by the whole wave: lane l takes the C
// consecutive voxels of chunk l, from a z-fastest copy of the volume.  The
// column core (u tap, fraction, distance weight) is the backprojector's own;
// the v coordinate sv(z) = A + z D of each voxel is formed in 32.32 fixed
// point from the column's FP64 A and D (integer row = high word, fraction =
// low word), within 2^-32 rows of the backprojector's value.
//
// Accumulation is a plain read-add-write of LDS, without atomics: in one
// instruction the active lanes' voxels are C apart along z, hence at least
// C |dsv| rows apart on the detector, and when C |dsv| > 1.01 no two lanes
// touch the same cell.  Columns with a smaller v-slope run in several phases
// over interleaved lane subsets that satisfy the same bound.  The upper tap
// row is updated by a second read-add-write after the first completes, and a
// wave's LDS operations execute in program order, so updates of a cell by
// neighbouring lanes, later voxels and later columns all see each other.
// LDS column kStripC0 + kStripW collects the right-tap spill into the next
// strip.  The kernel's speed follows the number of waves a CU holds, and a
// wave's LDS is its strip: with the column lists built once per geometry
// (below), one-column strips ran 13.1 ms at 325^3 / 512^2 / 360 views,
// against 14.7, 15.2 and 16.6 ms for strips of 2, 3 and 5 columns.  A row is
// then the pair (left tap, spill), read and written as one 8-byte access
// (11.8 ms, against 12.3 ms for pitch 3 and 13.0 ms for pitch 4).
constexpr int kStripW = 1;
constexpr int kStripP = 2;
constexpr int kStripC0 = 0;  // LDS column of the strip's first column

// A cell and its right neighbour (left and right tap of one row), as one
// 8-byte LDS access when the layout keeps them 8-byte aligned.
constexpr bool kPairAligned = kStripP % 2 == 0 && kStripC0 % 2 == 0;
__device__ inline float2 lds_get2(const float* strip, int i) {
  if constexpr (kPairAligned) return *(const float2*)(strip + i);
  return make_float2(strip[i], strip[i + 1]);
}
__device__ inline void lds_put2(float* strip, int i, float2 v) {
  if constexpr (kPairAligned) {
    *(float2*)(strip + i) = v;
  } else {
    strip[i] = v.x;
    strip[i + 1] = v.y;
  }
}
__device__ inline void lds_add2(float* strip, int i, float a, float b) {
  float2 x = lds_get2(strip, i);
  x.x += a;
  x.y += b;
  lds_put2(strip, i, x);
}

// Columns of one strip on each slab.  The strip's two edges su = s_lo and
// su = s_hi are lines through the source; on a slab (x fixed for x-slabs, y
// fixed for y-slabs) each crosses the other coordinate at
//   t = (q (c1 coord + c0) - a1 coord) / (a2 - q c2),  q = (s - su0) / suk,
// with (c1, c2, a1, a2) = (cx, cy, ax, ay) for x-slabs and (cy, cx, ay, ax)
// for y-slabs.  The denominators depend only on the view and the edge, so the
// per-slab work is two multiply-adds per edge.  The range is widened by one
// voxel each side; every column in it is then tested exactly.
struct SlabRanges {
  double q0, q1, id0, id1;  // edge parameters and reciprocal denominators
  double o0, ios;           // voxel index = (t - o0) * ios along the slab
  int n;                    // voxels along the slab
  bool whole;               // an edge, or a direction between them, runs along the slabs: take every column

  __device__ void init(double s_lo, double s_hi, const BpView& c, bool x_slabs, const BpGrid& g) {
    q0 = (s_lo - c.su0) / c.suk;
    q1 = (s_hi - c.su0) / c.suk;
    const double a2 = x_slabs ? c.ay : c.ax, c2 = x_slabs ? c.cy : c.cx;
    const double d0 = a2 - q0 * c2, d1 = a2 - q1 * c2;
    // (of opposite signs: a direction between the edges, 45 degrees or more off the axis, runs along the slabs)
    whole = fabs(d0) < 1e-12 || fabs(d1) < 1e-12 || (d0 < 0.0) != (d1 < 0.0);
    id0 = 1.0 / d0;
    id1 = 1.0 / d1;
    o0 = x_slabs ? g.gy0 : g.gx0;
    ios = 1.0 / (x_slabs ? g.gsy : g.gsx);
    n = x_slabs ? g.ny : g.nx;
  }
  __device__ void range(const BpView& c, bool x_slabs, double coord, int& a, int& b) const {
    if (whole) { a = 0; b = n - 1; return; }
    const double c1 = x_slabs ? c.cx : c.cy, a1 = x_slabs ? c.ax : c.ay;
    const double base = c1 * coord + c.c0;
    const double t0 = (q0 * base - a1 * coord) * id0, t1 = (q1 * base - a1 * coord) * id1;
    const double i0 = (t0 - o0) * ios, i1 = (t1 - o0) * ios;
    a = (int)fmax(floor(fmin(i0, i1)) - 1.0, 0.0);
    b = (int)fmin(ceil(fmax(i0, i1)) + 1.0, (double)(n - 1));
  }
};

__device__ inline int bcast_i(int v, int src) { return __builtin_amdgcn_readlane(v, src); }
__device__ inline float bcast_f(float v, int src) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), src));
}
__device__ inline double bcast_d(double v, int src) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffLL), src);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), src);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// Keeps the compiler from moving LDS accesses across this point; the hardware
// already executes one wave's LDS operations in order.
__device__ inline void lds_order() { asm volatile("" ::: "memory"); }

// Passes (64 chunks of C voxels) whose volume values are fetched one column
// ahead; columns longer than kPrefetchZ / C / 64 passes load the rest in place.
constexpr int kPrefetchZ = 512;
constexpr int kAhead = 2;
// Views per group of the projector's block order (see project_kernel): 4, 8
// and 16 took 10.4, 10.0 and 10.4 ms at 325^3 / 360 views (51 -> 35, 26 and
// 29 GB of fabric reads), 76.5, 74.1 and 75.3 ms at 512^3 / 720 views.
constexpr int kProjViewGroup = 8;
// LDS floats after the strip that absorb the updates of lanes with nothing to
// add (outside the v window or past the column end), so the updates need no
// branches: two per lane, two row pitches and one cell of overlap.  (Branches
// around the updates, or handing the upper-row update to the next lane by a
// DPP shift, both measured slower.)
constexpr int kTrash = 2 * 64 + 2 * kStripP + 2;

template <int C>
struct ColumnVals {
  static constexpr int NP = (kPrefetchZ / C + 63) / 64;
  float v[NP][C];
};

template <bool MASK>
__device__ inline bool in_mask_t(const BpGrid& g, int x, int y, int z) {
  if (!MASK) return true;
  const int dz = z - g.mcz, dy = y - g.mcy, dx = x - g.mcx;
  return (float)(dz * dz + dy * dy + dx * dx) <= g.mask_r2;
}

// Volume values of chunk (p * 64 + lane) of a column, zero past the end and
// outside the mask; the load itself is clamped into the column, so it is
// unconditional.
template <int C, bool MASK>
__device__ inline void load_chunk(float (&v)[C], const float* __restrict__ col, int p, int x, int y,
                                  const BpGrid& g, int lane) {
#pragma unroll
  for (int j = 0; j < C; ++j) {
    const int z = (p * 64 + lane) * C + j;
    const float val = col[min(z, g.nz - 1)];
    v[j] = (z < g.nz && in_mask_t<MASK>(g, x, y, z)) ? val : 0.f;
  }
}

template <int C, bool MASK>
__device__ inline void load_column(ColumnVals<C>& cv, const float* __restrict__ col, int x, int y, const BpGrid& g,
                                   int lane, int npass) {
#pragma unroll
  for (int p = 0; p < ColumnVals<C>::NP; ++p)
    if (p < npass) load_chunk<C, MASK>(cv.v[p], col, p, x, y, g, lane);
}

// The v coordinate of a column in 32.32 fixed point: sv(z) = a + z d, and the
// v window [lo, hi] (the backprojector's, inclusive).
struct ColumnFx {
  long long a, d, lo, hi;
};

__device__ inline ColumnFx column_fx(const ColumnCore& cc, const BpView& c, const BpGrid& g) {
  ColumnFx f;
  const double A = fma(cc.kv, g.gz0, c.sv0), D = cc.kv * g.gsz;
  f.a = __double2ll_rn(fmin(fmax(A, -1.0e6), 1.0e6) * 4294967296.0);
  f.d = __double2ll_rn(D * 4294967296.0);
  f.lo = (long long)g.lo_v * 4294967296LL;
  f.hi = (long long)g.hi_v * 4294967296LL;
  return f;
}

// Row (floor) and fraction of a fixed-point coordinate.
__device__ inline int fx_row(long long s) { return (int)(s >> 32); }
__device__ inline float fx_frac(long long s) { return (float)(uint32_t)s * 2.3283064365386963e-10f; }  // 2^-32

// The C voxel updates of one lane; lanes with `act` false (or nothing to add)
// update their trash floats instead.
template <int C>
__device__ inline void pass_updates(float* __restrict__ strip, const float (&v)[C], const ColumnCore& cc,
                                    long long s0, long long d, long long lo, long long hi, int z0, bool act,
                                    int cell0, int trash, const BpGrid& g) {
#pragma unroll
  for (int j = 0; j < C; ++j) {
    const long long sj = s0 + j * d;
    const int row = fx_row(sj);
    const float fv = fx_frac(sj);
    const bool live = act && sj >= lo && sj <= hi && z0 + j < g.nz;
    const float sw = cc.w * v[j];
    const float bb = sw * fv, aa = sw - bb;
    const float a1 = aa * cc.fu, b1 = bb * cc.fu;
    const int i0 = live ? cell0 + row * kStripP : trash;
    lds_add2(strip, i0, aa - a1, a1);
    lds_order();
    lds_add2(strip, i0 + kStripP, bb - b1, b1);
    lds_order();
  }
}

// Both voxels of a 2-voxel chunk, when the v-slope is in (0, 1): the second
// voxel's row is the first's or the one above, so the lane's four row updates
// fold into three consecutive rows r, r + 1, r + 2, added in three rounds.  In
// round k every lane updates its row r + k; the lanes' rows r strictly
// increase, so no two lanes of a round touch the same cell.
struct PairRows {
  int i0;            // LDS index of (row r, left tap), or the trash floats
  float q0, q1, q2;  // totals for rows r, r + 1, r + 2
};

__device__ inline PairRows pair_rows(const float (&v)[2], const ColumnCore& cc, long long s0, long long d,
                                     long long lo, long long hi, int z0, int cell0, int trash, const BpGrid& g) {
  const long long s1 = s0 + d;
  const int r0 = fx_row(s0), r1 = fx_row(s1);
  const bool live0 = s0 >= lo && s0 <= hi && z0 < g.nz, live1 = s1 >= lo && s1 <= hi && z0 + 1 < g.nz;
  const float sw0 = live0 ? cc.w * v[0] : 0.f, sw1 = live1 ? cc.w * v[1] : 0.f;
  const float b0 = sw0 * fx_frac(s0), a0 = sw0 - b0;
  const float b1 = sw1 * fx_frac(s1), a1 = sw1 - b1;
  const bool same = r1 == r0;
  PairRows p;
  p.q0 = a0 + (same ? a1 : 0.f);
  p.q1 = b0 + (same ? b1 : a1);
  p.q2 = same ? 0.f : b1;
  p.i0 = (live0 || live1) ? cell0 + r0 * kStripP : trash;
  return p;
}

__device__ inline float pair_q(const PairRows& p, int k) { return k == 0 ? p.q0 : (k == 1 ? p.q1 : p.q2); }

__device__ inline void pass_updates_pair(float* __restrict__ strip, const float (&v)[2], const ColumnCore& cc,
                                         long long s0, long long d, long long lo, long long hi, int z0, int cell0,
                                         int trash, const BpGrid& g) {
  const PairRows p = pair_rows(v, cc, s0, d, lo, hi, z0, cell0, trash, g);
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const int i = p.i0 + k * kStripP;
    const float q = pair_q(p, k), t = q * cc.fu;
    lds_add2(strip, i, q - t, t);
    lds_order();
  }
}

// Two pair passes whose rows cannot meet, run round by round together so each
// round's two reads are in flight at once.  Passes p and p + 2 of a column
// start 256 voxels apart, so at a v-slope above 0.505 rows per voxel the first
// row of the later pass lies more than 64 rows above the last row (r + 2) of
// the earlier.
__device__ inline void pass_updates_pair2(float* __restrict__ strip, const float (&va)[2], const float (&vb)[2],
                                          const ColumnCore& cc, long long sa, long long sb, long long d,
                                          long long lo, long long hi, int za, int zb, int cell0, int trash,
                                          const BpGrid& g) {
  const PairRows a = pair_rows(va, cc, sa, d, lo, hi, za, cell0, trash, g);
  const PairRows b = pair_rows(vb, cc, sb, d, lo, hi, zb, cell0, trash, g);
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const int ia = a.i0 + k * kStripP, ib = b.i0 + k * kStripP;
    const float qa = pair_q(a, k), ta = qa * cc.fu;
    const float qb = pair_q(b, k), tb = qb * cc.fu;
    const float2 xa = lds_get2(strip, ia), xb = lds_get2(strip, ib);
    lds_put2(strip, ia, make_float2(xa.x + (qa - ta), xa.y + ta));
    lds_put2(strip, ib, make_float2(xb.x + (qb - tb), xb.y + tb));
    lds_order();
  }
}

// Every pass of an unfolded column at once (npass <= NP, one lane phase),
// round by round: per voxel j of a lane's chunk, every pass updates the lower
// then the upper row of its voxel.  The rows of all lanes of all passes in one
// round are distinct (consecutive lanes, and the last lane of a pass and the
// first of the next, are C voxels apart, so their rows differ by at least
// C |dsv| > 1.01), so a round's reads of all passes are issued before its
// writes and the passes' LDS latencies overlap.  Rounds follow each other in
// program order.
template <int C, int NP>
__device__ inline void column_interleaved(float* __restrict__ strip, const float (&v)[NP][C], const ColumnCore& cc,
                                          const ColumnFx& fx, int cell0, int trash, int npass, const BpGrid& g,
                                          int lane) {
#pragma unroll
  for (int j = 0; j < C; ++j) {
    int i0[NP];
    float aa[NP], a1[NP], bb[NP], b1[NP];
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int z = (p * 64 + lane) * C + j;
      const long long sj = fx.a + (long long)z * fx.d;
      const bool live = p < npass && sj >= fx.lo && sj <= fx.hi && z < g.nz;
      const float sw = cc.w * v[p][j];
      bb[p] = sw * fx_frac(sj);
      aa[p] = sw - bb[p];
      a1[p] = aa[p] * cc.fu;
      b1[p] = bb[p] * cc.fu;
      i0[p] = live ? cell0 + fx_row(sj) * kStripP : trash;
    }
    float2 x[NP];
#pragma unroll
    for (int p = 0; p < NP; ++p)
      if (p < npass) x[p] = lds_get2(strip, i0[p]);
#pragma unroll
    for (int p = 0; p < NP; ++p)
      if (p < npass) lds_put2(strip, i0[p], make_float2(x[p].x + (aa[p] - a1[p]), x[p].y + a1[p]));
    lds_order();
#pragma unroll
    for (int p = 0; p < NP; ++p)
      if (p < npass) x[p] = lds_get2(strip, i0[p] + kStripP);
#pragma unroll
    for (int p = 0; p < NP; ++p)
      if (p < npass) lds_put2(strip, i0[p] + kStripP, make_float2(x[p].x + (bb[p] - b1[p]), x[p].y + b1[p]));
    lds_order();
  }
}

// One pass of a column: lane l takes the C voxels of chunk ch0 + l.  `cell0`
// is the LDS index of (row 0, left tap); `trash` the lane's trash floats;
// `phases` is the number of interleaved lane phases, or 0 for the folded
// two-voxel updates (C = 2 and a v-slope in (0.505, 0.999)).
template <int C>
__device__ inline void project_pass(float* __restrict__ strip, const float (&v)[C], const ColumnCore& cc,
                                    const ColumnFx& fx, int cell0, int trash, int ch0, int phases,
                                    const BpGrid& g, int lane) {
  const int z0 = (ch0 + lane) * C;
  const long long s0 = fx.a + (long long)z0 * fx.d;
  if constexpr (C == 2) {
    if (phases == 0) {
      pass_updates_pair(strip, v, cc, s0, fx.d, fx.lo, fx.hi, z0, cell0, trash, g);
      return;
    }
  }
  if (phases == 1) {
    pass_updates<C>(strip, v, cc, s0, fx.d, fx.lo, fx.hi, z0, true, cell0, trash, g);
  } else {
    const int ml = lane % phases;
    for (int ph = 0; ph < phases; ++ph)
      pass_updates<C>(strip, v, cc, s0, fx.d, fx.lo, fx.hi, z0, ml == ph, cell0, trash, g);
  }
}

// Up to 64 kept voxel columns of one strip, lane i holding the i-th.
struct ColumnBatch {
  int n = 0;
  int iu = 0, x = 0, y = 0;
  float fu = 0.f, w = 0.f, dsv = 0.f;
  double kv = 0.0;
};

// The projector's per-column constants, computed by lane i for the i-th
// listed column of a batch (all 64 columns at once), then read by the whole
// wave with readlane when the column's turn comes.
struct ColumnPrep {
  int x = 0, y = 0;
  float fu = 0.f, w = 0.f;
  long long a = 0, d = 0;  // sv(z) = a + z d in 32.32 fixed point
  int phases = 1;          // lane phases, 0 = folded two-voxel updates
  int cell0 = 0;           // LDS index of (padded row 0, left tap)
};

__device__ inline long long bcast_ll(long long v, int src) {
  const int lo = __builtin_amdgcn_readlane((int)(v & 0xffffffffLL), src);
  const int hi = __builtin_amdgcn_readlane((int)(v >> 32), src);
  return ((long long)hi << 32) | (unsigned int)lo;
}

__device__ inline int permute_i(int dst, int v) { return __builtin_amdgcn_ds_permute(dst << 2, v); }
__device__ inline float permute_f(int dst, float v) {
  return __int_as_float(__builtin_amdgcn_ds_permute(dst << 2, __float_as_int(v)));
}

// Whether column (x, y) of the first quadrant or half stands for its orbit: an odd
// volume's middle row holds whole orbits of half a turn, and turned middle columns.
__device__ inline bool orbit_first(int orbit, int x, int y, int nx, int ny) {
  if (orbit == 1 || 2 * y + 1 != ny || 2 * x + 1 == nx) return true;
  return orbit == 2 && 2 * x + 1 < nx;
}

// Walks the strip's slabs four at a time, 16 lanes per slab, and appends the
// kept columns to the batch (each kept lane pushes its column to lane n + its
// rank; the other lanes push to the lanes past the new end), until the batch
// is full or the slabs are exhausted.  Returns false when nothing is left.
struct Enumerator {
  SlabRanges sr;
  int s0 = 0;   // first slab of the current group of four
  int rnd = 0;  // 16-column round within the group

  __device__ bool fill(ColumnBatch& cb, const BpView& c, const BpGrid& g, bool x_slabs, int n_slabs, int u_lo,
                       int u_hi, int lane, int orbit, int full_ny) {
    cb.n = 0;
    for (;;) {
      if (s0 >= n_slabs) return cb.n > 0;
      const int sl = s0 + (lane >> 4);
      int a = 0, b = -1;
      if (sl < n_slabs) {
        const int sc = x_slabs ? g.x0 + sl : sl;
        sr.range(c, x_slabs, x_slabs ? voxel_x(g, sc) : voxel_y(g, sc), a, b);
        if (!x_slabs) {
          a = max(a, g.x0);
          b = min(b, g.x1 - 1);
        }
      }
      const int w = max(b - a + 1, 0);
      const int need = max(max(bcast_i(w, 0), bcast_i(w, 16)), max(bcast_i(w, 32), bcast_i(w, 48)));
      const int off = a + rnd * 16 + (lane & 15);
      const int o = min(off, max(b, a));
      const int xo = x_slabs ? g.x0 + sl : o, yo = x_slabs ? o : sl;
      const int x = min(xo, g.x1 - 1), y = min(yo, g.ny - 1);
      const double X = voxel_x(g, x), Y = voxel_y(g, y);
      const ColumnCore mine = column_core(c, X, Y, (float)X, (float)Y, g);
      const bool keep = sl < n_slabs && off <= b && mine.ok && mine.iu >= u_lo && mine.iu <= u_hi &&
                        orbit_first(orbit, x, y, g.nx, full_ny);
      const uint64_t m = __ballot(keep);
      const int cnt = (int)__popcll(m);
      if (cb.n + cnt > 64) return true;  // full: this round is taken again by the next fill
      if (++rnd * 16 >= need) {
        rnd = 0;
        s0 += 4;
      }
      if (!cnt) continue;
      const uint32_t rk = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
      const int dst = keep ? cb.n + (int)rk : (cb.n + cnt + (lane - (int)rk)) & 63;
      const bool fresh = lane >= cb.n && lane < cb.n + cnt;
      const long long kvb = __double_as_longlong(mine.kv);
      const int kv_lo = permute_i(dst, (int)(kvb & 0xffffffffLL)), kv_hi = permute_i(dst, (int)(kvb >> 32));
      const int piu = permute_i(dst, mine.iu), px = permute_i(dst, x), py = permute_i(dst, y);
      const float pfu = permute_f(dst, mine.fu), pw = permute_f(dst, mine.w), pdsv = permute_f(dst, mine.dsv);
      if (fresh) {
        cb.iu = piu; cb.x = px; cb.y = py;
        cb.fu = pfu; cb.w = pw; cb.dsv = pdsv;
        cb.kv = __longlong_as_double(((long long)kv_hi << 32) | (unsigned int)kv_lo);
      }
      cb.n += cnt;
      if (cb.n == 64) return true;
    }
  }
};

// The strip's geometry in a view: owned detector columns and slab setup.
struct StripSetup {
  int pu0, u_lo, u_hi, n_slabs;
  bool x_slabs;
  double s_lo, s_hi;
  __device__ StripSetup(const BpView& c, const BpGrid& g, int st) {
    pu0 = st * kStripW;   // first padded column of the strip
    u_lo = pu0 - kPadLo;  // first detector column index owned
    u_hi = u_lo + kStripW - 1;
    x_slabs = fabs(c.cx) >= fabs(c.cy);
    // columns whose left tap iu satisfies u_lo <= iu <= u_hi, i.e. su in [u_lo, u_hi + 1)
    s_lo = (double)u_lo - 0.5;
    s_hi = (double)(u_hi + 1) + 0.5;
    n_slabs = x_slabs ? (g.x1 - g.x0) : g.ny;
  }
};

// Column lists of the matched projector, built once per geometry: for view k
// and strip st, the voxel columns whose left tap lands in the strip, in the
// enumeration order above, packed as x | y << 16.  The first pass (WRITE
// false) stores each list's length at offs[k * n_strips + st]; the second
// writes the list at list + offs[k * n_strips + st] (offsets by then).
template <bool WRITE>
__global__ __launch_bounds__(64) void project_plan_kernel(const BpView* __restrict__ views, int n_strips, BpGrid g,
                                                          uint32_t* __restrict__ offs, uint32_t* __restrict__ list,
                                                          int orbit, int full_ny) {
  const int k = blockIdx.x / n_strips;
  const int st = blockIdx.x - k * n_strips;
  const int lane = threadIdx.x;
  const BpView& c = views[k];
  const StripSetup ss(c, g, st);
  Enumerator en;
  en.sr.init(ss.s_lo, ss.s_hi, c, ss.x_slabs, g);
  ColumnBatch cb;
  const uint32_t base = WRITE ? offs[blockIdx.x] : 0u;
  uint32_t n = 0;
  while (en.fill(cb, c, g, ss.x_slabs, ss.n_slabs, ss.u_lo, ss.u_hi, lane, orbit, full_ny)) {
    if (WRITE && lane < cb.n) list[base + n + lane] = (uint32_t)cb.x | ((uint32_t)cb.y << 16);
    n += (uint32_t)cb.n;
  }
  if (!WRITE && lane == 0) offs[blockIdx.x] = n;
}

template <int C, bool MASK>
__global__ __launch_bounds__(64) void project_kernel(const float* __restrict__ volT,
                                                     const BpView* __restrict__ views, int view0, int n_strips,
                                                     int nviews, BpGrid g, float* __restrict__ filt, int lds_r0,
                                                     int lds_rows,
                                                     const uint32_t* __restrict__ offs,
                                                     const uint32_t* __restrict__ list) {
  // [lds_rows][kStripP] (padded rows lds_r0.., column q = padded column pu0 + q - kStripC0), then kTrash floats
  extern __shared__ float strip[];
  // Block b runs on XCD b mod 8 (blocks are dealt to the XCDs round robin):
  // XCD x takes the views [x V / 8, (x + 1) V / 8) of the launch, in groups of
  // kProjViewGroup views, strip by strip within a group.  A voxel column lands
  // in nearby strips in nearby views, so the group's waves that read it run
  // together on one XCD and its L2 serves the column to most of them.
  const int xcd = (int)(blockIdx.x % 8u), jx = (int)(blockIdx.x / 8u);
  const int va = xcd * nviews / 8, vx = (xcd + 1) * nviews / 8 - va;
  if (jx >= vx * n_strips) return;  // (the whole one-wave block)
  const int grp = jx / (kProjViewGroup * n_strips), rem = jx - grp * kProjViewGroup * n_strips;
  const int gsize = min(kProjViewGroup, vx - grp * kProjViewGroup);
  const int st = rem / gsize;
  const int k = view0 + va + grp * kProjViewGroup + (rem - st * gsize);
  const int lane = threadIdx.x;
  const int trash = lds_rows * kStripP;
  for (int i = lane; i < trash + kTrash; i += 64) strip[i] = 0.f;
  __syncthreads();

  const BpView& c = views[k];
  const int pu0 = st * kStripW;  // first padded column of the strip
  const int nch = (g.nz + C - 1) / C;
  const int npass = (nch + 63) / 64;
  constexpr int NP = ColumnVals<C>::NP;
  const size_t cell = (size_t)k * n_strips + st;
  const uint32_t beg = offs[cell], end = offs[cell + 1];

  ColumnPrep cp;
  int ncols = 0;
  const ColumnFx win = {0, 0, (long long)g.lo_v * 4294967296LL, (long long)g.hi_v * 4294967296LL};
  // The volume values of the next kAhead columns are in flight while one is
  // accumulated: a column's accumulation takes less time than a load from HBM.
  auto fetch = [&](ColumnVals<C>& dst, int i) {
    const int x = bcast_i(cp.x, i), y = bcast_i(cp.y, i);
    load_column<C, MASK>(dst, volT + ((size_t)y * g.nx + x) * g.nz, x, y, g, lane, npass);
  };
  auto accumulate = [&](const ColumnVals<C>& vals, int i) {
    ColumnCore cc;
    cc.fu = bcast_f(cp.fu, i);
    cc.w = bcast_f(cp.w, i);
    cc.ok = true;
    const int phases = bcast_i(cp.phases, i);
    const int cell0 = bcast_i(cp.cell0, i);
    ColumnFx fx = win;
    fx.a = bcast_ll(cp.a, i);
    fx.d = bcast_ll(cp.d, i);
    if constexpr (C == 2) {
      // three folded passes: the first and last together, then the middle one
      if (npass == 3 && phases == 0) {
        const int za = 2 * lane, zb = 2 * (128 + lane);
        pass_updates_pair2(strip, vals.v[0], vals.v[2], cc, fx.a + (long long)za * fx.d,
                           fx.a + (long long)zb * fx.d, fx.d, fx.lo, fx.hi, za, zb, cell0, trash + 2 * lane, g);
        project_pass<C>(strip, vals.v[1], cc, fx, cell0, trash + 2 * lane, 64, phases, g, lane);
        return;
      }
    }
    if (npass <= NP && phases == 1) {  // every pass of an unfolded column at once
      column_interleaved<C, NP>(strip, vals.v, cc, fx, cell0, trash + 2 * lane, npass, g, lane);
      return;
    }
#pragma unroll
    for (int p = 0; p < NP; ++p)
      if (p < npass) project_pass<C>(strip, vals.v[p], cc, fx, cell0, trash + 2 * lane, p * 64, phases, g, lane);
    if (npass > NP) {  // columns longer than the prefetch window load the rest in place
      const int x = bcast_i(cp.x, i), y = bcast_i(cp.y, i);
      const float* col = volT + ((size_t)y * g.nx + x) * g.nz;
      for (int p = NP; p < npass; ++p) {
        float v[C];
        load_chunk<C, MASK>(v, col, p, x, y, g, lane);
        project_pass<C>(strip, v, cc, fx, cell0, trash + 2 * lane, p * 64, phases, g, lane);
      }
    }
  };
  // Batches of 64 listed columns: lane i prepares the i-th with the same column
  // arithmetic the enumeration used to select it.
  for (uint32_t b0 = beg; b0 < end; b0 += 64) {
    ncols = (int)min(64u, end - b0);
    if (lane < ncols) {
      const uint32_t e = list[b0 + lane];
      cp.x = (int)(e & 0xffffu);
      cp.y = (int)(e >> 16);
      const double X = voxel_x(g, cp.x), Y = voxel_y(g, cp.y);
      const ColumnCore mine = column_core(c, X, Y, (float)X, (float)Y, g);
      const ColumnFx f = column_fx(mine, c, g);
      cp.fu = mine.fu;
      cp.w = mine.w;
      cp.a = f.a;
      cp.d = f.d;
      const float step = (float)C * fabsf(mine.dsv);
      const int ph = step > 1.01f ? 1 : min(64, (int)ceilf(1.01f / fmaxf(step, 1e-6f)));
      cp.phases = (C == 2 && ph == 1 && mine.dsv > 0.f && mine.dsv < 0.999f) ? 0 : ph;
      cp.cell0 = (kPadLo - lds_r0) * kStripP + (mine.iu + kPadLo - pu0) + kStripC0;
    }
    ColumnVals<C> ring[kAhead];
#pragma unroll
    for (int q = 0; q < kAhead; ++q)
      if (q < ncols) fetch(ring[q], q);
    for (int i0 = 0; i0 < ncols; i0 += kAhead) {
#pragma unroll
      for (int q = 0; q < kAhead; ++q) {
        const int i = i0 + q;
        if (i < ncols) {
          const ColumnVals<C> vals = ring[q];
          if (i + kAhead < ncols) fetch(ring[q], i + kAhead);
          accumulate(vals, i);
        }
      }
    }
  }
  __syncthreads();
  // Strip column t (LDS column t + 1) is padded column pu0 + t.  Columns 1 ..
  // kStripW - 1 belong to this strip alone; column 0 also takes the previous
  // strip's spill, and the spill column kStripW is the next strip's column 0.
  // Those two are added atomically into the zeroed output: two addends onto
  // zero, so the sum is the same in either order.
  float* out = filt + (size_t)k * g.rows * g.pitch;
  constexpr int kOut = kStripW + 1;
  for (int i = lane; i < g.rows * kOut; i += 64) {
    const int r = i / kOut, t = i - r * kOut;
    const int lr = r - lds_r0;
    if (pu0 + t >= g.pitch) continue;
    float* o = out + (size_t)r * g.pitch + pu0 + t;
    const bool held = lr >= 0 && lr < lds_rows;
    if (t == 0 || t == kStripW) {
      if (held) {
        const float val = strip[lr * kStripP + t + kStripC0];
        if (val != 0.f) unsafeAtomicAdd(o, val);
      }
    } else {
      *o = held ? strip[lr * kStripP + t + kStripC0] : 0.f;
    }
  }
}

// ------------------------------------------------------------ L2 loss
// out = a - b and the FP64 sum of out^2: each block sums a fixed grid-stride
// share in a fixed order and reduces it in a fixed tree, so the result does
// not depend on scheduling.
__global__ __launch_bounds__(256) void residual_partial_kernel(const float* __restrict__ a,
                                                               const float* __restrict__ b, float* __restrict__ out,
                                                               size_t n, double* __restrict__ partial) {
  __shared__ double red[4];
  double acc = 0.0;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
    const float r = a[i] - b[i];
    out[i] = r;
    acc = fma((double)r, (double)r, acc);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) partial[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

__global__ __launch_bounds__(256) void loss_total_kernel(const double* __restrict__ partial, int n,
                                                         double* __restrict__ loss) {
  __shared__ double red[4];
  double acc = 0.0;
  for (int i = threadIdx.x; i < n; i += 256) acc += partial[i];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) *loss = 0.5 * ((red[0] + red[1]) + (red[2] + red[3]));
}

hipError_t launch_residual_loss(const float* a, const float* b, float* out, size_t n, double* partial, double* loss,
                                hipStream_t s) {
  hipLaunchKernelGGL(residual_partial_kernel, dim3(kLossBlocks), dim3(256), 0, s, a, b, out, n, partial);
  hipLaunchKernelGGL(loss_total_kernel, dim3(1), dim3(256), 0, s, partial, kLossBlocks, loss);
  return hipGetLastError();
}

// vol [z][y][x] -> volT [y][x][z] through 32 x 32 LDS tiles (per y).
__global__ __launch_bounds__(256) void transpose_zx_kernel(const float* __restrict__ vol, float* __restrict__ volT,
                                                           int nx, int ny, int nz) {
  __shared__ float t[32][33];
  const int x0 = blockIdx.x * 32, z0 = blockIdx.y * 32, y = blockIdx.z;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8
  for (int r = ty; r < 32; r += 8) {
    const int z = z0 + r, x = x0 + tx;
    t[r][tx] = (z < nz && x < nx) ? vol[((size_t)z * ny + y) * nx + x] : 0.f;
  }
  __syncthreads();
  for (int r = ty; r < 32; r += 8) {
    const int x = x0 + r, z = z0 + tx;
    if (x < nx && z < nz) volT[((size_t)y * nx + x) * nz + z] = t[tx][r];
  }
}

hipError_t launch_transpose_zx(const float* vol, float* volT, int nx, int ny, int nz, hipStream_t s) {
  dim3 gd((nx + 31) / 32, (nz + 31) / 32, ny);
  hipLaunchKernelGGL(transpose_zx_kernel, gd, dim3(256), 0, s, vol, volT, nx, ny, nz);
  return hipGetLastError();
}

int project_strips(const BpGrid& grid) { return (grid.pitch + kStripW - 1) / kStripW; }

hipError_t launch_project_plan(const BpView* views, int n_views, const BpGrid& grid, int orbit, uint32_t* offs,
                               uint32_t* list, bool write, hipStream_t s) {
  const long nblocks = (long)project_strips(grid) * n_views;
  if (nblocks <= 0) return hipSuccess;
  if (nblocks > (long)max_blocks(64) || grid.nx > 65536 || grid.ny > 65536) return hipErrorInvalidValue;
  BpGrid g = grid;  // the first quadrant or half
  if (orbit == 4) g.x1 = (g.nx + 1) / 2;
  if (orbit > 1) g.ny = (g.ny + 1) / 2;
  if (write)
    hipLaunchKernelGGL(project_plan_kernel<true>, dim3((unsigned)nblocks), dim3(64), 0, s, views,
                       project_strips(grid), g, offs, list, orbit, grid.ny);
  else
    hipLaunchKernelGGL(project_plan_kernel<false>, dim3((unsigned)nblocks), dim3(64), 0, s, views,
                       project_strips(grid), g, offs, list, orbit, grid.ny);
  return hipGetLastError();
}

// ------------------------------------------------ projector by rows
// The matched projector as a gather over detector rows, without read-add-writes:
// a wave owns one detector column (strip) of a view, its lanes the rows, and walks
// the strip's voxel columns.  Row r takes the voxels whose v coordinate lies
// within a row of it, with the bilinear tent max(0, 1 - |sv - r|): sv(z) = A + z D,
// so they are the J consecutive voxels from z0 = floor((r - 1 - A) / D) + 1, J =
// ceil(2 / D), at s0 = sv(z0) - r, s0 + D, ...  The sum is added to the lane's two
// registers per row, for the column itself and for the one to its right.
//   (r - 1 - A) / D is formed in 32.32 fixed point from the row's integer offset, and z0 is its
// high word; s0 = A + z0 D - r in 32.32 as well, as the projector by voxels forms it, and the
// tent of its upper 28 fraction bits in integers, to half an ulp of FP32.  (In FP32 from the
// low word of the first, weights were 2.7e-8 to 4.7e-8 rms off, for 1.1e-8 to 1.8e-8 by voxels.)
// A column's voxels come from memory straight into the wave's LDS, `depth` - 1
// columns ahead, between zeros that the rows past its ends read.
//   NQ > 1: as the backprojector, the NQ columns of an orbit share all of a row's
// geometry; the wave forms the strip in all NQ views that are a part of a turn
// apart, taking the lists of first columns of each in turn.
// Per row and column: (7 + 7 J / 2) / NQ VALU instructions of geometry, 2 J - 1 of sums and 2
// multiply-adds, J reads of LDS.  The kernel this one replaces in these cases (below:
// lanes own voxels, two read-add-writes of LDS per voxel) took 9.97 ms at 325^3 ->
// 360 views of 512^2.
constexpr int kRowPad = 4;  // zeros before and after a column in LDS (>= J)
constexpr float kTentUnit = 268435456.0f;  // 2^28: a whole row in the tents' fixed point

__device__ inline int mad_i24(int a, int b, int c) {  // a b + c of 24-bit a and b (uniform)
  int r;
  asm("v_mad_i32_i24 %0, %1, %2, %3" : "=v"(r) : "v"(a), "s"(b), "v"(c));
  return r;
}

__device__ inline int median0(int a, int b) {  // of a, b and 0
  int r;
  asm("v_med3_i32 %0, %1, %2, 0" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

__device__ inline void wait_copies(int n) {  // until at most n copies to LDS are in flight
#define MONTE_WAIT(N) asm volatile("s_waitcnt vmcnt(" #N ")" ::: "memory")
  if (n >= 48) MONTE_WAIT(48);
  else if (n >= 32) MONTE_WAIT(32);
  else if (n >= 24) MONTE_WAIT(24);
  else if (n >= 18) MONTE_WAIT(18);
  else if (n >= 12) MONTE_WAIT(12);
  else if (n >= 8) MONTE_WAIT(8);
  else if (n >= 6) MONTE_WAIT(6);
  else if (n >= 4) MONTE_WAIT(4);
  else if (n >= 3) MONTE_WAIT(3);
  else if (n >= 2) MONTE_WAIT(2);
  else if (n >= 1) MONTE_WAIT(1);
  else MONTE_WAIT(0);
#undef MONTE_WAIT
}

template <int NQ, int J, int NR>
__global__ __launch_bounds__(64) void project_rows_kernel(const float* __restrict__ volT,
                                                          const BpView* __restrict__ views, int view0, int n_strips,
                                                          int nviews, BpGrid g, float* __restrict__ filt, int row0,
                                                          int row_end, int row_chunks, int depth,
                                                          const uint32_t* __restrict__ offs,
                                                          const uint32_t* __restrict__ list, int turn) {
  extern __shared__ float cols[];  // [depth][NQ][kRowPad + nz + kRowPad]
  // XCD x takes the views [x V / 8, (x + 1) V / 8) of the launch in groups of
  // kProjViewGroup, strip by strip within a group (see project_kernel)
  const int per_view = n_strips * row_chunks;
  const int xcd = (int)(blockIdx.x % 8u), jx = (int)(blockIdx.x / 8u);
  const int va = xcd * nviews / 8, vx = (xcd + 1) * nviews / 8 - va;
  if (jx >= vx * per_view) return;  // (the whole one-wave block)
  const int grp = jx / (kProjViewGroup * per_view), rem = jx - grp * kProjViewGroup * per_view;
  const int gsize = min(kProjViewGroup, vx - grp * kProjViewGroup);
  const int sr = rem / gsize, st = sr / row_chunks;
  const int k = view0 + va + grp * kProjViewGroup + (rem - sr * gsize);
  const int u = st * kStripW - kPadLo;  // the strip's detector column
  if (u >= g.nu) return;
  const int lane = threadIdx.x;
  const int rbase = row0 + (sr - st * row_chunks) * 64 * NR;  // detector row of lane 0
  const int part = g.n_views / NQ;
  const int slot_words = kRowPad + g.nz + kRowPad;
  for (int i = lane; i < depth * NQ * slot_words; i += 64) cols[i] = 0.f;
  __builtin_amdgcn_wave_barrier();
  const int chunks = (g.nz + 63) / 64, per_column = NQ * chunks;

  float accl[NQ][NR], accr[NQ][NR];
  // careful: voxels that a row's tent leaves out are not multiplied
  auto walk = [&](auto careful) {
#pragma unroll
    for (int q = 0; q < NQ; ++q)
#pragma unroll
      for (int p = 0; p < NR; ++p) accl[q][p] = accr[q][p] = 0.f;

    for (int a = 0; a < NQ; ++a) {
      const int ka = k + a * part;
      const BpView& c = views[ka];
      const size_t cell = (size_t)ka * n_strips + st;
      const uint32_t beg = offs[cell], end = offs[cell + 1];
      for (uint32_t b0 = beg; b0 < end; b0 += 64) {
        const int ncols = (int)min(64u, end - b0);
        // lane i prepares the i-th column: its weights and its line in fixed point
        int cx = 0, cy = 0;
        float wl = 0.f, wr = 0.f;
        long long q0 = 0, s1 = 0;
        uint32_t inv = 0;
        int dl = 0, dh = 0;  // D's fraction and whole part
        int first = 0, last = -1;  // rows (from rbase) it reaches
        if (lane < ncols) {
          const uint32_t e = list[b0 + lane];
          cx = (int)(e & 0xffffu);
          cy = (int)(e >> 16);
          const double X = voxel_x(g, cx), Y = voxel_y(g, cy);
          const ColumnCore mine = column_core<true>(c, X, Y, (float)X, (float)Y, g);
          // the centre of an odd volume is an orbit of one, taken NQ times
          const float w = NQ > 1 && 2 * cx + 1 == g.nx && 2 * cy + 1 == g.ny ? mine.w / NQ : mine.w;
          wr = w * mine.fu;
          wl = w - wr;
          if (!careful) {  // the tents' scale
            wr *= 1.0f / kTentUnit;
            wl *= 1.0f / kTentUnit;
          }
          const double A = fma(mine.kv, g.gz0, c.sv0) - (double)rbase, D = mine.kv * g.gsz, iD = recip64(D);
          const long long df = __double2ll_rn(D * 4294967296.0);
          dl = (int)(uint32_t)df;
          dh = (int)((df - dl) >> 32);
          s1 = __double2ll_rn((fmin(fmax(A, -1.0e6), 1.0e6) + 1.0) * 4294967296.0);
          const double q = fmin(fmax((-1.0 - A) * iD, -1.0e8), 1.0e8);
          q0 = __double2ll_rn(q * 4294967296.0);
          inv = (uint32_t)__double2ll_rn(fmin(iD * 2147483648.0, 4294967295.0));
          first = (int)floor(fmin(fmax(A - 1.0, -1.0e6), 1.0e6));
          last = (int)ceil(fmin(fmax(fma((double)(g.nz - 1), D, A) + 1.0, -1.0e6), 1.0e6));
        }
        auto fetch = [&](int i, int slot) {
          const int x = bcast_i(cx, i), y = bcast_i(cy, i);
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slot's last reads are done
#pragma unroll
          for (int q = 0; q < NQ; ++q) {
            const int m = NQ == 2 ? 2 * q : (turn > 0 ? q : (4 - q) & 3);  // quarter turns (x, y) -> (n - 1 - y, x)
            const int xq = m == 0 ? x : (m == 1 ? g.nx - 1 - y : (m == 2 ? g.nx - 1 - x : y));
            const int yq = m == 0 ? y : (m == 1 ? x : (m == 2 ? g.ny - 1 - y : g.nx - 1 - x));
            const char* col = (const char*)(volT + ((size_t)yq * g.nx + xq) * g.nz);
            float* dst = cols + (slot * NQ + q) * slot_words + kRowPad;
            for (int ch = 0; ch < chunks; ++ch)
              if (ch * 64 + lane < g.nz) copy_to_lds(col + ch * 256, (uint32_t)lane * 4u, dst + ch * 64);
          }
        };
        const int ahead = min(depth - 1, ncols);
        for (int i = 0; i < ahead; ++i) fetch(i, i);
        int slot = 0, fslot = ahead;
        for (int i = 0; i < ncols; ++i) {
          if (i + ahead < ncols) fetch(i + ahead, fslot);
          if (++fslot == depth) fslot = 0;
          wait_copies(min(ahead, ncols - 1 - i) * per_column);
          const float wli = bcast_f(wl, i), wri = bcast_f(wr, i);
          const long long q0i = bcast_ll(q0, i), s1i = bcast_ll(s1, i);
          const int dli = bcast_i(dl, i), dhi = bcast_i(dh, i), step = dhi * (int)kTentUnit + (dli >> 4);
          const uint32_t invi = (uint32_t)bcast_i((int)inv, i);
          const int fi = bcast_i(first, i), la = bcast_i(last, i);
          const float* col = cols + slot * NQ * slot_words + kRowPad;
#pragma unroll
          for (int p = 0; p < NR; ++p) {
            if (fi > 64 * p + 63 || la < 64 * p) continue;  // (uniform)
            const uint64_t q = (uint64_t)invi * (uint32_t)(2 * lane + 128 * p) + (uint64_t)q0i;
            const int z = clamp_i((int)(uint32_t)(q >> 32) + 1, -kRowPad, g.nz);
            // sv(z) - r + 1, of which a tent's weight is the distance from the nearer of 0 and 2
            const uint64_t f = (uint64_t)((long long)z * dli + s1i);
            const int row = mad_i24(z, dhi, (int)(uint32_t)(f >> 32) - lane) - 64 * p;
            const uint32_t at = __builtin_amdgcn_alignbit((uint32_t)row, (uint32_t)f, 4);
            float t[J];
#pragma unroll
            for (int j = 0; j < J; ++j) {
              const uint32_t a = at + (uint32_t)(j * step);
              t[j] = (float)median0((int)a, (int)((uint32_t)(2 * kTentUnit) - a)) * (careful ? 1.0f / kTentUnit : 1.0f);
            }
#pragma unroll
            for (int qq = 0; qq < NQ; ++qq) {
              const float* v = col + qq * slot_words + z;
              auto value = [&](int j) { return careful && t[j] == 0.f ? 0.f : v[j]; };
              float sum = t[0] * value(0);
#pragma unroll
              for (int j = 1; j < J; ++j) sum = fmaf(t[j], value(j), sum);
              accl[qq][p] = fmaf(wli, sum, accl[qq][p]);
              accr[qq][p] = fmaf(wri, sum, accr[qq][p]);
            }
          }
          if (++slot == depth) slot = 0;
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // before the next batch's copies
      }
      // column q of the next list belongs to the view of this list's column q + 1
      if (NQ > 1) {
#pragma unroll
        for (int p = 0; p < NR; ++p) {
          const float l0 = accl[0][p], r0 = accr[0][p];
#pragma unroll
          for (int q = 0; q + 1 < NQ; ++q) {
            accl[q][p] = accl[q + 1][p];
            accr[q][p] = accr[q + 1][p];
          }
          accl[NQ - 1][p] = l0;
          accr[NQ - 1][p] = r0;
        }
      }
    }
  };
  walk(std::false_type{});
  // A voxel that is not finite reaches the rows it projects to, and no others: 0 times it is
  // not 0.  Such strips are walked again.
  bool finite = true;
#pragma unroll
  for (int q = 0; q < NQ; ++q)
#pragma unroll
    for (int p = 0; p < NR; ++p) finite = finite && fabsf(accl[q][p]) + fabsf(accr[q][p]) < INFINITY;
  if (__any(!finite)) walk(std::true_type{});
  // Two strips meet in a detector column: two addends onto zero, the same in
  // either order.  Guard cells are not used (standard preset).
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    float* out = filt + (size_t)(k + q * part) * g.rows * g.pitch;
#pragma unroll
    for (int p = 0; p < NR; ++p) {
      const int r = rbase + 64 * p + lane;
      if (r < 0 || r >= min(g.nv, row_end)) continue;
      float* o = out + (size_t)(r + kPadLo) * g.pitch + u + kPadLo;
      if (u >= 0 && accl[q][p] != 0.f) unsafeAtomicAdd(o, accl[q][p]);
      if (u + 1 < g.nu && accr[q][p] != 0.f) unsafeAtomicAdd(o + 1, accr[q][p]);
    }
  }
}

// The row kernel's orbit (4, 2 or 1 views that a wave forms together), or 0 for the
// voxel kernel above.  The rule takes the standard preset's zero guard cells and the
// automatic tuning, and these sizes (adjoint with its filter, ms, by rows : by
// voxels):
//  - between 0.8 and 1.9 rows a voxel.  Below, a row takes more than three voxels (0.090
//    against 0.085 at 65^3, 1.10 : 1.09 at 193^3, from 0.65 rows a voxel), above most rows
//    of a column see one voxel (0.50 : 0.39 at 97^3, up to 2.3 rows a voxel).  Launches of up
//    to 5000 waves wait for a wave's chain of read-add-writes by voxels, and gain up to 2.6
//    rows a voxel (0.046 : 0.055 at 33^3 / 30 views, 0.072 : 0.078 at 49^3 / 36 views, 2.5 rows).
//  - a column within 384 rows: more take a second wave that reads all columns again
//    (4.5 : 3.1 at 225^3, 434 rows).
//  - a volume of up to 48 MB.  Larger ones leave no columns for the next view in the
//    L2s: a launch reads the volume once per view, at 5.2 TB/s (325^3 / 360 views of 512^2, the
//    projection alone, without the second wave: 11.5 : 9.97, since the voxel kernel keeps columns).
// Within them: 0.051 : 0.072 at 49^3 (36 views of 64^2), 0.128 : 0.176 at 65^3 (90 of
// 96^2), 0.29 : 0.34 at 97^3 (90 of 160^2), 0.82 : 1.00 at 129^3 (180 of 192^2), 1.24 :
// 1.52 at 161^3 (180 of 256^2), 2.79 : 2.99 at 225^3 (180 of 384^2).
//   Orbits save geometry and take waves: of 4 from 10000 waves (in FP32 weights 2.75 : 3.10 with
// 2 at 17000, 0.72 : 0.68 at 7200), of 2 from 3000 (0.117 : 0.131 with 1 at 4300, 0.054 : 0.050
// at 1150).
int project_orbit(const BpGrid& g, const BpReach& r, const monte_tuning& t) {
  const double lo = r.svk * std::fabs(g.gsz) / (r.sod + r.rad), hi = r.svk * std::fabs(g.gsz) / (r.sod - r.rad);
  if (t.pj_zchunk != 0 || !r.zeros || g.gsz <= 0 || !(lo > 0.8) || !(hi * g.nz <= 384.0)) return 0;
  if ((double)g.nx * g.ny * g.nz > 12e6) return 0;
  const long waves = (long)g.n_views * project_strips(g);
  if (!(hi < (waves <= 5000 ? 2.6 : 1.9))) return 0;
  if (t.bp_view_chunk > 0 && t.bp_view_chunk < g.n_views) return 1;  // orbits need the whole turn
  return r.turn != 0 && waves >= 40000 ? 4 : (r.half && waves >= 6000 ? 2 : 1);
}

// Detector rows of a launch by rows, as blocks of 64 x nr rows, and the voxels a row takes of a column.
struct RowLaunch {
  int row0, row_end, chunks, nr, J;
};
static bool row_launch(const BpGrid& grid, const BpReach& reach, int lds_r0, int lds_rows, RowLaunch& L) {
  // detector rows that the window of padded rows holds
  L.row0 = std::max(lds_r0 - kPadLo, 0);
  L.row_end = std::min(lds_r0 - kPadLo + lds_rows, grid.nv);
  // a block fetches and sets up its columns once for all its rows: few chunks
  const int rows64 = std::max(0, (L.row_end - L.row0 + 63) / 64);
  L.chunks = (rows64 + 5) / 6;
  L.nr = L.chunks ? (rows64 + L.chunks - 1) / L.chunks : 0;
  const double lo = reach.svk * std::fabs(grid.gsz) / (reach.sod + reach.rad);
  L.J = lo >= 1.0 ? 2 : 3;
  return lo >= 2.0 / 3.0;  // (project_orbit)
}

void fdk_routes(const BpGrid& grid, const BpReach& reach, int nviews_chunk, int lds_r0, int lds_rows,
                const monte_tuning& t, int32_t out[kRouteWords]) {
  std::fill(out, out + kRouteWords, 0);
  BpLaunch B;
  out[0] = -1;
  if (bp_launch(grid, reach, nviews_chunk, t, B)) {
    const int32_t b[8] = {B.plan.orbit, B.plan.groups, B.zc, B.plan.stack, B.tile_x, B.rows, B.cols, (int32_t)B.blocks};
    std::copy(b, b + 8, out);
  }
  RowLaunch L;
  out[8] = project_orbit(grid, reach, t);
  if (out[8] && row_launch(grid, reach, lds_r0, lds_rows, L)) {
    out[9] = L.chunks;
    out[10] = L.nr;
    out[11] = L.J;
  }
}

hipError_t launch_project_rows(const float* volT, const BpView* views, int view0, int nviews_chunk, const BpGrid& grid,
                               const BpReach& reach, int orbit, float* filt_pad, int lds_r0, int lds_rows,
                               const uint32_t* plan_offs, const uint32_t* plan_list, hipStream_t s) {
  if (nviews_chunk <= 0) return hipSuccess;
  if (orbit != 1 && nviews_chunk != grid.n_views) return hipErrorInvalidValue;
  RowLaunch L;
  if (!row_launch(grid, reach, lds_r0, lds_rows, L)) return hipErrorInvalidValue;
  if (L.row_end <= L.row0) return hipSuccess;
  const int base_views = nviews_chunk / orbit, n_strips = project_strips(grid), chunks = L.chunks, J = L.J;
  const size_t slot = sizeof(float) * orbit * (2 * kRowPad + grid.nz);
  const int depth = (int)std::min<size_t>(6, std::max<size_t>(2, 12 * 1024 / slot));
  const long nblocks = (long)n_strips * chunks * 8 * ((base_views + 7) / 8);
  if (nblocks > (long)max_blocks(64)) return hipErrorInvalidValue;
#define MONTE_PR(NQ, JJ, RR)                                                                                   \
  hipLaunchKernelGGL((project_rows_kernel<NQ, JJ, RR>), dim3((unsigned)nblocks), dim3(64), slot * depth, s,    \
                     volT, views, view0, n_strips, base_views, grid, filt_pad, L.row0, L.row_end, chunks, depth, \
                     plan_offs, plan_list, reach.turn)
#define MONTE_PR_R(NQ, JJ)                                                                                     \
  switch (L.nr) {                                                                                              \
    case 1: MONTE_PR(NQ, JJ, 1); break;                                                                        \
    case 2: MONTE_PR(NQ, JJ, 2); break;                                                                        \
    case 3: MONTE_PR(NQ, JJ, 3); break;                                                                        \
    case 4: MONTE_PR(NQ, JJ, 4); break;                                                                        \
    case 5: MONTE_PR(NQ, JJ, 5); break;                                                                        \
    default: MONTE_PR(NQ, JJ, 6); break;                                                                       \
  }
#define MONTE_PR_J(NQ)                                                                                         \
  if (J == 2) { MONTE_PR_R(NQ, 2) } else { MONTE_PR_R(NQ, 3) }
  if (orbit == 4) { MONTE_PR_J(4) } else if (orbit == 2) { MONTE_PR_J(2) } else { MONTE_PR_J(1) }
#undef MONTE_PR_J
#undef MONTE_PR_R
#undef MONTE_PR
  return hipGetLastError();
}

hipError_t launch_project(const float* volT, const BpView* views, int view0, int nviews_chunk, const BpGrid& grid,
                          float* filt_pad, int lds_r0, int lds_rows, const uint32_t* plan_offs,
                          const uint32_t* plan_list, const monte_tuning& t, hipStream_t s) {
  const int n_strips = project_strips(grid);
  // (8 XCDs x the largest view share x strips; blocks past an XCD's share return)
  const long nblocks = (long)n_strips * 8 * ((nviews_chunk + 7) / 8);
  if (nblocks <= 0) return hipSuccess;
  if (nblocks > (long)max_blocks(64)) return hipErrorInvalidValue;
  if (lds_r0 < 0 || lds_rows < 1 || lds_r0 + lds_rows > grid.rows) return hipErrorInvalidValue;
  const size_t lds = sizeof(float) * ((size_t)lds_rows * kStripP + kTrash);
  if (lds > 64 * 1024) return hipErrorInvalidValue;
  // voxels per lane: 2 unless tuned otherwise.  Two voxels per lane need the
  // fewest dependent LDS read-add-writes per pass: 2 and 4 voxels per lane
  // took 10.6 and 13.8 ms at 325^3 / 512^2 / 360 views, 86 and 96 ms at
  // 512^3 / 1024 x 768 / 720 views (and 8 voxels per lane 163 ms).
  const int best = t.pj_zchunk ? t.pj_zchunk : 2;
  const dim3 gd((unsigned)nblocks), bd(64);
#define MONTE_PJ(CZ, MK)                                                                                      \
  hipLaunchKernelGGL((project_kernel<CZ, MK>), gd, bd, lds, s, volT, views, view0, n_strips, nviews_chunk, grid,   \
                     filt_pad,                                                                                  \
                     lds_r0, lds_rows, plan_offs, plan_list)
  const bool mk = grid.mask != 0;
  switch (best) {
    case 2: if (mk) MONTE_PJ(2, true); else MONTE_PJ(2, false); break;
    case 4: if (mk) MONTE_PJ(4, true); else MONTE_PJ(4, false); break;
    case 8: if (mk) MONTE_PJ(8, true); else MONTE_PJ(8, false); break;
    default: return hipErrorInvalidValue;
  }
#undef MONTE_PJ
  return hipGetLastError();
}

}  // namespace monte
