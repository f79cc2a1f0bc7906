// p0k_stats.hip — the statistics the convolution prologues read: PixelNorm scales (conv3 `pn`) and GroupNorm(32)
// affine coefficients (conv `gn`). Both are HBM-bound reductions over HWC / THWC fp16 activations.
//
//  pixstats  (src/ops/video.js:301-321): R[ro + v] = 1 / sqrt(sum_c x[v][c]^2 / C + eps), one value per voxel.
//            A group of 16 lanes owns one voxel and reads its C channels as 16-byte chunks, so a wave reads four whole
//            voxels per step; the 16 partial sums meet through shuffles.
//  GroupNorm (src/ops/misc.js:50-109): exact two-pass statistics per chunk of 64 pixels, written as partial rows
//            [chunk][group] = (n, mean, M2, 0) (the reference's layout, so partials of several calls - bands of one
//            tensor - merge), then Chan's parallel formula merges the rows: a[c] = gamma[c] / sqrt(M2 / n + eps),
//            b[c] = beta[c] - mean * a[c], so GN(x) = a x + b. The merge runs one workgroup per group; each thread
//            merges a strided subset of rows in order and the 256 partial states meet in a fixed tree, so the result
//            does not depend on timing.
#include "p0k_device.h"
#include "p0k_launch.h"

#include <type_traits>

namespace p0k {

// ------------------------------------------------------------------------------------------------------------ pixstats
__global__ __launch_bounds__(256) void k_pixstats(const uint8_t *x, uint32_t V, uint32_t C, float eps, float *r) {
  const uint32_t g = threadIdx.x & 15;
  const uint32_t v = (blockIdx.x * 256u + threadIdx.x) >> 4;
  const bool live = v < V;
  const uint16_t *row = (const uint16_t *)x + (size_t)(live ? v : 0u) * C;
  float s = 0.0f;
  if (live) {
    const uint32_t c8 = C / 8;
    if ((((uintptr_t)row) & 15u) == 0) {
      for (uint32_t i = g; i < c8; i += 16) {
        const u32x4 w = ((const u32x4 *)row)[i];
        const f16x2 a = as_h2(w.x), b = as_h2(w.y), c = as_h2(w.z), d = as_h2(w.w);
        s += ((float)a.x * (float)a.x + (float)a.y * (float)a.y) + ((float)b.x * (float)b.x + (float)b.y * (float)b.y) +
             ((float)c.x * (float)c.x + (float)c.y * (float)c.y) + ((float)d.x * (float)d.x + (float)d.y * (float)d.y);
      }
      for (uint32_t c = c8 * 8 + g; c < C; c += 16) { const float t = h_val(row[c]); s += t * t; }
    } else {
      for (uint32_t c = g; c < C; c += 16) { const float t = h_val(row[c]); s += t * t; }
    }
  }
  s = sum16(s);
  if (live && g == 0) r[v] = __frsqrt_rn(s / (float)C + eps);
}

hipError_t launch_pixstats(const void *x, uint32_t V, uint32_t C, float eps, float *r, hipStream_t s) {
  if (V == 0) return hipSuccess;
  const uint32_t blocks = (V + 15) / 16;
  hipLaunchKernelGGL(k_pixstats, dim3(blocks), dim3(256), 0, s, (const uint8_t *)x, V, C, eps, r);
  return hipGetLastError();
}

// ------------------------------------------------------------------------------------------------------------ GroupNorm
constexpr uint32_t GN_PIX = 64;   // pixels per partial row (the reference's chunk, so partial buffers interoperate)

// One workgroup per chunk of 64 pixels, its whole chunk in registers: thread t holds the 16-byte pieces t, t + 256, ...
// (8 channels each; C / 32 of them), and since C divides 2048 halves they all cover the same 8 channels, i.e. 8 / cpg
// whole groups (cpg = C / 32 channels each) or, at C = 512, half of one. Both passes (sums, then squared deviations
// from the group mean) run from the registers, so the chunk is read once with every load in flight; lanes that hold
// the same channels meet by shuffles, the four waves in LDS. HBM-latency-bound: 16384 pixels x 256 channels (8.4 MB)
// went from 117.6 us (2-byte loads, one in flight per thread, and 512-term serial group sums) to under 5: GroupNorm +
// 3x3 convolution of that image 220.8 -> 106.8 us.
// AL: x is 16-byte aligned (pieces are one load each), else eight 2-byte loads.
template <uint32_t C, bool AL>
__global__ __launch_bounds__(256) void k_gn_partial(const uint16_t *x, uint32_t pix, f32x4 *part, uint32_t wg_off) {
  constexpr uint32_t CPG = C / 32, NP = C / 32, SLOTS = C / 8;   // channels per group, pieces per thread, piece columns
  constexpr uint32_t G = CPG >= 8 ? 1 : 8 / CPG, PER = 8 / G;    // groups in a piece, channels of each
  __shared__ float red[2][4][32];
  const uint32_t t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const uint32_t px0 = blockIdx.x * GN_PIX, npx = pix - px0 < GN_PIX ? pix - px0 : GN_PIX;
  const uint16_t *base = x + (size_t)px0 * C;
  const uint32_t n8 = npx * (C / 8);                             // pieces of this chunk
  u32x4 v[NP];
#pragma unroll
  for (uint32_t i = 0; i < NP; i++) {
    const uint32_t e = t + 256 * i;
    v[i] = (u32x4){0u, 0u, 0u, 0u};
    if (e < n8) {
      if constexpr (AL) {
        v[i] = *(const u32x4 *)(base + (size_t)e * 8);
      } else {
#pragma unroll
        for (int j = 0; j < 4; j++) v[i][j] = base[(size_t)e * 8 + 2 * j] | ((uint32_t)base[(size_t)e * 8 + 2 * j + 1] << 16);
      }
    }
  }
  const uint32_t g0 = (t % SLOTS) * 8 / CPG;                     // the piece's first group
  // s[q]: this thread's sum for group g0 + q -> the chunk's, in every thread
  auto meet = [&](float *s, int pass) {
#pragma unroll
    for (uint32_t q = 0; q < G; q++) {
      if (CPG == 16) s[q] += __shfl_xor(s[q], 1, 64);            // the group's other half is in the next piece
#pragma unroll
      for (uint32_t o = SLOTS; o < 64; o <<= 1) s[q] += __shfl_xor(s[q], o, 64);
      if (lane < SLOTS) red[pass][wave][g0 + q] = s[q];
    }
    __syncthreads();
#pragma unroll
    for (uint32_t q = 0; q < G; q++)
      s[q] = (red[pass][0][g0 + q] + red[pass][1][g0 + q]) + (red[pass][2][g0 + q] + red[pass][3][g0 + q]);
  };
  const float cnt = (float)(npx * CPG);
  float s[G] = {}, mean[G];
#pragma unroll
  for (uint32_t i = 0; i < NP; i++)
#pragma unroll
    for (uint32_t j = 0; j < 8; j++) s[j / PER] += h_val((uint16_t)(v[i][j >> 1] >> (16 * (j & 1))));
  meet(s, 0);
#pragma unroll
  for (uint32_t q = 0; q < G; q++) {
    mean[q] = s[q] / cnt;
    s[q] = 0.0f;
  }
#pragma unroll
  for (uint32_t i = 0; i < NP; i++)
    if (t + 256 * i < n8) {
#pragma unroll
      for (uint32_t j = 0; j < 8; j++) {
        const float d = h_val((uint16_t)(v[i][j >> 1] >> (16 * (j & 1)))) - mean[j / PER];
        s[j / PER] += d * d;
      }
    }
  meet(s, 1);
  if (t < SLOTS) {                                               // (C = 512: two threads write the same row)
#pragma unroll
    for (uint32_t q = 0; q < G; q++)
      part[(size_t)(wg_off + blockIdx.x) * 32 + g0 + q] = (f32x4){cnt, mean[q], s[q], 0.0f};
  }
}

struct GnState { float n, mean, m2; };
__device__ __forceinline__ GnState gn_merge(GnState a, GnState b) {
  if (b.n <= 0.0f) return a;
  if (a.n <= 0.0f) return b;
  const float nn = a.n + b.n, d = b.mean - a.mean;
  return GnState{nn, a.mean + d * (b.n / nn), a.m2 + b.m2 + d * d * (a.n * b.n / nn)};
}

// One workgroup per group: merge the partial rows, then write the affine coefficients of the group's channels.
__global__ __launch_bounds__(256) void k_gn_finalize(const f32x4 *part, uint32_t nwg, uint32_t C, float eps,
                                                     const float *gamma, const float *beta, float *ab) {
  __shared__ float sn[256], sm[256], sq[256];
  const uint32_t g = blockIdx.x, t = threadIdx.x;
  GnState st{0.0f, 0.0f, 0.0f};
  for (uint32_t w = t; w < nwg; w += 256) {
    const f32x4 q = part[(size_t)w * 32 + g];
    st = gn_merge(st, GnState{q.x, q.y, q.z});
  }
  sn[t] = st.n; sm[t] = st.mean; sq[t] = st.m2;
  __syncthreads();
  for (uint32_t h = 128; h > 0; h >>= 1) {
    if (t < h) {
      const GnState m = gn_merge(GnState{sn[t], sm[t], sq[t]}, GnState{sn[t + h], sm[t + h], sq[t + h]});
      sn[t] = m.n; sm[t] = m.mean; sq[t] = m.m2;
    }
    __syncthreads();
  }
  const float rs = __frsqrt_rn(sq[0] / fmaxf(sn[0], 1.0f) + eps), mean = sm[0];
  const uint32_t cpg = C / 32;
  for (uint32_t c = g * cpg + t; c < (g + 1) * cpg; c += 256) {
    const float a = gamma[c] * rs;
    ab[c] = a;
    ab[C + c] = beta[c] - mean * a;
  }
}

hipError_t launch_gn_partial(const void *x, uint32_t pix, uint32_t C, float *part, uint32_t wg_off, hipStream_t s) {
  if (pix == 0) return hipSuccess;
  const dim3 grid((pix + GN_PIX - 1) / GN_PIX);
  const bool al = ((uintptr_t)x & 15u) == 0;
  auto go = [&](auto c) {
    constexpr uint32_t CC = decltype(c)::value;
    if (al) hipLaunchKernelGGL((k_gn_partial<CC, true>), grid, dim3(256), 0, s, (const uint16_t *)x, pix, (f32x4 *)part, wg_off);
    else hipLaunchKernelGGL((k_gn_partial<CC, false>), grid, dim3(256), 0, s, (const uint16_t *)x, pix, (f32x4 *)part, wg_off);
    return hipGetLastError();
  };
  switch (C) {
  case 32: return go(std::integral_constant<uint32_t, 32>{});
  case 64: return go(std::integral_constant<uint32_t, 64>{});
  case 128: return go(std::integral_constant<uint32_t, 128>{});
  case 256: return go(std::integral_constant<uint32_t, 256>{});
  case 512: return go(std::integral_constant<uint32_t, 512>{});
  }
  return hipErrorInvalidValue;
}

hipError_t launch_gn_finalize(const float *part, uint32_t nwg, uint32_t C, float eps, const float *gamma,
                              const float *beta, float *ab, hipStream_t s) {
  hipLaunchKernelGGL(k_gn_finalize, dim3(32), dim3(256), 0, s, (const f32x4 *)part, nwg, C, eps, gamma, beta, ab);
  return hipGetLastError();
}

}  // namespace p0k
