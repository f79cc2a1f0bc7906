// p0k_gemm_dma.hip — the host side of the load-to-LDS GEMM (p0k_gemm_dma.h): which calls qualify, the tile and the split
// of a call, and the passes that materialise X' once per element.
#include "p0k_gemm_dma.h"
#include "p0k_internal.h"

namespace p0k {

hipError_t launch_dma_q4(const Params &p, int xg, unsigned bm, unsigned bn, unsigned wv, hipStream_t s);
hipError_t launch_dma_q8(const Params &p, int xg, unsigned bm, unsigned bn, unsigned wv, hipStream_t s);
hipError_t launch_dma_f16(const Params &p, int xg, unsigned bm, unsigned bn, unsigned wv, hipStream_t s);

namespace {

// conv3 PixelNorm + SiLU, materialised once per input element (the fused prologue's exact fp16 values, xload8)
__global__ __launch_bounds__(256) void k_pnprep(Params p, uint16_t *xp) {
  const uint32_t c8 = p.Ci / 8;
  const uint64_t n = (uint64_t)p.nvox * c8;
  for (uint64_t t = (uint64_t)blockIdx.x * 256 + threadIdx.x; t < n; t += (uint64_t)gridDim.x * 256) {
    const uint64_t vox = t / c8;
    const uint32_t c0 = (uint32_t)(t - vox * c8) * 8;
    u32x4 v = *(const u32x4 *)(p.X + (vox * p.Ci + c0) * 2);
    const float sc = p.ST[vox];
    const f16x2 a = as_h2(v.x), b = as_h2(v.y), c = as_h2(v.z), d = as_h2(v.w);
    v = (u32x4){pack2(silu((float)a.x * sc), silu((float)a.y * sc)), pack2(silu((float)b.x * sc), silu((float)b.y * sc)),
                pack2(silu((float)c.x * sc), silu((float)c.y * sc)), pack2(silu((float)d.x * sc), silu((float)d.y * sc))};
    *(u32x4 *)(xp + vox * p.Ci + c0) = v;
  }
}

// 2-D convolution: GroupNorm-apply + SiLU, materialised once per input element (the fused prologue's exact fp16 values).
// The fused form recomputes them for each of the 9 taps and each column tile, and stages through registers: GroupNorm +
// 3x3 convolution 128 x 128 x 256 -> 256 106.8 us per pass, with this pass and the gather 55.0; 64 x 64 x 512 -> 512
// 183 -> 76, 256 x 256 x 128 -> 128 77 -> 50.
__global__ __launch_bounds__(256) void k_gnprep(Params p, uint16_t *xp) {
  const uint32_t c8 = p.Ci / 8;
  const uint64_t n = (uint64_t)p.nvox * c8;
  for (uint64_t t = (uint64_t)blockIdx.x * 256 + threadIdx.x; t < n; t += (uint64_t)gridDim.x * 256) {
    const uint64_t pix = t / c8;
    const uint32_t c0 = (uint32_t)(t - pix * c8) * 8;
    const u32x4 v = *(const u32x4 *)(p.X + (pix * p.Ci + c0) * 2);
    const f32x4 *a = (const f32x4 *)(p.PV + p.pvOff + c0), *b = (const f32x4 *)(p.PV + p.pvOff + p.pvStride + c0);
    const f32x4 a0 = a[0], a1 = a[1], b0 = b[0], b1 = b[1];
    const f16x2 h0 = as_h2(v.x), h1 = as_h2(v.y), h2 = as_h2(v.z), h3 = as_h2(v.w);
    *(u32x4 *)(xp + pix * p.Ci + c0) =
        (u32x4){pack2(silu((float)h0.x * a0.x + b0.x), silu((float)h0.y * a0.y + b0.y)),
                pack2(silu((float)h1.x * a0.z + b0.z), silu((float)h1.y * a0.w + b0.w)),
                pack2(silu((float)h2.x * a1.x + b1.x), silu((float)h2.y * a1.y + b1.y)),
                pack2(silu((float)h3.x * a1.z + b1.z), silu((float)h3.y * a1.w + b1.w))};
  }
}

// X' of the rms / lnmod prologues, materialised once: Xp[m][k] = xload8 (the fused prologue's exact values); one
// workgroup per row (and 2048 columns, with few rows), 8 k per thread and step
template <int XM>
__global__ __launch_bounds__(256) void k_xprep(Params p, uint16_t *xp) {
  const uint32_t k8 = p.K / 8, m = blockIdx.x;
  uint16_t *dst = xp + (size_t)m * p.K;
#pragma unroll 2
  for (uint32_t kq = blockIdx.y * 256 + threadIdx.x; kq < k8; kq += 256 * gridDim.y) *(u32x4 *)(dst + 8 * kq) = xload8<XM, 1>(p, m, RowCtx{0, 0, 0}, 8 * kq);
}

// The end of a call whose K was split: the slices' fp32 sums, added in slice order, and the epilogue. One workgroup per
// 16 rows x 128 columns; a thread's two 16-byte pieces of up to 4 slices are in flight together.
constexpr int SE_ROWS = 16;
__global__ __launch_bounds__(256) void k_split_epi(Params p) {
  __shared__ __attribute__((aligned(16))) float sC[SE_ROWS * 132];
  const uint32_t mB = blockIdx.x * SE_ROWS, nB = blockIdx.y * 128;
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const uint32_t r = (threadIdx.x >> 5) + 8 * i, c = (threadIdx.x & 31) * 4, m = mB + r < p.M ? mB + r : p.M - 1u;
    const float *src = p.part + (size_t)m * p.ldp + nB + c;
    const size_t step = (size_t)p.M * p.ldp;
    f32x4 sum = (f32x4){};
#pragma unroll 4
    for (uint32_t q = 0; q < p.slices; q++) sum += *(const f32x4 *)(src + q * step);
    *(f32x4 *)(sC + r * 132 + c) = sum;
  }
  __syncthreads();
  epilogue<256>(p, sC, 132, SE_ROWS, mB, nB, threadIdx.x);
}

}  // namespace

bool gemm_dma_ok(const Params &p, int we, int xm, uint64_t wbytes) {
  if (xm == X_CONV) {
    // 64-k steps inside one tap; first-tap coordinates in signed 16 bits
    const uint64_t rows = p.M ? ((uint64_t)p.M - 1) / p.Wo + 1 : 0;
    const uint64_t yspan = rows * p.stride + p.padT + p.ks, xspan = (uint64_t)p.Wo * p.stride + p.padL + p.ks;
    if (p.Ci % 64 != 0 || yspan > 32767 || xspan > 32767 || p.Hi > 16383 || p.Wi > 16383) return false;
  } else if (xm == X_CONV3) {
    // 64-k steps inside one tap; input frames of the three time taps packed in 10 bits; (oy, ox) in 16
    // f16 weights also with Ci 96, 160, ...: a tap per half step. us, register-staged kernel -> this one: 96 -> 128 channels
    // 3 x 41 x 123 58.2 -> 24.7 (with PixelNorm 102 -> 32.2), 13 x 92 x 160 216 -> 167 (385 -> 187); 160 -> 160
    // 13 x 92 x 160 515 -> 477 (757 -> 506). Ci 32 was not timed and stays on the register-staged kernel
    const bool half = we == W_F16 && p.Ci % 64 == 32 && p.Ci > 64;
    if ((p.Ci % 64 != 0 && !half) || p.stride > 1024 || p.ks > 1024 || p.Ho > 65535 || p.Wo > 65535 || p.nvox == 0xffffffffu)
      return false;
    if (half) return wbytes < (1ull << 32) && p.K != 0 && p.K % 32 == 0 && (p.flags & F_WALIGN8);
  } else {
    // 32-bit lane offsets from the X' base
    const uint64_t xbytes = xm == X_F16 ? ((uint64_t)p.M * p.ldx + p.kx0 + p.K) * 2 : (uint64_t)p.M * p.K * 2;
    if (xbytes >= (1ull << 32)) return false;
  }
  if (wbytes >= (1ull << 32)) return false;
  if (p.K % DBK != 0 || p.K == 0) return false;
  if (xm == X_F16 && !(p.flags & F_XALIGN8)) return false;
  if (we == W_F16 && !(p.flags & F_WALIGN8)) return false;
  if (we == W_Q4 && p.wk0 % 32 != 0) return false;
  if (we == W_Q8 && p.wk0 % 64 != 0) return false;
  return we == W_F16 || we == W_Q4 || we == W_Q8;
}

hipError_t launch_xprep(const Params &p, int xm, uint16_t *xp, hipStream_t s) {
  if (xm == X_CONV3 || xm == X_CONV) {
    const uint64_t n = (uint64_t)p.nvox * (p.Ci / 8);
    const unsigned blocks = (unsigned)(n / 256 < 4096 ? (n + 255) / 256 : 4096);
    if (n && xm == X_CONV3) hipLaunchKernelGGL(k_pnprep, dim3(blocks), dim3(256), 0, s, p, xp);
    else if (n) hipLaunchKernelGGL(k_gnprep, dim3(blocks), dim3(256), 0, s, p, xp);
    return hipGetLastError();
  }
  if (p.M == 0) return hipSuccess;
  // (few rows: a workgroup per 2048 columns, one trip to memory)
  const dim3 grid(p.M, p.M <= 512 ? (p.K + 2047) / 2048 : 1);
  if (xm == X_RMS) hipLaunchKernelGGL(k_xprep<X_RMS>, grid, dim3(256), 0, s, p, xp);
  else if (xm == X_LNMOD) hipLaunchKernelGGL(k_xprep<X_LNMOD>, grid, dim3(256), 0, s, p, xp);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

// The tile: each candidate scored by its relative per-CU rate times the fraction of workgroup slots (one or two per
// CU, as the tile's LDS allows) that hold real work over the rounds the grid needs.
// workgroups per CU of a tile for a grid of `tiles` (q4 256 x 128: 8 waves when the grid has one tile per CU at most)
unsigned dma_wgs(int we, unsigned m, unsigned n, uint64_t tiles, unsigned cus) {
  if (m == 256 && n == 256) return 1;
  if (m == 256 && (we != W_Q4 || tiles <= cus)) return 1;           // 8 waves
  if (m == 128 && n == 128 && we == W_Q4 && tiles <= cus) return 1;   // 8 waves
  if (we == W_F16) return m == 128 && n == 128 ? (DT<W_F16, 128, 128>::WGS) : (DT<W_F16, 128, 256>::WGS);
  if (we == W_Q4) return m == 128 && n == 128 ? DT<W_Q4, 128, 128>::WGS : (m == 128 ? DT<W_Q4, 128, 256>::WGS : DT<W_Q4, 256, 128>::WGS);
  return m == 128 && n == 128 ? DT<W_Q8, 128, 128>::WGS : (m == 128 ? DT<W_Q8, 128, 256>::WGS : DT<W_Q8, 256, 128>::WGS);
}

void dma_tile(uint32_t M, uint32_t N, int we, int xg, unsigned cus, unsigned *bm, unsigned *bn) {
  auto per_cu = [&](unsigned m, unsigned n) -> unsigned {
    return dma_wgs(we, m, n, (uint64_t)((M + m - 1) / m) * ((N + n - 1) / n), cus);
  };
  // relative per-CU rates measured on MI355X at 4096^3 (f16 prologue), per weight encoding: 256 x 256 and (f16, q8)
  // 256 x 128 run 8 waves (two per SIMD), the others 4; the quantised weights favour 256-row tiles (each decoded
  // weight feeds four 32-row blocks instead of two)
  struct C { unsigned m, n; double rate; };
  const C c16[] = {{256, 256, 1.0}, {128, 256, 0.94}, {256, 128, 0.99}, {128, 128, 0.91}};
  const C cq4[] = {{256, 256, 1.0}, {128, 256, 0.68}, {256, 128, 0.91}, {128, 128, 0.68}};
  const C cq8[] = {{256, 256, 1.0}, {128, 256, 0.75}, {256, 128, 0.84}, {128, 128, 0.78}};
  // the conv3 gather computes each row's tap address per step (f16 weights, 13 x 92 x 160 x 128 clip: 256 x 128 with
  // 8 waves 244 us, 128 x 128 (two workgroups per CU) 257, 256 x 256 382 and 128 x 256 409 with 4 waves)
  const C cg[] = {{256, 256, 0.66}, {128, 256, 0.62}, {256, 128, 1.05}, {128, 128, 1.0}};
  const C *cand = xg != X_F16 ? cg : (we == W_F16 ? c16 : (we == W_Q4 ? cq4 : cq8));
  double best = -1.0;
  for (int ci = 0; ci < 4; ci++) {
    const C &c = cand[ci];
    if (c.n == 256 && N <= 128) continue;
    if (c.m == 256 && M <= 128) continue;
    const uint64_t tiles = (uint64_t)((M + c.m - 1) / c.m) * ((N + c.n - 1) / c.n), slots = (uint64_t)cus * per_cu(c.m, c.n);
    const double rounds = (double)((tiles + slots - 1) / slots);
    const double useful = (double)M * N / ((double)c.m * c.n * rounds * slots);
    // q4 256 x 128 with 8 waves (a grid of one tile per CU at most): 2048 x 4096 x 4096 in 87.7 us against 143.7 for
    // twice the work at 256 x 256
    double rate = (we == W_Q4 && c.m == 256 && c.n == 128 && tiles <= cus) ? 0.80 : c.rate;
    // q4 128 x 128 with 8 waves (at most one tile per CU): DiT QKV's last 1024 columns as 256 such tiles instead of
    // 128 of 256 x 128 on half the CUs, 272 -> 265 us per call
    if (we == W_Q4 && c.m == 128 && c.n == 128 && tiles <= cus) rate = 0.6;
    const double score = rate * useful;
    if (score > best + 1e-9) { best = score; *bm = c.m; *bn = c.n; }
  }
}

// the tallest tile of the 1 x 4 x 2 wave layout: two stages of two steps within 160 KB
static unsigned dma_tall(int we) { return we == W_Q4 ? 256u : we == W_Q8 ? 224u : 192u; }

// the instances of launch_dma_we
bool dma_tile_ok(int we, int xg, unsigned bm, unsigned bn, unsigned wv) {
  if (bn == 256) return wv == 0 && (bm == 128 || bm == 256);
  if (bn != 128) return false;
  switch (wv) {
  case 0: return bm == 128 || bm == 256;                                   // (4 or 8 waves, as dma_wgs says)
  case 2: return xg == X_F16 && bm % 32 == 0 && bm != 0 && bm <= dma_tall(we);
  case 4: return bm == 128 || (bm == 256 && we == W_Q4);
  case 8: return bm == 256 || (bm == 128 && we != W_Q8) || (bm == 64 && we == W_F16 && xg != X_F16);
  }
  return false;
}

void dma_forced(uint32_t M, uint32_t N, uint32_t K, int we, int xg, uint64_t xbytes, const Tuning &t, DmaPlan *d) {
  for (unsigned wv : {t.tile_wv, 0u, 2u, 8u})
    if (t.tile_m && dma_tile_ok(we, xg, t.tile_m, t.tile_n, wv)) {
      *d = DmaPlan{t.tile_m, t.tile_n, wv, 1};
      break;
    }
  if (t.split && d->bn == 128 && dma_tile_ok(we, xg, d->bm, 128, 2)) {
    d->slices = t.split < K / DBK ? t.split : K / DBK;
    if (d->slices > 1 && xbytes + (uint64_t)d->slices * M * dma_ldp(N) * 4u > DMA_SPLIT_BYTES) d->slices = 1;
  }
}

// The plan of a call: dma_tile's tile; or, for grids that leave it idle or tiles half empty, a tile of the 1 x 4 x 2 wave
// layout (any 32 rows x 128 columns), with K in slices where its tiles are fewer than the CUs; or, with f16 weights, an
// 8-wave 128 x 128 tile. All are estimated, in us, in one form,
//   rounds of workgroups x (steps x (time of a 64-k step, less where the round leaves CUs idle) + fixed) (+ the slices'
//   exchange),
// whose constants are fitted to timed calls (q4, q8 and f16: 250-270 shapes each of 17..2048 rows x 1024..28672 columns x
// K 1024..14336, every tile and 1..8 slices; rms 5-7 %; over those shapes the picks are 1-1.7 % above the best and 1.8
// times as fast as dma_tile's). Taken where it is 10 % under the estimate of dma_tile's tile, so that
// the fit's errors do not pick a slower one. us, before -> after: q4 17 x 4096 x 4096 40.6 -> 11.0, 77 x 6144 x 4096
// 40.3 -> 16.8, 300 x 4096 x 14336 130 -> 48, 300 x 28672 x 4096 117 -> 88, 1000 x 4096 x 4096 55 -> 45; f16 77 x 6144 x
// 4096 42.9 -> 16.5.
struct TileCost { unsigned m, n, wgs; double step, fix, idle; };
struct SliceCost { double step[8], idle, fix, fix_row, split, split_mb; };   // step: of 32, 64 .. 256 rows
static double rounds_us(uint64_t wgs, uint64_t slots, double steps, double step, double idle, double fix) {
  const uint64_t rounds = (wgs + slots - 1) / slots, last = wgs - (rounds - 1) * slots;
  return (double)(rounds - 1) * (steps * step + fix) + steps * step * (idle + (1.0 - idle) * (double)last / (double)slots) + fix;
}

void dma_plan(uint32_t M, uint32_t N, uint32_t K, int we, int xg, uint64_t xbytes, unsigned cus, DmaPlan *d) {
  static const TileCost tiles[3][4] = {
      {{128, 128, 1, 0.699, 5.32, 0.724}, {256, 128, 1, 1.143, 8.37, 0.375}, {256, 256, 1, 2.016, 13.3, 0.245}, {}},
      {{128, 128, 2, 0.869, 4.96, 0.630}, {256, 128, 1, 1.000, 6.70, 0.530}, {256, 256, 1, 1.855, 14.2, 0.357}, {}},
      {{128, 128, 1, 0.521, 3.63, 0.539}, {128, 256, 1, 0.734, 8.52, 0.685}, {256, 128, 1, 0.824, 6.25, 0.506}, {256, 256, 1, 1.708, 13.4, 0.547}}};
  static const SliceCost slices[3] = {
      {{0.308, 0.374, 0.443, 0.512, 0.609, 0.743, 0.831, 0.910}, 0.670, 2.70, 0.020, 2.54, 0.359},
      {{0.278, 0.336, 0.410, 0.503, 0.711, 0.785, 0.851, 0.0}, 0.644, 2.77, 0.027, 2.49, 0.364},
      {{0.262, 0.326, 0.536, 0.608, 0.697, 0.761, 0.0, 0.0}, 0.689, 1.77, 0.024, 3.13, 0.341}};
  d->wv = 0;
  d->slices = 1;
  dma_tile(M, N, we, xg, cus, &d->bm, &d->bn);
  const uint32_t nk = (K + DBK - 1) / DBK;
  // (K of a few steps is all fixed cost; quantised convolution weights were not timed)
  if (M == 0 || N == 0 || nk < 8 || (xg != X_F16 && we != W_F16)) return;
  if (xg != X_F16) {
    // one order of K whatever the clip or the image (no halves, no slices): tiles of 64 and 128 rows x 128 with 8 waves for
    // calls of few tiles, the same estimate (conv3 61 shapes, 2-D 44, rms 2-5 %, picks within 0.5 % of the best on average).
    // us, before -> after: conv3 128 -> 128 32 x 32 51.3 -> 23.8, 3 x 41 x 123 52.5 -> 27.9, 2 x 92 x 160 53.1 -> 40.6; 256 ->
    // 256 2 x 27 x 101 92.9 -> 46.0; 2-D 512 -> 512 64 x 64 73.7 -> 36.1, 16 x 16 58.2 -> 29.4 (slices of K gave 34.1 and
    // 12.7, but an image taken in bands then had other bits than the whole one)
    static const TileCost conv[2][4] = {{{256, 128, 1, 0.956, 8.14, 0.779}, {128, 128, 2, 1.301, 3.22, 0.613},
                                         {128, 128, 1, 0.631, 4.45, 0.825}, {64, 128, 1, 0.403, 2.70, 0.857}},
                                        {{256, 128, 1, 0.983, 8.76, 0.729}, {128, 128, 2, 1.269, 6.69, 0.547},
                                         {128, 128, 1, 0.621, 5.99, 0.781}, {64, 128, 1, 0.404, 4.39, 0.848}}};
    const unsigned had = dma_wgs(we, d->bm, d->bn, 1, cus);
    double best = 0.0;
    for (const TileCost &c : conv[xg == X_CONV]) {
      const bool old = c.m == d->bm && c.n == d->bn && c.wgs == had;
      const double us = (old ? 0.95 : 1.0) * rounds_us((uint64_t)((M + c.m - 1) / c.m) * ((N + 127) / 128), (uint64_t)cus * c.wgs, nk,
                                                       c.step, c.idle, c.fix);
      if (best == 0.0 || us < best) { best = us; *d = DmaPlan{c.m, c.n, c.wgs == 2 ? 4u : 8u, 1}; }
    }
    return;
  }
  const int ei = we == W_Q4 ? 0 : we == W_Q8 ? 1 : 2;
  const uint64_t tn = (N + 127) / 128, had = (uint64_t)((M + d->bm - 1) / d->bm) * ((N + d->bn - 1) / d->bn);
  const unsigned wgs = dma_wgs(we, d->bm, d->bn, had, cus);
  double best = 0.0;
  for (const TileCost &c : tiles[ei])
    if (c.m == d->bm && c.n == d->bn && c.wgs == wgs && c.m) best = 0.9 * (2.0 + rounds_us(had, (uint64_t)cus * wgs, nk, c.step, c.idle, c.fix));
  if (best == 0.0) return;
  if (we == W_F16) {
    const TileCost &c = tiles[ei][0];
    const double us = 2.0 + rounds_us((uint64_t)((M + 127) / 128) * tn, cus, nk, c.step, c.idle, c.fix);
    if (us < best) { best = us; *d = DmaPlan{128, 128, 8, 1}; }
  }
  const SliceCost &c = slices[ei];
  for (unsigned bm = 32; bm <= dma_tall(we); bm += 32) {
    const uint64_t tm = (M + bm - 1) / bm;
    for (unsigned S = 1; S <= 8; S++) {
      const uint64_t part = S > 1 ? (uint64_t)S * M * dma_ldp(N) * 4u : 0u;
      if (S > 1 && (nk / S < 4 || tm * tn * S > 2ull * cus || xbytes + part > DMA_SPLIT_BYTES)) break;
      const double us = 2.0 + rounds_us(tm * tn * S, cus, (double)nk / S, c.step[bm / 32 - 1], c.idle, c.fix + c.fix_row * bm) +
                        (S > 1 ? c.split + c.split_mb * 1e-6 * (double)part : 0.0);
      if (us < best) { best = us; *d = DmaPlan{bm, 128, 2, S}; }
    }
  }
}

static hipError_t launch_dma_x(const Params &p, int we, int xg, unsigned bm, unsigned bn, unsigned wv, unsigned cus,
                               hipStream_t s) {
  const uint64_t tiles = (uint64_t)((p.M - p.mbase + bm - 1) / bm) * ((p.N - p.nbase + bn - 1) / bn);
  if (!wv && bn == 128 && bm % 128) wv = xg != X_F16 ? 8 : 2;
  if (!wv) wv = dma_wgs(we, bm, bn, tiles, cus) == 1 ? 8 : 4;
  switch (we) {
  case W_Q4: return launch_dma_q4(p, xg, bm, bn, wv, s);
  case W_Q8: return launch_dma_q8(p, xg, bm, bn, wv, s);
  case W_F16: return launch_dma_f16(p, xg, bm, bn, wv, s);
  }
  return hipErrorInvalidValue;
}

// Tail columns: when the grid's last round of tiles would leave at least half of the workgroup slots empty, the
// whole rounds run as one launch over the first columns (as many whole column bands of tiles as they hold) and the
// remaining columns as a second launch with the tile dma_tile picks for them (smaller tiles, more of them). Every tile
// sums K in the same order, so the output is the same bits as one launch. DiT QKV (576 tiles of 256 x 256 on 256 CUs,
// 2.25 rounds): 512 tiles, then the last 1024 columns in 128 x 128 tiles. P0K_DMA_TAIL=0 keeps one launch.
void dma_tail(uint32_t M, uint32_t N, int we, unsigned bm, unsigned bn, unsigned cus, uint32_t *ncut, unsigned *bm2,
              unsigned *bn2) {
  *ncut = N;
  *bm2 = bm;
  *bn2 = bn;
  const uint32_t tilesM = (M + bm - 1) / bm, tilesN = (N + bn - 1) / bn, T = tilesM * tilesN;
  const uint32_t slots = cus * dma_wgs(we, bm, bn, T, cus), full = T / slots * slots, tail = T - full;
  if (tail == 0 || 2 * tail > slots || full < tilesM) return;
  const uint32_t nA = full / tilesM;                           // column bands of the first launch
  if (nA >= tilesN) return;
  *ncut = nA * bn;
  dma_tile(M, N - *ncut, we, X_F16, cus, bm2, bn2);
}

hipError_t launch_gemm_dma(const Params &p, int we, int xg, const DmaPlan &d, unsigned cus, bool tail, hipStream_t s) {
  const unsigned bm = d.bm, bn = d.bn;
  if (p.slices > 1) {
    hipError_t e = launch_dma_x(p, we, xg, bm, bn, 2, cus, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_split_epi, dim3((p.M + SE_ROWS - 1) / SE_ROWS, p.ldp / 128), dim3(256), 0, s, p);
    return hipGetLastError();
  }
  uint32_t ncut = p.N;
  unsigned bm2 = bm, bn2 = bn;
  if (xg == X_F16 && tail && d.wv == 0) dma_tail(p.M, p.N, we, bm, bn, cus, &ncut, &bm2, &bn2);
  if (ncut >= p.N) return launch_dma_x(p, we, xg, bm, bn, d.wv, cus, s);
  Params a = p, b = p;
  a.N = ncut;                                                 // epilogue bounds: the first launch's columns only
  a.nbase = 0;
  b.nbase = ncut;
  hipError_t e = launch_dma_x(a, we, xg, bm, bn, 0, cus, s);
  if (e != hipSuccess) return e;
  return launch_dma_x(b, we, xg, bm2, bn2, 0, cus, s);
}

}  // namespace p0k
