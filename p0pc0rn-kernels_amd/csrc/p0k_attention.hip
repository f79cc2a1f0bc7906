// p0k_attention.hip — flash attention over the `heads` output of the QKV gemm (src/ops/attention.js:168-201), head
// size 128, on gfx950 matrix cores.
//
//   Q [Hq][Lq][128] f16, K / V [Hkv][Lk][128] f16 (head-major, as the heads epilogue writes them), O [Lq][ldo] f16
//   token-major at column h*128. Query head h reads kv head h / (Hq / Hkv). mode 0: no mask; 1: key j visible to query
//   i iff j <= min(i, nvalid - 1); 2: j < nvalid. Scores s = scale * q.k (scale defaults to 1/sqrt(128)), optionally
//   soft-capped to cap * tanh(s / cap); O = softmax(s) V with an exact online softmax in fp32.
//
// One workgroup owns 128 queries of one head (4 waves, 32 queries each, two workgroups per CU; a 256-query, 8-wave
// variant is selectable for tuning); each wave keeps its Q rows in registers. Everything is computed transposed, so
// that a lane owns ONE query and the softmax statistics stay in it:
//   S^T (keys x queries) = K Q^T           v_mfma_f32_32x32x16_f16, A = K from LDS, B = Q^T from registers
//   O^T (d x queries)   += V^T P           A = V^T from LDS, B = P = exp(S - m) from the S^T registers (fp16)
// In the 32x32 layout lane l holds column l % 32 (its query) and 16 rows 8 (r/4) + 4 (l/32) + r%4, so a row maximum
// or sum is a reduction over the lane's registers plus one exchange with lane l ^ 32. The 16 keys a lane contributes
// to one P.V step are exactly the keys its S^T registers hold, so P never leaves the registers. Keys come in tiles of
// 64 through a two-stage LDS ring (the next tile's loads are issued before this tile's MFMAs); K and V both arrive
// by the load-to-LDS path in their HBM layout [key][d], and the V^T operand is read with the transposing
// ds_read_b64_tr_b16 (four keys of one d per lane). Both tiles are XOR-swizzled so the 16-byte K reads and the
// transposed V reads of a wave hit distinct banks. Two waves per SIMD (256 registers each) let one wave's softmax
// run under the other's MFMAs.
#include "p0k_device.h"
#include "p0k_launch.h"
#include <algorithm>
#include <type_traits>

namespace p0k {

#ifndef P0K_AT_S
#define P0K_AT_S 2
#endif
constexpr int AT_S = P0K_AT_S, AT_BK = 64;

// AT_BQ queries per workgroup (128 or 256), 32 per wave. LPT: longest blocks first (mode 1), cxu = CUs of an XCD
template <int AT_BQ, bool CAP, bool LPT>
__global__ __launch_bounds__((2 * AT_BQ), (512 / (2 * AT_BQ))) void k_attention(AttnParams p, uint32_t cxu) {
  constexpr int AT_NT = 2 * AT_BQ, AT_NW = AT_NT / 64;
  __shared__ __attribute__((aligned(16))) f16 sK[AT_S][AT_BK * 128];   // [key][d], 16-byte chunk c at c ^ (key & 15)
  __shared__ __attribute__((aligned(16))) f16 sV[AT_S][AT_BK * 128];   // [key][d], 16-byte chunk c at c ^ 4 (key & 3)

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, gh = lane >> 5, l32 = lane & 31;
  // Workgroups go round-robin to the 8 XCDs; regroup them so each XCD walks whole heads (all query blocks of a head
  // in a row): the head's K / V (Lk x 256 B) then stays in that XCD's L2 instead of being fetched once per query block
  const uint32_t nqb = (p.Lq + AT_BQ - 1) / AT_BQ, nblk = nqb * p.Hq, b0 = blockIdx.x;
  uint32_t h, qblk;
  if constexpr (LPT) {
    // A causal block's work grows with its queries' position: the longest go first, so that the short ones fill the
    // ends. Where an XCD holds all of its blocks at once (two on a CU), the second on each CU comes in the opposite
    // order, so that every CU has the same sum (1999 queries x 32 heads: head by head, a CU got two blocks of the same
    // place, up to 64 key tiles against 34 on average: 61.0 -> 49.0 us)
    const uint32_t hx = (p.Hq & 7u) == 0u ? p.Hq >> 3 : p.Hq, n = nqb * hx;      // heads and blocks of an XCD
    uint32_t pos = (p.Hq & 7u) == 0u ? b0 >> 3 : b0;
    const uint32_t first = (p.Hq & 7u) == 0u ? cxu : 8 * cxu;
    if (n <= (512 / (2 * AT_BQ)) * first && pos >= first) pos = n - 1 - (pos - first);
    const uint32_t j = pos / hx;
    h = pos - j * hx + ((p.Hq & 7u) == 0u ? (b0 & 7u) * hx : 0u);
    qblk = nqb - 1 - j;
  } else {
    const uint32_t lin = (nblk & 7u) == 0u ? (b0 & 7u) * (nblk >> 3) + (b0 >> 3) : b0;
    h = lin / nqb;
    qblk = lin - h * nqb;
  }
  const uint32_t hk = h / (p.Hq / p.Hkv);
  const uint32_t q0 = qblk * AT_BQ, qw = q0 + wave * 32 + l32;
  const uint32_t qc = qw < p.Lq ? qw : p.Lq - 1u;

  // this lane's query row: 8 steps of 16 d, lane half gh holds d = 16 s + 8 gh .. + 7
  f16x8 qf[8];
  const uint16_t *qrow = p.Q + ((size_t)h * p.Lq + qc) * 128;
#pragma unroll
  for (int s = 0; s < 8; s++) qf[s] = *(const f16x8 *)(qrow + 16 * s + 8 * gh);

  uint32_t kend = p.Lk;
  if (p.mode == 1) {
    const uint32_t last = q0 + AT_BQ - 1 < p.nvalid - 1 ? q0 + AT_BQ - 1 : p.nvalid - 1;
    kend = p.Lk < last + 1 ? p.Lk : last + 1;
  } else if (p.mode == 2) {
    kend = p.Lk < p.nvalid ? p.Lk : p.nvalid;
  }
  // the keys this lane's query may see
  uint32_t qlim = p.Lk;
  if (p.mode == 1) qlim = (qc < p.nvalid - 1 ? qc : p.nvalid - 1) + 1;
  else if (p.mode == 2) qlim = p.nvalid;
  qlim = qlim < p.Lk ? qlim : p.Lk;
  const uint32_t ntile = (kend + AT_BK - 1) / AT_BK;
  const float sl2 = p.scale * 1.4426950408889634f;

  const uint16_t *Kb = p.K + (size_t)hk * p.Lk * 128, *Vb = p.V + (size_t)hk * p.Lk * 128;
  // K and V go global -> LDS by the load-to-LDS path: instruction i of wave w fills keys 4 (NW i + w) .. + 3 (1 KB),
  // lane l the 16-byte slot l % 16 of key l / 16, i.e. logical chunk (l % 16) ^ (key & 15) of K, (l % 16) ^ 4 (key & 3)
  // of V
  const int wv = __builtin_amdgcn_readfirstlane(wave);
  const uint32_t sk0 = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void *)&sK[0][0];
  auto kdma = [&](uint32_t t, int b) {
    const uint32_t k0 = t * AT_BK;
#pragma unroll
    for (int i = 0; i < 16 / AT_NW; i++) {
      const uint32_t kr = 4 * (AT_NW * i + wv) + lane / 16, key = k0 + kr, c = (lane & 15) ^ (kr & 15);
      const uint32_t off = ((key < p.Lk ? key : p.Lk - 1u) * 128 + c * 8) * 2;
      const uint32_t m0 = __builtin_amdgcn_readfirstlane(sk0 + (uint32_t)(b * AT_BK * 128 + 4 * (AT_NW * i + wv) * 128) * 2);
      asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(m0), "v"(off), "s"(Kb) : "memory");
    }
  };
  const uint32_t sv0 = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void *)&sV[0][0];
  auto vdma = [&](uint32_t t, int b) {
    const uint32_t k0 = t * AT_BK;
#pragma unroll
    for (int i = 0; i < 16 / AT_NW; i++) {
      const uint32_t kr = 4 * (AT_NW * i + wv) + lane / 16, key = k0 + kr, c = (lane & 15) ^ (4 * (kr & 3));
      const uint32_t off = ((key < p.Lk ? key : p.Lk - 1u) * 128 + c * 8) * 2;
      const uint32_t m0 = __builtin_amdgcn_readfirstlane(sv0 + (uint32_t)(b * AT_BK * 128 + 4 * (AT_NW * i + wv) * 128) * 2);
      asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(m0), "v"(off), "s"(Vb) : "memory");
    }
  };
  f32x16 oacc[4];
#pragma unroll
  for (int i = 0; i < 4; i++) oacc[i] = (f32x16){};
  float m = -1.0e30f, l = 0.0f;

  // AT_S-stage ring: tile t lives in buffer t % AT_S; tile t + AT_S - 1 is issued at the top of tile t into the buffer
  // every wave left at the barrier that ended tile t - 1. A wave's own loads complete in order, so waiting until at
  // most (AT_S - 2) tiles' worth of them are outstanding means its share of the next tile has landed.
  constexpr int PER = 32 / AT_NW;                           // load instructions per wave per tile (K and V)
  constexpr int NOUT = (AT_S - 2) * PER;
  constexpr int WAIT_RING = (NOUT & 15) | ((NOUT >> 4) << 14) | 0x0f70;
#pragma unroll
  for (int i = 0; i < AT_S - 1; i++)
    if ((uint32_t)i < ntile) {
      kdma(i, i);
      vdma(i, i);
    }
  if (ntile >= (uint32_t)(AT_S - 1)) __builtin_amdgcn_s_waitcnt(WAIT_RING);
  else __builtin_amdgcn_s_waitcnt(0x0f70);
  __syncthreads();
  int b = 0;
  for (uint32_t t = 0; t < ntile; t++) {
    const uint32_t k0 = t * AT_BK;
    if (t + AT_S - 1 < ntile) {
      const int bn = b == 0 ? AT_S - 1 : b - 1;
      kdma(t + AT_S - 1, bn);
      vdma(t + AT_S - 1, bn);
    }

    // ---- S^T for keys k0 .. k0+63: two 32-key blocks
    // (the two key blocks' MFMA chains alternate, and each K fragment read is issued one MFMA ahead of its use)
    f32x16 sacc[2];
    sacc[0] = (f32x16){};
    sacc[1] = (f32x16){};
#pragma unroll
    for (int s = 0; s < 8; s++)
#pragma unroll
      for (int kb = 0; kb < 2; kb++) {
        const uint32_t key = 32 * kb + l32;
        const f16x8 a = *(const f16x8 *)(sK[b] + key * 128 + (((2 * s + gh) ^ (key & 15u)) * 8));
        sacc[kb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, qf[s], sacc[kb], 0, 0, 0);
      }
    __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
    for (int q = 0; q < 14; q++) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
    __builtin_amdgcn_sched_barrier(0);
    // ---- scores to the log2 domain: max over the raw scores (the scale is positive), then exp2(s * sl2 - m) with one
    //      FMA per score. Soft cap: s -> cap * tanh(s * scale / cap) first. Keys past the lane's limit are masked only
    //      in tiles that reach past some lane's limit (a wave-uniform test).
    float sf = sl2;
    if constexpr (CAP) {
#pragma unroll
      for (int kb = 0; kb < 2; kb++)
#pragma unroll
        for (int r = 0; r < 16; r++) sacc[kb][r] = p.cap * (2.0f * sigmoid(2.0f * sacc[kb][r] * p.scale / p.cap) - 1.0f);
      sf = 1.4426950408889634f;
    }
    const uint32_t kl = qlim > k0 ? qlim - k0 : 0u;           // keys of this tile the lane's query sees: [0, kl)
    if (__any(kl < (uint32_t)AT_BK)) {
#pragma unroll
      for (int kb = 0; kb < 2; kb++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
          const uint32_t key = 32 * kb + 8 * (r >> 2) + 4 * gh + (r & 3);
          sacc[kb][r] = key < kl ? sacc[kb][r] : -1.0e30f;
        }
    }
    float mx = -1.0e30f;
#pragma unroll
    for (int kb = 0; kb < 2; kb++)
#pragma unroll
      for (int r = 0; r < 16; r++) mx = fmaxf(mx, sacc[kb][r]);
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    // m: running maximum in the log2 domain (-1e30: none yet)
    const float mxl = mx <= -1.0e29f ? -1.0e30f : mx * sf;
    // the maximum the exponents subtract stays where it is until some row's maximum grows past it by more than 8
    // (P <= 2^8 = 256 meanwhile: exact enough in fp16, and O and l keep the same common factor, which the final
    // division removes), so most tiles skip the rescale of O
    const float mn = __any(mxl > m + 8.0f) ? fmaxf(m, mxl) : m;
    // a masked score (-1e30) underflows exp2 to 0; a row with no visible key yet subtracts 0 instead of -1e30
    const float mns = mn <= -1.0e29f ? 0.0f : mn;
    float ps = 0.0f;
#pragma unroll
    for (int kb = 0; kb < 2; kb++)
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const float e = __builtin_amdgcn_exp2f(fmaf(sacc[kb][r], sf, -mns));
        sacc[kb][r] = e;
        ps += e;
      }
    if (__any(mn != m)) {                                       // rescale only when the subtracted maximum moved
      const float alpha = __builtin_amdgcn_exp2f(m - mn);
      l = l * alpha;
#pragma unroll
      for (int db = 0; db < 4; db++) oacc[db] *= alpha;
    }
    m = mn;
    l += ps;

    // ---- O^T += V^T P over four 16-key steps
#pragma unroll
    for (int c = 0; c < 4; c++) {
      const int kb = c >> 1, h2 = c & 1;
      const f16x8 bp = {(f16)sacc[kb][8 * h2 + 0], (f16)sacc[kb][8 * h2 + 1], (f16)sacc[kb][8 * h2 + 2],
                        (f16)sacc[kb][8 * h2 + 3], (f16)sacc[kb][8 * h2 + 4], (f16)sacc[kb][8 * h2 + 5],
                        (f16)sacc[kb][8 * h2 + 6], (f16)sacc[kb][8 * h2 + 7]};
#pragma unroll
      for (int db = 0; db < 4; db++) {
        // transposed read: lane 4 j + a of each 16-lane group addresses key j, d 4 a .. 4 a + 3; lane 4 a + b then
        // receives d 4 a + b of keys j = 0..3. Lanes 16..31 of a half take the next 16 d; half gh the keys 4 gh ..
        const uint32_t kr = 32 * kb + 16 * h2 + 4 * gh + ((lane >> 2) & 3), c = 4 * db + 2 * ((lane >> 4) & 1) + ((lane >> 1) & 1);
        const f16 *va = sV[b] + kr * 128 + ((c ^ (4 * (kr & 3))) * 8) + 4 * (lane & 1);
        typedef short v4s __attribute__((ext_vector_type(4)));
        const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4s *)va);
        const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4s *)(va + 8 * 128));
        const f16x8 av = __builtin_bit_cast(f16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        oacc[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av, bp, oacc[db], 0, 0, 0);
      }
    }
    // (this phase is left to the compiler's schedule: pinning each MFMA behind two transposed V reads, as the S phase
    // pins its K reads, ran 249-251 against 242-244 us)
    if (t + AT_S - 1 < ntile) __builtin_amdgcn_s_waitcnt(WAIT_RING);   // this wave's share of tile t + 1 has landed
    else __builtin_amdgcn_s_waitcnt(0x0f70);
    __syncthreads();
    b = b == AT_S - 1 ? 0 : b + 1;
  }

  // ---- O = O^T / l: lane writes its query's 128 values in runs of 4 d
  const float lt = l + __shfl_xor(l, 32, 64);
  const float inv = lt > 0.0f ? 1.0f / lt : 0.0f;
  if (qw < p.Lq) {
    uint16_t *orow = p.O + (size_t)qw * p.ldo + h * 128;
#pragma unroll
    for (int db = 0; db < 4; db++)
#pragma unroll
      for (int g4 = 0; g4 < 4; g4++) {
        const uint32_t d = 32 * db + 8 * g4 + 4 * gh;
        *(u32x2 *)(orow + d) = (u32x2){pack2(oacc[db][4 * g4] * inv, oacc[db][4 * g4 + 1] * inv),
                                       pack2(oacc[db][4 * g4 + 2] * inv, oacc[db][4 * g4 + 3] * inv)};
      }
  }
}

// ---------------------------------------------------------------------------------------- few queries, many keys
// k_attention gives a head 128 queries per workgroup and walks all of its keys with one: a decode step (one query, 32
// heads) fills 32 of 256 CUs and reads its cache one 64-key tile at a time. Here a workgroup owns 32 query ROWS of one
// kv head (the Hq / Hkv query heads that share it x their queries, packed, so GQA reads the cache once) and one of S
// runs of its keys; each of its 4 waves takes every fourth 32-key tile of the run through a private two-tile LDS ring
// (K and V 8 KB each, load-to-LDS, no barrier in the loop), so 128 KB per CU are in flight right after the launch. The
// matrix products, layouts and softmax are those of k_attention (a lane owns one row). The waves' (maximum, sum, O)
// meet in LDS; with S > 1 every workgroup leaves its rows in `part` (sc0 sc1 stores) and the last one of a kv head and
// row block to arrive merges them in run order, so the result does not depend on timing.
// HBM-latency-bound: one query, 32 heads on 8 kv heads, 3777 keys (15.5 MB): 68.9 -> 10.6 us.
constexpr int AS_W = 4, AS_K = 32, AS_LD = 132;           // waves, keys per tile, padded fp32 row of O in LDS
constexpr uint32_t AS_PART = 32 * 128 + 64;               // floats one workgroup leaves: O [32][128], m [32], l [32]

template <bool CAP>
__global__ __launch_bounds__(64 * AS_W, 1) void k_attention_split(AttnParams p, uint32_t nqb, uint32_t S,
                                                                float *part, uint32_t *cnt) {
  __shared__ __attribute__((aligned(16))) f16 ring[AS_W][2][2][AS_K * 128];   // wave, stage, K / V, [key][d]
  __shared__ float sm[AS_W][32], sl[AS_W][32];
  __shared__ uint32_t sLast;
  static_assert(sizeof(ring) >= sizeof(float) * AS_W * 32 * AS_LD, "O staging");

  const int tid = threadIdx.x, lane = tid & 63, gh = lane >> 5, l32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // row blocks of one run of keys go to one XCD (they read the same K / V)
  const uint32_t nblk = gridDim.x, b0 = blockIdx.x;
  const uint32_t lin = (nblk & 7u) == 0u ? (b0 & 7u) * (nblk >> 3) + (b0 >> 3) : b0;
  const uint32_t qb = lin % nqb, run = (lin / nqb) % S, hk = lin / nqb / S;
  const uint32_t rep = p.Hq / p.Hkv, R = rep * p.Lq;
  const uint32_t nrow = R - qb * 32 < 32u ? R - qb * 32 : 32u;                // live rows of this block
  const uint32_t row = qb * 32 + ((uint32_t)l32 < nrow ? l32 : nrow - 1u);
  const uint32_t h = hk * rep + row / p.Lq, qi = row % p.Lq;

  f16x8 qf[8];
  const uint16_t *qrow = p.Q + ((size_t)h * p.Lq + qi) * 128;
#pragma unroll
  for (int s = 0; s < 8; s++) qf[s] = *(const f16x8 *)(qrow + 16 * s + 8 * gh);
  uint32_t qlim = p.Lk;                                                       // the keys this lane's row may see
  if (p.mode == 1) qlim = (qi < p.nvalid - 1 ? qi : p.nvalid - 1) + 1;
  else if (p.mode == 2) qlim = p.nvalid;
  qlim = qlim < p.Lk ? qlim : p.Lk;
  const float sl2 = p.scale * 1.4426950408889634f;

  uint32_t kend = p.Lk;                                                       // the keys any row of the block sees
  if (p.mode == 1) {
    const uint32_t q0 = qb * 32 % p.Lq + nrow - 1, qmax = q0 < p.Lq - 1 ? q0 : p.Lq - 1;   // (rows may wrap to the next head)
    kend = (qmax < p.nvalid - 1 ? qmax : p.nvalid - 1) + 1;
  } else if (p.mode == 2) {
    kend = p.nvalid;
  }
  kend = kend < p.Lk ? kend : p.Lk;
  const uint32_t nt = (kend + AS_K - 1) / AS_K;
  const uint32_t t0 = (uint32_t)((uint64_t)nt * run / S), t1 = (uint32_t)((uint64_t)nt * (run + 1) / S);
  const uint16_t *Kb = p.K + (size_t)hk * p.Lk * 128, *Vb = p.V + (size_t)hk * p.Lk * 128;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void *)&ring[wave][0][0][0];
  // instruction i fills keys 4 i .. 4 i + 3 of the tile: lane l the slot l % 16 of key l / 16, i.e. logical chunk
  // (l % 16) ^ (key & 15) of K, (l % 16) ^ 4 (key & 3) of V
  auto fill = [&](uint32_t t, int st) {
#pragma unroll
    for (int kv = 0; kv < 2; kv++)
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const uint32_t kr = 4 * i + lane / 16, key = t * AS_K + kr;
        const uint32_t c = (lane & 15) ^ (kv == 0 ? (kr & 15) : 4 * (kr & 3));
        const uint32_t off = ((key < p.Lk ? key : p.Lk - 1u) * 128 + c * 8) * 2;
        const uint32_t m0 = __builtin_amdgcn_readfirstlane(lds0 + (uint32_t)((st * 2 + kv) * AS_K * 256 + i * 1024));
        asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(m0), "v"(off), "s"(kv == 0 ? Kb : Vb) : "memory");
      }
  };
  // (a wave's loads land in order, and the compiler does not count these: every wait on them is explicit)
  f32x16 oacc[4];
#pragma unroll
  for (int i = 0; i < 4; i++) oacc[i] = (f32x16){};
  float m = -1.0e30f, l = 0.0f;
  uint32_t t = t0 + wave;
  if (t < t1) fill(t, 0);
  if (t + AS_W < t1) fill(t + AS_W, 1);
  for (int st = 0; t < t1; t += AS_W, st ^= 1) {
    const bool more = t + AS_W < t1;                                          // the next tile's 16 loads are in flight
    if (more) asm volatile("s_waitcnt vmcnt(24)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    const f16 *sK = ring[wave][st][0], *sV = ring[wave][st][1];
    const uint32_t k0 = t * AS_K;
    f32x16 sacc = (f32x16){};
#pragma unroll
    for (int s = 0; s < 8; s++) {
      const f16x8 a = *(const f16x8 *)(sK + l32 * 128 + (((2 * s + gh) ^ (l32 & 15)) * 8));
      sacc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, qf[s], sacc, 0, 0, 0);
    }
    float sf = sl2;
    if constexpr (CAP) {
#pragma unroll
      for (int r = 0; r < 16; r++) sacc[r] = p.cap * (2.0f * sigmoid(2.0f * sacc[r] * p.scale / p.cap) - 1.0f);
      sf = 1.4426950408889634f;
    }
    const uint32_t kl = qlim > k0 ? qlim - k0 : 0u;
    if (__any(kl < (uint32_t)AS_K)) {
#pragma unroll
      for (int r = 0; r < 16; r++) sacc[r] = 8u * (r >> 2) + 4u * gh + (r & 3u) < kl ? sacc[r] : -1.0e30f;
    }
    float mx = -1.0e30f;
#pragma unroll
    for (int r = 0; r < 16; r++) mx = fmaxf(mx, sacc[r]);
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float mxl = mx <= -1.0e29f ? -1.0e30f : mx * sf;
    const float mn = fmaxf(m, mxl);
    const float mns = mn <= -1.0e29f ? 0.0f : mn;
    float ps = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const float e = __builtin_amdgcn_exp2f(fmaf(sacc[r], sf, -mns));
      sacc[r] = e;
      ps += e;
    }
    if (__any(mn != m)) {
      const float alpha = __builtin_amdgcn_exp2f(m - mn);
      l = l * alpha;
#pragma unroll
      for (int db = 0; db < 4; db++) oacc[db] *= alpha;
    }
    m = mn;
    l += ps;
    if (more) asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
    for (int h2 = 0; h2 < 2; h2++) {
      const f16x8 bp = {(f16)sacc[8 * h2 + 0], (f16)sacc[8 * h2 + 1], (f16)sacc[8 * h2 + 2], (f16)sacc[8 * h2 + 3],
                        (f16)sacc[8 * h2 + 4], (f16)sacc[8 * h2 + 5], (f16)sacc[8 * h2 + 6], (f16)sacc[8 * h2 + 7]};
#pragma unroll
      for (int db = 0; db < 4; db++) {
        const uint32_t kr = 16 * h2 + 4 * gh + ((lane >> 2) & 3), c = 4 * db + 2 * ((lane >> 4) & 1) + ((lane >> 1) & 1);
        const f16 *va = sV + kr * 128 + ((c ^ (4 * (kr & 3))) * 8) + 4 * (lane & 1);
        typedef short v4s __attribute__((ext_vector_type(4)));
        const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4s *)va);
        const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4s *)(va + 8 * 128));
        const f16x8 av = __builtin_bit_cast(f16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        oacc[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av, bp, oacc[db], 0, 0, 0);
      }
    }
    if (t + 2 * AS_W < t1) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                      // this tile's reads are done: refill it
      fill(t + 2 * AS_W, st);
    }
  }

  // ---- the four waves' rows: O scaled to the common maximum
  l += __shfl_xor(l, 32, 64);
  if (gh == 0) { sm[wave][l32] = m; sl[wave][l32] = l; }
  __syncthreads();                                                            // every wave is done with its ring
  float *sO = (float *)ring;
#pragma unroll
  for (int db = 0; db < 4; db++)
#pragma unroll
    for (int g4 = 0; g4 < 4; g4++)
      *(f32x4 *)(sO + (wave * 32 + l32) * AS_LD + 32 * db + 8 * g4 + 4 * gh) =
          (f32x4){oacc[db][4 * g4], oacc[db][4 * g4 + 1], oacc[db][4 * g4 + 2], oacc[db][4 * g4 + 3]};
  __syncthreads();
  auto put = [&](uint32_t r, uint32_t d, f32x4 o, float L) {                  // O row of block row r, d .. d + 3
    const uint32_t gr = qb * 32 + r, hh = hk * rep + gr / p.Lq, q = gr % p.Lq;
    const float inv = L > 0.0f ? 1.0f / L : 0.0f;
    *(u32x2 *)(p.O + (size_t)q * p.ldo + hh * 128 + d) = (u32x2){pack2(o.x * inv, o.y * inv), pack2(o.z * inv, o.w * inv)};
  };
  const srsrc pr = stream_rsrc((const uint8_t *)part);
  const uint32_t grp = hk * nqb + qb, slot0 = grp * S;                        // this block's rows in `part`
  for (uint32_t it = tid; it < nrow * 32; it += 64 * AS_W) {
    const uint32_t r = it >> 5, d = (it & 31u) * 4;
    float M = sm[0][r];
#pragma unroll
    for (int w = 1; w < AS_W; w++) M = fmaxf(M, sm[w][r]);
    f32x4 o = (f32x4){};
    float L = 0.0f;
#pragma unroll
    for (int w = 0; w < AS_W; w++) {
      const float f = __builtin_amdgcn_exp2f(sm[w][r] - M);
      o += f * *(const f32x4 *)(sO + (w * 32 + r) * AS_LD + d);
      L += f * sl[w][r];
    }
    if (S == 1) {
      put(r, d, o, L);
    } else {
      const uint32_t base = (slot0 + run) * AS_PART;
      sys_store128(pr, (base + r * 128 + d) * 4u, __builtin_bit_cast(u32x4, o));
      if (d == 0) __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, (f32x2){M, L}), pr, (int)((base + 32 * 128 + 2 * r) * 4u), 0, SC0_SC1);
    }
  }
  if (S == 1) return;
  __builtin_amdgcn_s_waitcnt(0);                                              // this thread's rows are in memory
  __syncthreads();
  if (tid == 0) sLast = __hip_atomic_fetch_add(cnt + grp, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) == S - 1 ? 1u : 0u;
  __syncthreads();
  if (!sLast) return;

  // ---- the last run to arrive merges all of them. np threads share one (row, d .. d + 3), each a contiguous part of
  //      the runs with 16 runs' loads in flight; their results meet in LDS
  const uint32_t items = nrow * 32;
  const uint32_t np = items <= 32 ? 8u : items <= 64 ? 4u : items <= 128 ? 2u : 1u;
  for (uint32_t it0 = 0; it0 < items; it0 += 64 * AS_W) {                     // (one pass whenever np > 1)
    const uint32_t pi = np > 1 ? tid / items : 0u, it = np > 1 ? tid % items : it0 + tid;
    const bool live = pi < np && it < items;
    const uint32_t r = it >> 5, d = (it & 31u) * 4;
    float M = -1.0e30f, L = 0.0f;
    f32x4 o = (f32x4){};
    if (live) {
      for (uint32_t s = S * pi / np, e = S * (pi + 1) / np; s < e; s += 16) {
        f32x4 ov[16];
        f32x2 ml[16];
#pragma unroll
        for (uint32_t u = 0; u < 16; u++) {
          const uint32_t base = (slot0 + (s + u < e ? s + u : e - 1u)) * AS_PART;
          ml[u] = __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(pr, (int)((base + 32 * 128 + 2 * r) * 4u), 0, SC0_SC1));
          ov[u] = __builtin_bit_cast(f32x4, sys_load128(pr, (base + r * 128 + d) * 4u));
        }
        float Mn = M;
#pragma unroll
        for (uint32_t u = 0; u < 16; u++) Mn = fmaxf(Mn, ml[u].x);            // (a repeated run changes no maximum)
        const float a = __builtin_amdgcn_exp2f(M - Mn);
        o *= a;
        L *= a;
#pragma unroll
        for (uint32_t u = 0; u < 16; u++) {
          const float f = s + u < e ? __builtin_amdgcn_exp2f(ml[u].x - Mn) : 0.0f;
          o += f * ov[u];
          L += f * ml[u].y;
        }
        M = Mn;
      }
    }
    if (np > 1) {
      // sO is free: this block's rows have left it (the barriers above)
      if (live) {
        *(f32x4 *)(sO + (pi * items + it) * 4) = o;
        *(f32x2 *)(sO + 4096 + (pi * items + it) * 2) = (f32x2){M, L};
      }
      __syncthreads();
      if (pi == 0 && live) {
        for (uint32_t q = 1; q < np; q++) {
          const f32x2 ml = *(const f32x2 *)(sO + 4096 + (q * items + it) * 2);
          const float Mn = fmaxf(M, ml.x), a = __builtin_amdgcn_exp2f(M - Mn), f = __builtin_amdgcn_exp2f(ml.x - Mn);
          o = a * o + f * *(const f32x4 *)(sO + (q * items + it) * 4);
          L = a * L + f * ml.y;
          M = Mn;
        }
      }
    }
    if (live && pi == 0) put(r, d, o, L);
  }
  if (tid == 0) __hip_atomic_store(cnt + grp, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

static uint32_t attention_kend(const AttnParams &p) {   // the keys any query sees
  uint32_t kend = p.Lk;
  if (p.mode == 1) kend = std::min(p.Lk, std::min(p.Lq, p.nvalid));
  else if (p.mode == 2) kend = std::min(p.Lk, p.nvalid);
  return kend;
}

int attention_bq(uint32_t Lq, uint32_t Hq, int cus, int force) {
  if (force == 128 || force == 256) return force;                 // tuning / tests (P0K_ATTN_BQ)
  // 128 (two workgroups per CU). 256 queries per workgroup halve the LDS fill per query but run one workgroup per CU:
  // 24 heads x 4096 queries, 300 us vs 280 us (its 384 blocks leave half the CUs idle in the second round, where
  // the 768 blocks of 128 let the last third of a CU's blocks run alone and faster)
  (void)Lq;
  (void)Hq;
  (void)cus;
  return 128;
}

uint64_t attention_part_bytes(int cus) { return (uint64_t)cus * AS_PART * sizeof(float); }

// Where the few-queries kernel is taken: its row blocks fit the CUs in one round (it holds one workgroup per CU, so a
// second round costs what the 128-query blocks save: 64 heads on 16, 256 queries, 512 blocks, 2048 keys 46.9 us
// against 36.4) and it has more than 128 keys or few rows to store. Measured against the 128-query blocks over
// 5 head layouts x 1..256 queries x 128..8192 keys: 1.1-1.5x at up to 16 rows and 128 / 512 keys, 2-5x at 2048 keys,
// 4-11x at 8192; with 192-256 blocks (256 queries) 1.2-1.7x.
// Runs: as many as the CUs hold, but the exchange at the end costs as much as 2 + rows / 10 tiles of a wave (3 us with 4
// live rows, 7 with 32: 512 keys in 4 runs 13.0-13.4 us, in one 9.7), so short calls keep one run.
unsigned attention_runs(const AttnParams &p, int cus, bool ws, int force) {
  if (force == 0) return 0;
  const uint64_t R = (uint64_t)(p.Hq / p.Hkv) * p.Lq, nqb = (R + 31) / 32, groups = nqb * p.Hkv;
  const uint32_t sets = (attention_kend(p) + AS_W * AS_K - 1) / (AS_W * AS_K);   // 128-key sets: a tile for each wave
  if (groups > 0xffffffu || (force < 0 && (groups > (uint64_t)cus || (sets == 1 && R > 16 && p.Lq < 64)))) return 0;
  const uint32_t S = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(sets, (uint64_t)cus / groups));
  const uint32_t saved = sets - (sets + S - 1) / S, rows = (uint32_t)std::min<uint64_t>(R, 32);
  if (!ws || groups > ATTN_COUNTERS || saved * 10 <= 20 + rows) return 1;
  return S;
}

hipError_t launch_attention(const AttnParams &p, int cus, int force_bq, unsigned runs, float *part, unsigned *cnt,
                            hipStream_t s) {
  if (p.Lq == 0 || p.Hq == 0) return hipSuccess;
  if (runs) {
    const uint32_t nqb = (uint32_t)(((uint64_t)(p.Hq / p.Hkv) * p.Lq + 31) / 32);
    const dim3 grid(p.Hkv * nqb * runs), block(64 * AS_W);
    if (p.cap > 0.0f) hipLaunchKernelGGL(k_attention_split<true>, grid, block, 0, s, p, nqb, runs, part, cnt);
    else hipLaunchKernelGGL(k_attention_split<false>, grid, block, 0, s, p, nqb, runs, part, cnt);
    return hipGetLastError();
  }
  const int bq = attention_bq(p.Lq, p.Hq, cus, force_bq);
  dim3 grid(((p.Lq + bq - 1) / bq) * p.Hq);
  const uint32_t cxu = (uint32_t)cus / 8u;
  // (a block per CU at most: the longest decides in any order, and head by head K / V stay in one L2: 2048 queries x 12
  // heads 39.2 us against 41.4)
  const bool lpt = p.mode == 1 && grid.x > (unsigned)cus;
  auto go = [&](auto cap, auto longest) {
    if (bq == 256) hipLaunchKernelGGL((k_attention<256, decltype(cap)::value, decltype(longest)::value>), grid, dim3(512), 0, s, p, cxu);
    else hipLaunchKernelGGL((k_attention<128, decltype(cap)::value, decltype(longest)::value>), grid, dim3(256), 0, s, p, cxu);
  };
  if (p.cap > 0.0f) lpt ? go(std::true_type{}, std::true_type{}) : go(std::true_type{}, std::false_type{});
  else lpt ? go(std::false_type{}, std::true_type{}) : go(std::false_type{}, std::false_type{});
  return hipGetLastError();
}

}  // namespace p0k
