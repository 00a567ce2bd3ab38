// Exact router logits of many tokens on the int8 matrix cores (HF:768-776).
//
//   logit[t, e] = bf16(f32(S)),  S = sum_k x[t, k] * w[e, k], exact
//
// The fp64 matrix rate bounds the direct form (route.hip: 45 us for 2048
// tokens x 256 experts x 2048).  A bf16 row is instead written as fixed-point integers of
// 23 bits, x[k] = X[k] 2^-s with s from the row's largest value, and X as three
// signed base-256 digits, so S is nine int8 products with exact int32 sums
// (at a seventh of the fp64 MFMA cycles), combined in 64-bit integers.
//
// A value below 2^-15 of its row's largest may not fit the grid.  Each row keeps the sum of
// those residues, R = sum_k |x[k] - X[k] 2^-s| (0 for most rows), and its
// largest value m, so |S - S'| <= R_t m_e + R_e m_t for the computed S', plus
// half an ulp where S' exceeds 53 bits.  Where the two ends of that
// interval round to the same bf16 value, that is the logit; the few others,
// and every logit of a row that is not finite or below 2^-100, are taken again
// by an fp64 dot product, the value the direct form computes.
//
// Rows with a strong channel (some 200 times the others and more) would leave many
// logits open, so a block of 16 token rows with a residue above kRdResidue
// also stores its residues: x[k] - X[k] 2^-s has at most 8 significant bits and is
// exact in bf16, and one bf16 product per logit adds sum_k (x - X 2^-s) w in
// fp32, which leaves 2^-11 of the bound above.  With a channel of 3000 or 30000
// times the others, 2048 tokens take 45 us (the direct form 46); without the
// residues they took 77 and 76.
//
// At 2048 tokens router_digits_kernel takes 13.7 us (it writes 14 MB of digits;
// half of that is its chain of load, largest value, barrier, digits) and
// router_digits_mfma 15 us (4 us of MFMAs; its operands come from L2 at 200 MB
// a call, and the 64-bit finish is not overlapped): 32 us with the top-k against
// 45; 22 against 27 at 700 tokens, 46 against 83 at 4096.
#include <algorithm>

#include "internal.hpp"

namespace lm {
namespace {

struct RowMeta {
  int s;        // x[k] = X[k] 2^-s
  float m;      // largest |x[k]|
  float r[2];   // sum of residues of each half of K (NaN: use fp64)
};

// Digits in MFMA operand order: block (16 rows x 64 K) b = row / 16 * (H / 64) +
// k / 64 holds three planes of 1 KB, byte 16 (16 p + row % 16) + j of a plane
// being digit k = 64 b + 16 p + j.
struct DigitArgs {
  const uint16_t *x, *w;
  const float *bias;
  float *logits;
  int8_t *xd, *wd;
  RowMeta *xm, *wm;
  u32x4 *xr;    // token residues x - X 2^-s, scaled by 2^s, bf16 in MFMA operand order:
                // K block b of row block j holds two steps of 64 pieces at ((j nk + b) 2 + h) 64
  uint8_t *xflag;  // [row blocks][halves of K]: the residues are stored
  int T, E, H;
};

// A half row block stores its residues where its 16 rows have more than
// kRdResidue in all, in units of each row's grid and counting up to one per wave (a
// sixteenth of the half row), so that one row alone does not decide.  A half row of
// normal values has 0.03, with a channel 300 times the others 2 (11 logits of a
// tile's 1024 open, taken again in 6 us of a call), 1000 times 7 (34 open, 17 us;
// the residues 13).
constexpr int kRdResidue = 80;

// One 16-row block per workgroup, K blocks dealt to its 16 waves: coalesced row
// loads into LDS (chunks XOR-swizzled by row), then lane l (row l & 15, quarter p
// = l >> 4) reads the 16 values it stores in every K block, first for the row's
// largest value, then for digits and residues, so a block's planes are written
// whole.  blockIdx.y takes the digits of one half of K; the largest value is
// each half's own work (2048 tokens give only 144 row blocks for 256 CUs).
constexpr int kRdWaves = 16;
__global__ __launch_bounds__(kRdWaves * 64) void router_digits_kernel(DigitArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];  // [16][H] values
  __shared__ uint32_t wmax[kRdWaves][16];
  __shared__ float wres[kRdWaves][16];
  __shared__ int large;  // the block's residues in sixteenths of a grid unit
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tblocks = (a.T + 15) / 16;  // the expert rows' blocks follow
  const bool tok = (int)blockIdx.x < tblocks;
  const int blk = tok ? blockIdx.x : blockIdx.x - tblocks;
  const int rows = min(16, (tok ? a.T : a.E) - blk * 16);
  const uint16_t *src = (tok ? a.x : a.w) + (int64_t)blk * 16 * a.H;
  int8_t *dst = (tok ? a.xd : a.wd) + (int64_t)blk * (a.H / 64) * 3072;
  const int nk = a.H / 64, pitch = a.H * 2;
  // wave load: 8 rows x one 128-byte K block; rows past the end repeat the last
  for (int kb = wave; kb < nk; kb += 2 * kRdWaves) {
    u32x4 v[2][2];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        v[u][h] = ldg16(src + (int64_t)min(8 * h + (lane >> 3), rows - 1) * a.H +
                        min(kb + u * kRdWaves, nk - 1) * 64 + (lane & 7) * 8);
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int row = 8 * h + (lane >> 3), ch = (kb + u * kRdWaves) * 8 + (lane & 7);
        if (kb + u * kRdWaves < nk)
          *reinterpret_cast<u32x4 *>(smem + row * pitch + ((ch ^ (row & 7)) * 16)) = v[u][h];
      }
  }
  wave_lds_sync();
  const int r = lane & 15, p = lane >> 4;
  auto piece = [&](int kb, int h) {  // values 64 kb + 16 p + 8 h .. + 7 of row r
    const int ch = 8 * kb + 2 * p + h;
    return *reinterpret_cast<const u32x4 *>(smem + r * pitch + ((ch ^ (r & 7)) * 16));
  };
  // scaled value j of a piece, and its distance from the grid
  auto scaled = [](u32x4 v, int j, int s) {
    return ldexpf(bf16_bits_to_f32((v[j >> 1] >> (16 * (j & 1))) & 0xFFFFu), s);
  };
  uint32_t mb = 0;  // largest |x| as bits: the order of finite values, inf and NaN above
  for (int kb = wave; kb < nk; kb += kRdWaves)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const u32x4 v = piece(kb, h);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        mb = max(mb, max((v[j] << 16) & 0x7FFF0000u, v[j] & 0x7FFF0000u));
    }
  mb = max(mb, (uint32_t)__shfl_xor((int)mb, 16, 64));
  mb = max(mb, (uint32_t)__shfl_xor((int)mb, 32, 64));
  if (p == 0) wmax[wave][r] = mb;
  if (threadIdx.x == 0) large = 0;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kRdWaves; ++w) mb = max(mb, wmax[w][r]);
  const float m = __uint_as_float(mb);
  const bool direct = mb >= 0x7F800000u || (mb != 0 && m < 0x1.0p-100f);
  // m in [2^(ex - 1), 2^ex): |X| <= 2^22
  const int ex = (int)(mb >> 23) - 126;
  const int s = direct || mb == 0 ? 0 : 22 - ex;
  float res = 0.0f;
  const int kh = (nk + 1) / 2, kb0 = blockIdx.y * kh, kb1 = min(kb0 + kh, nk);
  for (int kb = kb0 + wave; kb < kb1; kb += kRdWaves) {
    u32x4 d[3] = {{0u, 0u, 0u, 0u}, {0u, 0u, 0u, 0u}, {0u, 0u, 0u, 0u}};
    if (!direct) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const u32x4 v = piece(kb, h);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float f = scaled(v, j, s);
          const float g = rintf(f);
          // exact: f has 8 significant bits and |f - g| <= 1/2; a nonzero value
          // scaled into or below the subnormals counts as 2^-100
          const bool tiny = fabsf(f) < 0x1.0p-100f && ((v[j >> 1] >> (16 * (j & 1))) & 0x7FFFu);
          res += tiny ? 0x1.0p-100f : fabsf(f - g);
          const int X = (int)g;
          const int d0 = (int)(int8_t)X, x1 = (X - d0) >> 8;
          const int d1 = (int)(int8_t)x1, d2 = (x1 - d1) >> 8;
          const int at = 2 * h + (j >> 2), sh = 8 * (j & 3);
          d[0][at] |= (uint32_t)(d0 & 255) << sh;
          d[1][at] |= (uint32_t)(d1 & 255) << sh;
          d[2][at] |= (uint32_t)(d2 & 255) << sh;
        }
      }
    }
#pragma unroll
    for (int c = 0; c < 3; ++c)
      *reinterpret_cast<u32x4 *>(dst + (int64_t)kb * 3072 + c * 1024 + lane * 16) = d[c];
  }
  res += __shfl_xor(res, 16, 64);
  res += __shfl_xor(res, 32, 64);
  if (p == 0) {
    wres[wave][r] = res;
    if (tok && res > 0.0f) atomicAdd(&large, (int)(16.0f * fminf(res, 1.0f)));
  }
  __syncthreads();
  const bool store = large > 16 * kRdResidue;  // tokens only
  if (store) {
    u32x4 *out = a.xr + (int64_t)blk * nk * 128 + lane;
    for (int kb = kb0 + wave; kb < kb1; kb += kRdWaves)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const u32x4 v = piece(kb, h);
        u32x4 o = {0u, 0u, 0u, 0u};
        if (!direct) {
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const float f = scaled(v, j, s);
            o[j >> 1] |= (__float_as_uint(f - rintf(f)) >> 16) << (16 * (j & 1));
          }
        }
        out[(kb * 2 + h) * 64] = o;
      }
  }
  if (threadIdx.x < 16 && (int)threadIdx.x < rows) {  // wave 0: lane r holds row r's m and s
    if (tok && r == 0) a.xflag[blk * 2 + blockIdx.y] = store;
    res = 0.0f;
#pragma unroll
    for (int w = 0; w < kRdWaves; ++w) res += wres[w][r];
    RowMeta &o = (tok ? a.xm : a.wm)[blk * 16 + r];
    if (blockIdx.y == 0) {
      o.s = s;
      o.m = m;
    }
    // 1.001 covers the rounding of the sum
    o.r[blockIdx.y] = direct      ? __uint_as_float(0x7FC00000u)
          : res == 0.0f ? 0.0f
                        : fmaxf(ldexpf(res * 1.001f, -s), 0x1.0p-126f);
  }
}

constexpr int kRdTok = 32;  // tokens of a workgroup's tile
// Above this many open logits of its 1024 a workgroup takes its whole tile by
// fp64 MFMA instead of one dot product a wave and logit: with every third of a
// tile's logits open, 2048 tokens took 140 us by dot products, 112 with the line at
// 256, 76 at 128.  Such tiles are those of rows that are not finite, and of
// expert rows with a strong channel, whose residues are not stored.
constexpr int kRdDense = 128;

// A workgroup owns 32 tokens x 16 NJ experts, its waves the K blocks wave, wave
// + 4, ...  The int32 sums of digit pairs of equal weight share an accumulator
// (five per 16 x 16 tile).  Wave v then finishes the tiles v, v + 4, ..: it adds
// the four waves' sums through LDS and decides each logit.
template <int NJ, int OCC>
__global__ __launch_bounds__(256, OCC) void router_digits_mfma(DigitArgs a) {
  constexpr int kRdExp = 16 * NJ, NT = 2 * NJ, OWN = NT / 4;
  __shared__ i32x4 part[4][3][OWN][5][64];  // [owner][other wave][its tile][weight][lane]
  __shared__ int open[kRdTok * kRdExp];
  __shared__ int n_open;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // linear id b runs on XCD b % 8: a token tile's expert tiles share one
  const int ny = (a.E + kRdExp - 1) / kRdExp, b = blockIdx.x, jb = b >> 3;
  const int t0 = ((jb / ny) * 8 + (b & 7)) * kRdTok, e0 = (jb % ny) * kRdExp;
  if (t0 >= a.T) return;
  const int nk = a.H / 64;
  if (threadIdx.x == 0) n_open = 0;
  // byte 2 i + h: row block i of the tile stores the residues of half h
  uint32_t flags = ldg<uint32_t>(reinterpret_cast<const uint32_t *>(a.xflag) + t0 / 32);
  const int8_t *ap[2], *bp[NJ];
#pragma unroll
  for (int i = 0; i < 2; ++i)
    ap[i] = a.xd + (int64_t)min(t0 / 16 + i, (a.T - 1) / 16) * nk * 3072 + lane * 16;
#pragma unroll
  for (int j = 0; j < NJ; ++j)
    bp[j] = a.wd + (int64_t)min(e0 / 16 + j, (a.E - 1) / 16) * nk * 3072 + lane * 16;
  i32x4 acc[NT][5];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int w = 0; w < 5; ++w) acc[t][w] = i32x4{0, 0, 0, 0};
  // D K blocks in registers, D - 1 in flight: one wave per SIMD has the
  // registers for it, and the blocks come from L2
  constexpr int D = 3;
  i32x4 av[D][2][3], bv[D][NJ][3];
  auto load = [&](int slot, int s) {  // past the end: the last block again, not used
    const int64_t o = (int64_t)min(s, nk - 1) * 3072;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
#pragma unroll
      for (int i = 0; i < 2; ++i) av[slot][i][c] = ldg<i32x4>(ap[i] + o + c * 1024);
#pragma unroll
      for (int j = 0; j < NJ; ++j) bv[slot][j][c] = ldg<i32x4>(bp[j] + o + c * 1024);
    }
  };
  auto multiply = [&](int slot) {
#pragma unroll
    for (int ca = 0; ca < 3; ++ca)
#pragma unroll
      for (int cb = 0; cb < 3; ++cb)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < NJ; ++j)
            acc[i * NJ + j][ca + cb] = __builtin_amdgcn_mfma_i32_16x16x64_i8(
                av[slot][i][ca], bv[slot][j][cb], acc[i * NJ + j][ca + cb], 0, 0, 0);
  };
#pragma unroll
  for (int d = 0; d < D - 1; ++d) load(d, wave + 4 * d);
  int s = wave;
  for (; s + 4 * (D - 1) < nk; s += 4 * D) {
#pragma unroll
    for (int u = 0; u < D; ++u) {
      load((u + D - 1) % D, s + 4 * (u + D - 1));
      __builtin_amdgcn_sched_barrier(0);
      multiply(u);
    }
  }
#pragma unroll
  for (int u = 0; u < D - 1; ++u)
    if (s + 4 * u < nk) multiply(u);
  // The residues' products with w, where a row block has them: the wave's K blocks again.
  const int r = lane & 15, q = lane >> 4;
  const int kh = (nk + 1) / 2;
  flags = __builtin_amdgcn_readfirstlane(flags) & (t0 + 16 < a.T ? 0x01010101u : 0x00000101u);
  const bool residues = flags != 0;
  auto stored = [&](int i, int h) { return (flags >> (16 * i + 8 * h) & 1u) != 0; };
  f32x4 rs[OWN];  // of this wave's tiles
#pragma unroll
  for (int own = 0; own < OWN; ++own) rs[own] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (residues) {
    f32x4 racc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) racc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    const uint16_t *wr[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j)
      wr[j] = a.w + (int64_t)min(e0 + 16 * j + r, a.E - 1) * a.H + 16 * q;
    const u32x4 *xr[2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
      xr[i] = a.xr + (int64_t)min(t0 / 16 + i, (a.T - 1) / 16) * nk * 128 + lane;
    constexpr int R = 3;  // K blocks in registers
    u32x4 xv[R][2][2], wv[R][NJ][2];
    auto fetch = [&](int slot, int kb) {  // past the end: the last block again, not used
      kb = min(kb, nk - 1);
      const int half = kb >= kh ? 1 : 0;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
          xv[slot][i][h] = stored(i, half) ? ldg16(xr[i] + (kb * 2 + h) * 64)
                                                                : u32x4{0u, 0u, 0u, 0u};
#pragma unroll
        for (int j = 0; j < NJ; ++j) wv[slot][j][h] = ldg16(wr[j] + kb * 64 + 8 * h);
      }
    };
#pragma unroll
    for (int d = 0; d < R - 1; ++d) fetch(d, wave + 4 * d);
    int kb = wave;
    while (kb < nk) {
#pragma unroll
      for (int u = 0; u < R; ++u, kb += 4) {
        fetch((u + R - 1) % R, kb + 4 * (R - 1));
        __builtin_amdgcn_sched_barrier(0);
        if (kb >= nk) continue;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
              racc[i * NJ + j] = BF16::mfma16x16x32(xv[u][i][h], wv[u][j][h], racc[i * NJ + j]);
      }
    }
#pragma unroll
    for (int t = 0; t < NT; ++t)
      if ((t & 3) != wave)
        part[t & 3][wave - (wave > (t & 3) ? 1 : 0)][t >> 2][0][lane] =
            __builtin_bit_cast(i32x4, racc[t]);
    __syncthreads();
#pragma unroll
    for (int own = 0; own < OWN; ++own) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (wave == j) rs[own] = racc[4 * own + j];
#pragma unroll
      for (int o = 0; o < 3; ++o)
        rs[own] = rs[own] + __builtin_bit_cast(f32x4, part[wave][o][own][0][lane]);
    }
    __syncthreads();  // part is used again below
  }
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int owner = t & 3;
    if (owner == wave) continue;
#pragma unroll
    for (int w = 0; w < 5; ++w)
      part[owner][wave - (wave > owner ? 1 : 0)][t >> 2][w][lane] = acc[t][w];
  }
  __syncthreads();
#pragma unroll
  for (int own = 0; own < OWN; ++own) {
    // this wave's tile 4 own + wave
    i32x4 v[5];
#pragma unroll
    for (int w = 0; w < 5; ++w) {
      v[w] = acc[4 * own][w];
#pragma unroll
      for (int j = 1; j < 4; ++j)
        if (wave == j) v[w] = acc[4 * own + j][w];
#pragma unroll
      for (int o = 0; o < 3; ++o) v[w] = v[w] + part[wave][o][own][w][lane];
    }
    const int i = (4 * own + wave) / NJ, e = e0 + 16 * ((4 * own + wave) % NJ) + r;
    const RowMeta we = a.wm[min(e, a.E - 1)];
    const float be = a.bias ? a.bias[min(e, a.E - 1)] : 0.0f;
#pragma unroll
    for (int it = 0; it < 4; ++it) {
      const int t = t0 + 16 * i + 4 * q + it;
      if (t >= a.T || e >= a.E) continue;
      const RowMeta xt = a.xm[t];
      long long S = v[4][it];
#pragma unroll
      for (int w = 3; w >= 0; --w) S = S * 256 + v[w][it];
      double L = ldexp((double)S, -(xt.s + we.s)), slack = 0.0;
      double rx = (double)xt.r[0] + xt.r[1];
      if (residues) {
        const bool s0 = stored(i, 0), s1 = stored(i, 1);
        rx = (s0 ? 0x1.0p-11 : 1.0) * xt.r[0] + (s1 ? 0x1.0p-11 : 1.0) * xt.r[1];
        if ((s0 && xt.r[0] != 0.0f) || (s1 && xt.r[1] != 0.0f)) {
          // L in 53 bits, values that count as 2^-100, products below the normal range; a sum
          // that left fp32 opens the logit
          L += ldexp((double)rs[own][it], -xt.s);
          slack = fabs(L) * 0x1.0p-52 + ldexp(0x1.0p-87 * we.m + 0x1.0p-110, -xt.s) + 0.0 * rs[own][it];
        }
      }
      double eps = (rx * we.m + ((double)we.r[0] + we.r[1]) * xt.m) * 1.001 + slack;
      if (S >= (1LL << 53) || S <= -(1LL << 53)) eps += fabs(L) * 0x1.0p-52;
      const float lo = round_bf16((float)(L - eps)), hi = round_bf16((float)(L + eps));
      if (lo == hi && (lo != 0.0f || eps == 0.0))  // an interval around 0 leaves the sign open
        a.logits[(int64_t)t * a.E + e] = a.bias ? lo + be : lo;
      else
        open[atomicAdd(&n_open, 1)] = (t - t0) * kRdExp + (e - e0);
    }
  }
  __syncthreads();
  const int n = n_open;
  if (n > kRdDense) {  // uniform: every tile again, K in 32-wide stages as in route.hip
    for (int own = 0; own < OWN; ++own) {
      const int i = (4 * own + wave) / NJ, e = e0 + 16 * ((4 * own + wave) % NJ) + r;
      const uint16_t *xr = a.x + (int64_t)min(t0 + 16 * i + r, a.T - 1) * a.H + 8 * q;
      const uint16_t *wr = a.w + (int64_t)min(e, a.E - 1) * a.H + 8 * q;
      f64x4 d[2] = {{0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0}};
#pragma unroll 4
      for (int k = 0; k < a.H; k += 32) {
        const u32x4 xv = ldg16(xr + k), wv = ldg16(wr + k);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const uint32_t sh = (j & 1) ? 16u : 0u;
          d[j & 1] = __builtin_amdgcn_mfma_f64_16x16x4f64(
              (double)bf16_bits_to_f32((xv[j >> 1] >> sh) & 0xFFFFu),
              (double)bf16_bits_to_f32((wv[j >> 1] >> sh) & 0xFFFFu), d[j & 1], 0, 0, 0);
        }
      }
#pragma unroll
      for (int it = 0; it < 4; ++it) {
        const int t = t0 + 16 * i + 4 * it + q;  // fp64 tiles: row 4 it + q, column r
        if (t >= a.T || e >= a.E) continue;
        const float l = round_bf16((float)(d[0][it] + d[1][it]));
        a.logits[(int64_t)t * a.E + e] = a.bias ? l + a.bias[e] : l;
      }
    }
    return;
  }
  for (int c = wave; c < n; c += 4) {
    const int t = t0 + open[c] / kRdExp, ee = e0 + open[c] % kRdExp;
    const uint16_t *xr = a.x + (int64_t)t * a.H, *wr = a.w + (int64_t)ee * a.H;
    double d = 0.0;
    for (int k = lane * 8; k < a.H; k += 512) {
      const u32x4 xv = ldg16(xr + k), wv = ldg16(wr + k);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        d = __builtin_fma((double)bf16_bits_to_f32(xv[j] & 0xFFFFu),
                          (double)bf16_bits_to_f32(wv[j] & 0xFFFFu), d);
        d = __builtin_fma((double)bf16_bits_to_f32(xv[j] >> 16),
                          (double)bf16_bits_to_f32(wv[j] >> 16), d);
      }
    }
    d = wave_sum_f64_dpp(d);
    if (lane == 0) {
      float l = round_bf16((float)d);
      if (a.bias) l = l + a.bias[ee];
      a.logits[(int64_t)t * a.E + ee] = l;
    }
  }
}

// Tokens per pass over the workspace, which bounds it (336 MB): as few passes as
// do, of whole tiles and about the same size.  Each further one costs its launches and a
// last round (20000 tokens: 152 us in one pass, 183 in three).
int64_t slice_tokens(int64_t T, int64_t H) {
  const int64_t most = (int64_t(64) << 20) / H;
  const int64_t passes = (T + most - 1) / most;
  return std::min(most, ((T + passes - 1) / passes + 31) / 32 * 32);
}
int64_t row_blocks(int64_t rows) { return (rows + 15) / 16; }
int64_t digit_bytes(int64_t rows, int64_t h) { return row_blocks(rows) * 16 * h * 3; }
int64_t meta_bytes(int64_t rows) { return row_blocks(rows) * 16 * (int64_t)sizeof(RowMeta); }

}  // namespace

int64_t router_digits_bytes(int64_t T, int64_t E, int64_t H) {
  T = std::min(T, (int64_t(64) << 20) / H);
  return digit_bytes(T, H) + digit_bytes(E, H) + row_blocks(T) * 16 * H * 2 + meta_bytes(T) +
         meta_bytes(E) + (T + 31) / 32 * 4;
}

int router_logits_digits(const uint16_t *x, const uint16_t *w, const float *bias, float *logits,
                         int64_t T, int64_t E, int64_t H, void *workspace, hipStream_t st) {
  const int64_t slice = slice_tokens(T, H);
  DigitArgs a{};
  a.w = w;
  a.bias = bias;
  a.xd = static_cast<int8_t *>(workspace);
  a.wd = a.xd + digit_bytes(slice, H);
  a.xr = reinterpret_cast<u32x4 *>(a.wd + digit_bytes(E, H));
  a.xm = reinterpret_cast<RowMeta *>(a.xr + row_blocks(slice) * H * 2);
  a.wm = a.xm + row_blocks(slice) * 16;
  a.xflag = reinterpret_cast<uint8_t *>(a.wm + row_blocks(E) * 16);
  a.E = (int)E;
  a.H = (int)H;
  for (int64_t t = 0; t < T; t += slice) {
    a.x = x + t * H;
    a.logits = logits + t * E;
    a.T = (int)std::min(slice, T - t);
    const unsigned blocks = cdiv(a.T, 16) + (t ? 0 : cdiv(E, 16));  // the weights once
    router_digits_kernel<<<dim3(blocks, 2), kRdWaves * 64, (size_t)H * 32, st>>>(a);
    if (int rc = check_launch("router_digits_kernel")) return rc;
    constexpr int NJ = 2;  // 32 x 32 logits, two workgroups per CU (4, one per CU: no faster)
    const unsigned grid = 8 * cdiv(cdiv(a.T, kRdTok), 8) * cdiv(E, 16 * NJ);
    router_digits_mfma<NJ, 2><<<grid, 256, 0, st>>>(a);
    if (int rc = check_launch("router_digits_mfma")) return rc;
  }
  return LM_OK;
}

}  // namespace lm
