// W8A16 GEMM of few to a few hundred rows (gfx950): the waves of a workgroup
// split K.
//
//   y[m, n] = sum_k x[m, k] * T(q[n, k] * s[n, k/128])      (int8.py:9-37)
//
// With few rows a matrix gives few output tiles, and a workgroup that walks
// all of K alone is one long chain of dependent stages on a mostly idle chip.
// Here a workgroup owns a small tile (16 MS rows x 16 NI columns) and each of
// its kKsWaves waves takes a contiguous 1/kKsWaves of K for the whole tile, so
// the main loop shares nothing between the waves and has no barrier, and each
// activation and weight byte is loaded once per tile.  The fp32 partial tiles
// are added through LDS in wave order.
//
// A wave stages each 64-K unit through LDS of its own: loads in the MFMA
// operand layout would touch 16 rows in every quarter-wave, and their line
// accesses, not their bytes, then bound the kernel (a 64-row tile at K = 2048
// took 10.6 us instead of 8.3, a 64 x 64 one 14.8 instead of 10.6).  Staged, a
// quarter-wave reads two whole lines of activations or four half lines of
// weights.  Then lane l (quarter p = l >> 4) reads k = 16 p .. 16 p + 15 of
// weight column l & 15 and of activation row l & 15, and MFMA step `sub`
// multiplies the halves 16 p + 8 sub .. + 7 of both.
//
// What bounds it: a tile's loads, staging and dequantization in sequence, at
// two waves per SIMD for the largest tiles (10.6 us for one round of 64 x 64
// tiles at K = 2048: [230, 2048] by [4096, 2048] runs at 310 TFLOP/s); the
// smallest calls take one load latency, the wave sum and the launch (2.6 to
// 4.0 us).  Loading the weights non-temporally made every size slower, also
// over 500 MB of them.
#include <utility>

#include "internal.hpp"

namespace lm {
namespace {

constexpr int kKsWaves = 8;
constexpr int kKsUnit = 64;

struct KsArgs {
  const uint16_t *x;
  const int8_t *q;
  const float *s;
  uint16_t *y;
  int64_t M;
  int N, K;
  int nt_count, mt_count;
  bool by_columns;
};

// NU: units per wave (K / 64 / kKsWaves).  D: units held in registers, D - 1 of
// them in flight while one is consumed.
template <typename T, int MS, int NI, int NU, int D>
__global__ __launch_bounds__(kKsWaves * 64) void ksplit_kernel(KsArgs a) {
  static_assert(D >= 1 && D <= NU, "ring depth");
  constexpr int G = NU * kKsWaves * kKsUnit / 128;  // scale groups
  constexpr int BN = 16 * NI;
  constexpr int SC_P = BN * G / 4;  // 16-byte scale pieces of the tile
  constexpr int SC_W = (SC_P + kKsWaves * 64 - 1) / (kKsWaves * 64);
  constexpr int STG = MS * 2048 + NI * 1024;  // staging bytes of one wave
  constexpr int PART = MS * NI * 1024;        // partial tile bytes of one wave
  __shared__ __align__(16) unsigned char smem[kKsWaves * (STG > PART ? STG : PART)];
  __shared__ float scl[G * BN];  // [group][column]
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int p = lane >> 4, r = lane & 15;
  int mt, nt;
  if (!xcd_tile(a.mt_count, a.nt_count, a.by_columns, mt, nt)) return;
  const int64_t m0 = (int64_t)mt * (16 * MS);
  const int n0 = nt * BN;
  const int K = a.K;
  const int k0 = wave * NU * kKsUnit;

  // Rows past M and columns past N re-read the last one; they are not stored.
  u32x4 sreg[SC_W];
#pragma unroll
  for (int j = 0; j < SC_W; ++j) {
    const int piece = (tid + kKsWaves * 64 * j) % SC_P;
    sreg[j] = ldg16(a.s + (int64_t)min(n0 + piece / (G / 4), a.N - 1) * G + (piece % (G / 4)) * 4);
  }
  // Activation load j: row 8 j + lane / 8, 16-byte piece lane & 7 of the
  // row's 128-byte unit (a quarter-wave reads two whole lines); weight load
  // ni: row 16 ni + lane / 4, piece lane & 3 of its 64-byte unit.
  const uint16_t *asrc[2 * MS];
#pragma unroll
  for (int j = 0; j < 2 * MS; ++j)
    asrc[j] = a.x + min(m0 + j * 8 + (lane >> 3), a.M - 1) * K + k0 + 8 * (lane & 7);
  const int8_t *bsrc[NI];
#pragma unroll
  for (int ni = 0; ni < NI; ++ni)
    bsrc[ni] = a.q + (int64_t)min(n0 + ni * 16 + (lane >> 2), a.N - 1) * K + k0 + 16 * (lane & 3);
  u32x4 av[D][2 * MS], bv[D][NI];
  auto load = [&](int slot, int u) {
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) bv[slot][ni] = ldg16(bsrc[ni] + u * kKsUnit);
#pragma unroll
    for (int j = 0; j < 2 * MS; ++j) av[slot][j] = ldg16(asrc[j] + u * kKsUnit);
  };
#pragma unroll
  for (int u = 0; u < D; ++u) load(u, u);
#pragma unroll
  for (int j = 0; j < SC_W; ++j) {
    const int piece = tid + kKsWaves * 64 * j;
    if (piece < SC_P) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        scl[(4 * (piece % (G / 4)) + e) * BN + piece / (G / 4)] = __uint_as_float(sreg[j][e]);
    }
  }
  // lgkmcnt(0): the scales are written; the loads stay in flight
  __builtin_amdgcn_s_waitcnt(0xC07F);
  asm volatile("s_barrier" ::: "memory");

  // The wave's own staging area.  Chunks are XOR-swizzled by row so that the
  // 16 rows read by a quarter-wave fall in 16 different bank groups.
  unsigned char *sa = smem + wave * STG;
  unsigned char *sb = sa + MS * 2048;
  unsigned char *awr = sa + (lane >> 3) * 128;
  unsigned char *bwr = sb + (lane >> 2) * 64 + (((lane & 3) ^ (lane >> 4)) * 16);
  f32x4 acc[MS][NI];
#pragma unroll
  for (int mi = 0; mi < MS; ++mi)
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) acc[mi][ni] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    const int slot = u % D;
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) *reinterpret_cast<u32x4 *>(bwr + ni * 1024) = bv[slot][ni];
#pragma unroll
    for (int j = 0; j < 2 * MS; ++j) {
      const int row = (8 * j + (lane >> 3)) & 15;
      *reinterpret_cast<u32x4 *>(awr + j * 1024 + (((lane & 7) ^ (row >> 1)) * 16)) = av[slot][j];
    }
    wave_lds_sync();
    if (u + D < NU) load(slot, u + D);
    u32x4 bq[NI];
    float sc[NI];
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) {
      bq[ni] = *reinterpret_cast<const u32x4 *>(sb + ni * 1024 + r * 64 + ((p ^ (r >> 2)) * 16));
      sc[ni] = scl[((k0 + u * kKsUnit) >> 7) * BN + ni * 16 + r];
    }
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
      u32x4 af[MS];
#pragma unroll
      for (int mi = 0; mi < MS; ++mi)
        af[mi] = *reinterpret_cast<const u32x4 *>(sa + mi * 2048 + r * 128 +
                                                  (((2 * p + sub) ^ (r >> 1)) * 16));
#pragma unroll
      for (int ni = 0; ni < NI; ++ni) {
        const u32x4 w = dequant8s<T>(uint2{bq[ni][2 * sub], bq[ni][2 * sub + 1]}, sc[ni]);
#pragma unroll
        for (int mi = 0; mi < MS; ++mi) acc[mi][ni] = T::mfma16x16x32(af[mi], w, acc[mi][ni]);
      }
    }
    wave_lds_sync();  // every lane's reads before the next unit is staged
  }
  __syncthreads();  // the partial tiles reuse the staging areas
  f32x4(*part)[MS * NI][64] = reinterpret_cast<f32x4(*)[MS * NI][64]>(smem);
#pragma unroll
  for (int mi = 0; mi < MS; ++mi)
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) part[wave][mi * NI + ni][lane] = acc[mi][ni];
  __syncthreads();
  // MFMA 16x16 layout: lane l holds column l & 15, rows 4 (l >> 4) + it.
  for (int c = tid; c < MS * NI * 64; c += kKsWaves * 64) {
    const int ln = c & 63, t = c >> 6;
    f32x4 v = part[0][t][ln];
#pragma unroll
    for (int w = 1; w < kKsWaves; ++w) v = v + part[w][t][ln];
    const int n = n0 + (t % NI) * 16 + (ln & 15);
    const int64_t m = m0 + (t / NI) * 16 + (ln >> 4) * 4;
    if (n >= a.N) continue;
#pragma unroll
    for (int it = 0; it < 4; ++it)
      if (m + it < a.M) a.y[(m + it) * a.N + n] = T::from_f32(v[it]);
  }
}

template <typename T, int MS, int NI, int NU>
int launch_ks(KsArgs a, hipStream_t st) {
  constexpr int PER = NI * 4 + MS * 8;  // registers of one unit
  constexpr int D0 = PER * 4 + MS * NI * 4 <= 150 ? 4 : PER * 3 + MS * NI * 4 <= 190 ? 3 : 2;
  constexpr int D = D0 < NU ? D0 : NU;
  a.mt_count = (int)cdiv(a.M, 16 * MS);
  a.nt_count = (int)cdiv(a.N, 16 * NI);
  const int64_t grid = xcd_grid(a.mt_count, a.nt_count, a.by_columns);
  LM_REQUIRE(grid < (int64_t(1) << 31), LM_EINVAL, "problem too large for one launch");
  ksplit_kernel<T, MS, NI, NU, D><<<(unsigned)grid, kKsWaves * 64, 0, st>>>(a);
  return check_launch("ksplit_kernel");
}

constexpr int kKsCount = 8;
constexpr int kKsShapes[kKsCount][2] = {{1, 1}, {1, 2}, {1, 4}, {2, 2},
                                        {3, 2}, {4, 2}, {4, 4}, {6, 2}};

template <typename T, int NU, int... I>
int launch_shape(const KsArgs &a, int shape, hipStream_t st, std::integer_sequence<int, I...>) {
  int rc = LM_OK;
  (void)((shape == I && (rc = launch_ks<T, kKsShapes[I][0], kKsShapes[I][1], NU>(a, st), true)) ||
         ...);
  return rc;
}

template <typename T>
int launch_k(const KsArgs &a, int shape, hipStream_t st) {
  constexpr auto all = std::make_integer_sequence<int, kKsCount>{};
  return a.K == 512    ? launch_shape<T, 1>(a, shape, st, all)
         : a.K == 2048 ? launch_shape<T, 4>(a, shape, st, all)
                       : launch_shape<T, 8>(a, shape, st, all);
}

}  // namespace

// The tile shape with the smallest estimated time in us, for 8 XCDs of 32 CUs
// that work through their tiles in whole rounds.  A call takes 1.8 us, and a
// round 0.8 us per 16 rows or columns and 2048 of K (loads, staging,
// dequantization) plus 0.18 us per 16 x 16 tile (the sum over the waves):
// measured at K = 512, 2048 and 4096 from 4.7 us (1 x 1, one round) to 36 us (4
// x 4 at K = 4096, two rounds; 10 of 800 sizes further than 20 % off).  A tile's
// rows are all loaded, so a short last row tile counts whole.  Where the
// activations fit an XCD's 4 MB L2, every XCD may read all of them ([512, 2048]
// by [512, 2048]: 6.5 us by columns, 7.0 by rows in one round both); beyond it
// that costs a tenth.
KsPlan ksplit_plan(int64_t m, int64_t n, int64_t k) {
  KsPlan best{-1, 0.0, 0, 0, false};
  if (k != 512 && k != 2048 && k != 4096) return best;
  const bool in_l2 = 2 * m * k <= (4 << 20);
  for (int i = 0; i < kKsCount; ++i) {
    const int ms = kKsShapes[i][0], ni = kKsShapes[i][1];
    const int64_t mt = cdiv(m, 16 * ms), nt = cdiv(n, 16 * ni);
    const double round = 0.18 * ms * ni + 0.8 * (ms + ni) * (double)k / 2048.0;
    // a small call's host side: no deal is better than one tile on every CU in turn
    if (best.shape >= 0 && 1.8 + (double)((mt * nt + 255) / 256) * round >= best.cost) continue;
    const XcdDeal deal = xcd_deal(m, n, mt, nt, 16 * ms, false, in_l2 ? 0 : 2);
    const double cost = 1.8 + deal.rounds * round * (deal.by_columns && !in_l2 ? 1.1 : 1.0);
    if (best.shape < 0 || cost < best.cost)
      best = KsPlan{i, cost, 16 * ms, 16 * ni, deal.by_columns};
  }
  return best;
}

int w8a16_ksplit(const KsPlan &plan, const void *x, const int8_t *q, const float *s, void *y,
                 int64_t m, int64_t n, int64_t k, int dtype, hipStream_t st) {
  KsArgs a{};
  a.x = static_cast<const uint16_t *>(x);
  a.q = q;
  a.s = s;
  a.y = static_cast<uint16_t *>(y);
  a.M = m;
  a.N = (int)n;
  a.K = (int)k;
  a.by_columns = plan.by_columns;
  return dtype == LM_BF16 ? launch_k<BF16>(a, plan.shape, st) : launch_k<FP16>(a, plan.shape, st);
}

}  // namespace lm
