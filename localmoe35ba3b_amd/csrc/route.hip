// Routing side of the MoE block:
//   router logits (fp64 accumulation, bf16-rounded) + top-k + softmax renorm
//                                                   (HF:768-776)
//   device route plan: stable token sort / permute  (gpu_routes.py:17-63)
//   ordered combines for decode and prefill         (int8.py:240-250, prefill.py:37-49)
//   SwiGLU glue, RMSNorm                            (HF:715, HF:801-815)
#include <algorithm>

#include "internal.hpp"

namespace lm {

// ============================================================ router logits
// logit[t, e] = f32(bf16(f32(sum_k f64(x[t,k]) * f64(w[e,k])))) (+ bias[e]).
// Products of two bf16 values are exact in fp64 and the fp64 sum of 2048 of
// them is exact unless operands span more than ~37 binary orders of
// magnitude, so the result does not depend on the summation order; the
// kernels below may therefore permute k freely.

// Small token counts (decode): one wave per (expert, token-block), VALU fp64.
template <int MT>
__global__ __launch_bounds__(256) void router_logits_gemv(const uint16_t *__restrict__ x,
                                                          const uint16_t *__restrict__ w,
                                                          const float *__restrict__ bias,
                                                          float *__restrict__ logits, int T,
                                                          int E, int H) {
  const int lane = threadIdx.x & 63;
  const int e = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (e >= E) return;
  double acc[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) acc[m] = 0.0;
  const uint16_t *wr = w + (int64_t)e * H;
  for (int k0 = lane * 8; k0 < H; k0 += 512) {
    const u32x4 wv = ldg16(wr + k0);
    double wd[8];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      wd[2 * j] = (double)bf16_bits_to_f32(wv[j] & 0xFFFFu);
      wd[2 * j + 1] = (double)bf16_bits_to_f32(wv[j] >> 16);
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      if (m < T) {
        const u32x4 xv = ldg16(x + (int64_t)m * H + k0);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          acc[m] = __builtin_fma((double)bf16_bits_to_f32(xv[j] & 0xFFFFu), wd[2 * j], acc[m]);
          acc[m] = __builtin_fma((double)bf16_bits_to_f32(xv[j] >> 16), wd[2 * j + 1], acc[m]);
        }
      }
    }
  }
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    if (m < T) {
      const double s = wave_sum_f64_dpp(acc[m]);
      if (lane == 0) {
        float l = round_bf16((float)s);
        if (bias) l = l + bias[e];
        logits[(int64_t)m * E + e] = l;
      }
    }
  }
}

// More tokens: v_mfma_f64_16x16x4f64.  A workgroup owns 16 tokens x 16 NE
// experts and its waves split K (K in 32-wide stages dealt round robin, so any
// number of stages splits evenly); the fp64 partial tiles are added through
// LDS.  Lane quad q supplies k = k0 + 8 q + j at MFMA step j (the same
// permutation for both operands), so one 16-byte load per operand row feeds 8
// MFMA steps.  Two stages are held in registers, and even and odd K-steps
// accumulate into separate fp64 tiles.
//
// Bound: the fp64 matrix rate (64 cycles per MFMA and SIMD: 27 us for 2048
// tokens x 256 experts x 2048; 7 us for one 16 x 32 tile on a CU).  With all of
// K in one wave and 32 x 128 experts per workgroup a call of 9 tokens took as
// long as one of 2048 (46 us, top-k included); split it takes 12 us up to 256
// tokens, 17 up to 512, 27 up to 1024 and 45 at 2048.
constexpr int kRouterWaves = 4;
template <int NE>
__global__ __launch_bounds__(kRouterWaves * 64) void router_logits_mfma(
    const uint16_t *__restrict__ x, const uint16_t *__restrict__ w, const float *__restrict__ bias,
    float *__restrict__ logits, int T, int E, int H) {
  constexpr int NW = kRouterWaves, D = 2;
  __shared__ f64x4 part[NW][NE][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int t0 = blockIdx.x * 16;
  const int e0 = blockIdx.y * 16 * NE;
  const int q = lane >> 4;
  const int r = lane & 15;
  const uint16_t *xa = x + (int64_t)min(t0 + r, T - 1) * H + q * 8;
  const uint16_t *wb[NE];
#pragma unroll
  for (int c = 0; c < NE; ++c) wb[c] = w + (int64_t)min(e0 + 16 * c + r, E - 1) * H + q * 8;
  f64x4 acc[2][NE];
#pragma unroll
  for (int c = 0; c < NE; ++c) acc[0][c] = acc[1][c] = f64x4{0.0, 0.0, 0.0, 0.0};
  u32x4 ra[D], rb[D][NE];
  // this wave's stages: k = 32 (NW i + wave), i < stages; past the end the
  // row's last stage is re-read and never consumed
  const int stages = (H / 32 - wave + NW - 1) / NW;
  auto load = [&](int slot, int i) {
    const int k = min(32 * (NW * i + wave), H - 32);
    ra[slot] = ldg16(xa + k);
#pragma unroll
    for (int c = 0; c < NE; ++c) rb[slot][c] = ldg16(wb[c] + k);
  };
  auto step = [&](u32x4 av, const u32x4 (&bv)[NE]) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint32_t sh = (j & 1) ? 16u : 0u;
      const double a = (double)bf16_bits_to_f32((av[j >> 1] >> sh) & 0xFFFFu);
#pragma unroll
      for (int c = 0; c < NE; ++c) {
        const double b = (double)bf16_bits_to_f32((bv[c][j >> 1] >> sh) & 0xFFFFu);
        acc[j & 1][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc[j & 1][c], 0, 0, 0);
      }
    }
  };
#pragma unroll
  for (int d = 0; d < D; ++d) load(d, d);
  int i = 0;
  for (; i + D <= stages; i += D) {
#pragma unroll
    for (int u = 0; u < D; ++u) {
      const u32x4 av = ra[u];
      u32x4 bv[NE];
#pragma unroll
      for (int c = 0; c < NE; ++c) bv[c] = rb[u][c];
      load(u, i + u + D);
      step(av, bv);
    }
  }
#pragma unroll
  for (int u = 0; u < D; ++u)
    if (i + u < stages) step(ra[u], rb[u]);
#pragma unroll
  for (int c = 0; c < NE; ++c) part[wave][c][lane] = acc[0][c] + acc[1][c];
  __syncthreads();
  if (wave >= NE) return;  // wave c finishes 16 experts
  f64x4 v = part[0][wave][lane];
#pragma unroll
  for (int j = 1; j < NW; ++j) v = v + part[j][wave][lane];
  // D layout of the f64 16x16x4 MFMA: lane holds column (lane & 15) and
  // rows (lane >> 4) + 4 i, i = 0..3 (unlike the 4 (lane >> 4) + i rows of the
  // 32-bit-output 16x16 MFMAs).
  const int e = e0 + 16 * wave + r;
  if (e >= E) return;
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const int t = t0 + q + 4 * m;
    if (t >= T) continue;
    float l = round_bf16((float)v[m]);
    if (bias) l = l + bias[e];
    logits[(int64_t)t * E + e] = l;
  }
}

// ============================================================ top-k
__global__ __launch_bounds__(256) void topk_kernel(const float *__restrict__ logits, int T, int E,
                                                   int K, int64_t *__restrict__ ids,
                                                   uint16_t *__restrict__ weights) {
  __shared__ unsigned long long scratch[4][kTopkScratch];
  const int lane = threadIdx.x & 63;
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= T) return;
  topk_wave(logits + (int64_t)t * E, E, K, lane, scratch[threadIdx.x >> 6], ids + (int64_t)t * K,
            weights + (int64_t)t * K);
}

int router_logits(const uint16_t *x, const uint16_t *w, const float *bias, float *logits,
                  int64_t T, int64_t E, int64_t H, hipStream_t st) {
  if (T <= 6) {  // 11.5 us and rising with T; the MFMA tile takes 12
    const unsigned g = cdiv(E, 4);
    if (T == 1)
      router_logits_gemv<1><<<g, 256, 0, st>>>(x, w, bias, logits, (int)T, (int)E, (int)H);
    else
      router_logits_gemv<8><<<g, 256, 0, st>>>(x, w, bias, logits, (int)T, (int)E, (int)H);
  } else if (cdiv(T, 16) * cdiv(E, 16) <= 256) {  // narrow tiles while they fit the CUs once
    router_logits_mfma<1><<<dim3(cdiv(T, 16), cdiv(E, 16)), kRouterWaves * 64, 0, st>>>(
        x, w, bias, logits, (int)T, (int)E, (int)H);
  } else {
    router_logits_mfma<2><<<dim3(cdiv(T, 16), cdiv(E, 32)), kRouterWaves * 64, 0, st>>>(
        x, w, bias, logits, (int)T, (int)E, (int)H);
  }
  return check_launch("router_logits");
}

// Calls of more than kDigitTokens tokens take the int8 digits where the caller
// brings a workspace for them (with the top-k, 21 us against 26 at 513 tokens,
// 31 against 45 at 2048, 46 against 83 at 4096; up to 512 tokens the fp64 tiles
// run in one round, 17 us).
constexpr int64_t kDigitTokens = 512;
static bool router_digits_serves(int64_t T, int64_t H) {
  return T > kDigitTokens && H % 256 == 0 && H <= 4096;
}

// Whether the digits are the faster form, by estimates in us fitted over 480
// sizes of 513 to 16384 tokens, 16 to 256 experts and hidden 256 to 4096, where
// the choice is 0.1 % slower than the better of both.  The fp64 tiles cost their
// rounds of 16 x 32 on 256 CUs, the digits two launches and their passes, so few
// experts or a short row leave nothing to gain: 2048 tokens and 256 experts take
// 32 us against 46 at hidden 2048, 23 against 27 at 1024, 16 against 13 at 256; 32
// experts at 2048 hidden 26 against 12.  The margin is for rows with large
// residues, which cost the digits up to a third more.
static bool router_digits_pay(int64_t T, int64_t E, int64_t H) {
  const double h = (double)H / 1024.0;
  const int64_t tiles = ((T + 15) / 16) * ((E + 31) / 32);
  const double fp64 = 7.0 + 4.75 * h * (double)((tiles + 255) / 256);
  const double more = (double)std::max<int64_t>(T - 1024, 0) / 1024.0;
  const double digits = 12.0 + 4.2 * h + more * (0.8 + h * (1.75 + 0.0085 * (double)E));
  return H >= 512 && fp64 > 1.05 * digits;
}

int router_topk(const float *logits, int64_t T, int64_t E, int64_t K, int64_t *ids,
                uint16_t *weights, hipStream_t st) {
  topk_kernel<<<cdiv(T, 4), 256, 0, st>>>(logits, (int)T, (int)E, (int)K, ids, weights);
  return check_launch("topk_kernel");
}

// ============================================================ route plan
// Stable counting sort of the flat route ids by expert, in one launch without
// communication between workgroups.  Workgroup b ranks the routes of its own
// tokens; to place them it needs the count of every expert over all routes
// and over the routes before its own, which it takes itself: every workgroup
// reads all ids (128 KB for 2048 tokens x 8, served by L2) into LDS
// histograms.  A single workgroup had to rank all routes one 64-lane chunk
// after the other: 40 us for 2048 x 8 and 1644 us for 60000 x 8, against 8 and
// 102 us.  With up to 1024 routes per workgroup a wave ranks one chunk; a
// call then costs its launch, the ids' latency and four barriers (5.0 us for
// one slice).
//
// Within the slice, wave w owns a contiguous run of routes and walks it 64 at
// a time: lanes holding the same expert id find each other with eight ballots
// over the id bits, so a route's position is the wave's running position of
// that expert plus the equal ids in lower lanes.  The running positions start
// at the expert's offset, plus its routes before the slice, plus those of the
// slice's earlier waves.  A slice holds whole tokens, and a route's place in
// its token's ascending order is counted from the token's ids.  ids are
// clamped into [0, E), so a malformed id can never index out of bounds.  One
// further workgroup, without routes, writes the tile table.
constexpr int kPlanThreads = 1024;
constexpr int kPlanWaves = kPlanThreads / 64;
constexpr int kPlanBlocks = 255;  // at most this many slices, of at least kPlanThreads routes

// Exclusive scan of one value per thread over the first 256 threads of a
// 1024-thread block (the others pass 0); returns the prefix, *total = sum.
__device__ int block_scan_256(int v, int *scratch, int *total) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  int incl = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int u = __shfl_up(incl, o, 64);
    if (lane >= o) incl += u;
  }
  if (lane == 63 && wave < 4) scratch[wave] = incl;
  __syncthreads();
  int base = 0;
  for (int i = 0; i < wave && i < 4; ++i) base += scratch[i];
  const int all = scratch[0] + scratch[1] + scratch[2] + scratch[3];
  __syncthreads();
  *total = all;
  return base + incl - v;
}

__global__ __launch_bounds__(1024) void route_plan_kernel(const int64_t *__restrict__ ids, int T,
                                                          int K, int E, int bm, int tokens_per_block,
                                                          int64_t *__restrict__ pos,
                                                          int64_t *__restrict__ table,
                                                          int max_tiles,
                                                          int64_t *__restrict__ ordered,
                                                          int64_t *__restrict__ slots) {
  __shared__ int count[2][256];  // routes before the slice / from its start on
  __shared__ int wpos[kPlanWaves][256];
  __shared__ int offs[257], tends[256], scratch[4];
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = t >> 6;
  const int R = T * K;
  const bool tiles = blockIdx.x + 1 == gridDim.x;
  const int lo = tiles ? R : min((int)blockIdx.x * tokens_per_block, T) * K;
  const int hi = tiles ? R : min(((int)blockIdx.x + 1) * tokens_per_block, T) * K;
  const unsigned long long lt = (1ull << lane) - 1ull;
  auto eid = [&](int i) -> int {
    const int64_t e = ids[i];
    return (int)(e < 0 ? 0 : (e >= E ? E - 1 : e));
  };
  for (int i = t; i < 512; i += kPlanThreads) count[i >> 8][i & 255] = 0;
#pragma unroll
  for (int i = 0; i < kPlanWaves * 256 / kPlanThreads; ++i)
    wpos[(t + i * kPlanThreads) >> 8][t & 255] = 0;
  __syncthreads();

  // Counts: all routes, and per wave those of its own run.
#pragma unroll 8
  for (int r = t; r < R; r += kPlanThreads) atomicAdd(&count[r < lo ? 0 : 1][eid(r)], 1);
  const int run = ((hi - lo + kPlanWaves - 1) / kPlanWaves + 63) & ~63;
  const int wlo = min(lo + wave * run, hi), whi = min(wlo + run, hi);
  for (int r = wlo + lane; r < whi; r += 64) atomicAdd(&wpos[wave][eid(r)], 1);
  __syncthreads();
  int all;
  const int before = t < 256 ? count[0][t] : 0;
  const int ex = block_scan_256(t < E ? before + count[1][t] : 0, scratch, &all);
  if (t < 256) {
    offs[t] = ex;
    int p = ex + before;
    for (int w = 0; w < kPlanWaves; ++w) {
      const int c = wpos[w][t];
      wpos[w][t] = p;
      p += c;
    }
  }
  if (t == 0) offs[256] = all;
  __syncthreads();

  // Sorted position p of each route of the slice, and its place i in its
  // token: slots = argsort(ids, dim=1, stable), ordered[t, i] = p.
  for (int base = wlo; base < whi; base += 64) {
    const int r = base + lane;
    const bool valid = r < whi;
    const int e = valid ? eid(r) : 0;
    unsigned long long same = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const unsigned long long bit = __ballot(valid && ((e >> b) & 1));
      same &= ((e >> b) & 1) ? bit : ~bit;
    }
    const int in_chunk = __popcll(same & lt);
    const int first = wpos[wave][e];
    wave_lds_sync();
    if (valid && in_chunk == 0) wpos[wave][e] = first + __popcll(same);
    wave_lds_sync();
    if (valid) {
      const int p = first + in_chunk;
      const int tok = r / K, j = r - tok * K;
      int i = 0;
#pragma unroll 8
      for (int jj = 0; jj < K; ++jj) {
        const int o = eid(tok * K + jj);
        i += (o < e || (o == e && jj < j)) ? 1 : 0;
      }
      pos[p] = tok;
      slots[(int64_t)tok * K + i] = j;
      ordered[(int64_t)tok * K + i] = p;
    }
  }
  if (!tiles) return;

  // Tile table (gpu_routes._table): tiles of bm rows, expert by expert.
  const int nt = t < E ? (offs[t + 1] - offs[t] + bm - 1) / bm : 0;
  int ntot;
  const int tex = block_scan_256(nt, scratch, &ntot);
  if (t < 256) tends[t] = tex + nt;
  __syncthreads();
  for (int i = t; i < max_tiles; i += kPlanThreads) {
    int64_t ex_ = 0, st_ = 0, sp_ = 0;
    if (i < ntot) {
      int l = 0, h = E;
      while (l < h) {
        const int mid = (l + h) >> 1;
        if (tends[mid] <= i) l = mid + 1;
        else h = mid;
      }
      const int prior = l > 0 ? tends[l - 1] : 0;
      ex_ = l;
      st_ = offs[l] + (int64_t)(i - prior) * bm;
      sp_ = offs[l + 1];
    }
    table[i * 3] = ex_;
    table[i * 3 + 1] = st_;
    table[i * 3 + 2] = sp_;
  }
}

int route_plan(const int64_t *ids, int64_t T, int64_t K, int64_t E, int64_t bm, int64_t *pos,
               int64_t *table, int64_t max_tiles, int64_t *ordered, int64_t *slots,
               hipStream_t st) {
  const int64_t want = std::min<int64_t>((T * K + kPlanThreads - 1) / kPlanThreads, kPlanBlocks);
  const int64_t per = (T + want - 1) / want;
  const unsigned blocks = cdiv(T, per);
  route_plan_kernel<<<blocks + 1, kPlanThreads, 0, st>>>(ids, (int)T, (int)K, (int)E, (int)bm,
                                                         (int)per, pos, table, (int)max_tiles,
                                                         ordered, slots);
  return check_launch("route_plan_kernel");
}

// ============================================================ combines
__device__ __forceinline__ float load_weight(const void *w, int dtype, int64_t i) {
  if (dtype == LM_FP32) return static_cast<const float *>(w)[i];
  const uint16_t b = static_cast<const uint16_t *>(w)[i];
  return dtype == LM_FP16 ? f16_bits_to_f32(b) : bf16_bits_to_f32(b);
}

// int8._ordered_reduce: ascending table order, rounding to the output dtype T
// at every step.  A table slot outside [0, E) is clamped into it.
template <typename T>
__global__ __launch_bounds__(256) void ordered_reduce_kernel(const uint16_t *__restrict__ v,
                                                             const int64_t *__restrict__ table,
                                                             const void *w, int w_dtype,
                                                             uint16_t *__restrict__ y, int N,
                                                             int E) {
  const int n = blockIdx.x * 256 + threadIdx.x;
  if (n >= N) return;
  float acc = 0.0f;
  for (int e = 0; e < E; ++e) {
    const int64_t slot = clamp_index(table[e * 5 + 4], E);
    const float wt = load_weight(w, w_dtype, slot);
    const float val = T::round(T::to_f32(v[(int64_t)e * N + n]) * wt);
    acc = T::round(acc + val);
  }
  y[n] = T::from_f32(acc);
}

// prefill._reduce: per token, routes in ascending expert order, rounding to
// T at every step.  Routes are clamped into [0, tokens * K), slots into [0, K).
// A thread owns VEC adjacent columns (one 16-byte load per route at VEC = 8)
// and requests the rows of B routes before it adds the first.  Two are enough with
// the many waves of a call, and fewer registers and repeated rows than eight:
// 2048 tokens x 8 routes x 2048 columns take 57 us with 2-byte loads route by
// route, 17.6 with eight in flight, 14.2 with two (8192 tokens 274, 49 and 50 us,
// 6 TB/s); one route of 4096 columns 20.8, 14.1 and 7.5.
template <typename T, int VEC>
__global__ __launch_bounds__(256) void routed_reduce_kernel(const uint16_t *__restrict__ v,
                                                            const int64_t *__restrict__ ordered,
                                                            const int64_t *__restrict__ slots,
                                                            const void *w, int w_dtype,
                                                            uint16_t *__restrict__ y, int N,
                                                            int K, int64_t routes) {
  constexpr int B = VEC == 8 ? 2 : 1;  // routes per batch
  const int tok = blockIdx.y;
  const int n = (blockIdx.x * blockDim.x + threadIdx.x) * VEC;
  if (n >= N) return;
  float acc[VEC];
#pragma unroll
  for (int c = 0; c < VEC; ++c) acc[c] = 0.0f;
  for (int i0 = 0; i0 < K; i0 += B) {
    // routes past the last re-read it and are not added
    u32x4 raw[B];
    float wt[B];
#pragma unroll
    for (int i = 0; i < B; ++i) {
      const int64_t at = (int64_t)tok * K + min(i0 + i, K - 1);
      const uint16_t *p = v + clamp_index(ordered[at], routes) * N + n;
      if constexpr (VEC == 8)
        raw[i] = ldg16(p);
      else
        raw[i][0] = ldg<uint16_t>(p);
      wt[i] = load_weight(w, w_dtype, (int64_t)tok * K + clamp_index(slots[at], K));
    }
#pragma unroll
    for (int i = 0; i < B; ++i) {
      if (i0 + i < K) {
#pragma unroll
        for (int c = 0; c < VEC; ++c)
          acc[c] = T::round(
              acc[c] + T::round(T::to_f32((raw[i][c >> 1] >> (16 * (c & 1))) & 0xFFFFu) * wt[i]));
      }
    }
  }
  uint16_t *yp = y + (int64_t)tok * N + n;
  if constexpr (VEC == 8) {
    u32x4 out;
#pragma unroll
    for (int c = 0; c < 4; ++c) out[c] = T::pack2(acc[2 * c], acc[2 * c + 1]);
    *reinterpret_cast<u32x4 *>(yp) = out;
  } else {
    *yp = T::from_f32(acc[0]);
  }
}

template <typename T>
static int routed_reduce(const uint16_t *v, const int64_t *ordered, const int64_t *slots,
                         const void *w, int w_dtype, uint16_t *y, int64_t tokens, int64_t n,
                         int64_t top_k, hipStream_t st) {
  // whole 16-byte pieces where the rows allow them, else one column a thread; rows of
  // fewer than 256 columns too, whose pieces fill no wave (16 routes of 128 columns, 300
  // tokens: 6.5 us, with pieces 9.0)
  const bool wide = n >= 256 && n % 8 == 0 &&
                    ((reinterpret_cast<uintptr_t>(v) | reinterpret_cast<uintptr_t>(y)) & 15) == 0;
  const int64_t threads = wide ? n / 8 : n;
  const unsigned block = threads <= 64 ? 64 : threads <= 128 ? 128 : 256;
  const dim3 grid(cdiv(threads, block), (unsigned)tokens);
  if (wide)
    routed_reduce_kernel<T, 8><<<grid, block, 0, st>>>(v, ordered, slots, w, w_dtype, y, (int)n,
                                                       (int)top_k, tokens * top_k);
  else
    routed_reduce_kernel<T, 1><<<grid, block, 0, st>>>(v, ordered, slots, w, w_dtype, y, (int)n,
                                                       (int)top_k, tokens * top_k);
  return check_launch("routed_reduce_kernel");
}

// SwiGLU glue on a [rows, 2*half] gate_up tensor of dtype T.
template <typename T>
__global__ __launch_bounds__(256) void swiglu_kernel(const uint16_t *__restrict__ gu,
                                                     uint16_t *__restrict__ h, int64_t rows,
                                                     int64_t half) {
  const int64_t total = rows * half;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * 256) {
    const int64_t r = i / half, c = i - r * half;
    const float g = T::to_f32(gu[r * 2 * half + c]);
    const float u = T::to_f32(gu[r * 2 * half + half + c]);
    h[i] = T::from_f32(T::round(silu_f32(g)) * u);
  }
}

// RMSNorm (HF:807-815) on rows of n bf16 values; one block per row.  The sum
// of squares uses a fixed tree - thread t sums its contiguous chunk of
// ceil(n/256) elements in order, a 64-lane xor butterfly per wave, then the
// four wave sums left to right - and r = 1 / sqrt(mean + eps) with IEEE
// sqrt and division, so the result is reproducible bit for bit.
__global__ __launch_bounds__(256) void rmsnorm_kernel(const uint16_t *__restrict__ x,
                                                      const float *__restrict__ w,
                                                      uint16_t *__restrict__ y, int n,
                                                      float eps) {
  __shared__ float red[4];
  const uint16_t *xr = x + (int64_t)blockIdx.x * n;
  uint16_t *yr = y + (int64_t)blockIdx.x * n;
  const int per = (n + 255) / 256;
  const int lo = min(threadIdx.x * per, n), hi = min(lo + per, n);
  float ss = 0.0f;
  for (int i = lo; i < hi; ++i) {
    const float v = bf16_bits_to_f32(xr[i]);
    ss += v * v;
  }
  ss = wave_sum_f32(ss);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
  __syncthreads();
  const float tot = red[0] + red[1] + red[2] + red[3];
  const float r = 1.0f / sqrtf(tot / (float)n + eps);
  for (int i = lo; i < hi; ++i) {
    float v = bf16_bits_to_f32(xr[i]) * r;
    if (w) v = v * (1.0f + w[i]);
    yr[i] = f32_to_bf16_bits(v);
  }
}

}  // namespace lm

using namespace lm;

extern "C" int64_t lm_router_workspace_bytes(int64_t tokens, int64_t experts, int64_t hidden) {
  if (experts < 1 || experts > 256 || hidden < 1 || !router_digits_serves(tokens, hidden)) return 0;
  return router_digits_bytes(tokens, experts, hidden);
}

extern "C" int lm_router_workspace_pays(int64_t tokens, int64_t experts, int64_t hidden) {
  return lm_router_workspace_bytes(tokens, experts, hidden) > 0 &&
         router_digits_pay(tokens, experts, hidden);
}

extern "C" int lm_router_topk_ws(const void *x, const void *w, const float *bias, float *logits,
                                 int64_t *ids, void *weights, int64_t tokens, int64_t experts,
                                 int64_t hidden, int64_t top_k, void *workspace,
                                 int64_t workspace_bytes, void *stream) {
  LM_REQUIRE(experts >= 1 && experts <= 256, LM_EINVAL, "router supports 1..256 experts");
  LM_REQUIRE(top_k >= 1 && top_k <= 16 && top_k <= experts, LM_EINVAL, "invalid top_k");
  LM_REQUIRE(hidden > 0 && hidden % 32 == 0, LM_EINVAL, "hidden must be a multiple of 32");
  LM_REQUIRE(tokens >= 0, LM_EINVAL, "invalid token count");
  if (tokens == 0) return LM_OK;
  LM_REQUIRE(x && w && logits && ids && weights, LM_EINVAL, "null pointer");
  hipStream_t st = as_stream(stream);
  const uint16_t *xp = static_cast<const uint16_t *>(x), *wp = static_cast<const uint16_t *>(w);
  int rc;
  if (workspace && router_digits_serves(tokens, hidden)) {
    LM_REQUIRE(workspace_bytes >= router_digits_bytes(tokens, experts, hidden), LM_ENOMEM,
               "router workspace too small (lm_router_workspace_bytes)");
    LM_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 15) == 0, LM_EINVAL,
               "router workspace must be 16-byte aligned");
    rc = router_logits_digits(xp, wp, bias, logits, tokens, experts, hidden, workspace, st);
  } else {
    rc = router_logits(xp, wp, bias, logits, tokens, experts, hidden, st);
  }
  if (rc) return rc;
  return router_topk(logits, tokens, experts, top_k, ids, static_cast<uint16_t *>(weights), st);
}

extern "C" int lm_router_topk(const void *x, const void *w, const float *bias, float *logits,
                              int64_t *ids, void *weights, int64_t tokens, int64_t experts,
                              int64_t hidden, int64_t top_k, void *stream) {
  return lm_router_topk_ws(x, w, bias, logits, ids, weights, tokens, experts, hidden, top_k,
                           nullptr, 0, stream);
}

extern "C" int lm_route_plan(const int64_t *ids, int64_t tokens, int64_t top_k, int64_t experts,
                             int64_t bm, int64_t *pos, int64_t *table, int64_t max_tiles,
                             int64_t *ordered, int64_t *slots, void *stream) {
  LM_REQUIRE(tokens >= 1 && top_k >= 1 && top_k <= 16, LM_EINVAL,
             "Expected contiguous CUDA [tokens,top_k] routing IDs");
  LM_REQUIRE(experts >= 1 && experts <= 256, LM_EINVAL, "route plan supports 1..256 experts");
  LM_REQUIRE(bm >= 1, LM_EINVAL, "tile height must be positive");
  LM_REQUIRE(tokens * top_k < (1LL << 30), LM_EINVAL, "too many routes");
  LM_REQUIRE(max_tiles == (tokens * top_k + bm - 1) / bm + experts, LM_EINVAL,
             "max_tiles must be cdiv(routes, bm) + experts");
  LM_REQUIRE(ids && pos && table && ordered && slots, LM_EINVAL, "null pointer");
  return route_plan(ids, tokens, top_k, experts, bm, pos, table, max_tiles, ordered, slots,
                    as_stream(stream));
}

extern "C" int lm_ordered_reduce(const void *v, const int64_t *table, const void *w, int w_dtype,
                                 void *y, int64_t n, int64_t experts, int dtype, void *stream) {
  LM_REQUIRE(n > 0 && experts >= 0, LM_EINVAL, "invalid reduce geometry");
  LM_REQUIRE(w_dtype == LM_BF16 || w_dtype == LM_FP16 || w_dtype == LM_FP32, LM_EINVAL,
             "weights must be bf16, fp16 or fp32");
  LM_REQUIRE(dtype == LM_BF16 || dtype == LM_FP16, LM_EINVAL, "values must be bf16 or fp16");
  LM_REQUIRE(v && table && w && y, LM_EINVAL, "null pointer");
  const unsigned g = cdiv(n, 256);
  const uint16_t *vp = static_cast<const uint16_t *>(v);
  uint16_t *yp = static_cast<uint16_t *>(y);
  if (dtype == LM_BF16)
    ordered_reduce_kernel<BF16><<<g, 256, 0, as_stream(stream)>>>(vp, table, w, w_dtype, yp,
                                                                  (int)n, (int)experts);
  else
    ordered_reduce_kernel<FP16><<<g, 256, 0, as_stream(stream)>>>(vp, table, w, w_dtype, yp,
                                                                  (int)n, (int)experts);
  return check_launch("ordered_reduce_kernel");
}

extern "C" int lm_routed_reduce(const void *v, const int64_t *ordered, const int64_t *slots,
                                const void *w, int w_dtype, void *y, int64_t tokens, int64_t n,
                                int64_t top_k, int dtype, void *stream) {
  LM_REQUIRE(n > 0 && tokens >= 0 && top_k >= 1, LM_EINVAL, "invalid reduce geometry");
  LM_REQUIRE(w_dtype == LM_BF16 || w_dtype == LM_FP16 || w_dtype == LM_FP32, LM_EINVAL,
             "weights must be bf16, fp16 or fp32");
  LM_REQUIRE(dtype == LM_BF16 || dtype == LM_FP16, LM_EINVAL, "values must be bf16 or fp16");
  if (tokens == 0) return LM_OK;
  LM_REQUIRE(tokens < 65536, LM_EINVAL, "too many tokens for one launch");
  LM_REQUIRE(v && ordered && slots && w && y, LM_EINVAL, "null pointer");
  const uint16_t *vp = static_cast<const uint16_t *>(v);
  uint16_t *yp = static_cast<uint16_t *>(y);
  return dtype == LM_BF16 ? routed_reduce<BF16>(vp, ordered, slots, w, w_dtype, yp, tokens, n,
                                                top_k, as_stream(stream))
                          : routed_reduce<FP16>(vp, ordered, slots, w, w_dtype, yp, tokens, n,
                                                top_k, as_stream(stream));
}

extern "C" int lm_swiglu(const void *gu, void *h, int64_t rows, int64_t half, int dtype,
                         void *stream) {
  LM_REQUIRE(rows >= 0 && half > 0, LM_EINVAL, "invalid SwiGLU geometry");
  LM_REQUIRE(dtype == LM_BF16 || dtype == LM_FP16, LM_EINVAL, "SwiGLU input must be bf16 or fp16");
  if (rows == 0) return LM_OK;
  LM_REQUIRE(gu && h, LM_EINVAL, "null pointer");
  int64_t blocks = (rows * half + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  const uint16_t *gp = static_cast<const uint16_t *>(gu);
  uint16_t *hp = static_cast<uint16_t *>(h);
  if (dtype == LM_BF16)
    swiglu_kernel<BF16><<<(unsigned)blocks, 256, 0, as_stream(stream)>>>(gp, hp, rows, half);
  else
    swiglu_kernel<FP16><<<(unsigned)blocks, 256, 0, as_stream(stream)>>>(gp, hp, rows, half);
  return check_launch("swiglu_kernel");
}

extern "C" int lm_rmsnorm(const void *x, const float *w, void *y, int64_t rows, int64_t n,
                          float eps, void *stream) {
  LM_REQUIRE(rows >= 0 && n > 0, LM_EINVAL, "invalid RMSNorm geometry");
  if (rows == 0) return LM_OK;
  LM_REQUIRE(rows < (1LL << 31) && x && y, LM_EINVAL, "null pointer");
  rmsnorm_kernel<<<(unsigned)rows, 256, 0, as_stream(stream)>>>(
      static_cast<const uint16_t *>(x), w, static_cast<uint16_t *>(y), (int)n, eps);
  return check_launch("rmsnorm_kernel");
}
