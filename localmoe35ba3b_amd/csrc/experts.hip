// Decode experts of the operator layer (Int8Experts, one token; int8.py:127-210).
//
//   lm_expert_table          the descriptor table of the grouped GEMVs: the
//                            selected ids sorted, and each expert's bank
//                            pointers (int8.py:164-179)
//   lm_w8a16_experts_decode  the whole W8A16 expert pass in two kernels:
//                            gate_up + SwiGLU, then down + ordered combine
//
// One token is latency-bound: 26 MB of weights for 8 experts against the
// launches.  As separate operators (device sort, pointer arithmetic, two
// GEMVs, SwiGLU, combine) the pass took 121 us, most of it host work and a
// host-to-device copy; each kernel here sorts the few ids itself, so the pass
// needs two launches and nothing between them.  Arithmetic and order of every
// sum are those of the separate operators, so the bits are the same.
#include "gemv_core.hpp"

namespace lm {
namespace {

constexpr int kExPairs = 8;    // gate_up: SwiGLU columns per workgroup
constexpr int kExCols = 8;     // down: output columns per workgroup
constexpr int kExMax = 64;     // selected experts (one lane each)
constexpr int kExThreads = 256;
constexpr size_t kExLds = 128 * 1024;

struct ExpertsArgs {
  const void *ids;
  int ids32;
  int n;         // selected experts
  int experts;   // of the bank
  const uint16_t *x;
  const int8_t *gu_q, *dn_q;
  const float *gu_s, *dn_s;
  int64_t gu_qes, gu_ses, dn_qes, dn_ses;
  const void *w;
  int w_dtype;
  uint16_t *h;  // [n, inter]
  uint16_t *y;  // [hidden]
  int inter, hidden;
};

// Expert id of selection j, clamped into the bank.
__device__ __forceinline__ int selected_id(const void *ids, int ids32, int j, int experts) {
  const int64_t e = ids32 ? ldg<int>(static_cast<const int *>(ids) + j)
                          : ldg<int64_t>(static_cast<const int64_t *>(ids) + j);
  return (int)clamp_index(e, experts);
}

// Place of lane j's id among the n <= 64 ids of the wave (lane i holds id
// i): ascending ids, equal ids in selection order.
__device__ __forceinline__ int id_rank(int id, int n, int lane) {
  int rank = 0;
  for (int i = 0; i < n; ++i) {
    const int o = __builtin_amdgcn_readlane(id, i);
    rank += (o < id || (o == id && i < lane)) ? 1 : 0;
  }
  return rank;
}

__global__ __launch_bounds__(256) void expert_table_kernel(ExpertsArgs a, int64_t *table) {
  const int j = blockIdx.x * 256 + threadIdx.x;
  if (j < a.n) {
    const int e = selected_id(a.ids, a.ids32, j, a.experts);
    int rank = 0;
    for (int i = 0; i < a.n; ++i) {
      const int o = selected_id(a.ids, a.ids32, i, a.experts);
      rank += (o < e || (o == e && i < j)) ? 1 : 0;
    }
    int64_t *row = table + (int64_t)rank * 5;
    row[0] = reinterpret_cast<int64_t>(a.gu_q + e * a.gu_qes);
    row[1] = reinterpret_cast<int64_t>(a.gu_s + e * a.gu_ses);
    row[2] = reinterpret_cast<int64_t>(a.dn_q + e * a.dn_qes);
    row[3] = reinterpret_cast<int64_t>(a.dn_s + e * a.dn_ses);
    row[4] = j;
  }
}

// gate_up rows of slot blockIdx.y (the blockIdx.y-th smallest id) for
// kExPairs SwiGLU columns: gate rows n0 .. and up rows inter + n0 .., 32 KB of
// weights at K = 2048, all of them in flight at once (KC = 2048; KC = 0
// streams any K in batches).
template <typename T, int KC>
__global__ __launch_bounds__(kExThreads) void experts_gate_up_kernel(ExpertsArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int K = KC ? KC : a.hidden, G = K >> 7;
  uint16_t *xl = reinterpret_cast<uint16_t *>(smem);
  float *ws = reinterpret_cast<float *>(smem + K * 2);
  float *part = ws + 2 * kExPairs * G;
  const int t = threadIdx.x, lane = t & 63;
  const int id = selected_id(a.ids, a.ids32, min(lane, a.n - 1), a.experts);
  const int n0 = blockIdx.x * kExPairs;
  const int rh = min(kExPairs, a.inter - n0);
  const RowMap map{n0, a.inter + n0, rh};
  const int rows = 2 * rh;
  const int slot = blockIdx.y;
  const int8_t *q;
  const float *s;
  auto pick = [&] {
    const int rank = id_rank(id, a.n, lane);
    const unsigned long long m = __ballot(lane < a.n && rank == slot);
    const int e = __builtin_amdgcn_readlane(id, (int)__builtin_ctzll(m));
    q = a.gu_q + e * a.gu_qes;
    s = a.gu_s + e * a.gu_ses;
  };
  auto row_ptr = [&](int r) { return q + (int64_t)map(r) * K; };
  const int sub = t & 7;
  auto body = [&](u32x4 w, int r, int g, int f, bool ok) {
    uint32_t wd[8];
    dequant16<T>(w, ok ? ws[f] : 0.0f, wd);
    const uint16_t *xp = xl + g * 128 + sub * 16;
    const float p = octet_sum_f32(dot16_w16<T>(wd, *reinterpret_cast<const u32x4 *>(xp),
                                               *reinterpret_cast<const u32x4 *>(xp + 8)));
    if (ok && sub == 0) part[f] = p;
  };
  if constexpr (KC == 2048) {
    const u32x4 xv = ldg16(a.x + t * 8);
    pick();
    const int f = min(t, rows * G - 1);
    const float wsv = ldg_f32(s + (int64_t)map(f / G) * G + f % G);
    RowLoads<8, kExThreads> L;
    L.issue(rows, G, row_ptr);
    reinterpret_cast<u32x4 *>(xl)[t] = xv;
    ws[f] = wsv;  // surplus threads rewrite the last entry with its own value
    __syncthreads();
    L.consume(body);
  } else {
    pick();
    for (int i = t; i < K / 8; i += kExThreads)
      reinterpret_cast<u32x4 *>(xl)[i] = ldg16(a.x + i * 8);
    for (int i = t; i < rows * G; i += kExThreads)
      ws[i] = ldg_f32(s + (int64_t)map(i / G) * G + i % G);
    __syncthreads();
    stream_rows<8>(rows, G, row_ptr, body);
  }
  __syncthreads();
  if (t < rh) {
    const float gate = T::round(ordered_sum8(part + t * G, G));
    const float up = T::round(ordered_sum8(part + (rh + t) * G, G));
    a.h[(int64_t)slot * a.inter + n0 + t] = T::from_f32(T::round(silu_f32(gate)) * up);
  }
}

// down rows of every slot for kExCols output columns (row r = slot * kExCols
// + column), then the combine in ascending expert order, rounding at every
// step (int8.py:240-250).
template <typename T, int KC>
__global__ __launch_bounds__(kExThreads) void experts_down_kernel(ExpertsArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int K = KC ? KC : a.inter, G = K >> 7, n = a.n;
  const int R = n * kExCols;
  uint16_t *hl = reinterpret_cast<uint16_t *>(smem);
  float *ws = reinterpret_cast<float *>(smem + (size_t)n * K * 2);
  float *part = ws + R * G;
  float *prod = part + R * G;
  __shared__ int sid[kExMax];
  __shared__ float sw[kExMax];
  const int t = threadIdx.x, lane = t & 63;
  const int j = min(lane, n - 1);
  const int id = selected_id(a.ids, a.ids32, j, a.experts);
  float wj;
  if (a.w_dtype == LM_FP32) {
    wj = ldg_f32(static_cast<const float *>(a.w) + j);
  } else {
    const uint32_t b = ldg<uint16_t>(static_cast<const uint16_t *>(a.w) + j);
    wj = a.w_dtype == LM_FP16 ? f16_bits_to_f32(b) : bf16_bits_to_f32(b);
  }
  const int c0 = blockIdx.x * kExCols;
  // every wave writes the same sorted ids and weights, and reads only them
  const int rank = id_rank(id, n, lane);
  if (lane < n) {
    sid[rank] = id;
    sw[rank] = wj;
  }
  wave_lds_sync();
  // columns past the end re-read the last one; they are not stored
  auto row_ptr = [&](int r) {
    return a.dn_q + sid[r / kExCols] * a.dn_qes +
           (int64_t)min(c0 + r % kExCols, a.hidden - 1) * K;
  };
  auto scale_ptr = [&](int f) {
    const int r = f / G;
    return a.dn_s + sid[r / kExCols] * a.dn_ses +
           (int64_t)min(c0 + r % kExCols, a.hidden - 1) * G + f % G;
  };
  const int sub = t & 7;
  auto body = [&](u32x4 w, int r, int g, int f, bool ok) {
    uint32_t wd[8];
    dequant16<T>(w, ok ? ws[f] : 0.0f, wd);
    const uint16_t *hp = hl + (r / kExCols) * K + g * 128 + sub * 16;
    const float p = octet_sum_f32(dot16_w16<T>(wd, *reinterpret_cast<const u32x4 *>(hp),
                                               *reinterpret_cast<const u32x4 *>(hp + 8)));
    if (ok && sub == 0) part[f] = p;
  };
  if (KC == 512 && n <= 8) {
    u32x4 hv[2];  // n * 64 pieces; surplus ones re-read the last
    const int np = n * (K / 8);
#pragma unroll
    for (int u = 0; u < 2; ++u) hv[u] = ldg16(a.h + min(t + u * kExThreads, np - 1) * 8);
    const int f = min(t, R * G - 1);
    const float wsv = ldg_f32(scale_ptr(f));
    RowLoads<8, kExThreads> L;
    L.issue(R, G, row_ptr);
#pragma unroll
    for (int u = 0; u < 2; ++u)
      reinterpret_cast<u32x4 *>(hl)[min(t + u * kExThreads, np - 1)] = hv[u];
    ws[f] = wsv;
    __syncthreads();
    L.consume(body);
  } else {
    for (int i = t; i < n * (K / 8); i += kExThreads)
      reinterpret_cast<u32x4 *>(hl)[i] = ldg16(a.h + (int64_t)i * 8);
    for (int i = t; i < R * G; i += kExThreads) ws[i] = ldg_f32(scale_ptr(i));
    __syncthreads();
    stream_rows<8>(R, G, row_ptr, body);
  }
  __syncthreads();
  for (int i = t; i < R; i += kExThreads)
    prod[i] = T::round(T::round(ordered_sum8(part + i * G, G)) * sw[i / kExCols]);
  __syncthreads();
  if (t < kExCols && c0 + t < a.hidden) {
    float acc = 0.0f;
    for (int s = 0; s < n; ++s) acc = T::round(acc + prod[s * kExCols + t]);
    a.y[c0 + t] = T::from_f32(acc);
  }
}

size_t gate_up_lds(int64_t k) { return (size_t)k * 2 + 2 * kExPairs * (size_t)(k / 128) * 8; }
size_t down_lds(int64_t n, int64_t k) {
  return (size_t)n * k * 2 + (size_t)n * kExCols * (size_t)(k / 128) * 8 + (size_t)n * kExCols * 4;
}

template <typename T>
int experts_decode(const ExpertsArgs &a, hipStream_t st) {
  const dim3 gu(cdiv(a.inter, kExPairs), (unsigned)a.n);
  const unsigned dn = cdiv(a.hidden, kExCols);
  const size_t l1 = gate_up_lds(a.hidden), l2 = down_lds(a.n, a.inter);
  if (a.hidden == 2048)
    experts_gate_up_kernel<T, 2048><<<gu, kExThreads, l1, st>>>(a);
  else
    experts_gate_up_kernel<T, 0><<<gu, kExThreads, l1, st>>>(a);
  if (int rc = check_launch("experts_gate_up_kernel")) return rc;
  if (a.inter == 512)
    experts_down_kernel<T, 512><<<dn, kExThreads, l2, st>>>(a);
  else
    experts_down_kernel<T, 0><<<dn, kExThreads, l2, st>>>(a);
  return check_launch("experts_down_kernel");
}

int check_selection(const void *ids, int ids_bytes, int64_t n, int64_t experts) {
  LM_REQUIRE(ids_bytes == 4 || ids_bytes == 8, LM_EINVAL, "expert ids must be int32 or int64");
  LM_REQUIRE(n >= 0 && n < (1 << 20) && experts >= (n ? 1 : 0) && experts < (1LL << 31), LM_EINVAL,
             "invalid expert selection");
  LM_REQUIRE(n == 0 || ids, LM_EINVAL, "null pointer");
  return LM_OK;
}

}  // namespace
}  // namespace lm

using namespace lm;

extern "C" int lm_expert_table(const void *ids, int ids_bytes, int64_t n, int64_t experts,
                               const int8_t *gu_q, const float *gu_s, const int8_t *dn_q,
                               const float *dn_s, int64_t gu_q_expert_stride,
                               int64_t gu_s_expert_stride, int64_t dn_q_expert_stride,
                               int64_t dn_s_expert_stride, int64_t *table, void *stream) {
  if (int rc = check_selection(ids, ids_bytes, n, experts)) return rc;
  if (n == 0) return LM_OK;
  LM_REQUIRE(gu_q && gu_s && dn_q && dn_s && table, LM_EINVAL, "null pointer");
  ExpertsArgs a{};
  a.ids = ids;
  a.ids32 = ids_bytes == 4;
  a.n = (int)n;
  a.experts = (int)experts;
  a.gu_q = gu_q;
  a.gu_s = gu_s;
  a.dn_q = dn_q;
  a.dn_s = dn_s;
  a.gu_qes = gu_q_expert_stride;
  a.gu_ses = gu_s_expert_stride;
  a.dn_qes = dn_q_expert_stride;
  a.dn_ses = dn_s_expert_stride;
  expert_table_kernel<<<cdiv(n, 256), 256, 0, as_stream(stream)>>>(a, table);
  return check_launch("expert_table_kernel");
}

extern "C" int lm_w8a16_experts_decode_fits(int64_t n, int64_t hidden, int64_t inter) {
  return n >= 1 && n <= kExMax && hidden > 0 && inter > 0 && hidden % 128 == 0 &&
         inter % 128 == 0 && hidden <= 65536 && inter <= 65536 && gate_up_lds(hidden) <= kExLds &&
         down_lds(n, inter) <= kExLds;
}

extern "C" int lm_w8a16_experts_decode(const void *x, const void *ids, int ids_bytes, int64_t n,
                                       int64_t experts, const int8_t *gu_q, const float *gu_s,
                                       const int8_t *dn_q, const float *dn_s,
                                       int64_t gu_q_expert_stride, int64_t gu_s_expert_stride,
                                       int64_t dn_q_expert_stride, int64_t dn_s_expert_stride,
                                       const void *w, int w_dtype, void *h, void *y,
                                       int64_t hidden, int64_t inter, int dtype, void *stream) {
  if (int rc = check_selection(ids, ids_bytes, n, experts)) return rc;
  LM_REQUIRE(lm_w8a16_experts_decode_fits(n, hidden, inter), LM_EINVAL,
             "Invalid INT8 group geometry");
  LM_REQUIRE(dtype == LM_BF16 || dtype == LM_FP16, LM_EINVAL,
             "W8A16 requires CUDA FP16/BF16 activations");
  LM_REQUIRE(w_dtype == LM_BF16 || w_dtype == LM_FP16 || w_dtype == LM_FP32, LM_EINVAL,
             "weights must be bf16, fp16 or fp32");
  LM_REQUIRE(x && gu_q && gu_s && dn_q && dn_s && w && h && y, LM_EINVAL, "null pointer");
  ExpertsArgs a{};
  a.ids = ids;
  a.ids32 = ids_bytes == 4;
  a.n = (int)n;
  a.experts = (int)experts;
  a.x = static_cast<const uint16_t *>(x);
  a.gu_q = gu_q;
  a.gu_s = gu_s;
  a.dn_q = dn_q;
  a.dn_s = dn_s;
  a.gu_qes = gu_q_expert_stride;
  a.gu_ses = gu_s_expert_stride;
  a.dn_qes = dn_q_expert_stride;
  a.dn_ses = dn_s_expert_stride;
  a.w = w;
  a.w_dtype = w_dtype;
  a.h = static_cast<uint16_t *>(h);
  a.y = static_cast<uint16_t *>(y);
  a.inter = (int)inter;
  a.hidden = (int)hidden;
  return dtype == LM_BF16 ? experts_decode<BF16>(a, as_stream(stream))
                          : experts_decode<FP16>(a, as_stream(stream));
}
