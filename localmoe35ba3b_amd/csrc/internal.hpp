// Host-side launch helpers shared between translation units of the library.
#pragma once
#include "common.hpp"

namespace lm {

int router_logits(const uint16_t *x, const uint16_t *w, const float *bias, float *logits,
                  int64_t T, int64_t E, int64_t H, hipStream_t st);
// The same logits through int8 digits (router_digits.hip), which need a workspace.
int64_t router_digits_bytes(int64_t T, int64_t E, int64_t H);
int router_logits_digits(const uint16_t *x, const uint16_t *w, const float *bias, float *logits,
                         int64_t T, int64_t E, int64_t H, void *workspace, hipStream_t st);
int router_topk(const float *logits, int64_t T, int64_t E, int64_t K, int64_t *ids,
                uint16_t *weights, hipStream_t st);
int route_plan(const int64_t *ids, int64_t T, int64_t K, int64_t E, int64_t bm, int64_t *pos,
               int64_t *table, int64_t max_tiles, int64_t *ordered, int64_t *slots,
               hipStream_t st);
// One routed grouped W8A16 GEMM (gate_up with gather + optional SwiGLU
// epilogue, or down over contiguous rows) over a (expert, start, stop) tile
// table.  Table experts are clamped into [0, experts), starts and stops into
// [0, y_rows], gathered row indices into [0, x_rows).
struct RoutedGemm {
  const void *x;
  int64_t ldx, x_rows;
  const int8_t *q;
  const float *s;
  int64_t q_es, s_es, experts;
  const int64_t *pos;
  const int64_t *table;
  int64_t n_tiles, bm;
  void *y;
  int64_t y_rows, n, k;
  bool gather, swiglu;
  int dtype;
  const int8_t *q_tiles = nullptr;  // q in the lm_w8_tile_rows layout, or null
  // Non-null: x holds fp16 rows fp16(row r * 2^x_exp[r]) (exact) and q_tiles
  // is in the LM_TILES_F16 format; the output is bf16.
  const int *x_exp = nullptr;
  // Gathered GEMMs on q_tiles: the token of row r of table tile i at
  // ptile[i * bm + r] (any value for rows past the tile's end), read with the
  // table row instead of through pos; required with q_tiles and gather.
  const int *ptile = nullptr;
  // Output rows that choose the tile form where another call's GEMM runs at the
  // same time and has more rows (results are the same); 0: y_rows.
  int64_t form_rows = 0;
};
int routed_gemm(const RoutedGemm &r, hipStream_t st);

// How a dense matrix of row_tiles x col_tiles tiles is dealt to the 8 XCDs of 32
// CUs (xcd_tile, common.hpp), and the rounds of one tile per CU that the busiest
// XCD works through.  short_tail: the last row tile takes time by its rows;
// act_bytes: of an activation, 0 where an XCD's L2 holds them all.
struct XcdDeal {
  bool by_columns;
  double rounds;
};
XcdDeal xcd_deal(int64_t m, int64_t n, int64_t row_tiles, int64_t col_tiles, int tile_rows,
                 bool short_tail, int act_bytes);
// Workgroups of such a launch; callers reject counts beyond one launch's grid
// (2^31 - 1) before launching.
inline int64_t xcd_grid(int64_t row_tiles, int64_t col_tiles, bool by_columns = false) {
  return by_columns ? 8 * row_tiles * ((col_tiles + 7) / 8) : 8 * col_tiles * ((row_tiles + 7) / 8);
}

// Dense W8A16 over small tiles whose waves split K (ksplit.hip): the tile
// shape for an [m, n, k] problem (shape < 0: k not served) with its estimated
// time in us, and the launch.
struct KsPlan {
  int shape;
  double cost;
  int rows, cols;  // of a tile
  bool by_columns;
};
KsPlan ksplit_plan(int64_t m, int64_t n, int64_t k);
int w8a16_ksplit(const KsPlan &plan, const void *x, const int8_t *q, const float *s, void *y,
                 int64_t m, int64_t n, int64_t k, int dtype, hipStream_t st);

// W8A8 on few rows already quantized (gemv.hip): the same results as the GEMM.
bool w8a8_gemv_serves(int64_t m, int64_t k);
int w8a8_gemv_rows(const int8_t *xq, const float *xs, const int8_t *q, const float *s, void *y,
                   int64_t m, int64_t n, int64_t k, int swiglu, int y_dtype, hipStream_t st);

}  // namespace lm
