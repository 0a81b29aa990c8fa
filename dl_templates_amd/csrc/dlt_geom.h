// Window geometry shared by host code, the debug exports and every attention kernel.
//
// Tokens live on a 2D grid of `TR` rows; a row holds `XL` tokens (x = c * S + s for tile
// column c and in-tile slot s), token n = r * XL + x, which is the reference's tile-major
// numbering n = (r * t_width + c) * b_size + s (src/tiled_swa.py:63,104,216).
// Dense attention is the same structure with one row and an unrestricted x interval.
#pragma once
#include <stdint.h>

#if defined(__HIPCC__)
#define DLT_HD __host__ __device__ inline
#else
#define DLT_HD inline
#endif

enum { DLT_GEOM_SWA = 0, DLT_GEOM_DENSE = 1, DLT_GEOM_CAUSAL = 2 };

struct DltGeom {
  int32_t mode;
  int32_t TR;        // grid rows (1 for dense / causal)
  int32_t XLq, XLk;  // tokens per row on the query side / key side
  int32_t S, TC;     // tokens per tile, tiles per row (SWA only)
  int32_t WR, WC;    // window half sizes in tiles (SWA only)
};

DLT_HD int dlt_imin(int a, int b) { return a < b ? a : b; }
DLT_HD int dlt_imax(int a, int b) { return a > b ? a : b; }

// Keys attended by query (r, x): rows [rlo, rhi] (inclusive), x in [xlo, xhi).
// SWA: |r - r'| <= WR and |c - c'| <= WC, truncated at the border
// (src/tiled_swa.py:76-79, :212-214, :701-713).
DLT_HD void dlt_key_range(const DltGeom& g, int r, int x, int& rlo, int& rhi, int& xlo, int& xhi) {
  if (g.mode == DLT_GEOM_SWA) {
    const int c = x / g.S;
    rlo = dlt_imax(r - g.WR, 0);
    rhi = dlt_imin(r + g.WR, g.TR - 1);
    xlo = dlt_imax(c - g.WC, 0) * g.S;
    xhi = dlt_imin(c + g.WC + 1, g.TC) * g.S;
  } else if (g.mode == DLT_GEOM_DENSE) {
    rlo = rhi = 0; xlo = 0; xhi = g.XLk;
  } else {
    rlo = rhi = 0; xlo = 0; xhi = dlt_imin(x + 1, g.XLk);
  }
}

// Queries that attend key (r, x): the transpose of dlt_key_range.  The SWA window is
// symmetric (the reference's backward relies on the same fact, src/tiled_swa.py:475-488).
DLT_HD void dlt_query_range(const DltGeom& g, int r, int x, int& rlo, int& rhi, int& xlo, int& xhi) {
  if (g.mode == DLT_GEOM_SWA) {
    dlt_key_range(g, r, x, rlo, rhi, xlo, xhi);
  } else if (g.mode == DLT_GEOM_DENSE) {
    rlo = rhi = 0; xlo = 0; xhi = g.XLq;
  } else {
    rlo = rhi = 0; xlo = dlt_imin(x, g.XLq); xhi = g.XLq;
  }
}

// Bands of the marching kernels: `units` steps (or grid rows) split evenly, `per` of them in each of `nb` bands; one workgroup per
// band and column strip, `slots` of them on the chip at once.  A band costs its units plus a prologue of about two; workgroups
// beyond the slots wait for a whole band.  The cheapest split with the fewest bands wins.  Only band heights that occur are
// tried (about 2 sqrt(units)), and none beyond the band count at which the prologues alone cost more than the best split: a
// thin grid of 262 144 rows takes a few hundred steps of this loop, not 262 144 (1.1 ms).  Returns the splits tried.
DLT_HD int dlt_band_plan(int units, int64_t cols, int64_t slots, int& per, int& nb) {
  int64_t best = -1;
  int tried = 0;
  for (int n = 1;;) {
    const int h = (units + n - 1) / n;
    const int64_t cost = (cols * n + slots - 1) / slots * (h + 2);
    tried++;
    if (best < 0 || cost < best) { best = cost; per = h; nb = n; }
    // cost >= cols n (units / n + 2) / slots, which grows with n
    if (h == 1 || cols * (units + 2 * (int64_t)n) >= best * slots) return tried;
    n = (units + h - 2) / (h - 1);   // fewest bands of at most h - 1 units
  }
}

// Image layout, forward over 16-token tiles at d = 32 with a 3 x 3 window: whether one workgroup per CU runs (`cols` strips of 8 tiles).
// A pixel's heads lie side by side, so the workgroups of 8 heads and more share every 128-byte line and must meet in the L2.  Two
// workgroups per CU march strips apart and fetch 1.37 times the bytes; one per CU gives up half of the waves that hide latency.
// It wins where HBM is the bound and both launches would march strips: strips and rounds over the CUs at least 15/16 full, 1, 2 or 4 rounds, and
// rows enough, fewer with 16 heads.  Two per CU -> one, us, inputs in the caches / cycled through 800 MB: 8 heads, one round of 64 rows of
// 64 tiles 153 -> 141 / 160 -> 141, of 16 or 32 tiles 132 -> 132 / 136 -> 131, 48 rows of 64 101 -> 103 / 119 -> 107; two rounds of 40 rows of 8 to
// 64 tiles -11 ... +1 / -12 ... 0 %, 24 of 64 101 -> 106 / 118 -> 112, 8 rows 30 -> 34 / 43 -> 45; four of 48 rows -10 ... +3 %, of 24 -3 ... +8 %.
// 16 heads: one round of 32 rows of 64 tiles 64 -> 59 / 92 -> 82, two of 24 114 -> 108 / 130 -> 111, four of 32 -9 ... +1 %.  It loses in three
// rounds (64 rows of 48 tiles 422 -> 436) and five (407 -> 433), on ragged strips (two rounds of 33 tiles, 64 rows 262 -> 275; one
// tile 93 -> 149: most of a CU's waves own nothing) and with fewer heads (16 x 2 slabs of 64 x 64: 121 -> 122); 32-token tiles (179 ->
// 208) and windows of five columns (183 -> 186) are bound by arithmetic, d = 64 and five rows leave LDS for one anyway.
DLT_HD bool dlt_image_fwd_alone(int d, int S, int WR, int WC, int TR, int TC, int H, int64_t cols, int64_t cus) {
  if (d != 32 || S != 16 || WR != 1 || WC != 1 || H < 8 || cols < cus || 16 * TC < 15 * 8 * ((TC + 7) / 8)) return false;
  const int64_t rounds = (cols + cus - 1) / cus;
  if (16 * cols < 15 * rounds * cus) return false;
  return rounds == 1 ? TR >= (H < 16 ? 64 : 32) : rounds == 2 ? TR >= (H < 16 ? 40 : 24) : rounds == 4 && TR >= (H < 16 ? 48 : 32);
}

// Backward over tiles at d = 32 / 64: whether dQ, dK and dV leave in one launch (16-token tiles, 3 x 3 window; TC tile columns, `rows` grid
// rows of all (batch, head) slabs together).  At d = 32 a strip is 8 tiles wide and a CU holds one workgroup: on grids of a few tile
// columns most of its 16 waves own nothing, and once a CU has some 12 rows to march the two launches, two workgroups per CU each,
// are faster.  Token layout, 256 slabs of 24 rows, one launch -> two: 1 column 65 -> 56 us, 3 68 -> 63, 5 87 -> 78, 6 and more 87 -> 87, 9
// 162 -> 162; 1024 slabs of 6 rows of 5 97 -> 84.  Images are bound by HBM sooner: 1 column 65 -> 57, 2 66 -> 64, 3 67 -> 66, 4 67 -> 72, 5 88 -> 91.
// Fewer rows: 64 slabs of 6 rows, 1 ... 5 columns 10-12 against 13-15.  Where neither side wins clearly one launch stays: images of 3 columns
// (+ 10 ... - 6 %), many slabs of 6 rows (512 of 9 columns, inputs in the caches 96 against 90, not 99 against 97).  At d = 64 strips are 4 tiles wide (256 slabs of 24 x 1: 81 against 120).
DLT_HD bool dlt_tile_bwd_one_launch(int d, int S, int WR, int WC, bool img, int TC, int64_t rows, int64_t cus) {
  if (S != 16 || WR != 1 || WC != 1) return false;
  return d == 64 || TC > (img ? 2 : 5) || rows < 12 * cus;
}

// Backward passes of dense / causal attention that do not split the other side: whether a workgroup owns 64 tokens (4 waves of one block)
// instead of 128 (two blocks per wave).  `wgs`: workgroups of 64 tokens; `kv_64_128`: dK/dV at 64/128.  The same bits either way.
// They do while they all run at once, one per CU, or two under a mask, where the work is uneven.  8 slabs of 2048 x 2048, dQ and dK/dV:
// 64/64 32.3 -> 25.0 and 39.2 -> 30.0 us, 64/128 37.7 -> 28.5 and 50.5 -> 38.4, dQ at 128/128 52.0 -> 39.3; causal, 16 slabs: 35.4 -> 31.1 and
// 43.5 -> 39.3, 40.2 -> 35.3 and 67.0 -> 50.3, 53.0 -> 45.4.  12 slabs without a mask (384 workgroups): the same or slower.
// dK/dV at 64/128 under a mask, where two blocks per wave spill: always below 3072 keys (64 slabs of 2048: 160 -> 138; 32 of 4096: 232 ->
// 249), up to four per CU below 8192 (whole backward pass, causal: 10 slabs of 4096 203 -> 186, 8 of 6000 253 -> 219, 6 of 8192 384 -> 360;
// 10 of 6000 316 -> 327; beyond it loses: 4 of 12 000 510 -> 546).
DLT_HD bool dlt_flash_bwd_64(bool causal, bool kv_64_128, int own, int64_t wgs, int64_t cus) {
  if (causal && kv_64_128 && own < 3072) return true;
  return wgs <= (!causal ? 1 : kv_64_128 && own <= 8192 ? 4 : 2) * cus;
}

// idx decode of the rotary op: row = int16(idx >> 16), col = int16(idx & 0xFFFF)
// (src/fused_rope2d.py:41-42); an axis is rotated iff its value is >= 0 (:44-45).
DLT_HD int dlt_rope_row(int32_t idx) { return (int)(int16_t)(idx >> 16); }
DLT_HD int dlt_rope_col(int32_t idx) { return (int)(int16_t)(idx & 0xFFFF); }

// ---- image layout of the tokens --------------------------------------------------------------
// A caller that keeps q, k, v as images [B, IH, IW, heads, D] (the layout the reference's demo
// converts from and to around the operator, src/tiled_swa.py:753-755) maps pixel (y, x) of a tile
// of bh x bw pixels to token
//     n = ((y / bh * TC + x / bw) * bh + y % bh) * bw + x % bw,      S = bh * bw tokens per tile.
// The kernels go the other way: token n -> pixel (y, x) -> element offset y * stride_y + x * stride_x.
// Divisions by S, TC and bw are exact multiply-shift divisions (m = ceil(2^(31+l) / d), l = ceil(log2 d):
// floor(n m / 2^(31+l)) = floor(n / d) for every n < 2^31).
struct DltTokMap {
  int32_t img;  // 0: token n lies n * stride_n elements into its (batch, head) slab
  uint32_t S, TC, bh, bw;
  uint32_t mS, mTC, mbw;  // multipliers
  uint32_t sS, sTC, sbw;  // shifts (31 + l)
};

DLT_HD uint32_t dlt_fastdiv(uint32_t n, uint32_t m, uint32_t sh) { return (uint32_t)(((uint64_t)n * m) >> sh); }

DLT_HD void dlt_fastdiv_make(uint32_t d, uint32_t& m, uint32_t& sh) {
  uint32_t l = 0;
  while (l < 31 && ((uint32_t)1 << l) < d) l++;
  const uint64_t num = (uint64_t)1 << (31 + l);
  m = (uint32_t)((num + d - 1) / d);
  sh = 31 + l;
}

DLT_HD DltTokMap dlt_tokmap_none() {
  DltTokMap tm;
  tm.img = 0; tm.S = tm.TC = tm.bh = tm.bw = 1;
  tm.mS = tm.mTC = tm.mbw = (uint32_t)1 << 31;
  tm.sS = tm.sTC = tm.sbw = 31;
  return tm;
}

DLT_HD DltTokMap dlt_tokmap_image(uint32_t bh, uint32_t bw, uint32_t TC) {
  DltTokMap tm;
  tm.img = 1; tm.S = bh * bw; tm.TC = TC; tm.bh = bh; tm.bw = bw;
  dlt_fastdiv_make(tm.S, tm.mS, tm.sS);
  dlt_fastdiv_make(TC, tm.mTC, tm.sTC);
  dlt_fastdiv_make(bw, tm.mbw, tm.sbw);
  return tm;
}

// token n (tile-major order) -> pixel (y, x)
DLT_HD void dlt_token_pixel(const DltTokMap& tm, uint32_t n, uint32_t& y, uint32_t& x) {
  const uint32_t tile = dlt_fastdiv(n, tm.mS, tm.sS), s = n - tile * tm.S;
  const uint32_t tr = dlt_fastdiv(tile, tm.mTC, tm.sTC), tc = tile - tr * tm.TC;
  const uint32_t i = dlt_fastdiv(s, tm.mbw, tm.sbw), j = s - i * tm.bw;
  y = tr * tm.bh + i;
  x = tc * tm.bw + j;
}

// slot x' = tc * S + s inside a grid row (tile column tc, in-tile slot s) -> (pixel row inside the
// tile row, pixel x): what the kernels that walk a grid row at a time need
DLT_HD void dlt_slot_pixel(const DltTokMap& tm, uint32_t xs, uint32_t& i, uint32_t& x) {
  const uint32_t tc = dlt_fastdiv(xs, tm.mS, tm.sS), s = xs - tc * tm.S;
  i = dlt_fastdiv(s, tm.mbw, tm.sbw);
  x = tc * tm.bw + (s - i * tm.bw);
}
