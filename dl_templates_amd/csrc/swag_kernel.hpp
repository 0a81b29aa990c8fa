// Marching kernels for token grids (b_size == 1) at head dim 64 and windows up to 13 x 13, and at head dim 32 and windows up to 21
// x 21 (the ring of K and V of the widest class: 129 KB; at head dim 64 it would be twice that), with or without the fused
// rotation (head dim 64, 8 rotary pairs per axis, rotated q / k kept): the shape of the benchmark's headline configuration.
//
// The window is a compile-time class: NCH x NCG blocks of 4 x 4 keys.  (An earlier version always computed 16 x 16 keys at head
// dim 64, and head dim 32 ran zero-padded on the tile kernels, which stage every halo row once per band of 4 own rows: 32 slabs
// of 84 x 82 tokens, d = 64, 11 x 7 window: forward 62 -> 35 us, dQ 79 -> 51, dK/dV 88 -> 53; 64 slabs of the same at d = 32:
// 89 -> 42, 95 -> 50, 120 -> 56; 32 slabs of 89 x 98, d = 32, 15 x 21: 94 -> 54, 98 -> 67, 123 -> 78; 16 of 13 x 74, 17 x 17: 14.0 ->
// 9.6, 14.3 -> 10.3, 17.4 -> 11.4.)  A workgroup owns a strip of 4 PC columns and marches down the grid in steps of 4 PR rows
// (PR = 8 / PC); wave w owns the 4 x 4 patch of column w % PC and row group w / PC.  The halo rows a step sees
// (NCH + PR - 1 chunks of 4 rows, both streamed tensors) live in an LDS ring; the chunks of the next step travel HBM ->
// registers while the current one computes.  The whole window is resident: the softmax is one-shot.
//
// In the C layout of a block lane group g holds key row g and element i key column i, lane n is own token (n >> 2, n & 3): the
// row test enters as the C operand of the score products (0 or -inf), the column tests are lane masks that stay in scalar
// registers for the whole march.  -inf + inf and -inf + NaN are NaN: with an infinity or NaN in a key row, queries that do not see it
// find their row sum NaN (one test per patch of the forward pass), and the patch is formed again by swag_fwd_exact.  (Replacing
// masked scores always costs a scalar instruction in front of every select, and a second body inside the march costs registers: 89 x 98,
// d = 32, 15 x 21 window, 32 slabs 49 -> 65 and 58 us.)
//
// LDS: token rows of 2 D bytes, 16-byte piece p of the token at halo row r, column c at p ^ swz(r, c), where the swizzle only
// takes c & 3 and r & 1: operand reads and transposing reads are free of bank conflicts and their lane offsets are the same
// for every block of the window.
#pragma once
#include "swat_kernel.hpp"

struct SwagArgs {
  const void *q, *k, *v, *o, *d_o;
  void *out_o, *dq, *dk, *dv;
  float* lse;
  float* delta;
  int64_t qs[4], ks[4], vs[4], os[4], dos[4], dqs[4], dks[4], dvs[4], ls[3];
  DltGeom g;
  int32_t B, H;
  int32_t nstrips, band, nbands;   // band: grid rows per workgroup, a multiple of 4 PR
  uint32_t m_s, s_s, m_b, s_b, m_h, s_h;   // exact multiply-shift divisions by nstrips, nbands and H
  float scale_log2, sm_scale;
  RopeDev rope;              // ROPE kernels: 8 rotary pairs per axis
  void *q_rot, *k_rot;       // forward: where the rotated q and k go (NULL: nowhere)
  int64_t qrs[4], krs[4];
};

// ---- fused rotation (D = 64, 8 rotary pairs per axis: the 16-byte pieces 0, 1 of a row turn by the row angle, 2, 3 by the
// column angle) --------------------------------------------------------------------------------------------------------
// Both tables (64 bytes per position) are copied into LDS once per workgroup when they fit: a table row is then four LDS reads
// behind the arrival of the token's index instead of a dependent global load.
constexpr int SWAG_TAB_BYTES = 8192;
struct SwagTab {
  swat_lds lds;
  bool in_lds;
  f32x4 part;   // the 16 bytes this thread copies
  DLT_DEV void fetch(swat_lds at, const RopeDev& rope, int tid) {
    lds = at;
    in_lds = (rope.row_len + rope.col_len) * 64 <= SWAG_TAB_BYTES;
    const int row = dlt_imin(tid >> 2, rope.row_len + rope.col_len - 1);   // 128 rows of four 16-byte parts
    const float* p = (row < rope.row_len ? rope.row_cs + (int64_t)row * rope.rs0 : rope.col_cs + (int64_t)(row - rope.row_len) * rope.cs0) + 4 * (tid & 3);
    part = f32x4{p[0], p[1], p[2], p[3]};
  }
  DLT_DEV void store(int tid) const { if (in_lds) *reinterpret_cast<DLT_LDS f32x4*>(lds + 16 * tid) = part; }
  // NF pairs of (cos, sin) from pair `first` on; false: the axis is not rotated
  template <int NV4>
  DLT_DEV bool get(f32x4 (&t)[NV4], int32_t id, int axis, int first, const RopeDev& rope) const {
    int pos = axis == 0 ? dlt_rope_row(id) : dlt_rope_col(id);
    const bool rotated = pos >= 0;
    pos = dlt_imax(0, dlt_imin(pos, (axis == 0 ? rope.row_len : rope.col_len) - 1));
    if (in_lds) {
      swat_lds p = lds + ((axis == 0 ? 0 : rope.row_len) + pos) * 64 + 8 * first;
#pragma unroll
      for (int j = 0; j < NV4; j++) t[j] = *reinterpret_cast<DLT_LDS f32x4*>(p + 16 * j);
    } else {
      const float* p = (axis == 0 ? rope.row_cs + (int64_t)pos * rope.rs0 : rope.col_cs + (int64_t)pos * rope.cs0) + 2 * first;
#pragma unroll
      for (int j = 0; j < NV4; j++) t[j] = f32x4{p[4 * j], p[4 * j + 1], p[4 * j + 2], p[4 * j + 3]};
    }
    return rotated;
  }
};

// one 16-byte piece turned with its partner piece: the arithmetic of the standalone rotation (every product rounded)
template <typename CT>
DLT_DEV u32x4 swag_turn(u32x4 self, u32x4 partner, const f32x4 (&t)[4], bool is_x0) {
  float x[8], y[8];
  unpack8<CT>(self, x);
  unpack8<CT>(partner, y);
  const unsigned sm = rope_sign_mask(is_x0, false);
#pragma unroll
  for (int j = 0; j < 8; j++) x[j] = rope_mix_signed(x[j], y[j], t[j >> 1][2 * (j & 1)], t[j >> 1][2 * (j & 1) + 1], sm);
  return pack8<CT>(x);
}
DLT_DEV unsigned swag_lane_xor16(unsigned v, int g) {
  typedef unsigned pair_t __attribute__((ext_vector_type(2)));
  const pair_t r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  return (g & 1) ? r.x : r.y;
}
DLT_DEV float swag_lane_xor32(float v, int g) {
  typedef unsigned pair_t __attribute__((ext_vector_type(2)));
  const unsigned u = __builtin_bit_cast(unsigned, v);
  const pair_t r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __builtin_bit_cast(float, (unsigned)(g < 2 ? r.y : r.x));
}
// Gradient rows (C layout) of rotated q or k -> of the caller's: rounded to the element type first (as the composition of the
// plain operator and the rotation does), then blocks 0 (row axis) and 1 (column axis) turned back.  Lane group g holds dims
// 4 g .. 4 g + 3 of a block, its rotary partners sit 32 lanes away; t[axis]: the pairs 4 (g & 1) .. + 3.
template <typename CT>
DLT_DEV void swag_turn_back(f32x4 (&acc)[4], float mul, const f32x4 (&t)[2][2], const bool (&rot)[2], int g) {
#pragma unroll
  for (int ax = 0; ax < 2; ax++) {
    const unsigned sm = rope_sign_mask(g < 2, true);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const float x = (float)(CT)(acc[ax][i] * mul), y = swag_lane_xor32(x, g);
      const float z = rope_mix_signed(x, y, t[ax][i >> 1][2 * (i & 1)], t[ax][i >> 1][2 * (i & 1) + 1], sm);
      acc[ax][i] = rot[ax] ? z : x;
    }
#pragma unroll
    for (int i = 0; i < 4; i++) acc[2 + ax][i] *= mul;
  }
}

template <int D, int NCH, int NCG, int PC>
struct Swag {
  static constexpr int STRIP = 4 * PC;                                 // own columns of a workgroup
  static constexpr int PR = 8 / PC, NRES = NCH + PR - 1;               // row groups, resident chunks
  static constexpr int NB = NCH * NCG, NP = (NB + 1) / 2;              // 4 x 4 key blocks of a window, pairs of them
  static constexpr int HCW = 4 * PC + 4 * (NCG - 1), TOK = 4 * HCW;    // staged columns, tokens of a chunk
  static constexpr int ROWB = 2 * D, TB = TOK * ROWB, SLOT = 2 * TB;
  static constexpr int PIECES = D / 8, NV = 2 * TOK * PIECES, NIT = (NV + 511) / 512;
  static constexpr int KC = D / 32, DB = D / 16;
  static constexpr int RING = NRES * SLOT, SCAL = NRES * 2 * TOK * 4;
  // waves per SIMD: two workgroups per CU where two rings and the registers fit
  static constexpr int OCC = RING + SCAL <= 80 * 1024 ? 4 : 2, OCC_BWD = D == 32 ? OCC : 2;
  static_assert((TOK * PIECES) % 64 == 0, "a wave stages one tensor per vector");
  static_assert(RING + SCAL <= 160 * 1024, "the ring exceeds the LDS");
};

// patch columns per workgroup: strips of 16 columns (strips of 32 with one row group per step stage fewer halo columns, but
// measured within 3 % on large grids and up to 18 % slower where the grid's width is no multiple of 32)
constexpr int SWAG_PC = 4;

template <int D> DLT_DEV int swag_swz(int row, int col) { return D == 32 ? (row & 1) << 1 : (col & 3) | ((row & 1) << 2); }

struct SwagWho { int b, h, r0, r1, c0; };
DLT_DEV SwagWho swag_who(const SwagArgs& a, int strip) {
  const int lin = xcd_remap(blockIdx.x, gridDim.x);
  SwagWho w;
  const int row = (int)dlt_fastdiv(lin, a.m_s, a.s_s), s = lin - row * a.nstrips;
  const int bh = (int)dlt_fastdiv(row, a.m_b, a.s_b), bd = row - bh * a.nbands;
  w.b = (int)dlt_fastdiv(bh, a.m_h, a.s_h);
  w.h = bh - w.b * a.H;
  w.c0 = s * strip;
  w.r0 = bd * a.band;
  w.r1 = dlt_imin(w.r0 + a.band, a.g.TR);
  return w;
}

template <typename C>
struct SwagRing {
  swat_lds lds;
  const char *base0, *base1;
  uint32_t rs0, rs1;                  // bytes between grid rows
  uint32_t goff[C::NIT];              // offset inside a grid row
  int hrow[C::NIT], loff[C::NIT];     // halo row inside a chunk; LDS offset inside a slot
  bool second[C::NIT];                // wave-uniform
  int tid, TR;

  DLT_DEV void init(swat_lds lds_, const char* b0, int sn0, const char* b1, int sn1, const SwagArgs& a, int c0, int tid_, int wave) {
    lds = lds_; base0 = b0; base1 = b1; tid = tid_; TR = a.g.TR;
    const int TC = a.g.TC;
    rs0 = (uint32_t)(TC * sn0 * 2);
    rs1 = (uint32_t)(TC * sn1 * 2);
#pragma unroll
    for (int it = 0; it < C::NIT; it++) {
      const int id = tid + 512 * it;
      second[it] = 64 * wave + 512 * it >= C::NV / 2;
      const int v = second[it] ? id - C::NV / 2 : id;
      const int tok = v / C::PIECES, piece = v % C::PIECES;
      hrow[it] = tok / C::HCW;
      const int hc = tok - hrow[it] * C::HCW;
      // columns outside the grid are clamped onto it: the window tests drop them
      const int col = dlt_imax(0, dlt_imin(c0 - a.g.WC + hc, TC - 1));
      goff[it] = (uint32_t)(col * (second[it] ? sn1 : sn0) * 2) + 16 * piece;
      loff[it] = (second[it] ? C::TB : 0) + tok * C::ROWB + 16 * (piece ^ swag_swz<C::ROWB / 2>(hrow[it], hc));
    }
  }
  DLT_DEV bool has(int it) const { return C::NV % 512 == 0 || it + 1 < C::NIT || tid + 512 * it < C::NV; }
  // first: grid row of the chunk's first halo row (rows outside the grid are clamped onto it)
  DLT_DEV void issue(u32x4 (&r)[C::NIT], int first) const {
#pragma unroll
    for (int it = 0; it < C::NIT; it++)
      if (has(it)) {
        const uint32_t rc = (uint32_t)dlt_imax(0, dlt_imin(first + hrow[it], TR - 1));
        r[it] = *reinterpret_cast<const u32x4*>((second[it] ? base1 : base0) + (goff[it] + rc * (second[it] ? rs1 : rs0)));
      }
  }
  DLT_DEV void commit(const u32x4 (&r)[C::NIT], int slot) const {
#pragma unroll
    for (int it = 0; it < C::NIT; it++)
      if (has(it)) swat_write16(lds + slot * C::SLOT + loff[it], r[it]);
  }
  // chunks of the first step: all requested before the first is written
  DLT_DEV void fill(int first) const {
    u32x4 pre[C::NRES][C::NIT];
#pragma unroll
    for (int i = 0; i < C::NRES; i++) issue(pre[i], first + 4 * i);
#pragma unroll
    for (int i = 0; i < C::NRES; i++) commit(pre[i], i);
  }
};

// Staging of the rotating forward kernel, two chunks at a time (what a step brings in).  A K item is half of a token row, pieces
// (2 h, 2 h + 1) = the rotary pair of axis h and (4 + 2 h, 5 + 2 h): a thread turns both partners of its pair with one read of the
// table row.  Waves 0 ... 3 take the K items of the first chunk (160 ... 224 of 256 threads), waves 4 ... 7 those of the second; the V
// pieces of both chunks run through all threads.  A thread's items have the same place in every pair of chunks, so offsets inside a
// grid row and inside a slot are formed once.
template <typename C>
struct SwagTurnStage {
  static constexpr int NV = (2 * C::TOK * 8 + 511) / 512;
  static_assert(C::PR == 2 && 2 * C::TOK <= 256 && (C::TOK * 8) % 64 == 0, "two chunks per step, a K item per thread, waves of one chunk");
  struct Data { u32x4 k[4], v[NV]; };
  const char *kb, *vb;
  uint32_t krs, vrs, koff, voff[NV];        // bytes between grid rows; offsets inside one
  int kchunk, krow, kcol, kl, vchunk[NV], vrow[NV], vl[NV];   // chunk (wave-uniform), halo row of the pair, column; offset in a slot
  bool kon, kown;
  uint32_t kout;                            // offset of the own token's rotated row inside a grid row
  int TR, TC, h;
  DLT_DEV void init(const char* kb_, int ksn, const char* vb_, int vsn, int krsn, const SwagArgs& a, int c0, int tid, int wave) {
    kb = kb_; vb = vb_; TR = a.g.TR; TC = a.g.TC;
    krs = (uint32_t)(TC * ksn);
    vrs = (uint32_t)(TC * vsn);
    h = tid & 1;
    const int x = tid & 255, kt = dlt_imin(x >> 1, C::TOK - 1), khr = kt / C::HCW, khc = kt - khr * C::HCW;
    kon = x < 2 * C::TOK;
    kchunk = wave >> 2;
    krow = 4 * kchunk + khr;
    const int col = c0 - a.g.WC + khc;
    kcol = dlt_imax(0, dlt_imin(col, TC - 1));
    koff = (uint32_t)(kcol * ksn) + 32 * h;
    kl = (khr * C::HCW + khc) * C::ROWB + 16 * ((2 * h) ^ swag_swz<64>(khr, khc));
    kown = col >= c0 && col < c0 + C::STRIP && col < TC;
    kout = (uint32_t)(kcol * krsn) + 32 * h;
#pragma unroll
    for (int i = 0; i < NV; i++) {
      vchunk[i] = 64 * wave + 512 * i >= C::TOK * 8;
      const int y = tid + 512 * i - (vchunk[i] ? C::TOK * 8 : 0), vt = dlt_imin(y >> 3, C::TOK - 1), hr = vt / C::HCW, hc = vt - hr * C::HCW;
      vrow[i] = 4 * vchunk[i] + hr;
      voff[i] = (uint32_t)(dlt_imax(0, dlt_imin(c0 - a.g.WC + hc, TC - 1)) * vsn) + 16 * (y & 7);
      vl[i] = C::TB + (hr * C::HCW + hc) * C::ROWB + 16 * ((y & 7) ^ swag_swz<64>(hr, hc));
    }
  }
  DLT_DEV bool von(int i, int wave) const { return 512 * (i + 1) <= 2 * C::TOK * 8 || 64 * wave + 512 * i < 2 * C::TOK * 8; }
  DLT_DEV uint32_t grid_row(int row) const { return (uint32_t)dlt_imax(0, dlt_imin(row, TR - 1)); }
  // rotary index of the K item (first: see issue)
  DLT_DEV int32_t index(const SwagArgs& a, int first) const { return a.rope.idx[grid_row(first + krow) * (uint32_t)TC + (uint32_t)kcol]; }
  // first: grid row of the first chunk's first halo row, the second chunk starts four rows further down; n: chunks wanted
  DLT_DEV void issue(Data& d, int first, int n, int wave) const {
    if (kon && kchunk < n) {
      const uint32_t r = grid_row(first + krow);
      const char* p = kb + (r * krs + koff);
      d.k[0] = *reinterpret_cast<const u32x4*>(p);
      d.k[1] = *reinterpret_cast<const u32x4*>(p + 16);
      d.k[2] = *reinterpret_cast<const u32x4*>(p + 64);
      d.k[3] = *reinterpret_cast<const u32x4*>(p + 80);
    }
#pragma unroll
    for (int i = 0; i < NV; i++)
      if (von(i, wave) && vchunk[i] < n) d.v[i] = *reinterpret_cast<const u32x4*>(vb + (grid_row(first + vrow[i]) * vrs + voff[i]));
  }
  // the K pair turned in registers; the workgroup's own tokens are also stored to `out` (NULL: nowhere)
  template <typename CT>
  DLT_DEV void turn(Data& d, const f32x4 (&t)[4], bool rot, char* out, uint32_t outrs, int first, int n, int r0, int r1) const {
    if (!(kon && kchunk < n)) return;
    if (rot) {
      const u32x4 x0 = d.k[0];
      d.k[0] = swag_turn<CT>(x0, d.k[1], t, true);
      d.k[1] = swag_turn<CT>(d.k[1], x0, t, false);
    }
    const int row = first + krow;
    if (out != nullptr && kown && row >= r0 && row < r1) {
      char* q = out + ((uint32_t)row * outrs + kout);
      store_stream16(q, d.k[0]);
      store_stream16(q + 16, d.k[1]);
      store_stream16(q + 64, d.k[2]);
      store_stream16(q + 80, d.k[3]);
    }
  }
  static DLT_DEV int slot_of(int s) { return (s >= C::NRES ? s - C::NRES : s) * C::SLOT; }
  DLT_DEV void commit_k(const Data& d, swat_lds lds, int slot0, int n) const {
    if (!(kon && kchunk < n)) return;
    swat_lds s = lds + slot_of(slot0 + kchunk);
    swat_write16(s + kl, d.k[0]);
    swat_write16(s + (kl ^ 16), d.k[1]);
    swat_write16(s + (kl ^ 64), d.k[2]);
    swat_write16(s + (kl ^ 80), d.k[3]);
  }
  DLT_DEV void commit_v(const Data& d, swat_lds lds, int slot0, int n, int wave) const {
#pragma unroll
    for (int i = 0; i < NV; i++)
      if (von(i, wave) && vchunk[i] < n) swat_write16(lds + slot_of(slot0 + vchunk[i]) + vl[i], d.v[i]);
  }
};

// lane parts of the operand addresses of a 4 x 4 block
template <typename C>
struct SwagLane {
  int row[C::KC], tr[C::DB];
  DLT_DEV void init(int n, int g) {
    constexpr int D = C::ROWB / 2;
#pragma unroll
    for (int c = 0; c < C::KC; c++) row[c] = ((n >> 2) * C::HCW + (n & 3)) * C::ROWB + 16 * ((4 * c + g) ^ swag_swz<D>(n >> 2, n));
#pragma unroll
    for (int d = 0; d < C::DB; d++)
      tr[d] = (g * C::HCW + (n >> 2)) * C::ROWB + 16 * ((2 * d + ((n >> 1) & 1)) ^ swag_swz<D>(g, n >> 2)) + 8 * (n & 1);
  }
};

// Common frame of the three kernels: who the wave is and what its lanes own.
template <typename C, int PC>
struct SwagFrame {
  int lane, n, g, wave, pc, rg;
  SwagWho w;
  int TR, TC, WR, WC;
  int col;          // own column (unclamped)
  int clo, chi;     // visible window columns of the own token
  DLT_DEV void init(const SwagArgs& a, int tid) {
    lane = tid & 63; n = lane & 15; g = lane >> 4;
    wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    pc = wave % PC; rg = wave / PC;
    w = swag_who(a, 4 * PC);
    TR = a.g.TR; TC = a.g.TC; WR = a.g.WR; WC = a.g.WC;
    const int cp = w.c0 + 4 * pc;
    col = cp + (n & 3);
    clo = dlt_imax(n & 3, WC - cp);
    chi = dlt_imin((n & 3) + 2 * WC, TC - 1 - cp + WC);
    if (col >= TC) chi = -1;
  }
  DLT_DEV bool sees_col(int j) const { return j >= clo && j <= chi; }
  // key rows 4 i + g are in the own token's window
  DLT_DEV bool sees_row(int i, int rp) const {
    const int hr = 4 * i + g, qr = n >> 2;
    const int lo = dlt_imax(qr, WR - rp), hi = dlt_imin(qr + 2 * WR, TR - 1 - rp + WR);
    return hr >= lo && hr <= hi;
  }
  // the same as the C operand of the score products: 0 or -inf
  DLT_DEV float row_bias(int i, int rp) const { return sees_row(i, rp) ? 0.f : -INFINITY; }
  DLT_DEV int own_row(int rp) const { return rp + (n >> 2); }
  DLT_DEV bool own_ok(int rp) const { return own_row(rp) < TR && col < TC; }
  // clamped token index of the own token
  DLT_DEV int own_tok(int rp) const { return dlt_imin(own_row(rp), TR - 1) * TC + dlt_imin(col, TC - 1); }
};

// Own rows leave straight from the accumulators: a lane of the C layout holds 4 dims of its token in each 16-dim block; the
// lane swap of two blocks gives every lane 8 consecutive dims (16 bytes), four lanes a whole 64-byte piece.  p: row of the lane's token.
template <typename CT, int DB>
DLT_DEV void swag_store_row(char* p, const f32x4 (&acc)[DB], float mul, int g) {
  typedef unsigned pair_t __attribute__((ext_vector_type(2)));
#pragma unroll
  for (int d = 0; d < DB; d += 2) {
    const pair_t lo = __builtin_amdgcn_permlane16_swap(pack2<CT>(acc[d][0] * mul, acc[d][1] * mul), pack2<CT>(acc[d + 1][0] * mul, acc[d + 1][1] * mul),
                                                       false, false);
    const pair_t hi = __builtin_amdgcn_permlane16_swap(pack2<CT>(acc[d][2] * mul, acc[d][3] * mul), pack2<CT>(acc[d + 1][2] * mul, acc[d + 1][3] * mul),
                                                       false, false);
    store_stream16(p + 2 * (16 * d + 16 * (g & 1) + 8 * (g >> 1)), u32x4{lo.x, hi.x, lo.y, hi.y});
  }
}

// scores of block (i, j) on top of `bias`
template <typename C, typename CT>
DLT_DEV f32x4 swag_scores(swat_lds blk, const SwagLane<C>& L, const u32x4 (&own)[C::KC], float bias) {
  f32x4 s = {bias, bias, bias, bias};
#pragma unroll
  for (int c = 0; c < C::KC; c++) s = Mma<CT>::mfma(swat_read16(blk + L.row[c]), own[c], s);
  return s;
}

// The forward pass of one patch where a key row holds an infinity or a NaN: block by block (`block(i, j)`: where it lies in LDS), every
// score outside the window replaced, the softmax online.  Rare: rolled, so that it costs the common path few registers.
template <typename C, typename CT, int NCG, typename Frame, typename Block>
DLT_DEV void swag_fwd_exact(const Frame& F, const SwagLane<C>& L, int rp, const u32x4 (&q)[C::KC], float scale, f32x4 (&acc)[C::DB], float& l, float& m_use,
                            Block block) {
  float m = -INFINITY, sum = 0.f;
#pragma unroll
  for (int d = 0; d < C::DB; d++) acc[d] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (int k = 0; k < C::NB; k++) {
    const int i = k / NCG, j = k - i * NCG;
    swat_lds blk = block(i, j);
    const bool row = F.sees_row(i, rp);
    f32x4 t = swag_scores<C, CT>(blk, L, q, 0.f);
#pragma unroll
    for (int e = 0; e < 4; e++) t[e] = row && F.sees_col(4 * j + e) ? t[e] : -INFINITY;
    const float m_new = fmaxf(m, wave_max4(fmaxf(fmaxf(t[0], t[1]), fmaxf(t[2], t[3]))));
    const float alpha = m_new == m ? 1.f : fast_exp2((m - m_new) * scale), neg_m2 = m_new == -INFINITY ? 0.f : -m_new * scale;
    m = m_new;
    float p[8];
#pragma unroll
    for (int e = 0; e < 4; e++) {
      p[e] = fast_exp2(fmaf(t[e], scale, neg_m2));
      p[4 + e] = 0.f;
    }
    const u32x4 pb = pack8<CT>(p);
    const unsigned one2 = pack2<CT>(1.f, 1.f);
    sum = dot2_acc<CT>(pb.y, one2, dot2_acc<CT>(pb.x, one2, sum * alpha));
#pragma unroll
    for (int d = 0; d < C::DB; d++) {
      const u32x2 v = swat_read_tr(blk + C::TB + L.tr[d]);
      acc[d] = Mma<CT>::mfma(u32x4{v.x, v.y, v.x, v.y}, pb, acc[d] * alpha);
    }
  }
  l = wave_sum4(sum);
  m_use = m == -INFINITY ? 0.f : m;
}

// Forward pass without rotation.
//
// With one workgroup per CU (head dim 32, the largest windows: two waves per SIMD) the LDS reads are placed by hand, K one row of
// blocks ahead of its products and V one pair of blocks: left to the compiler the read-ahead depends on the scalar registers that
// happen to be free (89 x 98, 32 slabs: 19 x 21 window 66 -> 59 us; 15 x 21 49.5 and 58 us in two builds, 51.7 here).  Where two
// workgroups share a CU the placed reads cost registers (64 x 64, 9 x 19 window 18.4 -> 25.7 us).
template <typename TIO, int D, int NCH, int NCG, int PC>
__global__ __launch_bounds__(512, (Swag<D, NCH, NCG, PC>::OCC)) void swag_fwd_kernel(const SwagArgs a) {
  typedef Swag<D, NCH, NCG, PC> C;
  typedef typename ComputeOf<TIO>::type CT;
  constexpr bool AHEAD = D == 32 && C::OCC == 2;
  extern __shared__ __align__(16) char smem[];
  swat_lds lds = (swat_lds)smem;
  const int tid = threadIdx.x;
  SwagFrame<C, PC> F;
  F.init(a, tid);
  const int b = F.w.b, h = F.w.h, n = F.n, g = F.g;
  const char* kb_ = reinterpret_cast<const char*>(reinterpret_cast<const TIO*>(a.k) + b * a.ks[0] + h * a.ks[1]);
  const char* vb_ = reinterpret_cast<const char*>(reinterpret_cast<const TIO*>(a.v) + b * a.vs[0] + h * a.vs[1]);
  const int ksn = (int)a.ks[2] * 2, vsn = (int)a.vs[2] * 2;
  SwagRing<C> ring;
  ring.init(lds, kb_, (int)a.ks[2], vb_, (int)a.vs[2], a, F.w.c0, tid, F.wave);
  const char* qb = reinterpret_cast<const char*>(reinterpret_cast<const TIO*>(a.q) + b * a.qs[0] + h * a.qs[1]) + 16 * g;
  char* ob = reinterpret_cast<char*>(reinterpret_cast<TIO*>(a.out_o) + b * a.os[0] + h * a.os[1]);
  float* lseb = a.lse + b * a.ls[0] + h * a.ls[1];
  const int qsn = (int)a.qs[2] * 2, osn = (int)a.os[2] * 2;
  SwagLane<C> L;
  L.init(n, g);
  const float scale = a.scale_log2;
  const unsigned one2 = pack2<CT>(1.f, 1.f);
  const u32x4 ones = {one2, one2, one2, one2};

  u32x4 qn[C::KC];
  auto load_q = [&](int rp) {
    const int tok = F.own_tok(rp);
#pragma unroll
    for (int c = 0; c < C::KC; c++) qn[c] = *reinterpret_cast<const u32x4*>(qb + (uint32_t)(tok * qsn) + 64 * c);
  };
  load_q(F.w.r0 + 4 * F.rg);
  ring.fill(F.w.r0 - F.WR);
  __syncthreads();

  int slot0 = 0;   // slot of the step's first chunk
  uint64_t any_bad = 0;
  for (int r = F.w.r0; r < F.w.r1; r += 4 * C::PR) {
    const int rp = r + 4 * F.rg;
    u32x4 q[C::KC];
#pragma unroll
    for (int c = 0; c < C::KC; c++) q[c] = qn[c];
    pin_loaded(q);
    const bool more = r + 4 * C::PR < F.w.r1;
    u32x4 nx[C::PR][C::NIT];
    const int next = r - F.WR + 4 * C::NRES;   // first halo row of the chunks to come
    if (more) {
#pragma unroll
      for (int i = 0; i < C::PR; i++) ring.issue(nx[i], next + 4 * i);
      load_q(rp + 4 * C::PR);
    }
    if (rp < F.TR && F.w.c0 + 4 * F.pc < F.TC) {
      swat_lds rowp[NCH];
#pragma unroll
      for (int i = 0; i < NCH; i++) {
        const int s = slot0 + F.rg + i;
        rowp[i] = lds + (s >= C::NRES ? s - C::NRES : s) * C::SLOT + 4 * F.pc * C::ROWB;
      }
      f32x4 s[C::NB + 1];
      float mx[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
      u32x4 ka[2][NCG][C::KC];
      auto read_row = [&](int i) {
#pragma unroll
        for (int j = 0; j < NCG; j++)
#pragma unroll
          for (int c = 0; c < C::KC; c++) ka[i & 1][j][c] = swat_read16(rowp[i] + 4 * j * C::ROWB + L.row[c]);
      };
      if constexpr (AHEAD) read_row(0);
#pragma unroll
      for (int i = 0; i < NCH; i++) {
        const float bias = F.row_bias(i, rp);
        if constexpr (AHEAD) {
          if (i + 1 < NCH) read_row(i + 1);
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int j = 0; j < NCG; j++) {
          f32x4 t = {bias, bias, bias, bias};
          if constexpr (AHEAD) {
#pragma unroll
            for (int c = 0; c < C::KC; c++) t = Mma<CT>::mfma(ka[i & 1][j][c], q[c], t);
          } else {
            t = swag_scores<C, CT>(rowp[i] + 4 * j * C::ROWB, L, q, bias);
          }
#pragma unroll
          for (int e = 0; e < 4; e++) t[e] = F.sees_col(4 * j + e) ? t[e] : -INFINITY;
          s[i * NCG + j] = t;
        }
      }
#pragma unroll
      for (int k = 0; k < C::NB; k += 2)
#pragma unroll
        for (int e = 0; e < 4; e++) mx[e] = fmaxf(fmaxf(mx[e], s[k][e]), s[k + 1 < C::NB ? k + 1 : k][e]);
      const float m = wave_max4(fmaxf(fmaxf(mx[0], mx[1]), fmaxf(mx[2], mx[3])));
      const float m_use = m == -INFINITY ? 0.f : m;   // own positions outside the grid see nothing
      const float neg_m2 = -m_use * scale;
      f32x4 acc[C::DB], acc_l = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int d = 0; d < C::DB; d++) acc[d] = f32x4{0.f, 0.f, 0.f, 0.f};
      u32x4 va[2][C::DB];
      auto read_v = [&](int t) {
        const int b0 = 2 * t, b1 = 2 * t + 1 < C::NB ? 2 * t + 1 : 2 * t;
        swat_lds v0 = rowp[b0 / NCG] + C::TB + 4 * (b0 % NCG) * C::ROWB, v1 = rowp[b1 / NCG] + C::TB + 4 * (b1 % NCG) * C::ROWB;
#pragma unroll
        for (int d = 0; d < C::DB; d++) {
          const u32x2 lo = swat_read_tr(v0 + L.tr[d]), hi = swat_read_tr(v1 + L.tr[d]);
          va[t & 1][d] = u32x4{lo.x, lo.y, hi.x, hi.y};
        }
      };
      if constexpr (AHEAD) read_v(0);
#pragma unroll
      for (int t = 0; t < C::NP; t++) {
        const int b0 = 2 * t, b1 = 2 * t + 1 < C::NB ? 2 * t + 1 : 2 * t;
        if constexpr (AHEAD) {
          if (t + 1 < C::NP) read_v(t + 1);
          __builtin_amdgcn_sched_barrier(0);
        }
        float p[8];
#pragma unroll
        for (int e = 0; e < 4; e++) {
          p[e] = fast_exp2(fmaf(s[b0][e], scale, neg_m2));
          p[4 + e] = 2 * t + 1 < C::NB ? fast_exp2(fmaf(s[b1][e], scale, neg_m2)) : 0.f;
        }
        const u32x4 pb = pack8<CT>(p);
        if constexpr (AHEAD) {
#pragma unroll
          for (int d = 0; d < C::DB; d++) acc[d] = Mma<CT>::mfma(va[t & 1][d], pb, acc[d]);
        } else {
          swat_lds v0 = rowp[b0 / NCG] + C::TB + 4 * (b0 % NCG) * C::ROWB, v1 = rowp[b1 / NCG] + C::TB + 4 * (b1 % NCG) * C::ROWB;
#pragma unroll
          for (int d = 0; d < C::DB; d++) {
            const u32x2 lo = swat_read_tr(v0 + L.tr[d]), hi = swat_read_tr(v1 + L.tr[d]);
            acc[d] = Mma<CT>::mfma(u32x4{lo.x, lo.y, hi.x, hi.y}, pb, acc[d]);
          }
        }
        acc_l = Mma<CT>::mfma(ones, pb, acc_l);
      }
      const float l = acc_l[0];
      any_bad |= __builtin_amdgcn_ballot_w64(l != l);
      if (F.own_ok(rp)) {
        const int tok = F.own_tok(rp);
        swag_store_row<CT, C::DB>(ob + (uint32_t)(tok * osn), acc, fast_rcp(l), g);
        if (g == 0) store_stream4(lseb + tok * a.ls[2], m_use * scale + fast_log2(l));
      }
    }
    if (more) {
      __syncthreads();
#pragma unroll
      for (int i = 0; i < C::PR; i++) ring.commit(nx[i], slot0 + i >= C::NRES ? slot0 + i - C::NRES : slot0 + i);
      __syncthreads();
      slot0 = slot0 + C::PR >= C::NRES ? slot0 + C::PR - C::NRES : slot0 + C::PR;
    }
  }
  // Patches of a wave that met such a key are formed again behind the march, from memory: every block of the window passes through
  // the wave's own 4 x 4 tokens of the ring.
  __syncthreads();
  if (any_bad) {
    keep_branch();
    constexpr int PER = D / 32;   // 16-byte pieces of a tensor's block per lane
    int lane = F.lane;
    asm volatile("" : "+v"(lane));   // keeps the addresses below out of the march
    swat_lds own = lds + F.rg * C::SLOT + 4 * F.pc * C::ROWB;
    for (int rp = F.w.r0 + 4 * F.rg; rp < dlt_imin(F.w.r1, F.TR); rp += 4 * C::PR) {
      load_q(rp);
      f32x4 acc[C::DB];
      float l, m_use;
      swag_fwd_exact<C, CT, NCG>(F, L, rp, qn, scale, acc, l, m_use, [&](int i, int j) {
#pragma unroll
        for (int x = 0; x < PER; x++) {
          const int id = lane + 64 * x, t = id / C::PIECES, piece = id % C::PIECES, lr = t >> 2, lc = t & 3;
          const int row = dlt_imax(0, dlt_imin(rp - F.WR + 4 * i + lr, F.TR - 1));
          const int tok = row * F.TC + dlt_imax(0, dlt_imin(F.w.c0 + 4 * (F.pc + j) - F.WC + lc, F.TC - 1));
          swat_lds p = own + (lr * C::HCW + lc) * C::ROWB + 16 * (piece ^ swag_swz<D>(lr, lc));
          swat_write16(p, *reinterpret_cast<const u32x4*>(kb_ + (uint32_t)(tok * ksn) + 16 * piece));
          swat_write16(p + C::TB, *reinterpret_cast<const u32x4*>(vb_ + (uint32_t)(tok * vsn) + 16 * piece));
        }
        return own;
      });
      if (F.own_ok(rp)) {
        const int tok = F.own_tok(rp);
        swag_store_row<CT, C::DB>(ob + (uint32_t)(tok * osn), acc, fast_rcp(l), g);
        if (g == 0) store_stream4(lseb + tok * a.ls[2], m_use * scale + fast_log2(l));
      }
    }
  }
}

// Forward pass with rotation: K is turned in registers between HBM and LDS, the own queries in theirs.
//
// At two steps per workgroup (2 x 8 slabs of 64 x 64, 13 x 13 window: one workgroup per CU) the time is the fill of the ring and
// the turning between two steps.  The chunks of the prologue are turned and written pair by pair as their loads return; indices are
// loaded a step ahead and table rows together with the data, so that nothing dependent is left behind the products; the last
// step is peeled (a conditional prefetch leaves loads pending across the back edge and every later wait becomes a full one).  Two
// waves per SIMD get the registers for that, also in the small window classes (5 x 5 spilled 70 registers at four).  Kernel trace,
// against chunks staged with the plain kernel's frame: 64 x 64 19.3 -> 16.7 us, 128 x 128 63 -> 56, 5 x 5 window on 64 x 64 17.0 -> 10.7.
template <typename TIO, int D, int NCH, int NCG, int PC>
__global__ __launch_bounds__(512, 2) void swag_fwd_rope_kernel(const SwagArgs a) {
  typedef Swag<D, NCH, NCG, PC> C;
  typedef typename ComputeOf<TIO>::type CT;
  extern __shared__ __align__(16) char smem[];
  swat_lds lds = (swat_lds)smem;
  const int tid = threadIdx.x;
  SwagFrame<C, PC> F;
  F.init(a, tid);
  const int b = F.w.b, h = F.w.h, n = F.n, g = F.g;
  const char* kb_ = reinterpret_cast<const char*>(reinterpret_cast<const TIO*>(a.k) + b * a.ks[0] + h * a.ks[1]);
  const char* vb_ = reinterpret_cast<const char*>(reinterpret_cast<const TIO*>(a.v) + b * a.vs[0] + h * a.vs[1]);
  const int ksn = (int)a.ks[2] * 2, vsn = (int)a.vs[2] * 2;
  const char* qb = reinterpret_cast<const char*>(reinterpret_cast<const TIO*>(a.q) + b * a.qs[0] + h * a.qs[1]) + 16 * g;
  char* ob = reinterpret_cast<char*>(reinterpret_cast<TIO*>(a.out_o) + b * a.os[0] + h * a.os[1]);
  float* lseb = a.lse + b * a.ls[0] + h * a.ls[1];
  const int qsn = (int)a.qs[2] * 2, osn = (int)a.os[2] * 2;
  SwagLane<C> L;
  L.init(n, g);
  const float scale = a.scale_log2;
  const unsigned one2 = pack2<CT>(1.f, 1.f);
  const u32x4 ones = {one2, one2, one2, one2};

  SwagTab tab;
  char *krb = nullptr, *qrb = nullptr;
  tab.fetch(lds + C::RING, a.rope, tid);   // requested first: it does not depend on any index
  if (a.k_rot != nullptr) {
    krb = reinterpret_cast<char*>(reinterpret_cast<TIO*>(a.k_rot) + b * a.krs[0] + h * a.krs[1]);
    qrb = reinterpret_cast<char*>(reinterpret_cast<TIO*>(a.q_rot) + b * a.qrs[0] + h * a.qrs[1]) + 16 * g;
  }
  const int krsn = (int)a.krs[2] * 2, qrsn = (int)a.qrs[2] * 2;
  u32x4 qn[C::KC];
  auto load_q = [&](int rp) {
    const int tok = F.own_tok(rp);
#pragma unroll
    for (int c = 0; c < C::KC; c++) qn[c] = *reinterpret_cast<const u32x4*>(qb + (uint32_t)(tok * qsn) + 64 * c);
  };
  // the own queries of patch rp turned in registers and stored
  auto turn_q = [&](int rp, const f32x4 (&t)[4], bool rot) {
    const u32x4 partner = {swag_lane_xor16(qn[0].x, g), swag_lane_xor16(qn[0].y, g), swag_lane_xor16(qn[0].z, g), swag_lane_xor16(qn[0].w, g)};
    if (rot) qn[0] = swag_turn<CT>(qn[0], partner, t, (g & 1) == 0);
    if (qrb != nullptr && F.own_ok(rp)) {
#pragma unroll
      for (int c = 0; c < C::KC; c++) store_stream16(qrb + (uint32_t)(F.own_tok(rp) * qrsn) + 64 * c, qn[c]);
    }
  };
  typedef SwagTurnStage<C> Stage;
  Stage stage;
  const uint32_t outrs = (uint32_t)(F.TC * krsn);
  stage.init(kb_, ksn, vb_, vsn, krsn, a, F.w.c0, tid, F.wave);
  constexpr int NPAIR = (C::NRES + 1) / 2;
  typename Stage::Data pre[NPAIR];
  int32_t id[NPAIR];
#pragma unroll
  for (int j = 0; j < NPAIR; j++) id[j] = stage.index(a, F.w.r0 - F.WR + 8 * j);
  const int32_t idq0 = a.rope.idx[F.own_tok(F.w.r0 + 4 * F.rg)];
#pragma unroll
  for (int j = 0; j < NPAIR; j++) stage.issue(pre[j], F.w.r0 - F.WR + 8 * j, C::NRES - 2 * j, F.wave);
  load_q(F.w.r0 + 4 * F.rg);
  // rotary indices of the next step's K item and own queries: always loaded a step ahead
  int32_t idk = stage.index(a, F.w.r0 - F.WR + 4 * C::NRES);
  int32_t idq = a.rope.idx[F.own_tok(F.w.r0 + 4 * F.rg + 4 * C::PR)];
  tab.store(tid);
  __syncthreads();
#pragma unroll
  for (int j = 0; j < NPAIR; j++) {
    f32x4 t[4];
    const bool rot = tab.get(t, id[j], stage.h, 0, a.rope);
    stage.template turn<CT>(pre[j], t, rot, krb, outrs, F.w.r0 - F.WR + 8 * j, C::NRES - 2 * j, F.w.r0, F.w.r1);
    stage.commit_k(pre[j], lds, 2 * j, C::NRES - 2 * j);
    stage.commit_v(pre[j], lds, 2 * j, C::NRES - 2 * j, F.wave);
  }
  {
    f32x4 t[4];
    const bool rot = tab.get(t, idq0, g >> 1, 0, a.rope);
    turn_q(F.w.r0 + 4 * F.rg, t, rot);
  }
  __syncthreads();

  int slot0 = 0;   // slot of the step's first chunk
  auto store = [&](int rp, const f32x4 (&acc)[C::DB], float l, float m_use) {
    if (F.own_ok(rp)) {
      const int tok = F.own_tok(rp);
      swag_store_row<CT, C::DB>(ob + (uint32_t)(tok * osn), acc, fast_rcp(l), g);
      if (g == 0) store_stream4(lseb + tok * a.ls[2], m_use * scale + fast_log2(l));
    }
  };
  // scores, softmax and output of the patch whose first own row is rp; q: its queries
  auto attend = [&](int rp, const u32x4 (&q)[C::KC]) __attribute__((always_inline)) {
    if (rp < F.TR && F.w.c0 + 4 * F.pc < F.TC) {
      swat_lds rowp[NCH];
#pragma unroll
      for (int i = 0; i < NCH; i++) {
        const int s = slot0 + F.rg + i;
        rowp[i] = lds + (s >= C::NRES ? s - C::NRES : s) * C::SLOT + 4 * F.pc * C::ROWB;
      }
      f32x4 s[C::NB + 1];
      float mx[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
#pragma unroll
      for (int i = 0; i < NCH; i++) {
        const float bias = F.row_bias(i, rp);
#pragma unroll
        for (int j = 0; j < NCG; j++) {
          f32x4 t = swag_scores<C, CT>(rowp[i] + 4 * j * C::ROWB, L, q, bias);
#pragma unroll
          for (int e = 0; e < 4; e++) t[e] = F.sees_col(4 * j + e) ? t[e] : -INFINITY;
          s[i * NCG + j] = t;
        }
      }
#pragma unroll
      for (int k = 0; k < C::NB; k += 2)
#pragma unroll
        for (int e = 0; e < 4; e++) mx[e] = fmaxf(fmaxf(mx[e], s[k][e]), s[k + 1 < C::NB ? k + 1 : k][e]);
      const float m = wave_max4(fmaxf(fmaxf(mx[0], mx[1]), fmaxf(mx[2], mx[3])));
      float m_use = m == -INFINITY ? 0.f : m;   // own positions outside the grid see nothing
      const float neg_m2 = -m_use * scale;
      f32x4 acc[C::DB], acc_l = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int d = 0; d < C::DB; d++) acc[d] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < C::NP; t++) {
        const int b0 = 2 * t, b1 = 2 * t + 1 < C::NB ? 2 * t + 1 : 2 * t;
        float p[8];
#pragma unroll
        for (int e = 0; e < 4; e++) {
          p[e] = fast_exp2(fmaf(s[b0][e], scale, neg_m2));
          p[4 + e] = 2 * t + 1 < C::NB ? fast_exp2(fmaf(s[b1][e], scale, neg_m2)) : 0.f;
        }
        const u32x4 pb = pack8<CT>(p);
        swat_lds v0 = rowp[b0 / NCG] + C::TB + 4 * (b0 % NCG) * C::ROWB, v1 = rowp[b1 / NCG] + C::TB + 4 * (b1 % NCG) * C::ROWB;
#pragma unroll
        for (int d = 0; d < C::DB; d++) {
          const u32x2 lo = swat_read_tr(v0 + L.tr[d]), hi = swat_read_tr(v1 + L.tr[d]);
          acc[d] = Mma<CT>::mfma(u32x4{lo.x, lo.y, hi.x, hi.y}, pb, acc[d]);
        }
        acc_l = Mma<CT>::mfma(ones, pb, acc_l);
      }
      float l = acc_l[0];
      if (__builtin_amdgcn_ballot_w64(l != l)) {   // an infinite or NaN key in or beside the window of some query
        keep_branch();
        swag_fwd_exact<C, CT, NCG>(F, L, rp, q, scale, acc, l, m_use, [&](int i, int j) {
          const int s = slot0 + F.rg + i;
          return lds + (s >= C::NRES ? s - C::NRES : s) * C::SLOT + 4 * (F.pc + j) * C::ROWB;
        });
      }
      store(rp, acc, l, m_use);
    }
  };
  int r = F.w.r0;
  for (; r + 4 * C::PR < F.w.r1; r += 4 * C::PR) {
    const int rp = r + 4 * F.rg, next = r - F.WR + 4 * C::NRES;   // next: first halo row of the chunks to come
    u32x4 q[C::KC];
#pragma unroll
    for (int c = 0; c < C::KC; c++) q[c] = qn[c];
    // the table rows are requested with the data and there when the products are done
    f32x4 tk[4], tq[4];
    const bool rk = tab.get(tk, idk, stage.h, 0, a.rope), rq = tab.get(tq, idq, g >> 1, 0, a.rope);
    typename Stage::Data nt;
    stage.issue(nt, next, 2, F.wave);
    idk = stage.index(a, next + 4 * C::PR);
    idq = a.rope.idx[F.own_tok(rp + 8 * C::PR)];
    load_q(rp + 4 * C::PR);
    attend(rp, q);
    stage.template turn<CT>(nt, tk, rk, krb, outrs, next, 2, F.w.r0, F.w.r1);
    turn_q(rp + 4 * C::PR, tq, rq);
    __syncthreads();
    stage.commit_k(nt, lds, slot0, 2);
    stage.commit_v(nt, lds, slot0, 2, F.wave);
    __syncthreads();
    slot0 = slot0 + C::PR >= C::NRES ? slot0 + C::PR - C::NRES : slot0 + C::PR;
  }
  attend(r + 4 * F.rg, qn);
}

// dQ: own = queries, K and V in the ring; delta = rowsum(o dO) of the own queries is formed and stored on the way.
// ROPE (both backward kernels): q and k arrive rotated, the gradients are turned back on their way out.
template <typename TIO, int D, int NCH, int NCG, int PC, bool ROPE>
__global__ __launch_bounds__(512, (Swag<D, NCH, NCG, PC>::OCC_BWD)) void swag_bwd_q_kernel(const SwagArgs a) {
  typedef Swag<D, NCH, NCG, PC> C;
  typedef typename ComputeOf<TIO>::type CT;
  extern __shared__ __align__(16) char smem[];
  swat_lds lds = (swat_lds)smem;
  const int tid = threadIdx.x;
  SwagFrame<C, PC> F;
  F.init(a, tid);
  const int b = F.w.b, h = F.w.h, n = F.n, g = F.g;
  SwagRing<C> ring;
  ring.init(lds, reinterpret_cast<const char*>(reinterpret_cast<const TIO*>(a.k) + b * a.ks[0] + h * a.ks[1]), (int)a.ks[2],
            reinterpret_cast<const char*>(reinterpret_cast<const TIO*>(a.v) + b * a.vs[0] + h * a.vs[1]), (int)a.vs[2], a, F.w.c0, tid, F.wave);
  const char* qb = reinterpret_cast<const char*>(reinterpret_cast<const TIO*>(a.q) + b * a.qs[0] + h * a.qs[1]) + 16 * g;
  const char* dob = reinterpret_cast<const char*>(reinterpret_cast<const TIO*>(a.d_o) + b * a.dos[0] + h * a.dos[1]) + 16 * g;
  const char* ob = reinterpret_cast<const char*>(reinterpret_cast<const TIO*>(a.o) + b * a.os[0] + h * a.os[1]) + 16 * g;
  char* dqb = reinterpret_cast<char*>(reinterpret_cast<TIO*>(a.dq) + b * a.dqs[0] + h * a.dqs[1]);
  const float* lseb = a.lse + b * a.ls[0] + h * a.ls[1];
  float* delb = a.delta + b * a.ls[0] + h * a.ls[1];
  const int qsn = (int)a.qs[2] * 2, dosn = (int)a.dos[2] * 2, osn = (int)a.os[2] * 2, dqsn = (int)a.dqs[2] * 2;
  SwagLane<C> L;
  L.init(n, g);
  const float scale = a.scale_log2;

  SwagTab tab;
  tab.in_lds = false;
  int32_t idn = -1;
  u32x4 qn[C::KC], don[C::KC], on[C::KC];
  float lsen;
  auto load_own = [&](int rp) {
    const int tok = F.own_tok(rp);
#pragma unroll
    for (int c = 0; c < C::KC; c++) {
      qn[c] = *reinterpret_cast<const u32x4*>(qb + (uint32_t)(tok * qsn) + 64 * c);
      don[c] = *reinterpret_cast<const u32x4*>(dob + (uint32_t)(tok * dosn) + 64 * c);
      on[c] = *reinterpret_cast<const u32x4*>(ob + (uint32_t)(tok * osn) + 64 * c);
    }
    lsen = lseb[tok * a.ls[2]];
    if constexpr (ROPE) idn = a.rope.idx[tok];
  };
  load_own(F.w.r0 + 4 * F.rg);
  ring.fill(F.w.r0 - F.WR);
  __syncthreads();

  int slot0 = 0;
  for (int r = F.w.r0; r < F.w.r1; r += 4 * C::PR) {
    const int rp = r + 4 * F.rg;
    u32x4 q[C::KC], d_o[C::KC];
    float part = 0.f;
#pragma unroll
    for (int c = 0; c < C::KC; c++) {
      q[c] = qn[c];
      d_o[c] = don[c];
      float fo[8], fd[8];
      unpack8<CT>(on[c], fo);
      unpack8<CT>(d_o[c], fd);
#pragma unroll
      for (int j = 0; j < 8; j++) part += fo[j] * fd[j];
    }
    pin_loaded(q);
    const float nlse = -lsen;
    const float del = wave_sum4(part);
    const bool ok = F.own_ok(rp);
    f32x4 tr[2][2];
    bool rot[2];
    if constexpr (ROPE) {
#pragma unroll
      for (int ax = 0; ax < 2; ax++) rot[ax] = tab.get(tr[ax], idn, ax, 4 * (g & 1), a.rope);
    }
    if (g == 0 && ok) store_stream4(delb + F.own_tok(rp) * a.ls[2], del);
    const bool more = r + 4 * C::PR < F.w.r1;
    u32x4 nx[C::PR][C::NIT];
    if (more) {
#pragma unroll
      for (int i = 0; i < C::PR; i++) ring.issue(nx[i], r - F.WR + 4 * (C::NRES + i));
      load_own(rp + 4 * C::PR);
    }
    if (rp < F.TR && F.w.c0 + 4 * F.pc < F.TC) {
      swat_lds rowp[NCH];
#pragma unroll
      for (int i = 0; i < NCH; i++) {
        const int s = slot0 + F.rg + i;
        rowp[i] = lds + (s >= C::NRES ? s - C::NRES : s) * C::SLOT + 4 * F.pc * C::ROWB;
      }
      f32x4 acc[C::DB];
#pragma unroll
      for (int d = 0; d < C::DB; d++) acc[d] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < C::NP; t++) {
        float ds[8];
#pragma unroll
        for (int u = 0; u < 2; u++) {
          const int k = 2 * t + u;
          if (k >= C::NB) {
#pragma unroll
            for (int e = 0; e < 4; e++) ds[4 * u + e] = 0.f;
            continue;
          }
          swat_lds kp = rowp[k / NCG] + 4 * (k % NCG) * C::ROWB;
          const f32x4 s = swag_scores<C, CT>(kp, L, q, F.row_bias(k / NCG, rp));
          // the dP products start from -delta: the matrix pipe delivers dP - delta
          f32x4 dp = {-del, -del, -del, -del};
#pragma unroll
          for (int c = 0; c < C::KC; c++) dp = Mma<CT>::mfma(swat_read16(kp + C::TB + L.row[c]), d_o[c], dp);
#pragma unroll
          for (int e = 0; e < 4; e++) {
            const float pv = fast_exp2(fmaf(s[e], scale, nlse));
            ds[4 * u + e] = (F.sees_col(4 * (k % NCG) + e) ? pv : 0.f) * dp[e];
          }
        }
        const u32x4 dsb = pack8<CT>(ds);
        const int b0 = 2 * t, b1 = 2 * t + 1 < C::NB ? 2 * t + 1 : 2 * t;
        swat_lds k0 = rowp[b0 / NCG] + 4 * (b0 % NCG) * C::ROWB, k1 = rowp[b1 / NCG] + 4 * (b1 % NCG) * C::ROWB;
#pragma unroll
        for (int d = 0; d < C::DB; d++) {
          const u32x2 lo = swat_read_tr(k0 + L.tr[d]), hi = swat_read_tr(k1 + L.tr[d]);
          acc[d] = Mma<CT>::mfma(u32x4{lo.x, lo.y, hi.x, hi.y}, dsb, acc[d]);
        }
      }
      if constexpr (ROPE) swag_turn_back<CT>(acc, a.sm_scale, tr, rot, g);
      if (ok) swag_store_row<CT, C::DB>(dqb + (uint32_t)(F.own_tok(rp) * dqsn), acc, ROPE ? 1.f : a.sm_scale, g);
    }
    if (more) {
      __syncthreads();
#pragma unroll
      for (int i = 0; i < C::PR; i++) ring.commit(nx[i], slot0 + i >= C::NRES ? slot0 + i - C::NRES : slot0 + i);
      __syncthreads();
      slot0 = slot0 + C::PR >= C::NRES ? slot0 + C::PR - C::NRES : slot0 + C::PR;
    }
  }
}

// dK / dV: own = keys, Q and dO in the ring with -lse2 and delta of their tokens behind it (the window is symmetric).
template <typename TIO, int D, int NCH, int NCG, int PC, bool ROPE>
__global__ __launch_bounds__(512, (Swag<D, NCH, NCG, PC>::OCC_BWD)) void swag_bwd_kv_kernel(const SwagArgs a) {
  typedef Swag<D, NCH, NCG, PC> C;
  typedef typename ComputeOf<TIO>::type CT;
  extern __shared__ __align__(16) char smem[];
  swat_lds lds = (swat_lds)smem;
  const int tid = threadIdx.x;
  SwagFrame<C, PC> F;
  F.init(a, tid);
  const int b = F.w.b, h = F.w.h, n = F.n, g = F.g;
  SwagRing<C> ring;
  ring.init(lds, reinterpret_cast<const char*>(reinterpret_cast<const TIO*>(a.q) + b * a.qs[0] + h * a.qs[1]), (int)a.qs[2],
            reinterpret_cast<const char*>(reinterpret_cast<const TIO*>(a.d_o) + b * a.dos[0] + h * a.dos[1]), (int)a.dos[2], a, F.w.c0, tid, F.wave);
  const float* lseb = a.lse + b * a.ls[0] + h * a.ls[1];
  const float* delb = a.delta + b * a.ls[0] + h * a.ls[1];
  DLT_LDS float* scal = reinterpret_cast<DLT_LDS float*>(lds + C::RING);   // [slot][-lse2 | delta][token]
  const int shr = tid / C::HCW, shc = tid - shr * C::HCW;
  const int scol = dlt_imax(0, dlt_imin(F.w.c0 - F.WC + shc, F.TC - 1));
  auto issue_scal = [&](float& x, float& y, int first) {
    if (tid < C::TOK) {
      const int tok = dlt_imax(0, dlt_imin(first + shr, F.TR - 1)) * F.TC + scol;
      x = lseb[tok * a.ls[2]];
      y = delb[tok * a.ls[2]];
    }
  };
  auto commit_scal = [&](float x, float y, int slot) {
    if (tid < C::TOK) {
      scal[slot * 2 * C::TOK + tid] = -x;
      scal[slot * 2 * C::TOK + C::TOK + tid] = y;
    }
  };
  const char* kb = reinterpret_cast<const char*>(reinterpret_cast<const TIO*>(a.k) + b * a.ks[0] + h * a.ks[1]) + 16 * g;
  const char* vb = reinterpret_cast<const char*>(reinterpret_cast<const TIO*>(a.v) + b * a.vs[0] + h * a.vs[1]) + 16 * g;
  char* dkb = reinterpret_cast<char*>(reinterpret_cast<TIO*>(a.dk) + b * a.dks[0] + h * a.dks[1]);
  char* dvb = reinterpret_cast<char*>(reinterpret_cast<TIO*>(a.dv) + b * a.dvs[0] + h * a.dvs[1]);
  const int ksn = (int)a.ks[2] * 2, vsn = (int)a.vs[2] * 2, dksn = (int)a.dks[2] * 2, dvsn = (int)a.dvs[2] * 2;
  SwagLane<C> L;
  L.init(n, g);
  const float scale = a.scale_log2;

  SwagTab tab;
  tab.in_lds = false;
  int32_t idn = -1;
  u32x4 kn[C::KC], vn[C::KC];
  auto load_own = [&](int rp) {
    const int tok = F.own_tok(rp);
    if constexpr (ROPE) idn = a.rope.idx[tok];
#pragma unroll
    for (int c = 0; c < C::KC; c++) {
      kn[c] = *reinterpret_cast<const u32x4*>(kb + (uint32_t)(tok * ksn) + 64 * c);
      vn[c] = *reinterpret_cast<const u32x4*>(vb + (uint32_t)(tok * vsn) + 64 * c);
    }
  };
  load_own(F.w.r0 + 4 * F.rg);
  ring.fill(F.w.r0 - F.WR);
  {
    float x[C::NRES], y[C::NRES];
#pragma unroll
    for (int i = 0; i < C::NRES; i++) issue_scal(x[i], y[i], F.w.r0 - F.WR + 4 * i);
#pragma unroll
    for (int i = 0; i < C::NRES; i++) commit_scal(x[i], y[i], i);
  }
  __syncthreads();

  int slot0 = 0;
  for (int r = F.w.r0; r < F.w.r1; r += 4 * C::PR) {
    const int rp = r + 4 * F.rg;
    // the own values are negated and the dP products start from the staged delta: the matrix pipe delivers -(dP - delta)
    u32x4 k_[C::KC], v_[C::KC];
#pragma unroll
    for (int c = 0; c < C::KC; c++) {
      k_[c] = kn[c];
      v_[c] = u32x4{vn[c].x ^ 0x80008000u, vn[c].y ^ 0x80008000u, vn[c].z ^ 0x80008000u, vn[c].w ^ 0x80008000u};
    }
    pin_loaded(k_);
    pin_loaded(v_);
    f32x4 tr[2][2];
    bool rot[2];
    if constexpr (ROPE) {
#pragma unroll
      for (int ax = 0; ax < 2; ax++) rot[ax] = tab.get(tr[ax], idn, ax, 4 * (g & 1), a.rope);
    }
    const bool more = r + 4 * C::PR < F.w.r1;
    u32x4 nx[C::PR][C::NIT];
    float sx[C::PR], sy[C::PR];
    if (more) {
#pragma unroll
      for (int i = 0; i < C::PR; i++) {
        ring.issue(nx[i], r - F.WR + 4 * (C::NRES + i));
        issue_scal(sx[i], sy[i], r - F.WR + 4 * (C::NRES + i));
      }
      load_own(rp + 4 * C::PR);
    }
    if (rp < F.TR && F.w.c0 + 4 * F.pc < F.TC) {
      swat_lds rowp[NCH];
      DLT_LDS float* scp[NCH];
#pragma unroll
      for (int i = 0; i < NCH; i++) {
        const int s0 = slot0 + F.rg + i, s = s0 >= C::NRES ? s0 - C::NRES : s0;
        rowp[i] = lds + s * C::SLOT + 4 * F.pc * C::ROWB;
        scp[i] = scal + s * 2 * C::TOK + g * C::HCW + 4 * F.pc;
      }
      f32x4 acc_k[C::DB], acc_v[C::DB];
#pragma unroll
      for (int d = 0; d < C::DB; d++) acc_k[d] = acc_v[d] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < C::NP; t++) {
        float p[8], ds[8];
#pragma unroll
        for (int u = 0; u < 2; u++) {
          const int k = 2 * t + u;
          if (k >= C::NB) {
#pragma unroll
            for (int e = 0; e < 4; e++) p[4 * u + e] = ds[4 * u + e] = 0.f;
            continue;
          }
          swat_lds qp = rowp[k / NCG] + 4 * (k % NCG) * C::ROWB;
          DLT_LDS float* sp = scp[k / NCG] + 4 * (k % NCG);
          const f32x4 nl = *reinterpret_cast<DLT_LDS f32x4*>(sp);
          const f32x4 s = swag_scores<C, CT>(qp, L, k_, F.row_bias(k / NCG, rp));
          f32x4 dp = *reinterpret_cast<DLT_LDS f32x4*>(sp + C::TOK);
#pragma unroll
          for (int c = 0; c < C::KC; c++) dp = Mma<CT>::mfma(swat_read16(qp + C::TB + L.row[c]), v_[c], dp);
#pragma unroll
          for (int e = 0; e < 4; e++) {
            const float x = fast_exp2(fmaf(s[e], scale, nl[e])), pv = F.sees_col(4 * (k % NCG) + e) ? x : 0.f;
            p[4 * u + e] = pv;
            ds[4 * u + e] = -pv * dp[e];
          }
        }
        const u32x4 pb = pack8<CT>(p), dsb = pack8<CT>(ds);
        const int b0 = 2 * t, b1 = 2 * t + 1 < C::NB ? 2 * t + 1 : 2 * t;
        swat_lds q0 = rowp[b0 / NCG] + 4 * (b0 % NCG) * C::ROWB, q1 = rowp[b1 / NCG] + 4 * (b1 % NCG) * C::ROWB;
#pragma unroll
        for (int d = 0; d < C::DB; d++) {
          const u32x2 lo = swat_read_tr(q0 + C::TB + L.tr[d]), hi = swat_read_tr(q1 + C::TB + L.tr[d]);
          acc_v[d] = Mma<CT>::mfma(u32x4{lo.x, lo.y, hi.x, hi.y}, pb, acc_v[d]);
        }
#pragma unroll
        for (int d = 0; d < C::DB; d++) {
          const u32x2 lo = swat_read_tr(q0 + L.tr[d]), hi = swat_read_tr(q1 + L.tr[d]);
          acc_k[d] = Mma<CT>::mfma(u32x4{lo.x, lo.y, hi.x, hi.y}, dsb, acc_k[d]);
        }
      }
      if constexpr (ROPE) swag_turn_back<CT>(acc_k, a.sm_scale, tr, rot, g);
      if (F.own_ok(rp)) {
        const int tok = F.own_tok(rp);
        swag_store_row<CT, C::DB>(dvb + (uint32_t)(tok * dvsn), acc_v, 1.f, g);
        swag_store_row<CT, C::DB>(dkb + (uint32_t)(tok * dksn), acc_k, ROPE ? 1.f : a.sm_scale, g);
      }
    }
    if (more) {
      __syncthreads();
#pragma unroll
      for (int i = 0; i < C::PR; i++) {
        const int slot = slot0 + i >= C::NRES ? slot0 + i - C::NRES : slot0 + i;
        ring.commit(nx[i], slot);
        commit_scal(sx[i], sy[i], slot);
      }
      __syncthreads();
      slot0 = slot0 + C::PR >= C::NRES ? slot0 + C::PR - C::NRES : slot0 + C::PR;
    }
  }
}
