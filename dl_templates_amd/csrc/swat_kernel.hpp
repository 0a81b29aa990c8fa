// Marching kernels for windows over tiles of 16 or 32 tokens at head dim 32 / 64, forward also at 128 (the reference's demo regime,
// src/tiled_swa.py:142-244 and :741-750), in the token layout and in the image layout.
//
// What bounded the chunked kernels here: a query tile sees only 9 ... 25 tiles, so a workgroup of 128 queries walked nine
// 64-token chunks, each a load, two barriers and work for one or two of its four waves (image layout, B = 4, H = 8,
// 256 x 256 pixels, 4 x 4-pixel tiles, d = 32: forward 301 us for 537 MB, latency of 9 rounds, 1.8 TB/s).
// Here a workgroup owns a strip of 8 blocks of 16 tokens (one per wave; 4 at head dim 64 with five window rows and at 128) and marches down the grid rows.  The rows its
// window covers (2 WR + 1 grid rows of both streamed tensors) live in an LDS ring; a step needs one new row, which travels
// HBM -> registers while the step computes, so every row is fetched once per strip and the loads of a step have a whole
// step to arrive.  All tiles of the window are resident: the softmax is one-shot, there is no mask inside a tile (a block of
// 16 tokens lies inside one tile), and only tiles at the border of the grid test their neighbours' existence.
//
// LDS: token rows of 2 D bytes, 16-byte piece p of token t at p ^ swz(t): operand reads, transposing reads and staging
// writes are free of bank conflicts without padding, so that at D = 32 with a 3 x 3 window the ring takes 60 KB and two
// workgroups (16 waves) share a CU.
#pragma once
#include <type_traits>
#include "swa1_common.hpp"

struct SwatArgs {
  const void *q, *k, *v, *o, *d_o;
  void *out_o, *dq, *dk, *dv;
  float* lse;
  float* delta;
  int64_t qs[5], ks[5], vs[5], os[5], dos[5], dqs[5], dks[5], dvs[5], ls[3];
  const void* ring_p[4];   // swat_bwd_kernel: K, V, Q, dO as its ring holds them, picked by a wave-uniform index
  int64_t ring_s[4][5];
  DltTokMap tm;
  DltGeom g;
  int32_t B, H;
  int32_t nstrips, band, nbands;
  float scale_log2, sm_scale;
  int32_t lone;   // host only, forward: one workgroup per CU (dlt_image_fwd_alone)
  int32_t one;    // host only, backward: swat_bwd_kernel (dlt_tile_bwd_one_launch)
};

template <int D, int NTB, int WC, int WR>
struct Swat {
  static constexpr int NWB = (2 * WC + 1) * NTB, NR = 2 * WR + 1;   // 16-token blocks per window row, window rows
  static constexpr int NB = NR * NWB, NP = (NB + 1) / 2;            // blocks of a window, pairs of them (32 tokens of a product)
  // strips of four blocks where a ring of eight exceeds the LDS; one wave per SIMD then, with all of its registers
  static constexpr int SB = D == 128 || (D == 64 && WR == 2) ? 4 : 8, THREADS = 64 * SB;   // 16-token blocks of a strip, one per wave
  // Strips of four write slots outside the grid as zeros: their probabilities are 0, and 0 times an infinite value is not.  A workgroup there fills a
  // ring of up to 147 KB, beside which the ANDs are 0 ... 3 %; strips of eight, which it would cost 1 ... 4 % (32 slabs of 16 x 16 tiles, d = 32: 10.7 -> 11.1 us), hold copies of the edge
  static constexpr bool CLEAR = SB == 4;
  // The last of an odd number of blocks has zeros beside it instead of its values again, for the same reason: no time or less but at five columns and strips of
  // eight (d = 64, 16 slabs of 40 x 40 tiles: forward 52.4 -> 53.4 us, backward 151 -> 162)
  static constexpr bool ALONE = CLEAR || WC == 1;
  static constexpr int HB = SB + 2 * WC * NTB, TOK = 16 * HB;       // staged blocks / tokens per grid row
  static constexpr int ROWB = 2 * D, BLKB = 16 * ROWB, TB = TOK * ROWB, SLOT = 2 * TB;
  static constexpr int PIECES = D / 8, NV = 2 * TOK * PIECES, NIT = (NV + THREADS - 1) / THREADS;
  static constexpr int KC = D / 32, DB = D / 16;
  static constexpr int RING = NR * SLOT, SCAL = NR * 2 * TOK * 4;
  // waves per SIMD: two workgroups per CU where two rings fit
  static constexpr int OCC = (RING + SCAL <= 80 * 1024 ? 2 : 1) * SB / 4;
  // Forward rows leave in 64-byte runs (swat_store_row) where registers allow: at d = 32 five columns and 32-token tiles are held to 128 (with
  // five rows, to arithmetic) and take 1 and 3.5 % less without.  With them: d = 64, 3 x 3, 64 slabs of 40 x 40 tiles 180 -> 174 us, five
  // columns 214 -> 209, d = 32, five rows 138 -> 131.
  static constexpr bool RUNS = !(D == 32 && (WC == 2 || NTB == 2));
  static_assert((TOK * PIECES) % 64 == 0, "a wave stages one tensor per vector");
  static constexpr bool BWD = RING + SCAL <= 160 * 1024;   // else forward only
  static_assert(RING <= 160 * 1024, "the ring exceeds the LDS");
};

template <int D> DLT_DEV int swat_swz(int t) { return D == 32 ? ((t >> 2) & 1) << 1 : D / 64 * (t & 7); }

typedef DLT_LDS char* swat_lds;
DLT_DEV u32x4 swat_read16(swat_lds p) { return *reinterpret_cast<DLT_LDS u32x4*>(p); }
DLT_DEV void swat_write16(swat_lds p, u32x4 v) { *reinterpret_cast<DLT_LDS u32x4*>(p) = v; }
DLT_DEV u32x2 swat_read_tr(swat_lds p) {
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<DLT_LDS s16x4*>(p)));
}

// byte offset of slot x of grid row 0 inside a (batch, head) slab, and the bytes between grid rows
DLT_DEV uint32_t swat_slot_off(const DltTokMap& tm, const int64_t (&st)[5], int x) {
  if (!tm.img) return (uint32_t)(x * (int)st[2] * 2);
  uint32_t i, px;
  dlt_slot_pixel(tm, (uint32_t)x, i, px);
  return i * (uint32_t)((int)st[4] * 2) + px * (uint32_t)((int)st[2] * 2);
}
DLT_DEV uint32_t swat_row_bytes(const DltTokMap& tm, const int64_t (&st)[5], int XL) {
  return tm.img ? tm.bh * (uint32_t)((int)st[4] * 2) : (uint32_t)(XL * (int)st[2] * 2);
}
template <typename T> DLT_DEV const char* swat_slab(const void* p, const int64_t (&st)[5], int b, int h) {
  return reinterpret_cast<const char*>(reinterpret_cast<const T*>(p) + b * st[0] + h * st[1]);
}

// Who a workgroup is: heads innermost (image rows hold all heads of a pixel side by side: the workgroups that share its
// 128-byte lines run at the same time on one XCD), then strips, bands and batches.
struct SwatWho { int b, h, r0, r1, xs; };
DLT_DEV SwatWho swat_who(const SwatArgs& a, int width) {
  int lin = xcd_remap(blockIdx.x, gridDim.x);
  SwatWho w;
  if (a.tm.img) {
    w.h = lin % a.H; lin /= a.H;
    const int s = lin % a.nstrips; lin /= a.nstrips;
    const int bd = lin % a.nbands;
    w.b = lin / a.nbands;
    w.xs = s * width; w.r0 = bd * a.band;
  } else {
    const int s = lin % a.nstrips; lin /= a.nstrips;
    const int bd = lin % a.nbands; lin /= a.nbands;
    w.h = lin % a.H;
    w.b = lin / a.H;
    w.xs = s * width; w.r0 = bd * a.band;
  }
  w.r1 = dlt_imin(w.r0 + a.band, a.g.TR);
  return w;
}

// The ring of one workgroup: staging of grid rows of two tensors, slot addresses, operand reads.
template <typename TIO, typename C>
struct SwatRing {
  swat_lds lds;
  const char *base0, *base1;
  uint32_t rs0, rs1;               // bytes between grid rows
  uint32_t goff[C::NIT];           // this thread's pieces: offset inside a grid row, LDS offset inside a slot
  int loff[C::NIT];
  bool second[C::NIT];             // wave-uniform
  unsigned outside;                // wave-uniform, bit `it`: the slots of that vector lie outside the grid row
  bool row_in;                     // the row in flight lies inside the grid
  u32x4 r[C::NIT];
  int tid, TR;

  DLT_DEV void init(swat_lds lds_, const char* b0, const int64_t (&s0)[5], const char* b1, const int64_t (&s1)[5], const SwatArgs& a, int xs, int tid_,
                    int wave) {
    lds = lds_; base0 = b0; base1 = b1; tid = tid_; TR = a.g.TR;
    const int XL = a.g.XLq;
    rs0 = swat_row_bytes(a.tm, s0, XL);
    rs1 = swat_row_bytes(a.tm, s1, XL);
    const int xh = xs - (C::HB - C::SB) * 8;   // first staged slot: half of the extra blocks lie to the left
    outside = 0;
#pragma unroll
    for (int it = 0; it < C::NIT; it++) {
      const int id = tid + C::THREADS * it;
      second[it] = 64 * wave + C::THREADS * it >= C::NV / 2;
      const int v = second[it] ? id - C::NV / 2 : id;
      const int tok = v / C::PIECES, piece = v % C::PIECES;
      // slots outside the grid row are clamped onto it: they belong to tiles that nobody sees (CLEAR)
      const int x = dlt_imax(0, dlt_imin(xh + tok, XL - 1));
      const int x0 = xh + (64 * wave + C::THREADS * it - (second[it] ? C::NV / 2 : 0)) / C::PIECES;   // a vector's slots lie in one block of 16
      outside |= (unsigned)(x0 < 0 || x0 >= XL) << it;
      goff[it] = (second[it] ? swat_slot_off(a.tm, s1, x) : swat_slot_off(a.tm, s0, x)) + 16 * piece;
      loff[it] = (second[it] ? C::TB : 0) + tok * C::ROWB + 16 * (piece ^ swat_swz<C::ROWB / 2>(tok));
    }
  }
  // rows outside the grid likewise
  DLT_DEV void issue(int row) {
    row_in = row >= 0 && row < TR;
    const uint32_t rc = (uint32_t)dlt_imax(0, dlt_imin(row, TR - 1));
    const uint32_t o0 = rc * rs0, o1 = rc * rs1;
#pragma unroll
    for (int it = 0; it < C::NIT; it++)
      if (C::NV % C::THREADS == 0 || it + 1 < C::NIT || tid + C::THREADS * it < C::NV)
        r[it] = *reinterpret_cast<const u32x4*>((second[it] ? base1 : base0) + (goff[it] + (second[it] ? o1 : o0)));
  }
  DLT_DEV void commit(int slot) {
    const unsigned zero = row_in ? outside : ~0u;
#pragma unroll
    for (int it = 0; it < C::NIT; it++)
      if (C::NV % C::THREADS == 0 || it + 1 < C::NIT || tid + C::THREADS * it < C::NV)
        swat_write16(lds + slot * C::SLOT + loff[it], C::CLEAR ? r[it] & ((zero >> it & 1u) - 1u) : r[it]);
  }
  // window rows of the first step: all requested before the first is written
  DLT_DEV void fill(int first) {
    u32x4 pre[C::NR][C::NIT];
#pragma unroll
    for (int i = 0; i < C::NR; i++) {
      issue(first + i);
#pragma unroll
      for (int it = 0; it < C::NIT; it++) pre[i][it] = r[it];
    }
#pragma unroll
    for (int i = 0; i < C::NR; i++) {
#pragma unroll
      for (int it = 0; it < C::NIT; it++) r[it] = pre[i][it];
      row_in = first + i >= 0 && first + i < TR;
      commit(i);
    }
  }
};

// lane parts of the operand addresses of a 16-token block (see swat_swz)
template <typename C>
struct SwatLane {
  int row[C::KC], tr[C::DB];
  DLT_DEV void init(int n, int g) {
    constexpr int D = C::ROWB / 2;
#pragma unroll
    for (int c = 0; c < C::KC; c++) row[c] = n * C::ROWB + 16 * ((4 * c + g) ^ swat_swz<D>(n));
    const int t = 4 * g + (n >> 2);
#pragma unroll
    for (int d = 0; d < C::DB; d++) tr[d] = t * C::ROWB + 16 * ((2 * d + ((n >> 1) & 1)) ^ swat_swz<D>(t)) + 8 * (n & 1);
  }
};

// Own rows leave straight from the accumulators: a lane of the C layout holds 4 dims of its token in each 16-dim block, and the
// lane swap of two blocks gives every lane 8 consecutive dims (16 bytes) of token n.  The 16 lanes that the memory pipe takes at a
// time then write 16 bytes each into 16 rows, and streaming stores can leave in parts of a sector: 1.25 to 1.3 times the bytes
// (D = 64 forward, 210 MB of o: 268 MB written; 498 MB of gradients for 403 at D = 32).  With RUNS a permutation brings the four
// pieces of a 64-byte run to four consecutive lanes (lane l: token l / 4, piece l % 4).  That is 4 LDS permutes per 32 dims: it pays
// where HBM is the bound (Swat::RUNS, swat_bwd_kernel) and not in the two backward launches of the larger windows and tiles, bound by
// arithmetic: their passes take 1 to 3.5 % less without it (d = 64, 16-token tiles, five columns, 64 slabs of 40 x 40 tiles: 651 -> 629 us,
// two registers spilled with it; d = 32, five rows, 128 slabs of 8 x 8: 35.1 -> 33.9).
// p: row of token swat_store_tok plus swat_store_byte.  Blocks of 16 tokens lie inside the grid or outside as a whole.
DLT_DEV int swat_store_tok(int lane, bool runs) { return runs ? lane >> 2 : lane & 15; }
DLT_DEV int swat_store_byte(int lane, bool runs) { return runs ? 16 * (lane & 3) : 32 * ((lane >> 4) & 1) + 16 * (lane >> 5); }
template <typename CT, int DB, bool RUNS>
DLT_DEV void swat_store_row(char* p, const f32x4 (&acc)[DB], float mul, int lane) {
  typedef unsigned pair_t __attribute__((ext_vector_type(2)));
  const int from = 4 * ((lane >> 2) + 16 * (((lane >> 1) & 1) | ((lane & 1) << 1)));
#pragma unroll
  for (int d = 0; d < DB; d += 2) {
    const pair_t lo = __builtin_amdgcn_permlane16_swap(pack2<CT>(acc[d][0] * mul, acc[d][1] * mul), pack2<CT>(acc[d + 1][0] * mul, acc[d + 1][1] * mul),
                                                       false, false);
    const pair_t hi = __builtin_amdgcn_permlane16_swap(pack2<CT>(acc[d][2] * mul, acc[d][3] * mul), pack2<CT>(acc[d + 1][2] * mul, acc[d + 1][3] * mul),
                                                       false, false);
    unsigned v[4] = {lo.x, hi.x, lo.y, hi.y};
    if constexpr (RUNS)
#pragma unroll
      for (int i = 0; i < 4; i++) v[i] = (unsigned)__builtin_amdgcn_ds_bpermute(from, (int)v[i]);
    store_stream16(p + 32 * d, u32x4{v[0], v[1], v[2], v[3]});
  }
}

// Which tiles of a window exist (wave-uniform).
template <typename C, int NTB>
struct SwatSeen {
  int rlo, rhi, clo, chi;   // window rows / block columns inside the grid
  DLT_DEV void init(const SwatArgs& a, int r, int tile, int WC, int WR) {
    rlo = dlt_imax(0, WR - r); rhi = dlt_imin(C::NR - 1, a.g.TR - 1 - r + WR);
    clo = NTB * dlt_imax(0, WC - tile); chi = NTB * (dlt_imin(2 * WC, a.g.TC - 1 - tile + WC) + 1) - 1;
  }
  DLT_DEV bool all() const { return rlo == 0 && rhi == C::NR - 1 && clo == 0 && chi == C::NWB - 1; }
  DLT_DEV bool sees(int i, int j) const { return i >= rlo && i <= rhi && j >= clo && j <= chi; }
};

template <typename TIO, int D, int NTB, int WC, int WR>
__global__ __launch_bounds__((Swat<D, NTB, WC, WR>::THREADS), (Swat<D, NTB, WC, WR>::OCC)) void swat_fwd_kernel(const SwatArgs a) {
  typedef Swat<D, NTB, WC, WR> C;
  typedef typename ComputeOf<TIO>::type CT;
  extern __shared__ __align__(16) char smem[];
  swat_lds lds = (swat_lds)smem;
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const SwatWho w = swat_who(a, 16 * C::SB);
  const int XL = a.g.XLq;

  SwatRing<TIO, C> ring;
  ring.init(lds, swat_slab<TIO>(a.k, a.ks, w.b, w.h), a.ks, swat_slab<TIO>(a.v, a.vs, w.b, w.h), a.vs, a, w.xs, tid, wave);

  const int x = w.xs + 16 * wave + n;
  const bool own = w.xs + 16 * wave < XL;                     // wave-uniform: the wave has a block of the grid
  const int tile = (w.xs + 16 * wave) / (16 * NTB);
  const int blk = NTB == 1 ? wave : wave / NTB * NTB;         // first staged block of the wave's window
  const int xc = dlt_imin(x, XL - 1), xw = dlt_imin(w.xs + 16 * wave + swat_store_tok(lane, C::RUNS), XL - 1);   // token of the lane's loads, of its stores
  const char* qb = swat_slab<TIO>(a.q, a.qs, w.b, w.h) + swat_slot_off(a.tm, a.qs, xc) + 16 * g;
  char* ob = const_cast<char*>(swat_slab<TIO>(a.out_o, a.os, w.b, w.h)) + swat_slot_off(a.tm, a.os, xw) + swat_store_byte(lane, C::RUNS);
  float* lseb = a.lse + w.b * a.ls[0] + w.h * a.ls[1] + (int64_t)x * a.ls[2];
  const uint32_t qrs = swat_row_bytes(a.tm, a.qs, XL), ors = swat_row_bytes(a.tm, a.os, XL);
  SwatLane<C> L;
  L.init(n, g);
  const float scale = a.scale_log2;
  const unsigned one2 = pack2<CT>(1.f, 1.f);
  const u32x4 ones = {one2, one2, one2, one2};

  // 18 blocks of scores at 128 registers a lane: requested in front of them the next q was spilled, i.e. waited for with
  // every piece in flight; it is requested once half of the scores are gone
  constexpr bool LATE_Q = C::OCC == 4 && C::NB > 15;
  u32x4 qn[C::KC];
  auto load_q = [&](int r) {
#pragma unroll
    for (int c = 0; c < C::KC; c++) qn[c] = *reinterpret_cast<const u32x4*>(qb + (uint32_t)r * qrs + 64 * c);
  };
  load_q(w.r0);
  ring.fill(w.r0 - WR);
  __syncthreads();

  int slot0 = 0;   // slot of the window's first row
  for (int r = w.r0; r < w.r1; r++) {
    u32x4 q[C::KC];
#pragma unroll
    for (int c = 0; c < C::KC; c++) q[c] = qn[c];
    pin_loaded(q);
    const bool more = r + 1 < w.r1;
    if (more) {
      ring.issue(r + 1 + WR);
      if constexpr (!LATE_Q) load_q(r + 1);
    }
    SwatSeen<C, NTB> seen;
    seen.init(a, r, tile, WC, WR);
    auto step = [&](auto edge_tag) __attribute__((always_inline)) {
      constexpr bool EDGE = decltype(edge_tag)::value;
      swat_lds rowp[C::NR];
#pragma unroll
      for (int i = 0; i < C::NR; i++) {
        const int s = slot0 + i;
        rowp[i] = lds + (s >= C::NR ? s - C::NR : s) * C::SLOT + blk * C::BLKB;
      }
      f32x4 s[C::NB + 1];
#pragma unroll
      for (int i = 0; i < C::NR; i++)
#pragma unroll
        for (int j = 0; j < C::NWB; j++) {
          f32x4 t = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int c = 0; c < C::KC; c++) t = Mma<CT>::mfma(swat_read16(rowp[i] + L.row[c] + j * C::BLKB), q[c], t);
          if (EDGE && !seen.sees(i, j)) t = f32x4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
          s[i * C::NWB + j] = t;
        }
      float mx[4] = {s[0][0], s[0][1], s[0][2], s[0][3]};
#pragma unroll
      for (int b = 1; b + 1 < C::NB; b += 2)
#pragma unroll
        for (int i = 0; i < 4; i++) mx[i] = fmaxf(fmaxf(mx[i], s[b][i]), s[b + 1][i]);
      if (C::NB % 2 == 0)
#pragma unroll
        for (int i = 0; i < 4; i++) mx[i] = fmaxf(mx[i], s[C::NB - 1][i]);
      const float m = wave_max4(fmaxf(fmaxf(mx[0], mx[1]), fmaxf(mx[2], mx[3])));   // finite: a tile sees itself
      const float neg_m2 = -m * scale;
      f32x4 acc[C::DB], acc_l = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int d = 0; d < C::DB; d++) acc[d] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < C::NP; t++) {
        constexpr int LAST = C::NB - 1;
        const bool pair = 2 * t < LAST;
        const int b0 = 2 * t, b1 = pair ? 2 * t + 1 : 2 * t;
        float p[8];
#pragma unroll
        for (int i = 0; i < 4; i++) {
          p[i] = fast_exp2(fmaf(s[b0][i], scale, neg_m2));
          p[4 + i] = pair ? fast_exp2(fmaf(s[b1][i], scale, neg_m2)) : 0.f;
        }
        const u32x4 pb = pack8<CT>(p);
        if constexpr (LATE_Q)
          if (t == C::NP / 2 && more) load_q(r + 1);
        swat_lds v0 = rowp[b0 / C::NWB] + C::TB + (b0 % C::NWB) * C::BLKB, v1 = rowp[b1 / C::NWB] + C::TB + (b1 % C::NWB) * C::BLKB;
#pragma unroll
        for (int d = 0; d < C::DB; d++) {
          const u32x2 lo = swat_read_tr(v0 + L.tr[d]), hi = pair || !C::ALONE ? swat_read_tr(v1 + L.tr[d]) : u32x2{0u, 0u};
          acc[d] = Mma<CT>::mfma(u32x4{lo.x, lo.y, hi.x, hi.y}, pb, acc[d]);
        }
        acc_l = Mma<CT>::mfma(ones, pb, acc_l);
      }
      const float l = acc_l[0];
      swat_store_row<CT, C::DB, C::RUNS>(ob + (uint32_t)r * ors, acc, fast_rcp(l), lane);
      if (g == 0) store_stream4(lseb + (int64_t)r * XL * a.ls[2], m * scale + fast_log2(l));
    };
    if (own) {
      if (seen.all()) step(std::false_type{});
      else step(std::true_type{});
    }
    if (more) {
      __syncthreads();
      ring.commit(slot0);   // the row that left the window
      __syncthreads();
      slot0 = slot0 + 1 == C::NR ? 0 : slot0 + 1;
    }
  }
}

// dQ: own = queries, K and V in the ring; delta = rowsum(o dO) of the own queries is formed and stored on the way.
template <typename TIO, int D, int NTB, int WC, int WR>
__global__ __launch_bounds__((Swat<D, NTB, WC, WR>::THREADS), (Swat<D, NTB, WC, WR>::OCC)) void swat_bwd_q_kernel(const SwatArgs a) {
  typedef Swat<D, NTB, WC, WR> C;
  typedef typename ComputeOf<TIO>::type CT;
  extern __shared__ __align__(16) char smem[];
  swat_lds lds = (swat_lds)smem;
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const SwatWho w = swat_who(a, 16 * C::SB);
  const int XL = a.g.XLq;

  SwatRing<TIO, C> ring;
  ring.init(lds, swat_slab<TIO>(a.k, a.ks, w.b, w.h), a.ks, swat_slab<TIO>(a.v, a.vs, w.b, w.h), a.vs, a, w.xs, tid, wave);
  const int x = w.xs + 16 * wave + n;
  const bool own = w.xs + 16 * wave < XL;
  const int tile = (w.xs + 16 * wave) / (16 * NTB);
  const int blk = NTB == 1 ? wave : wave / NTB * NTB;
  const int xc = dlt_imin(x, XL - 1);
  const char* qb = swat_slab<TIO>(a.q, a.qs, w.b, w.h) + swat_slot_off(a.tm, a.qs, xc) + 16 * g;
  const char* dob = swat_slab<TIO>(a.d_o, a.dos, w.b, w.h) + swat_slot_off(a.tm, a.dos, xc) + 16 * g;
  const char* ob = swat_slab<TIO>(a.o, a.os, w.b, w.h) + swat_slot_off(a.tm, a.os, xc) + 16 * g;
  char* dqb = const_cast<char*>(swat_slab<TIO>(a.dq, a.dqs, w.b, w.h)) + swat_slot_off(a.tm, a.dqs, xc) + swat_store_byte(lane, false);
  const float* lseb = a.lse + w.b * a.ls[0] + w.h * a.ls[1] + (int64_t)xc * a.ls[2];
  float* delb = a.delta + w.b * a.ls[0] + w.h * a.ls[1] + (int64_t)xc * a.ls[2];
  const uint32_t qrs = swat_row_bytes(a.tm, a.qs, XL), dors = swat_row_bytes(a.tm, a.dos, XL), ors = swat_row_bytes(a.tm, a.os, XL),
                 dqrs = swat_row_bytes(a.tm, a.dqs, XL);
  SwatLane<C> L;
  L.init(n, g);
  const float scale = a.scale_log2;

  u32x4 qn[C::KC], don[C::KC], on[C::KC];
  float lsen;
  auto load_own = [&](int r) {
#pragma unroll
    for (int c = 0; c < C::KC; c++) {
      qn[c] = *reinterpret_cast<const u32x4*>(qb + (uint32_t)r * qrs + 64 * c);
      don[c] = *reinterpret_cast<const u32x4*>(dob + (uint32_t)r * dors + 64 * c);
      on[c] = *reinterpret_cast<const u32x4*>(ob + (uint32_t)r * ors + 64 * c);
    }
    lsen = lseb[(int64_t)r * XL * a.ls[2]];
  };
  load_own(w.r0);
  ring.fill(w.r0 - WR);
  __syncthreads();

  int slot0 = 0;
  for (int r = w.r0; r < w.r1; r++) {
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
    if (g == 0 && x < XL) store_stream4(delb + (int64_t)r * XL * a.ls[2], del);
    const bool more = r + 1 < w.r1;
    if (more) {
      ring.issue(r + 1 + WR);
      load_own(r + 1);
    }
    SwatSeen<C, NTB> seen;
    seen.init(a, r, tile, WC, WR);
    auto step = [&](auto edge_tag) __attribute__((always_inline)) {
      constexpr bool EDGE = decltype(edge_tag)::value;
      swat_lds rowp[C::NR];
#pragma unroll
      for (int i = 0; i < C::NR; i++) {
        const int s = slot0 + i;
        rowp[i] = lds + (s >= C::NR ? s - C::NR : s) * C::SLOT + blk * C::BLKB;
      }
      f32x4 acc[C::DB];
#pragma unroll
      for (int d = 0; d < C::DB; d++) acc[d] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < C::NP; t++) {
        float ds[8];
#pragma unroll
        for (int u = 0; u < 2; u++) {
          const int b = 2 * t + u;
          if (b >= C::NB) {
#pragma unroll
            for (int i = 0; i < 4; i++) ds[4 * u + i] = 0.f;
            continue;
          }
          swat_lds kp = rowp[b / C::NWB] + (b % C::NWB) * C::BLKB;
          // the dP products start from -delta: the matrix pipe delivers dP - delta
          f32x4 s = {0.f, 0.f, 0.f, 0.f}, dp = {-del, -del, -del, -del};
#pragma unroll
          for (int c = 0; c < C::KC; c++) {
            s = Mma<CT>::mfma(swat_read16(kp + L.row[c]), q[c], s);
            dp = Mma<CT>::mfma(swat_read16(kp + C::TB + L.row[c]), d_o[c], dp);
          }
          if (EDGE && !seen.sees(b / C::NWB, b % C::NWB)) s = f32x4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
#pragma unroll
          for (int i = 0; i < 4; i++) ds[4 * u + i] = fast_exp2(fmaf(s[i], scale, nlse)) * dp[i];
        }
        const u32x4 dsb = pack8<CT>(ds);
        const bool pair = 2 * t + 1 < C::NB;
        const int b0 = 2 * t, b1 = pair ? 2 * t + 1 : 2 * t;
        swat_lds k0 = rowp[b0 / C::NWB] + (b0 % C::NWB) * C::BLKB, k1 = rowp[b1 / C::NWB] + (b1 % C::NWB) * C::BLKB;
#pragma unroll
        for (int d = 0; d < C::DB; d++) {
          const u32x2 lo = swat_read_tr(k0 + L.tr[d]), hi = pair || !C::ALONE ? swat_read_tr(k1 + L.tr[d]) : u32x2{0u, 0u};
          acc[d] = Mma<CT>::mfma(u32x4{lo.x, lo.y, hi.x, hi.y}, dsb, acc[d]);
        }
      }
      if (x < XL) swat_store_row<CT, C::DB, false>(dqb + (uint32_t)r * dqrs, acc, a.sm_scale, lane);
    };
    if (own) {
      if (seen.all()) step(std::false_type{});
      else step(std::true_type{});
    }
    if (more) {
      __syncthreads();
      ring.commit(slot0);
      __syncthreads();
      slot0 = slot0 + 1 == C::NR ? 0 : slot0 + 1;
    }
  }
}

// dK / dV: own = keys, Q and dO in the ring with -lse2 and delta of their tokens behind it (the window is symmetric).
template <typename TIO, int D, int NTB, int WC, int WR>
__global__ __launch_bounds__((Swat<D, NTB, WC, WR>::THREADS), (Swat<D, NTB, WC, WR>::OCC)) void swat_bwd_kv_kernel(const SwatArgs a) {
  typedef Swat<D, NTB, WC, WR> C;
  typedef typename ComputeOf<TIO>::type CT;
  extern __shared__ __align__(16) char smem[];
  swat_lds lds = (swat_lds)smem;
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const SwatWho w = swat_who(a, 16 * C::SB);
  const int XL = a.g.XLq;

  SwatRing<TIO, C> ring;
  ring.init(lds, swat_slab<TIO>(a.q, a.qs, w.b, w.h), a.qs, swat_slab<TIO>(a.d_o, a.dos, w.b, w.h), a.dos, a, w.xs, tid, wave);
  const float* lseb = a.lse + w.b * a.ls[0] + w.h * a.ls[1];
  const float* delb = a.delta + w.b * a.ls[0] + w.h * a.ls[1];
  DLT_LDS float* scal = reinterpret_cast<DLT_LDS float*>(lds + C::RING);   // [slot][-lse2 | delta][token]
  const int xsc = dlt_imax(0, dlt_imin(w.xs - (C::HB - C::SB) * 8 + tid, XL - 1));
  float r_lse = 0.f, r_del = 0.f;
  auto issue_scal = [&](int row) {
    const int rc = dlt_imax(0, dlt_imin(row, a.g.TR - 1));
    if (tid < C::TOK) {
      const int64_t off = ((int64_t)rc * XL + xsc) * a.ls[2];
      r_lse = lseb[off];
      r_del = delb[off];
    }
  };
  auto commit_scal = [&](int slot) {
    if (tid < C::TOK) {
      scal[slot * 2 * C::TOK + tid] = -r_lse;
      scal[slot * 2 * C::TOK + C::TOK + tid] = r_del;
    }
  };
  const int x = w.xs + 16 * wave + n;
  const bool own = w.xs + 16 * wave < XL;
  const int tile = (w.xs + 16 * wave) / (16 * NTB);
  const int blk = NTB == 1 ? wave : wave / NTB * NTB;
  const int xc = dlt_imin(x, XL - 1);
  const char* kb = swat_slab<TIO>(a.k, a.ks, w.b, w.h) + swat_slot_off(a.tm, a.ks, xc) + 16 * g;
  const char* vb = swat_slab<TIO>(a.v, a.vs, w.b, w.h) + swat_slot_off(a.tm, a.vs, xc) + 16 * g;
  char* dkb = const_cast<char*>(swat_slab<TIO>(a.dk, a.dks, w.b, w.h)) + swat_slot_off(a.tm, a.dks, xc) + swat_store_byte(lane, false);
  char* dvb = const_cast<char*>(swat_slab<TIO>(a.dv, a.dvs, w.b, w.h)) + swat_slot_off(a.tm, a.dvs, xc) + swat_store_byte(lane, false);
  const uint32_t krs = swat_row_bytes(a.tm, a.ks, XL), vrs = swat_row_bytes(a.tm, a.vs, XL), dkrs = swat_row_bytes(a.tm, a.dks, XL),
                 dvrs = swat_row_bytes(a.tm, a.dvs, XL);
  SwatLane<C> L;
  L.init(n, g);
  const float scale = a.scale_log2;

  u32x4 kn[C::KC], vn[C::KC];
  auto load_own = [&](int r) {
#pragma unroll
    for (int c = 0; c < C::KC; c++) {
      kn[c] = *reinterpret_cast<const u32x4*>(kb + (uint32_t)r * krs + 64 * c);
      vn[c] = *reinterpret_cast<const u32x4*>(vb + (uint32_t)r * vrs + 64 * c);
    }
  };
  load_own(w.r0);
  ring.fill(w.r0 - WR);
#pragma unroll
  for (int i = 0; i < C::NR; i++) {
    issue_scal(w.r0 - WR + i);
    commit_scal(i);
  }
  __syncthreads();

  int slot0 = 0;
  for (int r = w.r0; r < w.r1; r++) {
    // The own values are negated and the dP products start from the staged delta: the matrix pipe delivers -(dP - delta)
    u32x4 k[C::KC], v[C::KC];
#pragma unroll
    for (int c = 0; c < C::KC; c++) {
      k[c] = kn[c];
      v[c] = u32x4{vn[c].x ^ 0x80008000u, vn[c].y ^ 0x80008000u, vn[c].z ^ 0x80008000u, vn[c].w ^ 0x80008000u};
    }
    pin_loaded(k);
    pin_loaded(v);
    const bool more = r + 1 < w.r1;
    if (more) {
      ring.issue(r + 1 + WR);
      issue_scal(r + 1 + WR);
      load_own(r + 1);
    }
    SwatSeen<C, NTB> seen;
    seen.init(a, r, tile, WC, WR);
    auto step = [&](auto edge_tag) __attribute__((always_inline)) {
      constexpr bool EDGE = decltype(edge_tag)::value;
      swat_lds rowp[C::NR];
      DLT_LDS float* scp[C::NR];
#pragma unroll
      for (int i = 0; i < C::NR; i++) {
        const int s0 = slot0 + i, s = s0 >= C::NR ? s0 - C::NR : s0;
        rowp[i] = lds + s * C::SLOT + blk * C::BLKB;
        scp[i] = scal + s * 2 * C::TOK + blk * 16 + 4 * g;
      }
      f32x4 acc_k[C::DB], acc_v[C::DB];
#pragma unroll
      for (int d = 0; d < C::DB; d++) acc_k[d] = acc_v[d] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < C::NP; t++) {
        float p[8], ds[8];
#pragma unroll
        for (int u = 0; u < 2; u++) {
          const int b = 2 * t + u;
          if (b >= C::NB) {
#pragma unroll
            for (int i = 0; i < 4; i++) p[4 * u + i] = ds[4 * u + i] = 0.f;
            continue;
          }
          swat_lds qp = rowp[b / C::NWB] + (b % C::NWB) * C::BLKB;
          DLT_LDS float* sp = scp[b / C::NWB] + (b % C::NWB) * 16;
          const f32x4 nl = *reinterpret_cast<DLT_LDS f32x4*>(sp);
          f32x4 s = {0.f, 0.f, 0.f, 0.f}, dp = *reinterpret_cast<DLT_LDS f32x4*>(sp + C::TOK);
#pragma unroll
          for (int c = 0; c < C::KC; c++) {
            s = Mma<CT>::mfma(swat_read16(qp + L.row[c]), k[c], s);
            dp = Mma<CT>::mfma(swat_read16(qp + C::TB + L.row[c]), v[c], dp);
          }
          if (EDGE && !seen.sees(b / C::NWB, b % C::NWB)) s = f32x4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
#pragma unroll
          for (int i = 0; i < 4; i++) {
            const float pv = fast_exp2(fmaf(s[i], scale, nl[i]));
            p[4 * u + i] = pv;
            ds[4 * u + i] = -pv * dp[i];
          }
        }
        const u32x4 pb = pack8<CT>(p), dsb = pack8<CT>(ds);
        const bool pair = 2 * t + 1 < C::NB;
        const int b0 = 2 * t, b1 = pair ? 2 * t + 1 : 2 * t;
        swat_lds q0 = rowp[b0 / C::NWB] + (b0 % C::NWB) * C::BLKB, q1 = rowp[b1 / C::NWB] + (b1 % C::NWB) * C::BLKB;
#pragma unroll
        for (int d = 0; d < C::DB; d++) {
          const u32x2 lo = swat_read_tr(q0 + C::TB + L.tr[d]), hi = pair || !C::ALONE ? swat_read_tr(q1 + C::TB + L.tr[d]) : u32x2{0u, 0u};
          acc_v[d] = Mma<CT>::mfma(u32x4{lo.x, lo.y, hi.x, hi.y}, pb, acc_v[d]);
        }
#pragma unroll
        for (int d = 0; d < C::DB; d++) {
          const u32x2 lo = swat_read_tr(q0 + L.tr[d]), hi = pair || !C::ALONE ? swat_read_tr(q1 + L.tr[d]) : u32x2{0u, 0u};
          acc_k[d] = Mma<CT>::mfma(u32x4{lo.x, lo.y, hi.x, hi.y}, dsb, acc_k[d]);
        }
      }
      if (x < XL) {
        swat_store_row<CT, C::DB, false>(dvb + (uint32_t)r * dvrs, acc_v, 1.f, lane);
        swat_store_row<CT, C::DB, false>(dkb + (uint32_t)r * dkrs, acc_k, a.sm_scale, lane);
      }
    };
    if (own) {
      if (seen.all()) step(std::false_type{});
      else step(std::true_type{});
    }
    if (more) {
      __syncthreads();
      ring.commit(slot0);
      commit_scal(slot0);
      __syncthreads();
      slot0 = slot0 + 1 == C::NR ? 0 : slot0 + 1;
    }
  }
}

// ---- dQ, dK and dV in one launch (16-token tiles, 3 x 3 window) ---------------------------------------------------
// What bounded the two launches above: HBM.  Both read q, k, v and dO, dQ also o: with the gradients, delta and lse2 that is
// 12 passes over a tensor of the operator where 8 are needed (B = 4, H = 8, 256 x 256 pixels in 4 x 4 tiles, d = 32, image
// layout: 210 + 243 us at 4.3 TB/s).  With all four tensors of the window's rows in the ring (K, V, Q, dO: 120 KB at D = 32, 147 at
// D = 64, one workgroup per CU) a strip's dQ, dK and dV leave in one march: the first half of the waves own query blocks, the
// second half key blocks; both take their own fragments, lse2 and delta from the ring, and delta is formed by the threads
// that stage dO (they fetch the pieces of o beside it), so nothing travels between launches.  Strips of 8 blocks and 16 waves
// at D = 32; at D = 64 the ring holds strips of 4 (8 waves).  Measured: the backward pass above 453 -> 290 us (1.18 GB, 4.1
// TB/s); d = 64, 16 slabs of 40 x 40 tiles x 4 batches 540 -> 433.  Narrow grids at D = 32 (dlt_tile_bwd_one_launch), larger windows and
// 32-token tiles stay on two launches: their
// rows would fit at D = 32, but there the arithmetic is the bound and one workgroup per CU ties (5 columns: 164 against 166 us)
// or loses (32-token tiles: 91 against 100).
template <int D, int NTB, int WC, int WR>
struct Swab : Swat<D, NTB, WC, WR> {
  typedef Swat<D, NTB, WC, WR> Base;
  static constexpr int SB = D == 32 ? 8 : 4;                        // 16-token blocks of a strip
  static constexpr int NWAVE = 2 * SB, THREADS = 64 * NWAVE;
  static constexpr int HB = SB + 2 * WC * NTB, TOK = 16 * HB;
  static constexpr int TB = TOK * Base::ROWB, SLOT = 4 * TB;        // K, V, Q, dO of a grid row
  static constexpr int WPT = TOK * Base::PIECES / 64;               // wave-wide vectors per tensor and row
  static constexpr int NIT = (4 * WPT + NWAVE - 1) / NWAVE;
  static constexpr int RING = Base::NR * SLOT, SCAL = Base::NR * 2 * TOK * 4, LDS = RING + SCAL;
  static constexpr bool USED = NTB == 1 && WC == 1 && WR == 1;
  static_assert(!USED || (TOK * Base::PIECES % 64 == 0 && TOK <= THREADS && LDS <= 160 * 1024), "staging map, LDS");
};

// sum over the lanes that hold the 16-byte pieces of one token (4 or 8 consecutive lanes)
template <int PIECES>
DLT_DEV float swat_sum_pieces(float v) {
  static_assert(PIECES == 4 || PIECES == 8, "a quad or half a row of lanes");
  auto dpp = [](float x, auto ctrl) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), decltype(ctrl)::value, 0xf, 0xf, true));
  };
  v += dpp(v, std::integral_constant<int, 0x4e>{});   // lane ^ 2
  v += dpp(v, std::integral_constant<int, 0xb1>{});   // lane ^ 1
  if constexpr (PIECES == 8) v += dpp(v, std::integral_constant<int, 0x141>{});   // the other quad of the eight
  return v;
}

template <typename TIO, int D, int NTB, int WC, int WR>
__global__ __launch_bounds__((Swab<D, NTB, WC, WR>::THREADS), (Swab<D, NTB, WC, WR>::NWAVE / 4)) void swat_bwd_kernel(const SwatArgs a) {
  typedef Swab<D, NTB, WC, WR> C;
  typedef typename ComputeOf<TIO>::type CT;
  extern __shared__ __align__(16) char smem[];
  swat_lds lds = (swat_lds)smem;
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const SwatWho w = swat_who(a, 16 * C::SB);
  const int XL = a.g.XLq, TR = a.g.TR;
  DLT_LDS float* scal = reinterpret_cast<DLT_LDS float*>(lds + C::RING);   // [slot][-lse2 | delta][token]

  // ---- staging: vector wave + NWAVE it of a grid row belongs to tensor (that) / WPT (K, V, Q, dO): wave-uniform
  const int xh = w.xs - 16 * WC * NTB;   // first staged slot
  const char* base[C::NIT];
  uint32_t rs[C::NIT], goff[C::NIT], ooff[C::NIT];
  int loff[C::NIT], tok_of[C::NIT];
  const char* ob = swat_slab<TIO>(a.o, a.os, w.b, w.h);
  const uint32_t ors = swat_row_bytes(a.tm, a.os, XL);
  auto may_be_do = [](int it) { return C::NWAVE * (it + 1) > 3 * C::WPT; };
#pragma unroll
  for (int it = 0; it < C::NIT; it++) {
    const int wv = wave + C::NWAVE * it, ten = dlt_imin(wv / C::WPT, 3);
    const int v = (wv - ten * C::WPT) * 64 + lane, tok = v / C::PIECES, piece = v % C::PIECES;
    // slots outside the grid row are clamped onto it: they belong to tiles that nobody sees
    const int x = dlt_imax(0, dlt_imin(xh + tok, XL - 1));
    base[it] = swat_slab<TIO>(a.ring_p[ten], a.ring_s[ten], w.b, w.h);
    rs[it] = swat_row_bytes(a.tm, a.ring_s[ten], XL);
    goff[it] = swat_slot_off(a.tm, a.ring_s[ten], x);
    goff[it] += 16 * piece;
    ooff[it] = may_be_do(it) ? swat_slot_off(a.tm, a.os, x) + 16 * piece : 0u;
    loff[it] = ten * C::TB + tok * C::ROWB + 16 * (piece ^ swat_swz<D>(tok));
    tok_of[it] = tok;
  }
  const int xsc = dlt_imax(0, dlt_imin(xh + tid, XL - 1));
  const float* lseb = a.lse + w.b * a.ls[0] + w.h * a.ls[1];
  struct Row { u32x4 r[C::NIT], o[C::NIT]; float lse; };
  auto on = [&](int it) { return wave + C::NWAVE * it < 4 * C::WPT; };                                // wave-uniform
  auto is_do = [&](int it) { return may_be_do(it) && wave + C::NWAVE * it >= 3 * C::WPT && on(it); };
  auto issue = [&](int row, Row& R) __attribute__((always_inline)) {
    const uint32_t rc = (uint32_t)dlt_imax(0, dlt_imin(row, TR - 1));   // rows outside the grid: clamped as well
#pragma unroll
    for (int it = 0; it < C::NIT; it++) {
      if (on(it)) R.r[it] = *reinterpret_cast<const u32x4*>(base[it] + (goff[it] + rc * rs[it]));
      if (may_be_do(it) && is_do(it)) R.o[it] = *reinterpret_cast<const u32x4*>(ob + (ooff[it] + rc * ors));
    }
    if (tid < C::TOK) R.lse = lseb[((int64_t)rc * XL + xsc) * a.ls[2]];
  };
  auto commit = [&](int slot, const Row& R) __attribute__((always_inline)) {
#pragma unroll
    for (int it = 0; it < C::NIT; it++) {
      if (on(it)) swat_write16(lds + slot * C::SLOT + loff[it], R.r[it]);
      if (may_be_do(it) && is_do(it)) {
        float fo[8], fd[8], part = 0.f;
        unpack8<CT>(R.o[it], fo);
        unpack8<CT>(R.r[it], fd);
#pragma unroll
        for (int j = 0; j < 8; j++) part += fo[j] * fd[j];
        const float del = swat_sum_pieces<C::PIECES>(part);
        if (lane % C::PIECES == 0) scal[slot * 2 * C::TOK + C::TOK + tok_of[it]] = del;
      }
    }
    if (tid < C::TOK) scal[slot * 2 * C::TOK + tid] = -R.lse;
  };

  const bool is_q = wave < C::SB;                            // this wave owns queries, else keys
  const int blk_w = is_q ? wave : wave - C::SB;              // own block of the strip
  const bool own = w.xs + 16 * blk_w < XL;
  const int tile = (w.xs + 16 * blk_w) / (16 * NTB);
  const int blk = NTB == 1 ? blk_w : blk_w / NTB * NTB;      // first staged block of the wave's window
  const int own_blk = blk_w + WC * NTB;                      // own block among the staged ones
  const int xw = dlt_imin(w.xs + 16 * blk_w + swat_store_tok(lane, true), XL - 1);   // token of the lane's stores
  char* out0 = is_q ? const_cast<char*>(swat_slab<TIO>(a.dq, a.dqs, w.b, w.h)) + swat_slot_off(a.tm, a.dqs, xw) + swat_store_byte(lane, true)
                    : const_cast<char*>(swat_slab<TIO>(a.dk, a.dks, w.b, w.h)) + swat_slot_off(a.tm, a.dks, xw) + swat_store_byte(lane, true);
  char* out1 = const_cast<char*>(swat_slab<TIO>(a.dv, a.dvs, w.b, w.h)) + swat_slot_off(a.tm, a.dvs, xw) + swat_store_byte(lane, true);
  const uint32_t out0rs = is_q ? swat_row_bytes(a.tm, a.dqs, XL) : swat_row_bytes(a.tm, a.dks, XL), out1rs = swat_row_bytes(a.tm, a.dvs, XL);
  SwatLane<C> L;
  L.init(n, g);
  const float scale = a.scale_log2;

  {
    Row pre[C::NR];
#pragma unroll
    for (int i = 0; i < C::NR; i++) issue(w.r0 - WR + i, pre[i]);
#pragma unroll
    for (int i = 0; i < C::NR; i++) commit(i, pre[i]);
  }
  __syncthreads();

  int slot0 = 0;   // slot of the window's first row
  for (int r = w.r0; r < w.r1; r++) {
    const bool more = r + 1 < w.r1;
    Row next;
    if (more) issue(r + 1 + WR, next);
    SwatSeen<C, NTB> seen;
    seen.init(a, r, tile, WC, WR);
    swat_lds rowp[C::NR];
    DLT_LDS float* scp[C::NR];
#pragma unroll
    for (int i = 0; i < C::NR; i++) {
      const int s0 = slot0 + i, s = s0 >= C::NR ? s0 - C::NR : s0;
      rowp[i] = lds + s * C::SLOT + blk * C::BLKB;
      scp[i] = scal + s * 2 * C::TOK + blk * 16;
    }
    const int to_own = (own_blk - blk) * C::BLKB;
    // queries: K and V stream past the own q, dO, lse2 and delta
    auto step_q = [&](auto edge_tag) __attribute__((always_inline)) {
      constexpr bool EDGE = decltype(edge_tag)::value;
      u32x4 q[C::KC], d_o[C::KC];
#pragma unroll
      for (int c = 0; c < C::KC; c++) {
        q[c] = swat_read16(rowp[WR] + 2 * C::TB + to_own + L.row[c]);
        d_o[c] = swat_read16(rowp[WR] + 3 * C::TB + to_own + L.row[c]);
      }
      DLT_LDS float* sp = scp[WR] + (own_blk - blk) * 16 + n;
      const float nlse = sp[0], del = sp[C::TOK];
      f32x4 acc[C::DB];
#pragma unroll
      for (int d = 0; d < C::DB; d++) acc[d] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < C::NP; t++) {
        float ds[8];
#pragma unroll
        for (int u = 0; u < 2; u++) {
          const int b = 2 * t + u;
          if (b >= C::NB) {
#pragma unroll
            for (int i = 0; i < 4; i++) ds[4 * u + i] = 0.f;
            continue;
          }
          swat_lds kp = rowp[b / C::NWB] + (b % C::NWB) * C::BLKB;
          // the dP products start from -delta: the matrix pipe delivers dP - delta
          f32x4 s = {0.f, 0.f, 0.f, 0.f}, dp = {-del, -del, -del, -del};
#pragma unroll
          for (int c = 0; c < C::KC; c++) {
            s = Mma<CT>::mfma(swat_read16(kp + L.row[c]), q[c], s);
            dp = Mma<CT>::mfma(swat_read16(kp + C::TB + L.row[c]), d_o[c], dp);
          }
          if (EDGE && !seen.sees(b / C::NWB, b % C::NWB)) s = f32x4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
#pragma unroll
          for (int i = 0; i < 4; i++) ds[4 * u + i] = fast_exp2(fmaf(s[i], scale, nlse)) * dp[i];
        }
        const u32x4 dsb = pack8<CT>(ds);
        const bool pair = 2 * t + 1 < C::NB;
        const int b0 = 2 * t, b1 = pair ? 2 * t + 1 : 2 * t;
        swat_lds k0 = rowp[b0 / C::NWB] + (b0 % C::NWB) * C::BLKB, k1 = rowp[b1 / C::NWB] + (b1 % C::NWB) * C::BLKB;
#pragma unroll
        for (int d = 0; d < C::DB; d++) {
          const u32x2 lo = swat_read_tr(k0 + L.tr[d]), hi = pair || !C::ALONE ? swat_read_tr(k1 + L.tr[d]) : u32x2{0u, 0u};
          acc[d] = Mma<CT>::mfma(u32x4{lo.x, lo.y, hi.x, hi.y}, dsb, acc[d]);
        }
      }
      swat_store_row<CT, C::DB, true>(out0 + (uint32_t)r * out0rs, acc, a.sm_scale, lane);
    };
    // keys: Q, dO, lse2 and delta stream past the own k and v (the window is symmetric)
    auto step_kv = [&](auto edge_tag) __attribute__((always_inline)) {
      constexpr bool EDGE = decltype(edge_tag)::value;
      // the own values are negated and the dP products start from delta: the matrix pipe delivers -(dP - delta)
      u32x4 k[C::KC], v[C::KC];
#pragma unroll
      for (int c = 0; c < C::KC; c++) {
        k[c] = swat_read16(rowp[WR] + to_own + L.row[c]);
        v[c] = swat_read16(rowp[WR] + C::TB + to_own + L.row[c]);
        v[c].x ^= 0x80008000u; v[c].y ^= 0x80008000u; v[c].z ^= 0x80008000u; v[c].w ^= 0x80008000u;
      }
      f32x4 acc_k[C::DB], acc_v[C::DB];
#pragma unroll
      for (int d = 0; d < C::DB; d++) acc_k[d] = acc_v[d] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < C::NP; t++) {
        float p[8], ds[8];
#pragma unroll
        for (int u = 0; u < 2; u++) {
          const int b = 2 * t + u;
          if (b >= C::NB) {
#pragma unroll
            for (int i = 0; i < 4; i++) p[4 * u + i] = ds[4 * u + i] = 0.f;
            continue;
          }
          swat_lds qp = rowp[b / C::NWB] + 2 * C::TB + (b % C::NWB) * C::BLKB;
          DLT_LDS float* sp = scp[b / C::NWB] + (b % C::NWB) * 16 + 4 * g;
          const f32x4 nl = *reinterpret_cast<DLT_LDS f32x4*>(sp);
          f32x4 s = {0.f, 0.f, 0.f, 0.f}, dp = *reinterpret_cast<DLT_LDS f32x4*>(sp + C::TOK);
#pragma unroll
          for (int c = 0; c < C::KC; c++) {
            s = Mma<CT>::mfma(swat_read16(qp + L.row[c]), k[c], s);
            dp = Mma<CT>::mfma(swat_read16(qp + C::TB + L.row[c]), v[c], dp);
          }
          if (EDGE && !seen.sees(b / C::NWB, b % C::NWB)) s = f32x4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
#pragma unroll
          for (int i = 0; i < 4; i++) {
            const float pv = fast_exp2(fmaf(s[i], scale, nl[i]));
            p[4 * u + i] = pv;
            ds[4 * u + i] = -pv * dp[i];
          }
        }
        const u32x4 pb = pack8<CT>(p), dsb = pack8<CT>(ds);
        const bool pair = 2 * t + 1 < C::NB;
        const int b0 = 2 * t, b1 = pair ? 2 * t + 1 : 2 * t;
        swat_lds q0 = rowp[b0 / C::NWB] + 2 * C::TB + (b0 % C::NWB) * C::BLKB, q1 = rowp[b1 / C::NWB] + 2 * C::TB + (b1 % C::NWB) * C::BLKB;
#pragma unroll
        for (int d = 0; d < C::DB; d++) {
          const u32x2 lo = swat_read_tr(q0 + C::TB + L.tr[d]), hi = pair || !C::ALONE ? swat_read_tr(q1 + C::TB + L.tr[d]) : u32x2{0u, 0u};
          acc_v[d] = Mma<CT>::mfma(u32x4{lo.x, lo.y, hi.x, hi.y}, pb, acc_v[d]);
        }
#pragma unroll
        for (int d = 0; d < C::DB; d++) {
          const u32x2 lo = swat_read_tr(q0 + L.tr[d]), hi = pair || !C::ALONE ? swat_read_tr(q1 + L.tr[d]) : u32x2{0u, 0u};
          acc_k[d] = Mma<CT>::mfma(u32x4{lo.x, lo.y, hi.x, hi.y}, dsb, acc_k[d]);
        }
        // 128 registers a lane: reads hoisted across pairs of blocks spilled the pieces in flight, a wait for them at the step's start
        __builtin_amdgcn_sched_barrier(0);
      }
      swat_store_row<CT, C::DB, true>(out1 + (uint32_t)r * out1rs, acc_v, 1.f, lane);
      swat_store_row<CT, C::DB, true>(out0 + (uint32_t)r * out0rs, acc_k, a.sm_scale, lane);
    };
    if (own) {
      if (is_q) {
        if (seen.all()) step_q(std::false_type{});
        else step_q(std::true_type{});
      } else {
        if (seen.all()) step_kv(std::false_type{});
        else step_kv(std::true_type{});
      }
    }
    if (more) {
      __syncthreads();
      commit(slot0, next);   // the row that left the window
      __syncthreads();
      slot0 = slot0 + 1 == C::NR ? 0 : slot0 + 1;
    }
  }
}
