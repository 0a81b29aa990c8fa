// Marching forward kernel for fp32 token grids (b_size == 1, head dim 32, no rotation): the frame of swag_kernel.hpp with
// the arithmetic of the generic kernels (q and k as hi + lo bf16 pairs, three products per score; v and the probabilities
// rounded to bf16 once).  o is normalised by the sum of the rounded probabilities its product uses; lse2, from which the
// backward kernels rebuild unrounded ones, comes from the sum of the probabilities as they are.
//
// These calls ran on the generic kernels, whose workgroups own 64 consecutive tokens of ONE grid row: on a 16 x 16 map three
// quarters of a workgroup had no token, and every row staged its whole halo for itself.  Back-to-back calls, before -> after:
// 2 heads of 16 x 16, 7 x 7 window 14.2 -> 6.0 us (the host path), 64 heads of 32 x 32, 9 x 9 window 73.6 -> 10.4 us (34 MB,
// 3.2 TB/s: the LDS reads of the three score products and the launch are the rest).
//
// A score outside the window is replaced, whatever it is (an infinite or NaN key row must not reach the queries that do not see it).  As
// an addend of 0 or -inf the row test was up to 5 % faster and let them through: 32 slabs of 64 x 64, 13 x 13 window 21.1 -> 22.1 us, 16 of
// 89 x 98, 11 x 7 22.6 -> 23.6, small maps the same.
//
// LDS: three planes per chunk (k hi, k lo, v), token rows of 2 D bytes, swizzled as in swag_kernel.hpp.
#pragma once
#include "swag_kernel.hpp"

template <int D, int NCH, int NCG>
struct SwagF : Swag<D, NCH, NCG, SWAG_PC> {
  typedef Swag<D, NCH, NCG, SWAG_PC> B;
  static constexpr int SLOT = 3 * B::TB, RING = B::NRES * SLOT, OCC = RING <= 80 * 1024 ? 4 : 2;
  static_assert(RING <= 160 * 1024, "the ring exceeds the LDS");
};

// 8 fp32 values -> bf16, and what is left of them as bf16
DLT_DEV void swagf_split(const f32x4& a, const f32x4& b, u32x4& hi, u32x4& lo) {
  float f[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]}, h[8];
  hi = pack8<bf16_t>(f);
  unpack8<bf16_t>(hi, h);
#pragma unroll
  for (int j = 0; j < 8; j++) f[j] -= h[j];
  lo = pack8<bf16_t>(f);
}

template <typename C>
struct SwagFRing {
  swat_lds lds;
  const char *kb, *vb;
  int ksn, vsn, tid, c0, WC, TR, TC;
  struct At { bool on, v; int hr, hc, piece; };
  DLT_DEV At at(int it) const {
    const int id = tid + 512 * it;
    At p;
    p.on = id < C::NV;
    p.v = id >= C::NV / 2;
    const int x = p.v ? id - C::NV / 2 : id, tok = x / C::PIECES;
    p.piece = x % C::PIECES;
    p.hr = tok / C::HCW;
    p.hc = tok - p.hr * C::HCW;
    return p;
  }
  DLT_DEV void issue(f32x4 (&r)[C::NIT][2], int first) const {
#pragma unroll
    for (int it = 0; it < C::NIT; it++) {
      const At p = at(it);
      if (!p.on) continue;
      const int tok = dlt_imax(0, dlt_imin(first + p.hr, TR - 1)) * TC + dlt_imax(0, dlt_imin(c0 - WC + p.hc, TC - 1));
      const char* q = (p.v ? vb + (uint32_t)(tok * vsn) : kb + (uint32_t)(tok * ksn)) + 32 * p.piece;
      r[it][0] = *reinterpret_cast<const f32x4*>(q);
      r[it][1] = *reinterpret_cast<const f32x4*>(q + 16);
    }
  }
  DLT_DEV void commit(const f32x4 (&r)[C::NIT][2], int slot) const {
#pragma unroll
    for (int it = 0; it < C::NIT; it++) {
      const At p = at(it);
      if (!p.on) continue;
      u32x4 hi, lo;
      swagf_split(r[it][0], r[it][1], hi, lo);
      swat_lds d = lds + slot * C::SLOT + (p.hr * C::HCW + p.hc) * C::ROWB + 16 * (p.piece ^ swag_swz<C::ROWB / 2>(p.hr, p.hc));
      if (p.v) {
        swat_write16(d + 2 * C::TB, hi);
      } else {
        swat_write16(d, hi);
        swat_write16(d + C::TB, lo);
      }
    }
  }
};

template <int D, int NCH, int NCG>
__global__ __launch_bounds__(512, (SwagF<D, NCH, NCG>::OCC)) void swag_fwd_f32_kernel(const SwagArgs a) {
  typedef SwagF<D, NCH, NCG> C;
  typedef bf16_t CT;
  extern __shared__ __align__(16) char smem[];
  const int tid = threadIdx.x;
  SwagFrame<C, SWAG_PC> F;
  F.init(a, tid);
  const int b = F.w.b, h = F.w.h, n = F.n, g = F.g;
  SwagFRing<C> ring;
  ring.lds = (swat_lds)smem;
  ring.kb = reinterpret_cast<const char*>(reinterpret_cast<const float*>(a.k) + b * a.ks[0] + h * a.ks[1]);
  ring.vb = reinterpret_cast<const char*>(reinterpret_cast<const float*>(a.v) + b * a.vs[0] + h * a.vs[1]);
  ring.ksn = (int)a.ks[2] * 4; ring.vsn = (int)a.vs[2] * 4;
  ring.tid = tid; ring.c0 = F.w.c0; ring.WC = F.WC; ring.TR = F.TR; ring.TC = F.TC;
  const char* qb = reinterpret_cast<const char*>(reinterpret_cast<const float*>(a.q) + b * a.qs[0] + h * a.qs[1]) + 32 * g;
  float* ob = reinterpret_cast<float*>(a.out_o) + b * a.os[0] + h * a.os[1] + 4 * g;
  float* lseb = a.lse + b * a.ls[0] + h * a.ls[1];
  const int qsn = (int)a.qs[2] * 4;
  SwagLane<C> L;
  L.init(n, g);
  const float scale = a.scale_log2;
  const unsigned one2 = pack2<CT>(1.f, 1.f);
  const u32x4 ones = {one2, one2, one2, one2};

  f32x4 qn[C::KC][2];
  auto load_q = [&](int rp) {
    const uint32_t off = (uint32_t)(F.own_tok(rp) * qsn);
#pragma unroll
    for (int c = 0; c < C::KC; c++) {
      qn[c][0] = *reinterpret_cast<const f32x4*>(qb + off + 128 * c);
      qn[c][1] = *reinterpret_cast<const f32x4*>(qb + off + 128 * c + 16);
    }
  };
  load_q(F.w.r0 + 4 * F.rg);
  {
    f32x4 pre[C::NRES][C::NIT][2];
#pragma unroll
    for (int i = 0; i < C::NRES; i++) ring.issue(pre[i], F.w.r0 - F.WR + 4 * i);
#pragma unroll
    for (int i = 0; i < C::NRES; i++) ring.commit(pre[i], i);
  }
  __syncthreads();

  int slot0 = 0;
  for (int r = F.w.r0; r < F.w.r1; r += 4 * C::PR) {
    const int rp = r + 4 * F.rg;
    u32x4 qh[C::KC], ql[C::KC];
#pragma unroll
    for (int c = 0; c < C::KC; c++) swagf_split(qn[c][0], qn[c][1], qh[c], ql[c]);
    const bool more = r + 4 * C::PR < F.w.r1;
    f32x4 nx[C::PR][C::NIT][2];
    if (more) {
#pragma unroll
      for (int i = 0; i < C::PR; i++) ring.issue(nx[i], r - F.WR + 4 * (C::NRES + i));
      load_q(rp + 4 * C::PR);
    }
    if (rp < F.TR && F.w.c0 + 4 * F.pc < F.TC) {
      swat_lds rowp[NCH];
#pragma unroll
      for (int i = 0; i < NCH; i++) {
        const int s = slot0 + F.rg + i;
        rowp[i] = ring.lds + (s >= C::NRES ? s - C::NRES : s) * C::SLOT + 4 * F.pc * C::ROWB;
      }
      f32x4 s[C::NB + 1];
      float mx[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
#pragma unroll
      for (int i = 0; i < NCH; i++) {
        const bool row = F.sees_row(i, rp);
#pragma unroll
        for (int j = 0; j < NCG; j++) {
          swat_lds blk = rowp[i] + 4 * j * C::ROWB;
          f32x4 t = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int c = 0; c < C::KC; c++) {
            const u32x4 kh = swat_read16(blk + L.row[c]), kl = swat_read16(blk + C::TB + L.row[c]);
            t = Mma<CT>::mfma(kl, qh[c], t);
            t = Mma<CT>::mfma(kh, ql[c], t);
            t = Mma<CT>::mfma(kh, qh[c], t);
          }
#pragma unroll
          for (int e = 0; e < 4; e++) {
            t[e] = (row & F.sees_col(4 * j + e)) ? t[e] : -INFINITY;
            mx[e] = fmaxf(mx[e], t[e]);
          }
          s[i * NCG + j] = t;
        }
        __builtin_amdgcn_sched_barrier(0);   // the scores of one row of blocks at a time: read further ahead, the operands spill
      }
      const float m = wave_max4(fmaxf(fmaxf(mx[0], mx[1]), fmaxf(mx[2], mx[3])));
      const float m_use = m == -INFINITY ? 0.f : m;
      const float neg_m2 = -m_use * scale;
      f32x4 acc[C::DB], acc_l = {0.f, 0.f, 0.f, 0.f};
      float psum = 0.f;   // of the probabilities as they are, for lse2
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
#pragma unroll
        for (int e = 0; e < 8; e++) psum += p[e];
        const u32x4 pb = pack8<CT>(p);
        swat_lds v0 = rowp[b0 / NCG] + 2 * C::TB + 4 * (b0 % NCG) * C::ROWB, v1 = rowp[b1 / NCG] + 2 * C::TB + 4 * (b1 % NCG) * C::ROWB;
#pragma unroll
        for (int d = 0; d < C::DB; d++) {
          const u32x2 lo = swat_read_tr(v0 + L.tr[d]), hi = swat_read_tr(v1 + L.tr[d]);
          acc[d] = Mma<CT>::mfma(u32x4{lo.x, lo.y, hi.x, hi.y}, pb, acc[d]);
        }
        acc_l = Mma<CT>::mfma(ones, pb, acc_l);
      }
      const float l = acc_l[0], lsum = wave_sum4(psum);
      if (F.own_ok(rp)) {
        const int tok = F.own_tok(rp);
        const float inv = fast_rcp(l);
#pragma unroll
        for (int d = 0; d < C::DB; d++) __builtin_nontemporal_store(acc[d] * inv, reinterpret_cast<f32x4*>(ob + tok * a.os[2] + 16 * d));
        if (g == 0) store_stream4(lseb + tok * a.ls[2], m_use * scale + fast_log2(lsum));
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
}
