// Windowed forward attention on fp32 tensors whose rows can be read in 16-byte pieces, without rotation: the generic forward kernel's
// arithmetic (attn_fwd_kernel.hpp: hi + lo pairs of q and k, three products to a score, fp32 softmax and sums) for maps that fit a few workgroups.
//
// What bounds such calls is latency: the generic kernel stages one halo row after the other, a wait for memory each, behind a prologue that
// fetches its arguments as it needs them.  Here
//   - the halo rows of a chunk are one list of tokens, 4 x 32 rows of K and as many of V in flight at once, and a small map is one chunk;
//   - a workgroup of 4 waves owns 16, 32 or 64 columns of 4, 2 or 1 grid rows (every halo row is staged once for all of them), or, while CUs would
//     be idle, of fewer rows with the parts of a row's window dealt over the waves that are left (WinArgs::wave_shift; their sums meet in LDS);
//   - a block of 32 keys is two halo rows where a row has at most 16 tokens, one whole row up to 32, else it starts at the wave's first column.
// A slab's bits do not depend on how many a call holds: a window's rows are summed in parts (WinArgs::parts), each from nothing, which are added in order
// whether one wave takes them one after the other or several side by side, and the blocks start at the window's first row whatever the
// rows of a workgroup and of a chunk (in pairs of rows chunks overlap by one).
// (figures at win_plan)
#pragma once
#include "attn_common.hpp"

struct WinArgs {
  const float *q, *k, *v;
  float *o, *lse;
  int64_t qs[2], ks[2], vs[2], os[2], ls[2];    // batch, head strides (elements)
  int32_t qn, kn, vn, on, ln;                   // token strides (elements; a slab spans less than 2^31 bytes)
  int32_t H, TR, XL, WR, WC;
  int32_t dk, dv;
  int32_t patch_shift;   // 1 << patch_shift blocks of 16 queries lie side by side
  int32_t parts;         // a window's rows are summed in 4, 2 or 1 parts (by the map's width and the window alone: win_plan)
  int32_t wave_shift;    // 1 << wave_shift waves share a grid row: the blocks, times the waves that its parts are dealt over
  int32_t chunk_rows, cx, pair;   // halo rows staged at once, LDS slots of a row, two rows to a block of keys
  float scale_log2;
};

constexpr int win_pitch_k(int DK) { return DK * 4 + 16; }
constexpr int win_pitch_v(int DV) { return DV * 2 + 16; }
constexpr int win_per_token(int DK, int DV) { return win_pitch_k(DK) + win_pitch_v(DV); }
constexpr int win_sum_bytes(int DV) { return 4 * 64 * (DV + 8); }   // DV / 16 fragments of 16 bytes, maximum and sum: per lane of up to four parts
// (in pairs of rows the half block beside a lone one may lie behind the chunk)
constexpr int win_lds_bytes(int DK, int DV, int rows, int cx, bool pair) {
  const int chunk = rows * cx * win_per_token(DK, DV) + (pair ? 16 * win_pitch_v(DV) : 0);
  return chunk > win_sum_bytes(DV) ? chunk : win_sum_bytes(DV);
}

// running maximum, row sum and output rows of a part
template <int VB>
struct WinSum {
  float m, l;
  f32x4 acc[VB];
  DLT_DEV void clear() {
    m = -INFINITY;
    l = 0.f;
#pragma unroll
    for (int d = 0; d < VB; d++) acc[d] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  template <typename F>
  DLT_DEV void add(float m2, float l2, const F& acc2) {
    const float m_new = fmaxf(m, m2), m_use = m_new == -INFINITY ? 0.f : m_new, f1 = fast_exp2(m - m_use), f2 = fast_exp2(m2 - m_use);
    m = m_new;
    l = l * f1 + l2 * f2;
#pragma unroll
    for (int d = 0; d < VB; d++) acc[d] = acc[d] * f1 + acc2(d) * f2;
  }
};

// U rows per thread of one operand: loads, then conversion and LDS writes.  Reads are clamped into the chunk and the head dims, not predicated.
template <int D, int U>
struct WinTile {
  static constexpr int CH = D / 8, RSTEP = 256 / CH;
  f32x4 r[U][2];
  DLT_DEV static int row(int tid, int j, int u) { return tid / CH + (j * U + u) * RSTEP; }
  DLT_DEV void load(const char* base, int sn, int d, int tok0, int xl, int w, unsigned magic, int total, int tid, int j) {
    const int c = tid % CH, off = 8 * c < d ? 32 * c : 0;
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int i = dlt_imin(row(tid, j, u), total - 1), ri = (int)(((unsigned)i * magic) >> 20);
      const char* p = base + (uint32_t)((tok0 + ri * xl + i - ri * w) * sn + off);
      r[u][0] = *reinterpret_cast<const f32x4*>(p);
      r[u][1] = *reinterpret_cast<const f32x4*>(p + 16);
    }
  }
  template <bool SPLIT>
  DLT_DEV void store(char* s, int pitch, int d, int w, int cx, unsigned magic, int total, int tid, int j) const {
    const int c = tid % CH;
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int i = row(tid, j, u), ri = (int)(((unsigned)i * magic) >> 20);
      if (i >= total) continue;
      float f[8];
#pragma unroll
      for (int e = 0; e < 8; e++) f[e] = 8 * c < d ? r[u][e / 4][e % 4] : 0.f;
      char* dst = s + (ri * cx + i - ri * w) * pitch + c * 16;
      lds_write16(dst, pack8<bf16_t>(f));
      if constexpr (SPLIT) {
#pragma unroll
        for (int e = 0; e < 8; e++) f[e] -= (float)(bf16_t)f[e];
        lds_write16(dst + D * 2, pack8<bf16_t>(f));
      }
    }
  }
};

// MULTI: a wave takes several parts
template <int DK, int DV, bool MULTI>
__global__ __launch_bounds__(256, 2) void attn_win_fwd_kernel(const WinArgs a) {
  typedef bf16_t CT;
  extern __shared__ __align__(16) char smem[];
  constexpr int PK = win_pitch_k(DK), PV = win_pitch_v(DV), KC = DK / 32, VB = DV / 16;
  constexpr int U = 4;
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = (int)blockIdx.x / a.H, h = (int)blockIdx.x - b * a.H;
  const int rows = 4 >> a.wave_shift;
  const int r0 = blockIdx.y * rows, rlast = dlt_imin(r0 + rows, a.TR) - 1;
  const int x0 = (int)blockIdx.z * (16 << a.patch_shift), xlast = dlt_imin(x0 + (16 << a.patch_shift), a.XL) - 1;
  const int r = r0 + (wave >> a.wave_shift);
  const int in_row = wave & ((1 << a.wave_shift) - 1), turn = in_row >> a.patch_shift;
  const int xw = x0 + 16 * (in_row & ((1 << a.patch_shift) - 1));   // first column of the wave's queries
  const bool live = r <= rlast && xw <= xlast;

  // columns [lo, hi) that queries x1 ... x2 see
  auto first = [&](int x) { return dlt_imax(x - a.WC, 0); };
  auto past = [&](int x) { return dlt_imin(x + a.WC + 1, a.XL); };
  const int rlo = dlt_imax(r0 - a.WR, 0), rhi = dlt_imin(rlast + a.WR, a.TR - 1);
  const int wrlo = dlt_imax(r - a.WR, 0), wrhi = live ? dlt_imin(r + a.WR, a.TR - 1) : -1;
  const int X0 = first(x0), w = past(xlast) - X0;
  const int wlo = first(xw) - X0, whi = past(dlt_imin(xw + 15, xlast)) - X0;   // of the wave, relative to X0
  const int xq = dlt_imin(xw + n, xlast);
  const int xlo = first(xq) - X0;
  const unsigned span = past(xq) - X0 - xlo;
  const int cx = a.cx;
  const bool whole = cx <= 32;    // a block of keys is a whole row (or two)

  const char* qb = reinterpret_cast<const char*>(a.q + b * a.qs[0] + h * a.qs[1]);
  const char* kb_ = reinterpret_cast<const char*>(a.k + b * a.ks[0] + h * a.ks[1]);
  const char* vb_ = reinterpret_cast<const char*>(a.v + b * a.vs[0] + h * a.vs[1]);
  char *sK = smem, *sV = smem + a.chunk_rows * cx * PK;

  // own queries as B operands
  f32x4 qr[KC][2];
  {
    const char* p = qb + (uint32_t)((dlt_imin(r, a.TR - 1) * a.XL + xq) * (a.qn * 4));
#pragma unroll
    for (int c = 0; c < KC; c++) {
      const int off = 32 * c + 8 * g < a.dk ? (32 * c + 8 * g) * 4 : 0;
      qr[c][0] = *reinterpret_cast<const f32x4*>(p + off);
      qr[c][1] = *reinterpret_cast<const f32x4*>(p + off + 16);
    }
  }
  u32x4 qf[KC], qlo[KC];

  // a probability of 0 times an infinite value is not 0: the columns of a block from kx on that no query of the wave sees are cleared
  auto seen_values = [&](int kx) {
    unsigned m[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const int x = kx + (i < 4 || a.pair ? 4 * g : 16 + 4 * g) + (i & 3);
      m[i] = x >= wlo && x < whi ? 0xffffu : 0u;
    }
    return u32x4{m[0] | m[1] << 16, m[2] | m[3] << 16, m[4] | m[5] << 16, m[6] | m[7] << 16};
  };
  // (the blocks of longer rows start at the first such column: it is their last one that holds others)
  const u32x4 vmask = seen_values(whole ? 0 : wlo + (whi - 1 - wlo) / 32 * 32), all = {~0u, ~0u, ~0u, ~0u};
  // slots past the halo's columns hold no value
  for (int i = tid; i < a.chunk_rows * (cx - w) * (DV / 8); i += 256) {
    const int t = i / (DV / 8), ri = t / (cx - w);
    lds_write16(sV + (ri * cx + w + t - ri * (cx - w)) * PV + i % (DV / 8) * 16, u32x4{0u, 0u, 0u, 0u});
  }

  // the wave's parts of the window: rows next ... stop in steps of part_rows; the first wave of a row adds them up, others keep theirs (two at most) apart
  const int parts = a.parts, own_parts = MULTI ? parts >> (a.wave_shift - a.patch_shift) : 1, nwin = wrhi - wrlo + 1;
  const int part_rows = a.pair ? ((nwin + 2 * parts - 1) / (2 * parts)) * 2 : (nwin + parts - 1) / parts;
  int next = wrlo + turn * own_parts * part_rows, part_end = next + part_rows;
  const int stop = dlt_imin(wrhi, next + own_parts * part_rows - 1);
  WinSum<VB> cur, sum;   // of the current part; of those before it
  cur.clear();
  if constexpr (MULTI) sum.clear();
  auto close = [&]() {
    cur.l = wave_sum4(cur.l);
    if constexpr (MULTI) {
      if (turn == 0) sum.add(cur.m, cur.l, [&](int d) { return cur.acc[d]; });
      else sum = cur;
    }
  };
  const float scale = a.scale_log2;
  const unsigned magic = (0x100000u + w - 1) / (unsigned)w;   // i / w while i * w < 2^20: a chunk holds some 1000 tokens at most

  for (int kr0 = rlo, last = 0; !last; kr0 += a.chunk_rows - a.pair) {
    const int nr = dlt_imin(a.chunk_rows, rhi - kr0 + 1), total = nr * w;
    last = kr0 + nr > rhi;
    if (kr0 != rlo) __syncthreads();
    for (int j = 0; j * U * (2048 / DK) < total; j++) {
      WinTile<DK, U> K;
      WinTile<DV, DK == DV ? U : U * DV / DK> V;    // as many rows a step
      K.load(kb_, a.kn * 4, a.dk, kr0 * a.XL + X0, a.XL, w, magic, total, tid, j);
      V.load(vb_, a.vn * 4, a.dv, kr0 * a.XL + X0, a.XL, w, magic, total, tid, j);
      K.template store<true>(sK, PK, a.dk, w, cx, magic, total, tid, j);
      V.template store<false>(sV, PV, a.dv, w, cx, magic, total, tid, j);
    }
    if (kr0 == rlo) {
#pragma unroll
      for (int c = 0; c < KC; c++) {
        float f[8];
#pragma unroll
        for (int e = 0; e < 8; e++) f[e] = 32 * c + 8 * g < a.dk ? qr[c][e / 4][e % 4] : 0.f;
        qf[c] = pack8<CT>(f);
#pragma unroll
        for (int e = 0; e < 8; e++) f[e] -= (float)(bf16_t)f[e];
        qlo[c] = pack8<CT>(f);
      }
    }
    __syncthreads();

    for (; next <= stop && next < kr0 + nr; next += 1 + a.pair) {
      const bool lone = a.pair && next == wrhi;   // the block's second half is no row of this wave
      if (a.pair && !lone && next + 1 == kr0 + nr) break;   // the pair lies in the next chunk
      const int ri = next - kr0;
      if constexpr (MULTI)
        if (next == part_end) {
          close();
          cur.clear();
          part_end += part_rows;
        }
      for (int kx = whole ? 0 : wlo; kx < whi; kx += 32) {
        const int kb = ri * cx + kx;
        u32x4 ka[2][KC], kl[2][KC], vt[VB];
#pragma unroll
        for (int mb = 0; mb < 2; mb++)
#pragma unroll
          for (int c = 0; c < KC; c++) {
            ka[mb][c] = lds_read16(sK + (kb + 16 * mb + n) * PK + (32 * c + 8 * g) * 2);
            kl[mb][c] = lds_read16(sK + (kb + 16 * mb + n) * PK + DK * 2 + (32 * c + 8 * g) * 2);
          }
#pragma unroll
        for (int d = 0; d < VB; d++) {
          vt[d] = lds_read_tokens_as_k(sV, PV, kb, 16 * d, n, g);
        }
        f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < KC; c++) {   // the small terms first
          s0 = Mma<CT>::mfma(kl[0][c], qf[c], s0);
          s1 = Mma<CT>::mfma(kl[1][c], qf[c], s1);
          s0 = Mma<CT>::mfma(ka[0][c], qlo[c], s0);
          s1 = Mma<CT>::mfma(ka[1][c], qlo[c], s1);
          s0 = Mma<CT>::mfma(ka[0][c], qf[c], s0);
          s1 = Mma<CT>::mfma(ka[1][c], qf[c], s1);
        }
        float t[8];
        const int k0 = kx + 4 * g - xlo, k1 = a.pair ? k0 : k0 + 16;
#pragma unroll
        for (int i = 0; i < 4; i++) {
          t[i] = (unsigned)(k0 + i) < span ? s0[i] * scale : -INFINITY;
          t[4 + i] = (unsigned)(k1 + i) < span && !lone ? s1[i] * scale : -INFINITY;
        }
        float mloc = fmaxf(fmaxf(fmaxf(t[0], t[1]), fmaxf(t[2], t[3])), fmaxf(fmaxf(t[4], t[5]), fmaxf(t[6], t[7])));
        mloc = wave_max4(mloc);
        const float m_new = fmaxf(cur.m, mloc);
        const float m_use = m_new == -INFINITY ? 0.f : m_new;
        const float alpha = fast_exp2(cur.m - m_use);
        cur.m = m_new;
        float psum = 0.f;
#pragma unroll
        for (int i = 0; i < 8; i++) { t[i] = fast_exp2(t[i] - m_use); psum += t[i]; }
        cur.l = cur.l * alpha + psum;
        if (__builtin_amdgcn_ballot_w64(alpha != 1.f)) {
#pragma unroll
          for (int d = 0; d < VB; d++) cur.acc[d] *= alpha;
        }
        const u32x4 pb = pack8<CT>(t), seen = whole || kx + 32 > whi ? vmask : all;
#pragma unroll
        for (int d = 0; d < VB; d++) {
          vt[d] &= seen;
          if (lone) vt[d].z = vt[d].w = 0u;
          cur.acc[d] = Mma<CT>::mfma(vt[d], pb, cur.acc[d]);
        }
      }
    }
  }

  WinSum<VB>& total = MULTI ? sum : cur;
  if (own_parts < parts) {   // the other waves' parts reach the first one through LDS
    __syncthreads();
    const int patches = 1 << a.patch_shift;
    auto slot = [&](int part) { return smem + (((wave >> a.wave_shift) * (parts - own_parts) + part - own_parts) * patches + (in_row & (patches - 1))) * 64 * (DV + 8); };
    auto put = [&](int part, const WinSum<VB>& p) {
      char* s = slot(part);
#pragma unroll
      for (int d = 0; d < VB; d++) lds_write16(s + (d * 64 + lane) * 16, __builtin_bit_cast(u32x4, p.acc[d]));
      float* ml = reinterpret_cast<float*>(s + 64 * DV);
      ml[lane] = p.m; ml[64 + lane] = p.l;
    };
    if (turn > 0) {
      cur.l = wave_sum4(cur.l);
      if (own_parts > 1) put(turn * own_parts, sum);
      put((turn + 1) * own_parts - 1, cur);
    }
    __syncthreads();
    if (turn > 0) return;
    close();
    for (int part = own_parts; part < parts; part++) {
      const char* s = slot(part);
      const float* ml = reinterpret_cast<const float*>(s + 64 * DV);
      total.add(ml[lane], ml[64 + lane], [&](int d) { return __builtin_bit_cast(f32x4, lds_read16(s + (d * 64 + lane) * 16)); });
    }
  } else close();
  if (!live || xw + n > xlast) return;
  const float inv = total.l > 0.f ? fast_rcp(total.l) : 0.f;
  float* o = reinterpret_cast<float*>(reinterpret_cast<char*>(a.o + b * a.os[0] + h * a.os[1]) + (uint32_t)((r * a.XL + xq) * (a.on * 4)));
#pragma unroll
  for (int d = 0; d < VB; d++)
    if (16 * d + 4 * g < a.dv) store_stream16f(o + 16 * d + 4 * g, total.acc[d][0] * inv, total.acc[d][1] * inv, total.acc[d][2] * inv, total.acc[d][3] * inv);
  if (g == 0) store_stream4(a.lse + (b * a.ls[0] + h * a.ls[1] + (int64_t)(r * a.XL + xq) * a.ln), total.m + fast_log2(total.l));
}
