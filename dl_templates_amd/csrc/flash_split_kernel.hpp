// Dense / causal flash attention for calls with too few own blocks to fill the chip: few queries against many keys (and
// the transpose), short sequences, few heads.
//
// What bounded those calls: the kernels that stream chunks through LDS give one wave 32 own tokens and walk the other side
// one 64-token chunk after the other, so 77 queries x 1500 keys x 16 heads were 16 workgroups of 24 dependent rounds
// (22.5 us on 6 % of the CUs).  Here a workgroup owns 16 NP tokens and its NW waves split the OTHER side: wave w takes the
// 32-token blocks w, w + NW, ...  The waves share nothing while they stream, so there is no barrier in the loop: row operands
// come straight from HBM / L2 one block ahead, the tensors that are also needed transposed pass through a wave-private LDS
// tile.  At the end the partial results meet in LDS: (m, l, o) of the forward pass by the usual rescaling, gradients by
// plain fp32 sums, in a fixed order (results do not depend on timing).
#pragma once
#include "flash_kernel.hpp"

template <int D> DLT_DEV int flashs_swz(int t) { return D == 32 ? ((t >> 2) & 1) << 1 : (t & 7) * (D / 64); }

// The other side's tokens as a list, in blocks of 32.  MODE 0 dense, 1 causal: tokens 0 ... len - 1, reads clamped to the last one.
template <int MODE>
struct FlashsList {
  int len;
  DLT_DEV int token(int b, int half, int i) const { return dlt_imin(32 * b + 16 * half + i, len - 1); }
};
// 2 (3: tensors in the image layout): the window of own token x0 over tiles of S = 16 k tokens, which its whole block shares: runs of `pieces` x 16 tokens, one per grid row, and no
// pair of tokens in it is masked.  The window is symmetric: queries that see a key are listed the same way.
template <>
struct FlashsList<2> {
  int len, first, row, pieces;
  unsigned magic;       // ceil(2^32 / pieces)
  DLT_DEV FlashsList(const DltGeom& g, int x0) {
    const int r = x0 / g.XLk, c = (x0 - r * g.XLk) / g.S;
    const int rlo = dlt_imax(r - g.WR, 0), rhi = dlt_imin(r + g.WR, g.TR - 1), clo = dlt_imax(c - g.WC, 0), chi = dlt_imin(c + g.WC, g.TC - 1);
    row = g.XLk;
    first = rlo * row + clo * g.S;
    pieces = (chi - clo + 1) * (g.S / 16);
    len = 16 * pieces * (rhi - rlo + 1);
    magic = 0xffffffffu / (unsigned)pieces + 1;
  }
  DLT_DEV int token(int b, int half, int i) const {
    const int p = dlt_imin(2 * b + half, len / 16 - 1), r = pieces == 1 ? p : (int)__umulhi((unsigned)p, magic);
    return first + r * row + 16 * (p - r * pieces) + i;
  }
};

template <> struct FlashsList<3> : FlashsList<2> { using FlashsList<2>::FlashsList; };
template <int MODE>
DLT_DEV FlashsList<MODE> flashs_list(const DltGeom& g, int len, int x0) {
  if constexpr (MODE >= 2) return FlashsList<MODE>(g, x0);
  else return FlashsList<MODE>{len};
}
// elements between a slab's start and token x; Rows: the same in 32 bits and bytes for the other side's tokens
template <int MODE>
DLT_DEV int64_t flashs_at(const DltTokMap& tm, const int64_t (&s)[5], int x) {
  if constexpr (MODE == 3) return tok_addr(s, tm)(x);
  else return x * s[2];
}
template <int MODE>
struct FlashsRows {
  int sn2;
  DLT_DEV FlashsRows(const DltTokMap&, const int64_t (&s)[5]) : sn2((int)s[2] * 2) {}
  DLT_DEV int operator()(int token) const { return token * sn2; }
};
template <>
struct FlashsRows<3> {
  int sn2, sy2;
  const DltTokMap& tm;
  DLT_DEV FlashsRows(const DltTokMap& m, const int64_t (&s)[5]) : sn2((int)s[2] * 2), sy2((int)s[4] * 2), tm(m) {}
  DLT_DEV int operator()(int token) const {
    uint32_t y, x;
    dlt_token_pixel(tm, (uint32_t)token, y, x);
    return (int)y * sy2 + (int)x * sn2;
  }
};

// wave-private [32 tokens][D] tile, rows of 2 D bytes, 16-byte piece p of token t at p ^ swz(t)
template <int D>
struct FlashsTile {
  static constexpr int BYTES = 64 * D, NV = D / 16;   // 16-byte vectors per lane of one block
  // rows of block `b`; pieces past `dact` are left as they are (zero, from the caller).  A lane has one piece of every row: one branch, inside which the
  // loads follow each other
  template <typename Rows, typename List>
  static DLT_DEV void load(u32x4 (&r)[NV], const char* base, const Rows& at, int b, const List& list, int dact, int lane) {
    const int p = lane % (D / 8);
    if (8 * p >= dact) return;
#pragma unroll
    for (int it = 0; it < NV; it++) {
      const int t = (lane + 64 * it) / (D / 8), half = 64 * it / (D / 8) / 16;
      r[it] = *reinterpret_cast<const u32x4*>(base + (uint32_t)(at(list.token(b, half, t - 16 * half)) + 16 * p));
    }
  }
  static DLT_DEV void write(char* s, const u32x4 (&r)[NV], int lane) {
#pragma unroll
    for (int it = 0; it < NV; it++) {
      const int v = lane + 64 * it, t = v / (D / 8), p = v % (D / 8);
      lds_write16(s + t * 2 * D + 16 * (p ^ flashs_swz<D>(t)), r[it]);
    }
  }
  // Tiles: a block's tokens from `left` on repeat the list's last one: their probabilities are 0, which times an infinite value is not, so that they are cleared
  // (dense calls, where that token is the sequence's last one, go without: it costs short backward passes 3 to 5 %)
  static DLT_DEV void clear_past(u32x4 (&r)[NV], int left, int lane) {
    if (left >= 32) return;   // wave-uniform
#pragma unroll
    for (int it = 0; it < NV; it++)
      if ((lane + 64 * it) / (D / 8) >= left) r[it] = u32x4{0u, 0u, 0u, 0u};
  }
  // A operand, 16 tokens (half mb) x dims 32 c ..
  static DLT_DEV u32x4 rows(const char* s, int mb, int c, int n, int g) {
    return lds_read16(s + (16 * mb + n) * 2 * D + 16 * ((4 * c + g) ^ flashs_swz<D>(n)));
  }
  // A operand, dims 16 d .. as rows, the 32 tokens along k
  static DLT_DEV u32x4 trans(const char* s, int d, int n, int g) {
    const int t = 4 * g + (n >> 2);
    const char* p = s + t * 2 * D + 16 * ((2 * d + ((n >> 1) & 1)) ^ flashs_swz<D>(t)) + 8 * (n & 1);
    const u32x2 lo = lds_read_tr16(p), hi = lds_read_tr16(p + 32 * D);   // token t + 16: same swizzle
    return u32x4{lo.x, lo.y, hi.x, hi.y};
  }
};

// A operand rows straight from HBM: 32 tokens of block b (pieces past `dact`: as above)
template <int D, typename Rows, typename List>
DLT_DEV void flashs_load_rows(u32x4 (&f)[2][D / 32], const char* base, const Rows& at, int b, const List& list, int dact, int n, int g) {
#pragma unroll
  for (int c = 0; c < D / 32; c++)
    if (8 * (4 * c + g) < dact) {
#pragma unroll
      for (int mb = 0; mb < 2; mb++) f[mb][c] = *reinterpret_cast<const u32x4*>(base + (uint32_t)(at(list.token(b, mb, n)) + 64 * c + 16 * g));
    }
}
// an own row's operands, one lane's 8 dims of every 32
template <int N, typename T>
DLT_DEV void flashs_own(u32x4 (&f)[N], const T* row, int dact, int g) {
#pragma unroll
  for (int c = 0; c < N; c++) f[c] = *reinterpret_cast<const u32x4*>(row + (8 * (4 * c + g) < dact ? 32 * c + 8 * g : 0));
}
template <int N>
DLT_DEV void flashs_own_zero(u32x4 (&f)[N], int dact, int g) {
#pragma unroll
  for (int c = 0; c < N; c++) f[c] = 8 * (4 * c + g) < dact ? f[c] : u32x4{0u, 0u, 0u, 0u};
}

// Partial [16 NP][D] results of NW waves (C layout: lane n = own token, dims 16 d + 4 g + i) -> their sum, 8 dims per thread and
// turn: out(row, first dim, 8 values).
template <int D, int NP, int NW>
struct FlashsSum {
  static constexpr int P = D + 4;                      // fp32 row pitch
  static constexpr int BYTES = NW * 16 * NP * P * 4;
  static DLT_DEV void put(float* s, const f32x4 (&acc)[NP][D / 16], int wave, int n, int g) {
#pragma unroll
    for (int p = 0; p < NP; p++)
#pragma unroll
      for (int d = 0; d < D / 16; d++) *reinterpret_cast<f32x4*>(s + ((wave * NP + p) * 16 + n) * P + 16 * d + 4 * g) = acc[p][d];
  }
  template <typename Out>
  static DLT_DEV void reduce(const float* s, int tid, Out out) {
    for (int id = tid; id < 16 * NP * (D / 8); id += 64 * NW) {
      const int row = id / (D / 8), c = id % (D / 8);
      f32x4 a = {0.f, 0.f, 0.f, 0.f}, b = a;
#pragma unroll
      for (int w = 0; w < NW; w++) {
        const float* q = s + (w * 16 * NP + row) * P + 8 * c;
        a += *reinterpret_cast<const f32x4*>(q);
        b += *reinterpret_cast<const f32x4*>(q + 4);
      }
      float v[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
      out(row, 8 * c, v);
    }
  }
};

// workgroup -> (batch * head, first own token)
DLT_DEV void flashs_block(int nblk, int own, int& bh, int& x0) {
  const int lin = xcd_remap(blockIdx.x, gridDim.x);
  bh = lin / nblk;
  x0 = (lin - bh * nblk) * own;
}

template <int DK, int DV, int NP, int NW>
constexpr int flashs_lds_fwd() {
  const int tiles = NW * FlashsTile<DV>::BYTES, sum = FlashsSum<DV, NP, NW>::BYTES + 2 * NW * 16 * NP * 4;
  return tiles > sum ? tiles : sum;
}

// a.parts workgroups take DV of an own block's output dims each: scores and softmax are formed in every one of them, K is read by all and V by
// one.  A CU reads the other side at 55 B/ns whatever the others do, so narrower parts take less time while CUs are idle (flash_forward has the
// line and figures), with the same bits.
template <typename TIO, int DK, int DV, int NP, int NW, int MODE>
__global__ __launch_bounds__(64 * NW, NW / 4) void flashs_fwd_kernel(const FlashArgs a) {
  typedef typename ComputeOf<TIO>::type CT;
  constexpr bool CAUSAL = MODE == 1;
  extern __shared__ __align__(16) char smem[];
  constexpr int KC = DK / 32, VB = DV / 16;
  typedef FlashsTile<DV> VT;
  typedef FlashsSum<DV, NP, NW> Sum;
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int bh, part, x0;
  flash_block(xcd_remap(blockIdx.x, gridDim.x), a.nblk, a.parts, 16 * NP, bh, part, x0);
  const int v0 = part * DV, dv = dlt_imin(a.dv - v0, DV);   // first output dim, their number
  const int b = bh / a.H, h = bh - b * a.H;
  const TIO* qb = reinterpret_cast<const TIO*>(a.q) + b * a.qs[0] + h * a.qs[1];
  const char* kb_ = reinterpret_cast<const char*>(reinterpret_cast<const TIO*>(a.k) + b * a.ks[0] + h * a.ks[1]);
  const char* vb_ = reinterpret_cast<const char*>(reinterpret_cast<const TIO*>(a.v) + b * a.vs[0] + h * a.vs[1] + v0);
  const FlashsRows<MODE> ksn(a.tm, a.ks), vsn(a.tm, a.vs);
  const FlashsList<MODE> keys = flashs_list<MODE>(a.g, a.Lk, x0);
  const int nkb = ((CAUSAL ? dlt_imin(keys.len, x0 + 16 * NP) : keys.len) + 31) / 32;   // causal: keys up to the last own query
  char* sV = smem + wave * VT::BYTES;

  u32x4 kf[2][KC] = {}, vr[VT::NV] = {};
  if (wave < nkb) {
    flashs_load_rows<DK>(kf, kb_, ksn, wave, keys, a.dk, n, g);
    VT::load(vr, vb_, vsn, wave, keys, dv, lane);
  }
  u32x4 qf[NP][KC];
#pragma unroll
  for (int p = 0; p < NP; p++) {
    const int x = x0 + 16 * p + n;
    flashs_own(qf[p], qb + flashs_at<MODE>(a.tm, a.qs, dlt_imin(x, a.Lq - 1)), a.dk, g);
  }
  float m_run[NP], l_run[NP];
  f32x4 acc[NP][VB];
#pragma unroll
  for (int p = 0; p < NP; p++) {
    flashs_own_zero(qf[p], x0 + 16 * p + n < a.Lq ? a.dk : 0, g);
    m_run[p] = -INFINITY;
    l_run[p] = 0.f;
#pragma unroll
    for (int d = 0; d < VB; d++) acc[p][d] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const float scale = a.scale_log2;
  for (int kb = wave; kb < nkb; kb += NW) {
    if constexpr (MODE >= 2) VT::clear_past(vr, keys.len - 32 * kb, lane);
    VT::write(sV, vr, lane);
    u32x4 ka[2][KC];
#pragma unroll
    for (int mb = 0; mb < 2; mb++)
#pragma unroll
      for (int c = 0; c < KC; c++) ka[mb][c] = kf[mb][c];
    if (kb + NW < nkb) {
      flashs_load_rows<DK>(kf, kb_, ksn, kb + NW, keys, a.dk, n, g);
      VT::load(vr, vb_, vsn, kb + NW, keys, dv, lane);
    }
    const bool tail = 32 * kb + 32 > keys.len || (CAUSAL && 32 * kb + 31 > x0);
    u32x4 pb[NP];
#pragma unroll
    for (int p = 0; p < NP; p++) {
      f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = s0;
#pragma unroll
      for (int c = 0; c < KC; c++) {
        s0 = Mma<CT>::mfma(ka[0][c], qf[p][c], s0);
        s1 = Mma<CT>::mfma(ka[1][c], qf[p][c], s1);
      }
      float t[8] = {s0[0], s0[1], s0[2], s0[3], s1[0], s1[1], s1[2], s1[3]};
      if (tail) {
        const int klim = CAUSAL ? dlt_imin(x0 + 16 * p + n, keys.len - 1) : keys.len - 1;
#pragma unroll
        for (int i = 0; i < 8; i++) t[i] = 32 * kb + 16 * (i >> 2) + 4 * g + (i & 3) <= klim ? t[i] : -INFINITY;
      }
      const float mloc = wave_max4(fmaxf(fmaxf(fmaxf(t[0], t[1]), fmaxf(t[2], t[3])), fmaxf(fmaxf(t[4], t[5]), fmaxf(t[6], t[7]))));
      if (__builtin_amdgcn_ballot_w64((mloc - m_run[p]) * scale > 8.f)) {   // the reference maximum moves (see flash_fwd_kernel)
        keep_branch();
        const float m_new = fmaxf(m_run[p], mloc);
        const float alpha = m_run[p] == m_new ? 1.f : fast_exp2((m_run[p] - m_new) * scale);
        m_run[p] = m_new;
#pragma unroll
        for (int d = 0; d < VB; d++) acc[p][d] *= alpha;
        l_run[p] *= alpha;
      }
      const float neg_m2 = m_run[p] == -INFINITY ? 0.f : -m_run[p] * scale;
#pragma unroll
      for (int i = 0; i < 8; i++) t[i] = fast_exp2(fmaf(t[i], scale, neg_m2));
      pb[p] = pack8<CT>(t);
      const unsigned one2 = pack2<CT>(1.f, 1.f);   // row sums of the rounded probabilities, per lane group
      l_run[p] = dot2_acc<CT>(pb[p].w, one2, dot2_acc<CT>(pb[p].z, one2, dot2_acc<CT>(pb[p].y, one2, dot2_acc<CT>(pb[p].x, one2, l_run[p]))));
    }
#pragma unroll
    for (int d = 0; d < VB; d++) {
      const u32x4 vt = VT::trans(sV, d, n, g);
#pragma unroll
      for (int p = 0; p < NP; p++) acc[p][d] = Mma<CT>::mfma(vt, pb[p], acc[p][d]);
    }
  }
  // ---- the waves' partial results meet
  float* sums = reinterpret_cast<float*>(smem);
  float* sm = reinterpret_cast<float*>(smem + Sum::BYTES);   // [wave][own] maxima, then row sums
  float* sl = sm + NW * 16 * NP;
  __syncthreads();
#pragma unroll
  for (int p = 0; p < NP; p++) {
    const float l = wave_sum4(l_run[p]);
    if (g == 0) {
      sm[wave * 16 * NP + 16 * p + n] = m_run[p];
      sl[wave * 16 * NP + 16 * p + n] = l;
    }
  }
  __syncthreads();
#pragma unroll
  for (int p = 0; p < NP; p++) {
    float m = -INFINITY;
#pragma unroll
    for (int w = 0; w < NW; w++) m = fmaxf(m, sm[w * 16 * NP + 16 * p + n]);
    const float f = m_run[p] == -INFINITY ? 0.f : fast_exp2((m_run[p] - m) * scale);
#pragma unroll
    for (int d = 0; d < VB; d++) acc[p][d] *= f;
  }
  Sum::put(sums, acc, wave, n, g);
  __syncthreads();
  auto total = [&](int row, float& m, float& l) {
    m = -INFINITY;
    l = 0.f;
#pragma unroll
    for (int w = 0; w < NW; w++) m = fmaxf(m, sm[w * 16 * NP + row]);
#pragma unroll
    for (int w = 0; w < NW; w++) {
      const float mw = sm[w * 16 * NP + row];
      l += mw == -INFINITY ? 0.f : sl[w * 16 * NP + row] * fast_exp2((mw - m) * scale);
    }
  };
  TIO* ob = reinterpret_cast<TIO*>(a.o) + b * a.os[0] + h * a.os[1];
  Sum::reduce(sums, tid, [&](int row, int d0, float* v) {
    if (x0 + row >= a.Lq || d0 >= dv) return;
    float m, l;
    total(row, m, l);
    const float inv = l > 0.f ? fast_rcp(l) : 0.f;
#pragma unroll
    for (int j = 0; j < 8; j++) v[j] *= inv;
    Io<TIO, CT>::store8(ob + flashs_at<MODE>(a.tm, a.os, x0 + row) + (v0 + d0) * a.os[3], v, a.o_vec != 0, a.os[3], dlt_imin(8, dv - d0));
    if (d0 == 0 && part == 0) store_stream4(a.lse + (b * a.ls[0] + h * a.ls[1] + (x0 + row) * a.ls[2]), m * scale + fast_log2(l));
  });
}

template <int DK, int DV, int NP, int NW>
constexpr int flashs_lds_q() {
  const int tiles = NW * FlashsTile<DK>::BYTES, sum = FlashsSum<DK, NP, NW>::BYTES;
  return tiles > sum ? tiles : sum;
}

// dQ: own = queries, the waves split the keys; delta of the own queries is formed (fuse_delta) and stored on the way
template <typename TIO, int DK, int DV, int NP, int NW, int MODE>
__global__ __launch_bounds__(64 * NW, NW / 4) void flashs_bwd_q_kernel(const FlashBwdArgs a) {
  typedef typename ComputeOf<TIO>::type CT;
  constexpr bool CAUSAL = MODE == 1;
  extern __shared__ __align__(16) char smem[];
  constexpr int KC = DK / 32, VC = DV / 32, KB = DK / 16;
  typedef FlashsTile<DK> KT;
  typedef FlashsSum<DK, NP, NW> Sum;
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int bh, x0;
  flashs_block(a.nblk_q, 16 * NP, bh, x0);
  const int b = bh / a.H, h = bh - b * a.H;
  const TIO* qb = reinterpret_cast<const TIO*>(a.q) + b * a.qs[0] + h * a.qs[1];
  const TIO* dob = reinterpret_cast<const TIO*>(a.d_o) + b * a.dos[0] + h * a.dos[1];
  const TIO* ob = reinterpret_cast<const TIO*>(a.o) + b * a.os[0] + h * a.os[1];
  const char* kb_ = reinterpret_cast<const char*>(reinterpret_cast<const TIO*>(a.k) + b * a.ks[0] + h * a.ks[1]);
  const char* vb_ = reinterpret_cast<const char*>(reinterpret_cast<const TIO*>(a.v) + b * a.vs[0] + h * a.vs[1]);
  const FlashsRows<MODE> ksn(a.tm, a.ks), vsn(a.tm, a.vs);
  const FlashsList<MODE> keys = flashs_list<MODE>(a.g, a.Lk, x0);
  const int nkb = ((CAUSAL ? dlt_imin(keys.len, x0 + 16 * NP) : keys.len) + 31) / 32;
  char* sK = smem + wave * KT::BYTES;

  u32x4 kr[KT::NV] = {}, vf[2][VC] = {};
  if (wave < nkb) {
    KT::load(kr, kb_, ksn, wave, keys, a.dk_, lane);
    flashs_load_rows<DV>(vf, vb_, vsn, wave, keys, a.dv_, n, g);
  }
  u32x4 qf[NP][KC], dof[NP][VC];
  float nlse[NP];
  f32x4 dinit[NP], acc[NP][KB];
#pragma unroll
  for (int p = 0; p < NP; p++) {
    const int x = x0 + 16 * p + n;
    const bool in = x < a.Lq;
    const int xc = dlt_imin(x, a.Lq - 1);
    flashs_own(qf[p], qb + flashs_at<MODE>(a.tm, a.qs, xc), a.dk_, g);
    flashs_own(dof[p], dob + flashs_at<MODE>(a.tm, a.dos, xc), a.dv_, g);
    const int64_t off = b * a.ls[0] + h * a.ls[1] + xc * a.ls[2];
    nlse[p] = a.lse[off];
    float del;
    if (a.fuse_delta != 0) {
      u32x4 of[VC];
      flashs_own(of, ob + flashs_at<MODE>(a.tm, a.os, xc), a.dv_, g);
      flashs_own_zero(of, in ? a.dv_ : 0, g);
      flashs_own_zero(dof[p], in ? a.dv_ : 0, g);
      float part = 0.f;
#pragma unroll
      for (int c = 0; c < VC; c++) {
        float fo[8], fd[8];
        unpack8<CT>(of[c], fo);
        unpack8<CT>(dof[p][c], fd);
#pragma unroll
        for (int j = 0; j < 8; j++) part += fo[j] * fd[j];
      }
      del = wave_sum4(part);
      if (wave == 0 && g == 0 && in) store_stream4(a.delta_out + off, del);
    } else {
      flashs_own_zero(dof[p], in ? a.dv_ : 0, g);
      del = in ? a.delta[off] : 0.f;
    }
    flashs_own_zero(qf[p], in ? a.dk_ : 0, g);
    nlse[p] = in ? -nlse[p] : 0.f;
    dinit[p] = f32x4{-del, -del, -del, -del};
#pragma unroll
    for (int d = 0; d < KB; d++) acc[p][d] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const float scale = a.scale_log2;
  for (int kb = wave; kb < nkb; kb += NW) {
    if constexpr (MODE >= 2) KT::clear_past(kr, keys.len - 32 * kb, lane);
    KT::write(sK, kr, lane);
    u32x4 va[2][VC];
#pragma unroll
    for (int mb = 0; mb < 2; mb++)
#pragma unroll
      for (int c = 0; c < VC; c++) va[mb][c] = vf[mb][c];
    if (kb + NW < nkb) {
      KT::load(kr, kb_, ksn, kb + NW, keys, a.dk_, lane);
      flashs_load_rows<DV>(vf, vb_, vsn, kb + NW, keys, a.dv_, n, g);
    }
    const bool tail = 32 * kb + 32 > keys.len || (CAUSAL && 32 * kb + 31 > x0);
    u32x4 dsb[NP];
    float ds[NP][8];
#pragma unroll
    for (int mb = 0; mb < 2; mb++) {
      u32x4 ka[KC];
#pragma unroll
      for (int c = 0; c < KC; c++) ka[c] = KT::rows(sK, mb, c, n, g);
#pragma unroll
      for (int p = 0; p < NP; p++) {
        f32x4 s = {0.f, 0.f, 0.f, 0.f}, dp = dinit[p];
#pragma unroll
        for (int c = 0; c < KC; c++) s = Mma<CT>::mfma(ka[c], qf[p][c], s);
#pragma unroll
        for (int c = 0; c < VC; c++) dp = Mma<CT>::mfma(va[mb][c], dof[p][c], dp);
        const int klim = CAUSAL ? dlt_imin(x0 + 16 * p + n, keys.len - 1) : keys.len - 1;
#pragma unroll
        for (int i = 0; i < 4; i++) {
          float pv = fast_exp2(fmaf(s[i], scale, nlse[p]));
          if (tail) pv = 32 * kb + 16 * mb + 4 * g + i <= klim ? pv : 0.f;
          ds[p][4 * mb + i] = pv * dp[i];
          if (MODE >= 2 && tail) ds[p][4 * mb + i] = 32 * kb + 16 * mb + 4 * g + i <= klim ? ds[p][4 * mb + i] : 0.f;
        }
      }
    }
#pragma unroll
    for (int p = 0; p < NP; p++) dsb[p] = pack8<CT>(ds[p]);
#pragma unroll
    for (int d = 0; d < KB; d++) {
      const u32x4 kt = KT::trans(sK, d, n, g);
#pragma unroll
      for (int p = 0; p < NP; p++) acc[p][d] = Mma<CT>::mfma(kt, dsb[p], acc[p][d]);
    }
  }
  float* sums = reinterpret_cast<float*>(smem);
  __syncthreads();
  Sum::put(sums, acc, wave, n, g);
  __syncthreads();
  TIO* dqb = reinterpret_cast<TIO*>(a.dq) + b * a.dqs[0] + h * a.dqs[1];
  Sum::reduce(sums, tid, [&](int row, int d0, float* v) {
    if (x0 + row >= a.Lq || d0 >= a.dk_) return;
#pragma unroll
    for (int j = 0; j < 8; j++) v[j] *= a.sm_scale;
    Io<TIO, CT>::store8(dqb + flashs_at<MODE>(a.tm, a.dqs, x0 + row) + d0 * a.dqs[3], v, a.dq_vec != 0, a.dqs[3], dlt_imin(8, a.dk_ - d0));
  });
}

template <int DK, int DV, int NP, int NW>
constexpr int flashs_lds_kv() {
  const int tiles = NW * (FlashsTile<DK>::BYTES + FlashsTile<DV>::BYTES + 256);
  const int sk = FlashsSum<DK, NP, NW>::BYTES, sv = FlashsSum<DV, NP, NW>::BYTES;
  return tiles > sk ? (tiles > sv ? tiles : sv) : (sk > sv ? sk : sv);
}

// dK / dV: own = keys, the waves split the queries
template <typename TIO, int DK, int DV, int NP, int NW, int MODE>
__global__ __launch_bounds__(64 * NW, NW / 4) void flashs_bwd_kv_kernel(const FlashBwdArgs a) {
  typedef typename ComputeOf<TIO>::type CT;
  constexpr bool CAUSAL = MODE == 1;
  extern __shared__ __align__(16) char smem[];
  constexpr int KC = DK / 32, VC = DV / 32, KB = DK / 16, VB = DV / 16;
  typedef FlashsTile<DK> QT;
  typedef FlashsTile<DV> DT;
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int bh, x0;
  flashs_block(a.nblk_k, 16 * NP, bh, x0);
  const int b = bh / a.H, h = bh - b * a.H;
  const TIO* kb_ = reinterpret_cast<const TIO*>(a.k) + b * a.ks[0] + h * a.ks[1];
  const TIO* vb_ = reinterpret_cast<const TIO*>(a.v) + b * a.vs[0] + h * a.vs[1];
  const char* qb = reinterpret_cast<const char*>(reinterpret_cast<const TIO*>(a.q) + b * a.qs[0] + h * a.qs[1]);
  const char* dob = reinterpret_cast<const char*>(reinterpret_cast<const TIO*>(a.d_o) + b * a.dos[0] + h * a.dos[1]);
  // lanes 0 ... 31 fetch lse2, lanes 32 ... 63 delta of a block's queries
  const float* scb = (lane < 32 ? a.lse : a.delta) + b * a.ls[0] + h * a.ls[1];
  const FlashsRows<MODE> qsn(a.tm, a.qs), dosn(a.tm, a.dos);
  const FlashsList<MODE> queries = flashs_list<MODE>(a.g, a.Lq, x0);
  const int nqb = (queries.len + 31) / 32;
  char* sQ = smem + wave * (QT::BYTES + DT::BYTES + 256);
  char* sD = sQ + QT::BYTES;
  float* sc = reinterpret_cast<float*>(sD + DT::BYTES);

  u32x4 qr[QT::NV] = {}, dr[DT::NV] = {};
  float scr = 0.f;
  const int first = (CAUSAL ? x0 / 32 : 0) + wave;   // causal: queries below the first own key see none of the own keys
  auto fetch = [&](int blk) {
    QT::load(qr, qb, qsn, blk, queries, a.dk_, lane);
    DT::load(dr, dob, dosn, blk, queries, a.dv_, lane);
    if constexpr (MODE >= 2) scr = scb[((lane & 16) ? queries.token(blk, 1, lane & 15) : queries.token(blk, 0, lane & 15)) * a.ls[2]];
    else scr = scb[dlt_imin(32 * blk + (lane & 31), queries.len - 1) * a.ls[2]];
  };
  if (first < nqb) fetch(first);
  u32x4 kf[NP][KC], vf[NP][VC];
  f32x4 acc_k[NP][KB], acc_v[NP][VB];
#pragma unroll
  for (int p = 0; p < NP; p++) {
    const int x = x0 + 16 * p + n;
    flashs_own(kf[p], kb_ + flashs_at<MODE>(a.tm, a.ks, dlt_imin(x, a.Lk - 1)), a.dk_, g);
    flashs_own(vf[p], vb_ + flashs_at<MODE>(a.tm, a.vs, dlt_imin(x, a.Lk - 1)), a.dv_, g);
    flashs_own_zero(kf[p], x < a.Lk ? a.dk_ : 0, g);
    flashs_own_zero(vf[p], x < a.Lk ? a.dv_ : 0, g);
    // negated: with the products started from delta the matrix pipe delivers -(dP - delta)
#pragma unroll
    for (int c = 0; c < VC; c++) {
      vf[p][c].x ^= 0x80008000u; vf[p][c].y ^= 0x80008000u; vf[p][c].z ^= 0x80008000u; vf[p][c].w ^= 0x80008000u;
    }
#pragma unroll
    for (int d = 0; d < KB; d++) acc_k[p][d] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int d = 0; d < VB; d++) acc_v[p][d] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const float scale = a.scale_log2;
  for (int qbk = first; qbk < nqb; qbk += NW) {
    if constexpr (MODE >= 2) {
      QT::clear_past(qr, queries.len - 32 * qbk, lane);
      DT::clear_past(dr, queries.len - 32 * qbk, lane);
    }
    QT::write(sQ, qr, lane);
    DT::write(sD, dr, lane);
    sc[lane] = scr;
    if (qbk + NW < nqb) fetch(qbk + NW);
    const bool tail = 32 * qbk + 32 > queries.len || (CAUSAL && 32 * qbk < x0 + 16 * NP - 1);
    float pr[NP][8], ds[NP][8];
#pragma unroll
    for (int mb = 0; mb < 2; mb++) {
      u32x4 qa[KC], da[VC];
#pragma unroll
      for (int c = 0; c < KC; c++) qa[c] = QT::rows(sQ, mb, c, n, g);
#pragma unroll
      for (int c = 0; c < VC; c++) da[c] = DT::rows(sD, mb, c, n, g);
      const f32x4 lq = *reinterpret_cast<const f32x4*>(sc + 16 * mb + 4 * g), dl = *reinterpret_cast<const f32x4*>(sc + 32 + 16 * mb + 4 * g);
#pragma unroll
      for (int p = 0; p < NP; p++) {
        f32x4 s = {0.f, 0.f, 0.f, 0.f}, dp = dl;
#pragma unroll
        for (int c = 0; c < KC; c++) s = Mma<CT>::mfma(qa[c], kf[p][c], s);
#pragma unroll
        for (int c = 0; c < VC; c++) dp = Mma<CT>::mfma(da[c], vf[p][c], dp);
        const int qmin = CAUSAL ? x0 + 16 * p + n : 0;
#pragma unroll
        for (int i = 0; i < 4; i++) {
          float pv = fast_exp2(fmaf(s[i], scale, -lq[i]));
          const int qi = 32 * qbk + 16 * mb + 4 * g + i;
          if (tail) pv = (qi >= qmin && qi < queries.len) ? pv : 0.f;
          pr[p][4 * mb + i] = pv;
          ds[p][4 * mb + i] = -pv * dp[i];
          if (MODE >= 2 && tail) ds[p][4 * mb + i] = qi < queries.len ? ds[p][4 * mb + i] : 0.f;
        }
      }
    }
    u32x4 pb[NP], dsb[NP];
#pragma unroll
    for (int p = 0; p < NP; p++) {
      pb[p] = pack8<CT>(pr[p]);
      dsb[p] = pack8<CT>(ds[p]);
    }
#pragma unroll
    for (int d = 0; d < VB; d++) {
      const u32x4 dt = DT::trans(sD, d, n, g);
#pragma unroll
      for (int p = 0; p < NP; p++) acc_v[p][d] = Mma<CT>::mfma(dt, pb[p], acc_v[p][d]);
    }
#pragma unroll
    for (int d = 0; d < KB; d++) {
      const u32x4 qt = QT::trans(sQ, d, n, g);
#pragma unroll
      for (int p = 0; p < NP; p++) acc_k[p][d] = Mma<CT>::mfma(qt, dsb[p], acc_k[p][d]);
    }
  }
  float* sums = reinterpret_cast<float*>(smem);
  __syncthreads();
  FlashsSum<DK, NP, NW>::put(sums, acc_k, wave, n, g);
  __syncthreads();
  TIO* dkb = reinterpret_cast<TIO*>(a.dk) + b * a.dks[0] + h * a.dks[1];
  FlashsSum<DK, NP, NW>::reduce(sums, tid, [&](int row, int d0, float* v) {
    if (x0 + row >= a.Lk || d0 >= a.dk_) return;
#pragma unroll
    for (int j = 0; j < 8; j++) v[j] *= a.sm_scale;
    Io<TIO, CT>::store8(dkb + flashs_at<MODE>(a.tm, a.dks, x0 + row) + d0 * a.dks[3], v, a.dk_vec != 0, a.dks[3], dlt_imin(8, a.dk_ - d0));
  });
  __syncthreads();
  FlashsSum<DV, NP, NW>::put(sums, acc_v, wave, n, g);
  __syncthreads();
  TIO* dvb = reinterpret_cast<TIO*>(a.dv) + b * a.dvs[0] + h * a.dvs[1];
  FlashsSum<DV, NP, NW>::reduce(sums, tid, [&](int row, int d0, float* v) {
    if (x0 + row >= a.Lk || d0 >= a.dv_) return;
    Io<TIO, CT>::store8(dvb + flashs_at<MODE>(a.tm, a.dvs, x0 + row) + d0 * a.dvs[3], v, a.dv_vec != 0, a.dvs[3], dlt_imin(8, a.dv_ - d0));
  });
}
