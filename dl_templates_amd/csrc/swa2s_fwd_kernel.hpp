// Forward kernel for token grids at head dims 64 and 128 (b_size == 1 and tiles of 2 ... 15 tokens, no rotation), two stacked
// patches per wave: the work of tiled_swa_fwd_kernel (src/tiled_swa.py:15-133) on the streaming structure of swa2_common.hpp.
// A workgroup of 4 waves owns a band of 8 rows x 16 columns, wave w the two 4x4 patches at column 4 w: both see the same
// window columns, so every K fragment read from LDS feeds the score products of both patches and every V^T fragment both
// output products.
//
// K and V of a chunk have ONE buffer each: V of a chunk is copied while its scores are formed, K of the next chunk during
// the output products, a barrier between the two.  A workgroup then fits into half the LDS of a CU (74 KB at head dim 128,
// 6 column groups), and the two (head dim 64: up to four) workgroups of a CU are in different phases: one fills the waits of the
// other.  An earlier version ran 8 waves over bands of 16 rows with both chunk buffers doubled, one workgroup per CU: the waves
// stood together at every barrier, and half of them had no row of the first two and last two chunks.  Back-to-back calls on one set
// of inputs, 16 slabs at d = 128, 21 x 21 window: 128 x 128 tokens 99.7 -> 94.7 us, 97 x 161 105.7 -> 94 (over three sets of inputs in
// turn 112.6 -> 104.5); 32 slabs of 103 x 36, 21 x 7: 54.2 -> 45.2; d = 64, 32 slabs of 89 x 98, 15 x 21: 74 -> 66.6 (there against one
// patch per wave).  Of 106 us in a short burst the
// matrix and vector instructions account for 71 (the issue port), LDS operand reads and the copies for the rest: without
// either of the two it runs in 91 ... 94.  Leaving out the column test where a whole group is inside every window, a longer
// read-ahead of K and copies issued earlier in their phase measured the same within 1 %.
//
// The row sums are two-element dot products on the vector pipe (fp32 accumulation of the rounded probabilities): the matrix
// instruction of swa2_fwd_kernel would take registers that are not there (256 at 6 column groups).
#pragma once
#include "swa2_fwd_kernel.hpp"

constexpr int SWA2S_THREADS = 256;
// waves per SIMD the register budget is sized for (head dim 64 at 6 column groups spills at 3)
constexpr int swa2s_occ(int D, int NCG) { return D == 64 && NCG == 4 ? 3 : 2; }

template <typename TIO, int D, int NCG, bool SAME, bool PAD, bool TALL>
__global__ __launch_bounds__(SWA2S_THREADS, swa2s_occ(D, NCG)) void swa2s_fwd_kernel(const Swa2FwdArgs a) {
  typedef typename ComputeOf<TIO>::type CT;
  typedef Swa2Cfg<D, NCG, PAD> C;
  constexpr int KC = C::KC, VB = C::VB, NKB = C::NKB;
  constexpr int NG = VB / 4;   // groups of four 16-dim blocks of the output
  static_assert(C::NI <= 2 * NCG && C::NI <= 2 * NKB * NG && 4 * C::TILE <= C::BUF, "copy slots of a phase; the store epilogue");
  extern __shared__ __align__(16) char smem[];
  const int tid = threadIdx.x;
  const int lane = tid & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const Swa2Geom G0 = swa2_geom<TALL>(a.p, a.plan);
  const int pc = wave & ((1 << G0.lpc) - 1), rg = 2 * (wave >> G0.lpc);

  const char* qb = reinterpret_cast<const char*>(a.q) + 2 * (G0.b * a.qs[0] + G0.h * a.qs[1]);
  const char* kb_ = reinterpret_cast<const char*>(a.k) + 2 * (G0.b * a.ks[0] + G0.h * a.ks[1]);
  const char* vb_ = reinterpret_cast<const char*>(a.v) + 2 * (G0.b * a.vs[0] + G0.h * a.vs[1]);
  TIO* ob = reinterpret_cast<TIO*>(a.o) + G0.b * a.os[0] + G0.h * a.os[1];
  float* lseb = a.lse + G0.b * a.ls[0] + G0.h * a.ls[1];
  const int64_t os2 = a.os[2], ls2 = a.ls[2];
  const float scale = a.scale_log2;

  // staging: wave w copies halo row w of every chunk, of K and of V.  SAME: one set of lane offsets serves both tensors (equal token
  // strides); V in another layout has offsets of its own (at head dim 128 and 6 column groups 6 more registers spill outside the
  // loops; 128 x 128, 21 x 21, 16 slabs, V as [B, N, H, D]: 105 us, 119 on the one-patch kernel that took these calls before)
  const int ksn2 = (int)a.ks[2] * 2, vsn2 = (int)a.vs[2] * 2;
  const uint32_t krow = (uint32_t)(G0.TC * ksn2), vrow = (uint32_t)(G0.TC * vsn2);
  Swa2Geom G = G0;   // column pass 0
  Swa2Stage<C> st, st_own;
  swa2_clear<C, SWA2S_THREADS>(smem, C::BUF, tid);
  swa2_stage_init(st, G, wave, lane, ksn2, a.p.dk);
  if constexpr (!SAME) swa2_stage_init(st_own, G, wave, lane, vsn2, a.p.dv);
  const Swa2Stage<C>& stv = SAME ? st : st_own;
  swa2_issue(st, G, G.ch_first, kb_, krow, smem, wave);

  // own queries of both patches straight into B-operand fragments
  const int c_p = G.c0 + 4 * pc;
  int r_p[2], tq[2];
  u32x4 qf[2][KC];
  Swa2Win W0[2], W[2];
#pragma unroll
  for (int p = 0; p < 2; p++) {
    r_p[p] = G.r0 + 4 * (rg + p);
    tq[p] = (r_p[p] + (n >> 2) < G.TR && c_p + (n & 3) < G.TC) ? (r_p[p] + (n >> 2)) * G.TC + c_p + (n & 3) : -1;
    swa2_own_frags<KC, PAD>(qf[p], qb, (int)a.qs[2] * 2, tq[p], g, a.p.dk);
    W0[p] = swa2_window(G0, rg + p, pc, n);
    W[p] = W0[p];
  }
  Swa2Lane<C> L;
  swa2_lane_init(L, pc, n, g);

  float m_run[2] = {-INFINITY, -INFINITY};
  f32x4 acc[2][VB];
  float lsum[2] = {0.f, 0.f};   // per lane: sum of the probabilities of its own token over the halo rows g of every chunk
#pragma unroll
  for (int p = 0; p < 2; p++) {
#pragma unroll
    for (int d = 0; d < VB; d++) acc[p][d] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const unsigned one2 = pack2<CT>(1.f, 1.f);

  swa2_wait_copies();   // also: the own fragments have arrived
  pin_loaded(qf);
  __syncthreads();

  // PM: the patches that see rows of the chunk (bit 0: the upper patch, bit 1: the lower one).  The chunks of a wave come
  // in the order "upper only" (at most one), "both", "lower only" (at most one); the one-patch bodies issue no product,
  // mask, exponential or reduction for the other patch.
  auto consume = [&](const int ch, auto more_tag, auto pm_tag) {
    constexpr bool more = decltype(more_tag)::value;   // a later chunk exists: its K is copied between the output products
    constexpr int PM = decltype(pm_tag)::value;
    constexpr bool P0 = (PM & 1) != 0, P1 = (PM & 2) != 0;
    Swa2Lds sK = (Swa2Lds)smem;
    Swa2Lds sV = sK + C::REGION;
    const char* nrow = swa2_issue_row(G, ch, vb_, vrow, wave);
    char* ndst = swa2_issue_dst<C>(smem + C::REGION, wave);
    const int hrow = 4 * ch + g;
    // a lane's keys of a chunk are columns of ONE halo row; the column test is the same for both patches (the own token of patch 1
    // lies below that of patch 0: inside the grid only where that one is).  The two tests are joined as lane masks (scalar pipe)
    // and a score outside the window is replaced, whatever it is: an infinite or NaN key row reaches only the queries that see it.
    const bool row_vis[2] = {(hrow >= W[0].rlo) && (hrow <= W[0].rhi), (hrow >= W[1].rlo) && (hrow <= W[1].rhi) && W[1].cspan >= 0};
    // ---- scores of the chunk, one column group (16 keys) at a time
    float t[2][NKB][8];
    float mx[2][4];
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
      for (int i = 0; i < 4; i++) mx[p][i] = -INFINITY;
    u32x4 ka[KC];
    f32x4 sc[2][2];
    auto mask_max = [&](const int p, const int cg, const f32x4& sv) {
      const int kb = cg >> 1, h4 = 4 * (cg & 1);
#pragma unroll
      for (int i = 0; i < 4; i++) t[p][kb][h4 + i] = (row_vis[p] & ((unsigned)(4 * cg + i - W[0].clo) <= (unsigned)W[0].cspan)) ? sv[i] : -INFINITY;
      mx[p][cg & 3] = fmaxf(fmaxf(mx[p][cg & 3], t[p][kb][h4]), t[p][kb][h4 + 1]);
      mx[p][(cg + 2) & 3] = fmaxf(fmaxf(mx[p][(cg + 2) & 3], t[p][kb][h4 + 2]), t[p][kb][h4 + 3]);
    };
    // K fragments live in ONE set of registers: piece c of the next group is requested as soon as the products of piece c
    // of this group are issued (with two patches every fragment feeds two products, so one group of read-ahead covers
    // the LDS latency)
    swa2_read_a<C, 0>(sK, L, ka);
    swa2_for<0, NCG>([&](auto cgc) {
      constexpr int cg = decltype(cgc)::value;
      f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
      swa2_for<0, KC>([&](auto cc) {
        constexpr int c = decltype(cc)::value;
        if constexpr (c == 0) swa2_issue_one<C, 2 * cg>(stv, nrow, ndst);
        if constexpr (c == KC / 2) swa2_issue_one<C, 2 * cg + 1>(stv, nrow, ndst);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (P0) s0 = Mma<CT>::mfma(ka[c], qf[0][c], s0);
        if constexpr (P1) s1 = Mma<CT>::mfma(ka[c], qf[1][c], s1);
        if constexpr (cg > 0) {
          if (P0 && c == 1) mask_max(0, cg - 1, sc[0][(cg - 1) & 1]);
          if (P1 && c == KC - 1) mask_max(1, cg - 1, sc[1][(cg - 1) & 1]);
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (cg + 1 < NCG) ka[c] = swa2_lds16(sK + swa2_read_a_off<C, cg + 1>(L, c));
        __builtin_amdgcn_sched_barrier(0);
      });
      if constexpr (P0) sc[0][cg & 1] = s0;
      if constexpr (P1) sc[1][cg & 1] = s1;
    });
    if constexpr (P0) mask_max(0, NCG - 1, sc[0][(NCG - 1) & 1]);
    if constexpr (P1) mask_max(1, NCG - 1, sc[1][(NCG - 1) & 1]);
    // reference maxima move only when some score exceeds them by more than 2^8 after scaling (see swa2_fwd_kernel)
    float mloc[2] = {-INFINITY, -INFINITY};
    if constexpr (P0) mloc[0] = wave_max4(fmaxf(fmaxf(mx[0][0], mx[0][1]), fmaxf(mx[0][2], mx[0][3])));
    if constexpr (P1) mloc[1] = wave_max4(fmaxf(fmaxf(mx[1][0], mx[1][1]), fmaxf(mx[1][2], mx[1][3])));
    swa2_for<0, 2>([&](auto pc_) {
      constexpr int p = decltype(pc_)::value;
      if constexpr ((PM >> p) & 1) {
        if (__builtin_amdgcn_ballot_w64((mloc[p] - m_run[p]) * scale > 8.f)) {
          keep_branch();
          const float m_new = fmaxf(m_run[p], mloc[p]);
          // a lane that has not seen a key yet keeps its (zero) accumulators as they are
          const float alpha = m_new == -INFINITY ? 1.f : fast_exp2((m_run[p] - m_new) * scale);
          m_run[p] = m_new;
#pragma unroll
          for (int d = 0; d < VB; d++) acc[p][d] *= alpha;
          lsum[p] *= alpha;
        }
      }
    });
    float neg_m2[2];
#pragma unroll
    for (int p = 0; p < 2; p++) neg_m2[p] = m_run[p] == -INFINITY ? 0.f : -m_run[p] * scale;
    // ---- O^T += V^T P^T, 32 keys at a time: with two patches every V^T fragment feeds two products
    u32x4 va[4];
    u32x4 pb[2][2];
    // V^T fragments live in one set of registers too: fragment d of the next step is requested behind the products of
    // fragment d of this step
    auto read_v = [&](auto ic, const int d) {
      constexpr int i = decltype(ic)::value, kb = i / NG, grp = i % NG;
      const u32x2 lo = swa2_lds_tr(sV + swa2_read_tr_off<C, kb>(L, 4 * grp + d, 0));
      const u32x2 hi = swa2_lds_tr(sV + swa2_read_tr_off<C, kb>(L, 4 * grp + d, 1));
      va[d].x = lo.x; va[d].y = lo.y; va[d].z = hi.x; va[d].w = hi.y;
    };
    // probability of element e (0 .. 7) of block kb for the active patches; the pair (e - 1, e) is packed behind odd e
    auto prob = [&](const int kb, const int e) {
#pragma unroll
      for (int p = 0; p < 2; p++)
        if ((PM >> p) & 1) {
          t[p][kb][e] = fast_exp2(fmaf(t[p][kb][e], scale, neg_m2[p]));
          if (e & 1) pb[p][kb & 1][e >> 1] = pack2<CT>(t[p][kb][e - 1], t[p][kb][e]);
        }
    };
#pragma unroll
    for (int e = 0; e < 8; e++) prob(0, e);
    swa2_wait_copies();
    __syncthreads();   // V of the chunk has landed, every wave is done with its K
    nrow = swa2_issue_row(G, ch + 1, kb_, krow, wave);
    ndst = swa2_issue_dst<C>(smem, wave);
#pragma unroll
    for (int d = 0; d < 4; d++) read_v(std::integral_constant<int, 0>{}, d);
    swa2_for<0, NKB * NG>([&](auto ic) {
      constexpr int i = decltype(ic)::value, kb = i / NG, grp = i % NG;
      const u32x4 pk0 = pb[0][kb & 1], pk1 = pb[1][kb & 1];
      swa2_for<0, 4>([&](auto dc) {
        constexpr int d = decltype(dc)::value;
        if constexpr (more && d == 0) swa2_issue_one<C, 2 * i>(st, nrow, ndst);
        if constexpr (more && d == 2) swa2_issue_one<C, 2 * i + 1>(st, nrow, ndst);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (P0) acc[0][4 * grp + d] = Mma<CT>::mfma(va[d], pk0, acc[0][4 * grp + d]);
        if constexpr (P1) acc[1][4 * grp + d] = Mma<CT>::mfma(va[d], pk1, acc[1][4 * grp + d]);
        if constexpr (kb + 1 < NKB) {
          // the exponentials of the next 32 keys, EPS elements per patch behind every fragment's products
          constexpr int EPS = 2 / NG;
#pragma unroll
          for (int e = (4 * grp + d) * EPS; e < (4 * grp + d + 1) * EPS; e++) prob(kb + 1, e);
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (i + 1 < NKB * NG) read_v(std::integral_constant<int, i + 1>{}, d);
        __builtin_amdgcn_sched_barrier(0);
      });
      if constexpr (grp == NG - 1) {
        // row sums of the rounded probabilities (the values the products above use)
#pragma unroll
        for (int j = 0; j < 4; j++) {
          if constexpr (P0) lsum[0] = dot2_acc<CT>(pk0[j], one2, lsum[0]);
          if constexpr (P1) lsum[1] = dot2_acc<CT>(pk1[j], one2, lsum[1]);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  };

  // Chunk ranges of the two patches (a patch outside the grid has an empty range; the lower patch starts and ends at or
  // after the upper one, and their ranges touch or overlap): upper only, both, lower only.  One loop per kind, in that
  // order, and copy-only rounds before and after, keep the accumulators in place (see swa2_fwd_kernel).
  const bool ok1 = W[1].ch_lo <= W[1].ch_hi;
  const int a_lo = W[0].ch_lo, a_hi = W[0].ch_hi;
  const int b_lo = ok1 ? W[1].ch_lo : a_hi + 1, b_hi = ok1 ? W[1].ch_hi : a_hi;
  const int w_lo = a_lo;
  const int both_lo = dlt_imax(a_lo, b_lo), both_hi = dlt_imin(a_hi, b_hi);
  // a wave without rows in a chunk copies its halo row of V, then of the next chunk's K, at the barriers of consume() and round()
  auto copy_v = [&](int ch) {
    swa2_issue(stv, G, ch, vb_, vrow, smem + C::REGION, wave);
    swa2_wait_copies();
    __syncthreads();
  };
  auto copy_only = [&](int ch) {
    copy_v(ch);
    swa2_issue(st, G, ch + 1, kb_, krow, smem, wave);
    swa2_wait_copies();
    __syncthreads();
  };
  auto round = [&](int ch, auto pm_tag) {
    consume(ch, std::true_type{}, pm_tag);
    swa2_wait_copies();
    __syncthreads();
  };
  typedef std::integral_constant<int, 1> PmUpper;
  typedef std::integral_constant<int, 2> PmLower;
  typedef std::integral_constant<int, 3> PmBoth;
  for (int pass = 0;;) {
    int ch = G.ch_first;
    for (; ch < G.ch_last && ch < w_lo; ch++) copy_only(ch);
    for (; ch < G.ch_last && ch <= a_hi && ch < both_lo; ch++) round(ch, PmUpper{});
    for (; ch < G.ch_last && ch <= both_hi; ch++) round(ch, PmBoth{});
    for (; ch < G.ch_last && ch <= b_hi; ch++) round(ch, PmLower{});
    for (; ch < G.ch_last; ch++) copy_only(ch);
    {
      const int cl = G.ch_last;
      const bool in0 = cl >= a_lo && cl <= a_hi, in1 = ok1 && cl >= b_lo && cl <= b_hi;
      if (in0 && in1) consume(cl, std::false_type{}, PmBoth{});
      else if (in0) consume(cl, std::false_type{}, PmUpper{});
      else if (in1) consume(cl, std::false_type{}, PmLower{});
      else copy_v(cl);   // one barrier, as in consume(): the waves of a workgroup stay in step for the next column pass
    }
    __syncthreads();   // every wave is done with the chunk
    if (++pass >= a.plan.npass) break;
    G = swa2_pass_geom(G0, NCG, pass);
    W[0] = swa2_pass_window(W0[0], NCG, pass);
    W[1] = swa2_pass_window(W0[1], NCG, pass);
    swa2_stage_init(st, G, wave, lane, ksn2, a.p.dk);
    if constexpr (!SAME) swa2_stage_init(st_own, G, wave, lane, vsn2, a.p.dv);
    swa2_issue(st, G, G.ch_first, kb_, krow, smem, wave);
    swa2_wait_copies();
    __syncthreads();
  }

  // ---- epilogue (the loop ended with a barrier: the chunk buffers are free), one patch after the other
#pragma unroll
  for (int p = 0; p < 2; p++) {
    const float lt = wave_sum4(lsum[p]);
    const float inv = lt > 0.f ? fast_rcp(lt) : 0.f;
    if (g == 0 && tq[p] >= 0) store_stream4(lseb + (int64_t)tq[p] * ls2, m_run[p] * scale + fast_log2(lt));
    swa2_store_own<C, TIO, CT>(smem + wave * C::TILE, acc[p], inv, ob, os2, G, r_p[p], c_p, lane, a.p.dv);
  }
}
