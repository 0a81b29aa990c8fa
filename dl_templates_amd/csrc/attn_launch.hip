// Host side of the attention core: validation that depends on the kernels' limits, the
// per-launch LDS / chunking plan, and dispatch to the instantiation for the padded head dims.
#include "attn_fwd_kernel.hpp"
#include "attn_win_kernel.hpp"
#include "attn_bwd_kernel.hpp"
#include "swa1_fwd_kernel.hpp"
#include "swa1_bwd_kernel.hpp"
#include "flash_kernel.hpp"
#include "swa2_bwd_kernel.hpp"
#include "swat_kernel.hpp"
#include "swag_kernel.hpp"

int dlt_launch_fwd_32_32(const FwdArgs&, int, int, hipStream_t);
int dlt_launch_fwd_64_64(const FwdArgs&, int, int, hipStream_t);
int dlt_launch_win_32_32(const WinArgs&, int, int, hipStream_t);
int dlt_launch_win_64_64(const WinArgs&, int, int, hipStream_t);
int dlt_launch_win_64_128(const WinArgs&, int, int, hipStream_t);
int dlt_launch_win_128_128(const WinArgs&, int, int, hipStream_t);
int dlt_launch_fwd_128_128(const FwdArgs&, int, int, hipStream_t);
int dlt_launch_fwd_64_128(const FwdArgs&, int, int, hipStream_t);
int dlt_launch_fwd_256_256(const FwdArgs&, int, int, hipStream_t);

int dlt_launch_bwd_32_32(const BwdArgs&, int, const BwdArgs&, int, int, hipStream_t);
int dlt_launch_bwd_64_64(const BwdArgs&, int, const BwdArgs&, int, int, hipStream_t);
int dlt_launch_bwd_128_128(const BwdArgs&, int, const BwdArgs&, int, int, hipStream_t);
int dlt_launch_bwd_64_128(const BwdArgs&, int, const BwdArgs&, int, int, hipStream_t);
int dlt_launch_bwd_256_256(const BwdArgs&, int, const BwdArgs&, int, int, hipStream_t);

int dlt_flash_launch_fwd_32_32(const FlashArgs&, int, int, hipStream_t);
int dlt_flash_launch_fwdc_32_32(const FlashArgs&, int, int, hipStream_t);
int dlt_flash_launch_fwd_64_64(const FlashArgs&, int, int, hipStream_t);
int dlt_flash_launch_fwdc_64_64(const FlashArgs&, int, int, hipStream_t);
int dlt_flash_launch_fwd_128_128(const FlashArgs&, int, int, hipStream_t);
int dlt_flash_launch_fwdc_128_128(const FlashArgs&, int, int, hipStream_t);
int dlt_flash_launch_fwd_64_128(const FlashArgs&, int, int, hipStream_t);
int dlt_flash_launch_fwdc_64_128(const FlashArgs&, int, int, hipStream_t);
int dlt_flash_launch_bwd_q_32_32(const FlashBwdArgs&, int dtype, int grid, hipStream_t);
int dlt_flash_launch_bwd_kv_32_32(const FlashBwdArgs&, int dtype, int grid, hipStream_t);
int dlt_flash_launch_bwd_q_64_64(const FlashBwdArgs&, int dtype, int grid, hipStream_t);
int dlt_flash_launch_bwd_kv_64_64(const FlashBwdArgs&, int dtype, int grid, hipStream_t);
int dlt_flash_launch_bwd_q_128_128(const FlashBwdArgs&, int dtype, int grid, hipStream_t);
int dlt_flash_launch_bwd_kv_128_128(const FlashBwdArgs&, int dtype, int grid, hipStream_t);
int dlt_flash_launch_bwd_q_64_128(const FlashBwdArgs&, int dtype, int grid, hipStream_t);
int dlt_flash_launch_bwd_kv_64_128(const FlashBwdArgs&, int dtype, int grid, hipStream_t);
int dlt_flashs_fwd_32_32(const FlashArgs&, int dtype, int np, hipStream_t);
int dlt_flashs_bwd_q_32_32(const FlashBwdArgs&, int dtype, int np, hipStream_t);
int dlt_flashs_bwd_kv_32_32(const FlashBwdArgs&, int dtype, int np, hipStream_t);
int dlt_flashs_fwd_64_64(const FlashArgs&, int dtype, int np, hipStream_t);
int dlt_flashs_bwd_q_64_64(const FlashBwdArgs&, int dtype, int np, hipStream_t);
int dlt_flashs_bwd_kv_64_64(const FlashBwdArgs&, int dtype, int np, hipStream_t);
int dlt_flashs_fwd_64_128(const FlashArgs&, int dtype, int np, hipStream_t);
int dlt_flashs_bwd_q_64_128(const FlashBwdArgs&, int dtype, int np, hipStream_t);
int dlt_flashs_bwd_kv_64_128(const FlashBwdArgs&, int dtype, int np, hipStream_t);
int dlt_flashs_fwd_128_128(const FlashArgs&, int dtype, int np, hipStream_t);
int dlt_flashs_bwd_q_128_128(const FlashBwdArgs&, int dtype, int np, hipStream_t);
int dlt_flashs_bwd_kv_128_128(const FlashBwdArgs&, int dtype, int np, hipStream_t);
int dlt_flash_share_fwd(const FlashArgs&, int dtype, hipStream_t);
int dlt_flash_share_bwd_q(const FlashBwdArgs&, int dtype, hipStream_t);
int dlt_flash_share_bwd_kv(const FlashBwdArgs&, int dtype, hipStream_t);
int dlt_swag_launch_f32(const SwagArgs&, int nch, int ncg, int grid, hipStream_t);
int dlt_swag_launch_32_2(const SwagArgs&, int dtype, int ncg, bool bwd, int grid, hipStream_t);
int dlt_swag_launch_32_3(const SwagArgs&, int dtype, int ncg, bool bwd, int grid, hipStream_t);
int dlt_swag_launch_32_4(const SwagArgs&, int dtype, int ncg, bool bwd, int grid, hipStream_t);
int dlt_swag_launch_32_5(const SwagArgs&, int dtype, int ncg, bool bwd, int grid, hipStream_t);
int dlt_swag_launch_32_6(const SwagArgs&, int dtype, int ncg, bool bwd, int grid, hipStream_t);
int dlt_swag_launch_64_2(const SwagArgs&, int dtype, int ncg, bool bwd, int grid, hipStream_t);
int dlt_swag_launch_64_3(const SwagArgs&, int dtype, int ncg, bool bwd, int grid, hipStream_t);
int dlt_swag_launch_64_4(const SwagArgs&, int dtype, int ncg, bool bwd, int grid, hipStream_t);
int dlt_swat_launch_32(const SwatArgs&, int dtype, bool bwd, int grid, hipStream_t);
int dlt_swat_launch_64(const SwatArgs&, int dtype, bool bwd, int grid, hipStream_t);
int dlt_swat_launch_128(const SwatArgs&, int dtype, bool bwd, int grid, hipStream_t);
int dlt_launch_delta_32_32(const BwdArgs&, hipStream_t);
int dlt_launch_delta_64_64(const BwdArgs&, hipStream_t);
int dlt_launch_delta_128_128(const BwdArgs&, hipStream_t);
int dlt_launch_delta_64_128(const BwdArgs&, hipStream_t);
int dlt_launch_delta_256_256(const BwdArgs&, hipStream_t);
int dlt_swa1_launch_bwd_64(const Swa1BwdArgs&, int, int, int, int, hipStream_t);
int dlt_swa1_launch_bwd_128(const Swa1BwdArgs&, int, int, int, int, hipStream_t);
int dlt_swa1_launch_fwd_64(const Swa1FwdArgs&, int, int, hipStream_t);
int dlt_swa1_launch_fwd_128(const Swa1FwdArgs&, int, int, hipStream_t);
int dlt_swa2_launch_fwd_64(const Swa2FwdArgs&, int, int, hipStream_t);
int dlt_swa2_launch_bwd_64(const Swa2BwdArgs&, int, int, hipStream_t);
int dlt_swa2_launch_fwd_128(const Swa2FwdArgs&, int, int, hipStream_t);
int dlt_swa2_launch_bwd_128(const Swa2BwdArgs&, int, int, hipStream_t);

bool dlt_flash_async() {
  static const bool on = [] { const char* e = getenv("DLT_FLASH_SYNC_STAGING"); return !(e != nullptr && e[0] == '1'); }();
  return on;
}

namespace {

constexpr int LDS_TOTAL = 160 * 1024;

struct DimClass { int DK, DV, id; };

int pick_dims(const AttnProblem& p, DimClass& dc) {
  if (p.dk <= 32 && p.dv <= 32) dc = {32, 32, 3};  // the reference's demo and test head dims (src/tiled_swa.py:741, src/flash_attn.py:653)
  else if (p.dk <= 64 && p.dv <= 64) dc = {64, 64, 0};
  else if (p.dk <= 64 && p.dv <= 128) dc = {64, 128, 2};
  else if (p.dk <= 128 && p.dv <= 128) dc = {128, 128, 1};
  else if (p.dk <= 256 && p.dv <= 256) dc = {256, 256, 4};  // the largest head dim the reference admits (src/flash_attn.py:460-462): generic kernels only
  else return dlt_set_error(DLT_ERR_UNSUPPORTED, "head dims dk=%d dv=%d: at most 256 is supported", p.dk, p.dv);
  return DLT_OK;
}

int roundup(int v, int m) { return (v + m - 1) / m * m; }

// 16-byte vector access is possible when the last stride is 1 and every row start is aligned
bool vec_ok(const void* ptr, const int64_t* st, int nd, int d, int elem) {
  const int vb = 8 * elem;  // bytes of one 8-element chunk
  if (st[nd - 1] != 1 || d % 8 != 0) return false;
  if ((uintptr_t)ptr % (vb > 16 ? 16 : vb) != 0) return false;
  for (int i = 0; i < nd - 1; i++)
    if ((st[i] * elem) % 16 != 0) return false;
  return true;
}

// [B, H, N, D] tensor (entry 4 of the strides: pixel-row stride of an image-layout tensor, else 0)
bool tvec_ok(const void* ptr, const int64_t* st, int d, int elem) {
  return vec_ok(ptr, st, 4, d, elem) && (st[4] * elem) % 16 == 0;
}

// elements between the first and one past the last token of a (batch, head) slab
int64_t slab_span(const AttnProblem& p, const int64_t* st, int64_t ntok) {
  if (!p.tm.img) return ntok * st[2];
  return ((int64_t)p.g.TR * p.tm.bh - 1) * st[4] + ((int64_t)p.g.TC * p.tm.bw - 1) * st[2] + 1;
}

// chunking plan for a kernel whose halo buffers need `per_tok` bytes per staged token and
// whose own-tile region needs `own_bytes`
int make_plan(const AttnProblem& p, int own, int own_bytes, int per_tok, int XL_own, int XL_halo, AttnPlan& plan) {
  const DltGeom& g = p.g;
  plan.nblk_x = (XL_own + own - 1) / own;
  own_bytes = roundup(own_bytes, 16);
  const int budget2 = LDS_TOTAL / 2 - own_bytes;       // two workgroups per CU
  const int budget1 = LDS_TOTAL - own_bytes - 512;     // one workgroup per CU
  plan.rowfit = 0; plan.chunk_rows = 1; plan.chunk_x = 128;
  if (g.mode == DLT_GEOM_SWA) {
    const int whmax = dlt_imin(XL_halo, own + (2 * g.WC + 2) * g.S);
    const int cx = roundup(whmax + 32, 8);
    const int64_t row_bytes = (int64_t)cx * per_tok;
    const int nrows = 2 * g.WR + 1;
    if (row_bytes <= budget2) {
      plan.rowfit = 1; plan.chunk_x = cx; plan.chunk_rows = dlt_imin((int)(budget2 / row_bytes), nrows);
    } else if (row_bytes <= budget1) {
      plan.rowfit = 1; plan.chunk_x = cx; plan.chunk_rows = dlt_imin((int)(budget1 / row_bytes), nrows);
    }
  }
  if (!plan.rowfit) {
    int cx = 128;
    while (cx > 32 && (int64_t)cx * per_tok > budget2) cx -= 32;
    if ((int64_t)cx * per_tok > budget1) return dlt_set_error(DLT_ERR_UNSUPPORTED, "attention: LDS plan does not fit");
    plan.chunk_x = cx;
  }
  plan.off_a = own_bytes;
  plan.lds_bytes = own_bytes + plan.chunk_rows * plan.chunk_x * per_tok;
  return DLT_OK;
}

// ---- token-grid (b_size == 1) fast path ----------------------------------------------------
struct Swa1Class { int D, wclass, pbit, rope_mode; };
constexpr int SWA2_MAX_PASSES = 4;   // column passes of the streaming kernels: windows up to 93 columns

// Can the token-grid kernels take this problem?  They need 16-byte vector access to the
// streamed tensors, both head dims in one padded class, a window of at most 21 columns and,
// with rotation, rotary partners a power-of-two number of 8-dim chunks apart.
bool swa1_eligible(const AttnProblem& p, const bool* streamed_vec, int n_streamed, Swa1Class& c) {
  if (p.g.mode != DLT_GEOM_SWA || p.g.S != 1 || p.tm.img) return false;
  if (p.dtype != DLT_BF16 && p.dtype != DLT_FP16) return false;
  if (!(p.sm_scale > 0.f)) return false;  // the running max is kept on raw scores: needs a positive scale
  if (p.dk % 32 != 0 || p.dv % 32 != 0) return false;  // 64-byte staging pieces
  if (p.dk <= 64 && p.dv <= 64) c.D = 64;
  else if (p.dk <= 128 && p.dv <= 128 && p.dk > 64 && p.dv > 64) c.D = 128;
  else return false;
  for (int i = 0; i < n_streamed; i++)
    if (!streamed_vec[i]) return false;
  if ((int64_t)p.g.TR * p.g.TC >= ((int64_t)1 << 31) / 1024) return false;  // 32-bit element offsets inside a slab
  // column groups of a wave's window: up to 4 / 6 per class; wider windows (class 2) only run on the streaming kernels,
  // which walk them in column passes
  const int ncg = (4 + 2 * p.g.WC + 3) / 4;
  if (ncg > SWA2_MAX_PASSES * 6) return false;
  c.wclass = ncg <= 4 ? 0 : ncg <= 6 ? 1 : 2;
  c.pbit = 1;
  c.rope_mode = 0;
  if (p.rope.enabled && p.rope.R > 0) {
    const int r8 = p.rope.R / 8;
    if (p.rope.R % 8 != 0 || (r8 & (r8 - 1)) != 0 || 4 * p.rope.R > c.D) return false;
    if ((uintptr_t)p.rope.row_cs % 4 != 0) return false;
    c.pbit = r8;
    // balanced staging map: the rotation covers exactly half of a fully used head dim, so there
    // are as many rotary chunk pairs per token as staging threads
    c.rope_mode = (2 * r8 == c.D / 32 && p.dk == c.D && p.dv == c.D) ? 2 : 1;
    // plain staging map: a thread holds 4 neighbouring chunks of a token, so rotary partners must be 1 or 2
    // chunks apart; farther partners (R = 32: 4 chunks) sit in another thread's piece.  Tensors that arrive
    // rotated are staged without rotation and are not affected.
    if (c.rope_mode == 1 && r8 > 2 && !p.rope_prerot) return false;
  }
  return true;
}

// n_regions: [8 rows x HCW tokens] LDS regions the kernel keeps resident
void swa1_make_plan(const AttnProblem& p, const Swa1Class& c, int n_regions, int extra_bytes, Swa1Plan& plan, int cr = 8, bool kv = false) {
  plan.ncg = (4 + 2 * p.g.WC + 3) / 4;
  const int hcw = swa1_hcw(c.wclass == 0 ? 4 : 6);
  plan.HRP = roundup(4 + 2 * p.g.WR, cr);
  plan.nblk_r = (p.g.TR + 3) / 4;
  plan.nblk_c = (p.g.TC + 15) / 16;
  const int ncgmax = c.wclass == 0 ? 4 : 6;
  const bool wide = c.rope_mode == 0 || c.rope_mode == 3;  // must match WIDE in the kernels
  plan.lds_bytes = cr * hcw * (swa1_pitch(c.D, ncgmax, 0, wide, kv) + swa1_pitch(c.D, ncgmax, 1, wide, kv)) + extra_bytes;
  const int own_tile = 64 * (c.D * 2 + 16);  // output tile of the epilogue
  if (plan.lds_bytes < own_tile) plan.lds_bytes = own_tile;
}

// the token-grid kernels address the streamed tensors with 32-bit BYTE offsets inside a (batch, head) slab
bool swa1_strides_fit(const AttnProblem& p, const AttnTensors& t) {
  const int64_t ntok = (int64_t)p.g.TR * p.g.TC, lim = ((int64_t)1 << 31) - 1;
  const int64_t row = 2 * (int64_t)(p.dk > p.dv ? p.dk : p.dv);   // bytes of the last row
  auto fits = [&](const int64_t* st) { return st[2] >= 0 && (ntok - 1) * st[2] * 2 + row <= lim; };
  // lse2 / delta of the halo tokens are fetched with 32-bit element offsets (backward)
  const bool scalars_fit = t.ls[2] >= 0 && (ntok - 1) * t.ls[2] <= lim;
  return fits(t.qs) && fits(t.ks) && fits(t.vs) && (t.d_o == nullptr || (fits(t.dos) && scalars_fit));
}

int swa1_backward(const AttnProblem& p, const AttnTensors& t, const Swa1Class& c_in, hipStream_t stream) {
  if (dlt_route_note(DLT_FAMILY_TILE)) return DLT_OK;
  Swa1Class c = c_in;
  if (p.rope_prerot && c.rope_mode != 0) c.rope_mode = 3;  // rotated q, k: plain tile loads, gradients rotated back on store
  const int es = dlt_elem_size(p.dtype);
  // delta = rowsum(o * dO): folded into the dQ kernel when o can be read in 16-byte pieces like the
  // other operands, else the pre-pass kernel shared with the generic path
  const bool fuse_delta = tvec_ok(t.o, t.os, p.dv, es) && t.os[2] < ((int64_t)1 << 20);
  BwdArgs d;
  d.p = p;
  d.o = t.o; d.d_o = t.d_o; d.delta = t.delta;
  for (int i = 0; i < 5; i++) { d.os[i] = t.os[i]; d.dos[i] = t.dos[i]; }
  for (int i = 0; i < 3; i++) d.ls[i] = t.ls[i];
  d.o_vec = tvec_ok(t.o, t.os, p.dv, es);
  d.do_vec = tvec_ok(t.d_o, t.dos, p.dv, es);
  d.n_tokens_q = (int64_t)p.g.TR * p.g.XLq;
  if (!fuse_delta) {
    int rc = c.D == 64 ? dlt_launch_delta_64_64(d, stream) : dlt_launch_delta_128_128(d, stream);
    if (rc != DLT_OK) return rc;
  }

  Swa1BwdArgs a;
  a.p = p;
  // chunk heights of the two kernels may differ; the plan fields the kernels read (ncg, block
  // counts) do not depend on it
  Swa1Plan plan_q;
  swa1_make_plan(p, c, 2, 0, plan_q, SWA1_FWD_CR);
  const int hcw = swa1_hcw(c.wclass == 0 ? 4 : 6);
  swa1_make_plan(p, c, 2, 2 * SWA1_KV_CR * hcw * 4, a.plan, SWA1_KV_CR, true);
  const int lds_q = plan_q.lds_bytes, lds_kv = a.plan.lds_bytes;
  a.q = t.q; a.k = t.k; a.v = t.v; a.o = t.o; a.d_o = t.d_o; a.lse = t.lse; a.delta = t.delta;
  a.delta_out = t.delta;
  a.fuse_delta = fuse_delta ? 1 : 0;
  a.dq = t.dq; a.dk = t.dk; a.dv = t.dv;
  for (int i = 0; i < 4; i++) {
    a.qs[i] = t.qs[i]; a.ks[i] = t.ks[i]; a.vs[i] = t.vs[i]; a.os[i] = t.os[i]; a.dos[i] = t.dos[i];
    a.dqs[i] = t.dqs[i]; a.dks[i] = t.dks[i]; a.dvs[i] = t.dvs[i];
  }
  for (int i = 0; i < 3; i++) a.ls[i] = t.ls[i];
  a.q_vec = 1; a.k_vec = 1; a.v_vec = 1; a.do_vec = 1;
  a.dq_vec = tvec_ok(t.dq, t.dqs, p.dk, es);
  a.dk_vec = tvec_ok(t.dk, t.dks, p.dk, es);
  a.dv_vec = tvec_ok(t.dv, t.dvs, p.dv, es);
  a.rope_pbit = c.pbit;
  a.rope_mode = c.rope_mode;
  a.scale_log2 = p.sm_scale * 1.4426950408889634f;
  const int64_t grid = (int64_t)p.B * p.H * a.plan.nblk_r * a.plan.nblk_c;
  if (grid > 0x7fffffff) return dlt_set_error(DLT_ERR_UNSUPPORTED, "attention backward: grid too large");
  return c.D == 64 ? dlt_swa1_launch_bwd_64(a, c.wclass, (int)grid, lds_kv, lds_q, stream)
                   : dlt_swa1_launch_bwd_128(a, c.wclass, (int)grid, lds_kv, lds_q, stream);
}

int swa1_forward(const AttnProblem& p, const AttnTensors& t, const Swa1Class& c, hipStream_t stream) {
  if (dlt_route_note(DLT_FAMILY_TILE)) return DLT_OK;
  const int es = dlt_elem_size(p.dtype);
  Swa1FwdArgs a;
  a.p = p;
  swa1_make_plan(p, c, 2, 0, a.plan, SWA1_FWD_CR);
  a.q = t.q; a.k = t.k; a.v = t.v; a.o = t.out_o; a.lse = t.lse;
  for (int i = 0; i < 4; i++) { a.qs[i] = t.qs[i]; a.ks[i] = t.ks[i]; a.vs[i] = t.vs[i]; a.os[i] = t.os[i]; }
  for (int i = 0; i < 3; i++) a.ls[i] = t.ls[i];
  a.q_rot = c.rope_mode != 0 ? t.q_rot : nullptr;
  a.k_rot = c.rope_mode != 0 ? t.k_rot : nullptr;
  for (int i = 0; i < 4; i++) { a.qrs[i] = t.qrs[i]; a.krs[i] = t.krs[i]; }
  a.q_vec = tvec_ok(t.q, t.qs, p.dk, es);
  a.o_vec = tvec_ok(t.out_o, t.os, p.dv, es);
  a.rope_pbit = c.pbit;
  a.rope_mode = c.rope_mode;
  a.scale_log2 = p.sm_scale * 1.4426950408889634f;
  const int64_t grid = (int64_t)p.B * p.H * a.plan.nblk_r * a.plan.nblk_c;
  if (grid > 0x7fffffff) return dlt_set_error(DLT_ERR_UNSUPPORTED, "attention forward: grid too large");
  return c.D == 64 ? dlt_swa1_launch_fwd_64(a, c.wclass, (int)grid, stream)
                   : dlt_swa1_launch_fwd_128(a, c.wclass, (int)grid, stream);
}

// ---- streaming kernels: head dim 64 or 128 exactly, no rotation, windows up to 21 columns ---------------------------
bool swa2_eligible(const AttnProblem& p, const Swa1Class& c) {
  return (c.D == 64 || c.D == 128) && p.dk == c.D && p.dv == c.D && c.rope_mode == 0;
}
// token slots per grid row, and the largest column extent of a window in slots (tiles of S tokens: S WC + S - 1)
int swa2_slots(const AttnProblem& p) { return p.g.TC * p.g.S; }
int swa2_extent(const AttnProblem& p) { return p.g.S * p.g.WC + p.g.S - 1; }
// Kernel class (column groups of a wave's window per pass: 4 x 4 columns cover windows up to 13 columns, 6 x 4 up to 21)
// and number of column passes.  Wider windows take the split that computes the fewest groups (7 groups: 2 passes of 4,
// not 2 of 6), the larger class on a tie (fewer passes).
void swa2_split(const AttnProblem& p, int& ncg_class, int& npass) {
  const int ncg = (4 + 2 * swa2_extent(p) + 3) / 4;
  if (ncg <= 4) { ncg_class = 4; npass = 1; return; }
  const int n4 = (ncg + 3) / 4, n6 = (ncg + 5) / 6;
  if (4 * n4 < 6 * n6 && n4 <= SWA2_MAX_PASSES) { ncg_class = 4; npass = n4; }
  else { ncg_class = 6; npass = n6; }
}
int swa2_ncg(const AttnProblem& p) { int c, n; swa2_split(p, c, n); return c; }
// The problem without its rotation would run on the streaming kernels, and the two extra launches (q and k rotated out of place,
// dq and dk rotated back in place) cost less than the tile kernels' repeated rotation.  Measured step, tile kernels -> composed:
// d = 64, 8 slabs of 134 x 66, 19 x 19 window 153 -> 117 us, 2 of 20 x 20, 17 x 17 43 -> 39; d = 128, 8 of 60 x 66, 19 x 19 149 -> 109, 4
// of 33 x 40, 17 x 17 73 -> 58.  Narrow windows, of which the streaming kernels compute 16 columns, gain little or lose on small
// grids (d = 128, 2 of 20 x 20, 7 x 7 40 -> 37; 4 of 13 x 17, 5 x 5 29.7 -> 32.2; d = 64, 32 of 24 x 30, 21 x 5 40.9 -> 43.4): up to 7 columns,
// the tile kernels' place in the routing table, they are composed from 10^5 tokens on.
bool swa2_compose_ok(const AttnProblem& p, const Swa1Class& c) {
  return (c.D == 64 || c.D == 128) && p.dk == c.D && p.dv == c.D && (p.g.WC > 3 || (int64_t)p.B * p.H * p.g.TR * p.g.TC >= 131072);
}

// Time of a launch in rounds of one chunk, the last columns on 2^lpc patch columns (2: workgroups of 8 rows as everywhere): a workgroup takes its chunks
// and three more for its start and end, a CU one at a time in the backward pass and two in the forward pass; behind the mean load of the CUs, the longest one stands
// alone for part of its time (fitted to the shapes below).
float swa2_estimate(const AttnProblem& p, int lpc, bool backward) {
  const int64_t bh = (int64_t)p.B * p.H, blocks = (swa2_slots(p) + 15) / 16, full = bh * (lpc == 2 ? blocks : blocks - 1) * ((p.g.TR + 7) / 8);
  auto len = [&](int band) { return (float)((dlt_imin(p.g.TR, band + 2 * p.g.WR) + 3) / 4 + 3); };
  const int band = 32 >> lpc;
  const int64_t tall = lpc == 2 ? 0 : bh * ((p.g.TR + band - 1) / band), n = full + tall, cap = (backward ? 1 : 2) * (int64_t)dlt_device_cus();
  const float longest = tall ? len(band) : len(8), mean = ((float)full * len(8) + (float)tall * len(band)) / (float)cap;
  return n > cap ? mean + 0.35f * longest : fmaxf(mean, longest) + (backward ? 0.f : 0.14f * longest);
}
// log2 of the patch columns for the last `rest` slots of a row: 1, 0 (up to 4 slots), or 2, plain workgroups, unless the estimate falls by 7 % (less is lost as often as won)
int swa2_pick_tall(const AttnProblem& p, int rest, bool backward) {
  float best = 0.93f * swa2_estimate(p, 2, backward);
  int pick = 2;
  for (int lpc = rest <= 4 ? 0 : 1; lpc < 2; lpc++) {
    const float e = swa2_estimate(p, lpc, backward);
    if (e < best) { best = e; pick = lpc; }
  }
  return pick;
}

// returns the workgroups of 8 rows x 16 columns that the grids of all slabs take
int64_t swa2_make_plan(const AttnProblem& p, bool backward, bool may_tall, Swa2Plan& plan) {
  // Bands of four rows (the waves of the lower four only copy; the same bits) while those too have a CU each: a band's time is its halo's copies and
  // chunks, 4 + 2 WR rows instead of 8 + 2 WR.  Over 3508 shapes of up to 128 workgroups forward 0.81 ... 0.87 of the time, backward 0.76 ... 0.82
  // (d = 128, 4 slabs of 47 x 25, 15 x 5 window, forward 10.3 -> 8.5 us); from 129 on, where workgroups of 4 rows would queue, 0.9 ... 1.1 and 1.1 ... 1.3.
  const int64_t bands = (int64_t)p.B * p.H * ((p.g.TR + 7) / 8) * ((swa2_slots(p) + 15) / 16);
  const int band = 2 * bands <= dlt_device_cus() ? 4 : 8;
  plan.pairs = 0;
  { int c; swa2_split(p, c, plan.npass); }
  plan.S = p.g.S; plan.WCt = p.g.WC;
  dlt_fastdiv_make((uint32_t)p.g.S, plan.m_S, plan.s_S);
  plan.band = band;
  plan.nblk_r = (p.g.TR + band - 1) / band;
  plan.nblk_c = (swa2_slots(p) + 15) / 16;
  plan.ntall = 0; plan.lpc = 2;
  const int rest = swa2_slots(p) & 15;
  if (may_tall && rest >= 1 && rest <= 8 && bands > dlt_device_cus()) {
    // The last columns fill half a workgroup or less: 2 or 1 patch columns and bands of 16 or 32 rows (the same bits), where the estimate says that
    // it pays.  90 shapes of 257 ... 2300 bands, backward 0.945 of the time in the mean of all, 0.61 ... 1.016, taken for 34 of them (d = 128, 16
    // slabs of 71 x 17, 17 x 7 window 0.64; 64 of 99 x 18, 15 x 9 184 -> 139 us); forward at d = 128, taken for 10, 0.98 in the mean, 56 -> 49 there; at
    // d = 64, where more workgroups share a CU, under 0.01.  Up to one band per CU the longer workgroups take 1.1 to 1.6 times as long.
    const int pick = swa2_pick_tall(p, rest, backward);
    if (pick < 2) swa2_plan_tall(plan, p.g.TR, swa2_slots(p), pick);
  }
  dlt_fastdiv_make((uint32_t)swa2_groups(plan), plan.m_bh, plan.s_bh);
  dlt_fastdiv_make((uint32_t)dlt_imax(1, plan.nblk_c), plan.m_c, plan.s_c);
  dlt_fastdiv_make((uint32_t)p.H, plan.m_h, plan.s_h);
  return bands;
}

bool swa2_rows_ok(const AttnProblem& p, const void* ptr, const int64_t* st) {
  return tvec_ok(ptr, st, p.dk, 2) && st[2] >= 0 && ((int64_t)p.g.TR * swa2_slots(p) - 1) * st[2] * 2 + 2 * dlt_imax(p.dk, p.dv) <= (((int64_t)1 << 31) - 1);
}
bool swa2_scalars_ok(const AttnProblem& p, const AttnTensors& t) {
  return t.ls[2] >= 0 && ((int64_t)p.g.TR * swa2_slots(p) - 1) * t.ls[2] * 4 + 4 <= (((int64_t)1 << 31) - 1);
}

// Tiles of 2 ... 15 tokens (the regime of the reference's small-tile kernel, src/tiled_swa.py:15-133, b_size < 16 at
// :611): the streaming kernels on the grid of token slots, with the window of a token given by its tile
// (csrc/swa2_index.h).  Head dim 64 or 128 exactly (calls that ask for it: multiples of 8 below 64), 2-byte types, no rotation, plain token layout.
bool swa2_tiles_eligible(const AttnProblem& p, const AttnTensors& t, bool backward) {
  if (p.g.mode != DLT_GEOM_SWA || p.g.S < 2 || p.g.S > 15 || p.tm.img) return false;
  if (p.dtype != DLT_BF16 && p.dtype != DLT_FP16) return false;
  if (!(p.sm_scale > 0.f)) return false;
  if (!((p.dk == 64 || p.dk == 128) && p.dv == p.dk) && !(p.narrow && p.dk <= 64 && p.dv <= 64 && p.dv % 8 == 0)) return false;
  if (p.rope.enabled && p.rope.R > 0) return false;
  if ((4 + 2 * swa2_extent(p) + 3) / 4 > SWA2_MAX_PASSES * 6) return false;
  if ((int64_t)p.g.TR * swa2_slots(p) >= ((int64_t)1 << 31) / 1024) return false;
  if (!swa2_rows_ok(p, t.q, t.qs) || !swa2_rows_ok(p, t.k, t.ks) || !swa2_rows_ok(p, t.v, t.vs)) return false;
  if (!backward) return t.q_rot == nullptr && swa2_rows_ok(p, t.out_o, t.os);
  return swa2_rows_ok(p, t.o, t.os) && swa2_rows_ok(p, t.d_o, t.dos) && swa2_rows_ok(p, t.dq, t.dqs) && swa2_rows_ok(p, t.dk, t.dks) &&
         swa2_rows_ok(p, t.dv, t.dvs) && swa2_scalars_ok(p, t);
}

int swa2_forward(const AttnProblem& p, const AttnTensors& t, hipStream_t stream) {
  if (dlt_route_note(DLT_FAMILY_STREAMING)) return DLT_OK;
  Swa2FwdArgs a;
  a.p = p;
  // Two stacked patches per wave (4 waves per workgroup, two workgroups per CU) from more than one workgroup per CU on; below, a
  // CU has one workgroup either way and 8 waves of one patch each finish it sooner (64 workgroups 12.8 against 14.2 us, 224
  // 11.2 / 12.2, 352 26.8 / 25.8).
  // DLT_SWA2_SINGLE_PATCH=1 (read once per process) keeps the one-patch kernel for A/B timing and for its tests.
  static const bool single_patch = [] { const char* e = getenv("DLT_SWA2_SINGLE_PATCH"); return e != nullptr && e[0] == '1'; }();
  const int64_t bands = swa2_make_plan(p, false, p.dk == 128 && !single_patch, a.plan);   // tall workgroups: two patches per wave only
  a.plan.pairs = !single_patch && bands > dlt_device_cus();
  a.q = t.q; a.k = t.k; a.v = t.v; a.o = t.out_o; a.lse = t.lse;
  for (int i = 0; i < 4; i++) { a.qs[i] = t.qs[i]; a.ks[i] = t.ks[i]; a.vs[i] = t.vs[i]; a.os[i] = t.os[i]; }
  for (int i = 0; i < 3; i++) a.ls[i] = t.ls[i];
  a.scale_log2 = p.sm_scale * 1.4426950408889634f;
  const int64_t grid = (int64_t)p.B * p.H * swa2_groups(a.plan);
  if (grid > 0x7fffffff) return dlt_set_error(DLT_ERR_UNSUPPORTED, "attention forward: grid too large");
  return p.dk <= 64 ? dlt_swa2_launch_fwd_64(a, swa2_ncg(p), (int)grid, stream) : dlt_swa2_launch_fwd_128(a, swa2_ncg(p), (int)grid, stream);
}

int swa2_backward(const AttnProblem& p, const AttnTensors& t, hipStream_t stream) {
  if (dlt_route_note(DLT_FAMILY_STREAMING)) return DLT_OK;
  Swa2BwdArgs a;
  a.p = p;
  swa2_make_plan(p, true, true, a.plan);
  a.q = t.q; a.k = t.k; a.v = t.v; a.o = t.o; a.d_o = t.d_o; a.lse = t.lse; a.delta = t.delta;
  a.dq = t.dq; a.dk = t.dk; a.dv = t.dv;
  for (int i = 0; i < 4; i++) {
    a.qs[i] = t.qs[i]; a.ks[i] = t.ks[i]; a.vs[i] = t.vs[i]; a.os[i] = t.os[i]; a.dos[i] = t.dos[i];
    a.dqs[i] = t.dqs[i]; a.dks[i] = t.dks[i]; a.dvs[i] = t.dvs[i];
  }
  for (int i = 0; i < 3; i++) a.ls[i] = t.ls[i];
  a.scale_log2 = p.sm_scale * 1.4426950408889634f;
  const int64_t grid = (int64_t)p.B * p.H * swa2_groups(a.plan);
  if (grid > 0x7fffffff) return dlt_set_error(DLT_ERR_UNSUPPORTED, "attention backward: grid too large");
  return p.dk <= 64 ? dlt_swa2_launch_bwd_64(a, swa2_ncg(p), (int)grid, stream) : dlt_swa2_launch_bwd_128(a, swa2_ncg(p), (int)grid, stream);
}

// ---- marching token-grid kernels: head dim 32 (windows up to 21 x 21) or 64 (13 x 13) exactly, by window class ----------------------
int swag_class(int w) { return w <= 2 ? 2 : (4 + 2 * w + 3) / 4; }   // 4-wide blocks a patch's window spans
bool swag_rows_ok(const AttnProblem& p, const void* ptr, const int64_t* st) {
  return tvec_ok(ptr, st, p.dk, 2) && st[2] >= 0 && ((int64_t)p.g.TR * p.g.TC - 1) * st[2] * 2 + 2 * p.dk <= (((int64_t)1 << 31) - 1);
}
bool swag_eligible(const AttnProblem& p, const AttnTensors& t, const Swa1Class& c, bool bwd) {
  // rotation: 8 pairs per axis at head dim 64 in the forward pass, gradients turned back where q and k arrive rotated
  if (c.rope_mode != 0 && !(p.dk == 64 && p.rope.R == 8 && (!bwd || p.rope_prerot))) return false;
  if (p.dk != p.dv || (p.dk != 32 && p.dk != 64)) return false;
  const int wmax = p.dk == 32 ? 10 : 6;
  if (p.g.WR > wmax || p.g.WC > wmax) return false;
  if (!swag_rows_ok(p, t.q, t.qs) || !swag_rows_ok(p, t.k, t.ks) || !swag_rows_ok(p, t.v, t.vs)) return false;
  if (!bwd)
    return swag_rows_ok(p, t.out_o, t.os) && (t.q_rot == nullptr || (swag_rows_ok(p, t.q_rot, t.qrs) && swag_rows_ok(p, t.k_rot, t.krs)));
  return swag_rows_ok(p, t.o, t.os) && swag_rows_ok(p, t.d_o, t.dos) && swag_rows_ok(p, t.dq, t.dqs) && swag_rows_ok(p, t.dk, t.dks) &&
         swag_rows_ok(p, t.dv, t.dvs);
}

// fp32 tensors of head dim 32, forward pass: the marching kernel on hi + lo pairs.  Head dim 64 in fp32 belongs to the generic
// family in the routing table that callers of the C ABI rely on, and stays there.
bool swag_f32_eligible(const AttnProblem& p, const AttnTensors& t) {
  if (p.g.mode != DLT_GEOM_SWA || p.g.S != 1 || p.tm.img || p.dtype != DLT_FP32 || !(p.sm_scale > 0.f) || t.q_rot != nullptr) return false;
  if ((p.rope.enabled && p.rope.R > 0) || p.dk != p.dv || p.dk != 32) return false;
  if (p.g.WR > 6 || p.g.WC > 6) return false;
  const void* const ptrs[4] = {t.q, t.k, t.v, t.out_o};
  const int64_t* const st[4] = {t.qs, t.ks, t.vs, t.os};
  for (int i = 0; i < 4; i++)
    if (!tvec_ok(ptrs[i], st[i], p.dk, 4) || st[i][2] < 0 || ((int64_t)p.g.TR * p.g.TC - 1) * st[i][2] * 4 + 4 * p.dk > ((int64_t)1 << 31) - 1) return false;
  return true;
}

// fp32 windows on the kernel of attn_win_kernel.hpp: one token to a tile (larger ones keep the bits of the image layout, which the generic kernel
// serves), rows readable in 16-byte pieces, slabs of less than 2^31 bytes, no rotation, and one halo row
// at least fits the LDS; false: the generic kernel.  Generic -> this, us, over 97 shapes (1 ... 128 slabs, maps of 3 x 3 to 160 x 160, every head
// dim class) some 0.4 of the time in the mean: head dim 64, 9 x 7 columns: 2 slabs of 22 x 15 23.0 -> 7.5, 32 of 25 x 11 39.8 -> 9.9, 16 of
// 30 x 30 30.0 -> 14.6; 2 slabs of 3 x 128 at head dim 96 24 -> 14.  166 registers at 64/64 where one wave takes one part (176 with the sums of all
// cases in one kernel) let a third workgroup onto a CU where chunks are one wide row: 64 slabs of 27 x 127, 11 x 19 columns 212 -> 168, 16 of 96 x 96, 13 x 13 177 -> 138.
bool win_plan(const AttnProblem& p, const AttnTensors& t, const DimClass& dc, WinArgs& a, int& lds) {
  if (p.g.mode != DLT_GEOM_SWA || p.g.S != 1 || p.tm.img || p.dtype != DLT_FP32 || dc.id == 4 || t.q_rot != nullptr || (p.rope.enabled && p.rope.R > 0)) return false;
  const void* const ptrs[4] = {t.q, t.k, t.v, t.out_o};
  const int64_t* const st[4] = {t.qs, t.ks, t.vs, t.os};
  const int dims[4] = {p.dk, p.dk, p.dv, p.dv};
  const int64_t ntok = (int64_t)p.g.TR * p.g.XLq, lim = ((int64_t)1 << 31) - 1, bh = (int64_t)p.B * p.H;
  for (int i = 0; i < 4; i++)
    if (!tvec_ok(ptrs[i], st[i], dims[i], 4) || st[i][2] < 0 || (ntok - 1) * st[i][2] * 4 + 4 * dims[i] > lim) return false;
  if (t.ls[2] < 0 || (ntok - 1) * t.ls[2] > lim || bh > 1 << 23) return false;
  a.patch_shift = p.g.XLq <= 16 ? 0 : p.g.XLq <= 32 ? 1 : 2;
  const int cols = 16 << a.patch_shift;
  const int64_t nx = (p.g.XLq + cols - 1) / cols, cus = dlt_device_cus();
  auto grid = [&](int ws) { return bh * ((p.g.TR + (4 >> ws) - 1) / (4 >> ws)) * nx; };
  // Parts of a window where a row has at most 32 columns and wave slots are left: two, and four in 9 rows and more of up to 16 columns.  Against four for all of
  // those, 140 shapes of 2 ... 128 slabs take 0.98 of the time, with three rows up to 0.82 (16 slabs of 29 x 16, 3 x 9, 6.8 -> 5.8 us); few slabs with five rows and seven 1.03
  a.parts = a.patch_shift == 2 ? 1 : a.patch_shift == 0 && p.g.WR >= 4 ? 4 : 2;
  // They are dealt over as many waves as keeps one and a half workgroups per CU: against lines at two and three, 60 shapes of 8 ... 128 slabs
  // take 1.007 and 1.034 of the time.  Taking several parts costs the merges of their sums: 64 slabs of 25 x 11, 9 x 7, 10.6 -> 12.3 us
  a.wave_shift = a.patch_shift + (a.parts >> 1);
  while (a.wave_shift > a.patch_shift && 2 * grid(a.wave_shift) > 3 * cus) a.wave_shift--;
  if (((int64_t)p.g.TR + 3) / (4 >> a.wave_shift) > 65535 || nx > 65535) return false;
  const int nrows = dlt_imin(2 * p.g.WR + (4 >> a.wave_shift), p.g.TR);
  a.pair = p.g.XLq <= 16;
  a.cx = a.pair ? 16 : p.g.XLq <= 32 ? 32 : roundup(dlt_imin(p.g.XLk, cols + 2 * p.g.WC + 2) + 32, 8);
  auto bytes = [&](int rows) { return win_lds_bytes(dc.DK, dc.DV, rows, a.cx, a.pair != 0); };
  const int least = 1 + a.pair;   // rows of a chunk
  // chunks leave room for two workgroups per CU where so many run: one takes 1.1 times the time of two in the mean of those shapes, three 1.06 times
  int budget = grid(a.wave_shift) <= cus ? LDS_TOTAL : LDS_TOTAL / 2;
  if (bytes(least) > budget) budget = LDS_TOTAL;
  if (bytes(least) > budget) return false;
  a.chunk_rows = dlt_imax(least, nrows);
  while (bytes(a.chunk_rows) > budget) a.chunk_rows--;
  lds = bytes(a.chunk_rows);
  return true;
}

int win_forward(const AttnProblem& p, const AttnTensors& t, const DimClass& dc, WinArgs& a, int lds, hipStream_t stream) {
  a.q = (const float*)t.q; a.k = (const float*)t.k; a.v = (const float*)t.v; a.o = (float*)t.out_o; a.lse = t.lse;
  for (int i = 0; i < 2; i++) { a.qs[i] = t.qs[i]; a.ks[i] = t.ks[i]; a.vs[i] = t.vs[i]; a.os[i] = t.os[i]; a.ls[i] = t.ls[i]; }
  a.qn = (int32_t)t.qs[2]; a.kn = (int32_t)t.ks[2]; a.vn = (int32_t)t.vs[2]; a.on = (int32_t)t.os[2]; a.ln = (int32_t)t.ls[2];
  a.H = p.H; a.TR = p.g.TR; a.XL = p.g.XLq; a.WR = p.g.WR; a.WC = p.g.WC; a.dk = p.dk; a.dv = p.dv;
  a.scale_log2 = p.sm_scale * 1.4426950408889634f;
  switch (dc.id) {
    case 0: return dlt_launch_win_64_64(a, p.B * p.H, lds, stream);
    case 1: return dlt_launch_win_128_128(a, p.B * p.H, lds, stream);
    case 3: return dlt_launch_win_32_32(a, p.B * p.H, lds, stream);
    default: return dlt_launch_win_64_128(a, p.B * p.H, lds, stream);
  }
}

int swag_run(const AttnProblem& p, const AttnTensors& t, bool bwd, hipStream_t stream) {
  if (dlt_route_note(DLT_FAMILY_MARCHING)) return DLT_OK;
  SwagArgs a;
  a.q = t.q; a.k = t.k; a.v = t.v; a.o = t.o; a.d_o = t.d_o; a.out_o = t.out_o; a.dq = t.dq; a.dk = t.dk; a.dv = t.dv;
  a.lse = t.lse; a.delta = t.delta;
  for (int i = 0; i < 4; i++) {
    a.qs[i] = t.qs[i]; a.ks[i] = t.ks[i]; a.vs[i] = t.vs[i]; a.os[i] = t.os[i]; a.dos[i] = t.dos[i];
    a.dqs[i] = t.dqs[i]; a.dks[i] = t.dks[i]; a.dvs[i] = t.dvs[i];
  }
  for (int i = 0; i < 3; i++) a.ls[i] = t.ls[i];
  a.g = p.g; a.B = p.B; a.H = p.H;
  a.scale_log2 = p.sm_scale * 1.4426950408889634f;
  a.sm_scale = p.sm_scale;
  a.rope = p.rope;
  a.rope.enabled = p.rope.enabled && p.rope.R > 0;
  a.q_rot = t.q_rot; a.k_rot = t.k_rot;
  for (int i = 0; i < 4; i++) { a.qrs[i] = t.qrs[i]; a.krs[i] = t.krs[i]; }
  const int nch = swag_class(p.g.WR), ncg = swag_class(p.g.WC);
  constexpr int pc = SWAG_PC, step = 4 * (8 / pc);
  a.nstrips = (p.g.TC + 4 * pc - 1) / (4 * pc);
  // Rows per workgroup: a band's prologue fills the ring; one or two workgroups per CU are on the chip at once.
  const int nres = nch + 8 / pc - 1, tok = 4 * (4 * pc + 4 * (ncg - 1)), lds = nres * tok * (p.dtype == DLT_FP32 ? 6 * p.dk : 4 * p.dk + 8);
  const bool two = lds <= 80 * 1024 && (bwd || !a.rope.enabled);   // the rotating forward kernel's registers leave room for one
  const int64_t slots = (int64_t)dlt_device_cus() * (two ? 2 : 1);
  const int64_t cols = (int64_t)p.B * p.H * a.nstrips;
  dlt_band_plan((p.g.TR + step - 1) / step, cols, slots, a.band, a.nbands);
  a.band *= step;
  dlt_fastdiv_make((uint32_t)a.nstrips, a.m_s, a.s_s);
  dlt_fastdiv_make((uint32_t)a.nbands, a.m_b, a.s_b);
  dlt_fastdiv_make((uint32_t)p.H, a.m_h, a.s_h);
  const int64_t grid = cols * a.nbands;
  if (grid > 0x7fffffff) return dlt_set_error(DLT_ERR_UNSUPPORTED, "attention: grid too large");
  if (p.dtype == DLT_FP32) return dlt_swag_launch_f32(a, nch, ncg, (int)grid, stream);
  if (p.dk == 32) {
    switch (nch) {
      case 2: return dlt_swag_launch_32_2(a, p.dtype, ncg, bwd, (int)grid, stream);
      case 3: return dlt_swag_launch_32_3(a, p.dtype, ncg, bwd, (int)grid, stream);
      case 4: return dlt_swag_launch_32_4(a, p.dtype, ncg, bwd, (int)grid, stream);
      case 5: return dlt_swag_launch_32_5(a, p.dtype, ncg, bwd, (int)grid, stream);
      default: return dlt_swag_launch_32_6(a, p.dtype, ncg, bwd, (int)grid, stream);
    }
  }
  switch (nch) {
    case 2: return dlt_swag_launch_64_2(a, p.dtype, ncg, bwd, (int)grid, stream);
    case 3: return dlt_swag_launch_64_3(a, p.dtype, ncg, bwd, (int)grid, stream);
    default: return dlt_swag_launch_64_4(a, p.dtype, ncg, bwd, (int)grid, stream);
  }
}

// ---- flash fast path: dense, causal, and sliding windows over tiles of 16 k tokens -----------
// needs 2-byte elements, 16-byte vector access to q, k, v and 32-bit byte offsets inside a slab;
// tile mode takes no fused rotation (those calls use the generic kernels)
bool flash_eligible(const AttnProblem& p, const AttnTensors& t, bool with_do) {
  if (p.g.mode == DLT_GEOM_SWA) {
    if (p.g.S < 16 || p.g.S % 16 != 0) return false;
    if (p.rope.enabled && p.rope.R > 0) return false;
  }
  if (p.dtype != DLT_BF16 && p.dtype != DLT_FP16) return false;
  if (!(p.sm_scale > 0.f)) return false;  // the running max is kept on raw scores: needs a positive scale
  if (p.dk > 128 || p.dv > 128) return false;
  const int es = 2;
  if (!tvec_ok(t.q, t.qs, p.dk, es) || !tvec_ok(t.k, t.ks, p.dk, es) || !tvec_ok(t.v, t.vs, p.dv, es)) return false;
  if (with_do && !tvec_ok(t.d_o, t.dos, p.dv, es)) return false;
  const int64_t lim = ((int64_t)1 << 31) - 1;
  const int64_t nq = (int64_t)p.g.TR * p.g.XLq, nk = (int64_t)p.g.TR * p.g.XLk;  // tokens of one (batch, head)
  if (slab_span(p, t.ks, nk) * es > lim || slab_span(p, t.vs, nk) * es > lim) return false;
  if (slab_span(p, t.qs, nq) * es > lim) return false;
  if (with_do && slab_span(p, t.dos, nq) * es > lim) return false;
  return true;
}

// ---- marching tile-window kernels: tiles of 16 or 32 tokens, head dim 32 or 64 exactly, forward also 128 -----------------
// What they take beyond flash_eligible: windows whose rows fit the LDS ring (3 x 3 tiles; with 16-token tiles also 5 tile
// columns, 5 tile rows at head dim 32, 5 x 3 tiles at 64 and 5 x 5 there in the forward pass), and 16-byte rows with 32-bit offsets for every tensor.  Larger tiles stay on the
// flash kernels: a window row of 64-token tiles gives a 64-token chunk work for every wave, and its rows do not fit the ring.
bool swat_rows_ok(const AttnProblem& p, const void* ptr, const int64_t* st) {
  return tvec_ok(ptr, st, p.dk, 2) && st[2] >= 0 && st[4] >= 0 && slab_span(p, st, (int64_t)p.g.TR * p.g.XLq) * 2 <= ((int64_t)1 << 31) - 1;
}
bool swat_eligible(const AttnProblem& p, const AttnTensors& t, bool bwd) {
  if (p.g.mode != DLT_GEOM_SWA || (p.g.S != 16 && p.g.S != 32)) return false;
  if (p.dk != p.dv || (p.dk != 32 && p.dk != 64 && (p.dk != 128 || bwd))) return false;
  if (p.g.WR < 1 || p.g.WC < 1 || p.g.WR > 2 || p.g.WC > 2) return false;
  if (p.g.S == 32 && (p.g.WR != 1 || p.g.WC != 1)) return false;
  // Strips of four tiles, of which a ring of eight does not fit the LDS, against the flash kernels.  The lines follow from a slab's shape alone, so that its
  // bits do not depend on how many a call holds.
  // d = 64, five rows of three columns, 190 shapes of 1 ... 256 slabs: forward 0.28 ... 0.90 of the time of the chunked kernels, backward 0.38 ... 1.04 where two
  // strips hold seven columns or more (5 and 6 columns, whose second strip is mostly empty, up to 1.24 there and left to the others): 2 slabs of 30 x 30 tiles
  // 25.3 -> 10 and 52.4 -> 31 us, 64 of 21 x 33 206 -> 136 and 537 -> 445.  On up to 20 tiles or so the window's keys over a workgroup's waves
  // (flash_tiles_split) take 0.9 of the forward and 0.65 of the backward time (2 of 14 x 6, forward, 5.8 against 6.3).
  // The same with five columns, forward (the scalars of the backward pass do not fit beside the ring): 0.41 ... 0.98, 64 slabs of 21 x 33 225 -> 177, 4 of 40 x 12
  // 28.9 -> 11.2.
  // d = 128, 3 x 3 tiles, forward: 0.40 ... 0.98 where strips are three quarters full (2 slabs of 30 x 30 23.8 -> 13.4, 64 of 30 x 10 174 -> 106), five columns
  // up to 1.10; the backward kernels take 0.95 ... 1.5 of the time and stay there.
  if (p.dk == 128 && (p.g.S != 16 || p.g.WR != 1)) return false;
  if (p.dk == 128 || (p.g.WR == 2 && p.dk == 64)) {
    const int sb = Swat<64, 1, 1, 2>::SB, strips = (p.g.TC + sb - 1) / sb;
    if (p.g.WC == 2 && (p.dk == 128 || bwd)) return false;
    if (p.g.TC < sb || (p.dk == 128 && 4 * p.g.TC < 3 * sb * strips)) return false;
    if (bwd && strips == 2 && p.g.TC <= 6) return false;
  }
  if (!swat_rows_ok(p, t.q, t.qs) || !swat_rows_ok(p, t.k, t.ks) || !swat_rows_ok(p, t.v, t.vs)) return false;
  if (!bwd) return swat_rows_ok(p, t.out_o, t.os);
  return swat_rows_ok(p, t.o, t.os) && swat_rows_ok(p, t.d_o, t.dos) && swat_rows_ok(p, t.dq, t.dqs) && swat_rows_ok(p, t.dk, t.dks) &&
         swat_rows_ok(p, t.dv, t.dvs);
}

int swat_run(const AttnProblem& p, const AttnTensors& t, bool bwd, hipStream_t stream) {
  if (dlt_route_note(DLT_FAMILY_FLASH)) return DLT_OK;
  SwatArgs a;
  a.q = t.q; a.k = t.k; a.v = t.v; a.o = t.o; a.d_o = t.d_o; a.out_o = t.out_o; a.dq = t.dq; a.dk = t.dk; a.dv = t.dv;
  a.lse = t.lse; a.delta = t.delta;
  for (int i = 0; i < 5; i++) {
    a.qs[i] = t.qs[i]; a.ks[i] = t.ks[i]; a.vs[i] = t.vs[i]; a.os[i] = t.os[i]; a.dos[i] = t.dos[i];
    a.dqs[i] = t.dqs[i]; a.dks[i] = t.dks[i]; a.dvs[i] = t.dvs[i];
  }
  for (int i = 0; i < 3; i++) a.ls[i] = t.ls[i];
  a.tm = p.tm; a.g = p.g; a.B = p.B; a.H = p.H;
  a.scale_log2 = p.sm_scale * 1.4426950408889634f;
  a.sm_scale = p.sm_scale;
  const int64_t cus = dlt_device_cus(), slabs = (int64_t)p.B * p.H;
  a.one = bwd && dlt_tile_bwd_one_launch(p.dk, p.g.S, p.g.WR, p.g.WC, p.tm.img != 0, p.g.TC, slabs * p.g.TR, cus);
  const void* const ring_p[4] = {t.k, t.v, t.q, t.d_o};
  const int64_t* const ring_s[4] = {t.ks, t.vs, t.qs, t.dos};
  for (int i = 0; i < 4; i++) {
    a.ring_p[i] = ring_p[i];
    for (int j = 0; j < 5; j++) a.ring_s[i][j] = ring_s[i][j];
  }
  const int sb = a.one ? (p.dk == 32 ? Swab<32, 1, 1, 1>::SB : Swab<64, 1, 1, 1>::SB) : p.dk == 128 || (p.dk == 64 && p.g.WR == 2) ? Swat<64, 1, 1, 2>::SB : 8, strip = 16 * sb;
  a.nstrips = (p.g.XLq + strip - 1) / strip;
  const int64_t cols = slabs * a.nstrips;
  a.lone = !bwd && p.tm.img && dlt_image_fwd_alone(p.dk, p.g.S, p.g.WR, p.g.WC, p.g.TR, p.g.TC, p.H, cols, cus);
  // Rows per workgroup: a band's prologue fills the ring (the latency of its loads) and re-reads 2 WR rows.
  const int halo = sb + 2 * p.g.WC * (p.g.S / 16), ring = (2 * p.g.WR + 1) * halo * 64 * p.dk;
  const bool two = !a.one && !a.lone && ring + (2 * p.g.WR + 1) * halo * 128 <= 80 * 1024;   // workgroups per CU
  dlt_band_plan(p.g.TR, cols, two ? 2 * cus : cus, a.band, a.nbands);
  const int64_t grid = cols * a.nbands;
  if (grid > 0x7fffffff) return dlt_set_error(DLT_ERR_UNSUPPORTED, "attention: grid too large");
  if (p.dk == 128) return dlt_swat_launch_128(a, p.dtype, bwd, (int)grid, stream);
  return p.dk == 32 ? dlt_swat_launch_32(a, p.dtype, bwd, (int)grid, stream) : dlt_swat_launch_64(a, p.dtype, bwd, (int)grid, stream);
}

// Which kernels a dense / causal pass runs on:
//   CHUNKED: the streamed side passes through LDS chunk by chunk, 32 own tokens per wave (64 ... 256 per workgroup);
//   SLIM:    the same with 16 own tokens per wave: half the work per wave and chunk.  Forward 8 waves (twice the workgroups of 64/128 and
//            128/128) or 4 (flash_forward), backward 4 (twice the workgroups);
//   SPLIT1, SPLIT2: the streamed side is split over the waves of workgroups that own one or two blocks of 16 tokens
//            (csrc/flash_split_kernel.hpp).
// CHUNKED wins once its workgroups fill the chip.  Below that the time of a chunked pass is a start and the chunks of 64 streamed
// tokens one after the other, however few the workgroups; the split ones take
//     fixed + rounds over the CUs * (start and final sum of a workgroup + its 32-token blocks * time of a block on a CU).
// The constants of the split kernels (us) are least-squares fits to launches of 32 ... 8192 tokens on either side and 4 ... 128 heads, dense
// and causal.  Those of the chunked kernels were fitted the same way to two blocks per wave; in the backward passes they were then scaled, by
// class, to what decides best now that few workgroups run one block per wave (dlt_flash_bwd_64; 7900 shapes of up to 4000 tokens); of the
// scales of start and chunk within 0.3 % of the best, those with the fewest passes over 5 % slower than before (some 140 against 329 with one scale
// for both).  Gained by it, on the whole backward pass: by dQ at 128/128 1.046, at 64/128 1.022, at 64/64 1.020, by dK/dV 1.00 ... 1.02 (32 slabs of
// 300 x 300, 64/64, both 20.8 -> 15.4 us).  In the forward pass the same scaling gained 1 % in the mean
// and lost up to 40 % with few slabs (8 of 480 x 2581, 64/64, 16 -> 27 us): left.
//   77 queries x 1500 keys, 16 heads, 64/64: forward 22 -> 10 us, dQ 24 -> 11; 482 keys x 5450 queries, 4 heads: dK/dV 86 -> 26
//   16 heads, 2048 x 2048: forward 64/128 46 -> 34 us, 128/128 55 -> 41 (SLIM)
//
// A slab's results do not depend on how many slabs its call holds: the order of summation is chosen for the shape of a slab, as
// if the call held FLASH_SLABS of them, and only among kernels that give the same bits by the slabs it really holds.  Measured
// over 1364 shapes of 4 ... 128 slabs against a free choice (time of a pass, geometric mean): 32 slabs - 1 %, 16 + 1 %, 64 + 2 %, 8 + 7 %,
// 128 + 10 %, 4 + 14 % (1024 keys x 4096 queries, 4 heads, 64/128: dK/dV 35 -> 91 us, the chunked kernel).  FLASH_SLABS = 16 or 24
// costs less with few slabs, but 128 slabs then pay 27 or 15 %: at 32 the fewest passes are slower than on chunked kernels alone.
// Forward passes at 64/128 and 128/128 that do not split the keys: slim workgroups below 3072 queries, where they take 0.70 of the
// chunked time while they fit the chip at once and 0.75 ... 1.2 beyond; from there on chunked ones (4096 queries, 32 slabs: 1.1 ... 1.2).
enum { FLASH_CHUNKED = 0, FLASH_SPLIT1 = 1, FLASH_SPLIT2 = 2, FLASH_SLIM = 3 };
constexpr int FLASH_SLABS = 32, FLASH_SLIM_BELOW = 3072;
constexpr unsigned FLASH_ALL = 15u;   // bit per kind
struct FlashCost { int own; float start, chunk, slim_start, slim_chunk, fixed1, wg1, block1, fixed2, wg2, block2; };   // own: tokens of a chunked workgroup
int flash_fastest(int pass, const DimClass& dc, int dims, int64_t bh, int own, int other, bool causal, unsigned kinds) {
  constexpr float NONE = 1e9f;
  static const FlashCost COST[3][4] = {   // by pass (forward, dQ, dK/dV) and DimClass::id
      {{128, 3.50f, .822f, 2.60f, .730f, 2.31f, 1.36f, .137f, 1.09f, 3.79f, .141f},    // 64/64
       {256, 6.78f, 1.493f, 2.40f, 1.125f, .59f, 3.70f, .272f, 0.f, 5.81f, .322f},     // 128/128
       {256, 6.06f, 1.272f, 2.40f, .960f, 1.53f, 2.57f, .174f, 0.f, 5.73f, .185f},     // 64/128
       {128, 2.94f, .698f, NONE, NONE, 2.84f, .52f, .055f, 2.41f, 1.13f, .094f}},      // 32/32
      {{128, 3.48f, .748f, NONE, NONE, 2.07f, 2.19f, .138f, .43f, 5.72f, .144f},
       {128, 2.63f, 1.236f, NONE, NONE, .67f, 4.25f, .289f, NONE, NONE, NONE},
       {128, 3.04f, .773f, NONE, NONE, .99f, 4.27f, .244f, NONE, NONE, NONE},
       {128, 4.44f, .825f, NONE, NONE, 2.73f, .68f, .057f, 2.36f, 1.44f, .090f}},
      {{128, 4.35f, .953f, NONE, NONE, 1.85f, 2.73f, .134f, 1.36f, 4.59f, .171f},
       {64, 4.95f, 1.275f, NONE, NONE, 1.31f, 4.42f, .283f, NONE, NONE, NONE},
       {128, 5.79f, 1.627f, NONE, NONE, 1.32f, 4.15f, .185f, NONE, NONE, NONE},
       {128, 4.28f, 1.038f, NONE, NONE, 2.51f, 1.14f, .072f, 2.79f, 1.38f, .114f}}};
  FlashCost c = COST[pass][dc.id];
  if (pass > 0 && dc.id == 1 && dims <= 192) {   // the split kernels leave out missing pieces of a row, of the chunked ones' work more stays (flashd_dims)
    // dQ: scaled for other sides of more than seven chunks only, dK/dV not at all: scaled, 80/80 was split where chunked workgroups take 0.64 of the time on 64
    // slabs and more and as long on fewer (272 x 272 causal, 324 keys of 1710 queries)
    const bool scaled = pass == 1 && other > 448;
    c.start = pass == 2 ? 5.62f : scaled ? 7.58f : 6.58f;
    c.chunk = pass == 2 ? 1.226f : scaled ? 1.26f : 1.404f;
  }
  const float cus = (float)dlt_device_cus();
  const auto wgs = [&](int n) { return (float)(bh * ((own + n - 1) / n)); };
  const auto may = [&](int kind) { return (kinds >> kind & 1u) != 0; };
  const float chunks = (float)((other + 63) / 64);
  int best = -1;
  float least = 0.f;
  const auto consider = [&](int kind, float t) {
    if (may(kind) && (best < 0 || t < least)) { least = t; best = kind; }
  };
  // backward: split or not; which of the others runs is dlt_flash_bwd_64's choice (dK/dV at 64/128 under a mask: 0.65 on one block per wave)
  const float whole = c.start + (pass == 2 && causal && dc.id == 2 ? 0.65f : 1.f) * c.chunk * chunks;
  consider(FLASH_CHUNKED, whole);
  if (pass > 0) {
    if (wgs(128) > cus && may(FLASH_CHUNKED)) return FLASH_CHUNKED;
  } else if (wgs(128) > cus) {
    // A CU has more than one slim workgroup.  Up to two of them run side by side, which still beats the chunked workgroups
    // at 64/64 and where a mask makes the work uneven (32 heads, 2048 x 2048, causal: 64/128 52 -> 46 us, 128/128 60 -> 49)
    if (c.slim_chunk < NONE && (causal || dc.id == 0)) {
      const int kind = wgs(128) <= 2.f * cus ? FLASH_SLIM : FLASH_CHUNKED;
      if (may(kind)) return kind;
    }
    if (wgs(c.own) > cus && may(FLASH_CHUNKED)) return FLASH_CHUNKED;
  } else {
    consider(FLASH_SLIM, c.slim_start + c.slim_chunk * chunks);
  }
  // the pieces of a row that a head dim below its class does not have are not read
  const float blocks = (float)((other + 31) / 32) * ((float)dims / (float)(dc.DK + dc.DV));
  for (int np = 1; np <= 2; np++) {
    float rounds = wgs(16 * np) / cus;
    if (dc.DK + dc.DV > 128) rounds = 0.5f * (rounds + ceilf(rounds));   // one workgroup per CU: a started round is half a round
    // under a causal mask the workgroups of several rounds see about half of the other side
    const float seen = causal && rounds > 1.f ? 0.55f * blocks : blocks;
    consider(np == 1 ? FLASH_SPLIT1 : FLASH_SPLIT2,
             (np == 1 ? c.fixed1 : c.fixed2) + (rounds > 1.f ? rounds : 1.f) * (np == 1 ? c.wg1 + c.block1 * seen : c.wg2 + c.block2 * seen));
  }
  return best < 0 ? FLASH_SLIM : best;   // SLIM alone, beyond one workgroup per CU
}
// Kinds that give a slab the same bits as `kind`: one and two own blocks per split workgroup; slim and chunked workgroups where both
// pass 64 tokens at a time (the chunked forward kernels at 64/128 and 128/128 pass 128: other reference maxima of the softmax).
// Asked about backward passes only where they are split.
unsigned flash_same_bits(int pass, const DimClass& dc, int kind) {
  if (kind == FLASH_SPLIT1 || kind == FLASH_SPLIT2) return 1u << FLASH_SPLIT1 | 1u << FLASH_SPLIT2;
  if (pass == 0 && (dc.id == 1 || dc.id == 2)) return 1u << kind;
  return 1u << FLASH_CHUNKED | 1u << FLASH_SLIM;
}
int flash_pick(int pass, const DimClass& dc, int dims, int64_t bh, int own, int other, bool causal) {
  int order = flash_fastest(pass, dc, dims, FLASH_SLABS, own, other, causal, FLASH_ALL);
  if (pass == 0 && (dc.id == 1 || dc.id == 2) && order != FLASH_SPLIT1 && order != FLASH_SPLIT2) order = own < FLASH_SLIM_BELOW ? FLASH_SLIM : FLASH_CHUNKED;
  if (pass > 0 && order != FLASH_SPLIT1 && order != FLASH_SPLIT2)
    return dlt_flash_bwd_64(causal, pass == 2 && dc.id == 2, own, bh * ((own + 63) / 64), dlt_device_cus()) ? FLASH_SLIM : FLASH_CHUNKED;
  return flash_fastest(pass, dc, dims, bh, own, other, causal, flash_same_bits(pass, dc, order));
}

// How a dense / causal pass runs: the kind, and over how many workgroups the other side of an own block is split (n; len: FlashShare).
//
// A dense pass with few own tokens and many others leaves most CUs idle, or has each of its small workgroups read all of the other side
// (16 slabs, forward: 64 queries x 4000 keys at 64/64 ran on 64 CUs).  Its other side is cut into n shares of chunked workgroups instead; their
// fp32 partial results are summed by a second launch, which costs some 3 us and 8 bytes per own element and share.  n follows from a
// slab's shape alone (see above), as other / (a + b own) up to 8: the lines were fitted to 2100 shapes of 4 ... 128 slabs (n = 2, 3, 4, 6, 8), a loss
// counted eightfold.  Inside them, not split -> split, geometric mean of the pass by slabs (4, 8, 16, 32, 64, 128): forward 1.7 ... 2.2,
// 1.55 ... 2.0, 1.33 ... 1.8, 1.22 ... 1.6, 1.2, 1.15; both backward passes together 1.4 ... 1.8 down to 1.05 ... 1.3.  Shorter other sides and
// longer own ones lose more to the sums than idle CUs cost (128 slabs of 734 x 3321, 64/64: 98 -> 144 us with n = 4).  The slowest against no
// shares: forward 1.26 on 128 slabs (53 x 3868, 64/128: 33 -> 42 us; one share of a handful of tokens is half a workgroup), backward 1.14 (30 x 1149, 128/128).
//
// Once workgroups fill the chip without it, partial results only cost: one workgroup then takes all shares of its own block (FlashShare::walk, the same
// bits), from 1.5 workgroups of 64 own tokens per CU on, 0.75 where they are all there are.  Over 110 shapes of 4 ... 256 slabs, walked against split
// in the mean below and above that line: up to 64 own tokens forward 1.27 and 0.9, dQ 1.04 and 0.89, dK/dV 1.08 and 0.87; more own tokens 1.03 and 0.93,
// 0.99 and 0.95, 0.95 and 0.9.  Long own sides of forward and dQ stay split (128/128 forward beyond 512 queries 1.03, dQ 1.04): their shares are few and
// long.  All of those shapes against no shares, forward and backward, split alone -> so: 128 slabs 1.01 and 1.00 -> 0.99 and 0.96, 256 slabs 1.01 and 1.01 -> 0.96
// and 0.93; the slowest of 256 slabs 1.30 -> 1.14 (995 x 5280, 128/128).  A pass whose partial results would take more than half of
// DLT_FLASH_WORKSPACE_MAX is walked as well, whatever its sides (128 MiB; at 64 MiB 32 slabs of 8943 x 294, 128/128, were, backward 211 -> 252 us).
constexpr int64_t FLASH_PART_MAX = (int64_t)DLT_FLASH_WORKSPACE_MAX / 4;   // floats
struct FlashShares { int n, len; bool walk; };
FlashShares flash_shares(int pass, const DimClass& dc, int dk, int dv, int64_t bh, int own, int other) {
  // other side of at least `least` tokens and `times` the own one; a, 4 b
  static const struct { int least, times, a, b4; } RULE[3][4] = {   // by pass; 64/64, 64/128, 128/128 with up to 192 dims in all, 128/128
      {{3000, 3, 150, 6}, {3000, 3, 500, 5}, {2500, 3, 150, 6}, {1200, 3, 150, 9}},
      {{1600, 1, 350, 4}, {600, 1, 150, 4}, {1600, 1, 150, 4}, {600, 4, 150, 8}},
      {{2500, 1, 150, 6}, {1600, 4, 250, 4}, {2000, 1, 500, 4}, {1200, 4, 150, 8}}};
  const auto& r = RULE[pass][dc.id == 0 ? 0 : dc.id == 2 ? 1 : dk + dv <= 192 ? 2 : 3];
  if (other < r.least || other < (int64_t)r.times * own) return {1, other, false};
  int n = dlt_imin((int)(4 * (int64_t)other / (4 * r.a + (int64_t)r.b4 * own)), FLASH_SHARES_MAX);
  if (n <= 1) return {1, other, false};
  const int len = roundup((other + n - 1) / n, 128);
  n = (other + len - 1) / len;
  const int64_t row = pass == 0 ? dv + 2 : pass == 1 ? dk : dk + dv;
  const int most = pass == 2 ? 1 << 30 : (pass == 0 ? dk + dv <= 192 : dc.id != 1) ? 1024 : 512;
  const bool full = own <= most && 4 * bh * ((own + 63) / 64) >= (own <= 64 ? 3 : 6) * (int64_t)dlt_device_cus();
  const bool walk = full || bh * n * own * row > FLASH_PART_MAX / 2;
  return {n, len, walk};
}

struct FlashPlan { int kind, n, len; bool walk; };
FlashPlan flash_plan(int pass, const DimClass& dc, int dk, int dv, int64_t bh, int own, int other, bool causal, bool may_split) {
  if (may_split && !causal) {
    const FlashShares s = flash_shares(pass, dc, dk, dv, bh, own, other);
    // one own block per wave or two (the same bits): one while its workgroups are few.  Forward at 64/64, 8 waves of one against 4 of two: 0.92 of the
    // time below a workgroup of 128 queries per four CUs, 0.96 up to one per CU, 1.01 to two, 1.05 beyond; at 64/128 and 128/128 always
    // 8 waves (their two-block kernel passes 128 keys at a time).  Backward, whole pass, one against two: 0.82 ... 0.89 below 64 workgroups of
    // 64, 0.87 ... 0.96 to one per CU, 0.97 ... 1.0 to two, 0.95 ... 1.09 beyond; up to 64 own tokens always, which the others' waves would idle beside
    // (and forward on 4 waves: 47 shapes of 128 and 256 slabs forward 0.98 of the time, backward 0.97)
    const int64_t cus = dlt_device_cus();
    const bool slim = own <= 64 || (pass == 0 ? dc.id != 0 || bh * s.n * ((own + 127) / 128) <= cus : bh * s.n * ((own + 63) / 64) <= 2 * cus);
    if (s.n > 1) return {slim ? FLASH_SLIM : FLASH_CHUNKED, s.n, s.len, s.walk};
  }
  return {flash_pick(pass, dc, dk + dv, bh, own, other, causal), 1, other, false};
}
// the asynchronously staged kernels know shares
// (partial rows are counted in 32 bits: beyond that nothing is split)
bool flash_may_split(const AttnProblem& p, const DimClass& dc) {
  const int64_t rows = (int64_t)p.B * p.H * dlt_imax(p.g.XLq, p.g.XLk);
  return p.g.mode == DLT_GEOM_DENSE && dc.id <= 2 && p.dtype != DLT_FP32 && p.dk % 8 == 0 && p.dv % 8 == 0 && rows <= 0x7fffffff / 16 && dlt_flash_async();
}
// floats of partial results that a pass leaves for a second launch
int64_t flash_part_fwd(const AttnProblem& p, int n, bool walk) { return n > 1 && !walk ? (int64_t)p.B * p.H * n * p.g.XLq * (p.dv + 2) : 0; }
int64_t flash_part_q(const AttnProblem& p, int n, bool walk) { return n > 1 && !walk ? (int64_t)p.B * p.H * n * p.g.XLq * p.dk : 0; }
int64_t flash_part_kv(const AttnProblem& p, int n, bool walk) { return n > 1 && !walk ? (int64_t)p.B * p.H * n * p.g.XLk * (p.dk + p.dv) : 0; }

// Windows over tiles of 16 k tokens off the marching kernels: whether the kernels of flash_split_kernel.hpp run, which take 16 own tokens to a
// workgroup and deal the window's keys over its waves, so that a call of few tiles is not a handful of workgroups with 64 keys after the other.
// This is the one choice for tiles that looks at the number of slabs, and with it their bits depend on it: by the shape alone it would cost calls of
// one to eight slabs up to 4 times, or calls of 64 and more up to 3 times the time (130 shapes; the split kernels take 0.45 of the chunked time on one slab, 1.8 on 32).
// Tiles of 64 k tokens stay on the asynchronously staged kernels (0.67 ... 1.1 of whose time it takes up to 256 blocks), where a slab's bits do not
// depend on the call.  A workgroup's time is a0 + a1 + a2 per key, one per CU and a3 of them at once, that of the chunked kernels
// b0 + b1 + b2 per 64 keys, b3 workgroups per CU at once; fitted to 1717 shapes (us), rms 7 and 13 %, so 15 % are asked for.  Chosen that way a forward pass takes
// 0.59 (d = 32), 0.73 and 0.80 (128) of the chunked time in the mean of shapes of 9 ... 60000 tiles, a backward pass 0.63, 0.74, 0.94, none over 1.10:
// windows of 5 x 3 tiles of 16, d = 64, 8 slabs of 7 x 6 forward 17.5 -> 7.6 us and backward 32.7 -> 17.1, 2 slabs of 6 x 11 forward 22.9 -> 6.2.
bool flash_tiles_split(const AttnProblem& p, const DimClass& dc, bool backward) {
  const DltGeom& g = p.g;
  if (g.mode != DLT_GEOM_SWA || g.S % 64 == 0) return false;
  const int64_t cus = dlt_device_cus(), bh = (int64_t)p.B * p.H, blocks = bh * g.TR * (g.XLk / 16);
  if (blocks > 0x7fffffff || (int64_t)g.TR * g.XLk > 0x7fffffff) return false;
  static const struct { float a0, a1, a2, a3, b0, b1, b2, b3; } COST[3][2] = {   // d = 32, 64, 128; forward, backward
    {{4.9f, .52f, .00068f, .54f, 4.8f, .52f, 1.1f, 2.2f}, {7.9f, 1.4f, .0019f, .60f, 7.9f, 2.8f, 1.9f, 2.2f}},
    {{4.7f, 1.2f, .0027f, .79f, 3.5f, 1.8f, 1.3f, 1.8f}, {7.4f, 3.3f, .0051f, .65f, 4.0f, 6.5f, 2.7f, 1.6f}},
    {{4.0f, 2.9f, .0056f, .69f, 2.8f, 3.9f, 1.8f, 1.4f}, {7.5f, 8.4f, .0100f, .66f, 6.5f, 7.0f, 2.1f, 1.3f}}};
  const auto& c = COST[dc.id == 3 ? 0 : dc.id == 0 ? 1 : 2][backward];
  const int rows = dlt_imin(g.TR, 2 * g.WR + 1), own = 64 * (backward ? flash_np_q(dc.DK, dc.DV) : FLASH_NP);
  const int64_t cols = own + 2 * (int64_t)g.WC * g.S + (own % g.S ? g.S : 0), wgs = bh * g.TR * ((g.XLk + own - 1) / own);
  const float keys = (float)rows * dlt_imin(g.TC, 2 * g.WC + 1) * g.S, chunks = (float)rows * (((cols < g.XLk ? cols : g.XLk) + 63) / 64);
  const float split = c.a0 + fmaxf(1.f, blocks / (c.a3 * cus)) * (c.a1 + c.a2 * keys), chunked = c.b0 + fmaxf(1.f, wgs / (c.b3 * cus)) * (c.b1 + c.b2 * chunks);
  return split < .85f * chunked;
}

int flash_forward(const AttnProblem& p, const AttnTensors& t, const DimClass& dc, hipStream_t stream) {
  if (dlt_route_note(DLT_FAMILY_FLASH)) return DLT_OK;
  FlashArgs a;
  a.q = t.q; a.k = t.k; a.v = t.v; a.o = t.out_o; a.lse = t.lse;
  for (int i = 0; i < 5; i++) { a.qs[i] = t.qs[i]; a.ks[i] = t.ks[i]; a.vs[i] = t.vs[i]; a.os[i] = t.os[i]; }
  for (int i = 0; i < 3; i++) a.ls[i] = t.ls[i];
  a.tm = p.tm;
  a.B = p.B; a.H = p.H; a.Lq = p.g.XLq; a.Lk = p.g.XLk; a.dk = p.dk; a.dv = p.dv;
  const int own = 64 * FLASH_NP;
  a.nblk = (a.Lq + own - 1) / own;
  a.causal = p.g.mode == DLT_GEOM_CAUSAL;
  a.causal_group = flash_causal_group(a.Lk, p.dk, p.dv);
  a.slim = 0; a.chunk = 64;
  a.tile = p.g.mode == DLT_GEOM_SWA;
  a.g = p.g;
  a.o_vec = tvec_ok(t.out_o, t.os, p.dv, 2);
  const int chunk = flash_ck_fwd(dc.DK, dc.DV) * (dc.DK * 2 + FLASH_PAD + dc.DV * 2 + FLASH_PAD), tile = own * (dc.DV * 2 + 16);
  a.lds_bytes = chunk > tile ? chunk : tile;
  a.scale_log2 = p.sm_scale * 1.4426950408889634f;
  const int64_t grid = (int64_t)p.B * p.H * p.g.TR * a.nblk;
  if (grid > 0x7fffffff) return dlt_set_error(DLT_ERR_UNSUPPORTED, "flash forward: grid too large");
  a.share = {t.part, 1, a.Lk, 0};
  int np = FLASH_CHUNKED;
  if (p.g.mode != DLT_GEOM_SWA) {
    const FlashPlan f = flash_plan(0, dc, p.dk, p.dv, (int64_t)p.B * p.H, a.Lq, a.Lk, a.causal != 0, t.shares && flash_may_split(p, dc));
    np = f.kind;
    // One own block per wave, with the bits of the kernel it stands for: 8 waves (workgroups of 128 queries) or, while workgroups of 64 all
    // run at once, one per CU (two under a mask, where the work is uneven), 4 waves.  Slim workgroups, 8 waves -> 4: 0.83 ... 0.89 of
    // the time up to one per CU (head dims of 80: 0.92 ... 0.96), under a mask 0.80 ... 0.88 and 0.83 ... 0.96 up to two; beyond 1.0 and
    // more.  Chunked ones of 64/128 and 128/128 (from 3072 queries on; two blocks on 8 waves): 4 waves 0.53 ... 0.64 up to one workgroup of 64 per
    // CU, then 8 waves 0.65 ... 0.76 up to one of 128, under a mask 0.62 ... 0.70 and 0.66 ... 0.85 up to two (4 slabs of 7232, causal,
    // 64/128: 151 -> 78 us)
    const int64_t cus = dlt_device_cus(), nbh = (int64_t)p.B * p.H * f.n, most = a.causal ? 2 * cus : cus;
    const bool long_chunks = np == FLASH_CHUNKED && dc.DV == 128;
    const bool four = (f.n > 1 && a.Lq <= 64) || nbh * ((a.Lq + 63) / 64) <= (long_chunks ? cus : most);
    a.chunk = long_chunks ? 128 : 64;
    a.slim = np == FLASH_SLIM ? (four ? 4 : 8) : long_chunks ? (four ? 4 : nbh * ((a.Lq + 127) / 128) <= most ? 8 : 0) : 0;
    a.share.n = f.n; a.share.len = f.len; a.share.walk = f.walk;
  }
  if (flash_tiles_split(p, dc, false)) {
    np = FLASH_SPLIT1;
    a.Lq = a.Lk = p.g.TR * p.g.XLq;
  }
  const bool split = np == FLASH_SPLIT1 || np == FLASH_SPLIT2;
  // Dense split calls with one block of 16: as many workgroups to a block as leave one per CU (bits are equal, so the line may look at the real
  // count).  Over 18096 shapes of 1 ... 16 slabs two take 0.94 ... 0.96 of one's time at 64/64, 0.89 ... 0.92 at 64/128 and 0.94 ... 0.97 at
  // 128/128, four another 0.94 ... 0.98 of two's there (77 x 1500, 16 slabs, 64/64: 11.5 -> 10.8 us); with more workgroups than CUs either takes
  // 1.17 ... 1.3, and under a mask, where the longest row decides, 0.99 ... 1.01.
  a.part_dv = dc.DV;
  if (np == FLASH_SPLIT1 && !a.causal && !a.tile)
    for (int w = dc.DV / 2; w >= 32 && 4 * w >= dc.DV; w /= 2)
      if ((int64_t)p.B * p.H * ((a.Lq + 15) / 16) * ((a.dv + w - 1) / w) <= dlt_device_cus()) a.part_dv = w;
  int rc;
#define DLT_FLASH_FWD(C) \
  rc = split ? dlt_flashs_fwd_##C(a, p.dtype, np, stream) : a.causal ? dlt_flash_launch_fwdc_##C(a, p.dtype, (int)grid, stream) : dlt_flash_launch_fwd_##C(a, p.dtype, (int)grid, stream); \
  break
  switch (dc.id) {
    case 0: DLT_FLASH_FWD(64_64);
    case 1: DLT_FLASH_FWD(128_128);
    case 3: DLT_FLASH_FWD(32_32);
    default: DLT_FLASH_FWD(64_128);
  }
#undef DLT_FLASH_FWD
  return rc == DLT_OK && a.share.n > 1 && !a.share.walk ? dlt_flash_share_fwd(a, p.dtype, stream) : rc;
}

int flash_backward(const AttnProblem& p, const AttnTensors& t, const DimClass& dc, hipStream_t stream) {
  if (dlt_route_note(DLT_FAMILY_FLASH)) return DLT_OK;
  BwdArgs d;
  d.p = p;
  d.o = t.o; d.d_o = t.d_o; d.delta = t.delta;
  for (int i = 0; i < 5; i++) { d.os[i] = t.os[i]; d.dos[i] = t.dos[i]; }
  for (int i = 0; i < 3; i++) d.ls[i] = t.ls[i];
  d.o_vec = tvec_ok(t.o, t.os, p.dv, 2);
  d.do_vec = 1;
  d.n_tokens_q = (int64_t)p.g.TR * p.g.XLq;
  // delta = rowsum(o * dO): folded into the dQ kernel when o can be read in 16-byte pieces
  const bool fuse_delta = tvec_ok(t.o, t.os, p.dv, 2) && slab_span(p, t.os, (int64_t)p.g.TR * p.g.XLq) * 2 < ((int64_t)1 << 31);
  if (!fuse_delta) {
    int rc = dc.id == 0 ? dlt_launch_delta_64_64(d, stream) : dc.id == 1 ? dlt_launch_delta_128_128(d, stream)
           : dc.id == 3 ? dlt_launch_delta_32_32(d, stream) : dlt_launch_delta_64_128(d, stream);
    if (rc != DLT_OK) return rc;
  }

  FlashBwdArgs a;
  a.q = t.q; a.k = t.k; a.v = t.v; a.o = t.o; a.d_o = t.d_o; a.lse = t.lse; a.delta = t.delta;
  a.delta_out = t.delta;
  a.fuse_delta = fuse_delta ? 1 : 0;
  a.dq = t.dq; a.dk = t.dk; a.dv = t.dv;
  for (int i = 0; i < 5; i++) {
    a.qs[i] = t.qs[i]; a.ks[i] = t.ks[i]; a.vs[i] = t.vs[i]; a.os[i] = t.os[i]; a.dos[i] = t.dos[i];
    a.dqs[i] = t.dqs[i]; a.dks[i] = t.dks[i]; a.dvs[i] = t.dvs[i];
  }
  for (int i = 0; i < 3; i++) a.ls[i] = t.ls[i];
  a.tm = p.tm;
  a.B = p.B; a.H = p.H; a.Lq = p.g.XLq; a.Lk = p.g.XLk; a.dk_ = p.dk; a.dv_ = p.dv;
  const int own = 64 * flash_np_q(dc.DK, dc.DV), own_kv = 64 * flash_np_kv(dc.DK, dc.DV);
  a.nblk_q = (a.Lq + own - 1) / own;
  a.nblk_k = (a.Lk + own_kv - 1) / own_kv;
  a.causal = p.g.mode == DLT_GEOM_CAUSAL;
  a.causal_group = flash_causal_group(a.Lk, p.dk, p.dv);
  a.tile = p.g.mode == DLT_GEOM_SWA;
  a.g = p.g;
  a.dq_vec = tvec_ok(t.dq, t.dqs, p.dk, 2);
  a.dk_vec = tvec_ok(t.dk, t.dks, p.dk, 2);
  a.dv_vec = tvec_ok(t.dv, t.dvs, p.dv, 2);
  const int row = dc.DK * 2 + FLASH_PAD + dc.DV * 2 + FLASH_PAD;   // one streamed token in both LDS regions
  const int chunk_q = flash_ck_q(dc.DK, dc.DV) * row, ck_kv = flash_ck_kv(dc.DK, dc.DV);
  const int tile_q = own * (dc.DK * 2 + 16);
  const int tile_k = own_kv * (dc.DK * 2 + 16), tile_v = own_kv * (dc.DV * 2 + 16);
  a.lds_q = chunk_q > tile_q ? chunk_q : tile_q;
  a.lds_kv = ck_kv * row + 2 * ck_kv * 4;
  if (tile_k > a.lds_kv) a.lds_kv = tile_k;
  if (tile_v > a.lds_kv) a.lds_kv = tile_v;
  a.scale_log2 = p.sm_scale * 1.4426950408889634f;
  a.sm_scale = p.sm_scale;
  const int64_t grid_q = (int64_t)p.B * p.H * p.g.TR * a.nblk_q, grid_kv = (int64_t)p.B * p.H * p.g.TR * a.nblk_k;
  if (grid_q > 0x7fffffff || grid_kv > 0x7fffffff) return dlt_set_error(DLT_ERR_UNSUPPORTED, "flash backward: grid too large");
  // each pass streams its other side through LDS or splits it over the waves, whichever suits its own shape
  const int64_t nbh = (int64_t)p.B * p.H;
  const bool seq = p.g.mode != DLT_GEOM_SWA;
  FlashPlan fq = {FLASH_CHUNKED, 1, a.Lk, false}, fkv = {FLASH_CHUNKED, 1, a.Lq, false};
  if (seq) {
    bool may_split = t.shares && flash_may_split(p, dc);
    fq = flash_plan(1, dc, p.dk, p.dv, nbh, a.Lq, a.Lk, a.causal != 0, may_split);
    may_split = may_split && dlt_flash_scalars_fit(a);   // else dK/dV stays on the register-staged kernel
    fkv = flash_plan(2, dc, p.dk, p.dv, nbh, a.Lk, a.Lq, a.causal != 0, may_split);
  }
  if (flash_tiles_split(p, dc, true)) {
    fq.kind = fkv.kind = FLASH_SPLIT1;
    a.Lq = a.Lk = p.g.TR * p.g.XLq;
  }
  const int np_q = fq.kind, np_kv = fkv.kind;
  a.share_q = {t.part, fq.n, fq.len, fq.walk};
  a.share_kv = {t.part + flash_part_q(p, fq.n, fq.walk), fkv.n, fkv.len, fkv.walk};
  a.slim = np_kv == FLASH_SLIM;
  // dQ with one workgroup of 128 queries per CU: 8 waves of one block (16 slabs of 2048 x 2048: 64/64 36.6 -> 34.6 us, 64/128 43.8 -> 41.0,
  // 128/128 58.0 -> 54.2; from two workgroups per CU on slower, 32 slabs 54.8 -> 56.0, 70.4 -> 70.5, 94.9 -> 108.5)
  // (under a mask 4 waves run up to there and beyond)
  a.slim_q = np_q == FLASH_SLIM ? 4 : p.g.mode == DLT_GEOM_DENSE && fq.n == 1 && nbh * ((a.Lq + 127) / 128) <= dlt_device_cus() ? 8 : 0;
  int rc;
#define DLT_FLASH_PASS(C)                                                                                                  \
  rc = np_q == FLASH_SPLIT1 || np_q == FLASH_SPLIT2 ? dlt_flashs_bwd_q_##C(a, p.dtype, np_q, stream) : dlt_flash_launch_bwd_q_##C(a, p.dtype, (int)grid_q, stream); \
  if (rc != DLT_OK) return rc;                                                                                             \
  rc = np_kv == FLASH_SPLIT1 || np_kv == FLASH_SPLIT2 ? dlt_flashs_bwd_kv_##C(a, p.dtype, np_kv, stream) : dlt_flash_launch_bwd_kv_##C(a, p.dtype, (int)grid_kv, stream); \
  break
  switch (dc.id) {
    case 0: DLT_FLASH_PASS(64_64);
    case 1: DLT_FLASH_PASS(128_128);
    case 3: DLT_FLASH_PASS(32_32);
    default: DLT_FLASH_PASS(64_128);
  }
  if (rc == DLT_OK && fq.n > 1 && !fq.walk) rc = dlt_flash_share_bwd_q(a, p.dtype, stream);
  if (rc == DLT_OK && fkv.n > 1 && !fkv.walk) rc = dlt_flash_share_bwd_kv(a, p.dtype, stream);
  return rc;
#undef DLT_FLASH_PASS
}

}  // namespace

int dlt_attn_forward(const AttnProblem& p, const AttnTensors& t, hipStream_t stream) {
  dlt_route_reset();
  DimClass dc;
  int rc = pick_dims(p, dc);
  if (rc != DLT_OK) return rc;
  const int es = dlt_elem_size(p.dtype);
  {
    // q is not streamed, but its own-token fragments are read as 16-byte pieces too
    const bool streamed[3] = {tvec_ok(t.q, t.qs, p.dk, es), tvec_ok(t.k, t.ks, p.dk, es), tvec_ok(t.v, t.vs, p.dv, es)};
    Swa1Class c;
    if (swa1_eligible(p, streamed, 3, c) && swa1_strides_fit(p, t)) {
      // rotated side outputs come from the fused kernels only (16-byte rows); otherwise see below
      const bool side_ok = t.q_rot == nullptr || (c.rope_mode != 0 && tvec_ok(t.q_rot, t.qrs, p.dk, es) &&
                                                  tvec_ok(t.k_rot, t.krs, p.dk, es));
      if (side_ok) {
        if (swag_eligible(p, t, c, false)) return swag_run(p, t, false, stream);
        if (swa2_eligible(p, c) && t.q_rot == nullptr && swa2_rows_ok(p, t.out_o, t.os)) return swa2_forward(p, t, stream);
        // Rotation the marching kernels do not take, with the rotated q / k wanted by the caller: rotating both out of place
        // first (below) and running the streaming kernels on the result is faster than the tile kernels, which rotate every
        // halo row again in each workgroup that stages it (128 x 128 grid, d = 128, 21 x 21, 16 rotary pairs, fwd+bwd:
        // 0.90 -> 0.64 ms)
        const bool compose = c.rope_mode != 0 && t.q_rot != nullptr && swa2_compose_ok(p, c) && swa2_rows_ok(p, t.out_o, t.os) &&
                             swa2_rows_ok(p, t.q_rot, t.qrs) && swa2_rows_ok(p, t.k_rot, t.krs);
        if (c.wclass < 2 && !compose) return swa1_forward(p, t, c, stream);
      }
    }
  }
  if (t.q_rot != nullptr) {
    // rotate q and k out of place, then run the plain operator on the rotated tensors (any kernel family)
    const void* const src[2] = {t.q, t.k};
    void* const dst[2] = {t.q_rot, t.k_rot};
    const int64_t *const ss[2] = {t.qs, t.ks}, *const ds[2] = {t.qrs, t.krs};
    rc = dlt_rope_rotate_copy(src, ss, dst, ds, 2, p.B, p.H, (int64_t)p.g.TR * p.g.XLq, p.dk, p.rope, p.dtype, stream);
    if (rc != DLT_OK) return rc;
    AttnProblem p2 = p;
    p2.rope = dlt_make_rope_dev(nullptr, 0);
    AttnTensors t2 = t;
    t2.q = t.q_rot; t2.k = t.k_rot; t2.q_rot = t2.k_rot = nullptr;
    for (int i = 0; i < 5; i++) { t2.qs[i] = t.qrs[i]; t2.ks[i] = t.krs[i]; }
    return dlt_attn_forward(p2, t2, stream);
  }
  if (swag_f32_eligible(p, t)) return swag_run(p, t, false, stream);
  if (flash_eligible(p, t, false) && swat_eligible(p, t, false)) return swat_run(p, t, false, stream);
  if (flash_eligible(p, t, false)) return flash_forward(p, t, dc, stream);
  if (swa2_tiles_eligible(p, t, false)) return swa2_forward(p, t, stream);
  if (dlt_route_note(DLT_FAMILY_GENERIC)) return DLT_OK;
  WinArgs win;
  int win_lds;
  if (win_plan(p, t, dc, win, win_lds)) return win_forward(p, t, dc, win, win_lds, stream);
  const int np = (p.g.mode == DLT_GEOM_SWA || dc.id == 4) ? 1 : 2;
  const int own = 64 * np;
  // fp32 tensors: q and k rows are staged as hi + lo bf16 pairs (must match SPLIT in attn_fwd_kernel.hpp)
  const int PQ = dc.DK * (p.dtype == DLT_FP32 ? 4 : 2) + 16, PK = PQ, PV = dc.DV * 2 + 16, PO = dc.DV * es + 16;
  FwdArgs a;
  a.p = p;
  rc = make_plan(p, own, own * (PQ > PO ? PQ : PO), PK + PV, p.g.XLq, p.g.XLk, a.plan);
  if (rc != DLT_OK) return rc;
  a.plan.off_b = a.plan.off_a + a.plan.chunk_rows * a.plan.chunk_x * PK;
  a.plan.off_c = a.plan.off_d = 0;
  a.q = t.q; a.k = t.k; a.v = t.v; a.o = t.out_o; a.lse = t.lse;
  for (int i = 0; i < 5; i++) { a.qs[i] = t.qs[i]; a.ks[i] = t.ks[i]; a.vs[i] = t.vs[i]; a.os[i] = t.os[i]; }
  for (int i = 0; i < 3; i++) a.ls[i] = t.ls[i];
  a.q_vec = tvec_ok(t.q, t.qs, p.dk, es);
  a.k_vec = tvec_ok(t.k, t.ks, p.dk, es);
  a.v_vec = tvec_ok(t.v, t.vs, p.dv, es);
  a.o_vec = tvec_ok(t.out_o, t.os, p.dv, es);
  a.scale_log2 = p.sm_scale * 1.4426950408889634f;
  const int64_t grid = (int64_t)p.B * p.H * p.g.TR * a.plan.nblk_x;
  if (grid > 0x7fffffff) return dlt_set_error(DLT_ERR_UNSUPPORTED, "attention forward: grid too large");
  switch (dc.id) {
    case 0: return dlt_launch_fwd_64_64(a, np, (int)grid, stream);
    case 1: return dlt_launch_fwd_128_128(a, np, (int)grid, stream);
    case 3: return dlt_launch_fwd_32_32(a, np, (int)grid, stream);
    case 4: return dlt_launch_fwd_256_256(a, np, (int)grid, stream);
    default: return dlt_launch_fwd_64_128(a, np, (int)grid, stream);
  }
}

int64_t dlt_attn_part_floats(const AttnProblem& p, bool backward) {
  DimClass dc;
  if (p.g.mode != DLT_GEOM_DENSE || p.dk > 128 || p.dv > 128 || pick_dims(p, dc) != DLT_OK) return 0;
  if (!flash_may_split(p, dc)) return 0;
  const int64_t bh = (int64_t)p.B * p.H;
  const FlashShares f = flash_shares(backward ? 1 : 0, dc, p.dk, p.dv, bh, p.g.XLq, p.g.XLk);
  if (!backward) return flash_part_fwd(p, f.n, f.walk);
  const FlashShares kv = flash_shares(2, dc, p.dk, p.dv, bh, p.g.XLk, p.g.XLq);
  return flash_part_q(p, f.n, f.walk) + flash_part_kv(p, kv.n, kv.walk);
}

int dlt_attn_backward(const AttnProblem& p, const AttnTensors& t, hipStream_t stream) {
  dlt_route_reset();
  DimClass dc;
  int rc = pick_dims(p, dc);
  if (rc != DLT_OK) return rc;
  const int es = dlt_elem_size(p.dtype);
  {
    const bool streamed[4] = {tvec_ok(t.q, t.qs, p.dk, es), tvec_ok(t.k, t.ks, p.dk, es),
                              tvec_ok(t.v, t.vs, p.dv, es), tvec_ok(t.d_o, t.dos, p.dv, es)};
    Swa1Class c;
    if (swa1_eligible(p, streamed, 4, c) && swa1_strides_fit(p, t)) {
      if (swag_eligible(p, t, c, true)) return swag_run(p, t, true, stream);
      // lse2 / delta rows are copied with 32-bit byte offsets inside a (batch, head) slab
      if (swa2_eligible(p, c) && swa2_rows_ok(p, t.o, t.os) && swa2_rows_ok(p, t.dq, t.dqs) && swa2_rows_ok(p, t.dk, t.dks) &&
          swa2_rows_ok(p, t.dv, t.dvs) && swa2_scalars_ok(p, t))
        return swa2_backward(p, t, stream);
      // rotated q, k that the marching kernels do not take: the streaming kernels on the rotated tensors, then dq / dk
      // rotated back in place (below), instead of the tile kernels (see the forward pass)
      const bool compose = p.rope_prerot && c.rope_mode != 0 && swa2_compose_ok(p, c) && swa2_rows_ok(p, t.o, t.os) &&
                           swa2_rows_ok(p, t.dq, t.dqs) && swa2_rows_ok(p, t.dk, t.dks) && swa2_rows_ok(p, t.dv, t.dvs) && swa2_scalars_ok(p, t);
      if (c.wclass < 2 && !compose) return swa1_backward(p, t, c, stream);
    }
  }
  if (p.rope_prerot && p.rope.enabled && p.rope.R > 0 && !p.tm.img) {
    // rotated q, k and no token-grid kernel: the plain operator (any kernel family) yields the gradients of the
    // rotated tensors; the standalone rotation turns them back in place
    AttnProblem p2 = p;
    p2.rope = dlt_make_rope_dev(nullptr, 0);
    p2.rope_prerot = 0;
    rc = dlt_attn_backward(p2, t, stream);
    if (rc != DLT_OK) return rc;
    dlt_rope_t r;
    r.idx = p.rope.idx; r.row_cs = p.rope.row_cs; r.col_cs = p.rope.col_cs;
    r.row_cs_stride0 = p.rope.rs0; r.col_cs_stride0 = p.rope.cs0;
    r.n_rdim = p.rope.R; r.row_len = p.rope.row_len; r.col_len = p.rope.col_len;
    void* const x[2] = {t.dq, t.dk};
    const int64_t* const st[2] = {t.dqs, t.dks};
    return dlt_rope_inplace_4d(x, st, 2, p.B, p.H, (int64_t)p.g.TR * p.g.XLq, p.dk, &r, 1, p.dtype, stream);
  }
  if (flash_eligible(p, t, true) && swat_eligible(p, t, true)) return swat_run(p, t, true, stream);
  if (flash_eligible(p, t, true)) return flash_backward(p, t, dc, stream);
  if (swa2_tiles_eligible(p, t, true)) return swa2_backward(p, t, stream);
  if (dlt_route_note(DLT_FAMILY_GENERIC)) return DLT_OK;
  const int np = 1;
  const int own = 64 * np;
  // fp32 tensors: q and k rows are staged as hi + lo bf16 pairs (must match SPLIT in attn_bwd_kernel.hpp)
  const int PQ = dc.DK * (p.dtype == DLT_FP32 ? 4 : 2) + 16, PV = dc.DV * 2 + 16;
  const int tile_k = dc.DK * es + 16, tile_v = dc.DV * es + 16;
  int own_bytes = own * (PQ + PV);
  if (own * tile_k > own_bytes) own_bytes = own * tile_k;
  if (own * tile_v > own_bytes) own_bytes = own * tile_v;

  BwdArgs a;
  a.p = p;
  a.q = t.q; a.k = t.k; a.v = t.v; a.o = t.o; a.d_o = t.d_o; a.lse = t.lse; a.delta = t.delta;
  a.dq = t.dq; a.dk = t.dk; a.dv = t.dv;
  for (int i = 0; i < 5; i++) {
    a.qs[i] = t.qs[i]; a.ks[i] = t.ks[i]; a.vs[i] = t.vs[i]; a.os[i] = t.os[i]; a.dos[i] = t.dos[i];
    a.dqs[i] = t.dqs[i]; a.dks[i] = t.dks[i]; a.dvs[i] = t.dvs[i];
  }
  for (int i = 0; i < 3; i++) a.ls[i] = t.ls[i];
  a.q_vec = tvec_ok(t.q, t.qs, p.dk, es);
  a.k_vec = tvec_ok(t.k, t.ks, p.dk, es);
  a.v_vec = tvec_ok(t.v, t.vs, p.dv, es);
  a.o_vec = tvec_ok(t.o, t.os, p.dv, es);
  a.do_vec = tvec_ok(t.d_o, t.dos, p.dv, es);
  a.dq_vec = tvec_ok(t.dq, t.dqs, p.dk, es);
  a.dk_vec = tvec_ok(t.dk, t.dks, p.dk, es);
  a.dv_vec = tvec_ok(t.dv, t.dvs, p.dv, es);
  a.scale_log2 = p.sm_scale * 1.4426950408889634f;
  a.n_tokens_q = (int64_t)p.g.TR * p.g.XLq;

  // dK/dV: keys are the own side, queries (Q, dO, lse2, delta) are streamed
  BwdArgs akv = a;
  rc = make_plan(p, own, own_bytes, PQ + PV + 8, p.g.XLk, p.g.XLq, akv.plan);
  if (rc != DLT_OK) return rc;
  {
    const int toks = akv.plan.chunk_rows * akv.plan.chunk_x;
    akv.plan.off_b = akv.plan.off_a + toks * PQ;
    akv.plan.off_c = akv.plan.off_b + toks * PV;
    akv.plan.off_d = akv.plan.off_c + toks * 4;
  }
  // dQ: queries are the own side, K and V are streamed
  BwdArgs aq = a;
  rc = make_plan(p, own, own_bytes, PQ + PV, p.g.XLq, p.g.XLk, aq.plan);
  if (rc != DLT_OK) return rc;
  aq.plan.off_b = aq.plan.off_a + aq.plan.chunk_rows * aq.plan.chunk_x * PQ;
  aq.plan.off_c = aq.plan.off_d = 0;

  const int64_t grid_kv = (int64_t)p.B * p.H * p.g.TR * akv.plan.nblk_x;
  const int64_t grid_q = (int64_t)p.B * p.H * p.g.TR * aq.plan.nblk_x;
  if (grid_kv > 0x7fffffff || grid_q > 0x7fffffff) return dlt_set_error(DLT_ERR_UNSUPPORTED, "attention backward: grid too large");
  switch (dc.id) {
    case 0: return dlt_launch_bwd_64_64(akv, (int)grid_kv, aq, (int)grid_q, np, stream);
    case 1: return dlt_launch_bwd_128_128(akv, (int)grid_kv, aq, (int)grid_q, np, stream);
    case 3: return dlt_launch_bwd_32_32(akv, (int)grid_kv, aq, (int)grid_q, np, stream);
    case 4: return dlt_launch_bwd_256_256(akv, (int)grid_kv, aq, (int)grid_q, np, stream);
    default: return dlt_launch_bwd_64_128(akv, (int)grid_kv, aq, (int)grid_q, np, stream);
  }
}
