// Included by flash_{fwd,fwdc,dq,dkv}_<DK>_<DV>.hip with DLT_DK / DLT_DV defined: flash kernels for one pair of padded head dims;
// DLT_FLASH_PART 0: forward, 3: forward under a mask, 1: dQ, 2: dK/dV (units of their own, since they take minutes to compile).
#include "flash_dma_kernel.hpp"

#define DLT_FCAT3_(a, b, c) a##b##_##c
#define DLT_FCAT3(a, b, c) DLT_FCAT3_(a, b, c)

namespace {
// shape of the asynchronously staged forward kernel: keys per chunk, waves per workgroup (16 NP queries per wave).
// 8 waves on 128-key chunks at 64/128 and 128/128 (K / V copied once per 256 queries), 4 waves on 64-key chunks at 64/64
// (there the 8-wave shape only ties with the register-staged kernel)
#ifndef FLASHD_FWD_NP
#define FLASHD_FWD_NP FLASH_NP
#endif
#ifndef FLASHD_FWD_CK
#define FLASHD_FWD_CK(dk, dv) ((dk) + (dv) > 128 ? 128 : 64)
#endif
#ifndef FLASHD_FWD_NW
#define FLASHD_FWD_NW(dk, dv) ((dk) + (dv) > 128 ? 8 : 4)
#endif
// query blocks per wave of the asynchronously staged dQ kernel: two in every class (without staging registers two blocks
// fit at 128/128 as well: -18 % there; three blocks measured 8 % slower at 64/64 and 64/128)
#ifndef FLASHD_DQ_NP
#define FLASHD_DQ_NP(dk, dv) 2
#endif
// waves per workgroup of the asynchronously staged backward kernels (64-token chunks)
#ifndef FLASHD_BWD_NW
#define FLASHD_BWD_NW 4
#endif

// PAD of the asynchronously staged kernels for head dims dk, dv: 2 where the class's 128 dims hold 96 at most, 3 where they hold 80
// (all sides measured at flashd_dims)
inline int flashd_pad(int dk, int dv) {
  if (dk == DLT_DK && dv == DLT_DV) return 0;
  const int d = DLT_DV < 128 || dv > 96 || (DLT_DK > 64 && dk > 96) ? 128 : DLT_DK > 64 && dk > dv ? dk : dv;
  return d > 96 ? 1 : d > 80 ? 2 : 3;
}

// Windows over tiles of 64 k tokens run on the asynchronously staged kernels: exact head dims, chunks of whole pixel rows in the image layout.
inline bool flashd_tiles(int dk, int dv, const DltGeom& g, const DltTokMap& tm) {
  return dk == DLT_DK && dv == DLT_DV && g.S % 64 == 0 && (!tm.img || 64 % tm.bw == 0) && dlt_flash_async();
}
// ... in workgroups of 64 own tokens (one block per wave) while they are few, and where workgroups of 128 would be a sixth empty.  Two blocks
// per wave -> one, 3 x 3 tiles of 64 unless said, us, forward and backward: 4 slabs of 15 x 4, d = 64 14.9 -> 11.1 and 34.5 -> 26.0; images, 8 of 11 x 5
// 21 -> 14.5 and 46 -> 31; 64 of 11 x 5 60 -> 56 and 155 -> 145; 32 of 17 x 30 249 -> 278 and 611 -> 639; d = 128, 4 of 15 x 4 21 -> 16 and 46 -> 39, but 64 of
// 11 x 5 (8 waves of one block in the forward pass there) 92 -> 105 and 261 -> 261.
inline bool flashd_tiles_one(int slabs, int xl, const DltGeom& g) {
  const int64_t n = (xl + 63) / 64;
  return slabs * (int64_t)g.TR * n <= 3 * (int64_t)dlt_device_cus() || (DLT_DK + DLT_DV <= 192 && 6 * n <= 5 * ((n + 1) / 2 * 2));
}

template <typename KernT>
int flash_set_lds(KernT kern, int bytes) { return dlt_ensure_lds(reinterpret_cast<const void*>(kern), bytes); }

#if DLT_FLASH_PART == 0 || DLT_FLASH_PART == 3
template <typename TIO, int MODE, int NP, int CK, int NW, bool WALK = false>
int flashd_launch_fwd(FlashArgs a, hipStream_t stream) {
  // head dims below the padded ones (multiples of 8): the kernel variant whose copies skip the missing pieces
  const int pad = flashd_pad(a.dk, a.dv);
  auto kern = flashd_fwd_kernel<TIO, DLT_DK, DLT_DV, NP, CK, NW, MODE, 0, WALK>;
  if constexpr (MODE < 2)
    if (pad == 1) kern = flashd_fwd_kernel<TIO, DLT_DK, DLT_DV, NP, CK, NW, MODE, 1, WALK>;
  if constexpr (MODE < 2 && DLT_DV == 128) {
    if (pad == 2) kern = flashd_fwd_kernel<TIO, DLT_DK, DLT_DV, NP, CK, NW, MODE, 2, WALK>;
    if (pad == 3) kern = flashd_fwd_kernel<TIO, DLT_DK, DLT_DV, NP, CK, NW, MODE, 3, WALK>;
  }
  constexpr int own = 16 * NP * NW;
  constexpr int tile = own * (DLT_DV * 2 + 16);
  constexpr int bufs = flashd_bufs(DLT_DK, DLT_DV, NP, NW) * FlashDBuf<DLT_DK, DLT_DV, CK>::BUF;
  constexpr int lds = bufs > tile ? bufs : tile;
  const int rc = flash_set_lds(kern, lds);
  if (rc != DLT_OK) return rc;
  a.nblk = (a.Lq + own - 1) / own;
  const int rows = MODE >= 2 ? a.g.TR : WALK ? 1 : a.share.n;
  dlt_timing_before(DLT_K_FWD, stream);
  hipLaunchKernelGGL(kern, dim3(a.B * a.H * a.nblk * rows), dim3(64 * NW), lds, stream, a);
  dlt_timing_after(stream);
  DLT_CHECK_LAUNCH("flash forward launch");
  return DLT_OK;
}

template <typename TIO, int MODE>
int flash_launch_fwd_c(const FlashArgs& a, int grid, hipStream_t stream) {
  if constexpr (DLT_DK >= 64 && DLT_DV >= 64 && MODE < 2) {
    // dense / causal, head dims that are multiples of 8: chunks are copied HBM -> LDS asynchronously.  Measured per
    // class and mode against the register-staged kernel: dense -2 % (64/64), -4 % (64/128), -7 % (128/128); causal -4 %
    // (64/64), -18 % (128/128); head dims below the class (80/80, 96/96): -18 % on the step.
    if (a.dk % 8 == 0 && a.dv % 8 == 0 && dlt_flash_async()) {
      if constexpr (MODE == 0)
        if (a.share.walk)   // workgroups of 64 queries or 128
          return a.Lq <= 64 ? flashd_launch_fwd<TIO, 0, 1, 64, 4, true>(a, stream) : flashd_launch_fwd<TIO, 0, (DLT_DV == 128 ? 1 : 2), 64, (DLT_DV == 128 ? 8 : 4), true>(a, stream);
      // few workgroups: one own block per wave (see flash_forward)
      if constexpr (DLT_DV == 128)
        if (a.slim != 0 && a.chunk == 128)
          return a.slim == 4 ? flashd_launch_fwd<TIO, MODE, 1, 128, 4>(a, stream) : flashd_launch_fwd<TIO, MODE, 1, 128, 8>(a, stream);
      if (a.slim != 0) return a.slim == 4 ? flashd_launch_fwd<TIO, MODE, 1, 64, 4>(a, stream) : flashd_launch_fwd<TIO, MODE, 1, 64, 8>(a, stream);
      return flashd_launch_fwd<TIO, MODE, FLASHD_FWD_NP, FLASHD_FWD_CK(DLT_DK, DLT_DV), FLASHD_FWD_NW(DLT_DK, DLT_DV)>(a, stream);
    }
  }
  if constexpr (MODE >= 2)
    if (flashd_tiles(a.dk, a.dv, a.g, a.tm)) {
      if (flashd_tiles_one(a.B * a.H, a.Lq, a.g)) return flashd_launch_fwd<TIO, MODE, 1, 64, 4>(a, stream);
      return flashd_launch_fwd<TIO, MODE, (DLT_DK + DLT_DV > 192 ? 1 : 2), 64, (DLT_DK + DLT_DV > 192 ? 8 : 4)>(a, stream);
    }
  auto kern = flash_fwd_kernel<TIO, DLT_DK, DLT_DV, FLASH_NP, flash_ck_fwd(DLT_DK, DLT_DV), MODE>;
  {
    const int rc = dlt_ensure_lds(reinterpret_cast<const void*>(kern), a.lds_bytes);
    if (rc != DLT_OK) return rc;
  }
  dlt_timing_before(DLT_K_FWD, stream);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(256), a.lds_bytes, stream, a);
  dlt_timing_after(stream);
  DLT_CHECK_LAUNCH("flash forward launch");
  return DLT_OK;
}

#if DLT_FLASH_PART == 0
template <typename TIO>
int flash_launch_fwd_t(const FlashArgs& a, int grid, hipStream_t stream) {
  if (a.tile) return a.tm.img ? flash_launch_fwd_c<TIO, 3>(a, grid, stream) : flash_launch_fwd_c<TIO, 2>(a, grid, stream);
  return flash_launch_fwd_c<TIO, 0>(a, grid, stream);
}
}  // namespace

int DLT_FCAT3(dlt_flash_launch_fwd_, DLT_DK, DLT_DV)(const FlashArgs& a, int dtype, int grid, hipStream_t stream) {
  return dtype == DLT_BF16 ? flash_launch_fwd_t<bf16_t>(a, grid, stream) : flash_launch_fwd_t<f16_t>(a, grid, stream);
}
#else
}  // namespace

int DLT_FCAT3(dlt_flash_launch_fwdc_, DLT_DK, DLT_DV)(const FlashArgs& a, int dtype, int grid, hipStream_t stream) {
  return dtype == DLT_BF16 ? flash_launch_fwd_c<bf16_t, 1>(a, grid, stream) : flash_launch_fwd_c<f16_t, 1>(a, grid, stream);
}
#endif

#elif DLT_FLASH_PART == 1
template <typename TIO, int MODE, int NP, int NW, bool WALK = false>
int flashd_launch_bwd_q(FlashBwdArgs a, hipStream_t stream) {
  constexpr int CK = 64;
  const int pad = flashd_pad(a.dk_, a.dv_);
  auto kern = flashd_bwd_q_kernel<TIO, DLT_DK, DLT_DV, NP, CK, NW, MODE, 0, WALK>;
  if constexpr (MODE < 2)
    if (pad == 1) kern = flashd_bwd_q_kernel<TIO, DLT_DK, DLT_DV, NP, CK, NW, MODE, 1, WALK>;
  if constexpr (MODE < 2 && DLT_DV == 128) {
    if (pad == 2) kern = flashd_bwd_q_kernel<TIO, DLT_DK, DLT_DV, NP, CK, NW, MODE, 2, WALK>;
    if (pad == 3) kern = flashd_bwd_q_kernel<TIO, DLT_DK, DLT_DV, NP, CK, NW, MODE, 3, WALK>;
  }
  constexpr int own = 16 * NP * NW;
  constexpr int tile = own * (DLT_DK * 2 + 16);
  constexpr int bufs = flashd_dq_bufs(DLT_DK, DLT_DV, NP, NW) * FlashDBuf<DLT_DK, DLT_DV, CK>::BUF;
  constexpr int lds = bufs > tile ? bufs : tile;
  const int rc = flash_set_lds(kern, lds);
  if (rc != DLT_OK) return rc;
  a.nblk_q = (a.Lq + own - 1) / own;
  dlt_timing_before(DLT_K_BWD_Q, stream);
  hipLaunchKernelGGL(kern, dim3(a.B * a.H * a.nblk_q * (MODE >= 2 ? a.g.TR : WALK ? 1 : a.share_q.n)), dim3(64 * NW), lds, stream, a);
  dlt_timing_after(stream);
  DLT_CHECK_LAUNCH("flash dQ launch");
  return DLT_OK;
}

template <typename TIO, int MODE>
int flash_launch_bwd_q_c(const FlashBwdArgs& a, int grid_q, hipStream_t stream) {
  if constexpr (DLT_DK >= 64 && DLT_DV >= 64 && MODE < 2) {
    if (a.dk_ % 8 == 0 && a.dv_ % 8 == 0 && dlt_flash_async()) {
      if constexpr (MODE == 0)
        if (a.share_q.walk) {   // (two blocks' sums of 128 dims do not fit the registers)
          if constexpr (DLT_DK == 64)
            if (a.Lq > 256) return flashd_launch_bwd_q<TIO, 0, 2, 4, true>(a, stream);
          return flashd_launch_bwd_q<TIO, 0, 1, 4, true>(a, stream);
        }
      // few workgroups: one own block per wave, in 4 waves (twice the workgroups) or, without a mask, 8 (see flash_backward)
      if (a.slim_q == 4) return flashd_launch_bwd_q<TIO, MODE, 1, 4>(a, stream);
      if constexpr (MODE == 0)
        if (a.slim_q == 8) return flashd_launch_bwd_q<TIO, MODE, 1, 8>(a, stream);
      return flashd_launch_bwd_q<TIO, MODE, FLASHD_DQ_NP(DLT_DK, DLT_DV), FLASHD_BWD_NW>(a, stream);
    }
  }
  if constexpr (MODE >= 2)
    if (flashd_tiles(a.dk_, a.dv_, a.g, a.tm))
      return flashd_tiles_one(a.B * a.H, a.Lq, a.g) ? flashd_launch_bwd_q<TIO, MODE, 1, 4>(a, stream) : flashd_launch_bwd_q<TIO, MODE, 2, 4>(a, stream);
  auto kern = flash_bwd_q_kernel<TIO, DLT_DK, DLT_DV, flash_np_q(DLT_DK, DLT_DV), flash_ck_q(DLT_DK, DLT_DV), MODE>;
  int rc = flash_set_lds(kern, a.lds_q);
  if (rc != DLT_OK) return rc;
  dlt_timing_before(DLT_K_BWD_Q, stream);
  hipLaunchKernelGGL(kern, dim3(grid_q), dim3(256), a.lds_q, stream, a);
  dlt_timing_after(stream);
  DLT_CHECK_LAUNCH("flash dQ launch");
  return DLT_OK;
}

template <typename TIO>
int flash_launch_bwd_q_t(const FlashBwdArgs& a, int grid_q, hipStream_t stream) {
  if (a.tile) return a.tm.img ? flash_launch_bwd_q_c<TIO, 3>(a, grid_q, stream) : flash_launch_bwd_q_c<TIO, 2>(a, grid_q, stream);
  return a.causal ? flash_launch_bwd_q_c<TIO, 1>(a, grid_q, stream) : flash_launch_bwd_q_c<TIO, 0>(a, grid_q, stream);
}
}  // namespace

int DLT_FCAT3(dlt_flash_launch_bwd_q_, DLT_DK, DLT_DV)(const FlashBwdArgs& a, int dtype, int grid_q, hipStream_t stream) {
  return dtype == DLT_BF16 ? flash_launch_bwd_q_t<bf16_t>(a, grid_q, stream) : flash_launch_bwd_q_t<f16_t>(a, grid_q, stream);
}

#else
template <typename TIO, int MODE, int NP, int NW, bool WALK = false>
int flashd_launch_bwd_kv(FlashBwdArgs a, hipStream_t stream) {
  constexpr int CK = 64;
  const int pad = flashd_pad(a.dk_, a.dv_);
  auto kern = flashd_bwd_kv_kernel<TIO, DLT_DK, DLT_DV, NP, CK, NW, MODE, 0, WALK>;
  if constexpr (MODE < 2)
    if (pad == 1) kern = flashd_bwd_kv_kernel<TIO, DLT_DK, DLT_DV, NP, CK, NW, MODE, 1, WALK>;
  if constexpr (MODE < 2 && DLT_DV == 128) {
    if (pad == 2) kern = flashd_bwd_kv_kernel<TIO, DLT_DK, DLT_DV, NP, CK, NW, MODE, 2, WALK>;
    if (pad == 3) kern = flashd_bwd_kv_kernel<TIO, DLT_DK, DLT_DV, NP, CK, NW, MODE, 3, WALK>;
  }
  constexpr int own = 16 * NP * NW;
  constexpr int tile_k = own * (DLT_DK * 2 + 16), tile_v = own * (DLT_DV * 2 + 16);
  constexpr int bufs = flashd_bufs(DLT_DK, DLT_DV, NP, NW) * FlashDBuf<DLT_DK, DLT_DV, CK>::BUF_KV;
  constexpr int lds = bufs > tile_v ? (bufs > tile_k ? bufs : tile_k) : (tile_v > tile_k ? tile_v : tile_k);
  const int rc = flash_set_lds(kern, lds);
  if (rc != DLT_OK) return rc;
  a.nblk_k = (a.Lk + own - 1) / own;
  dlt_timing_before(DLT_K_BWD_KV, stream);
  hipLaunchKernelGGL(kern, dim3(a.B * a.H * a.nblk_k * (MODE >= 2 ? a.g.TR : WALK ? 1 : a.share_kv.n)), dim3(64 * NW), lds, stream, a);
  dlt_timing_after(stream);
  DLT_CHECK_LAUNCH("flash dK/dV launch");
  return DLT_OK;
}

template <typename TIO, int MODE>
int flash_launch_bwd_kv_c(const FlashBwdArgs& a, int grid_kv, hipStream_t stream) {
  if constexpr (DLT_DK >= 64 && DLT_DV >= 64 && MODE < 2) {
    // dense / causal, head dims that are multiples of 8: chunks are copied HBM -> LDS asynchronously (tiles that are no multiple of 64
    // tokens: parts of a chunk are skipped, the register-staged kernel measured 1.5 % faster)
    if (a.dk_ % 8 == 0 && a.dv_ % 8 == 0 && dlt_flash_scalars_fit(a) && dlt_flash_async()) {
      if constexpr (MODE == 0)
        if (a.share_kv.walk) {
          if constexpr (DLT_DV == 64)
            if (a.Lk > 64) return flashd_launch_bwd_kv<TIO, 0, 2, 4, true>(a, stream);
          return flashd_launch_bwd_kv<TIO, 0, 1, 4, true>(a, stream);
        }
      if (a.slim) return flashd_launch_bwd_kv<TIO, MODE, 1, 4>(a, stream);
      return flashd_launch_bwd_kv<TIO, MODE, flash_np_kv(DLT_DK, DLT_DV), FLASHD_BWD_NW>(a, stream);
    }
  }
  if constexpr (MODE >= 2)
    if (flashd_tiles(a.dk_, a.dv_, a.g, a.tm) && dlt_flash_scalars_fit(a))
      return flashd_tiles_one(a.B * a.H, a.Lk, a.g) ? flashd_launch_bwd_kv<TIO, MODE, 1, 4>(a, stream) : flashd_launch_bwd_kv<TIO, MODE, flash_np_kv(DLT_DK, DLT_DV), 4>(a, stream);
  {
    auto kern = flash_bwd_kv_kernel<TIO, DLT_DK, DLT_DV, flash_np_kv(DLT_DK, DLT_DV), flash_ck_kv(DLT_DK, DLT_DV), MODE>;
    int rc = flash_set_lds(kern, a.lds_kv);
    if (rc != DLT_OK) return rc;
    dlt_timing_before(DLT_K_BWD_KV, stream);
    hipLaunchKernelGGL(kern, dim3(grid_kv), dim3(256), a.lds_kv, stream, a);
    dlt_timing_after(stream);
    DLT_CHECK_LAUNCH("flash dK/dV launch");
  }
  return DLT_OK;
}

template <typename TIO>
int flash_launch_bwd_kv_t(const FlashBwdArgs& a, int grid_kv, hipStream_t stream) {
  if (a.tile) return a.tm.img ? flash_launch_bwd_kv_c<TIO, 3>(a, grid_kv, stream) : flash_launch_bwd_kv_c<TIO, 2>(a, grid_kv, stream);
  return a.causal ? flash_launch_bwd_kv_c<TIO, 1>(a, grid_kv, stream) : flash_launch_bwd_kv_c<TIO, 0>(a, grid_kv, stream);
}
}  // namespace

int DLT_FCAT3(dlt_flash_launch_bwd_kv_, DLT_DK, DLT_DV)(const FlashBwdArgs& a, int dtype, int grid_kv, hipStream_t stream) {
  return dtype == DLT_BF16 ? flash_launch_bwd_kv_t<bf16_t>(a, grid_kv, stream) : flash_launch_bwd_kv_t<f16_t>(a, grid_kv, stream);
}
#endif
