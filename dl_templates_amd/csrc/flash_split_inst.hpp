// Included by flash_split_<DK>_<DV>.hip with DLT_DK / DLT_DV defined: launchers of the kernels that split the streamed side
// over the waves of a workgroup.
#include "flash_split_kernel.hpp"

#define DLT_FCAT3_(a, b, c) a##b##_##c
#define DLT_FCAT3(a, b, c) DLT_FCAT3_(a, b, c)

namespace {
constexpr int NW = 8;
// own blocks per workgroup of the backward kernels: two fit the registers up to 64/64
constexpr int NPB = DLT_DK + DLT_DV <= 128 ? 2 : 1;

template <typename KernT, typename Args>
int flashs_run(KernT kern, const Args& a, int lds, int grid, int id, hipStream_t stream) {
  const int rc = dlt_ensure_lds(reinterpret_cast<const void*>(kern), lds);
  if (rc != DLT_OK) return rc;
  dlt_timing_before(id, stream);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(64 * NW), lds, stream, a);
  dlt_timing_after(stream);
  DLT_CHECK_LAUNCH("flash split launch");
  return DLT_OK;
}

// (tiles: one own block, all output dims)
template <typename Args, typename KernT>
KernT flashs_mode(const Args& a, KernT dense, KernT causal, KernT tiles, KernT image) { return a.tile ? (a.tm.img ? image : tiles) : a.causal ? causal : dense; }

template <typename TIO, int NP, int DV>
int flashs_fwd_dv(FlashArgs a, hipStream_t stream) {
  a.parts = (a.dv + DV - 1) / DV;
  return flashs_run(flashs_mode(a, flashs_fwd_kernel<TIO, DLT_DK, DV, NP, NW, 0>, flashs_fwd_kernel<TIO, DLT_DK, DV, NP, NW, 1>, 
                                flashs_fwd_kernel<TIO, DLT_DK, DV, NP, NW, NP == 1 && DV == DLT_DV ? 2 : 0>, flashs_fwd_kernel<TIO, DLT_DK, DV, NP, NW, NP == 1 && DV == DLT_DV ? 3 : 0>), a,
                    flashs_lds_fwd<DLT_DK, DV, NP, NW>(), a.B * a.H * a.nblk * a.parts, DLT_K_FWD, stream);
}
template <typename TIO, int NP>
int flashs_fwd(FlashArgs a, hipStream_t stream) {
  a.nblk = (a.Lq + 16 * NP - 1) / (16 * NP);
  if constexpr (NP == 1 && DLT_DV == 128)
    if (a.part_dv == DLT_DV / 4) return flashs_fwd_dv<TIO, NP, DLT_DV / 4>(a, stream);
  if constexpr (NP == 1 && DLT_DV >= 64)
    if (a.part_dv == DLT_DV / 2) return flashs_fwd_dv<TIO, NP, DLT_DV / 2>(a, stream);
  return flashs_fwd_dv<TIO, NP, DLT_DV>(a, stream);
}
template <typename TIO, int NP>
int flashs_bwd_q(FlashBwdArgs a, hipStream_t stream) {
  a.nblk_q = (a.Lq + 16 * NP - 1) / (16 * NP);
  return flashs_run(flashs_mode(a, flashs_bwd_q_kernel<TIO, DLT_DK, DLT_DV, NP, NW, 0>, flashs_bwd_q_kernel<TIO, DLT_DK, DLT_DV, NP, NW, 1>, 
                                flashs_bwd_q_kernel<TIO, DLT_DK, DLT_DV, NP, NW, NP == 1 ? 2 : 0>, flashs_bwd_q_kernel<TIO, DLT_DK, DLT_DV, NP, NW, NP == 1 ? 3 : 0>), a,
                    flashs_lds_q<DLT_DK, DLT_DV, NP, NW>(), a.B * a.H * a.nblk_q, DLT_K_BWD_Q, stream);
}
template <typename TIO, int NP>
int flashs_bwd_kv(FlashBwdArgs a, hipStream_t stream) {
  a.nblk_k = (a.Lk + 16 * NP - 1) / (16 * NP);
  return flashs_run(flashs_mode(a, flashs_bwd_kv_kernel<TIO, DLT_DK, DLT_DV, NP, NW, 0>, flashs_bwd_kv_kernel<TIO, DLT_DK, DLT_DV, NP, NW, 1>, 
                                flashs_bwd_kv_kernel<TIO, DLT_DK, DLT_DV, NP, NW, NP == 1 ? 2 : 0>, flashs_bwd_kv_kernel<TIO, DLT_DK, DLT_DV, NP, NW, NP == 1 ? 3 : 0>), a,
                    flashs_lds_kv<DLT_DK, DLT_DV, NP, NW>(), a.B * a.H * a.nblk_k, DLT_K_BWD_KV, stream);
}
}  // namespace

// np: 16-token blocks a workgroup owns (1 or 2)
int DLT_FCAT3(dlt_flashs_fwd_, DLT_DK, DLT_DV)(const FlashArgs& a, int dtype, int np, hipStream_t stream) {
  if (dtype == DLT_BF16) return np == 1 ? flashs_fwd<bf16_t, 1>(a, stream) : flashs_fwd<bf16_t, 2>(a, stream);
  return np == 1 ? flashs_fwd<f16_t, 1>(a, stream) : flashs_fwd<f16_t, 2>(a, stream);
}
int DLT_FCAT3(dlt_flashs_bwd_q_, DLT_DK, DLT_DV)(const FlashBwdArgs& a, int dtype, int np, hipStream_t stream) {
  if (dtype == DLT_BF16) return np == 1 ? flashs_bwd_q<bf16_t, 1>(a, stream) : flashs_bwd_q<bf16_t, NPB>(a, stream);
  return np == 1 ? flashs_bwd_q<f16_t, 1>(a, stream) : flashs_bwd_q<f16_t, NPB>(a, stream);
}
int DLT_FCAT3(dlt_flashs_bwd_kv_, DLT_DK, DLT_DV)(const FlashBwdArgs& a, int dtype, int np, hipStream_t stream) {
  if (dtype == DLT_BF16) return np == 1 ? flashs_bwd_kv<bf16_t, 1>(a, stream) : flashs_bwd_kv<bf16_t, NPB>(a, stream);
  return np == 1 ? flashs_bwd_kv<f16_t, 1>(a, stream) : flashs_bwd_kv<f16_t, NPB>(a, stream);
}
