// Included by swag_inst_<D>_<NCH>.hip with DLT_D, DLT_NCH defined: instantiations and launchers of the marching token-grid
// kernels by window class.
#include "swag_kernel.hpp"

#define DLT_CAT4_(a, b, c, d) a##b##c##d
#define DLT_CAT4(a, b, c, d) DLT_CAT4_(a, b, c, d)

namespace {
constexpr int PC = SWAG_PC;

template <typename TIO, int NCG, bool ROPE>
int swag_fwd(const SwagArgs& a, int grid, hipStream_t stream) {
  typedef Swag<DLT_D, DLT_NCH, NCG, PC> C;
  void (*kern)(SwagArgs);
  if constexpr (ROPE) kern = swag_fwd_rope_kernel<TIO, DLT_D, DLT_NCH, NCG, PC>;
  else kern = swag_fwd_kernel<TIO, DLT_D, DLT_NCH, NCG, PC>;
  constexpr int lds = C::RING + (ROPE ? SWAG_TAB_BYTES : 0);
  static_assert(lds <= 160 * 1024, "ring and tables exceed the LDS");
  const int rc = dlt_ensure_lds(reinterpret_cast<const void*>(kern), lds);
  if (rc != DLT_OK) return rc;
  dlt_timing_before(DLT_K_FWD, stream);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(512), lds, stream, a);
  dlt_timing_after(stream);
  DLT_CHECK_LAUNCH("marching token-grid forward launch");
  return DLT_OK;
}

template <typename TIO, int NCG, bool ROPE>
int swag_bwd(const SwagArgs& a, int grid, hipStream_t stream) {
  typedef Swag<DLT_D, DLT_NCH, NCG, PC> C;
  // dQ first: it produces the delta vector the dK/dV kernel consumes
  auto kq = swag_bwd_q_kernel<TIO, DLT_D, DLT_NCH, NCG, PC, ROPE>;
  auto kkv = swag_bwd_kv_kernel<TIO, DLT_D, DLT_NCH, NCG, PC, ROPE>;
  int rc = dlt_ensure_lds(reinterpret_cast<const void*>(kq), C::RING);
  if (rc == DLT_OK) rc = dlt_ensure_lds(reinterpret_cast<const void*>(kkv), C::RING + C::SCAL);
  if (rc != DLT_OK) return rc;
  dlt_timing_before(DLT_K_BWD_Q, stream);
  hipLaunchKernelGGL(kq, dim3(grid), dim3(512), C::RING, stream, a);
  dlt_timing_after(stream);
  DLT_CHECK_LAUNCH("marching token-grid dQ launch");
  dlt_timing_before(DLT_K_BWD_KV, stream);
  hipLaunchKernelGGL(kkv, dim3(grid), dim3(512), C::RING + C::SCAL, stream, a);
  dlt_timing_after(stream);
  DLT_CHECK_LAUNCH("marching token-grid dK/dV launch");
  return DLT_OK;
}

template <typename TIO, bool ROPE>
int swag_pick(const SwagArgs& a, int ncg, bool bwd, int grid, hipStream_t stream) {
  switch (ncg) {
    case 2: return bwd ? swag_bwd<TIO, 2, ROPE>(a, grid, stream) : swag_fwd<TIO, 2, ROPE>(a, grid, stream);
    case 3: return bwd ? swag_bwd<TIO, 3, ROPE>(a, grid, stream) : swag_fwd<TIO, 3, ROPE>(a, grid, stream);
    case 4: return bwd ? swag_bwd<TIO, 4, ROPE>(a, grid, stream) : swag_fwd<TIO, 4, ROPE>(a, grid, stream);
    default: break;
  }
  if constexpr (DLT_D == 32) {   // head dim 32: the ring of a 24-column window fits as well
    if (ncg == 5) return bwd ? swag_bwd<TIO, 5, ROPE>(a, grid, stream) : swag_fwd<TIO, 5, ROPE>(a, grid, stream);
    if (ncg == 6) return bwd ? swag_bwd<TIO, 6, ROPE>(a, grid, stream) : swag_fwd<TIO, 6, ROPE>(a, grid, stream);
  }
  return dlt_set_error(DLT_ERR_UNSUPPORTED, "marching token-grid kernels: no instantiation for %d column groups", ncg);
}
template <typename TIO>
int swag_pick_rope(const SwagArgs& a, int ncg, bool bwd, int grid, hipStream_t stream) {
  if constexpr (DLT_D == 64)
    if (a.rope.enabled) return swag_pick<TIO, true>(a, ncg, bwd, grid, stream);
  return swag_pick<TIO, false>(a, ncg, bwd, grid, stream);
}
}  // namespace

int DLT_CAT4(dlt_swag_launch_, DLT_D, _, DLT_NCH)(const SwagArgs& a, int dtype, int ncg, bool bwd, int grid, hipStream_t stream) {
  return dtype == DLT_BF16 ? swag_pick_rope<bf16_t>(a, ncg, bwd, grid, stream) : swag_pick_rope<f16_t>(a, ncg, bwd, grid, stream);
}
