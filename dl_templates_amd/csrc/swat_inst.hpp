// Included by swat_inst_<D>.hip with DLT_D defined: instantiations and launchers of the marching tile-window kernels.
#include "swat_kernel.hpp"

#define DLT_CAT_(a, b) a##b
#define DLT_CAT(a, b) DLT_CAT_(a, b)

namespace {
template <typename TIO, int NTB, int WC, int WR>
int swat_launch_fwd(const SwatArgs& a, int grid, hipStream_t stream) {
  typedef Swat<DLT_D, NTB, WC, WR> C;
  auto kern = swat_fwd_kernel<TIO, DLT_D, NTB, WC, WR>;
  const int lds = a.lone ? dlt_imax(C::RING, 81 * 1024) : C::RING;   // more than half of a CU's: a second workgroup does not fit
  const int rc = dlt_ensure_lds(reinterpret_cast<const void*>(kern), lds);
  if (rc != DLT_OK) return rc;
  dlt_timing_before(DLT_K_FWD, stream);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(C::THREADS), lds, stream, a);
  dlt_timing_after(stream);
  DLT_CHECK_LAUNCH("marching tile-window forward launch");
  return DLT_OK;
}

// dQ, dK and dV in one launch (booked as the dK/dV kernel by dlt_timing_collect)
template <typename TIO, int NTB, int WC, int WR>
int swat_launch_bwd_one(const SwatArgs& a, int grid, hipStream_t stream) {
  typedef Swab<DLT_D, NTB, WC, WR> C;
  auto kern = swat_bwd_kernel<TIO, DLT_D, NTB, WC, WR>;
  const int rc = dlt_ensure_lds(reinterpret_cast<const void*>(kern), C::LDS);
  if (rc != DLT_OK) return rc;
  dlt_timing_before(DLT_K_BWD_KV, stream);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(C::THREADS), C::LDS, stream, a);
  dlt_timing_after(stream);
  DLT_CHECK_LAUNCH("marching tile-window backward launch");
  return DLT_OK;
}

template <typename TIO, int NTB, int WC, int WR>
int swat_launch_bwd_two(const SwatArgs& a, int grid, hipStream_t stream) {
  typedef Swat<DLT_D, NTB, WC, WR> C;
  static_assert(C::BWD, "ring and scalars exceed the LDS");
  // dQ first: it produces the delta vector the dK/dV kernel consumes
  auto kq = swat_bwd_q_kernel<TIO, DLT_D, NTB, WC, WR>;
  auto kkv = swat_bwd_kv_kernel<TIO, DLT_D, NTB, WC, WR>;
  int rc = dlt_ensure_lds(reinterpret_cast<const void*>(kq), C::RING);
  if (rc == DLT_OK) rc = dlt_ensure_lds(reinterpret_cast<const void*>(kkv), C::RING + C::SCAL);
  if (rc != DLT_OK) return rc;
  dlt_timing_before(DLT_K_BWD_Q, stream);
  hipLaunchKernelGGL(kq, dim3(grid), dim3(C::THREADS), C::RING, stream, a);
  dlt_timing_after(stream);
  DLT_CHECK_LAUNCH("marching tile-window dQ launch");
  dlt_timing_before(DLT_K_BWD_KV, stream);
  hipLaunchKernelGGL(kkv, dim3(grid), dim3(C::THREADS), C::RING + C::SCAL, stream, a);
  dlt_timing_after(stream);
  DLT_CHECK_LAUNCH("marching tile-window dK/dV launch");
  return DLT_OK;
}

template <typename TIO, int NTB, int WC, int WR>
int swat_launch_bwd(const SwatArgs& a, int grid, hipStream_t stream) {
  if constexpr (!Swab<DLT_D, NTB, WC, WR>::USED) return swat_launch_bwd_two<TIO, NTB, WC, WR>(a, grid, stream);
  else if constexpr (DLT_D == 64) return swat_launch_bwd_one<TIO, NTB, WC, WR>(a, grid, stream);   // see dlt_tile_bwd_one_launch
  else return a.one ? swat_launch_bwd_one<TIO, NTB, WC, WR>(a, grid, stream) : swat_launch_bwd_two<TIO, NTB, WC, WR>(a, grid, stream);
}

template <typename TIO>
int swat_pick(const SwatArgs& a, bool bwd, int grid, hipStream_t stream) {
#define DLT_SWAT(NTB, WC, WR) return bwd ? swat_launch_bwd<TIO, NTB, WC, WR>(a, grid, stream) : swat_launch_fwd<TIO, NTB, WC, WR>(a, grid, stream)
  const int ntb = a.g.S / 16;
#if DLT_D == 128   // forward only (swat_eligible)
  if (!bwd && ntb == 1 && a.g.WR == 1 && a.g.WC == 1) return swat_launch_fwd<TIO, 1, 1, 1>(a, grid, stream);
#else
  if (ntb == 2) DLT_SWAT(2, 1, 1);
  if (a.g.WR == 1) {
    if (a.g.WC == 1) DLT_SWAT(1, 1, 1);
    DLT_SWAT(1, 2, 1);
  }
  if (a.g.WC == 1) DLT_SWAT(1, 1, 2);
#if DLT_D == 32
  DLT_SWAT(1, 2, 2);
#else
  if (!bwd) return swat_launch_fwd<TIO, 1, 2, 2>(a, grid, stream);   // swat_eligible
#endif
#endif
  return dlt_set_error(DLT_ERR_UNSUPPORTED, "marching tile-window kernels: no instantiation for this window");
#undef DLT_SWAT
}
}  // namespace

int DLT_CAT(dlt_swat_launch_, DLT_D)(const SwatArgs& a, int dtype, bool bwd, int grid, hipStream_t stream) {
  return dtype == DLT_BF16 ? swat_pick<bf16_t>(a, bwd, grid, stream) : swat_pick<f16_t>(a, bwd, grid, stream);
}
