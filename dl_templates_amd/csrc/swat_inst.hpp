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
  hipLaunchKernelGGL(kern, dim3(grid), dim3(SWAT_THREADS), lds, stream, a);
  dlt_timing_after(stream);
  DLT_CHECK_LAUNCH("marching tile-window forward launch");
  return DLT_OK;
}

template <typename TIO, int NTB, int WC, int WR>
int swat_launch_bwd(const SwatArgs& a, int grid, hipStream_t stream) {
  typedef Swat<DLT_D, NTB, WC, WR> C;
  if constexpr (Swab<DLT_D, NTB, WC, WR>::USED) {   // one launch where HBM is the bound (figures at swat_bwd_kernel)
    typedef Swab<DLT_D, NTB, WC, WR> CB;
    auto kern = swat_bwd_kernel<TIO, DLT_D, NTB, WC, WR>;
    const int rc = dlt_ensure_lds(reinterpret_cast<const void*>(kern), CB::LDS);
    if (rc != DLT_OK) return rc;
    SwatArgs b = a;
    b.nstrips = (a.g.XLq + 16 * CB::SB - 1) / (16 * CB::SB);
    const void* const ring_p[4] = {a.k, a.v, a.q, a.d_o};
    const int64_t* const ring_s[4] = {a.ks, a.vs, a.qs, a.dos};
    for (int t = 0; t < 4; t++) {
      b.ring_p[t] = ring_p[t];
      for (int i = 0; i < 5; i++) b.ring_s[t][i] = ring_s[t][i];
    }
    const int64_t cols = (int64_t)a.B * a.H * b.nstrips;
    dlt_band_plan(a.g.TR, cols, dlt_device_cus(), b.band, b.nbands);
    if (cols * b.nbands > 0x7fffffff) return dlt_set_error(DLT_ERR_UNSUPPORTED, "attention: grid too large");
    dlt_timing_before(DLT_K_BWD_KV, stream);
    hipLaunchKernelGGL(kern, dim3((unsigned)(cols * b.nbands)), dim3(CB::THREADS), CB::LDS, stream, b);
    dlt_timing_after(stream);
    DLT_CHECK_LAUNCH("marching tile-window backward launch");
    return DLT_OK;
  } else {
  // dQ first: it produces the delta vector the dK/dV kernel consumes
  auto kq = swat_bwd_q_kernel<TIO, DLT_D, NTB, WC, WR>;
  auto kkv = swat_bwd_kv_kernel<TIO, DLT_D, NTB, WC, WR>;
  int rc = dlt_ensure_lds(reinterpret_cast<const void*>(kq), C::RING);
  if (rc == DLT_OK) rc = dlt_ensure_lds(reinterpret_cast<const void*>(kkv), C::RING + C::SCAL);
  if (rc != DLT_OK) return rc;
  dlt_timing_before(DLT_K_BWD_Q, stream);
  hipLaunchKernelGGL(kq, dim3(grid), dim3(SWAT_THREADS), C::RING, stream, a);
  dlt_timing_after(stream);
  DLT_CHECK_LAUNCH("marching tile-window dQ launch");
  dlt_timing_before(DLT_K_BWD_KV, stream);
  hipLaunchKernelGGL(kkv, dim3(grid), dim3(SWAT_THREADS), C::RING + C::SCAL, stream, a);
  dlt_timing_after(stream);
  DLT_CHECK_LAUNCH("marching tile-window dK/dV launch");
  return DLT_OK;
  }
}

template <typename TIO>
int swat_pick(const SwatArgs& a, bool bwd, int grid, hipStream_t stream) {
#define DLT_SWAT(NTB, WC, WR) return bwd ? swat_launch_bwd<TIO, NTB, WC, WR>(a, grid, stream) : swat_launch_fwd<TIO, NTB, WC, WR>(a, grid, stream)
  const int ntb = a.g.S / 16;
  if (ntb == 2) DLT_SWAT(2, 1, 1);
  if (a.g.WR == 1) {
    if (a.g.WC == 1) DLT_SWAT(1, 1, 1);
    DLT_SWAT(1, 2, 1);
  }
#if DLT_D == 32
  if (a.g.WC == 1) DLT_SWAT(1, 1, 2);
  DLT_SWAT(1, 2, 2);
#endif
  return dlt_set_error(DLT_ERR_UNSUPPORTED, "marching tile-window kernels: no instantiation for this window");
#undef DLT_SWAT
}
}  // namespace

int DLT_CAT(dlt_swat_launch_, DLT_D)(const SwatArgs& a, int dtype, bool bwd, int grid, hipStream_t stream) {
  return dtype == DLT_BF16 ? swat_pick<bf16_t>(a, bwd, grid, stream) : swat_pick<f16_t>(a, bwd, grid, stream);
}
