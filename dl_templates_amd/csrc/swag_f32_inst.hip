// Instantiations and launcher of the fp32 marching forward kernel.
#include "swag_f32_kernel.hpp"

namespace {
template <int NCH, int NCG>
int run(const SwagArgs& a, int grid, hipStream_t stream) {
  auto kern = swag_fwd_f32_kernel<32, NCH, NCG>;
  constexpr int lds = SwagF<32, NCH, NCG>::RING;
  const int rc = dlt_ensure_lds(reinterpret_cast<const void*>(kern), lds);
  if (rc != DLT_OK) return rc;
  dlt_timing_before(DLT_K_FWD, stream);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(512), lds, stream, a);
  dlt_timing_after(stream);
  DLT_CHECK_LAUNCH("marching fp32 token-grid forward launch");
  return DLT_OK;
}
template <int NCH>
int pick(const SwagArgs& a, int ncg, int grid, hipStream_t stream) {
  return ncg == 2 ? run<NCH, 2>(a, grid, stream) : ncg == 3 ? run<NCH, 3>(a, grid, stream) : run<NCH, 4>(a, grid, stream);
}
}  // namespace

int dlt_swag_launch_f32(const SwagArgs& a, int nch, int ncg, int grid, hipStream_t stream) {
  return nch == 2 ? pick<2>(a, ncg, grid, stream) : nch == 3 ? pick<3>(a, ncg, grid, stream) : pick<4>(a, ncg, grid, stream);
}
