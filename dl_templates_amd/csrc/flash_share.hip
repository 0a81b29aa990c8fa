// Second launch of the dense flash passes whose streamed side is split over workgroups (FlashShare): the partial rows of an own
// token are summed in the order of the shares, so that results depend on the split alone and not on timing.
//
// Bound by latency and HBM / memory-side cache: a thread takes 8 dims of one row, requests all its pieces at once (the number of
// shares is a template argument) and stores 16 bytes.
#include "flash_kernel.hpp"

namespace {

// one tensor of partial rows and where their sum goes
struct ShareOut {
  const float* part;
  void* out;
  int64_t st[4];
  float mul;
  int32_t L, d, vec;   // rows per (batch, head), head dim
  int64_t items;       // pieces of 8 dims
};

template <int S>
DLT_DEV void share_load(const float* part, int64_t step, f32x4 (&lo)[S], f32x4 (&hi)[S]) {
#pragma unroll
  for (int s = 0; s < S; s++) {
    lo[s] = *reinterpret_cast<const f32x4*>(part + s * step);
    hi[s] = *reinterpret_cast<const f32x4*>(part + s * step + 4);
  }
}

struct ShareItem { int bh, row, d0; };
DLT_DEV ShareItem share_item(const ShareOut& o, uint32_t id) {
  const uint32_t pieces = (uint32_t)o.d >> 3, r = id / pieces;
  ShareItem it;
  it.d0 = 8 * (int)(id - r * pieces);
  it.bh = (int)(r / (uint32_t)o.L);
  it.row = (int)(r - (uint32_t)it.bh * (uint32_t)o.L);
  return it;
}

template <typename TIO, int S>
__global__ __launch_bounds__(256) void flash_share_fwd_kernel(const ShareOut o, int H, float* lse, int64_t ls0, int64_t ls1, int64_t ls2, float scale) {
  const uint32_t id = blockIdx.x * 256u + threadIdx.x;
  if (id >= o.items) return;
  const ShareItem it = share_item(o, id);
  const int64_t row0 = (int64_t)it.bh * S * o.L + it.row;
  const float* ml = o.part + (o.items / (o.d >> 3)) * S * o.d;   // behind the rows
  f32x4 lo[S], hi[S];
  float2 w[S];
#pragma unroll
  for (int s = 0; s < S; s++) w[s] = *reinterpret_cast<const float2*>(ml + 2 * (row0 + (int64_t)s * o.L));
  share_load<S>(o.part + row0 * o.d + it.d0, (int64_t)o.L * o.d, lo, hi);
  float m = -INFINITY, l = 0.f;
  f32x4 a = {0.f, 0.f, 0.f, 0.f}, b = a;
#pragma unroll
  for (int s = 0; s < S; s++) {
    float f1, f2;
    flash_merge(m, w[s].x, scale, f1, f2);
    l = flash_add(l, f1, w[s].y, f2);
#pragma unroll
    for (int j = 0; j < 4; j++) {
      a[j] = flash_add(a[j], f1, lo[s][j], f2);
      b[j] = flash_add(b[j], f1, hi[s][j], f2);
    }
  }
  const float inv = l > 0.f ? fast_rcp(l) : 0.f;
  const float v[8] = {a[0] * inv, a[1] * inv, a[2] * inv, a[3] * inv, b[0] * inv, b[1] * inv, b[2] * inv, b[3] * inv};
  const int bb = it.bh / H, h = it.bh - bb * H;
  Io<TIO, TIO>::store8(reinterpret_cast<TIO*>(o.out) + bb * o.st[0] + h * o.st[1] + it.row * o.st[2] + it.d0 * o.st[3], v, o.vec != 0, o.st[3], 8);
  if (it.d0 == 0) store_stream4(lse + bb * ls0 + h * ls1 + it.row * ls2, flash_lse2(m, scale, l));
}

// workgroups [0, split) sum `x`, the others `y`
template <typename TIO, int S>
__global__ __launch_bounds__(256) void flash_share_grad_kernel(const ShareOut x, const ShareOut y, uint32_t split, int H) {
  const bool first = blockIdx.x < split;
  const ShareOut& o = first ? x : y;
  const uint32_t id = (blockIdx.x - (first ? 0u : split)) * 256u + threadIdx.x;
  if (id >= o.items) return;
  const ShareItem it = share_item(o, id);
  f32x4 lo[S], hi[S];
  share_load<S>(o.part + ((int64_t)it.bh * S * o.L + it.row) * o.d + it.d0, (int64_t)o.L * o.d, lo, hi);
  float v[8];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    float a = 0.f, b = 0.f;
#pragma unroll
    for (int s = 0; s < S; s++) { a += lo[s][j]; b += hi[s][j]; }
    v[j] = a * o.mul;
    v[4 + j] = b * o.mul;
  }
  const int bb = it.bh / H, h = it.bh - bb * H;
  Io<TIO, TIO>::store8(reinterpret_cast<TIO*>(o.out) + bb * o.st[0] + h * o.st[1] + it.row * o.st[2] + it.d0 * o.st[3], v, o.vec != 0, o.st[3], 8);
}

ShareOut share_out(const float* part, void* out, const int64_t (&st)[5], float mul, int bh, int L, int d, int vec) {
  ShareOut o;
  o.part = part; o.out = out; o.mul = mul; o.L = L; o.d = d; o.vec = vec;
  for (int i = 0; i < 4; i++) o.st[i] = st[i];
  o.items = (int64_t)bh * L * (d / 8);
  return o;
}
uint32_t share_blocks(const ShareOut& o) { return (uint32_t)((o.items + 255) / 256); }

static_assert(FLASH_SHARES_MAX == 8, "share_switch");
template <typename F>
int share_switch(int n, F&& f) {
  switch (n) {
    case 2: return f(std::integral_constant<int, 2>{});
    case 3: return f(std::integral_constant<int, 3>{});
    case 4: return f(std::integral_constant<int, 4>{});
    case 5: return f(std::integral_constant<int, 5>{});
    case 6: return f(std::integral_constant<int, 6>{});
    case 7: return f(std::integral_constant<int, 7>{});
    case 8: return f(std::integral_constant<int, 8>{});
    default: return dlt_set_error(DLT_ERR_UNSUPPORTED, "flash: %d shares of a streamed side", n);
  }
}

int share_grad(const ShareOut& x, const ShareOut& y, int n, int H, int dtype, int id, hipStream_t stream) {
  const uint32_t split = share_blocks(x), grid = split + share_blocks(y);
  return share_switch(n, [&](auto sc) {
    constexpr int S = decltype(sc)::value;
    dlt_timing_before(id, stream);
    if (dtype == DLT_BF16) hipLaunchKernelGGL((flash_share_grad_kernel<bf16_t, S>), dim3(grid), dim3(256), 0, stream, x, y, split, H);
    else hipLaunchKernelGGL((flash_share_grad_kernel<f16_t, S>), dim3(grid), dim3(256), 0, stream, x, y, split, H);
    dlt_timing_after(stream);
    DLT_CHECK_LAUNCH("flash: sum of shares");
    return DLT_OK;
  });
}

}  // namespace

int dlt_flash_share_fwd(const FlashArgs& a, int dtype, hipStream_t stream) {
  const ShareOut o = share_out(a.share.part, a.o, a.os, 1.f, a.B * a.H, a.Lq, a.dv, a.o_vec);
  return share_switch(a.share.n, [&](auto sc) {
    constexpr int S = decltype(sc)::value;
    dlt_timing_before(DLT_K_FWD, stream);
    if (dtype == DLT_BF16)
      hipLaunchKernelGGL((flash_share_fwd_kernel<bf16_t, S>), dim3(share_blocks(o)), dim3(256), 0, stream, o, a.H, a.lse, a.ls[0], a.ls[1], a.ls[2], a.scale_log2);
    else
      hipLaunchKernelGGL((flash_share_fwd_kernel<f16_t, S>), dim3(share_blocks(o)), dim3(256), 0, stream, o, a.H, a.lse, a.ls[0], a.ls[1], a.ls[2], a.scale_log2);
    dlt_timing_after(stream);
    DLT_CHECK_LAUNCH("flash forward: sum of shares");
    return DLT_OK;
  });
}
int dlt_flash_share_bwd_q(const FlashBwdArgs& a, int dtype, hipStream_t stream) {
  ShareOut none{};
  return share_grad(share_out(a.share_q.part, a.dq, a.dqs, a.sm_scale, a.B * a.H, a.Lq, a.dk_, a.dq_vec), none, a.share_q.n, a.H, dtype, DLT_K_BWD_Q, stream);
}
int dlt_flash_share_bwd_kv(const FlashBwdArgs& a, int dtype, hipStream_t stream) {
  const float* pv = a.share_kv.part + (int64_t)a.B * a.H * a.share_kv.n * a.Lk * a.dk_;
  return share_grad(share_out(a.share_kv.part, a.dk, a.dks, a.sm_scale, a.B * a.H, a.Lk, a.dk_, a.dk_vec),
                    share_out(pv, a.dv, a.dvs, 1.f, a.B * a.H, a.Lk, a.dv_, a.dv_vec), a.share_kv.n, a.H, dtype, DLT_K_BWD_KV, stream);
}
