// out = x W^T + bias for the few rows of a lightly loaded draft step (one or two requests
// of 16 slots): the DiT's projections, whose weights are read once and used by 32 rows at
// most (flashmap/modeling_flashmap.py:118-192 runs them as torch Linears).
//
// Bound: HBM, the weights (8 MB for a 2048 x 2048 projection, 34 MB for an MLP half);
// each call is so short that what matters is how many of those bytes are in flight at
// once. A workgroup owns 16 rows of W (output columns) and its wavefronts (16, or 8) split the
// reduction, so that a 2048 x 2048 projection has all of its weights in flight over 128
// CUs; the partials meet in LDS in a fixed order.
//   wavefront: out^T[n][m] += v_mfma_f32_16x16x32_bf16, A = W rows n, B = x rows m, both
//              as loaded (16 bytes per lane: row lane % 16, k 8 * (lane / 16))
//   LDS:       (wavefront, row block, lane) fp32x4, summed by one wavefront per row block
// bias is added in fp32 before the one rounding to bf16.
// Measured (weights from HBM, 16 rows, this kernel and the library's): 2048 x 2048 6.7 us
// (1.25 TB/s) and 11.1, 8192 x 2048 12.6 (2.7 TB/s) and 14.5; one row reads x from one line
// and takes 5.5 and 9.6 us: past the launch it is the reads of x, as many bytes as the
// weights and all of them from L2, that a second row block doubles.
#include <stdint.h>

#include <type_traits>

#include "fm_device.h"
#include "fm_host.h"

namespace fm {

constexpr int LIN_ROWS = 16;  // rows of W per workgroup

struct LinearArgs {
  const uint16_t *x, *w, *bias;
  uint16_t *out;
  int64_t xs, ws, os;  // row strides (elements)
  int32_t rows, n, k;
};

template <int MB, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void linear_rows_kernel(const LinearArgs a) {
  __shared__ f32x4_t part[WAVES][MB][64];
  const int lane = threadIdx.x & 63, wave = wave_id();
  const int r = lane & 15, g = lane >> 4;
  const int32_t n0 = (int32_t)blockIdx.x * LIN_ROWS;
  const int32_t steps = a.k >> 5;
  const int32_t s0 = (int32_t)((int64_t)steps * wave / WAVES), s1 = (int32_t)((int64_t)steps * (wave + 1) / WAVES);
  // Rows past the end read the last one: their results are not stored.
  const uint16_t *wr = a.w + (int64_t)(n0 + r < a.n ? n0 + r : a.n - 1) * a.ws + 8 * g;
  const uint16_t *xr[MB];
#pragma unroll
  for (int b = 0; b < MB; ++b) xr[b] = a.x + (int64_t)(16 * b + r < a.rows ? 16 * b + r : a.rows - 1) * a.xs + 8 * g;
  f32x4_t acc[MB];
#pragma unroll
  for (int b = 0; b < MB; ++b) acc[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // `live` of the G k-steps from s count; the loads of the others repeat the last one.
  auto take = [&](auto group, int32_t s, int32_t live) {
    constexpr int G = decltype(group)::value;
    u32x4_t wf[G], xf[MB][G];
#pragma unroll
    for (int i = 0; i < G; ++i) {
      const int64_t at = 32 * (int64_t)(s + (i < live ? i : live - 1));
      wf[i] = load16(wr + at);
#pragma unroll
      for (int b = 0; b < MB; ++b) xf[b][i] = load16(xr[b] + at);
    }
#pragma unroll
    for (int i = 0; i < G; ++i)
      if (i < live) {
#pragma unroll
        for (int b = 0; b < MB; ++b) acc[b] = mfma_16x16x32(wf[i], xf[b][i], acc[b]);
      }
  };
  int32_t s = s0;
  if constexpr (MB == 1)
    for (; s + 8 <= s1; s += 8) take(std::integral_constant<int, 8>{}, s, 8);
  for (; s + 4 <= s1; s += 4) take(std::integral_constant<int, 4>{}, s, 4);
  if (s < s1) take(std::integral_constant<int, 4>{}, s, s1 - s);
#pragma unroll
  for (int b = 0; b < MB; ++b) part[wave][b][lane] = acc[b];
  __syncthreads();
  if (wave >= MB) return;
  f32x4_t sum = part[0][wave][lane];
#pragma unroll
  for (int w = 1; w < WAVES; ++w) sum += part[w][wave][lane];
  // Lane: row m of out, columns n0 + 4 g .. + 3.
  const int32_t m = 16 * wave + r, n = n0 + 4 * g;
  if (m >= a.rows) return;
  uint16_t *dst = a.out + m * a.os + n;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (n + i >= a.n) break;
    float v = sum[i];
    if (a.bias != nullptr) v += bf16_to_f32(a.bias[n + i]);
    dst[i] = (uint16_t)(pack_bf16x2(v, 0.f) & 0xffffu);
  }
}

}  // namespace fm

extern "C" int fm_linear_rows(const void *x, int64_t x_stride, const void *weight, int64_t w_stride, const void *bias,
                              void *out, int64_t out_stride, int32_t rows, int32_t n, int32_t k,
                              void *stream) {
  using namespace fm;
  FM_REQUIRE(rows >= 0 && n >= 0 && k > 0, "bad sizes: rows=%d n=%d k=%d", rows, n, k);
  if (rows == 0 || n == 0) return FM_OK;
  if (rows > 32 || k % 32 != 0)
    return fail(FM_ERR_UNSUPPORTED, "%d rows of %d: at most 32 rows, a multiple of 32 values", rows, k);
  if (n > 1 << 26)  // a launch counts at most 2^32 threads
    return fail(FM_ERR_UNSUPPORTED, "%d output columns: at most 2^26", n);
  FM_REQUIRE(x && weight && out, "NULL tensor pointer");
  FM_REQUIRE((((uintptr_t)x | (uintptr_t)weight) & 15) == 0, "x / weight must be 16-byte aligned");
  FM_REQUIRE(x_stride % 8 == 0 && w_stride % 8 == 0 && x_stride >= k && w_stride >= k && out_stride >= n,
             "row strides must cover a row (x / weight: multiples of 8 elements)");
  LinearArgs a{(const uint16_t *)x, (const uint16_t *)weight, (const uint16_t *)bias, (uint16_t *)out,
               x_stride, w_stride, out_stride, rows, n, k};
  DeviceInfo info;
  const int rc = device_info(&info);
  if (rc != FM_OK) return rc;
  const unsigned tiles = (unsigned)((n + LIN_ROWS - 1) / LIN_ROWS);
  // More than a workgroup per CU: 8 wavefronts, so that several fit; fewer: 16, for the
  // loads in flight.
  const int waves = tiles <= (unsigned)info.cus ? 16 : 8;
  auto launch = [&](auto mb) {
    constexpr int MB = decltype(mb)::value;
    auto *kernel = waves == 16 ? linear_rows_kernel<MB, 16> : linear_rows_kernel<MB, 8>;
    kernel<<<dim3(tiles), dim3(64 * waves), 0, (hipStream_t)stream>>>(a);
  };
  if (rows <= 16)
    launch(std::integral_constant<int, 1>{});
  else
    launch(std::integral_constant<int, 2>{});
  FM_CHECK_HIP(hipGetLastError());
  return FM_OK;
}
