// Weight-streaming products of a decode step's few rows (vy_rows.h) as launches of their own: y = act(x W^T + bias).
#include "vy_rows.h"

namespace {

using vy_rows::Dense;

// (32 and 48 rows: eight k-steps ahead instead of four, 6144 x 1024 7.1 -> 6.7 us)
template <int ACT, int MB, int NW, int NT, bool HALF = false>
__global__ __launch_bounds__(64 * NW) void rows_linear_kernel(Dense a) {
  __shared__ f32x4 red[vy_rows::DENSE_RED<NT, MB, NW>];
  vy_rows::dense<MB, NW, NT, HALF, ACT, NT == 2 || NT == 3 ? 8 : vy_rows::STEPS<NT, MB>>(a, red, blockIdx.x, a.K);
}

// K cut into slices of `len` columns: fp32 partial sums [slice][M][N]
template <int MB, int NT>
__global__ __launch_bounds__(256) void rows_parts_kernel(Dense a, int len, int tiles) {
  __shared__ f32x4 red[vy_rows::DENSE_RED<NT, MB>];
  const int slice = blockIdx.x / tiles, tile = blockIdx.x - slice * tiles, k0 = slice * len;
  a.x += k0;
  a.w += k0;
  a.y = (float*)a.y + (int64_t)slice * a.M * a.N;
  vy_rows::dense<MB, 4, NT>(a, red, tile, min(len, a.K - k0));
}

// Weight rows of a workgroup.  What one CU takes in (25 to 40 GB/s) sets the time, and a workgroup reads x -- 16 MB rows of K -- beside
// its weights: so the rows that make the fullest CU read least.  24 are one workgroup a CU where 16 are two on half of them.  32 rows,
// weights from HBM: 6144 x 1024 8.3 us on 16, 6.7 on 24, 6.9 on 32 (8.6 before dense() spread its last part over the waves); 8192 x 1024
// 8.4, 10.3, 6.9 (9.3); 6144 x 2048 14.5, 11.0, 11.5 (12.9); 12288 x 2048 15.7 on 48, 18.9 on 24 (19.4); 32000 x 1024 18.7 on 64, 20.1 on
// 32 (23.0).  Up to 16 rows x weighs half and wide products stream from HBM, so only 24 in place of 16 pays, up to 16384: 8 rows,
// 6144 x 1024 6.1 -> 5.2, 6144 x 2048 9.3 -> 8.5, 32000 x 1024 16.3 (24: 17.6).
template <int ACT, int MB>
void rows_go(const Dense& a, hipStream_t st) {
  // few workgroups with long rows: twice the waves each
  if (a.N <= 4096 && a.K >= 2048) {
    hipLaunchKernelGGL((rows_linear_kernel<ACT, MB, 8, 1>), dim3((unsigned)vy_cdiv(a.N, 16)), dim3(512), 0, st, a);
    return;
  }
  auto rounds = [&](int r) { return vy_cdiv(vy_cdiv(a.N, r), 256); };
  int best = 16;
  if constexpr (MB == 1) {
    if (a.N <= 16384 && rounds(24) < rounds(16)) best = 24;
  } else {
    for (const int r : {24, 32, 48, 64})
      if (rounds(r) * (16 * MB + r) < rounds(best) * (16 * MB + best)) best = r;
  }
  const dim3 grid((unsigned)vy_cdiv(a.N, best)), block(256);
  if (best == 16) hipLaunchKernelGGL((rows_linear_kernel<ACT, MB, 4, 1>), grid, block, 0, st, a);
  else if (best == 24) hipLaunchKernelGGL((rows_linear_kernel<ACT, MB, 4, 2, true>), grid, block, 0, st, a);
  else if constexpr (MB > 1) {
    if (best == 32) hipLaunchKernelGGL((rows_linear_kernel<ACT, MB, 4, 2>), grid, block, 0, st, a);
    else if (best == 48) hipLaunchKernelGGL((rows_linear_kernel<ACT, MB, 4, 3>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((rows_linear_kernel<ACT, MB, 4, 4>), grid, block, 0, st, a);
  }
}

template <int ACT>
void rows_of(const Dense& a, hipStream_t st) {
  if (a.M <= 16) rows_go<ACT, 1>(a, st);
  else rows_go<ACT, 2>(a, st);
}

}  // namespace

// internal (vy_hybrid.hip): bf16 y[M][N], 5 .. 32 rows of x (stride K) against w [N][K].  VY_ERR_UNSUPPORTED: other sizes.
int vy_rows_linear(const void* x, const void* w, const void* bias, int act, float act_arg, void* y, int64_t ldy, int64_t M, int64_t N,
                   int64_t K, hipStream_t st) {
  if (M < 5 || M > 32 || N > INT32_MAX || K > INT32_MAX || N < 16 || K < 8 || K % 8 || ldy % 8 || (uintptr_t)x % 16 || (uintptr_t)w % 16 ||
      (uintptr_t)y % 16 || (act != VY_ACT_NONE && act != VY_ACT_RELU2 && act != VY_ACT_SOFTCAP))
    return VY_ERR_UNSUPPORTED;
  const Dense a{(const bf16*)x, K, (int)M, (const bf16*)w, (int)N, (int)K, y, ldy, 0, (const bf16*)bias, act_arg};
  if (act == VY_ACT_RELU2) rows_of<VY_ACT_RELU2>(a, st);
  else if (act == VY_ACT_SOFTCAP) rows_of<VY_ACT_SOFTCAP>(a, st);
  else rows_of<VY_ACT_NONE>(a, st);
  VY_CHECK_LAUNCH("vy_rows_linear");
  return VY_OK;
}

// internal (vy_hybrid.hip): the product of a sublayer's output, whose rows vy_residual_norm_parts adds to the stream: fp32 partial sums
// parts[slice][M][N] of K cut into that many slices (returned; 0: other sizes).  A product with as few columns as the stream has 32
// or 64 workgroups of 32 columns, and what one CU takes in (25 to 40 GB/s) sets its time; slices bring the workgroups to 256, and
// wider tiles halve the times x is read: 64 columns where they still are 256 workgroups.  32 rows, 1024 x 6144: 23.3 -> 6.8 us;
// 2048 x 8192: 11.4 (32 columns: 12.7); 2048 x 12288: 43.2 -> 16.6 (17.9); 1024 x 1024: 6.1 -> 3.5; 8 rows: 13.3 -> 5.4, 24.8 -> 14.2,
// 4.2 -> 3.2 (weights from HBM).  A slice keeps at least 128 columns: 8 waves' lines.
int vy_rows_parts(const void* x, const void* w, float* parts, int64_t M, int64_t N, int64_t K, hipStream_t st) {
  if (M < 5 || M > 32 || N < 512 || N > 4096 || K > INT32_MAX || K < 1024 || K % 8 || (uintptr_t)x % 16 || (uintptr_t)w % 16 ||
      (uintptr_t)parts % 16)
    return 0;
  const int slices = N <= 1024 ? 8 : N <= 2048 ? (K >= 8192 ? 8 : 4) : 2;
  const int len = (int)((K + slices - 1) / slices + 63) / 64 * 64;
  if ((slices - 1) * (int64_t)len >= K) return 0;
  const bool wide = (N + 63) / 64 * slices >= 256;
  const int tiles = (int)((N + (wide ? 63 : 31)) / (wide ? 64 : 32));
  const Dense a{(const bf16*)x, K, (int)M, (const bf16*)w, (int)N, (int)K, parts, N, 1, nullptr, 0.f};
  const dim3 grid(tiles * slices), block(256);
  if (M <= 16 && wide) hipLaunchKernelGGL((rows_parts_kernel<1, 4>), grid, block, 0, st, a, len, tiles);
  else if (M <= 16) hipLaunchKernelGGL((rows_parts_kernel<1, 2>), grid, block, 0, st, a, len, tiles);
  else if (wide) hipLaunchKernelGGL((rows_parts_kernel<2, 4>), grid, block, 0, st, a, len, tiles);
  else hipLaunchKernelGGL((rows_parts_kernel<2, 2>), grid, block, 0, st, a, len, tiles);
  return slices;
}
