// Weight-streaming products of a decode step's few rows (vy_rows.h) as launches of their own: y = act(x W^T + bias).
#include "vy_rows.h"

namespace {

using vy_rows::Dense;

// D: lines of K that a wave has on their way (vy_rows::share_lds)
template <int ACT, int MB, int NW, int NT, bool HALF, int D>
__global__ __launch_bounds__(64 * NW) void rows_linear_kernel(Dense a) {
  __shared__ __attribute__((aligned(16))) char lds[vy_rows::DENSE<MB, NW, NT, HALF, D>];
  vy_rows::dense<MB, NW, NT, HALF, ACT, D>(a, lds, blockIdx.x, a.K);
}

// K cut into slices of `len` columns: fp32 partial sums [slice][M][N]
template <int MB, int NT>
__global__ __launch_bounds__(256) void rows_parts_kernel(Dense a, int len, int tiles) {
  __shared__ __attribute__((aligned(16))) char lds[vy_rows::DENSE<MB, 4, NT, false, 2>];
  const int slice = blockIdx.x / tiles, tile = blockIdx.x - slice * tiles, k0 = slice * len;
  a.x += k0;
  a.w += k0;
  a.y = (float*)a.y + (int64_t)slice * a.M * a.N;
  vy_rows::dense<MB, 4, NT>(a, lds, tile, min(len, a.K - k0));
}

// Weight rows of a workgroup.  What one CU takes in sets the time, and a workgroup reads x -- 16 MB rows of K -- beside its weights: so the
// rows that make the fullest CU read least, as long as 64 of them bring everything in one round; wider products (vocabularies) have 64
// rows, beside 32 rows of x 48, and two lines on their way instead of three, so that two workgroups share a CU.  With the operands by
// whole lines through LDS instead of 16 rows a load straight into the product's registers (which a CU takes in at 25 to 30 KB a
// microsecond: 4.5 of the 6.8 us below): 32 rows, 6144 x 1024 6.8 -> 5.2 us, 8192 x 1024 7.1 -> 5.7, 2048 x 1024 5.5 -> 3.7, 6144 x 2048
// 11.5 -> 7.8, 12288 x 2048 16.7 -> 12.6, 16384 x 2048 21.5 -> 14.6, 32000 x 1024 20.0 -> 15.3 (64 rows a workgroup 17.6), 32000 x 2048 38.2 ->
// 27.7; 8 rows 5.4 -> 4.6, 6.6 -> 5.2, 4.3 -> 3.4, 8.8 -> 6.9, 14.7 -> 12.0, 20.1 -> 13.8, 18.8 -> 13.9, 34.9 -> 24.8.  The same bits.
// Wide and beside 32 rows of x, up to 256 columns of K are one line a wave, so room for one: 40 KB, four workgroups on a CU.  32 rows, 38360 x 64,
// 6.4 -> 4.8 us (5.5 straight into registers), 27072 x 168 6.5 -> 5.2 (6.6), 17000 x 256 5.2 -> 4.9 (6.6).
template <int ACT, int MB>
void rows_go(const Dense& a, hipStream_t st) {
  // few workgroups with long rows: twice the waves each (32 rows, 2048 x 2048 8.2 -> 4.9 us)
  if (a.N <= 4096 && a.K >= 2048) {
    hipLaunchKernelGGL((rows_linear_kernel<ACT, MB, 8, 1, false, 2>), dim3((unsigned)vy_cdiv(a.N, 16)), dim3(512), 0, st, a);
    return;
  }
  auto rounds = [&](int r) { return vy_cdiv(vy_cdiv(a.N, r), 256); };
  int best = 16;
  for (const int r : {24, 32, 48, 64})
    if (rounds(r) * (16 * MB + r) < rounds(best) * (16 * MB + best)) best = r;
  if (rounds(64) > 1) best = MB == 1 ? 64 : 48;
  const dim3 grid((unsigned)vy_cdiv(a.N, best)), block(256);
  if (best == 16) hipLaunchKernelGGL((rows_linear_kernel<ACT, MB, 4, 1, false, 3>), grid, block, 0, st, a);
  else if (best == 24) hipLaunchKernelGGL((rows_linear_kernel<ACT, MB, 4, 2, true, 3>), grid, block, 0, st, a);
  else if (best == 32) hipLaunchKernelGGL((rows_linear_kernel<ACT, MB, 4, 2, false, 3>), grid, block, 0, st, a);
  else if (best == 48) {
    if constexpr (MB == 2) {
      if (rounds(64) > 1 && a.K <= 256) {
        hipLaunchKernelGGL((rows_linear_kernel<ACT, MB, 4, 3, false, 1>), grid, block, 0, st, a);
        return;
      }
    }
    hipLaunchKernelGGL((rows_linear_kernel<ACT, MB, 4, 3, false, 2>), grid, block, 0, st, a);
  }
  else hipLaunchKernelGGL((rows_linear_kernel<ACT, MB, 4, 4, false, 2>), grid, block, 0, st, a);
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
// or 64 workgroups of 32 columns, and what one CU takes in sets its time; slices bring the workgroups to 256, and
// wider tiles halve the times x is read: 64 columns where they still are 256 workgroups.  32 rows, 1024 x 6144: 23.3 -> 6.8 us;
// 2048 x 8192: 11.4 (32 columns: 12.7); 2048 x 12288: 43.2 -> 16.6 (17.9); 1024 x 1024: 6.1 -> 3.5; 8 rows: 13.3 -> 5.4, 24.8 -> 14.2,
// 4.2 -> 3.2 (weights from HBM); with whole lines through LDS 5.1, 9.4, 12.7, 3.3 and 4.6, 11.3, 3.0.  A slice keeps at least 128 columns:
// 8 waves' lines.
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
