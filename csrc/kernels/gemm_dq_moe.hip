// Routed experts of a prompt: the grouped form of the dequantising tiles (gemm_dq_slots.h), all weight types. Tiles come from a
// device-side table {expert, first row, rows} over (token, expert) pairs sorted by expert (X in that order), the expert's matrix at
// row expert * N; outputs go to the sorted row (gate / up) or, with moe_scatter, to the pair's own row, unweighted (moe_combine sums
// a token's pairs). One launch for all experts, and the routed counts stay on the device.
#include "gemm_dq_slots.h"

namespace omx {
namespace {

// An expert's rows in tiles of 256 and a rest; a rest of up to 128 rows takes a tile of half the products. What bounds it: as the
// plain tiles, and the padding of the rests. Measured, 1,000 rows through the top 2 of 8 experts of 14,336 x 4,096, 128 x 128 tiles
// of eight waves -> this: gate / up 873 -> 680 us, down 528 -> 367 (Q4_K), 718 -> 543 (Q6_K); 128 x 256 tiles alone 712, 496, 813.
template <int QT>
__global__ __launch_bounds__(256, 1) void dq_moe_kernel(GemvParams P, const f16* __restrict__ X, int Kp) {
  const int nt = (P.w.N + 255) / 256, nwg = *P.moe_ntiles * nt;
  if ((int)blockIdx.x >= nwg) return;
  const int wg = ring::xcd_range(blockIdx.x, nwg);
  const int *t = P.moe_tiles + 3 * (wg / nt), m0 = t[1], rows = t[2], n0 = wg % nt * 256;
  const long long erow = (long long)t[0] * P.w.N;
  if (rows > 128) ds_tile<QT, 8, 2, true>(P, X, Kp, 1, 0, m0, m0 + rows, n0, erow);
  else ds_tile<QT, 4, 2, true>(P, X, Kp, 1, 0, m0, m0 + rows, n0, erow);
}

// The same in tiles of 128 x 128, a table's tile in two halves, two blocks a CU: for up to 128 rows an expert, where the products
// are bound by the weights' way in and 256 columns a block leave CUs without one (8 experts x 4,096 columns: 128 blocks). us, 128 x
// 128 tiles of eight waves / the kernel above / this, 8 experts, top 2: down 4,096 x 14,336 (Q4_K), (Q6_K), gate / up 28,672 x 4,096:
//   17 rows 200 / 207 / 132, 241 / 314 / 185, 318 / 271 / 254;  260 rows 210 / 215 / 149, 246 / 347 / 226, 336 / 292 / 275
//   400 rows 214 / 227 / 171, 251 / 361 / 241, 345 / 303 / 288
//   600 rows - / 307 / 282, - / 429 / 429, - / 469 / 551;  1,000 rows - / 341 / 424, - / 477 / 672, - / 704 / 808
template <int QT>
__global__ __launch_bounds__(256, 2) void dq_moe_half_kernel(GemvParams P, const f16* __restrict__ X, int Kp) {
  const int nt = (P.w.N + 127) / 128, nwg = *P.moe_ntiles * 2 * nt;
  if ((int)blockIdx.x >= nwg) return;
  const int wg = ring::xcd_range(blockIdx.x, nwg), u = wg / nt;
  const int *t = P.moe_tiles + 3 * (u >> 1), m0 = t[1] + 128 * (u & 1), rows = t[2] - 128 * (u & 1);
  if (rows <= 0) return;
  ds_tile<QT, 4, 1, true>(P, X, Kp, 1, 0, m0, m0 + min(rows, 128), wg % nt * 128, (long long)t[0] * P.w.N);
}

template <int QT>
void run_moe(const GemvParams& P, f16* xp, int Kp, hipStream_t s) {
  static_assert(DQ_MOE_TILE_M == 256, "rows of the tiles above");
  hipLaunchKernelGGL(prep_xp_kernel<QT>, dim3(P.B), dim3(256), (size_t)Kp * sizeof(float), s, P, xp, Kp);
  const int experts = P.moe_max_tiles - (P.B + DQ_MOE_TILE_M - 1) / DQ_MOE_TILE_M;  // (the table's bound: a rest for each)
  if (P.B <= 128 * experts) {
    hipLaunchKernelGGL(dq_moe_half_kernel<QT>, dim3(P.moe_max_tiles * 2 * ((P.w.N + 127) / 128)), dim3(256), (ds_lds<4, 1>()), s, P, xp,
                       Kp);
    return;
  }
  hipLaunchKernelGGL(dq_moe_kernel<QT>, dim3(P.moe_max_tiles * ((P.w.N + 255) / 256)), dim3(256), (ds_lds<8, 2>()), s, P, xp, Kp);
}

}  // namespace

void run_dq_moe(const GemvParams& P, f16* xp, int Kp, hipStream_t s) {
  switch (P.w.qtype) {
    case QT_Q4_K: run_moe<QT_Q4_K>(P, xp, Kp, s); break;
    case QT_Q5_K: run_moe<QT_Q5_K>(P, xp, Kp, s); break;
    case QT_Q6_K: run_moe<QT_Q6_K>(P, xp, Kp, s); break;
    case QT_Q4_0: run_moe<QT_Q4_0>(P, xp, Kp, s); break;
    default: run_moe<QT_Q8_0>(P, xp, Kp, s); break;
  }
}

}  // namespace omx
