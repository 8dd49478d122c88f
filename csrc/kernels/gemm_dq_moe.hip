// Routed experts of a prompt: the grouped form of the stream-order dequant GEMM (gemm_dq_impl.h), all weight types
#include "gemm_dq_impl.h"

namespace omx {
namespace {

template <int QT>
void run_moe(const GemvParams& P, f16* xp, int Kp, hipStream_t s) {
  constexpr int BM = MOE_TILE_M, BN = 128;  // BM: the tiles of P.moe_tiles
  hipLaunchKernelGGL(prep_xp_kernel<QT>, dim3(P.B), dim3(256), (size_t)Kp * sizeof(float), s, P, xp, Kp);
  hipLaunchKernelGGL((dq_gemm_ring_kernel<QT, BM, BN, 2, 4, true>), dim3(P.moe_max_tiles * ((P.w.N + BN - 1) / BN)), dim3(DQ_NT),
                     (dq_lds<BM, BN>()), s, P, xp, Kp, 1);
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
