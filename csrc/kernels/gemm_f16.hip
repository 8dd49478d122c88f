// fp16 weights (QT_F16, the vision tower) times prompt-sized activations: norm and conversion to fp16 in prep_f16_kernel, then
// the register-ring tiles of gemm_ring.h. What bounds it: 577 rows make few tiles, so a product lasts as long as its chain of
// K steps; tiles of 64 x 64 or 128 x 64 with K split over a block's waves keep a step at 0.16 .. 0.45 us, and nothing is left
// to add up in a second launch.
// Measured against 128-row tiles with K split over blocks and a finalize launch, 23 layers of 1,024 x 4,096, 577 rows: products
// 2.47 -> 2.06 ms, with the preparation 3.18 -> 2.53.
#include "common.h"
#include "epilogue.h"
#include "gemm_ring.h"
#include "ops.h"

namespace omx {
namespace {

// Rows of activations to fp16, normed on the way, K padded to Kp with zeros; a wave per row (four rows a block), or per 1,024
// columns of one where no statistics are needed. What bounds it: one round trip to memory, so a row's loads are all on their way
// at once, the norm's weights with them; rows of up to 1,024 stay in registers, longer ones are read again for the conversion.
// VEC: all rows start on 16 bytes. Measured against a block per row, element by element, 577 rows: of 1,024 normed 7.6 -> 5.5 us,
// of 4,096 not normed 7.9 -> 4.6.
template <bool NORM, bool VEC>
__global__ __launch_bounds__(256) void prep_f16_kernel(GemvParams P, f16* out, int Kp) {
  constexpr int NP = 4, CH = 256 * NP;
  const int K = P.w.K, lane = threadIdx.x & 63, b = 4 * blockIdx.x + (threadIdx.x >> 6);
  if (b >= P.B) return;
  const float* x = P.x + (long long)b * P.ldx;
  f16* o = out + (long long)b * Kp;
  auto load = [&](const float* p, int k) {
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (VEC && k + 4 <= K) return *(const f32x4*)(p + k);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (k + j < K) v[j] = p[k + j];
    return v;
  };
  f32x4 v[NP], w[NP], c[NP];
  auto fetch = [&](int k0, bool xs, bool ws) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int k = k0 + 256 * i + 4 * lane;
      if (xs) v[i] = load(x, k);
      if (NORM && ws) w[i] = load(P.norm_w, k), c[i] = P.norm == NORM_LAYER && P.norm_b ? load(P.norm_b, k) : f32x4{0.f, 0.f, 0.f, 0.f};
    }
  };
  float mean = 0.f, rstd = 1.f;
  const int first = NORM ? 0 : CH * blockIdx.y, last = NORM ? Kp : min(Kp, first + CH);
  fetch(first, true, true);
  if constexpr (NORM) {
    float s = 0.f, ss = 0.f;
    for (int k0 = 0;;) {
#pragma unroll
      for (int i = 0; i < NP; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) s += v[i][j], ss += v[i][j] * v[i][j];
      k0 += CH;
      if (k0 >= K) break;
      fetch(k0, true, false);
    }
    ss = wave_sum(ss);
    if (P.norm == NORM_LAYER) {
      mean = wave_sum(s) / K;
      rstd = rsqrtf(fmaxf(ss / K - mean * mean, 0.f) + P.eps);
    } else {
      rstd = rsqrtf(ss / K + P.eps);
    }
  }
  for (int k0 = first; k0 < last; k0 += CH) {
    if (NORM && K > CH) fetch(k0, true, true);
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int k = k0 + 256 * i + 4 * lane;
      f16x4 h;
#pragma unroll
      for (int j = 0; j < 4; ++j) h[j] = k + j < K ? (f16)(NORM ? (v[i][j] - mean) * rstd * w[i][j] + c[i][j] : v[i][j]) : (f16)0.f;
      if (k < Kp) *(f16x4*)(o + k) = h;
    }
  }
}

template <int E>
struct Out {
  GemvParams P;
  typedef EpiOperands Pre;
  __device__ __forceinline__ Pre fetch(int m, int n) const { return epi_fetch<E>(P, m, n + P.row_offset); }
  __device__ __forceinline__ void put(int m, int n, float v, float pv, Pre f) const { epi_put<E>(P, m, n + P.row_offset, v, pv, f); }
};

template <int E>
void run(const GemvParams& P, const ring::Operands& o, hipStream_t s) {
  using ring::launch_ring;
  const Out<E> e{P};
  const ring::Group g{};
  const int m64 = (o.M + 63) / 64, m128 = (o.M + 127) / 128;
  switch (ring::choose_tile(o.M, o.N, o.K, 1)) {
    case 1: launch_ring<ring::F16, Out<E>, 256, 128, 4, 2, 1, 2, false>(o, e, g, (o.M + 255) / 256, s); break;
    case 2: launch_ring<ring::F16, Out<E>, 128, 128, 2, 2, 2, 4, false>(o, e, g, m128, s); break;
    case 3: launch_ring<ring::F16, Out<E>, 128, 128, 2, 2, 2, 2, false>(o, e, g, m128, s); break;
    case 4: launch_ring<ring::F16, Out<E>, 128, 64, 2, 1, 4, 4, false>(o, e, g, m128, s); break;
    default: launch_ring<ring::F16, Out<E>, 64, 64, 2, 1, 4, 4, false>(o, e, g, m64, s); break;
  }
}

}  // namespace

void run_dq_f16(const GemvParams& P, f16* xp, int Kp, hipStream_t s) {
  const bool norm = P.norm != NORM_NONE;
  const bool vec = P.ldx % 4 == 0 && (((uintptr_t)P.x | (norm ? (uintptr_t)P.norm_w | (uintptr_t)P.norm_b : 0)) & 15) == 0;
  const dim3 grid((P.B + 3) / 4, norm ? 1 : (Kp + 1023) / 1024);
  if (norm && vec) hipLaunchKernelGGL((prep_f16_kernel<true, true>), grid, dim3(256), 0, s, P, xp, Kp);
  else if (norm) hipLaunchKernelGGL((prep_f16_kernel<true, false>), grid, dim3(256), 0, s, P, xp, Kp);
  else if (vec) hipLaunchKernelGGL((prep_f16_kernel<false, true>), grid, dim3(256), 0, s, P, xp, Kp);
  else hipLaunchKernelGGL((prep_f16_kernel<false, false>), grid, dim3(256), 0, s, P, xp, Kp);
  const ring::Operands o{(const uint16_t*)xp, Kp, (const uint16_t*)P.w.s0, P.B, P.w.N, Kp};
  switch (P.epi) {
    case EPI_STORE: run<EPI_STORE>(P, o, s); break;
    case EPI_ADD: run<EPI_ADD>(P, o, s); break;
    case EPI_GELU: run<EPI_GELU>(P, o, s); break;
    case EPI_GLU: run<EPI_GLU>(P, o, s); break;
    case EPI_GEGLU: run<EPI_GEGLU>(P, o, s); break;
    case EPI_QKV: run<EPI_QKV>(P, o, s); break;
    case EPI_GELU_ERF: run<EPI_GELU_ERF>(P, o, s); break;
    default: run<EPI_QGELU>(P, o, s); break;
  }
}

}  // namespace omx
