// Fused output epilogues shared by the decode GEMV (gemv.hip) and the prefill MFMA GEMM (gemm.hip):
// one output element (batch row bb, virtual matrix row vn) with its pair partner (row vn ^ 1) for
// the epilogues that combine adjacent rows (SiLU-GLU gate/up, RoPE pairs).
#pragma once
#include "common.h"
#include "ops.h"

namespace omx {

// rotation of column d of a head in row bb
__device__ __forceinline__ void epi_angle(const GemvParams& P, int bb, int d, float& cs, float& sn) {
  if (P.rope) {
    const float2 t = ((const float2*)P.rope)[(long long)bb * (P.n_rot >> 1) + (d >> 1)];
    cs = t.x, sn = t.y;
  } else {
    sincosf((float)P.pos[bb] * P.inv_freq[d >> 1], &sn, &cs);
  }
}

// `zsel`: MoE selected-expert slot of this output (blockIdx.z in the GEMV), 0 otherwise.
// One epilogue kind per instantiation: kernels that unroll many outputs per thread (gemm_dq.hip)
// dispatch on P.epi once and keep the unrolled body small.
template <int E>
__device__ __forceinline__ void epi_apply_t(const GemvParams& P, int bb, int vn, float v, float pv, int zsel) {
  if constexpr (E == EPI_STORE) {
    if (P.bias) v += P.bias[vn];
    P.y[(long long)bb * P.ldy + vn] = v;
  } else if constexpr (E == EPI_ADD) {
    if (P.bias) v += P.bias[vn];
    if (P.expert_w) v *= P.expert_w[bb * P.n_sel + zsel];
    float* dst = P.y + (long long)bb * P.ldy + vn;
    if (P.expert_ids && P.n_sel > 1) atomicAdd(dst, v);
    else *dst += v;
  } else if constexpr (E == EPI_GELU) {
    if (P.bias) v += P.bias[vn];
    P.y[(long long)bb * P.ldy + vn] = gelu_tanh(v);
  } else if constexpr (E == EPI_GELU_ERF) {
    if (P.bias) v += P.bias[vn];
    P.y[(long long)bb * P.ldy + vn] = 0.5f * v * (1.f + erff(v * 0.70710678f));
  } else if constexpr (E == EPI_QGELU) {
    if (P.bias) v += P.bias[vn];
    P.y[(long long)bb * P.ldy + vn] = v / (1.f + __expf(-1.702f * v));
  } else if constexpr (E == EPI_GLU) {
    if ((vn & 1) == 0)  // even row = gate, odd row = up
      P.y[(long long)bb * P.ldy + (long long)zsel * P.y_sel_stride + vn / 2] = silu(v) * pv;
  } else if constexpr (E == EPI_GEGLU) {  // Gemma: gelu(gate) * up
    if ((vn & 1) == 0)
      P.y[(long long)bb * P.ldy + (long long)zsel * P.y_sel_stride + vn / 2] = gelu_tanh(v) * pv;
  } else {  // EPI_QKV
    const int Eq = P.Eq, Ekv = P.Ekv, D = P.D;
    int which, hh, d;
    if (vn < Eq) { which = 0; hh = vn / D; d = vn % D; }
    else if (vn < Eq + Ekv) { which = 1; hh = (vn - Eq) / D; d = (vn - Eq) % D; }
    else { which = 2; hh = (vn - Eq - Ekv) / D; d = (vn - Eq - Ekv) % D; }
    if (P.bias) v += P.bias[vn];
    float out = v;
    if (which < 2 && d < P.n_rot) {
      if (P.bias) pv += P.bias[vn ^ 1];
      float sn, cs;
      epi_angle(P, bb, d, cs, sn);
      out = (d & 1) ? (pv * sn + v * cs) : (v * cs - pv * sn);
    }
    if (which == 0) {
      P.y[(long long)bb * P.ldy + vn] = out;
    } else {
      const int slot = P.slot[bb];
      const long long blk = slot / P.bs, off = slot % P.bs;
      const long long idx = ((blk * P.n_kv + hh) * P.bs + off) * (P.Dc > 0 ? P.Dc : D) + d;
      // two explicit stores: a pointer select here is lowered to an indexed scratch array
      if (which == 1) kv_store(P.kc, idx, out, P.kv8);
      else kv_store(P.vc, idx, out, P.kv8);
    }
  }
}

// The same in two parts for kernels whose threads have many outputs: what an output needs from memory (a store before a load keeps
// the load behind it, so all of a thread's loads go first), then the rest. Experts (expert_ids) take epi_apply_t.
struct EpiOperands {
  float was;   // EPI_ADD: the sum so far
  float bias;
  int slot;    // EPI_QKV
};
template <int E>
__device__ __forceinline__ EpiOperands epi_fetch(const GemvParams& P, int bb, int vn) {
  EpiOperands f{0.f, 0.f, 0};
  if (E != EPI_GLU && E != EPI_GEGLU && P.bias) f.bias = P.bias[vn];
  if constexpr (E == EPI_ADD) f.was = P.y[(long long)bb * P.ldy + vn];
  if constexpr (E == EPI_QKV) f.slot = vn >= P.Eq ? P.slot[bb] : 0;
  return f;
}
template <int E>
__device__ __forceinline__ void epi_put(const GemvParams& P, int bb, int vn, float v, float pv, EpiOperands f) {
  if constexpr (E == EPI_GLU || E == EPI_GEGLU) {
    epi_apply_t<E>(P, bb, vn, v, pv, 0);
    return;
  }
  v += f.bias;
  if constexpr (E == EPI_QKV) {
    const int which = vn < P.Eq ? 0 : vn < P.Eq + P.Ekv ? 1 : 2, h0 = vn - (which > 0 ? P.Eq : 0) - (which > 1 ? P.Ekv : 0);
    const int hh = h0 / P.D, d = h0 - hh * P.D;
    if (which < 2 && d < P.n_rot) {
      if (P.bias) pv += P.bias[vn ^ 1];
      float sn, cs;
      epi_angle(P, bb, d, cs, sn);
      v = (d & 1) ? (pv * sn + v * cs) : (v * cs - pv * sn);
    }
    if (which == 0) {
      P.y[(long long)bb * P.ldy + vn] = v;
      return;
    }
    const bool p2 = (P.bs & (P.bs - 1)) == 0;  // blocks of a power of two rows: no division per output
    const long long blk = p2 ? f.slot >> (__ffs(P.bs) - 1) : f.slot / P.bs, off = f.slot - blk * P.bs;
    kv_store(which == 1 ? P.kc : P.vc, ((blk * P.n_kv + hh) * P.bs + off) * (P.Dc > 0 ? P.Dc : P.D) + d, v, P.kv8);
    return;
  }
  if constexpr (E == EPI_ADD) {
    if (P.expert_w) v *= P.expert_w[bb * P.n_sel];
    v += f.was;
  }
  if constexpr (E == EPI_GELU) v = gelu_tanh(v);
  if constexpr (E == EPI_GELU_ERF) v = 0.5f * v * (1.f + erff(v * 0.70710678f));
  if constexpr (E == EPI_QGELU) v = v / (1.f + __expf(-1.702f * v));
  P.y[(long long)bb * P.ldy + vn] = v;
}

__device__ __forceinline__ void epi_apply(const GemvParams& P, int bb, int vn, float v, float pv, int zsel) {
  switch (P.epi) {
    case EPI_STORE: epi_apply_t<EPI_STORE>(P, bb, vn, v, pv, zsel); break;
    case EPI_ADD: epi_apply_t<EPI_ADD>(P, bb, vn, v, pv, zsel); break;
    case EPI_GELU: epi_apply_t<EPI_GELU>(P, bb, vn, v, pv, zsel); break;
    case EPI_GLU: epi_apply_t<EPI_GLU>(P, bb, vn, v, pv, zsel); break;
    case EPI_GEGLU: epi_apply_t<EPI_GEGLU>(P, bb, vn, v, pv, zsel); break;
    case EPI_QKV: epi_apply_t<EPI_QKV>(P, bb, vn, v, pv, zsel); break;
    case EPI_GELU_ERF: epi_apply_t<EPI_GELU_ERF>(P, bb, vn, v, pv, zsel); break;
    case EPI_QGELU: epi_apply_t<EPI_QGELU>(P, bb, vn, v, pv, zsel); break;
  }
}

}  // namespace omx
