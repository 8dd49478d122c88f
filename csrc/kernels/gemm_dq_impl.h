// Prompt products on quantised weights, shared parts: Y[M][N] = epi(X[M][K] . W[N][K]^T) for M = prompt tokens, W
// in the resident layout v2 (no second weight copy, no fp16 weight scratch). gemm_dq_slots.h holds the tiles of 65 rows and more,
// gemm_rows.hip those of up to 64.
//
//  * K in STORAGE order. Layout v2 keeps each row's codes piece-major (piece t of super-block sb at byte (t * SB + sb) *
//    piece_bytes), so the row's code stream is one contiguous run. A dot product is invariant under a common permutation of K, so
//    the kernels walk K in exactly that stream order: K step ks is the 32 (64 for Q8_0) contiguous code bytes of pieces 2 ks, 2 ks + 1
//    of every weight row. The activations are written once per product in the same order by `prep_xp_kernel` (RMSNorm / LayerNorm
//    fused there), so X is a plain row-major [M][Kp] fp16 slab.
//  * Inside a piece the packed-fp16 dequant produces weights in the order lo(0,2,1,3, 4,6,5,7, ...), hi(same):
//    `(q >> {0,8,4,12}) & 0x000F000F | 0x64006400` is two exact halves 1024 + n per VALU op, then one v_pk_add (remove 1024) + one
//    v_pk_fma (scale, zero point).
// Parity: replaces llama.cpp's prefill matmul inside `ollama/ollama` (reference pkg/model/pod.go:10-12);
// numerics vs fp32 torch on the dequantised weights in tests/test_gemm_gpu.py (dq cases).
#pragma once
#include <stdexcept>

#include "common.h"
#include "epilogue.h"
#include "ops.h"

namespace omx {

namespace {

constexpr unsigned DQ_MAGIC = 0x64006400u;

typedef _Float16 dh2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
__device__ __forceinline__ dh2 dq_h2(unsigned v) { return __builtin_bit_cast(dh2, v); }
__device__ __forceinline__ unsigned dq_u(dh2 v) { return __builtin_bit_cast(unsigned, v); }
__device__ __forceinline__ dh2 dq_splat(float f) { return (dh2){(f16)f, (f16)f}; }
// (n + 1024) pairs -> (n - off') * s + c  (off' = 1024 + zero point)
__device__ __forceinline__ unsigned dq2(unsigned p, dh2 off, dh2 sc, dh2 c) {
  return dq_u((dq_h2(p) - off) * sc + c);
}
__device__ __forceinline__ unsigned dsel(const u32x4& v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }

// weight offsets (natural K) of the lo / hi 16-weight halves of piece t of super-block sb
template <int QT>
__host__ __device__ __forceinline__ int piece_off(int t, int sb, int g) {
  if constexpr (QT == QT_Q4_K || QT == QT_Q5_K) return 256 * sb + 64 * (t >> 1) + 16 * (t & 1) + 32 * g;
  else if constexpr (QT == QT_Q6_K) return 256 * sb + 128 * (t >> 2) + 16 * (t & 3) + 64 * g;
  else return 256 * sb + 32 * t + 16 * g;  // Q4_0 / Q8_0
}

// LDS place of element k of a staged row: the 16-B slot index xor bits of the super-block (and, where a piece's
// halves are 64 apart, of that bit), so that the four chunks of four neighbouring pieces, slots {0, 2, 8, 10}
// (Q4_K / Q5_K, Q6_K) or {0, 2, 4, 6} (Q4_0 / Q8_0) of as many super-blocks, cover all 16 slots of the banks
template <int QT>
__host__ __device__ __forceinline__ int prep_at(int k) {
  const int sb = k >> 8, hi = QT == QT_Q4_0 || QT == QT_Q8_0 ? 8 : 4;
  int m = (sb & 1) | ((sb & 2) ? hi : 0);
  if (QT == QT_Q6_K) m ^= (k >> 3) & 8;
  return k ^ (4 * m);
}

// ------------------------------------------------------------------------------------------------
// activations: x fp32 [B][ldx] -> (norm) -> fp16 [B][Kp] in storage order; one block per row.
// Stream position kp: piece P = kp / 32 (t = P / SB, sb = P % SB), slot p = kp % 32: half g = p / 16,
// byte i = 4 ((p & 15) / 4) + (0, 2, 1, 3)[p & 3] -> natural k = piece_off(t, sb, g) + i
// ROWS (gemm_rows.hip): [16-row tile][32-K piece][8-K run][row], so that a wave reads a run of 16 rows as one block
// (PREP_MAX_KP: the longest row that fits)
template <int QT, bool ROWS = false>
__global__ __launch_bounds__(256) void prep_xp_kernel(GemvParams P, f16* out, int Kp) {
  // The row is staged in LDS in natural order (coalesced reads of x), normed there in place (coalesced reads of the
  // weights), then every thread gathers its 8 stream positions and writes them as one 16-B store. Neighbouring
  // chunks of the stream are whole super-blocks apart, the same banks: prep_at() swaps 16-B slots inside each
  // super-block so that the gathers of 16 lanes take 16 different ones. What bounds it: its bytes, 6 per element.
  // Measured against gathers that met in the banks (four or eight at a time) and applied the norm's weights from
  // memory in stream order: 2,048 rows of 4,096 20.6 -> 15.1 us, of 11,008 31.4 -> 23.2; 500 tokens' 1,000 pairs of
  // 14,336 66 -> 48.
  extern __shared__ float xs[];  // [Kp]
  __shared__ float red[4];
  const int b = blockIdx.x, K = P.w.K, SB = Kp >> 8;
  const float* x = P.x + (long long)(P.moe_gather ? P.moe_rows[b] / P.n_sel : b) * P.ldx;  // routed pairs: their token's row
  const bool nrm = P.norm != NORM_NONE, lnb = P.norm == NORM_LAYER && P.norm_b;
  float s = 0.f, ss = 0.f;
  for (int i = threadIdx.x; i < K / 4; i += 256) {
    const f32x4 v = *(const f32x4*)(x + 4 * i);
    *(f32x4*)(xs + prep_at<QT>(4 * i)) = v;
    s += v.x + v.y + v.z + v.w;
    ss += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
  }
  for (int k = (K & ~3) + threadIdx.x; k < K; k += 256) {  // K % 4 tail
    const float v = x[k];
    xs[prep_at<QT>(k)] = v;
    s += v;
    ss += v * v;
  }
  if (nrm) {
    float mean = 0.f, rstd;
    ss = block_sum<256>(ss, red);
    if (P.norm == NORM_LAYER) {
      s = block_sum<256>(s, red);
      mean = s / K;
      rstd = rsqrtf(fmaxf(ss / K - mean * mean, 0.f) + P.eps);
    } else {
      rstd = rsqrtf(ss / K + P.eps);
    }
    for (int i = threadIdx.x; i < K / 4; i += 256) {  // each thread its own elements
      f32x4* p = (f32x4*)(xs + prep_at<QT>(4 * i));
      f32x4 v = (*p - mean) * rstd * *(const f32x4*)(P.norm_w + 4 * i);
      if (lnb) v += *(const f32x4*)(P.norm_b + 4 * i);
      *p = v;
    }
    for (int k = (K & ~3) + threadIdx.x; k < K; k += 256) {
      float v = (xs[prep_at<QT>(k)] - mean) * rstd * P.norm_w[k];
      if (lnb) v += P.norm_b[k];
      xs[prep_at<QT>(k)] = v;
    }
  }
  f16* o = ROWS ? out + (long long)(b & ~15) * Kp + 8 * (b & 15) : out + (long long)b * Kp;
  __syncthreads();
  // a 16-B output chunk is 8 CONSECUTIVE natural positions base .. base + 7 in the order
  // 0 2 1 3 4 6 5 7: two 16-B LDS reads, permuted in registers
  for (int c = threadIdx.x; c < Kp / 8; c += 256) {
    const int kp = 8 * c, pc = kp >> 5, p0 = kp & 31;
    const int t = pc / SB, sb = pc - t * SB;
    const int base = piece_off<QT>(t, sb, p0 >> 4) + 4 * ((p0 & 15) >> 2);
    f16x8 v;
    if (base + 8 <= K) {
      const f32x4 a = *(const f32x4*)(xs + prep_at<QT>(base)), b = *(const f32x4*)(xs + prep_at<QT>(base + 4));
      v = (f16x8){(f16)a.x, (f16)a.z, (f16)a.y, (f16)a.w, (f16)b.x, (f16)b.z, (f16)b.y, (f16)b.w};
    } else {  // the row's K padding (Q4_0 / Q8_0 with K % 256 != 0)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int r = j & 3, k = base + 4 * (j >> 2) + (r == 1 ? 2 : r == 2 ? 1 : r);
        v[j] = (f16)(k < K ? xs[prep_at<QT>(k)] : 0.f);
      }
    }
    *(f16x8*)(o + (ROWS ? 16 * kp : kp)) = v;
  }
}

// ------------------------------------------------------------------------------------------------
// one weight-row piece (32 codes) in registers: codes + the scale bytes it needs
template <int QT>
struct Piece {
  u32x4 a;                                   // 16 code bytes (Q8_0: first 16)
  u32x4 b;                                   // Q8_0: last 16 code bytes
  u32x4 m;                                   // Q4_K / Q5_K meta (d, dmin, scales12); Q6_K int8 scales
  u32x2 h;                                   // Q6_K high-bit pairs
  unsigned e;                                // Q5_K 5th bits; Q6_K / Q4_0 / Q8_0: fp16 d (low half)
};

// Q4_K / Q5_K 6-bit scale and min of sub-block j (no branch: j differs between the lanes of a wave)
__device__ __forceinline__ void k_scale(const u32x4& m, int j, float& sc, float& mn) {
  const float d = h2f(m.x & 0xFFFF), dmin = h2f(m.x >> 16);
  const int sh = 8 * (j & 3);
  const unsigned hi = (unsigned)-(j >> 2), a = m.y >> sh, b = m.z >> sh, e = m.w >> sh;
  const unsigned s = (a & 63u & ~hi) | (((e & 15u) | ((a >> 2) & 48u)) & hi);
  const unsigned n = (b & 63u & ~hi) | ((((e >> 4) & 15u) | ((b >> 2) & 48u)) & hi);
  sc = d * (float)s;
  mn = -dmin * (float)n;
}

// two of a piece's fp16 weights (dword 2 e + odd of its lo / hi half in stream order): q: code dword e (Q8_0: of that half), H: the
// piece's high bits (Q5_K: all, Q6_K: that half's), S, C: that half's scale and minimum
template <int QT>
__device__ __forceinline__ unsigned dq_word(unsigned q, unsigned H, int half, int e, int odd, dh2 S, dh2 C) {
  if constexpr (QT == QT_Q8_0) {  // bytes are offset-binary after ^ 0x80
    return dq2((((q >> (8 * odd)) & 0x00FF00FFu) | DQ_MAGIC) ^ 0x00800080u, dq_splat(1152.f), S, C);  // 1024 + 128
  } else {
    if (QT == QT_Q4_K || QT == QT_Q4_0) q ^= 0x80808080u;  // undo the signed-high-nibble repack
    unsigned v = ((q >> (4 * half + 8 * odd)) & 0x000F000Fu) | DQ_MAGIC;
    if constexpr (QT == QT_Q5_K) {  // 5th bit of weight 4e + j: byte j of H, bit e (lo) / 4 + e (hi)
      const int sh = 4 * half + 8 * odd + e - 4;
      v |= (sh >= 0 ? H >> sh : H << -sh) & 0x00100010u;
    }
    if constexpr (QT == QT_Q6_K) {  // high 2 bits of weight 4e + j: byte j, bits 2e..2e+1 of H -> bits 4..5
      const int sh = 8 * odd + 2 * e - 4;
      v |= (sh >= 0 ? H >> sh : H << -sh) & 0x00300030u;
    }
    return dq2(v, dq_splat(QT == QT_Q6_K ? 1056.f : QT == QT_Q4_0 ? 1032.f : 1024.f), S, C);  // 1024 + zero point
  }
}
// scale and minimum of half `half` of piece t; m: Q4_K / Q5_K meta, Q6_K: the half's int8 scale in the low byte of m.x; e: fp16 d
template <int QT>
__device__ __forceinline__ void dq_scale(const u32x4& m, unsigned e, int t, int half, dh2& S, dh2& C) {
  C = dq_splat(0.f);
  if constexpr (QT == QT_Q4_K || QT == QT_Q5_K) {
    float s, c;
    k_scale(m, 2 * (t >> 1) + half, s, c);
    S = dq_splat(s), C = dq_splat(c);
  } else if constexpr (QT == QT_Q6_K) {
    S = dq_splat(h2f((uint16_t)e) * (float)(int8_t)(m.x & 0xFF));
  } else {
    S = dq_splat(h2f((uint16_t)e));
  }
}

}  // namespace

}  // namespace omx
