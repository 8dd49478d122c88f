// Prompt portions of fewer rows than a tile of the prefill GEMM (gemm_dq_slots.h): Y[M][N] = epi(X[M][K] . W[N][K]^T) for
// M <= 64, W in the resident layout v2, X in storage order (prep_xp_kernel, as for the larger GEMMs).
//
// What bounds it: the weights' way from memory; the products need a fifth of that time. So a block takes 16 NT weight rows
// over all of K, its 8 waves split K, and a weight goes from memory straight to the registers of the one lane that
// dequantises it: the four lane groups of a wave own one super-block each, lane (n, group) holds a 32-weight piece of row n,
// and the piece's four runs of 8 weights are the B operands of four v_mfma_f32_16x16x32_f16 per row tile (K runs in an order
// of its own, the same for the activations, which lane (m, group) finds in 256-byte runs of 16 rows). The next pieces are in
// flight while one is multiplied. No LDS until the waves' partial sums meet at the end; the epilogue follows in the same launch.
// (64 x 128 tiles through LDS left two thirds of the chip idle at N = 4096, and split K into slabs with a second launch.)
// The activations come from L2 once per block, in an order that makes a wave's reads of them whole lines (row by row they cost
// 16 lines a request and more time than the weights).
// Beside the bytes, the address unit: a lane's 16 bytes are alone in their line of the wave's request, so a scale block is loaded
// once for the four pieces of a unit instead of with each (and its scales worked out once): gate_up 32.6 -> 27 us. Weights two steps
// ahead instead of one were no faster.
// Measured, Llama-2-7B Q4_K_M at 33 rows, tile kernel + finalize -> this: gate_up 82 -> 27 us, q k v (Q4_K) 49 -> 20, o 34 ->
// 12, down (Q6_K) 48 -> 22; with 65 rows and more the 128-row tiles of the larger GEMM are ahead.
#include <type_traits>

#include "gemm_dq_impl.h"
#include "wave_shuffle.h"

namespace omx {

namespace {

template <int QT, int MT, int NT, int NW>
__global__ __launch_bounds__(64 * NW, 2) void dq_rows_kernel(GemvParams P, const f16* __restrict__ X, int Kp) {
  extern __shared__ float red[];  // [NW][mt * NT][256]
  const QMat& w = P.w;
  const int M = P.B, N = w.N, SB = Kp >> 8;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 15, g = lane >> 4, n0 = blockIdx.x * 16 * NT;
  const int mt = (M + 15) >> 4;  // row tiles of 16
  int row[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) row[j] = min(n0 + 16 * j + fr, N - 1);  // rows past the end repeat the last (not stored)
  f32x4 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
  // a unit: four super-blocks (one per lane group) x four of their eight pieces, 4 odd .. 4 odd + 3; units go to the waves in turn,
  // so a wave's are all of one half. A lane's scales serve the whole unit: loaded once, worked out once per sub-block
  const int odd = wave & 1, units = 2 * ((SB + 3) >> 2), mine = (units - wave + NW - 1) / NW;
  constexpr bool KM = QT == QT_Q4_K || QT == QT_Q5_K;
  auto block = [&](int n) { return 4 * ((wave + NW * n) >> 1) + g; };  // super-block of this lane group in the wave's unit n
  struct Scales {
    u32x4 m;
    unsigned e;
  };
  Piece<QT> pa[NT], pb[NT];
  Scales sa[NT], sb_[NT];
  u32x4 xa[MT][4], xb[MT][4];
  auto load_scales = [&](int n, Scales (&c)[NT]) {
    const int sb = min(block(n), SB - 1);
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const long long at = (long long)row[j] * SB + sb;
      if constexpr (KM) c[j].m = *(const u32x4*)(w.s1 + 16 * at);
      if constexpr (QT == QT_Q6_K) {
        const u32x2 v = *(const u32x2*)(w.s2 + 16 * at + 8 * odd);
        c[j].m.x = v.x, c[j].m.y = v.y;
        c[j].e = *(const uint16_t*)(w.s3 + 2 * at);
      }
      if constexpr (QT == QT_Q4_0 || QT == QT_Q8_0) {
        const u32x2 v = *(const u32x2*)(w.s1 + 16 * at + 8 * odd);
        c[j].m.x = v.x, c[j].m.y = v.y;
      }
    }
  };
  auto load = [&](int n, int k, Piece<QT> (&p)[NT], u32x4 (&a)[MT][4]) {  // piece 4 odd + k of unit n
    const int pc = (4 * odd + k) * SB + min(block(n), SB - 1);
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const long long r = (long long)row[j] * SB;
      p[j].a = *(const u32x4*)(w.s0 + r * (QT == QT_Q8_0 ? 256 : 128) + (QT == QT_Q8_0 ? 32LL : 16LL) * pc);
      if constexpr (QT == QT_Q8_0) p[j].b = *(const u32x4*)(w.s0 + r * 256 + 32LL * pc + 16);
      if constexpr (QT == QT_Q5_K) p[j].e = *(const unsigned*)(w.s2 + r * 32 + 4LL * pc);
      if constexpr (QT == QT_Q6_K) p[j].h = *(const u32x2*)(w.s1 + r * 64 + 8LL * pc);
    }
    const f16* x = X + 512 * pc + 8 * fr;  // (rows past the end hold anything: not stored)
#pragma unroll
    for (int i = 0; i < MT; ++i)
      if (i < mt) {
#pragma unroll
        for (int c = 0; c < 4; ++c) a[i][c] = *(const u32x4*)(x + i * 16 * Kp + 128 * c);
      }
  };
  dh2 S[NT][2], C[NT][2];
  auto multiply = [&](int n, auto kc, const Piece<QT> (&p)[NT], const Scales (&sc)[NT], u32x4 (&a)[MT][4]) {
    constexpr int k = decltype(kc)::value;
    // a lane group past the last super-block multiplies zeros: what it loaded is the last one's again, whose weights its row
    // multiplies anyway
    if (block(n) >= SB) {
#pragma unroll
      for (int i = 0; i < MT; ++i)
        if (i < mt) {
#pragma unroll
          for (int c = 0; c < 4; ++c) a[i][c] = (u32x4){0u, 0u, 0u, 0u};
        }
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) {
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        u32x4 m = sc[j].m;
        unsigned e = sc[j].e;
        if constexpr (QT == QT_Q6_K) m.x = (half ? m.y : m.x) >> (8 * k);
        if constexpr (QT == QT_Q4_0 || QT == QT_Q8_0) e = (k < 2 ? m.x : m.y) >> (16 * (k & 1));
        if (!KM || (k & 1) == 0) dq_scale<QT>(m, e, 4 * odd + k, half, S[j][half], C[j][half]);
        unsigned o[8];
#pragma unroll
        for (int x = 0; x < 8; ++x)
          o[x] = dq_word<QT>(dsel(QT == QT_Q8_0 && half ? p[j].b : p[j].a, x >> 1), QT == QT_Q6_K ? (half ? p[j].h.y : p[j].h.x) : p[j].e,
                             half, x >> 1, x & 1, S[j][half], C[j][half]);
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const f16x8 b = __builtin_bit_cast(f16x8, (u32x4){o[4 * c], o[4 * c + 1], o[4 * c + 2], o[4 * c + 3]});
#pragma unroll
          for (int i = 0; i < MT; ++i)
            if (i < mt)
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a[i][2 * half + c]), b, acc[i][j], 0, 0, 0);
        }
      }
    }
  };
  if (mine > 0) {
    typedef std::integral_constant<int, 0> k0;
    typedef std::integral_constant<int, 1> k1;
    typedef std::integral_constant<int, 2> k2;
    typedef std::integral_constant<int, 3> k3;
    load_scales(0, sa);
    load(0, 0, pa, xa);
    for (int n = 0; n < mine; ++n) {
      load(n, 1, pb, xb);
      multiply(n, k0{}, pa, sa, xa);
      load(n, 2, pa, xa);
      multiply(n, k1{}, pb, sa, xb);
      load(n, 3, pb, xb);
      multiply(n, k2{}, pa, sa, xa);
      const int next = min(n + 1, mine - 1);  // the last one: a repeated load that nobody multiplies
      load_scales(next, sb_);
      load(next, 0, pa, xa);
      multiply(n, k3{}, pb, sa, xb);
#pragma unroll
      for (int j = 0; j < NT; ++j) sa[j] = sb_[j];
    }
  }
#pragma unroll
  for (int i = 0; i < MT; ++i)
    if (i < mt) {
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) red[(wave * mt * NT + i * NT + j) * 256 + 64 * r + lane] = acc[i][j][r];
    }
  auto out = [&](auto ec) {  // element r of lane l: row 4 (l >> 4) + r, column l & 15; what the elements need from memory goes first
    constexpr int E = decltype(ec)::value, XN = (MT * NT * 4 + NW - 1) / NW;
    EpiOperands pre[XN];
    auto place = [&](int u, int& x, int& m, int& n) {
      x = tid + 64 * NW * u;
      const int f = x >> 8, r = (x >> 6) & 3, l = x & 63;
      m = 16 * (f / NT) + 4 * (l >> 4) + r, n = n0 + 16 * (f % NT) + (l & 15);
      return m < M && n < N;
    };
    int x, m, n;
#pragma unroll
    for (int u = 0; u < XN; ++u)
      if (place(u, x, m, n)) pre[u] = epi_fetch<E>(P, m, n + P.row_offset);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < XN; ++u) {
      const bool in = place(u, x, m, n);
      if (x >= mt * NT * 256) break;
      float v = 0.f;
#pragma unroll
      for (int k = 0; k < NW; ++k) v += red[k * mt * NT * 256 + x];
      const float pv = xor_shfl<1>(v);  // the row pair's partner: the next lane
      if (in) epi_put<E>(P, m, n + P.row_offset, v, pv, pre[u]);
    }
  };
  switch (P.epi) {
    case EPI_STORE: out(std::integral_constant<int, EPI_STORE>{}); break;
    case EPI_ADD: out(std::integral_constant<int, EPI_ADD>{}); break;
    case EPI_GELU: out(std::integral_constant<int, EPI_GELU>{}); break;
    case EPI_GLU: out(std::integral_constant<int, EPI_GLU>{}); break;
    case EPI_GEGLU: out(std::integral_constant<int, EPI_GEGLU>{}); break;
    case EPI_QKV: out(std::integral_constant<int, EPI_QKV>{}); break;
    case EPI_GELU_ERF: out(std::integral_constant<int, EPI_GELU_ERF>{}); break;
    default: out(std::integral_constant<int, EPI_QGELU>{}); break;
  }
}

template <int QT, int MT, int NT, int NW = 8>
void launch_rows(const GemvParams& P, const f16* xp, int Kp, hipStream_t s) {
  const int mt = (P.B + 15) / 16;
  hipLaunchKernelGGL((dq_rows_kernel<QT, MT, NT, NW>), dim3((P.w.N + 16 * NT - 1) / (16 * NT)), dim3(64 * NW),
                     (size_t)NW * mt * NT * 1024, s, P, xp, Kp);
}

template <int QT>
void run_rows(const GemvParams& P, f16* xp, int Kp, hipStream_t s) {
  hipLaunchKernelGGL((prep_xp_kernel<QT, true>), dim3(P.B), dim3(256), (size_t)Kp * sizeof(float), s, P, xp, Kp);
  const int N = P.w.N;
  // columns per block by what still leaves a block for most CUs (Q4_K, 48 rows: N = 22016 43 us at 48 columns, 49 at 64, 47
  // at 32; 6144 17.9 at 32, 21.5 at 48, 22.8 at 16; 4096 14.7 at 16, 16.9 at 32); at 64 rows three column tiles do not fit
  // the registers. Over 22 matrices of 512 .. 32,000 rows, five weight types and 16 .. 64 rows the launch takes 0.51 of the
  // tile kernel's time on average, and no point takes more
  // Four waves a block instead of eight where 257 to 512 blocks of 48 columns then run at once, two on each of the 256 CUs (33 rows,
  // us, four / eight: Q4_K x 4,096 N = 12,032 23.0 / 21.3, 12,800 29.0 / 33.2, 22,016 30.9 / 34.5, 24,576 31.6 / 35.7; Q6_K 25.9 / 25.6,
  // 36.8 / 41.7, 39.3 / 44.1, 39.7 / 45.1). Past 512 blocks four were ahead too when this was measured again (28,672: Q4_K 43.2 / 47.9,
  // Q6_K 54.2 / 61.7); the line was drawn at the round.
  const bool wide = N >= 48 * 208, middle = N >= 32 * 160;
  if (P.B <= 48) {
    if (wide && N > 48 * 256 && N <= 48 * 512) launch_rows<QT, 3, 3, 4>(P, xp, Kp, s);
    else if (wide) launch_rows<QT, 3, 3>(P, xp, Kp, s);
    else if (middle) launch_rows<QT, 3, 2>(P, xp, Kp, s);
    else launch_rows<QT, 3, 1>(P, xp, Kp, s);
  } else {
    if (middle) launch_rows<QT, 4, 2>(P, xp, Kp, s);
    else launch_rows<QT, 4, 1>(P, xp, Kp, s);
  }
}

}  // namespace

bool dq_rows(const GemvParams& P, hipStream_t s) {
  if (!dq_gemm_enabled() || P.B < 2 || P.B > 64 || !P.xws || P.expert_ids || P.moe_tiles || P.w.K % 8) return false;
  const int Kp = ((P.w.K + 255) >> 8) * 256;
  const long long cap = P.xws_elems ? P.xws_elems : (long long)P.B * P.w.K;
  if ((long long)((P.B + 15) & ~15) * Kp > cap || Kp > PREP_MAX_KP) return false;  // whole 16-row tiles
  f16* xp = (f16*)P.xws;
  switch (P.w.qtype) {
    case QT_Q4_K: run_rows<QT_Q4_K>(P, xp, Kp, s); break;
    case QT_Q5_K: run_rows<QT_Q5_K>(P, xp, Kp, s); break;
    case QT_Q6_K: run_rows<QT_Q6_K>(P, xp, Kp, s); break;
    case QT_Q4_0: run_rows<QT_Q4_0>(P, xp, Kp, s); break;
    case QT_Q8_0: run_rows<QT_Q8_0>(P, xp, Kp, s); break;
    default: return false;
  }
  count_launch(LC_GEMM_ROWS);
  return true;
}

}  // namespace omx
