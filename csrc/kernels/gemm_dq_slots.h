// Dequantising products of prompts on large tiles: Y[M][N] = epi(X[M][K] . W[N][K]^T), X in storage order (prep_xp_kernel), W in the
// resident layout v2. Only the activations pass through LDS: each of a block's four waves owns 32 TN weight rows, dequantises them
// straight into the fragments of its own products and multiplies them with all of the tile's 32 TM activation rows.
//
// What bounds it: at 256 x 256 a step of 64 K is 64 products of 32 x 32 x 16 for each wave, 2,048 cycles, and everything else has to
// fit beside them. One wave a SIMD issues an instruction every 4 cycles (8 if it needs the one before; measured), so a step has
// room for some 380 others: it has 250. The LDS moves 160 KiB of 256 that it could (the eight waves with both operands in LDS that
// this replaces needed all 256). What is left are the chip's power, which holds the clock of a full chip down (1.8 us a step against
// 1.3 with half the CUs idle; fp16 operands without any dequantisation take 1.57), and prologue and epilogue, some 20 us.
//  * Slots. A step is four phases (8 of the 32 weights of a lane's piece each), a phase TM * TN slots of one product, and a slot also
//    holds one or two instructions of every other kind: a fragment for the next phase, a share of its dequantisation (in stages
//    whose instructions do not wait for each other), of the next step's scales, of the next activations. Scheduling barriers keep
//    the slots apart; left to itself the compiler bunches them.
//  * Places in memory advance in scalar registers (buffer descriptors): no vector instruction computes an address.
//  * Loads return in order, so all of them are as old as the oldest: activations wait two steps in registers, weights four.
//  * A lane holds whole pieces: lanes 0 .. 31 piece 2 s of 32 rows, lanes 32 .. 63 piece 2 s + 1, and the fragments of phase p take
//    quarter p of both, so a piece's scales are worked out once. The activations' fragments are read in the same order.
// Measured, eight waves with both operands in LDS -> this, Llama-2-7B at 2,048 rows in the model: gate_up (Q4_K) 481 -> 418 us,
// q k v 412 -> 283, o 119 -> 93, down 245 -> 185; 509 rows x 28,672 x 4,096 (Q5_K) 170 -> 140. Over 65 .. 2,048 rows x 7 matrices x
// 3 types 0.79 of the time, no point slower.
#pragma once
#include <type_traits>

#include "gemm_dq_impl.h"
#include "gemm_dq_places.h"
#include "gemm_ring.h"

namespace omx {

namespace {

using ring::each;
template <int I>
using ic = std::integral_constant<int, I>;

constexpr int DS_RING = 4;  // steps that a weight piece is loaded ahead
template <int TM, int TN>
constexpr size_t ds_lds() {  // two buffers of activations, or 32 rows of results
  const size_t a = 2 * 32 * TM * 128, e = 32 * (128 * TN + 4) * 4 + 128 * TM;
  return a > e ? a : e;
}
constexpr bool slab_kind(int e) { return e < 0; }

// the tile of rows m0 .. M - 1 (up to 32 TM of them) and columns n0 .. (up to 128 TN), slice z of sk of K; erow: W's row 0
template <int QT, int TM, int TN, bool GROUPED>
__device__ __forceinline__ void ds_tile(const GemvParams& P, const f16* __restrict__ X, int Kp, int sk, int z, int m0, int M, int n0,
                                        long long erow) {
  constexpr int BM = 32 * TM, BN = 128 * TN, NS = TM * TN, XI = TM / 4, R = DS_RING, BUF = BM * 128;
  constexpr bool KM = QT == QT_Q4_K || QT == QT_Q5_K, K8 = QT == QT_Q8_0, Q6 = QT == QT_Q6_K;
  static_assert(TM % 4 == 0 && NS >= 4, "every phase stages as many pieces");
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const QMat& w = P.w;
  const int N = w.N, SB = Kp >> 8;
  const int ks0 = 4 * (int)((long long)z * SB / sk), ks1 = 4 * (int)((long long)(z + 1) * SB / sk), kl = ks1 - 1;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int fr = lane & 31, fq = lane >> 5, xr = tid >> 3, xc = tid & 7;
  // operands through buffer descriptors of the tile's rows: places advance in scalar registers
  auto rsrc = [](const void* p, long long bytes) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, (int)(unsigned)(bytes < 0xFFFFFFF0LL ? bytes : 0xFFFFFFF0LL), 0x00027000);
  };
  auto b128 = [](auto r, unsigned v, unsigned s) { return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, v, s, 0)); };
  const int rows = min(BM, M - m0);
  const auto bx = rsrc(X + (long long)m0 * Kp, 2LL * rows * Kp);
  const long long wf = (erow + n0) * SB, wl = (long long)(N - n0) * SB;  // super-blocks before the tile's rows, from there to the end
  constexpr int CB = K8 ? 256 : 128, B1 = Q6 ? 64 : 16, B2 = QT == QT_Q5_K ? 32 : Q6 ? 16 : 0, B3 = Q6 ? 2 : 0;  // bytes per super-block
  const auto bc = rsrc(w.s0 + wf * CB, wl * CB), b1 = rsrc(w.s1 + wf * B1, wl * B1);
  const auto b2 = rsrc(B2 ? w.s2 + wf * B2 : w.s1, wl * B2), b3 = rsrc(B3 ? w.s3 + wf * B3 : w.s1, wl * B3);
  unsigned ox[TM], rw[TN];
#pragma unroll
  for (int i = 0; i < TM; ++i) ox[i] = ds_x_at(min(xr + 32 * i, rows - 1), Kp, xc);
#pragma unroll
  for (int j = 0; j < TN; ++j) rw[j] = (unsigned)min(32 * TN * wave + 32 * j + fr, N - 1 - n0) * (unsigned)SB;
  u32x4 xv[2][TM];
  Piece<QT> wv[R][TN];
  unsigned wt[R];
  // the next piece to load is piece lt of super-block lsb: step s takes pieces 2 s (lanes 0 .. 31) and 2 s + 1 of the stream
  unsigned lt = (unsigned)(2 * ks0 + fq) / (unsigned)SB, lsb = 2 * ks0 + fq - lt * SB;
  const unsigned da = SB == 1 ? 0 : 2, db = SB == 1 ? 2 : 0;
  auto load_x = [&](int ks, auto b, auto c) {
    constexpr int C = decltype(c)::value;
    xv[decltype(b)::value][C] = b128(bx, ox[C], ds_x_step(ks, kl));
  };
  auto load_w = [&](int ks, int j, int part, int slot) {
    Piece<QT>& q = wv[slot][j];
    if (part == 0) {
      const unsigned at = ds_w_at(rw[j], CB, fq);
      q.a = b128(bc, at, ds_w_step(ks, kl, CB));
      if constexpr (K8) q.b = b128(bc, at + 16, ds_w_step(ks, kl, CB));
      if constexpr (QT == QT_Q5_K) q.e = __builtin_amdgcn_raw_buffer_load_b32(b2, ds_w_at(rw[j], 32, fq), ds_w_step(ks, kl, 32), 0);
      if constexpr (Q6)
        q.h = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(b1, ds_w_at(rw[j], 64, fq), ds_w_step(ks, kl, 64), 0));
    } else {
      const unsigned at = rw[j] + lsb;
      if constexpr (KM) q.m = b128(b1, 16 * at, 0);
      if constexpr (Q6) {
        q.m = b128(b2, 16 * at, 0);
        q.e = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(b3, 2 * at, 0, 0);
      }
      if constexpr (K8 || QT == QT_Q4_0) q.e = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(b1, ds_scale_at(at, lt), 0, 0);
      if (j == TN - 1) {  // two pieces of the stream further
        wt[slot] = lt;
        lsb += da, lt += db;
        const bool over = lsb >= (unsigned)SB;
        lsb = over ? lsb - SB : lsb;
        lt += over;
      }
    }
  };
  const int xw = xr * 128 + 16 * (xc ^ ((xr >> 1) & 7));
  const int fa = fr * 128 + 16 * ((4 * fq) ^ ((fr >> 1) & 7));  // chunk 4 fq + kk of a fragment row: this, with 16 kk flipped in
  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  f16x8 a[TM];
  unsigned o[2][TN][4], hb[TN][4];  // weight fragments of a phase and the next; high bits on their way there
  f16 S[2][TN][2], C[2][TN][2];     // scales and minima of a piece's halves, of a step and the next
  unsigned g[4], h[3], tt;
  float fs[4];
  auto stage = [&](auto phase, auto item, auto b, int ks, int buf) {  // piece of step ks to LDS, that of ks + 2 into its registers
    constexpr int c = decltype(phase)::value * XI + decltype(item)::value;
    *(u32x4*)(smem + buf * BUF + xw + 4096 * c) = xv[decltype(b)::value][c];
    load_x(ks + 2, b, ic<c>{});
  };
  auto read = [&](int i, int kk, int buf) { a[i] = *(const f16x8*)(smem + buf * BUF + (fa ^ (16 * kk)) + 4096 * i); };
  // scales of slot r's piece j, set n, in nine stages of independent instructions (k_scale and dq_scale, both halves at once)
  constexpr int SST = 9;
  auto scale = [&](auto rc, auto nc, auto jc, auto st) {
    constexpr int r = decltype(rc)::value, n = decltype(nc)::value, j = decltype(jc)::value, I = decltype(st)::value;
    const Piece<QT>& p = wv[r][j];
    if constexpr (KM) {
      if constexpr (I == 0) tt = wt[r], g[3] = 8 * (tt & 2), g[2] = -(int)(tt >> 2);
      else if constexpr (I == 1) g[0] = p.m.y >> g[3], g[1] = p.m.z >> g[3];
      else if constexpr (I == 2) tt = p.m.w >> g[3], h[0] = g[0] >> 2, h[1] = g[1] >> 2;
      else if constexpr (I == 3) g[0] &= 0x3F3Fu, g[1] &= 0x3F3Fu, h[2] = tt >> 4;
      else if constexpr (I == 4) h[0] &= 0x3030u, h[1] &= 0x3030u, tt &= 0x0F0Fu, h[2] &= 0x0F0Fu;
      else if constexpr (I == 5) h[0] |= tt, h[1] |= h[2];
      else if constexpr (I == 6) g[0] = (h[0] & g[2]) | (g[0] & ~g[2]), g[1] = (h[1] & g[2]) | (g[1] & ~g[2]);
      else if constexpr (I == 7) {
        fs[0] = (float)(g[0] & 0xFFu), fs[1] = (float)((g[0] >> 8) & 0xFFu);
        fs[2] = (float)(g[1] & 0xFFu), fs[3] = (float)((g[1] >> 8) & 0xFFu);
      } else {
        const float d = h2f(p.m.x & 0xFFFF), dm = -h2f(p.m.x >> 16);
        S[n][j][0] = (f16)(d * fs[0]), S[n][j][1] = (f16)(d * fs[1]);
        C[n][j][0] = (f16)(dm * fs[2]), C[n][j][1] = (f16)(dm * fs[3]);
      }
    } else if constexpr (Q6) {
      if constexpr (I == 0) g[2] = -(int)(wt[r] >> 2), g[3] = 8 * (wt[r] & 3);
      else if constexpr (I == 1) g[0] = (p.m.x & ~g[2]) | (p.m.z & g[2]), g[1] = (p.m.y & ~g[2]) | (p.m.w & g[2]);
      else if constexpr (I == 2) g[0] >>= g[3], g[1] >>= g[3];
      else if constexpr (I == 3) fs[0] = (float)(int8_t)(g[0] & 0xFF), fs[1] = (float)(int8_t)(g[1] & 0xFF);
      else if constexpr (I == 4) {
        const float d = h2f((uint16_t)p.e);
        S[n][j][0] = (f16)(d * fs[0]), S[n][j][1] = (f16)(d * fs[1]);
      }
    } else if constexpr (I == 0) {
      S[n][j][0] = S[n][j][1] = __builtin_bit_cast(f16, (uint16_t)p.e);
    }
  };
  // quarter q (8 weights a lane) of slot r's piece j with scale set n, two dwords at a time in five stages: shift; to fp16 (codes
  // of the high half stay in place: 64 + n in mantissa bits 4 .. 7, so only odd bytes are shifted); high bits; zero point; scale
  constexpr int DST = 5;
  auto deq = [&](auto qc, auto rc, auto nc, auto jc, auto st, auto wc) {
    constexpr int q = decltype(qc)::value, r = decltype(rc)::value, n = decltype(nc)::value;
    constexpr int j = decltype(jc)::value, I = decltype(st)::value;
    constexpr int Wd = decltype(wc)::value, half = q >> 1, e = 2 * (q & 1) + Wd;
    constexpr bool hi = half && !K8, hbits = QT == QT_Q5_K || Q6;
    const Piece<QT>& p = wv[r][j];
    unsigned &oa = o[q & 1][j][2 * Wd], &ob = o[q & 1][j][2 * Wd + 1];
    const unsigned c = dsel(K8 && half ? p.b : p.a, e);
    constexpr unsigned mask = K8 ? 0x00FF00FFu : hi ? 0x00F000F0u : 0x000F000Fu;
    constexpr unsigned flip = K8 || (hi && (QT == QT_Q4_K || QT == QT_Q4_0)) ? 0x00800080u : 0u;  // signed codes to offset binary
    constexpr unsigned magic = (hi ? 0x54005400u : 0x64006400u) ^ flip;
    constexpr float zero = (hi ? 64.f : 1024.f) + (K8 ? 128.f : Q6 ? 32.f : QT == QT_Q4_0 ? 8.f : 0.f);
    constexpr unsigned hmask = Q6 ? (half ? 0x03000300u : 0x00300030u) : (half ? 0x01000100u : 0x00100010u);
    if constexpr (I == 0) {
      ob = c >> 8;
      if constexpr (hbits) {
        const unsigned H = Q6 ? (half ? p.h.y : p.h.x) : p.e;
#pragma unroll
        for (int odd = 0; odd < 2; ++odd) {
          const int sh = Q6 ? 8 * odd + 2 * e - (half ? 8 : 4) : 8 * odd + e - 4;
          hb[j][2 * Wd + odd] = sh >= 0 ? H >> sh : H << -sh;
        }
      }
    } else if constexpr (I == 1) {
      oa = __builtin_amdgcn_bitop3_b32(c, mask, magic, 0x6a), ob = __builtin_amdgcn_bitop3_b32(ob, mask, magic, 0x6a);  // (a & b) ^ c
    } else if constexpr (I == 2) {
      if constexpr (hbits) oa |= hb[j][2 * Wd] & hmask, ob |= hb[j][2 * Wd + 1] & hmask;
    } else if constexpr (I == 3) {
      const dh2 zp = dq_splat(zero);
      oa = dq_u(dq_h2(oa) - zp), ob = dq_u(dq_h2(ob) - zp);
    } else {
      const dh2 s = (dh2){S[n][j][half], S[n][j][half]}, m = KM ? (dh2){C[n][j][half], C[n][j][half]} : dq_splat(0.f);
      oa = dq_u(dq_h2(oa) * s + m), ob = dq_u(dq_h2(ob) * s + m);
    }
  };
  constexpr int DI = 2 * DST * TN, SI = SST * TN;
  auto deq_item = [&](auto qc, auto rc, auto nc, auto c) {
    constexpr int x = decltype(c)::value;
    deq(qc, rc, nc, ic<x % TN>{}, ic<x / (2 * TN)>{}, ic<x / TN % 2>{});
  };
  // phase p of step s (U = s mod R): products of the pieces' quarter p; each activation fragment is read again, for the next phase,
  // behind its last product; the next phase's weights and, in phases 1 and 2, the next step's scales are worked out; pieces of the
  // next step's activations go to the other LDS buffer. The step's barrier lies a few products into phase 3: by then its own last
  // reads are back, and what follows reads the next step and writes the one after it
  auto phase = [&](auto pc, auto uc, int s) {
    constexpr int p = decltype(pc)::value, U = decltype(uc)::value, B = U & 1, q = (p + 1) & 3, KB = NS / 4;
    constexpr int rbuf = p == 3 ? B ^ 1 : B, sbuf = p == 3 ? B : B ^ 1, slot = (p == 3 ? U + 1 : U) % R, set = (p == 3 ? U + 1 : U) & 1;
    each<0, NS>([&](auto sc) {
      constexpr int I = decltype(sc)::value, i = I / TN, j = I % TN, H = NS / 2;
      acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
          a[i], __builtin_bit_cast(f16x8, (u32x4){o[p & 1][j][0], o[p & 1][j][1], o[p & 1][j][2], o[p & 1][j][3]}), acc[i][j], 0, 0, 0);
      if constexpr (p == 3 && I == KB - 1) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        each<0, KB / TN>([&](auto c) { read(decltype(c)::value, q, rbuf); });
      } else if constexpr (j == TN - 1 && (p < 3 || I >= KB)) {
        read(i, q, rbuf);
      }
      constexpr int F = p == 2 ? NS / 4 : H;  // (before the barrier in time for it, behind it otherwise)
      if constexpr (I >= F && I < F + H)
        each<(I - F) * XI / H, (I - F + 1) * XI / H>([&](auto c) { stage(ic<q>{}, c, ic<sbuf>{}, p == 3 ? s + 2 : s + 1, sbuf); });
      each<I * DI / NS, (I + 1) * DI / NS>([&](auto c) { deq_item(ic<q>{}, ic<slot>{}, ic<set>{}, c); });
      if constexpr (p == 1 || p == 2) {
        constexpr int v = (p - 1) * NS + I;
        each<v * SI / (2 * NS), (v + 1) * SI / (2 * NS)>([&](auto c) {
          constexpr int x = decltype(c)::value;
          scale(ic<(U + 1) % R>{}, ic<(U + 1) & 1>{}, ic<x / SST>{}, ic<x % SST>{});
        });
      }
      if constexpr (p == 3)  // the piece just used up makes room for the one R steps later
        each<I * 2 * TN / NS, (I + 1) * 2 * TN / NS>([&](auto c) { load_w(s + R, decltype(c)::value % TN, decltype(c)::value / TN, U); });
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  each<0, TM>([&](auto c) { load_x(ks0, ic<0>{}, c); });
  each<0, R>([&](auto u) {
#pragma unroll
    for (int x = 0; x < 2 * TN; ++x) load_w(ks0 + decltype(u)::value, x % TN, x / TN, decltype(u)::value);
    if constexpr (decltype(u)::value == 0) each<0, TM>([&](auto c) { load_x(ks0 + 1, ic<1>{}, c); });
  });
  each<0, 4>([&](auto p) { each<0, XI>([&](auto c) { stage(p, c, ic<0>{}, ks0, 0); }); });
  each<0, XI>([&](auto c) { stage(ic<0>{}, c, ic<1>{}, ks0 + 1, 1); });
  each<0, SI>([&](auto c) { scale(ic<0>{}, ic<0>{}, ic<decltype(c)::value / SST>{}, ic<decltype(c)::value % SST>{}); });
  each<0, DI>([&](auto c) { deq_item(ic<0>{}, ic<0>{}, ic<0>{}, c); });
  __syncthreads();
#pragma unroll
  for (int i = 0; i < TM; ++i) read(i, 0, 0);
  for (int s = ks0; s < ks1; s += R)
    each<0, R>([&](auto u) { each<0, 4>([&](auto ph) { phase(ph, u, s + decltype(u)::value); }); });

  // Results go out 32 rows at a time through LDS: a thread then has four neighbouring columns of a row (gate / up and rotation pairs
  // side by side, 16-byte accesses, a row of the tile in one wave's instruction) and the same four in all rows, so what depends on
  // the column is worked out once. And there is one copy of each epilogue: straight from the fragments, every kind 16 times over,
  // they spilled registers and a file took four minutes to compile.
  // C fragment: column (weight row) = lane & 31, row = (r & 3) + 8 (r >> 2) + 4 (lane >> 5)
  constexpr int LDE = BN + 4, QD = BN / 4, NIT = 32 * QD / 256;
  float* ep = (float*)smem;
  int* kvr = (int*)(ep + 32 * LDE);  // [BM]
  const bool slab = !GROUPED && sk > 1;
  float* y = slab ? P.gws + (long long)z * M * N : P.y;
  const int ld = slab ? N : P.ldy, c0 = slab ? 0 : P.row_offset;
  const bool v4 = ((N | ld | c0) & 3) == 0 && ((uintptr_t)y & 15) == 0;
  auto epilogue = [&](auto ec) {
    constexpr int E = decltype(ec)::value;  // -1: a split's slab
    constexpr bool glu = E == EPI_GLU || E == EPI_GEGLU;
    // EPI_QKV: q4: a thread's columns lie in one head
    const int vc = n0 + 4 * (tid % QD) + c0, Dc = P.Dc > 0 ? P.Dc : P.D;
    const bool q4 = E == EPI_QKV && v4 && ((P.D | P.Eq | P.Ekv | P.n_rot | Dc) & 3) == 0 && P.rope &&
                    (((uintptr_t)P.rope | (uintptr_t)P.kc | (uintptr_t)P.vc) & 15) == 0;
    int which = 0, d = 0;
    long long hoff = 0;
    if (E == EPI_QKV) {
      which = vc < P.Eq ? 0 : vc < P.Eq + P.Ekv ? 1 : 2;
      const int h0 = vc - (which > 0 ? P.Eq : 0) - (which > 1 ? P.Ekv : 0), hh = h0 / P.D;
      d = h0 - hh * P.D;
      hoff = (long long)hh * P.bs * Dc + d;
    }
    const bool turn = which < 2 && d < P.n_rot;
    // what the next 32 rows need from memory, requested before these are worked on: EPI_ADD the sums so far, EPI_QKV the angles
    f32x4 was[NIT], next[NIT];
    auto fetch = [&](int i) {
#pragma unroll
      for (int u = 0; u < NIT; ++u) {
        const int x = tid + 256 * u, m = m0 + 32 * i + x / QD, gn = n0 + 4 * (x % QD);
        if (m >= M || gn >= N) continue;
        if constexpr (E == EPI_ADD) {
          const float* q = y + (long long)m * ld + c0 + gn;
          if (v4) next[u] = *(const f32x4*)q;
          else
#pragma unroll
            for (int k = 0; k < 4; ++k) next[u][k] = gn + k < N ? q[k] : 0.f;
        }
        if (E == EPI_QKV && q4 && turn) next[u] = *(const f32x4*)(P.rope + ((long long)m * (P.n_rot >> 1) + (d >> 1)) * 2);
      }
    };
    fetch(0);
    if (E == EPI_QKV) __syncthreads();
    if (E == EPI_QKV && tid < BM && m0 + tid < M) {  // a row's place in the cache, in units of Dc
      const int slot = P.slot[m0 + tid], blk = slot / P.bs;
      kvr[tid] = blk * P.n_kv * P.bs + slot - blk * P.bs;
    }
    for (int i = 0; i < TM && m0 + 32 * i < M; ++i) {
#pragma unroll
      for (int u = 0; u < NIT; ++u) was[u] = next[u];
      if (i + 1 < TM) fetch(i + 1);
      __syncthreads();  // the loop's (or the last rows') readers are done
      each<0, TM>([&](auto cc) {
        constexpr int c = decltype(cc)::value;
        if (i == c) {
#pragma unroll
          for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) ep[((r & 3) + 8 * (r >> 2) + 4 * fq) * LDE + 32 * (TN * wave + j) + fr] = acc[c][j][r];
          asm volatile("; rows %0" ::"n"(c));  // keeps the branches apart: merged, they would index the accumulators, in memory
        }
      });
      __syncthreads();
      constexpr int UN = E == EPI_GELU || E == EPI_GELU_ERF || E == EPI_GEGLU || E == EPI_QGELU ? 1 : NIT;
#pragma unroll UN
      for (int u = 0; u < NIT; ++u) {
        const int x = tid + 256 * u, rr = x / QD, gn = n0 + 4 * (x % QD), m = m0 + 32 * i + rr, vn = gn + c0;
        if (m >= M || gn >= N) continue;
        f32x4 v = *(const f32x4*)(ep + rr * LDE + 4 * (x % QD));
        const int row = GROUPED && P.moe_scatter ? P.moe_rows[m] : m;
        if constexpr (glu) {
          float* q = y + (long long)row * ld + vn / 2;
          const float a0 = (E == EPI_GLU ? silu(v.x) : gelu_tanh(v.x)) * v.y, a1 = (E == EPI_GLU ? silu(v.z) : gelu_tanh(v.z)) * v.w;
          if (v4) {
            *(f32x2*)q = (f32x2){a0, a1};
          } else {
            q[0] = a0;
            if (gn + 2 < N) q[1] = a1;
          }
          continue;
        }
        if constexpr (!slab_kind(E)) {
          if (P.bias && (E != EPI_QKV || q4)) {
#pragma unroll
            for (int k = 0; k < 4; ++k) v[k] += gn + k < N ? P.bias[vn + k] : 0.f;
          }
        }
        if constexpr (E == EPI_QKV) {
          if (q4) {  // four columns of one head
            const f32x4 t = was[u];
            if (turn) v = (f32x4){v.x * t.x - v.y * t.y, v.x * t.y + v.y * t.x, v.z * t.z - v.w * t.w, v.z * t.w + v.w * t.z};
            if (which == 0) {
              *(f32x4*)(y + (long long)m * ld + vn) = v;
            } else {
              const long long at = (long long)kvr[32 * i + rr] * Dc + hoff;
              void* kv = which == 1 ? P.kc : P.vc;
              if (P.kv8) *(unsigned*)((uint8_t*)kv + at) = f2e4m3(v.x) | f2e4m3(v.y) << 8 | f2e4m3(v.z) << 16 | (unsigned)f2e4m3(v.w) << 24;
              else *(f16x4*)((f16*)kv + at) = (f16x4){(f16)v.x, (f16)v.y, (f16)v.z, (f16)v.w};
            }
          } else {
#pragma unroll
            for (int k = 0; k < 4; ++k)
              if (gn + k < N) epi_apply_t<EPI_QKV>(P, m, vn + k, ep[rr * LDE + 4 * (x % QD) + k], ep[rr * LDE + 4 * (x % QD) + (k ^ 1)], 0);
          }
          continue;
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          if constexpr (E == EPI_ADD) v[k] += was[u][k];
          if constexpr (E == EPI_GELU) v[k] = gelu_tanh(v[k]);
          if constexpr (E == EPI_GELU_ERF) v[k] = 0.5f * v[k] * (1.f + erff(v[k] * 0.70710678f));
          if constexpr (E == EPI_QGELU) v[k] = v[k] / (1.f + __expf(-1.702f * v[k]));
        }
        float* q = y + (long long)row * ld + vn;
        if (v4 && slab_kind(E)) __builtin_nontemporal_store(v, (f32x4*)q);
        else if (v4) *(f32x4*)q = v;
        else
#pragma unroll
          for (int k = 0; k < 4; ++k)
            if (gn + k < N) q[k] = v[k];
      }
    }
  };
  if (slab) {
    epilogue(ic<-1>{});
    return;
  }
  if constexpr (GROUPED) {
    if (P.epi == EPI_GLU) epilogue(ic<EPI_GLU>{});
    else if (P.epi == EPI_GEGLU) epilogue(ic<EPI_GEGLU>{});
    else epilogue(ic<EPI_STORE>{});
  } else {
    switch (P.epi) {
      case EPI_STORE: epilogue(ic<EPI_STORE>{}); break;
      case EPI_ADD: epilogue(ic<EPI_ADD>{}); break;
      case EPI_GELU: epilogue(ic<EPI_GELU>{}); break;
      case EPI_GLU: epilogue(ic<EPI_GLU>{}); break;
      case EPI_GEGLU: epilogue(ic<EPI_GEGLU>{}); break;
      case EPI_GELU_ERF: epilogue(ic<EPI_GELU_ERF>{}); break;
      case EPI_QGELU: epilogue(ic<EPI_QGELU>{}); break;
      default: epilogue(ic<EPI_QKV>{}); break;
    }
  }
}

template <int QT, int TM, int TN>
__global__ __launch_bounds__(256, 1) void dq_slots_kernel(GemvParams P, const f16* __restrict__ X, int Kp, int sk) {
  const int nt = (P.w.N + 128 * TN - 1) / (128 * TN), wg = ring::xcd_range(blockIdx.x, gridDim.x), z = wg % sk, tile = wg / sk;
  ds_tile<QT, TM, TN, false>(P, X, Kp, sk, z, tile / nt * 32 * TM, P.B, tile % nt * 128 * TN, 0);
}

template <int QT, int TM, int TN>
void launch_slots(const GemvParams& P, const f16* xp, int Kp, int sk, hipStream_t s) {
  const int mt = (P.B + 32 * TM - 1) / (32 * TM), nt = (P.w.N + 128 * TN - 1) / (128 * TN);
  hipLaunchKernelGGL((dq_slots_kernel<QT, TM, TN>), dim3(mt * nt * sk), dim3(256), (ds_lds<TM, TN>()), s, P, xp, Kp, sk);
}

template <int QT>
void run_dq(const GemvParams& P, f16* xp, int Kp, hipStream_t s) {
  const DqChoice c = dq_choose(P);
  const int sk = c.sk;
  hipLaunchKernelGGL(prep_xp_kernel<QT>, dim3(P.B), dim3(256), (size_t)Kp * sizeof(float), s, P, xp, Kp);
  switch (c.tile) {
    case 0: launch_slots<QT, 8, 2>(P, xp, Kp, sk, s); break;
    case 1: launch_slots<QT, 8, 1>(P, xp, Kp, sk, s); break;
    case 2: launch_slots<QT, 4, 2>(P, xp, Kp, sk, s); break;
    default: launch_slots<QT, 4, 1>(P, xp, Kp, sk, s); break;
  }
  if (sk > 1) gemm_finalize(P, sk, s);
}

}  // namespace
}  // namespace omx
