// Stream-order dequant prefill GEMM: dispatcher and knobs. Kernels are in
// gemm_dq_slots.h (shared parts in gemm_dq_impl.h), instantiated once per weight type in gemm_dq_<type>.hip.
#include <cstdlib>
#include <stdexcept>
#include <string>

#include "common.h"
#include "ops.h"

namespace omx {

int g_dq_enable = -1;  // -1: OMX_GEMM_DQ (default on), read once
int g_dq_cfg = -2;     // OMX_DQ_CFG: force tile config 0..3 (microbenchmarks); -2 = not read yet
int g_dq_sk = 0;       // > 0: force the split-K factor (microbenchmarks, set_dq_tuning)

void run_dq_q4k(const GemvParams& P, f16* xp, int Kp, hipStream_t s);  // gemm_dq_q4k.hip
void run_dq_q5k(const GemvParams& P, f16* xp, int Kp, hipStream_t s);  // gemm_dq_q5k.hip
void run_dq_q6k(const GemvParams& P, f16* xp, int Kp, hipStream_t s);  // gemm_dq_q6k.hip
void run_dq_q40(const GemvParams& P, f16* xp, int Kp, hipStream_t s);  // gemm_dq_q40.hip
void run_dq_q80(const GemvParams& P, f16* xp, int Kp, hipStream_t s);  // gemm_dq_q80.hip
void run_dq_moe(const GemvParams& P, f16* xp, int Kp, hipStream_t s);  // gemm_dq_moe.hip
void run_dq_f16(const GemvParams& P, f16* xp, int Kp, hipStream_t s);  // gemm_f16.hip: tiles of its own

bool dq_gemm_enabled() {
  if (g_dq_enable < 0) {
    const char* e = getenv("OMX_GEMM_DQ");
    g_dq_enable = e ? atoi(e) != 0 : 1;
  }
  if (g_dq_cfg == -2) {
    const char* c = getenv("OMX_DQ_CFG");
    g_dq_cfg = c ? atoi(c) : -1;
  }
  return g_dq_enable != 0;
}

void set_dq_gemm(int on) { g_dq_enable = on ? 1 : 0; }

void set_dq_tuning(int cfg, int sk) {
  dq_gemm_enabled();  // env defaults read first, then overridden
  g_dq_cfg = cfg;
  g_dq_sk = sk;
}

// tile x K split with the least time by a model of measured launches: the first and last steps of a wave of blocks cost `fixed`,
// every further wave `again`, a step of 64 K c0 while few blocks run and c1 on a full chip, on 128 x 128 tiles c2 with two blocks a
// CU (us); a split adds a launch that sums the slabs. Over 65 .. 2,048 rows x 7 matrices of 1,024 .. 22,016 rows and K = 4,096 ..
// 14,336 (all tiles and splits timed) the choice takes 0.3 % more time than the best on average and 5 % at most, Q6_K, whose
// unpacking is longer, with values of its own the same.
struct DsTile {
  int bm, bn;
  double fixed, again, c0, c1, c2;
};
constexpr DsTile DS_TILES[4] = {{256, 256, 12.0, 6.1, 1.14, 1.51, 0}, {256, 128, 10.0, 1.3, 0.59, 0.92, 0},
                                {128, 256, 6.9, 0.8, 0.78, 1.05, 0},  {128, 128, 6.7, 0.0, 0.42, 0.62, 1.05}};
constexpr DsTile DS_TILES6[4] = {{256, 256, 9.8, 3.8, 1.34, 1.99, 0}, {256, 128, 4.3, 2.8, 0.77, 1.13, 0},
                                 {128, 256, 5.7, 1.4, 1.08, 1.50, 0}, {128, 128, 2.6, 0.0, 0.64, 0.91, 1.51}};
DqChoice dq_choose(const GemvParams& P) {
  dq_gemm_enabled();  // OMX_DQ_CFG is read
  const bool q6 = P.w.qtype == QT_Q6_K;
  const int M = P.B, N = P.w.N, SB = (P.w.K + 255) >> 8;
  const int rule[6] = {1, 2, 3, 4, 6, 8}, *ks = g_dq_sk > 0 ? &g_dq_sk : rule, n_ks = g_dq_sk > 0 ? 1 : 6;
  const double g = q6 ? 8.4 : 3.0, bw = q6 ? 8.6e6 : 5.4e6;
  double least = -1.0;
  DqChoice best{3, 1};
  for (int c = 0; c < 4; ++c) {
    if (g_dq_cfg >= 0 && g_dq_cfg <= 3 && c != g_dq_cfg) continue;
    const DsTile& t = q6 ? DS_TILES6[c] : DS_TILES[c];
    for (int i = 0; i < n_ks; ++i) {
      const int k = ks[i];
      const long long units = (long long)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn) * k;
      if (k > 1 && (!P.gws || (long long)k * M * N > P.gws_elems || SB < k || (units > 640 && g_dq_sk <= 0))) break;
      const double slots = c == 3 ? 512 : 256, waves = (double)(long long)((units + slots - 1) / slots);
      const double fill = units < 256 ? units / 256.0 : 1.0, step = t.c2 > 0 && units > 256 ? t.c2 : t.c0 + (t.c1 - t.c0) * fill;
      const double us = t.fixed + (waves - 1) * t.again + waves * 4 * SB / k * step + (k > 1 ? g + 8.0 * k * M * N / bw : 0.0);
      if (least < 0.0 || us < least) least = us, best = {c, k};
    }
  }
  if (least < 0.0)  // a forced split
    throw std::runtime_error("dq GEMM: " + std::to_string(g_dq_sk) + " splits of K do not fit " + std::to_string(SB) +
                             " super-blocks or the slabs");
  return best;
}

bool dq_gemm(const GemvParams& P, hipStream_t s) {
  if (!dq_gemm_enabled() || P.B <= 64 || !P.xws || P.expert_ids || P.moe_tiles) return false;
  const int qt = P.w.qtype;
  if (qt == QT_F16 && P.B < 128) return false;
  if (qt != QT_Q4_K && qt != QT_Q5_K && qt != QT_Q6_K && qt != QT_Q4_0 && qt != QT_Q8_0 && qt != QT_F16) return false;
  const int Kp = ((P.w.K + 255) >> 8) * 256;
  const long long cap = P.xws_elems ? P.xws_elems : (long long)P.B * P.w.K;
  if ((long long)P.B * Kp > cap || (qt != QT_F16 && Kp > PREP_MAX_KP)) return false;
  f16* xp = (f16*)P.xws;
  count_launch(LC_DQ_GEMM);
  switch (qt) {
    case QT_Q4_K: run_dq_q4k(P, xp, Kp, s); break;
    case QT_Q5_K: run_dq_q5k(P, xp, Kp, s); break;
    case QT_Q6_K: run_dq_q6k(P, xp, Kp, s); break;
    case QT_Q4_0: run_dq_q40(P, xp, Kp, s); break;
    case QT_F16: run_dq_f16(P, xp, Kp, s); break;
    default: run_dq_q80(P, xp, Kp, s); break;
  }
  return true;
}

// Routed experts: gate / up of every (token, expert) pair, then down with the pairs' own output rows in P.y.
// Whole prompts (Q4_K_M) on this path / on the others (executor.cpp ffn_block), us. Four layers of 8 experts, top 2, of 1,024 x 1,024
// (width x feed-forward: 2,048 rows of gate and up): 17 rows 335 / 463, 130 463 / 1,606, 400 576 / 1,819; of 2,048 x 4,096: 17 rows 596 /
// 1,037, 1,000 1,622 / 3,237. Two layers of 64 experts, top 8, of 1,024 x 2,048: 17 rows 365 / 488, 1,000 1,413 / 6,667; of 8 of 4,096 x
// 14,336: 17 rows 1,039 / 2,265, 64 1,076 / 2,362, 260 1,293 / 4,182, 1,000 2,733 / 5,357. Smaller experts (not measured) stay with
// the others.
static bool moe_matrix(const QMat& w) {
  const int qt = w.qtype;
  return w.K % 4 == 0 && ((w.K + 255) >> 8) * 256 <= PREP_MAX_KP &&
         (qt == QT_Q4_K || qt == QT_Q5_K || qt == QT_Q6_K || qt == QT_Q4_0 || qt == QT_Q8_0);
}
bool moe_grouped(const QMat& gu, const QMat& down) {
  return dq_gemm_enabled() && gu.N >= 2048 && moe_matrix(gu) && moe_matrix(down);
}
bool dq_moe_covered(const GemvParams& P) {
  const int Kp = ((P.w.K + 255) >> 8) * 256;
  return dq_gemm_enabled() && moe_matrix(P.w) && P.xws && P.moe_tiles && P.moe_rows && (long long)P.B * Kp <= P.xws_elems &&
         (P.epi == EPI_GLU || P.epi == EPI_GEGLU || P.epi == EPI_STORE);
}
void dq_moe(const GemvParams& P, hipStream_t s) {
  const int Kp = ((P.w.K + 255) >> 8) * 256;
  f16* xp = (f16*)P.xws;
  count_launch(LC_DQ_GEMM);
  run_dq_moe(P, xp, Kp, s);
}

}  // namespace omx
