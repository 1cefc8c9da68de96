// Workgroup shapes of the skinny GEMM kernels (gemm.hip): host code without HIP, so that the choice
// can be checked on the CPU.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstdint>

namespace rg {

constexpr int kGemmWaves = 4;
constexpr int kGemmMaxRows = 128;
#ifndef RG_GEMM_AHEAD
#define RG_GEMM_AHEAD 2
#endif
// Chunks of 128 k: 256 bytes of every row of X and W.
constexpr int kChunkK = 128;
constexpr int kChunkBytes = 2 * kChunkK;
constexpr int kLdsBytes = 160 * 1024;
// Largest K of the NORM kernels (their norm weight is staged whole in LDS).
constexpr int kNormMaxK = 8192;

// Chunks in flight and LDS bytes of a workgroup of the (NB, MB) instantiation (GemmRing<NB, MB,
// reserve>::AHEAD and ::BYTES + reserve, the norm weight's bytes of the NORM kernels).
inline int ring_ahead(int nb, int mb, int reserve = 0) {
  const int fit = (kLdsBytes - reserve) / (16 * (mb + nb) * kChunkBytes);
  return fit >= RG_GEMM_AHEAD + 2 ? RG_GEMM_AHEAD : fit >= 3 ? fit - 2 : fit - 1;
}
inline int ring_bytes(int nb, int mb, int reserve = 0) {
  const int slot = 16 * (mb + nb) * kChunkBytes;
  const int fit = (kLdsBytes - reserve) / slot;
  const int ahead = ring_ahead(nb, mb, reserve);
  const int slots = fit >= ahead + 2 ? ahead + 2 : ahead + 1;
  return std::max(slots * slot, nb * mb * kGemmWaves * 1024) + reserve;
}

// Workgroup shape: 16-column n-blocks (NB) and 16-row blocks (MB) per workgroup, row tiles
// ceil(M / 16 MB) and splits of K, chosen by a cost model of the per-CU operand stream
// calibrated on MI355X (a sweep of every shape at 1 to 128 rows of the projections of three model
// sizes, weights cold):
//   workgroups = row tiles x column tiles x splits, R = CUs x resident workgroups per CU (LDS),
//   stream = 3 us x ceil(workgroups / R) + 0.047 us x ceil(workgroups / CUs) x (MB + NB) x chunks / S
//            (0.047 us per 16 rows x 128 k: 4 KB of copies),
//   turn = 3 us + 0.18 us x sqrt(2 / chunks in flight) x chunks / S: a workgroup walks its chunks one
//          after the other, a copy's round trip over the chunks in flight each, however few bytes
//          they hold (4096 x 14336 unsplit, 112 chunks in turn, took 30 us at 1 and at 16 rows alike),
//   serial = max(stream, ceil(workgroups / R) x turn), weights = N K 2 B / 5.5 TB/s,
//   time = max(serial, weights) + 0.2 min(serial, weights) + 0.1 stream + (S > 1: 2 us + S M N 8 B /
//          3 TB/s for the partials and their reduce).
// Without the turn the model left deep layers unsplit: 4096 x 14336 at 1 / 27 / 64 rows 30.3 / 32.7
// / 35.9 us against 21.9 / 22.9 / 27.3 now (the weights alone 18.9 at 6.2 TB/s), 3072 x 8192 at 1
// to 16 rows 17.4 against 13.6; of 182 shapes one is slower than without it, by 2 % (3072 x 3072 at 8
// rows).  The pick is 2.4 % from the best of all plans on average, 21 % at worst (2048 x 8192 at 33
// rows; profiles/skinny_gemm_plan_sweep.txt).
// Each workgroup streams its rows of X and its columns of W once per K range; small row tiles
// cut the X bytes of narrow layers, and the XCD-aware order keeps their re-reads of W in L2.
struct GemmPlan { int nb, mb, mtiles, splits, xcd; };
inline GemmPlan gemm_plan(int M, int N, int K, int cus, bool pairs = false, int only_nb = 0, bool norm = false,
                          int max_splits = 4) {
  auto ceil_div = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
  const int nblk = N / 16, chunks = K / kChunkK;
  GemmPlan best{1, 1, M, 1, 0};
  double best_t = 1e30;
  for (int mb : {1, 2, 4, 8}) {
    if (mb > 1 && 16 * (mb / 2) >= M) continue;  // a smaller row tile already holds every row
    const int mtiles = (M + 16 * mb - 1) / (16 * mb);
    for (int nb : {4, 2, 1}) {
      if (nblk % nb != 0 || (pairs && nb == 1) || (only_nb && nb != only_nb)) continue;
      const int resident = std::max(1, std::min(4, kLdsBytes / ring_bytes(nb, mb, norm ? 2 * kNormMaxK : 0)));
      for (int splits : {1, 2, 4}) {
        if (splits > 1 && (splits > max_splits || pairs || norm || chunks / splits < 8)) continue;
        const int64_t wgs = (int64_t)mtiles * (nblk / nb) * splits;
        const double stream = 3.0 * (double)ceil_div(wgs, (int64_t)cus * resident) +
                              0.047 * (double)ceil_div(wgs, cus) * (mb + nb) * (chunks / splits);
        const int ahead = ring_ahead(nb, mb, norm ? 2 * kNormMaxK : 0);
        const double turn = 3.0 + 0.18 * std::sqrt(2.0 / ahead) * chunks / splits;
        const double serial = std::max(stream, (double)ceil_div(wgs, (int64_t)cus * resident) * turn);
        const double weights = (double)N * K * 2 / 5.5e6;
        double t = std::max(serial, weights) + 0.2 * std::min(serial, weights) + 0.1 * stream;
        if (splits > 1) t += 2.0 + (double)splits * M * N * 8 / 3.0e6;
        if (t < best_t - 1e-9) {
          best_t = t;
          best = GemmPlan{nb, mb, mtiles, splits, mtiles > 1 && (nblk / nb) % 8 == 0 ? 1 : 0};
        }
      }
    }
  }
  return best;
}

// Bytes of the fp32 partials of a plan that splits K.
inline size_t split_bytes(const GemmPlan& p, int M, int N) {
  return p.splits > 1 ? (size_t)p.splits * M * N * sizeof(float) : 0;
}

// The plan of a projection whose caller brought `workspace_bytes` (0: none): the best of those with
// at most 4, 2 and 1 splits whose partials it holds.  The shape is chosen again for fewer splits: a
// plan that splits K has few wide tiles, and those tiles unsplit leave most CUs idle.
inline GemmPlan linear_plan(int M, int N, int K, int cus, size_t workspace_bytes) {
  for (int most : {4, 2}) {
    const GemmPlan p = gemm_plan(M, N, K, cus, false, 0, false, most);
    if (split_bytes(p, M, N) <= workspace_bytes) return p;
  }
  return gemm_plan(M, N, K, cus, false, 0, false, 1);
}

}  // namespace rg
