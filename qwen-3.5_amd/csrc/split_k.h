// How many splits of K a GEMM launch takes, how it deals its steps to them, and their partials' room;
// free of HIP so that host tests compile it too.
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>
#if defined(__HIPCC__)
#define Q35_SPLIT_HD __host__ __device__
#else
#define Q35_SPLIT_HD
#endif

namespace q35 {

// Every split takes each = steps / splits steps of K in a row, the first extra = steps % splits of
// them one more.  With steps >= splits none is empty: a kernel loads its split's first step before
// its loop, and a split that lay past K would read past the operands.
struct SplitK {
  int32_t each, extra;
};
inline SplitK split_k(int32_t steps, int32_t splits) { return SplitK{steps / splits, steps % splits}; }
// First K step of split s (s == splits: the end of the last one)
Q35_SPLIT_HD inline int32_t split_begin(const SplitK& k, int32_t s) {
  return s * k.each + (s < k.extra ? s : k.extra);
}

// K splits of the fp32 launches; of the MB launches while half as many would leave half of the CUs
// idle (few rows make few tiles: one 64-row tile of a 2048-wide projection is 16 blocks for 256 CUs)
constexpr int kGemmMaxSplit = 4, kGemmMaxSplitMb = 16;
constexpr int kMbTileM = 64, kMbTileN = 128, kMbStepK = 64;

// K splits of an MB launch of M rows over N columns in all: the least estimated time whose partials
// fit `room` floats.  Measured at 512 rows: a block alone on a CU takes ~1.09 us per 64-row K step, and
// a CU holding two or more blocks retires one block-step every ~0.91 us; a split adds the reduction
// (reads every split's partials, writes y: ~4 TB/s, plus a launch unless the caller's next kernel
// does it).
inline int mb_splits(int M, int64_t N, int K, int cus, bool deferred, size_t room) {
  const int64_t tiles = (N / kMbTileN) * ((M + kMbTileM - 1) / kMbTileM);
  double best = 1e300;
  int splits = 1;
  for (int ks = 1; ks <= kGemmMaxSplitMb; ks *= 2) {
    if (ks > 1 && (room < (size_t)ks * M * N || K / kMbStepK < 2 * ks)) break;
    // past 4 splits the splits' reading back costs more than the model's rate unless half of them
    // would leave half the CUs idle (2048 x 6144, 64 rows: 8 splits 23.3 us, 4 splits 22.4)
    if (ks > kGemmMaxSplit && tiles * (ks / 2) > cus / 2) break;
    const int steps = (K / kMbStepK + ks - 1) / ks;
    const int64_t per_cu = (tiles * ks + cus - 1) / cus;
    double cost = per_cu <= 1 ? steps * 1.09e-6 : (double)per_cu * steps * 0.91e-6;
    if (ks > 1) cost += (double)M * N * (ks + 1) * 4.0 / 4e12 + (deferred ? 0.0 : 3e-6);
    if (cost < best * 0.97) { best = cost; splits = ks; }
  }
  return splits;
}

// Partial floats with which no launch of up to M rows of N columns is held to fewer splits than its
// rule prefers.  A workspace that holds fewer changes a call's splits, hence its sums' order and bits:
// with requests below this, the same call gave other bits once a larger one had grown a shared
// workspace.
inline size_t gemm_part_floats(int M, int64_t N) { return (size_t)kGemmMaxSplit * M * N; }
inline size_t mb_part_room(int M, int64_t N, int cus) {
  int64_t rows = (int64_t)kGemmMaxSplit * M;
  for (int ks = 2 * kGemmMaxSplit; ks <= kGemmMaxSplitMb; ks *= 2) {
    // the most rows that may take ks splits: tiles * ks / 2 <= cus / 2 (mb_splits)
    const int64_t most = (int64_t)(cus / 2) / (ks / 2) / std::max<int64_t>(1, N / kMbTileN) * kMbTileM;
    rows = std::max(rows, ks * std::min<int64_t>(M, most));
  }
  return (size_t)(rows * N);
}

// Rows up to which a prompt's gate | up splits K and applies the SwiGLU in a second kernel: the fused
// epilogue needs whole sums, and one 64-row tile is 96 blocks of the 2B shape's 12288 columns
constexpr int kPrefillSplitGu = 64;
// Partials of a prompt pass of up to cap rows: the residual projections' (hidden columns), and at
// least one whole gate | up launch of the rows above, which has no other way out
inline size_t prompt_part_floats(int cap, int64_t hidden, int64_t ffn, int cus) {
  return std::max(mb_part_room(cap, hidden, cus), (size_t)std::min(cap, kPrefillSplitGu) * 2 * ffn);
}

}  // namespace q35
