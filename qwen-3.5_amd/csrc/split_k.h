// How a GEMM deals its steps of K to the splits of a launch, and the room their partial sums take;
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

// Partial floats that let gemm_launch consider up to kGemmMaxSplit K splits for M rows of N columns.
// Few rows make few tiles, so the MB launches split further: one 64-row tile of a 2048-wide projection
// is 16 blocks for 256 CUs.
constexpr int kGemmMaxSplit = 4, kGemmMaxSplitMb = 16;
inline size_t gemm_part_floats(int M, int64_t N) {
  return (size_t)(M <= 64 ? 16 : (M <= 128 ? 8 : kGemmMaxSplit)) * M * N;
}

// Rows up to which a prompt's gate | up splits K and applies the SwiGLU in a second kernel: the fused
// epilogue needs whole sums, and one 64-row tile is 96 blocks of the 2B shape's 12288 columns
constexpr int kPrefillSplitGu = 64;
// Partials of a prompt pass of up to cap rows: the residual projections' (hidden columns), and at
// least one whole gate | up launch of the rows above, which has no other way out
inline size_t prompt_part_floats(int cap, int64_t hidden, int64_t ffn) {
  return std::max(gemm_part_floats(cap, hidden), (size_t)std::min(cap, kPrefillSplitGu) * 2 * ffn);
}

}  // namespace q35
