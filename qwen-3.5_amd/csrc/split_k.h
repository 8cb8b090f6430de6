// How a GEMM deals its steps of K to the splits of a launch, free of HIP so that host tests
// compile it too.
#pragma once
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

}  // namespace q35
