// Instantiations of cbk_gemm_skinny.h for 2-bit codes.
#include "cbk_gemm_skinny.h"

namespace cbk {
int launch_skinny_b2(const SkArgs& a, int keep, int group, int ti, int blocks, hipStream_t st) {
  return launch_skinny_bits<2>(a, keep, group, ti, blocks, st);
}
}  // namespace cbk
