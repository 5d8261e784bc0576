// Instantiations of cbk_gemm_skinny.h for BLK1632_6 and for dense 8-bit codes.
#include "cbk_gemm_skinny.h"

namespace cbk {
int launch_skinny_b68(const SkArgs& a, int bits, int group, int ti, int blocks, hipStream_t st) {
  if (bits == 6) return launch_skinny_cfg<6, 16, 128>(a, ti, blocks, st);
  return group == 64 ? launch_skinny_cfg<8, 0, 64>(a, ti, blocks, st) : launch_skinny_cfg<8, 0, 128>(a, ti, blocks, st);
}
}  // namespace cbk
