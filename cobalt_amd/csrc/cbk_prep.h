// Eight activations times their column scales, shared by the preparation kernels of the two GEMMs.
#pragma once
#include "cbk_device.h"

namespace cbk {

__device__ inline void prep8(const uint4 v, const uint4 c, int xdt, float (&a)[8]) {
  const uint32_t xw[4] = {v.x, v.y, v.z, v.w}, cw[4] = {c.x, c.y, c.z, c.w};
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (xdt == CBK_F16) { a[2 * e] = h2f((uint16_t)(xw[e] & 0xffffu)); a[2 * e + 1] = h2f((uint16_t)(xw[e] >> 16)); }
    else { a[2 * e] = bf2f((uint16_t)(xw[e] & 0xffffu)); a[2 * e + 1] = bf2f((uint16_t)(xw[e] >> 16)); }
    a[2 * e] *= h2f((uint16_t)(cw[e] & 0xffffu)); a[2 * e + 1] *= h2f((uint16_t)(cw[e] >> 16));
  }
}

}  // namespace cbk
