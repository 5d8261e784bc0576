// What the Python extension (cbk_torch.cpp) uses of libcbk_hip.so beyond the C ABI.
#pragma once
#include <stddef.h>
#include <stdint.h>
#include "../../include/cbk.h"

namespace cbk {

// What cbk_gemv uses of a workspace at M rows (cbk_workspace_bytes covers every entry point).
size_t decode_workspace_bytes(const cbk_desc*, int M);

// The rest of a module's image, written by the packing kernel along with the rows: the column
// scales, the bytes between the arrays (zero), and two figures about what was packed.
constexpr int PACK_SLOTS = 64, PACK_SLOT_WORDS = 16;
struct PackExtra {
  // PACK_SLOTS x PACK_SLOT_WORDS, zeroed by the caller: status bits, groups re-derived, largest zero
  // point stored, survivors in the mask.  Workgroup b adds to slot b % PACK_SLOTS, a cache line each:
  // all workgroups on one address cost 25 us of a 50 us kernel.
  uint32_t* counts;
  const void* cs_src;          // column scales to copy (16-byte aligned), or nullptr
  void* cs_dst;
  uint32_t cs_units;           // in 16-byte units
  uint8_t* gap[4];
  uint32_t gap_bytes[4];       // below 256 each
};
int pack_image(const cbk_desc* dst, const void* mask_bits, const void* q, const void* scale, const void* zero,
               int zero_dtype, int fix_zero, int* status, const PackExtra* extra, void* stream);

}  // namespace cbk
