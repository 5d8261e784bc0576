// What the Python extension (cbk_torch.cpp) uses of libcbk_hip.so beyond the C ABI.
#pragma once
#include <stddef.h>
#include <stdint.h>
#include "../../include/cbk.h"

namespace cbk {

// What cbk_gemv uses of a workspace at M rows (cbk_workspace_bytes covers every entry point).
size_t decode_workspace_bytes(const cbk_desc*, int M);
size_t decode_batch_workspace_bytes(int n, const cbk_desc* descs, int M);   // and cbk_gemv_batch

// What a decode call of M rows launches when it has a workspace, or none: the selector table (0 the small one, 1 the wide one, -1:
// no such launch) of the main and of the column-split kernel, the main kernel's reduction slots, and the column slabs it stages a row in.
// For tests.
struct DecodeChoice { int main_table = -1, main_slots = 0, split_table = -1, main_slabs = 0; };
int decode_choice(int n, const cbk_desc* descs, int M, bool room, DecodeChoice*);   // CBK_ERR_UNSUPPORTED: not in one pass of these kernels

// How a prefill call runs, and the same call on a kernel, token tile and split of the columns that the caller
// names: for tests, which have to know which of the instantiations they run.  kernel: 0 none of the two (cbk_linear in a gated
// call), 1 the kernel of cbk_gemm_skinny.h (32 ti tokens, ti 1 - 3), 2 that of cbk_gemm_big.h (64 ti tokens, ti 1 / 2 / 4).
// act: -1 for cbk_gemm, an activation for cbk_linear_act (y_dtype counts only there).
struct GemmChoice { int kernel, ti, nsplit; };
GemmChoice gemm_choice(const cbk_desc*, int M, int act);
void gemm_last_round(const cbk_desc*, int M, const GemmChoice&, int* row_tiles, int* ti);   // of such a call: LastRound in cbk_gemm_plan.h
void gemm_column_parts(const cbk_desc*, int M, const GemmChoice&, int* parts, int* first, int* rest);   // of such a call: GbCut there; parts 0: not that kernel's
size_t gemm_as_workspace_bytes(const cbk_desc*, int M, const GemmChoice&, int act, int y_dtype);   // 0: it cannot be run so
int gemm_as(const cbk_desc*, const GemmChoice&, const void* x, int x_dtype, int M, int64_t ldx, void* y, int y_dtype, int64_t ldy,
            const void* bias, int act, void* workspace, size_t workspace_bytes, void* stream);

// The rest of a module's image, written by the packing kernel along with the rows: the column
// scales, the bytes between the arrays (zero), and two figures about what was packed.
constexpr int PACK_ROWS = 16, PACK_COLS = 4096, PACK_RECORDS = 4096;  // a workgroup's slab; workgroups at most
inline int pack_records(int64_t K, int64_t N) {
  const int64_t b = (K + PACK_ROWS - 1) / PACK_ROWS * ((N + PACK_COLS - 1) / PACK_COLS);
  return (int)(b < PACK_RECORDS ? b : PACK_RECORDS);
}
struct PackExtra {
  // pack_records(K, N) x 4 words, one record per workgroup: status bits, groups re-derived, largest zero
  // point stored, survivors in the mask.  Plain stores that the host adds up: nothing has to be cleared before the
  // kernel, and no cache line is shared (atomics of all workgroups on one line cost 25 us of a 50 us kernel).
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
