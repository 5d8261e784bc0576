// How a prefill call runs: the kernel, its token tile and the split of its column range.  A plan depends on the
// matrix and the number of activation rows alone, so a call's results do not depend on the workspace it is given.
#pragma once
#include <stddef.h>
#include "cbk_device.h"

namespace cbk {

enum GemmKernel { GEMM_NONE = 0, GEMM_ROWS = 1, GEMM_TILE = 2 };      // cbk_gemm_skinny.h, cbk_gemm_big.h
struct GemmPlan {
  int kernel = GEMM_NONE;
  int ti = 0;                // token tile: 32 ti (GEMM_ROWS, 1 - 3) or 64 ti (GEMM_TILE, 1 / 2 / 4) tokens
  int nsplit = 1;            // workgroups the column range of a tile is cut over
  double t = 0;              // what the kernel's model expects, in microseconds
  size_t bytes = 0;          // workspace
};
constexpr size_t ANY_ROOM = (size_t)-1;

// The fastest plan of a kernel whose workspace is at most `room`; kernel GEMM_NONE if there is none.
GemmPlan plan_skinny(const DMat&, int M, size_t room);
GemmPlan plan_big(const DMat&, int M, size_t room);
// A given tile and split as a plan, for callers that name one; GEMM_NONE where the kernel cannot run it.
GemmPlan fixed_plan_skinny(const DMat&, int M, int ti, int nsplit);
GemmPlan fixed_plan_big(const DMat&, int M, int ti, int nsplit);
// The row tiles of a plan of 256-token tiles that run as smaller tiles (64 ti tokens) in a launch of their own; rows 0: none.
struct LastRound { int rows = 0, ti = 0; };
LastRound last_round_big(const DMat&, const GemmPlan&, int M);
// The column parts of a launch of the tile kernel: nsplit of them, in 64-column stages `first` for the first and `part` for
// each further one (the last takes what is left).
struct GbCut { int nsplit, first, part; };
GbCut cut_big(const DMat&, const GemmPlan&, int M);
// What the tile kernel takes with every q|k|v matrix in one piece (see gemm_room in cbk_api.hip).
size_t big_unsplit_space(const DMat&, int M);
bool gemm_skinny_takes(const DMat&);

// act: -1, or CBK_ACT_*: y = act(gate) * up of a gate/up matrix, [M, K / 2]
int launch_gemm_skinny(const DMat&, const GemmPlan&, const void* x, int xdt, int M, int64_t ldx, void* y, int ydt, int64_t ldy,
                       const void* bias, int act, void* ws, size_t ws_bytes, hipStream_t);
// halves: a gate/up matrix's outputs as two halves of y (GbArgs::halves) instead of interleaved
int launch_gemm_big(const DMat&, const GemmPlan&, const void* x, int xdt, int M, int64_t ldx, void* y, int ydt, int64_t ldy,
                    const void* bias, void* ws, size_t ws_bytes, hipStream_t, bool halves = false);

}  // namespace cbk
