// Prefill GEMM for many tokens:  Y[M, K] = X[M, N] . W_hat[K, N]^T on the gfx950 matrix cores.  (Calls of nine to a
// few hundred rows and small matrices: cbk_gemm_skinny.h, which has a decoder for 8-bit codes too.)
//
// Workgroup tile 256 tokens x 256 weight rows, 64 input columns per stage, four wavefronts
// each owning a 128 x 128 sub-tile (8 x 8 blocks of v_mfma_f32_16x16x32_f16, 256 accumulator
// registers), one wavefront per SIMD.  Both operands are double-buffered in LDS (64 KB of
// activations, 64 KB of weights): while the matrix cores work on stage s, the same wavefronts
// dequantise the weights of stage s + 1 into the other buffer, and the activation tile is
// copied there from global memory without passing through registers.
//
// Operands.  The activation side is X' = fp16(x * col_scale / s_m), written once per call into
// the caller's workspace by a small row-wise kernel (bf16 inputs are widened exactly; the
// product is rounded once to fp16).  s_m is 1 unless token m holds a product of magnitude 2^15
// or more; then it is the power of two that brings the token's largest below 2^15, and the
// epilogue multiplies the token's outputs by it, so nothing saturates at fp16's 65504 and the
// scaling itself is exact.  The weight side is
// fp16((q - zero) * scale) for a kept column and exactly 0 for a pruned one, so
// Y = sum_j X'[m,j] * W'[k,j] carries two roundings of relative size 2^-12.  Feeding bf16
// operands instead would round to 2^-9, which alone exceeds the 1e-3 relative-Frobenius
// budget of this layer; the f16 and bf16 MFMA rates are identical.
//
// Weight decode.  Each of the 256 threads owns one weight row of the tile and decodes its
// 64 columns of the stage.  For 2/3/4-bit codes (bitmap layouts with 10, 16 or 23 of 32 kept,
// and the dense layouts) and for BLK1632_6, zero points <= 128, this is the byte-permute decoder
// of the decode kernel (selector table in LDS) followed by two packed-half operations per column
// pair; the remaining layouts (8-bit codes, larger zero points) go through the generic
// 32-column reader.  One wavefront per SIMD issues an instruction every five cycles, later if it waits
// for the one before, and two fit beside a matrix instruction of 16 cycles.  So the decode is counted in
// instructions (an entry's address is one four-byte dot product of the mask dword, the entry holds what
// would be counted or compared, codes stay unsigned until the exact subtraction of 1024 + zero point, a
// pruned column reads the zero point from the place of the eighth survivor) and dealt out by hand, two independent
// ones beside a matrix instruction; but what a chunk and a block take once (the alignment and widening of their codes) and the
// high bit pairs of 6-bit codes stand in one place, up to forty.  Vector instructions per matrix instruction of the 256-token tile: 4-bit,
// 16 of 32 1.2, dense 1.1, 3-bit 23 of 32 2.0, 6-bit 2.3; of the 128- and 64-token tiles two and four times that, and there
// they bind.  (The 64-token tile in 32 x 32 blocks, half as many products: with the same decode 0.5 to 2 % slower in the mean of 24 decoders.
// Over these, plain, gate/up, q|k|v and split, 8192 x 5376: the 256- / 128- / 64-token tile 1.07 - 1.12 / 1.04 - 1.10 / 1.00 - 1.07 times as
// fast in the mean as the kernel with 32 x 32 blocks throughout, on five GPUs.)
//
// What bounds it: power.  The clock falls with the load: a loop of nothing but these matrix instructions on
// halves, half of one operand zeros, runs at 2.08 PFLOP/s, of v_mfma_f32_32x32x16_f16 (a fourth of the sums moved per
// product, but twice as often) at 1.85 at the same operands: hence the 16 x 16 x 32 form here.  N = 5376, 2048 tokens,
// 8192 rows (one tile on every CU), 4-bit, 16 of 32, one box: 181 us with 32 x 32 blocks and the decode left to the
// compiler's interleave, 169 now, 141 with the decode taken out, 119 with the matrix instructions alone (266, 196 and 183
// thousand cycles of the loop at about 1.6 GHz).  Gated block of 21504 x 5376 at 2048 tokens with both its products
// 1421 -> 1346 us; since the wait before a barrier is one that the compiler counts (wait_loads) 1.6 % less again.
//
// Workgroups are ordered so that those running at the same time on one XCD (blockIdx % 8)
// share their token tile, which then stays in that XCD's L2.
//
// Reference semantics: cbk::gemm_tile (src/cobaltkernel/csrc/cobalt_gemm.cuh:243-609).
#pragma once
#include <atomic>
#include <type_traits>
#include <utility>
#include "cbk_decode.h"

namespace cbk {

constexpr int GB_T = 256;       // tokens per workgroup tile (TI = 4); the TI = 1 kernels take 64
constexpr int GB_R = 256;       // weight rows per workgroup tile
constexpr int GB_K = 64;        // input columns per stage
constexpr int GB_LUT = 256 * 8 * 16;  // selector table, 8 lane-private copies of 256 x 16 B
// one stage of either operand in LDS: rows of 128 B, unpadded, swizzled
constexpr int gb_xbuf(int ti) { return 64 * ti * GB_K * 2; }
constexpr int GB_WBUF = GB_R * GB_K * 2;
constexpr size_t gb_lds(int ti) { return (size_t)2 * gb_xbuf(ti) + (size_t)2 * GB_WBUF + GB_LUT; }

typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));

struct GbArgs {
  DMat m;
  const uint16_t* xp;      // X' fp16 [Mpad, Npad]
  const float* row_scale;  // [Mpad] per X': power of two each of its rows was divided by
  int rss;                 // elements between the row scales of two X'
  int M, Npad;
  void* y;
  int ydt;
  int64_t ldy;
  const void* bias;
  int tiles_t, tiles_r;    // token tiles, row tiles of this launch
  int tr0;                 // its first row tile
  int halves;              // gate/up matrix (par): 1 = write the gate outputs to columns [0, K/2) and the up outputs to
                           // [K/2, K) of y instead of interleaving them (whole 16-byte stores; for cbk_linear_act)
  int ti;                  // 32-token blocks per wavefront: 4, 2 or 1 (tiles of 256, 128 or 64 tokens)
  // par = 1: gate/up matrix, two col_scale vectors by row parity.  A workgroup then takes 256
  // rows of one parity out of 512 (rows r0 + 2 i + p), and X' of that parity's vector, which
  // starts xps elements after the other one.
  int par;
  size_t xps;
  // q|k|v matrix whose ranges start on row tiles: rows from vs0 on use the second X', rows from
  // vs1 on the third (both INT_MAX for any other matrix)
  int vs0, vs1;
  // split of the column range (PAR 3): nsplit workgroups per output tile take nst_part stages
  // each, the first one nst_first, and leave float32 partial tiles [nsplit][.][part_ld] at part; a second kernel adds them
  int nsplit, nst_part, nst_first;
  float* part;
  size_t part_stride;      // elements between the partial matrices
  int64_t part_ld;
};

// One wavefront-wide copy of 64 x 16 bytes from global memory straight into LDS (no VGPRs, no
// ds_write): lane l reads base + soff + voff and its 16 bytes land at LDS byte lds + AT + 16 * l.  The
// compiler does not know that this instruction counts on vmcnt or that it writes LDS; the
// kernel waits for it by hand before the barrier that publishes the stage.
// Nor does it put the five wait states between a vector instruction that writes a scalar register and a memory instruction
// that reads it, as it does around its own.  SPILLS: kernels that keep the descriptor or an offset in vector registers
// and read it back right before (the generic reader's): the wait is here.  The others have them in scalar registers from
// long before, which build.py (wait_hazards) looks at.
template <int AT, bool SPILLS>
__device__ inline void dma_x16(v4u buffer, uint32_t voff, uint32_t soff, uint32_t lds) {
  asm volatile("s_add_u32 m0, %3, %4\n\ts_nop %5\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds"
               ::"v"(voff), "s"(buffer), "s"(soff), "s"(lds), "i"(AT), "i"(SPILLS ? 4 : 0) : "memory", "m0", "scc");
}
// Waits for all of a wavefront's loads and direct copies, in a form that the compiler's own count of loads takes in: behind an assembly
// statement it still holds its loads for outstanding, and at their first use waits for the copies issued since
__device__ inline void wait_loads() {
  __builtin_amdgcn_s_waitcnt(0x0F70);                               // vmcnt 0, the other counters at their largest
  asm volatile("" ::: "memory");
}
// the same in every lane, in a scalar register
__device__ inline uint32_t uniform(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }

// f(integral_constant 0), f(1), ... f(N - 1)
template <typename F, int... I>
__device__ inline void static_for_seq(F&& f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, typename F>
__device__ inline void static_for(F&& f) { static_for_seq(f, std::make_integer_sequence<int, N>{}); }

// d += w . x^T of 16 weight rows, 16 tokens and 32 columns.  Written as the instruction, with the sum in place in
// accumulation registers: the compiler's own choice of a destination beside the addend left 912 register copies in
// a trip of the loop (the gated block of the header 1395 -> 1663 us).  So the compiler knows of no wait states: two behind what
// writes an operand, eight before anything else reads a sum.  The sums are tied to the wait behind the loop (gb_mfma_done); that nothing
// comes between, a copy or a spill, is looked at in every build (build.py, wait_hazards).  SPILLS: the generic reader's kernels, which
// move sums around the calls of their decoder, leave it to the compiler.
template <bool SPILLS>
__device__ inline void gb_mfma(v4f& d, const v8h& w, const v8h& x) {
  if (SPILLS) d = __builtin_amdgcn_mfma_f32_16x16x32_f16(w, x, d, 0, 0, 0);
  else asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(d) : "v"(w), "v"(x));
}
template <int N>
__device__ inline void gb_mfma_done(v4f (&acc)[N][8]) {
  asm volatile("s_nop 15" ::: "memory");
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) asm volatile("" : "+a"(acc[i][j]));
}

// One wavefront's 128 x 128 accumulators -> y, 32 tokens at a time through LDS.  D[i][j] holds, in
// lane l and register r, token l%16 and weight row 4*(l/16) + r of its 16 x 16 block: four consecutive
// output columns, one LDS store.  Turning the tile around in LDS makes the global stores whole 16-byte
// pieces of consecutive output columns: 256 B (f16) or 512 B (f32) per token.  Compile-time indexed and
// branch-free per element: the 256 accumulators make this straight-line code, and it has to stay small.
template <int YDT, int kstep, int TI>                            // local row i is output column row0 + kstep * i
__device__ inline void gb_epilogue(const GbArgs& a, v4f (&acc)[2 * TI][8], uint8_t* smem, int lane, int wave, int tok0,
                                   int row0, const float* rs) {   // rs: the row scales of this tile's X'
  constexpr int ESZ = YDT == CBK_F32 ? 4 : 2;
  constexpr int PITCH = 128 * ESZ + 16;                          // bytes per token row in LDS
  constexpr int EPP = 16 / ESZ, PPR = 128 / EPP;                 // elements per 16-byte piece, pieces per row
  const int K = a.m.K;
  uint8_t* ep = smem + (size_t)wave * (32 * (128 * 4 + 16));
  uint8_t* epl = ep + (lane & 15) * PITCH + 4 * (lane >> 4) * ESZ;
  float bv[8][4];
#pragma unroll
  for (int j = 0; j < 8; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int k = row0 + kstep * (16 * j + 4 * (lane >> 4) + r);
      bv[j][r] = 0.f;
      if (a.bias && k < K) bv[j][r] = load_act<YDT>(a.bias, k);
    }
  // (a tile's 32-bit offsets; stores that go on to memory: the gated block of the header 1310.4 -> 1302.5 us)
  const bool vec_ok = ((a.ldy * ESZ) & 15) == 0 && (((uintptr_t)a.y) & 15) == 0 && a.ldy < (1 << 22);
  const uint64_t yb = (uint64_t)((uint8_t*)a.y + (size_t)tok0 * a.ldy * ESZ);
  const auto ybuf = through_buffer((void*)((uint64_t)uniform((uint32_t)yb) | ((uint64_t)uniform((uint32_t)(yb >> 32)) << 32)));
#pragma unroll
  for (int i = 0; i < TI; ++i) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const float ts = rs[tok0 + 32 * i + 16 * h + (lane & 15)];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = acc[2 * i + h][j][r] * ts + bv[j][r];
        uint8_t* d = epl + 16 * h * PITCH + 16 * j * ESZ;
        if (YDT == CBK_F32) *(float4*)d = make_float4(v[0], v[1], v[2], v[3]);
        else if (YDT == CBK_F16) *(uint2*)d = make_uint2((uint32_t)f2h(v[0]) | ((uint32_t)f2h(v[1]) << 16), (uint32_t)f2h(v[2]) | ((uint32_t)f2h(v[3]) << 16));
        else {                                                     // v_cvt_pk_bf16_f32: round to nearest even
          typedef __bf16 b2 __attribute__((ext_vector_type(2)));
          const b2 lo = {(__bf16)v[0], (__bf16)v[1]}, hi = {(__bf16)v[2], (__bf16)v[3]};
          *(uint2*)d = make_uint2(__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi));
        }
      }
    }
    if (kstep == 1 && !vec_ok) {
      // Rows of y that start anywhere (heights that are no multiple of 8): a wavefront stores 128 outputs of one token at a time,
      // neighbouring lanes neighbouring elements, two of 16 bits to a store where they share a dword.  (2954 x 1664 at 2138
      // tokens, against the tree with 32 x 32 blocks: 7 % faster, with the pieces below an element at a time 1 to 2 % slower.)
      const bool two = ESZ == 2 && (((uintptr_t)a.y | (uintptr_t)(a.ldy * ESZ)) & 3) == 0;
#pragma unroll 4
      for (int row = 0; row < 32; ++row) {
        const int tok = tok0 + 32 * i + row;
        if (tok >= a.M) break;
        const uint8_t* src = ep + row * PITCH;
        uint8_t* dst = (uint8_t*)a.y + ((size_t)tok * a.ldy + row0) * ESZ;
        if (two && row0 + 2 * lane + 1 < K) ((uint32_t*)dst)[lane] = ((const uint32_t*)src)[lane];
        else
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int e = two ? 2 * lane + h : lane + 64 * h;
            if (row0 + e >= K) continue;
            if (ESZ == 4) ((float*)dst)[e] = ((const float*)src)[e];
            else ((uint16_t*)dst)[e] = ((const uint16_t*)src)[e];
          }
      }
      continue;
    }
#pragma unroll
    for (int t = 0; t < 32 * PPR / 64; ++t) {
      const int pc = t * 64 + lane;
      const int row = pc / PPR, c = pc % PPR;
      const int tok = tok0 + 32 * i + row, k = row0 + kstep * (c * EPP);
      if (tok >= a.M || k >= K) continue;
      const uint8_t* src = ep + row * PITCH + c * 16;
      uint8_t* dst = (uint8_t*)a.y + ((size_t)tok * a.ldy + k) * ESZ;
      if (vec_ok && kstep == 1 && k + EPP <= K) store16_through(ybuf, ((uint32_t)(32 * i + row) * (uint32_t)a.ldy + (uint32_t)k) * ESZ, *(const uint4*)src);
      else
        for (int e = 0; e < EPP && k + kstep * e < K; ++e) {
          if (ESZ == 4) ((float*)dst)[kstep * e] = ((const float*)src)[e];
          else ((uint16_t*)dst)[kstep * e] = ((const uint16_t*)src)[e];
        }
    }
  }
}

// The generic reader: block t (32 columns) of row wrc as halfs, into pieces c ... c + 3 of the weight tile's row at LDS address
// `row` (swizzled with `sw`).  Long, and called from many places, so a function; it is given values and not, as a closure would,
// the caller's variables, which would then live in memory around every call.
static __device__ __attribute__((noinline)) void gb_generic_block(const DMat& m, const RowView rv, int wrc, bool wok, int t, uint32_t row,
                                                                  uint32_t sw, uint32_t c) {
  uint32_t packed[16];
  if (wok) {
    int q[32];
    const uint32_t keep = decode_block32(m, rv, t, q);
    const int g = (t * BLOCK) / m.group;
    const float sc = h2f(m.scale[meta_index(m, wrc, g)]);
    const float z = (float)m.zero[meta_index(m, wrc, g)];
    const bool dense = family_of(m.layout) == FAM_DENSE;
#pragma unroll
    for (int p = 0; p < 32; p += 2) {
      float v0 = __fmul_rn((float)q[p] - z, sc), v1 = __fmul_rn((float)q[p + 1] - z, sc);
      if (!dense) { v0 = ((keep >> p) & 1u) ? v0 : 0.f; v1 = ((keep >> (p + 1)) & 1u) ? v1 : 0.f; }
      packed[p >> 1] = (uint32_t)f2h(v0) | ((uint32_t)f2h(v1) << 16);
    }
  } else {
#pragma unroll
    for (int e = 0; e < 16; ++e) packed[e] = 0;
  }
#pragma unroll
  for (uint32_t e = 0; e < 4; ++e)
    *(__attribute__((address_space(3))) v4u*)(uintptr_t)(row + (sw ^ (c + e)) * 16u) = v4u{packed[4 * e], packed[4 * e + 1], packed[4 * e + 2], packed[4 * e + 3]};
}

// Code stream of 32-column block jb of a chunk (block_stream in cbk_decode.h).  3-bit codes are widened by three shifts and three
// selects, which leaves bits of a neighbour above every code; a dense block takes them off with the mask that it needs
// anyway (CODES), a bitmap's rank 7 has none.  Few instructions less, but a shorter chain, which shows where a block has three dwords
// or four (8192 x 5376, 512 tokens on the 64-token tile: dense 80.7 -> 75.3 us, group 64 80.1 -> 77.3; 23 of 32 100 -> 96, 103 -> 97) and not
// where it has two (10 of 32 88.4 -> 91.3, 16 of 32 86.5 -> 88.6: those keep the general form).
template <class C, int BITS>
__device__ inline void gb_block_stream(const uint32_t (&cw)[C::ND], int jb, uint32_t (&st)[C::NW]) {
  if (BITS != 3 || C::NW < 3) { block_stream<C, BITS>(cw, jb, st); return; }
#pragma unroll
  for (int k = 0; k < C::NW; ++k) {
    uint32_t x = get32<C::ND>(cw, jb * C::CB + 24 * k);
    x = mask_select(0x00000FFFu, x << 4, x);
    x = mask_select(0x003F003Fu, x << 2, x);
    x = mask_select(0x07070707u, x << 1, x);
    st[k] = C::DENSE ? x : x & 0x77777777u;
  }
}

// BITS 2 / 3 / 4: byte-permute decoder for (BITS, KEEP, GRP), KEEP = 0 for the dense layouts.
// BITS 0: generic 32-column reader, any fixed-stride layout.
// PAR 0: one col_scale vector.  1: gate/up matrix (GbArgs::par).  2: q|k|v matrix (GbArgs::vs0, vs1).
// 3: one vector or q|k|v, column range split over several workgroups (GbArgs::nsplit).
// Three instantiations rather than run-time switches: the schedule of the main loop is tuned
// to the instruction and measurably shifts with every value that is added to it.
// TI: 32-token blocks per wavefront.  4: the 256-token tile described above.  2: a 128-token tile
// (each wavefront 64 tokens x 128 rows) for calls of 65 to 128 activation rows.  1: a 64-token tile
// (each wavefront 32 tokens x 128 rows) for calls of at most 64 activation rows, whose time is
// the weight decode: a quarter of the matrix instructions per stage, the same decode.
template <int BITS, int KEEP, int GRP, int PAR, int TI = 4>
__global__ __launch_bounds__(256) void gemm_big_kernel(GbArgs a) {
  // All 256 registers of a wavefront (LDS holds one workgroup per CU either way), so that the shift amounts of the decode
  // are not in the last one (build.py, shift_hazards, which found two 64-token kernels with theirs in v127 of 128).
  asm volatile("" ::: "v255");
  constexpr int GB_XBUF = gb_xbuf(TI);
  constexpr bool FASTD = BITS != 0;
  using C = CodeCfg<FASTD ? BITS : 4, KEEP, FASTD ? GRP : 128>;
  constexpr bool BITMAP = FASTD && !C::DENSE;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  // Xs [2][GB_T][64 halfs], Ws [2][GB_R][64 halfs]: row r, logical 16-byte piece c at physical piece c ^ ((r >> 1) & 7),
  // of Ws at c ^ (r & 7).  A 16-byte read or write goes through LDS in sets of sixteen lanes, 0-3 12-15 20-27 and so on: with the fragments' rows
  // (l % 16) and pieces (l / 16) as with one piece of 64 rows, a set's pieces so lie in different banks.  (Rows padded to
  // 144 bytes, which serve fragments of 32 rows and one piece, triple the conflicts of the call: 14 -> 43 million cycles.)
  _Float16* Xs = (_Float16*)smem;
  uint8_t* Ws = smem + 2 * GB_XBUF;
  uint4* lut = (uint4*)(Ws + 2 * GB_WBUF);                        // [256][8]
  const DMat& m = a.m;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wt = wave >> 1, wr = wave & 1;
  // XCD-aware order: blockIdx % 8 picks the XCD; give each XCD whole token tiles
  constexpr bool SPLIT = PAR == 3;
  const int xcd = blockIdx.x & 7, idx = blockIdx.x >> 3;
  int part = 0, tile;                                              // token-tile-major tile
  if (SPLIT && a.nst_first == a.nst_part) {                        // equal parts: side by side
    const int nb = a.tiles_t * a.tiles_r * a.nsplit, lin = xcd * ((nb + 7) >> 3) + idx;
    if (lin >= nb) return;
    tile = lin / a.nsplit; part = lin - tile * a.nsplit;
  } else {                                                         // the first parts of all of an XCD's tiles, then the second ones
    const int nb = a.tiles_t * a.tiles_r, per = (nb + 7) >> 3;
    if (SPLIT) part = idx >= per ? 1 : 0;
    tile = xcd * per + idx - part * per;
    if (tile >= nb) return;
  }
  const int tt = tile / a.tiles_r, tr = tile % a.tiles_r + a.tr0;
  constexpr int kstep = PAR == 1 ? 2 : 1;                         // row stride of this workgroup's rows
  const int pp = PAR == 1 ? (tr & 1) : 0;                         // and their parity
  const int t0 = tt * (64 * TI), r0 = PAR == 1 ? (tr >> 1) * (2 * GB_R) + pp : tr * GB_R;
  const int N = m.N, Npad = a.Npad;
  // stages of this workgroup: all of them, or its part of them; a multiple of 4 either way;
  // stages past N see X' = 0
  const int s_begin = SPLIT && part ? a.nst_first + (part - 1) * a.nst_part : 0, s_len = part ? a.nst_part : a.nst_first;
  const int nst = SPLIT && s_len < Npad / GB_K - s_begin ? s_len : Npad / GB_K - s_begin;
  const int c_begin = s_begin >> 1;                               // first 128-column chunk
  const int nch = N >> 7;                                         // 128-column chunks of the weight rows

  if (BITMAP) {
    // an entry: the two selectors (a pruned column reads rank 7's byte); which bits of the upper pool are the codes' (rank 7's
    // byte only if all eight columns are kept); the bits its survivors take in the code stream
    const uint2 e = make_selectors<0x07070707u>((uint32_t)tid, C::SEL_KIND);
    const uint32_t full = C::HI2 ? 0x00FFFFFFu : C::SB == 4 ? 0x000F0F0Fu : 0x00030303u;
    const uint4 v = make_uint4(e.x, e.y, tid == 255 ? full | 0xFF000000u : full, (uint32_t)__builtin_popcount(tid) * C::SB);
#pragma unroll
    for (int j = 0; j < 8; ++j) lut[table_slot<8, 16>(tid, j)] = v;
  }
  const uint32_t lut_lane = (uint32_t)(uintptr_t)lut + 16 * (lane & 7);      // LDS address of this lane's copy of entry 0

  v4f acc[2 * TI][8];                                             // 16 tokens x 16 weight rows each
#pragma unroll
  for (int i = 0; i < 2 * TI; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[i][j][e] = 0.f;

  // this thread's weight row
  const int wrow = r0 + kstep * tid;
  const bool wok = wrow < m.K;
  const int wrc = wok ? wrow : m.K - 1;
  const RowView rv = row_view(m, wrc);
  const size_t meta0 = meta_index(m, wrc, 0), meta_step = m.tiled ? 16 : 1;
  // Activation tile: wavefront w copies rows 16 TI w .. 16 TI (w+1) - 1 of every stage with 2 TI
  // direct copies of eight rows each; lane l of copy q takes row 16 TI w + 8q + l/8 and fills
  // physical piece l%8 of it, i.e. fetches logical piece (l%8) ^ ((4q + l/16) & 7).  That is one
  // of two values per lane (q even / odd), so two lane offsets and a scalar base per copy suffice.
  const int wv = __builtin_amdgcn_readfirstlane(wave);
  const uint32_t xvo_e = (uint32_t)((lane >> 3) * Npad * 2 + (((lane & 7) ^ (lane >> 4)) * 16));
  const uint32_t xvo_o = (uint32_t)((lane >> 3) * Npad * 2 + (((lane & 7) ^ (4 + (lane >> 4))) * 16));
  const int xv = PAR == 1 ? pp : PAR >= 2 ? (r0 >= a.vs0 ? 1 : 0) + (r0 >= a.vs1 ? 1 : 0) : 0;   // which col_scale vector
  const uint64_t xsb = (uint64_t)(a.xp + (size_t)xv * a.xps + (size_t)(t0 + 16 * TI * wv) * Npad + (size_t)s_begin * GB_K);
  const uint64_t xsu = (uint64_t)uniform((uint32_t)xsb) | ((uint64_t)uniform((uint32_t)(xsb >> 32)) << 32);
  const uint32_t xlds0 = uniform((uint32_t)(uintptr_t)Xs + (uint32_t)wv * (2048u * TI)), xrow8 = uniform(16u * Npad);
  v4u xbuf;                                                       // the stage that is being copied, as a buffer
  auto dma_stage = [&](int s) {
    const uint64_t b = xsu + (uint64_t)(uint32_t)((s < nst ? s : nst - 1) * (GB_K * 2));
    xbuf = v4u{uniform((uint32_t)b), uniform((uint32_t)(b >> 32)), 0xFFFFFFFFu, 0x00027000u};
  };
  auto dma_x = [&](auto buf_, auto q_) {                          // copy q of that stage -> Xs[buf]
    constexpr int q = decltype(q_)::value;
    dma_x16<decltype(buf_)::value * GB_XBUF + q * 1024, !FASTD>(xbuf, (q & 1) ? xvo_o : xvo_e, q * xrow8, xlds0);
  };
  // fragment reads: this lane's row inside a 16-row block of either operand and its two swizzled piece offsets
  uint32_t xpc[2], wpc[2];
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
    xpc[kk] = ((4 * kk + (lane >> 4)) ^ ((lane & 15) >> 1)) * 16;
    wpc[kk] = ((4 * kk + (lane >> 4)) ^ (lane & 7)) * 16;
  }

  // one 128-column chunk of this thread's weight row: two stages' worth
  struct WChunk {
    uint32_t m[4];                       // bitmap
    uint32_t raw[C::NL];                 // code dwords as loaded (whole 16-byte units)
    uint32_t c[C::ND];                   // code bits, first bit of the chunk at bit 0
    uint32_t z[C::NGC];                  // zero points of the chunk's groups, and scales as loaded: nothing that needs
    uint32_t s[C::NGC];                  // their values may stand beside the loads, where it would wait for them
    uint32_t ci;                         // chunk index the units were loaded for
    uint32_t h2[C::HI2 ? 4 : 1];         // BLK1632_6: high bit pairs, one dword per block
  };
  WChunk wA, wB;
  uint32_t st[C::NW];                                             // code stream of the block being decoded

  auto load_chunk = [&](int c, WChunk& w) {
    if (!FASTD) return;
    c += c_begin;
    c = c < nch ? c : nch - 1;
    w.ci = (uint32_t)c;
    if (BITMAP) {
      const uint4 mk = *(const uint4*)rv.unit((uint32_t)c);                         // 16 B of bitmap
      w.m[0] = mk.x; w.m[1] = mk.y; w.m[2] = mk.z; w.m[3] = mk.w;
    }
    const uint32_t u0 = (m.code_off >> 4) + (C::VEC16 ? (uint32_t)c * (C::CHB / 128) : (((uint32_t)c * C::CHB) >> 7));
#pragma unroll
    for (int i = 0; i < C::NL / 4; ++i) {
      const uint4 v = *(const uint4*)rv.unit(u0 + i);
      w.raw[4 * i] = v.x; w.raw[4 * i + 1] = v.y; w.raw[4 * i + 2] = v.z; w.raw[4 * i + 3] = v.w;
    }
    if (C::HI2) {                                                   // the plane behind mask and nibbles
      const uint4 v = *(const uint4*)rv.unit(3u * (uint32_t)nch + (uint32_t)c);
      w.h2[0] = v.x; w.h2[1] = v.y; w.h2[2] = v.z; w.h2[3] = v.w;
    }
    const size_t mi = meta0 + (size_t)c * C::NGC * meta_step;
#pragma unroll
    for (int g = 0; g < C::NGC; ++g) {
      w.z[g] = m.zero[mi + g * meta_step];
      w.s[g] = m.scale[mi + g * meta_step];
    }
  };

  // Decode of mask byte b8 (8 columns) of a stage = half h of chunk w into Ws[buf], in PIECES pieces of at most two vector
  // instructions that do not depend on each other, one piece beside each matrix instruction of a 256-token tile: with one
  // wavefront on a SIMD an instruction that waits for the one before it takes eight cycles and more, and of the rest two fit
  // beside a 16-cycle matrix instruction.  Pieces 0 and 1 fetch the table entry of the byte two ahead (half ha of chunk wa).
  constexpr int PIECES = 16;
  constexpr uint32_t CODES = BITS == 3 ? 0x07070707u : C::SB == 4 ? 0x0F0F0F0Fu : 0x03030303u;
  // The stream is shifted on from byte to byte, of three dwords as two 64-bit pieces (a byte's survivors take at most 32 bits): five
  // shifts a block, 18 instructions fewer than windows at a running position (8192 x 5376, 4-bit, 23 of 32, 512 / 1024 / 2048 tokens on
  // the 64- / 128- / 256-token tile: 104 / 120 / 166 -> 92 / 110 / 162 us).
  constexpr bool CHAIN = !C::HI2;
  struct Sel { uint32_t x, y, full, bits; };
  Sel sel[4];                                                       // by byte mod 4
  uint32_t sel_at = 0;
  struct Dec { uint32_t win, rank, p0, p1, t, b0, b1, o[4]; } de;
  uint32_t wdst[8];                                                 // 16-byte pieces of this thread's row in Ws[0]
#pragma unroll
  for (int c = 0; c < 8; ++c) wdst[c] = (uint32_t)(uintptr_t)Ws + (uint32_t)tid * 128u + (((uint32_t)tid & 7u) ^ c) * 16u;
  auto decode_piece = [&](int s, WChunk& w, int h, int buf, int b8, int piece, const WChunk& wa, int ha) {
    auto put = [&](int c, uint32_t x, uint32_t y, uint32_t z, uint32_t v) {
      *(__attribute__((address_space(3))) v4u*)(uintptr_t)(wdst[c] + (uint32_t)buf * GB_WBUF) = v4u{x, y, z, v};
    };
    if (!FASTD) {
      if ((b8 & 3) || piece) return;                              // the generic reader works on 32 columns
      const int t = ((s + s_begin) * GB_K >> 5) + (b8 >> 2);
      gb_generic_block(m, rv, wrc, wok, t < (N >> 5) ? t : (N >> 5) - 1,
                       (uint32_t)(uintptr_t)Ws + (uint32_t)buf * GB_WBUF + (uint32_t)tid * 128u, (uint32_t)tid & 7u, (uint32_t)b8);
      return;
    }
    const int blk = 2 * h + (b8 >> 2);                              // 32-column block of the chunk
    const int jj = b8 & 3;                                          // mask byte inside the block
    const int gi = C::NGC == 2 ? h : 0;                             // quantisation group of this stage
    const _Float16 sh = __builtin_bit_cast(_Float16, (uint16_t)(wok ? w.s[gi] : 0u));
    const h2_t s2 = {sh, sh};
    const uint32_t z = w.z[gi];
    // eight codes (the zero point z for a pruned column) -> eight halfs (q - z) * scale: a code in the low byte of
    // 0x64xx is the half 1024 + q; the difference to 1024 + z is exact, the product rounds once
    const h2_t off2 = __builtin_bit_cast(h2_t, 0xE400E400u + z * 0x00010001u);
    if (piece == 0) {
      if (h == 0 && b8 == 0) align_chunk_codes<C>(w.raw, w.ci, w.c);  // once per chunk, at its first use
      if (jj == 0) gb_block_stream<C, BITS>(w.c, blk, st);            // once per block
      if (BITMAP) {
        const int ja = 8 * ha + ((b8 + 2) & 7);                       // mask byte of the chunk, 0..15
        // byte ja % 4 of the mask dword, times 128 bytes per entry, plus the base
        sel_at = __builtin_amdgcn_udot4(wa.m[ja >> 2], 128u << (8 * (ja & 3)), lut_lane, false);
      }
    } else if (piece == 1) {
      if (BITMAP) {
        const v4u e = *(const __attribute__((address_space(3))) v4u*)(uintptr_t)sel_at;
        sel[(b8 + 2) & 3] = Sel{e[0], e[1], e[2], e[3]};
      }
    } else if (piece == 2) {
      if (BITMAP) {                                                   // past the survivors of the byte before
        const uint32_t n = sel[(b8 - 1) & 3].bits;
        if (!CHAIN) de.rank = jj == 0 ? 0u : jj == 1 ? n : de.rank + n;
        else if (jj && C::NW == 1) st[0] >>= n;
        else if (jj) {
          constexpr int B = C::NW > 1 ? 1 : 0, E = C::NW - 1;
          const uint64_t v = (((uint64_t)st[B] << 32) | st[0]) >> n;
          st[0] = (uint32_t)v;
          if (C::NW == 2) st[B] = (uint32_t)(v >> 32);
          else {
            const uint64_t u = (((uint64_t)st[E] << 32) | st[B]) >> n;
            st[B] = (uint32_t)u; st[E] = (uint32_t)(u >> 32);
          }
        }
      }
    } else if (piece == 3) {
      if (BITMAP) de.win = CHAIN || jj == 0 ? st[0] : window<C::NW>(st, de.rank);
      else de.win = C::SB == 4 ? st[jj] : (st[jj >> 1] >> (16 * (jj & 1)));
    } else if (piece == 4) {
      if (C::SB == 2) { const uint32_t lo16 = de.win & 0xFFFFu; de.win = (lo16 << 14) | lo16; }   // bytes c0 c4 c1 c5; four bits up c2 c6 c3 c7
    } else if (piece == 5) {
      de.p0 = de.win & CODES;                                         // even codes (of two bits: c0 c4 c1 c5)
      de.t = de.win >> 4;
    } else if (piece == 6) {
      // p0 | p1: the codes of the survivors from this byte's first on, even and odd ranks (four bits), or 0 2 .. and 4 6 ..
      // Rank 7, the top byte of p1, is asked for only if all eight columns are kept: otherwise the zero point takes its
      // place, which is what a pruned column reads.
      if (C::HI2) {
        uint32_t h0, h1;
        hi2_pools(w.h2[C::HI2 ? blk : 0], de.rank >> 2, h0, h1);
        de.p0 |= h0;
        de.t = (de.t & 0x0F0F0F0Fu) | h1;
      }
    } else if (piece == 7) {
      if (BITMAP) de.p1 = (de.t & sel[b8 & 3].full) | ((z << 24) & ~sel[b8 & 3].full);
      else de.p1 = de.t & CODES;
    } else if (piece == 8) {
      de.b0 = perm(de.p1, de.p0, BITMAP ? sel[b8 & 3].x : C::SB == 4 ? 0x05010400u : 0x06040200u);
      de.b1 = perm(de.p1, de.p0, BITMAP ? sel[b8 & 3].y : C::SB == 4 ? 0x07030602u : 0x07050301u);
    } else if (piece < 15) {
      const int i = piece < 11 ? 2 * (piece - 9) : 2 * ((piece - 11) & 1);
#pragma unroll
      for (int e = i; e < i + 2; ++e) {
        if (piece < 11) de.o[e] = __builtin_amdgcn_perm(0x64646464u, e < 2 ? de.b0 : de.b1, e & 1 ? 0x04030402u : 0x04010400u);
        else {
          const h2_t v = __builtin_bit_cast(h2_t, de.o[e]);
          de.o[e] = __builtin_bit_cast(uint32_t, piece < 13 ? v + off2 : v * s2);
        }
      }
    } else {
      put(b8, de.o[0], de.o[1], de.o[2], de.o[3]);
    }
  };

  // Fragment registers: the two halves of the tile's token blocks and of its row blocks, 32 columns each.  The 64-token tile
  // has registers for both 32-column steps of a stage (DEEP): a phase of its four matrix instructions is shorter than the
  // LDS latency (4096 x 14336, 2-bit dense, 64 rows: 216 us with the half that the next phase needs read one phase ahead as in
  // the larger tiles, 189 so; the 128-token tile gains nothing by it).
  constexpr bool DEEP = TI == 1;
  constexpr int BP = DEEP ? 4 : 6;                                // the phase that begins with the barrier
  v8h af[DEEP ? 2 : 1][2][TI], bf[DEEP ? 2 : 1][2][4];
  auto read_x = [&](int buf, int kk, int h, int i) {
    const uint8_t* xb = (const uint8_t*)Xs + (size_t)buf * GB_XBUF + (32 * TI * wt + 16 * TI * h + (lane & 15)) * 128;
    af[DEEP ? kk : 0][h][i] = *(const v8h*)(xb + 2048 * i + xpc[kk]);
  };
  auto read_w = [&](int buf, int kk, int h, int j) {
    const uint8_t* wb = Ws + (size_t)buf * GB_WBUF + (128 * wr + 64 * h + (lane & 15)) * 128;
    bf[DEEP ? kk : 0][h][j] = *(const v8h*)(wb + 2048 * j + wpc[kk]);
  };
  auto read_all = [&](int buf, int kk) {
    static_for<2 * TI>([&](auto i_) { constexpr int i = decltype(i_)::value; read_x(buf, kk, i / TI, i % TI); });
    static_for<8>([&](auto j_) { constexpr int j = decltype(j_)::value; read_w(buf, kk, j / 4, j % 4); });
  };

  // Decode of a stage: mask byte d / PIECES, piece d % PIECES; the first DEC0 pieces run behind the barrier of the stage
  // before the one that precedes it.
  constexpr int MF = 32 * TI, DEC0 = PIECES * (8 - BP);            // MFMAs of a stage
  // The copies of a stage start there too, one every DMAX MFMAs: a wavefront that issues the next before the last one's
  // 1 KB has passed waits for it (all eight behind the barrier: 1840 -> 2000 thousand cycles for the call)
  constexpr int DMAX = 12, DMA0 = (4 * TI * (8 - BP) - 3) / DMAX + 1;
  auto decode_step = [&](int s, auto d_, WChunk& wd, auto hd_tag, const WChunk& wn, auto hn_tag, int buf) {
    constexpr int d = decltype(d_)::value, b8 = d / PIECES, HD = decltype(hd_tag)::value, HN = decltype(hn_tag)::value;
    decode_piece(s, wd, HD, buf, b8, d % PIECES, b8 < 6 ? wd : wn, b8 < 6 ? HD : HN);
  };
  using T = std::true_type; using Fl = std::false_type;
  using H0 = std::integral_constant<int, 0>; using H1 = std::integral_constant<int, 1>;

  // ---- prologue: chunk 0 into registers and stage 0 into buffer 0; then, in the order every
  // stage leaves them, the copies of stage 1, the loads of chunk 1 and the first pieces of stage 1
  dma_stage(0);
  static_for<2 * TI>([&](auto q_) { dma_x(std::integral_constant<int, 0>{}, q_); });
  load_chunk(0, wA);
  load_chunk(1, wB);
  __syncthreads();                                                // selector table visible
  if (FASTD) {                                                    // selectors of bytes 0 and 1: as bytes 6 and 7 before them leave them
    decode_piece(0, wA, 0, 0, 6, 0, wA, 0); decode_piece(0, wA, 0, 0, 6, 1, wA, 0);
    decode_piece(0, wA, 0, 0, 7, 0, wA, 0); decode_piece(0, wA, 0, 0, 7, 1, wA, 0);
  }
  static_for<8 * PIECES>([&](auto d_) { decode_step(0, d_, wA, H0{}, wA, H1{}, 0); });
  wait_loads();
  __syncthreads();
  if constexpr (DEEP) read_all(0, 0);
  else {
#pragma unroll
    for (int i = 0; i < TI; ++i) read_x(0, 0, 0, i);
#pragma unroll
    for (int j = 0; j < 4; ++j) read_w(0, 0, 0, j);
  }
  dma_stage(1);
  static_for<DMA0>([&](auto q_) { dma_x(std::integral_constant<int, 1>{}, q_); });
  static_for<DEC0>([&](auto d_) { decode_step(1, d_, wA, H1{}, wB, H0{}, 1); });

  // One stage = eight phases of 4 TI MFMAs on buffer s % 2: for each 32 columns the four quarters (half of the
  // token blocks) x (half of the row blocks), in an order in which every phase needs one new half, read a phase
  // early into the registers that have just become free.  Phase BP first waits for the direct copies of stage
  // s + 1 (issued a stage ago) and passes the barrier; nobody reads buffer s % 2 after it, so the copies of
  // stage s + 2 start there and its weights begin to be decoded; the phases before it decode the rest
  // of stage s + 1: the same number of vector instructions beside every MFMA.
  // Stage s + 1 is half HD of chunk wd, stage s + 2 half HN of chunk wn; the stage behind that begins with chunk wo, half
  // HD.  With LOADW, phase BP loads chunk `cl` into wd, which is decoded.
  // No branches inside.
  auto stage = [&](int s, auto buf_, auto loadw_tag, WChunk& wd, auto hd_tag, WChunk& wn, auto hn_tag, WChunk& wo, int cl) {
    constexpr bool LOADW = decltype(loadw_tag)::value;
    constexpr int BUF = decltype(buf_)::value, buf = BUF;
    static_for<8>([&](auto p_) {
      constexpr int p = decltype(p_)::value, kk = p >> 2, q = p & 3;
      constexpr int hx = q >> 1, hw = (q == 1 || q == 2) ? 1 - kk : kk;
      if constexpr (p == BP) {
        // the direct copies of stage s + 1 must have landed before the barrier publishes them
        // (the weight chunk loads of the previous stage wait here as well: they were issued a
        // whole stage ago, and counting them out of the wait would rest on how many load
        // instructions the compiler keeps)
        wait_loads();
        __syncthreads();
        if (LOADW) load_chunk(cl, wd);
      }
      static_for<4 * TI>([&](auto t_) {
        constexpr int t = decltype(t_)::value, i = t / 4, j = t % 4, at = 4 * TI * p + t;
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (DEEP) {
          if constexpr (p == 0 && t == 0) read_all(buf, 1);
          if constexpr (p == BP && t == 0) read_all(buf ^ 1, 0);
        } else if constexpr (q == 1 || q == 2) {                    // the half that the next phase needs
          if constexpr (t < TI) read_x(p == 6 ? buf ^ 1 : buf, p == 2 ? 1 : kk & (p != 6), q == 1, t);
        } else if constexpr (t < 4) {
          if constexpr (q == 0) read_w(buf, kk, 1 - kk, t);
          else read_w(p == 7 ? buf ^ 1 : buf, p == 3, p == 3, t);
        }
        constexpr int g = p >= BP ? at - 4 * TI * BP : at + 4 * TI * (8 - BP);      // MFMAs since the barrier
        if constexpr (g == 0) dma_stage(s + 2);
        if constexpr (g % DMAX == 2 && g / DMAX < 2 * TI) dma_x(std::integral_constant<int, p >= BP ? BUF : 1 - BUF>{}, std::integral_constant<int, g / DMAX>{});
        gb_mfma<!FASTD>(acc[TI * hx + i][4 * hw + j], bf[DEEP ? kk : 0][hw][j], af[DEEP ? kk : 0][hx][i]);
        if constexpr (p < BP) {
          constexpr int d0 = DEC0 + at * 8 * PIECES / MF, d1 = DEC0 + (at + 1) * 8 * PIECES / MF;
          static_for<d1 - d0>([&](auto d_) { decode_step(s + 1, std::integral_constant<int, d0 + decltype(d_)::value>{}, wd, hd_tag, wn, hn_tag, buf ^ 1); });
        } else {
          constexpr int a6 = at - 4 * TI * BP, d0 = a6 * 8 * PIECES / MF, d1 = (a6 + 1) * 8 * PIECES / MF;
          static_for<d1 - d0>([&](auto d_) { decode_step(s + 2, std::integral_constant<int, d0 + decltype(d_)::value>{}, wn, hn_tag, wo, hd_tag, buf); });
        }
      });
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  // Four stages per trip (two chunks): stage 2p decodes the rest of the upper half of chunk p and, behind its
  // barrier, loads chunk p+2 into the registers chunk p has just left, two stages before their first use.
  for (int s = 0; s < nst; s += 4) {
    const int p = s >> 1;
    stage(s,     H0{}, T{},  wA, H1{}, wB, H0{}, wB, p + 2);
    stage(s + 1, H1{}, Fl{}, wB, H0{}, wB, H1{}, wA, 0);
    stage(s + 2, H0{}, T{},  wB, H1{}, wA, H0{}, wA, p + 3);
    stage(s + 3, H1{}, Fl{}, wA, H0{}, wA, H1{}, wB, 0);
  }
  gb_mfma_done(acc);
  // the last stage issued copies of a stage that does not exist: let them land before the
  // epilogue reuses LDS
  wait_loads();
  __syncthreads();

  const int tok0 = t0 + 32 * TI * wt, row0 = r0 + kstep * 128 * wr;
  const float* rs = a.row_scale + (size_t)xv * a.rss;
  if (SPLIT) {                                                    // float32 partial tile, no bias
    GbArgs b = a;
    b.y = a.part + (size_t)part * a.part_stride;
    b.ldy = a.part_ld;
    b.bias = nullptr;
    gb_epilogue<CBK_F32, 1, TI>(b, acc, smem, lane, wave, tok0, row0, rs);
    return;
  }
  if (PAR == 1 && a.halves) {
    // this workgroup's rows are one parity of the matrix: consecutive columns of that half of y
    GbArgs b = a;
    const int K2 = a.m.K >> 1;
    b.y = (uint8_t*)a.y + (size_t)pp * K2 * (a.ydt == CBK_F32 ? 4 : 2);
    b.m.K = K2;
    b.bias = nullptr;
    const int hrow0 = (r0 >> 1) + 128 * wr;
    if (a.ydt == CBK_F32) gb_epilogue<CBK_F32, 1, TI>(b, acc, smem, lane, wave, tok0, hrow0, rs);
    else if (a.ydt == CBK_F16) gb_epilogue<CBK_F16, 1, TI>(b, acc, smem, lane, wave, tok0, hrow0, rs);
    else gb_epilogue<CBK_BF16T, 1, TI>(b, acc, smem, lane, wave, tok0, hrow0, rs);
    return;
  }
  if (a.ydt == CBK_F32) gb_epilogue<CBK_F32, kstep, TI>(a, acc, smem, lane, wave, tok0, row0, rs);
  else if (a.ydt == CBK_F16) gb_epilogue<CBK_F16, kstep, TI>(a, acc, smem, lane, wave, tok0, row0, rs);
  else gb_epilogue<CBK_BF16T, kstep, TI>(a, acc, smem, lane, wave, tok0, row0, rs);
}

template <int BITS, int KEEP, int GRP, int PAR, int TI>
static int launch_big_par(const GbArgs& a, int blocks, hipStream_t st) {
  auto kern = gemm_big_kernel<BITS, KEEP, GRP, PAR, TI>;
  static std::atomic<int> configured{0};
  if (!configured.load(std::memory_order_acquire)) {
    if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024) != hipSuccess)
      return CBK_ERR_HIP;
    configured.store(1, std::memory_order_release);
  }
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(256), gb_lds(TI), st, a);
  return hipGetLastError() == hipSuccess ? CBK_OK : CBK_ERR_HIP;
}

template <int BITS, int KEEP, int GRP, int TI>
static int launch_big_ti(const GbArgs& a, int blocks, hipStream_t st) {
  if (a.par) return launch_big_par<BITS, KEEP, GRP, 1, TI>(a, blocks, st);
  if (a.nsplit > 1) {
    if constexpr (BITS == 0) return CBK_ERR_UNSUPPORTED;             // (the generic reader's launches are never split)
    else return launch_big_par<BITS, KEEP, GRP, 3, TI>(a, blocks, st);
  }
  if (a.vs0 != 0x7fffffff) return launch_big_par<BITS, KEEP, GRP, 2, TI>(a, blocks, st);
  return launch_big_par<BITS, KEEP, GRP, 0, TI>(a, blocks, st);
}

template <int BITS, int KEEP, int GRP>
static int launch_big_cfg(const GbArgs& a, int blocks, hipStream_t st) {
  return a.ti == 1 ? launch_big_ti<BITS, KEEP, GRP, 1>(a, blocks, st)
       : a.ti == 2 ? launch_big_ti<BITS, KEEP, GRP, 2>(a, blocks, st) : launch_big_ti<BITS, KEEP, GRP, 4>(a, blocks, st);
}

// the (keep, group) instantiations of one code width and one token tile (a translation unit each:
// the 32 kernels of such a set are what one compiler process takes a minute and a half for)
template <int BITS, int TI>
static int launch_big_bits(const GbArgs& a, int keep, int group, int blocks, hipStream_t st) {
#define CBK_GB_CASE(KEEP)                                                                            \
  case KEEP: return group == 64 ? launch_big_ti<BITS, KEEP, 64, TI>(a, blocks, st)                   \
                                : launch_big_ti<BITS, KEEP, 128, TI>(a, blocks, st);
  switch (keep) {
    CBK_GB_CASE(0) CBK_GB_CASE(10) CBK_GB_CASE(16) CBK_GB_CASE(23)
    default: return CBK_ERR_UNSUPPORTED;
  }
#undef CBK_GB_CASE
}

}  // namespace cbk
