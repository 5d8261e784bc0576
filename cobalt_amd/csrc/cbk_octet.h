// Codes of eight consecutive columns of a packed row, for the kernels that walk a matrix without
// multiplying it (dequantise, unpack, re-pack): a thread owns the columns of one mask byte, so
// neighbouring threads write neighbouring 16-byte pieces of the output, and a code is expanded
// with two byte permutes per mask byte instead of a 32-step bit loop.
#pragma once
#include "cbk_decode.h"

namespace cbk {

constexpr int OCT_LUT_LANES = 4;                                    // lane-private copies of the selector table

__device__ inline void octet_table(uint2 (&lut)[256 * OCT_LUT_LANES]) {   // 256 threads; the caller synchronises
  const uint2 e = make_selectors(threadIdx.x, 0);
#pragma unroll
  for (int j = 0; j < OCT_LUT_LANES; ++j) lut[table_slot<OCT_LUT_LANES, 8>(threadIdx.x, j)] = e;
}

// eight 2-bit codes -> eight nibbles
__device__ inline uint32_t expand2to4(uint32_t x) {
  x = (x | (x << 8)) & 0x00FF00FFu;
  x = (x | (x << 4)) & 0x0F0F0F0Fu;
  return (x | (x << 2)) & 0x33333333u;
}
template <int BITS> __device__ inline uint32_t to_nibbles(uint32_t w) {   // BITS 6: the low nibbles
  return BITS == 2 ? expand2to4(w & 0xFFFFu) : BITS == 3 ? expand3to4(w & 0xFFFFFFu) : w;
}

// The codes of eight columns, one per byte in column order; pruned columns hold 0.  `keep`: the mask byte.
struct Octet { uint32_t lo, hi, keep; };

__device__ inline Octet octet_from_nibbles(uint32_t nib, uint32_t mb, const uint2* lut, uint32_t h0 = 0, uint32_t h1 = 0) {
  const uint2 sel = lut[mb * OCT_LUT_LANES + (threadIdx.x & (OCT_LUT_LANES - 1))];
  const uint32_t p0 = (nib & 0x0F0F0F0Fu) | h0, p1 = ((nib >> 4) & 0x0F0F0F0Fu) | h1;
  return {perm(p1, p0, sel.x), perm(p1, p0, sel.y), mb};
}

// Columns 8 j8 ... 8 j8 + 7 of a row of a fixed-stride layout: FAM / BITS as the descriptor says, any
// survivor count.  Reads at most eight bytes past the row (the tail every image has).
template <int FAM, int BITS>
__device__ inline Octet octet_fixed(const DMat& m, const RowView& row, uint32_t j8, const uint2* lut) {
  if (FAM == FAM_DENSE) {
    const uint32_t d = (j8 * BITS) >> 2, sh = (j8 * BITS & 3u) * 8u;
    if (BITS == 8) {
      const uint2 v = *(const uint2*)(row.unit(j8 >> 1) + (j8 & 1u) * 8u);
      return {v.x, v.y, 0xFFu};
    }
    uint32_t w = row.dword(d);
    if (BITS == 3) w = __builtin_amdgcn_alignbit(row.dword(d + 1), w, sh);
    else if (BITS == 2) w >>= sh;
    const uint32_t n = to_nibbles<BITS>(w);
    const uint32_t p0 = n & 0x0F0F0F0Fu, p1 = (n >> 4) & 0x0F0F0F0Fu;
    return {perm(p1, p0, 0x05010400u), perm(p1, p0, 0x07030602u), 0xFFu};
  }
  const uint32_t t = j8 >> 2, jb = 8u * (j8 & 3u);
  const uint32_t mw = row.dword(t);
  const uint32_t r = (uint32_t)__builtin_popcount(mw & ((1u << jb) - 1u)), mb = (mw >> jb) & 0xFFu;
  constexpr int PB = BITS == 6 ? 4 : BITS;
  const uint32_t bit = (t * (uint32_t)m.keep + r) * PB;
  const uint32_t d = (m.code_off >> 2) + (bit >> 5);
  const uint32_t w = __builtin_amdgcn_alignbit(row.dword(d + 1), row.dword(d), bit & 31u);
  uint32_t h0 = 0, h1 = 0;
  if (BITS == 6) hi2_pools(row.dword(3u * (uint32_t)(m.N >> 5) + t), r, h0, h1);
  return octet_from_nibbles(to_nibbles<BITS>(w), mb, lut, h0, h1);
}

// ---- survivor streams (SPARSE4 / SPARSE4X / SPARSE4E; src/cobaltkernel/pack_cobalt.py:201-250): per row
// [bitmap N/8][uint16 byte offset per group, padded to 16 B; 4X / 4E only][nibbles, every group padded to a byte]
__device__ inline uint32_t stream_header(const DMat& m) {
  return (uint32_t)(((m.N >> 3) + (m.layout != CBK_SPARSE4 ? ((m.G * 2 + 15) & ~15) : 0) + 15) & ~15);
}
constexpr int STREAM_MAX_G = 8192;                                  // groups whose offsets fit the 32 KB a workgroup gives them
inline bool stream_sums(const DMat& m) { return m.layout == CBK_SPARSE4 && m.G <= STREAM_MAX_G; }
// Byte offsets of the groups of a row whose layout does not store them (SPARSE4), into goff[G]: a
// running sum over the groups, by one wavefront.
__device__ inline void stream_offsets(const DMat& m, const uint8_t* row, uint32_t* goff) {
  uint32_t base = 0;
  const int lane = threadIdx.x & 63;
  for (int g0 = 0; g0 < m.G; g0 += 64) {
    const int g = g0 + lane;
    uint32_t c = 0;
    if (g < m.G) {
      const uint4 k = *(const uint4*)(row + (size_t)g * 16);
      c = (uint32_t)(__popc(k.x) + __popc(k.y) + __popc(k.z) + __popc(k.w) + 1) >> 1;
    }
    uint32_t s = c;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t v = (uint32_t)__shfl_up((int)s, o);
      if (lane >= o) s += v;
    }
    if (g < m.G) goff[g] = base + s - c;
    base += (uint32_t)__shfl((int)s, 63);
  }
}
__device__ inline Octet octet_stream(const DMat& m, const uint8_t* row, uint32_t hdr, const uint32_t* goff, uint32_t j8,
                                     const uint2* lut) {
  const uint32_t g = j8 >> 4, i = (j8 >> 2) & 3u, jb = 8u * (j8 & 3u);
  const uint4 k = *(const uint4*)(row + (size_t)g * 16);
  const uint32_t mw = i == 0 ? k.x : i == 1 ? k.y : i == 2 ? k.z : k.w;
  uint32_t r = (uint32_t)__builtin_popcount(mw & ((1u << jb) - 1u));
  r += i > 0 ? (uint32_t)__popc(k.x) : 0u;
  r += i > 1 ? (uint32_t)__popc(k.y) : 0u;
  r += i > 2 ? (uint32_t)__popc(k.z) : 0u;
  uint32_t off = 0;
  if (goff) off = goff[g];
  else if (m.layout != CBK_SPARSE4) off = ((const uint16_t*)(row + (m.N >> 3)))[g];
  else                                                              // more groups than a workgroup keeps offsets of
    for (uint32_t e = 0; e < g; ++e) {
      const uint4 b = *(const uint4*)(row + (size_t)e * 16);
      off += (uint32_t)(__popc(b.x) + __popc(b.y) + __popc(b.z) + __popc(b.w) + 1) >> 1;
    }
  const uint32_t nib = 2u * (hdr + off) + r;                        // nibble of the row (its first byte is 16-byte aligned)
  const uint32_t* w = (const uint32_t*)row + (nib >> 3);
  return octet_from_nibbles(__builtin_amdgcn_alignbit(w[1], w[0], 4u * (nib & 7u)), (mw >> jb) & 0xFFu, lut);
}

// 0 / 1 in every byte: the four low bits of n
__device__ inline uint32_t bits_to_bytes(uint32_t n) { return __umul24(n & 0xFu, 0x204081u) & 0x01010101u; }

}  // namespace cbk
