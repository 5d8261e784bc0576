// RAW arrays (bitmap, codes, scale, zero point) -> the byte image the kernels read, on the GPU.
// The byte layouts are those of the reference's packer (src/cobaltkernel/pack_cobalt.py:98-250,
// docs/FORMAT.md:83-122) and of the two bit-stream layouts of this library (include/cbk.h);
// the destination is either the row-major order or the 16-row tiled order.
//
// A workgroup packs a slab of 4096 columns of sixteen rows (one tile of the tiled order).  A thread
// takes a 32-column block at a time: survivors are moved together by byte permutes from a table
// indexed by the mask byte, narrowed to the code width, and or-ed into the slab's image in LDS; the
// image leaves in whole 16-byte units.  A slab's codes start on a 16-byte unit whatever the code
// width and the survivors per block (128 blocks: 16 * keep * bits bytes).  Bound: reading K*N code
// bytes.  One thread per 256 columns with byte stores, the form before, took 147 us for
// 14336 x 4096 (plus 5 us to clear the destination, every byte of which is written here).
#include <atomic>
#include "cbk_internal.h"
#include "cbk_octet.h"

namespace cbk {

struct PackArgs {
  const uint8_t* mask;     // [K, N/8] or nullptr
  const uint8_t* q;        // [K, N]
  const uint16_t* scale;   // fp16 [K, G]
  const void* zero;        // fp16 or uint8 [K, G]
  uint8_t* data;
  uint16_t* oscale;
  uint8_t* ozero;
  int K, N, G, group, keep, tiled, zero_f16, fix_zero;
  uint32_t stride;
  int slabs, blocks;       // slabs of a row tile, and of the image
  int krows;               // rows of the image: K, or K padded to a multiple of 16 in the tiled order
  uint32_t tail;           // readable bytes behind the last row, zeroed
  int* status;             // see below, or nullptr
  PackExtra extra;         // all zero: rows, scale and zero point only
};

// The quantisation of one group as it is stored: the RAW one, or, when the RAW zero point is off
// the code grid [0, 2^bits - 1], one re-derived from the hull of the group's dequantised
// survivors and 0 (src/cobaltkernel/pack_cobalt.py:55-87).  Every step is a single correctly
// rounded float32 operation in the reference's order, so the bytes do not depend on the device.
struct GroupQ {
  bool redo;
  float z_raw, s_raw, s_new, z_new;
  uint32_t z_out;
  uint16_t s_out;
  bool small;                                                       // redo, and codes of the group: at most 15, map[c / 4] byte c % 4 is the new one
  uint32_t map[4];
  __device__ inline uint32_t code(uint32_t q, float nl) const {
    if (!redo) return q > (uint32_t)nl ? (uint32_t)nl : q;
    const float v = __fmul_rn((float)q - z_raw, s_raw);
    return (uint32_t)fminf(fmaxf(rintf(__fadd_rn(__fdiv_rn(v, s_new), z_new)), 0.f), nl);
  }
};

// sz: the group's scale and, in the upper half, its zero point as given.  q, m: codes and mask of one 32-column block of the group; the blocks of a group are in consecutive
// lanes (four or two of them, all active), which agree on the hull by lane exchanges.  any: bits of q that no code has.
//
// A group that is re-derived costs its whole workgroup the time, as the others wait for it (one group in 500 off the grid
// is two workgroups in three).  So its lanes do not take its 32 codes each through the arithmetic, a division apiece:
// where all codes are at most 2^BITS - 1, the dequantised values are monotonic in the code and none is NaN (the zero
// point is no code), so the hull is that of the smallest and the largest kept one; and the lanes work out the new code of the 16
// there are between them and look theirs up by byte permutes.  14336 x 4096, one group in 500: 28.8 -> 25.7 us (23 without such groups), 24.4 with stores that go on to memory.
template <int BITS>
__device__ inline GroupQ group_quant(const PackArgs& a, float nl, uint32_t sz, const uint32_t (&q)[8], uint32_t m, uint32_t any) {
  GroupQ r;
  r.s_out = (uint16_t)sz;
  r.s_raw = h2f(r.s_out);
  const int zi = a.zero_f16 ? (int)rintf(h2f((uint16_t)(sz >> 16))) : (int)(sz >> 16);
  r.z_raw = (float)zi;
  r.redo = a.fix_zero && (zi < 0 || zi > (int)nl);
  r.z_out = (uint32_t)zi & 0xffu;
  r.s_new = r.s_raw; r.z_new = r.z_raw;
  r.small = false;
  if (!r.redo) return r;
  constexpr float BIG = 3.4028234663852886e38f;
  const int lanes = a.group >> 5;
  float vmin = BIG, vmax = -BIG;
  if (BITS <= 4) {
    for (int o = 1; o < lanes; o <<= 1) any |= (uint32_t)__shfl_xor((int)any, o);
    r.small = any == 0;
  }
  if (r.small) {
    typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
    u16x2 lo = {255, 255}, hi = {0, 0};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t kp = bits_to_bytes(m >> (4 * i)) * 0xFFu, l = q[i] | ~kp, h = q[i] & kp;
      lo = __builtin_elementwise_min(lo, __builtin_bit_cast(u16x2, l & 0x00FF00FFu));
      lo = __builtin_elementwise_min(lo, __builtin_bit_cast(u16x2, (l >> 8) & 0x00FF00FFu));
      hi = __builtin_elementwise_max(hi, __builtin_bit_cast(u16x2, h & 0x00FF00FFu));
      hi = __builtin_elementwise_max(hi, __builtin_bit_cast(u16x2, (h >> 8) & 0x00FF00FFu));
    }
    int least = lo[0] < lo[1] ? lo[0] : lo[1], most = hi[0] > hi[1] ? hi[0] : hi[1];
    for (int o = 1; o < lanes; o <<= 1) {
      const int l = __shfl_xor(least, o), h = __shfl_xor(most, o);
      least = least < l ? least : l; most = most > h ? most : h;
    }
    if (least != 255) {                                             // (a kept code is at most 15)
      const float v0 = __fmul_rn((float)least - r.z_raw, r.s_raw), v1 = __fmul_rn((float)most - r.z_raw, r.s_raw);
      vmin = fminf(v0, v1); vmax = fmaxf(v0, v1);                   // (the scale may be negative)
    }
  } else {
#pragma unroll
    for (int j = 0; j < 32; ++j) {
      const float v = __fmul_rn((float)((q[j >> 2] >> (8 * (j & 3))) & 0xFFu) - r.z_raw, r.s_raw);
      const bool kept = (m >> j) & 1u;
      vmin = kept ? fminf(vmin, v) : vmin;
      vmax = kept ? fmaxf(vmax, v) : vmax;
    }
    for (int o = 1; o < lanes; o <<= 1) {
      vmin = fminf(vmin, __shfl_xor(vmin, o));
      vmax = fmaxf(vmax, __shfl_xor(vmax, o));
    }
  }
  vmin = fminf(vmin, 0.f); vmax = fmaxf(vmax, 0.f);                // (a group without survivors: 0 and 0)
  r.s_new = fmaxf(__fdiv_rn(__fsub_rn(vmax, vmin), nl), 1e-12f);
  r.z_new = fminf(fmaxf(rintf(__fdiv_rn(-vmin, r.s_new)), 0.f), nl);
  r.z_out = (uint32_t)r.z_new;
  r.s_out = f2h(r.s_new);
  if (r.small) {
    auto four = [&](uint32_t c) {
      uint32_t w = 0;
      for (uint32_t e = 0; e < 4; ++e) w |= r.code(c + e, nl) << (8 * e);
      return w;
    };
    const uint32_t at = threadIdx.x & (uint32_t)(lanes - 1);
    if (lanes == 4) {                                               // lane i of the four: codes 4 i ... 4 i + 3
      const int w = (int)four(4 * at);
      r.map[0] = (uint32_t)__builtin_amdgcn_update_dpp(0, w, 0x00, 0xf, 0xf, false);
      r.map[1] = (uint32_t)__builtin_amdgcn_update_dpp(0, w, 0x55, 0xf, 0xf, false);
      r.map[2] = (uint32_t)__builtin_amdgcn_update_dpp(0, w, 0xAA, 0xf, 0xf, false);
      r.map[3] = (uint32_t)__builtin_amdgcn_update_dpp(0, w, 0xFF, 0xf, 0xf, false);
    } else {                                                        // of the two: eight each
      const int w0 = (int)four(8 * at), w1 = (int)four(8 * at + 4);
      r.map[0] = (uint32_t)__builtin_amdgcn_update_dpp(0, w0, 0xA0, 0xf, 0xf, false);
      r.map[1] = (uint32_t)__builtin_amdgcn_update_dpp(0, w1, 0xA0, 0xf, 0xf, false);
      r.map[2] = (uint32_t)__builtin_amdgcn_update_dpp(0, w0, 0xF5, 0xf, 0xf, false);
      r.map[3] = (uint32_t)__builtin_amdgcn_update_dpp(0, w1, 0xF5, 0xf, 0xf, false);
    }
  }
  return r;
}

constexpr int PK_ROWS = PACK_ROWS, PK_COLS = PACK_COLS, PK_THREADS = 512;

// permute selectors that move the survivors of eight bytes together: output byte i takes the i-th
// survivor (zero past the last)
__device__ inline uint2 compress_selectors(uint32_t mb) {
  uint32_t lo = 0x0C0C0C0Cu, hi = 0x0C0C0C0Cu, r = 0;
#pragma unroll
  for (uint32_t p = 0; p < 8; ++p) {
    if ((mb >> p) & 1u) {
      const uint32_t sh = 8 * (r & 3u), put = (p ^ 0x0Cu) << sh;   // 0x0C -> p
      if (r < 4) lo ^= put; else hi ^= put;
      ++r;
    }
  }
  return make_uint2(lo, hi);
}

// eight bytes holding codes of `bits` bits -> 8 * bits bits, first code lowest
template <int bits>
__device__ inline uint64_t narrow8(uint32_t lo, uint32_t hi) {
  if (bits == 8) return (uint64_t)lo | ((uint64_t)hi << 32);
  // (bytes 0 and 2 of x | x >> 4 are the pairs of nibbles, as no code has bits above them)
  if (bits == 4) return (uint64_t)perm(hi | (hi >> 4), lo | (lo >> 4), 0x06040200u);
  auto four = [&](uint32_t x) -> uint32_t {                         // four bytes -> 4 * bits bits
    const uint32_t mask = ((1u << bits) - 1u) * 0x00010001u;
    const uint32_t y = (x & mask) | (((x >> 8) & mask) << bits);    // pairs at bits 0 and 16
    return (y & ((1u << (2 * bits)) - 1u)) | ((y >> 16) << (2 * bits));
  };
  return (uint64_t)four(lo) | ((uint64_t)four(hi) << (4 * bits));
}

// status[0] |= 1: a block without exactly `keep` survivors; |= 2: a dense layout had to store a zero
// point above 2^bits - 1 at a pruned column (its low bits are stored; the column no longer
// dequantises to 0); status[1] += groups re-derived
template <int FAM, int BITS>
__global__ __launch_bounds__(PK_THREADS) void pack_rows_kernel(PackArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint32_t img[];   // [PK_ROWS][code bytes of a slab (+ its BLK6 high plane)]
  __shared__ uint2 lut[256];
  __shared__ uint4 tot[PK_THREADS / 64];                            // status bits, groups re-derived, largest zero, survivors
  const int tid = threadIdx.x;
  constexpr bool dense = FAM == FAM_DENSE, blk6 = FAM == FAM_BLK6;
  if (tid < 256) lut[tid] = compress_selectors((uint32_t)tid);
  uint32_t st = 0, fixed = 0, zmax = 0, surv = 0;
  // (one slab per workgroup but for images of more than PACK_RECORDS slabs)
  for (int slab = blockIdx.x; slab < a.blocks; slab += gridDim.x) {
  const int rt = slab / a.slabs, c0 = (slab % a.slabs) * PK_COLS, k0 = rt * PK_ROWS;
  const int cols = a.N - c0 < PK_COLS ? a.N - c0 : PK_COLS, nb = cols >> 5;
  constexpr int pb = blk6 ? 4 : BITS;                               // bits per code of the code plane
  const int cb = (dense ? 32 : a.keep) * pb;                       // code bits of a block
  const uint32_t plane = (uint32_t)a.N >> 3;
  const uint32_t cbytes = ((uint32_t)nb * cb + 127) / 128 * 16;    // code bytes of the slab's rows, whole units
  const uint32_t hbytes = blk6 ? (uint32_t)nb * 4u : 0u;
  const uint32_t pitch = (cbytes + hbytes) >> 2;                   // dwords per row of the image
  for (uint32_t i = tid; i < PK_ROWS * pitch; i += PK_THREADS) img[i] = 0;
  __syncthreads();
  const float nl = (float)((1u << BITS) - 1u);
  const uint32_t over = ~((uint32_t)nl * 0x01010101u);             // bits that no code of this width has
  // codes, mask, scale and zero point of the next block are in flight while one is packed
  struct In { uint4 qa, qb; uint32_t m, sz; };
  const int rows_in = a.K - k0 < PK_ROWS ? a.K - k0 : PK_ROWS;      // (padding rows have no blocks)
  // a thread's blocks: every PK_THREADS-th of the slab's, row by row
  const int drow = PK_THREADS / nb, dt = PK_THREADS % nb, lg = a.group == 64 ? 6 : 7;
  const uint8_t* qb = a.q + (size_t)k0 * a.N + c0;
  const uint8_t* mb = a.mask ? a.mask + (size_t)k0 * plane + (c0 >> 3) : nullptr;
  const size_t gb = (size_t)k0 * a.G + (c0 >> lg);
  const uint16_t* sb = a.scale + gb;
  const uint8_t* zb = (const uint8_t*)a.zero + (a.zero_f16 ? 2 * gb : gb);
  auto load = [&](int row, int t) -> In {
    if (row >= rows_in) { row = rows_in - 1; t = 0; }
    // (sixteen rows: 32-bit offsets from an address all threads share)
    const uint32_t gi = (uint32_t)row * (uint32_t)a.G + (((uint32_t)t * 32u) >> lg), qo = (uint32_t)row * (uint32_t)a.N + (uint32_t)t * 32u;
    In x;
    x.qa = *(const uint4*)(qb + qo); x.qb = *(const uint4*)(qb + 16 + qo);
    x.m = mb ? *(const uint32_t*)(mb + (uint32_t)row * plane + (uint32_t)t * 4u) : 0xffffffffu;
    x.sz = (uint32_t)sb[gi] | ((a.zero_f16 ? (uint32_t)((const uint16_t*)zb)[gi] : (uint32_t)zb[gi]) << 16);
    return x;
  };
  int row = tid / nb, t = tid % nb;
  In nx = load(row, t);
  for (int nrow, nt; row < rows_in; row = nrow, t = nt) {
    const In cur = nx;
    nrow = row + drow; nt = t + dt;
    if (nt >= nb) { nt -= nb; ++nrow; }
    nx = load(nrow, nt);
    const int k = k0 + row, c = c0 + 32 * t, g = c >> lg;
    uint32_t q[8] = {cur.qa.x, cur.qa.y, cur.qa.z, cur.qa.w, cur.qb.x, cur.qb.y, cur.qb.z, cur.qb.w};
    const uint32_t m = cur.m;
    surv += (uint32_t)__popc(m);
    uint32_t any = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) any |= q[i] & over;
    const GroupQ gq = group_quant<BITS>(a, nl, cur.sz, q, m, any);
    if ((c & (a.group - 1)) == 0) {                                // the group's first block stores its quantisation
      const size_t mi = a.tiled ? ((size_t)rt * a.G + g) * 16 + row : (size_t)k * a.G + g;
      a.oscale[mi] = gq.s_out;
      a.ozero[mi] = (uint8_t)gq.z_out;
      fixed += gq.redo ? 1u : 0u;
      zmax = zmax > gq.z_out ? zmax : gq.z_out;
    }
    if (BITS <= 4 && gq.small) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const uint32_t sel = q[i] & 0x07070707u, up = ((q[i] >> 3) & 0x01010101u) * 0xFFu;
        q[i] = (perm(gq.map[1], gq.map[0], sel) & ~up) | (perm(gq.map[3], gq.map[2], sel) & up);
      }
    } else if (gq.redo || any) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        uint32_t w = 0;
        for (int e = 0; e < 4; ++e) w |= gq.code((q[i] >> (8 * e)) & 0xFFu, nl) << (8 * e);
        q[i] = w;
      }
    }
    uint32_t* dst = img + row * pitch;
    if (dense) {
      if (m != 0xffffffffu && gq.z_out > (uint32_t)nl) st |= 2u;
      const uint32_t z4 = (gq.z_out & (uint32_t)nl) * 0x01010101u;
      uint64_t w[4];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const uint32_t kp = bits_to_bytes(m >> (4 * i)) * 0xFFu;
        q[i] = (q[i] & kp) | (z4 & ~kp);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) w[i] = narrow8<pb>(q[2 * i], q[2 * i + 1]);
      uint32_t* d = dst + t * pb;                                  // a block is pb whole dwords
      if (pb == 8) {
#pragma unroll
        for (int i = 0; i < 4; ++i) { d[2 * i] = (uint32_t)w[i]; d[2 * i + 1] = (uint32_t)(w[i] >> 32); }
      } else if (pb == 4) {
#pragma unroll
        for (int i = 0; i < 4; ++i) d[i] = (uint32_t)w[i];
      } else if (pb == 3) {
        const uint64_t x = w[0] | (w[1] << 24), y = w[2] | (w[3] << 24);     // 48 bits each
        d[0] = (uint32_t)x; d[1] = (uint32_t)(x >> 32) | ((uint32_t)y << 16); d[2] = (uint32_t)(y >> 16);
      } else {
        d[0] = (uint32_t)w[0] | ((uint32_t)w[1] << 16); d[1] = (uint32_t)w[2] | ((uint32_t)w[3] << 16);
      }
      continue;
    }
    if (__popc(m) != a.keep) st |= 1u;
    // survivors of the block, at most `keep` of them, as one bit string of at most 128 bits
    static_assert(dense || pb <= 4, "the codes of a mask byte are at most 32 bits");
    uint32_t hw = 0, w[4], at[4];                                  // codes of a mask byte, bits of those before it
    int r = 0;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const uint32_t mb = (m >> (8 * b)) & 0xFFu;
      const uint2 sel = lut[mb];
      uint32_t lo = perm(q[2 * b + 1], q[2 * b], sel.x), hi = perm(q[2 * b + 1], q[2 * b], sel.y);
      if (blk6) {                                                  // high bit pairs: even survivors from bit 0, odd ones from bit 16
        for (int i = 0; i < 8; ++i) {
          const uint32_t cd = ((i < 4 ? lo : hi) >> (8 * (i & 3))) & 0xFFu;
          const int e = r + i;
          if (e < 16) hw |= (cd >> 4) << (2 * (e >> 1) + 16 * (e & 1));
        }
        lo &= 0x0F0F0F0Fu; hi &= 0x0F0F0F0Fu;
      }
      w[b] = (uint32_t)narrow8<pb>(lo, hi);
      at[b] = (uint32_t)(r * pb);
      r += __popc(mb);
    }
    // two mask bytes at a time (at most 64 bits), then the second two behind the first
    const uint64_t front = w[0] | ((uint64_t)w[1] << at[1]), back = w[2] | ((uint64_t)w[3] << (at[3] - at[2]));
    uint64_t s0 = front | (at[2] < 64 ? back << (at[2] & 63u) : 0), s1 = at[2] == 0 ? 0 : at[2] < 64 ? back >> ((64u - at[2]) & 63u) : back;
    if (cb < 64) { s0 &= (1ull << (cb & 63)) - 1ull; s1 = 0; }            // (too many survivors: an error, but never into the next block)
    else if (cb < 128) s1 &= (1ull << (cb & 63)) - 1ull;
    const uint32_t bit = (uint32_t)t * cb, sh = bit & 31u;
    uint32_t* d = dst + (bit >> 5);
    const uint32_t x[4] = {(uint32_t)s0, (uint32_t)(s0 >> 32), (uint32_t)s1, (uint32_t)(s1 >> 32)};
    const int nd = (int)(sh + cb + 31) >> 5;
    if ((cb & 31) == 0) {                                          // whole dwords: nobody shares them
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (i < nd) d[i] = x[i];
    } else {
#pragma unroll
      for (int i = 0; i < 5; ++i) {
        if (i >= nd) break;
        const uint32_t lo = i < 4 ? x[i] : 0u, pre = i > 0 ? x[i - 1] : 0u;
        const uint32_t v = sh ? (lo << sh) | (pre >> (32 - sh)) : lo;
        if (v) atomicOr(d + i, v);
      }
    }
    if (blk6) dst[(cbytes >> 2) + t] = hw;
  }
  __syncthreads();
  // the image, unit by unit: consecutive threads write the rows of a unit (tiled: a 256-byte run) or the units of a row
  const auto rows_at = through_buffer(a.data + (size_t)rt * 16 * a.stride);
  auto unit_at = [&](int row, uint32_t o) -> uint32_t {            // o: byte offset in the row, a multiple of 16
    return a.tiled ? o * 16 + (uint32_t)row * 16 : (uint32_t)row * a.stride + o;
  };
  const int rows = a.krows - k0 < PK_ROWS ? a.krows - k0 : PK_ROWS;
  auto put = [&](uint32_t units, uint32_t o0, auto&& get) {
    for (uint32_t i = tid; i < PK_ROWS * units; i += PK_THREADS) {
      const int row = a.tiled ? (int)(i & 15u) : (int)(i / units);
      const uint32_t u = a.tiled ? i >> 4 : i % units;
      if (row < rows) store16_through(rows_at, unit_at(row, o0 + u * 16), get(row, u));
    }
  };
  put(cbytes >> 4, (dense ? 0u : plane) + (uint32_t)(c0 >> 5) * (uint32_t)cb / 8,
      [&](int row, uint32_t u) { return *(const uint4*)(img + row * pitch + 4 * u); });
  if (blk6) put(hbytes >> 4, plane * 3u + (uint32_t)(c0 >> 3),
                [&](int row, uint32_t u) { return *(const uint4*)(img + row * pitch + (cbytes >> 2) + 4 * u); });
  if (!dense)
    put((uint32_t)cols >> 7, (uint32_t)(c0 >> 3), [&](int row, uint32_t u) {
      if (k0 + row >= a.K) return make_uint4(0, 0, 0, 0);
      if (!a.mask) return make_uint4(~0u, ~0u, ~0u, ~0u);
      const uint32_t* p = (const uint32_t*)(a.mask + (size_t)(k0 + row) * plane + (c0 >> 3)) + 4 * u;
      return make_uint4(p[0], p[1], p[2], p[3]);
    });
  // padding rows have no groups of their own; the bytes behind the last row
  if (c0 == 0 && k0 + PK_ROWS > a.K && a.tiled)
    for (int i = tid; i < (k0 + PK_ROWS - a.K) * a.G; i += PK_THREADS) {
      const size_t mi = ((size_t)rt * a.G + i % a.G) * 16 + (a.K - k0) + i / a.G;
      a.oscale[mi] = 0;
      a.ozero[mi] = 0;
    }
  if (slab + (int)gridDim.x < a.blocks) __syncthreads();           // the image has been read
  }
  if (blockIdx.x == 0 && tid < (int)(a.tail >> 4)) ((uint4*)(a.data + (size_t)a.krows * a.stride))[tid] = make_uint4(0, 0, 0, 0);
  for (uint32_t i = blockIdx.x * (uint32_t)PK_THREADS + tid; i < a.extra.cs_units; i += gridDim.x * (uint32_t)PK_THREADS)
    ((uint4*)a.extra.cs_dst)[i] = ((const uint4*)a.extra.cs_src)[i];
  if (blockIdx.x == 0)
    for (int i = 0; i < 4; ++i)
      if (tid < (int)a.extra.gap_bytes[i]) a.extra.gap[i][tid] = 0;
  if (a.status || a.extra.counts) {                                 // one record per workgroup, added over lanes, then wavefronts
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      st |= (uint32_t)__shfl_xor((int)st, o);
      fixed += (uint32_t)__shfl_xor((int)fixed, o);
      const uint32_t z = (uint32_t)__shfl_xor((int)zmax, o);
      zmax = zmax > z ? zmax : z;
      surv += (uint32_t)__shfl_xor((int)surv, o);
    }
    if ((tid & 63) == 0) tot[tid >> 6] = make_uint4(st, fixed, zmax, surv);
    __syncthreads();
    if (tid == 0) {
      uint4 t = tot[0];
      for (int w = 1; w < PK_THREADS / 64; ++w) {
        const uint4 u = tot[w];
        t.x |= u.x; t.y += u.y; t.z = t.z > u.z ? t.z : u.z; t.w += u.w;
      }
      if (a.status && t.x) atomicOr(a.status, (int)t.x);
      if (a.status && t.y) atomicAdd(a.status + 1, (int)t.y);
      if (a.extra.counts) ((uint4*)a.extra.counts)[blockIdx.x] = t;
    }
  }
}

// ------------------------------------------------------------------ the way back: image -> RAW
// Codes (0 at a pruned column of a bitmap or survivor-stream layout, the stored code, i.e. the
// zero point, at a pruned column of a dense layout) and the keep bitmap of any layout.
// A thread per eight columns.
template <int FAM, int BITS>
__global__ __launch_bounds__(256) void unpack_fixed_kernel(DMat m, uint8_t* q, uint8_t* mask) {
  __shared__ uint2 lut[256 * OCT_LUT_LANES];
  if (FAM != FAM_DENSE) { octet_table(lut); __syncthreads(); }
  const uint32_t n8 = (uint32_t)m.N >> 3;
  const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int rt = (int)(id / n8);
  const uint32_t j8 = (uint32_t)(id % n8);
  const int k1 = rt * 16 + 16 < m.K ? rt * 16 + 16 : m.K;
#pragma unroll 4
  for (int k = rt * 16; k < k1; ++k) {
    const Octet o = octet_fixed<FAM, BITS>(m, row_view(m, k), j8, lut);
    *(uint2*)(q + (size_t)k * m.N + 8 * (size_t)j8) = make_uint2(o.lo, o.hi);
    if (mask) mask[(size_t)k * n8 + j8] = (uint8_t)o.keep;
  }
}

// Survivor streams, a workgroup per four rows.
__global__ __launch_bounds__(256) void unpack_sparse_kernel(DMat m, uint8_t* q, uint8_t* mask, int summed) {
  extern __shared__ uint32_t goff[];
  __shared__ uint2 lut[256 * OCT_LUT_LANES];
  octet_table(lut);
  const uint32_t hdr = stream_header(m), n8 = (uint32_t)m.N >> 3;
  const int k0 = blockIdx.x * 4, k1 = m.K - k0 < 4 ? m.K : k0 + 4;
  for (int k = k0; k < k1; ++k) {
    const uint8_t* row = m.data + m.row_off[k];
    __syncthreads();                                                // the table; the offsets of the row before
    if (summed) {
      if (threadIdx.x < 64) stream_offsets(m, row, goff);
      __syncthreads();
    }
    for (uint32_t j8 = threadIdx.x; j8 < n8; j8 += 256) {
      const Octet o = octet_stream(m, row, hdr, summed ? goff : nullptr, j8, lut);
      *(uint2*)(q + (size_t)k * m.N + 8 * (size_t)j8) = make_uint2(o.lo, o.hi);
      if (mask) mask[(size_t)k * n8 + j8] = (uint8_t)o.keep;
    }
  }
}

// A survivor-stream matrix as dense 4-bit rows in tiled order (a pruned column holds its group's zero
// point), which is how a prefill call re-packs it: one pass over the stream.
//
// A workgroup takes a tile of sixteen rows; lane 16 b + r decodes block b (32 columns) of a group of row
// r, so the sixteen rows' units of a block leave as 256 contiguous bytes, and the wavefronts walk
// neighbouring groups together: the cache lines of the sixteen rows' masks and codes are read once.
// (A thread per octet of four rows wrote four bytes at a time and looked its group's offset, mask words,
// zero point and scale up for each.  A call of 21504 x 5376 at 128 rows 226 us, 99 now.)
constexpr int RP_WIN = 256;                                         // groups whose offsets are summed at a time (SPARSE4)
__global__ __launch_bounds__(1024) void repack_tile_kernel(DMat m, uint8_t* out, uint16_t* oscale, uint8_t* ozero) {
  __shared__ uint2 lut[256 * OCT_LUT_LANES];
  __shared__ uint32_t goff[16][RP_WIN + 1];                         // (+1: the sixteen rows of a group in different banks)
  __shared__ uint32_t carry[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nw = (int)blockDim.x >> 6;
  if (tid < 256) octet_table(lut);
  const int r = lane & 15, b = lane >> 4, k = (int)blockIdx.x * 16 + r, kc = k < m.K ? k : m.K - 1;
  const uint32_t hdr = stream_header(m);
  const uint8_t* row = m.data + m.row_off[kc];
  const bool sums = m.layout == CBK_SPARSE4;
  uint8_t* tile = out + (size_t)blockIdx.x * 16 * (m.N >> 1);
  for (int g0 = 0; g0 < m.G; g0 += RP_WIN) {
    const int g1 = m.G - g0 < RP_WIN ? m.G : g0 + RP_WIN;
    __syncthreads();                                                // the table; the offsets of the window before
    if (sums) {
      for (int rr = wave; rr < 16; rr += nw) {                      // a wavefront keeps its rows over the windows
        const int kr = (int)blockIdx.x * 16 + rr;
        const uint8_t* rp = m.data + m.row_off[kr < m.K ? kr : m.K - 1];
        uint32_t base = g0 ? carry[rr] : 0u;
        for (int gw = g0; gw < g1; gw += 64) {
          const int g = gw + lane;
          uint32_t c = 0;
          if (g < g1) {
            const uint4 w = *(const uint4*)(rp + (size_t)g * 16);
            c = (uint32_t)(__popc(w.x) + __popc(w.y) + __popc(w.z) + __popc(w.w) + 1) >> 1;
          }
          uint32_t s = c;
#pragma unroll
          for (int o = 1; o < 64; o <<= 1) {
            const uint32_t v = (uint32_t)__shfl_up((int)s, o);
            if (lane >= o) s += v;
          }
          if (g < g1) goff[rr][g - g0] = base + s - c;
          base += (uint32_t)__shfl((int)s, 63);
        }
        if (lane == 0) carry[rr] = base;
      }
      __syncthreads();
    }
    struct Head { uint4 k; uint32_t off, z, sc; };
    auto head = [&](int g) -> Head {
      g = g < g1 ? g : g1 - 1;
      Head h;
      h.k = *(const uint4*)(row + (size_t)g * 16);
      h.off = sums ? goff[r][g - g0] : ((const uint16_t*)(row + (m.N >> 3)))[g];
      const size_t mi = (size_t)kc * m.G + g;
      h.z = m.zero[mi]; h.sc = m.scale[mi];
      return h;
    };
    Head nx = head(g0 + wave);
    for (int g = g0 + wave; g < g1; g += nw) {
      const Head h = nx;
      const uint32_t c0 = (uint32_t)__popc(h.k.x), c1 = c0 + (uint32_t)__popc(h.k.y), c2 = c1 + (uint32_t)__popc(h.k.z);
      const uint32_t mw = b == 0 ? h.k.x : b == 1 ? h.k.y : b == 2 ? h.k.z : h.k.w;
      const uint32_t nib = 2u * (hdr + h.off) + (b == 0 ? 0u : b == 1 ? c0 : b == 2 ? c1 : c2);   // the block's first code
      const uint32_t* cp = (const uint32_t*)row + (nib >> 3);
      uint32_t e[5];
#pragma unroll
      for (int i = 0; i < 4; ++i) e[i] = cp[i];                     // rows end in a readable tail
      e[4] = 0;
      if ((nib & 7u) + (uint32_t)__popc(mw) > 32u) e[4] = cp[4];
      nx = head(g + nw);
      uint32_t st[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) st[i] = __builtin_amdgcn_alignbit(e[i + 1], e[i], 4u * (nib & 7u));
      const uint32_t z4 = (h.z & 0xFu) * 0x01010101u;
      uint32_t w[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t before = i ? (uint32_t)__popc(mw & ((1u << (8 * i)) - 1u)) : 0u;
        const Octet o = octet_from_nibbles(i ? window<4>(st, 4u * before) : st[0], (mw >> (8 * i)) & 0xFFu, lut);
        const uint32_t lo = mask_select(bits_to_bytes(o.keep) * 0xFFu, z4, o.lo), hi = mask_select(bits_to_bytes(o.keep >> 4) * 0xFFu, z4, o.hi);
        w[i] = (uint32_t)narrow8<4>(lo, hi);
      }
      const bool ok = k < m.K;                                      // (the padding rows of the last tile are zero)
      *(uint4*)(tile + ((size_t)g * 4 + b) * 256 + r * 16) = ok ? make_uint4(w[0], w[1], w[2], w[3]) : make_uint4(0, 0, 0, 0);
      if (b == 0) {
        const size_t at = ((size_t)blockIdx.x * m.G + g) * 16 + r;
        oscale[at] = (uint16_t)(ok ? h.sc : 0u);
        ozero[at] = (uint8_t)(ok ? h.z : 0u);
      }
    }
  }
  if (blockIdx.x == 0 && tid < 32)                                  // readable bytes behind the last tile
    ((uint4*)(out + (size_t)gridDim.x * 16 * (m.N >> 1)))[tid] = make_uint4(0, 0, 0, 0);
}

int launch_unpack(const DMat& m, void* q, void* mask, hipStream_t st) {
  const int fam = family_of(m.layout);
  const dim3 blk(256);
  uint8_t *qb = (uint8_t*)q, *mb = (uint8_t*)mask;
  if (fam == FAM_SPARSE) {
    const int summed = stream_sums(m) ? 1 : 0;
    hipLaunchKernelGGL(unpack_sparse_kernel, dim3((unsigned)((m.K + 3) / 4)), blk, summed ? (size_t)m.G * 4 : 0, st, m, qb, mb, summed);
  } else {
    const dim3 grid((unsigned)(((int64_t)((m.K + 15) / 16) * (m.N / 8) + 255) / 256));
    if (fam == FAM_BLK6) hipLaunchKernelGGL((unpack_fixed_kernel<FAM_BLK6, 6>), grid, blk, 0, st, m, qb, mb);
    else if (fam == FAM_DENSE) {
      if (m.bits == 2) hipLaunchKernelGGL((unpack_fixed_kernel<FAM_DENSE, 2>), grid, blk, 0, st, m, qb, mb);
      else if (m.bits == 3) hipLaunchKernelGGL((unpack_fixed_kernel<FAM_DENSE, 3>), grid, blk, 0, st, m, qb, mb);
      else if (m.bits == 4) hipLaunchKernelGGL((unpack_fixed_kernel<FAM_DENSE, 4>), grid, blk, 0, st, m, qb, mb);
      else hipLaunchKernelGGL((unpack_fixed_kernel<FAM_DENSE, 8>), grid, blk, 0, st, m, qb, mb);
    } else {
      if (m.bits == 2) hipLaunchKernelGGL((unpack_fixed_kernel<FAM_BLK, 2>), grid, blk, 0, st, m, qb, mb);
      else if (m.bits == 3) hipLaunchKernelGGL((unpack_fixed_kernel<FAM_BLK, 3>), grid, blk, 0, st, m, qb, mb);
      else hipLaunchKernelGGL((unpack_fixed_kernel<FAM_BLK, 4>), grid, blk, 0, st, m, qb, mb);
    }
  }
  return hipGetLastError() == hipSuccess ? CBK_OK : CBK_ERR_HIP;
}

// A survivor-stream matrix as dense 4-bit rows in tiled order: d.data, d.scale, d.zero of the sizes
// that layout has.
int launch_repack_dense4(const DMat& m, const DMat& d, hipStream_t st) {
  // about 4096 wavefronts and more; a wavefront of a wide workgroup has a few groups only
  const int tiles = (m.K + 15) / 16, threads = tiles >= 1024 ? 256 : tiles >= 512 ? 512 : 1024;
  hipLaunchKernelGGL(repack_tile_kernel, dim3((unsigned)tiles), dim3(threads), 0, st, m, (uint8_t*)d.data, (uint16_t*)d.scale,
                     (uint8_t*)d.zero);
  return hipGetLastError() == hipSuccess ? CBK_OK : CBK_ERR_HIP;
}

template <int FAM, int BITS>
static int launch_pack_cfg(const PackArgs& a, size_t lds, hipStream_t st) {
  auto kern = pack_rows_kernel<FAM, BITS>;
  static std::atomic<int> configured{0};
  if (!configured.load(std::memory_order_acquire)) {               // 64 KB for a slab of 8-bit codes, and the table
    if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 128 * 1024) != hipSuccess)
      return CBK_ERR_HIP;
    configured.store(1, std::memory_order_release);
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)pack_records(a.K, a.N)), dim3(PK_THREADS), lds, st, a);
  return hipGetLastError() == hipSuccess ? CBK_OK : CBK_ERR_HIP;
}

int launch_pack(const DMat& m, const void* mask, const void* q, const void* scale, const void* zero, int zero_f16,
                int fix_zero, int* status, const PackExtra* extra, hipStream_t st) {
  const int fam = family_of(m.layout);
  if (fam == FAM_SPARSE) return CBK_ERR_UNSUPPORTED;
  PackArgs a;
  a.mask = (const uint8_t*)mask; a.q = (const uint8_t*)q; a.scale = (const uint16_t*)scale; a.zero = zero;
  a.data = (uint8_t*)m.data; a.oscale = (uint16_t*)m.scale; a.ozero = (uint8_t*)m.zero;
  a.K = m.K; a.N = m.N; a.G = m.G; a.group = m.group; a.keep = m.keep; a.tiled = m.tiled;
  a.zero_f16 = zero_f16; a.fix_zero = fix_zero;
  a.stride = m.stride;
  a.krows = m.tiled ? (m.K + 15) / 16 * 16 : m.K;
  a.tail = m.tiled ? 512 : 64;
  a.status = status;
  a.extra = extra ? *extra : PackExtra{};
  a.slabs = (m.N + PK_COLS - 1) / PK_COLS;
  a.blocks = (m.K + PK_ROWS - 1) / PK_ROWS * a.slabs;
  const int cols = m.N < PK_COLS ? m.N : PK_COLS, pb = fam == FAM_BLK6 ? 4 : m.bits;
  const size_t row = (size_t)((cols / 32) * (fam == FAM_DENSE ? 32 : m.keep) * pb + 127) / 128 * 16 +
                     (fam == FAM_BLK6 ? (size_t)cols / 8 : 0);
  if (fam == FAM_BLK6) return launch_pack_cfg<FAM_BLK6, 6>(a, PK_ROWS * row, st);
  if (fam == FAM_DENSE)
    return m.bits == 2 ? launch_pack_cfg<FAM_DENSE, 2>(a, PK_ROWS * row, st)
         : m.bits == 3 ? launch_pack_cfg<FAM_DENSE, 3>(a, PK_ROWS * row, st)
         : m.bits == 4 ? launch_pack_cfg<FAM_DENSE, 4>(a, PK_ROWS * row, st)
                       : launch_pack_cfg<FAM_DENSE, 8>(a, PK_ROWS * row, st);
  return m.bits == 2 ? launch_pack_cfg<FAM_BLK, 2>(a, PK_ROWS * row, st)
       : m.bits == 3 ? launch_pack_cfg<FAM_BLK, 3>(a, PK_ROWS * row, st)
                     : launch_pack_cfg<FAM_BLK, 4>(a, PK_ROWS * row, st);
}

}  // namespace cbk
