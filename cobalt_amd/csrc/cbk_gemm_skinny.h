// GEMM for calls of nine to a few hundred activation rows:  Y[M, K] = X[M, N] . W_hat[K, N]^T.
//
// What bounds such a call is decoding the weights once, in vector instructions per weight, so the kernel
// is built around that.
//  * A decoded octet of columns never leaves the registers of the lane that decoded it: the B operand of
//    v_mfma_f32_32x32x16_f16 is, per lane, eight columns of one weight row, what one mask byte decodes
//    to.  A wavefront owns 64 weight rows (two such operands) and up to 64 activation rows.  There is no
//    weight tile in LDS and no barrier in the loop; two wavefronts per SIMD cover each other's waits.
//  * Everything is a byte permute: codes to their columns, the zero point into the pruned columns (which
//    so subtract to 0), bytes to halves BASE + code (SkCfg::BASE), exact.
//  * Tiles of up to 64 tokens multiply these halves as they are.  Once per quantisation group the float32
//    sum is corrected by -(BASE + zero) * sum(X' of the group), one more matrix step whose A operand is
//    that sum (as two halves), and multiplied by the group's scale on its way into the result: 37 vector
//    instructions per step of 16 columns x 64 rows where a subtraction and a multiplication per weight
//    need 52, and weights that are not rounded at all.  BASE is as small as a byte allows, because the matrix pipe
//    does not round its sums but cuts them off (measured), and what it cuts off a sum of BASE * X' of one sign adds
//    up: all activations positive, 2-bit codes with 10 of 32 kept in groups of 128, error against float64 2.2e-4
//    with BASE 1024, 0.7e-4 with 4; operands rounded to halves have 1.3e-4.  (Subnormal halves, code * 2^-24, need
//    no BASE, but the pipe loses more of those: 1.8e-4 for rows of 14336 columns.)
//    Tiles of 96 tokens have no registers for a second set of sums; they subtract and multiply per weight.
//  * What a step costs is counted in vector instructions at their price: with two or more wavefronts on a SIMD and, or,
//    xor, add, right shift, three-input logic, v_fma_f32 and v_mul_f32 on registers take 2.3 to 2.7 cycles, permutes, left
//    and 64-bit shifts, counts, packed halves, v_fma_mix_f32 and anything with a scalar operand 4.4.  So memory is read
//    through buffer descriptors (lane offset + scalar offset, no vector addition), the table starts LDS (an entry's
//    offset is its address), and scales are floats before they multiply: 4-bit codes, 64 tokens, 168 -> 135 cycles per
//    step of 16 columns x 64 rows beside 144 of matrix instructions.  With the preparation, before and after: feed-forward
//    block 14336 x 4096 at 48 rows 61.7 -> 58.9 us, 2-bit 6144 x 4096 at 333 rows 43.2 -> 41.6, fixed-stride 8-bit down
//    projection 4096 x 14336 at 512 rows 90.0 -> 85.3.
//  * No one unit is full.  Of a SIMD's cycles at 48, 333 and 512 rows of these three calls the matrix instructions take
//    34, 35 and 46 %, the other vector instructions (four cycles each) 42, 42 and 39 %, both at once 15, 17 and 22 %; a
//    wavefront waits at a counter or a barrier for 31, 33 and 25 % of its life; L2 sends a CU 28, 20 and 38 bytes per cycle.
//    The clock falls as the matrix share grows (1.8, 1.9 and 1.6 GHz, life over duration).  (The older of the two
//    wavefronts of a SIMD ends 25 % early; priorities that keep them level leave the end where it is.)
//
// k order.  A step is eight columns of the first half of a group (lanes 0-31) and eight of the second
// (lanes 32-63): a lane walks half a group of its own row, nothing is loaded or ranked twice.  The
// activations X' = fp16(x * col_scale / s_m) are written in that order by the preparation kernel, as
// whole 1 KB fragments [group][step][32-token block][lane], and come from L2 straight into registers,
// several steps ahead.  s_m is the power of two that brings the largest |x * col_scale| of a token and
// column part into [128, 256): neither X' nor the sum of a group leaves the range of a half, and the
// scaling is exact.
//
// A workgroup is eight wavefronts: two row groups of 64 rows (for a gate/up matrix: the even and the
// odd rows of 128) times four parts of the column range.  The parts are added through LDS in part
// order, so results do not depend on timing; where the rows alone do not fill the chip the column
// range is also split over workgroups, which leave float32 partial tiles for a second kernel.
// Because gate and up of an output meet in that sum, act(gate) * up costs no pass of its own.
#pragma once
#include <atomic>
#include <type_traits>
#include "cbk_octet.h"

namespace cbk {

constexpr int SK_WC = 4, SK_WR = 2;            // column parts and row groups of a workgroup
constexpr int SK_ROWS = 64;                    // weight rows per wavefront
constexpr int SK_PITCH = 72;                   // floats per token row of a wavefront's tile in LDS: lanes l and l + 32 write
                                               // four token rows apart, 288 floats = 32 banks
constexpr int SK_LUT_LANES = 16;               // lane-private copies of the selector table (16 lanes read 256 bytes at a time)
constexpr int SK_LUT = 256 * SK_LUT_LANES * 16;
constexpr size_t SK_LDS = (size_t)SK_WC * SK_WR * 32 * SK_PITCH * 4 + SK_LUT;

typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));

// A wavefront's view of global memory: base in scalar registers, loads at lane offset + scalar offset (32 bits each).
__device__ inline __amdgpu_buffer_rsrc_t sk_buffer(const void* base) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, -1, 0x00027000);
}
template <typename T>
__device__ inline T sk_load(__amdgpu_buffer_rsrc_t b, uint32_t lane_off, uint32_t off) {
  if constexpr (sizeof(T) == 16) return __builtin_amdgcn_raw_buffer_load_b128(b, lane_off, off, 0);
  else if constexpr (sizeof(T) == 8) return __builtin_amdgcn_raw_buffer_load_b64(b, lane_off, off, 0);
  else if constexpr (sizeof(T) == 4) return __builtin_amdgcn_raw_buffer_load_b32(b, lane_off, off, 0);
  else if constexpr (sizeof(T) == 2) return __builtin_amdgcn_raw_buffer_load_b16(b, lane_off, off, 0);
  else return __builtin_amdgcn_raw_buffer_load_b8(b, lane_off, off, 0);
}

// The scale of a token and column part with an infinite activation: above every scale of a finite one (2^120)
constexpr float SK_INFINITE = 2658455991569831745807614120560689152.f;   // 2^121

struct SkArgs {
  DMat m;
  const uint16_t* xp;      // fragments of X' [vector][token tile][group][steps][TI][64][8]
  const uint32_t* xc;      // sums of X' over the halves of a group, two halfs each [vector][token tile][group][2][32 TI]
  size_t xcs;              // their distance between two vectors
  const float* row_scale;  // [vector][part of the column range][rss]
  int rss, rvs;            // floats between two parts / two vectors
  size_t xps;              // halfs between the fragments of two col_scale vectors
  int M;
  void* y;
  int ydt;
  int64_t ldy;
  const void* bias;
  int tiles_t, tiles_r, nsplit;
  int par;                 // gate/up matrix: row group w of a workgroup takes the rows of parity w, with vector w
  int act;                 // par only: -1, or the activation of act(gate) * up (y is [M, K / 2])
  int vs0, vs1;            // q|k|v matrix: rows from vs0 / vs1 on use vector 1 / 2 (multiples of 64)
  float* part;             // nsplit > 1: partial tiles [nsplit][M][part_ld] instead of y
  size_t part_stride;
  int64_t part_ld;
};

__device__ inline float sk_act(int act, float g) {
  if (act == CBK_ACT_SILU) return g / (1.f + __expf(-g));
  const float k = 0.7978845608028654f;                              // sqrt(2 / pi)
  return 0.5f * g * (1.f + tanhf(k * (g + 0.044715f * g * g * g)));
}

// four consecutive outputs
__device__ inline void sk_store4(void* y, int ydt, size_t at, const float (&v)[4], int n, bool vec) {
  if (ydt == CBK_F32) {
    if (vec && n == 4) *(float4*)((float*)y + at) = make_float4(v[0], v[1], v[2], v[3]);
    else for (int e = 0; e < 4; ++e) { if (e < n) ((float*)y)[at + e] = v[e]; }
    return;
  }
  uint16_t h[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) h[e] = ydt == CBK_F16 ? f2h(v[e]) : f2bf(v[e]);
  if (vec && n == 4) *(uint2*)((uint16_t*)y + at) = make_uint2((uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16));
  else for (int e = 0; e < 4; ++e) { if (e < n) ((uint16_t*)y)[at + e] = h[e]; }
}

// What a lane reads of a row per group: half a group's columns, PBLK 32-column blocks.
constexpr int sk_gcd(int a, int b) { return b ? sk_gcd(b, a % b) : a; }
template <int BITS, int KEEP, int GRP, int TI>
struct SkCfg {
  static constexpr bool DENSE = KEEP == 0, HI2 = BITS == 6, B8 = BITS == 8;
  static constexpr int PB = HI2 ? 4 : BITS;                         // bits per code in the stream
  static constexpr int CB = (DENSE ? 32 : KEEP) * PB;               // code bits of a block
  static constexpr int PBLK = GRP / 64, ST = GRP / 16;              // blocks per lane and steps per group
  static constexpr int HB = PBLK * CB;                              // code bits of a lane's run
  static constexpr int ND = (HB + 31) / 32;
  static constexpr bool WHOLE = HB == 32 || HB == 64 || HB % 128 == 0;   // the run starts on a dword / 8 / 16 bytes of its own
  static constexpr int UNITS = (128 - sk_gcd(HB, 128) + HB + 127) / 128; // else: 16-byte units that hold it at any skew
  static constexpr int NL = WHOLE ? ND : 4 * UNITS;
  static constexpr int SB = BITS == 3 ? 4 : PB;                     // stream code width after expansion
  static constexpr int NW = ((DENSE ? 32 : KEEP) * SB + 31) / 32;   // dwords of a block's stream
  static constexpr int NG = GRP == 64 ? 3 : 2;                      // groups in flight
  static constexpr int RG = (DENSE ? 0 : PBLK) + NL + (HI2 ? PBLK : 0) + 2;   // registers of a group and row
  // scale and zero point per group instead of per weight: where the registers hold a second set of sums
  // (without spilling: read off the compiler's report)
  static constexpr bool DEFER = TI == 1 || (TI == 2 && 2 * NG * RG <= (DENSE ? 40 : GRP == 128 ? 32 : 24));
  static constexpr int NA = TI == 1 || (TI == 2 && !DEFER) ? 8 : 4; // activation fragments in flight (steps)
  // A code c becomes the half BASE + c, exactly, from one byte: the low byte of 0x6400 + c (8- and 6-bit codes), of
  // 0x5400 + (c << 4) (nibbles, kept in the high half of their byte), or the high byte of 0x4400 + (c << 8) (2-bit)
  static constexpr int BASE = B8 || HI2 ? 1024 : BITS == 2 ? 4 : 64;
  // order of the columns of an octet in a fragment: the order the codes come out of the stream
  static constexpr int ORDER = !DENSE || B8 ? 0 : BITS == 2 ? 2 : 1;
};

// BITS 2 / 3 / 4 / 6 with KEEP survivors per 32 columns, or KEEP = 0 for dense 2 / 3 / 4 / 8-bit codes; any zero
// point.  TI: 32-token blocks of the tile.
template <int BITS, int KEEP, int GRP, int TI>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_skinny_kernel(SkArgs a) {
  // All 256 registers of a wavefront (there is one workgroup per CU either way), so that the shift amounts of
  // window() are not in the last one: with 224 given and an amount in v223, the 64-token tile of 6-bit codes returned
  // sums off by 1e-2 that changed from run to run (build.py, shift_hazards, which looks at every kernel built).
  asm volatile("" ::: "v255");
  using C = SkCfg<BITS, KEEP, GRP, TI>;
  constexpr bool BITMAP = !C::DENSE;
  constexpr bool DEFER = C::DEFER;
  constexpr int ST = C::ST, NG = C::NG, NA = C::NA;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  // [256][copies]: selectors, byte masks.  First: an entry's address is its offset, so this kernel and what it inlines have
  // no static __shared__ (the build refuses one)
  uint4* lut = (uint4*)smem;
  float* red = (float*)(smem + SK_LUT);
  const DMat& m = a.m;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wave & 1, wc = wave >> 1, half = lane >> 5;
  // XCD-aware order: workgroups of one XCD (blockIdx % 8) take neighbouring tiles: the parts and token tiles of a
  // row range read the same weights
  const int nb = a.tiles_t * a.tiles_r * a.nsplit, per = (nb + 7) >> 3;
  const int lin = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || lin >= nb) return;
  const int tt = lin % a.tiles_t, rest = lin / a.tiles_t, sp = rest % a.nsplit, tr = rest / a.nsplit;
  const int kstep = a.par ? 2 : 1;
  const int r0 = tr * (SK_ROWS * SK_WR) + (a.par ? wr : SK_ROWS * wr);       // first row of this wavefront
  // its groups: the row's cut into nsplit * SK_WC parts
  const int q = sp * SK_WC + wc, nq = a.nsplit * SK_WC;
  const int g0 = m.G * q / nq, g1 = m.G * (q + 1) / nq;
  const int xv = a.par ? wr : (r0 >= a.vs0 ? 1 : 0) + (r0 >= a.vs1 ? 1 : 0);

  v16f tot[TI][2];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) tot[i][j][e] = 0.f;

  // Selector table, built while the first loads are in flight
  auto build_table = [&]() {
    if (BITMAP) {
      if (tid < 256) {
        const uint2 e = make_selectors((uint32_t)tid, BITS == 2 ? 1 : 0);
        // 6-bit: all ones in the pruned bytes; else the field of a code in the kept ones
        constexpr uint32_t F = C::HI2 ? 0xFFu : C::SB == 4 ? 0xF0u : 0x03u;
        const uint32_t k0 = bits_to_bytes((uint32_t)tid) * F, k1 = bits_to_bytes((uint32_t)tid >> 4) * F;
#pragma unroll
        for (int j = 0; j < SK_LUT_LANES; ++j) lut[table_slot<SK_LUT_LANES, 16>(tid, j)] = make_uint4(e.x, e.y, C::HI2 ? ~k0 : k0, C::HI2 ? ~k1 : k1);
      }
      // (a barrier over LDS only: __syncthreads() would wait for the loads in flight)
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    }
  };

  if (g0 >= g1) build_table();
  if (g0 < g1) {
    // Addresses: a scalar base that moves with the group plus a 32-bit offset per lane that does not.  The base row
    // is inside the matrix even where the wavefront's rows are not (those are decoded and never stored).
    const int rb = r0 < m.K ? r0 : m.K - 1;
    const uint32_t ush = m.tiled ? 256u : 16u;                      // bytes between the 16-byte units of a row
    const uint8_t* dbase = m.data + (m.tiled ? (size_t)(rb >> 4) * m.stride * 16 : (size_t)rb * m.stride);
    const size_t mbase = m.tiled ? (size_t)(rb >> 4) * m.G * 16 : (size_t)rb * m.G;
    uint32_t roff[2], moff[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int r = r0 + kstep * (32 * j + (lane & 31)), rc = r < m.K ? r : m.K - 1;
      roff[j] = m.tiled ? (uint32_t)((rc >> 4) - (rb >> 4)) * m.stride * 16u + (uint32_t)(rc & 15) * 16u : (uint32_t)(rc - rb) * m.stride;
      moff[j] = m.tiled ? (uint32_t)((rc >> 4) - (rb >> 4)) * (uint32_t)m.G * 16u + (uint32_t)(rc & 15) : (uint32_t)(rc - rb) * (uint32_t)m.G;
    }
    const uint32_t lut_lane = (uint32_t)(lane & (SK_LUT_LANES - 1)) * 16u;
    // Read as buffers: a scalar offset that moves with the group and a lane's that does not cost no vector instruction
    // (as pointers, every group's base and every step's went through a 64-bit vector addition)
    const auto data_b = sk_buffer(dbase), zero_b = sk_buffer(m.zero + mbase), scale_b = sk_buffer(m.scale + mbase);
    struct Grp {
      uint32_t m[BITMAP ? C::PBLK : 1];
      uint32_t raw[C::NL];
      uint32_t h2[C::HI2 ? C::PBLK : 1];
      uint32_t z, s;
    };
    auto load_group = [&](int g, Grp (&w)[2]) {
      g = g < g1 ? g : g1 - 1;
      const uint32_t ug = (uint32_t)g;
      // mask words (and, for one-dword runs, codes): 8 PBLK bytes per group and row, the upper half's behind the lower's
      const uint32_t go8 = C::PBLK == 2 ? ug * ush : (ug >> 1) * ush + (ug & 1u) * 8u, lo8 = (uint32_t)half * (C::PBLK * 4u);
      // first unit of a skewed run
      const uint32_t uskew = ((2u * ug + (uint32_t)half) * (uint32_t)C::HB >> 7) * ush;
      const uint32_t plane = (m.code_off >> 4) * ush;               // (the mask plane is whole units)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        if (BITMAP) {
          if (C::PBLK == 2) { const v2u v = sk_load<v2u>(data_b, roff[j] + lo8, go8); w[j].m[0] = v[0]; w[j].m[C::PBLK - 1] = v[1]; }
          else w[j].m[0] = sk_load<uint32_t>(data_b, roff[j] + lo8, go8);
        }
        if (C::HI2) {                                               // behind the mask and nibble planes
          const v2u v = sk_load<v2u>(data_b, roff[j] + (uint32_t)half * 8u, (uint32_t)(m.N * 3 >> 7) * ush + ug * ush);
          w[j].h2[0] = v[0]; w[j].h2[C::HI2 ? C::PBLK - 1 : 0] = v[1];
        }
        if constexpr (C::HB == 32) w[j].raw[0] = sk_load<uint32_t>(data_b, roff[j] + lo8, plane + go8);
        else if constexpr (C::HB == 64) {
          const v2u v = sk_load<v2u>(data_b, roff[j] + (uint32_t)half * 8u, plane + ug * ush);
          w[j].raw[0] = v[0]; w[j].raw[1] = v[1];
        } else {
#pragma unroll
          for (int i = 0; i < C::NL / 4; ++i) {
            const v4u v = C::WHOLE ? sk_load<v4u>(data_b, roff[j] + (uint32_t)half * (C::HB / 128) * ush, plane + (ug * (2 * C::HB / 128) + i) * ush)
                                   : sk_load<v4u>(data_b, roff[j] + uskew, plane + i * ush);
            w[j].raw[4 * i] = v[0]; w[j].raw[4 * i + 1] = v[1]; w[j].raw[4 * i + 2] = v[2]; w[j].raw[4 * i + 3] = v[3];
          }
        }
        const uint32_t mg = m.tiled ? ug * 16u : ug;
        w[j].z = sk_load<uint8_t>(zero_b, moff[j], mg);
        w[j].s = sk_load<uint16_t>(scale_b, moff[j] * 2u, mg * 2u);
      }
    };
    // activation fragments of step t and group sums of group g (counted from the wavefront's first)
    const uint8_t* xb = (const uint8_t*)(a.xp + (size_t)xv * a.xps) + ((size_t)tt * m.G + g0) * (ST * TI * 1024);
    const uint32_t* xcb = a.xc + (size_t)xv * a.xcs + ((size_t)tt * m.G + g0) * (2 * TI * 32);
    v8h af[NA][TI];
    uint32_t xs[TI];
    const uint32_t lane16 = (uint32_t)lane * 16u;
    const auto act_b = sk_buffer(xb);
    const int steps = (g1 - g0) * ST;
    auto load_a = [&](int t, int buf) {
      const uint32_t at = (uint32_t)(t < steps ? t : steps - 1) * (TI * 1024u);
#pragma unroll
      for (int i = 0; i < TI; ++i) af[buf][i] = __builtin_bit_cast(v8h, sk_load<v4u>(act_b, lane16, at + i * 1024u));
    };
    auto load_sums = [&](int g) {
      const uint32_t* p = xcb + (size_t)((uint32_t)(g < g1 - g0 ? g : g1 - g0 - 1) * (2u * TI * 32u));
#pragma unroll
      for (int i = 0; i < TI; ++i)
        if (DEFER) xs[i] = p[(uint32_t)(lane & 31) + (uint32_t)half * (TI * 32u) + i * 32u];
    };
    // Does this part of a token of the tile hold an infinity (see SK_INFINITE)?
    const int rtok = tt * (32 * TI) + (TI == 1 ? lane & 31 : lane);
    float rs = 0.f;
    if (DEFER) rs = a.row_scale[(size_t)xv * a.rvs + (size_t)q * a.rss + rtok];
    Grp ring[NG][2];
    load_sums(0);
#pragma unroll
    for (int u = 0; u < NG; ++u) load_group(g0 + u, ring[u]);
#pragma unroll
    for (int t = 0; t < NA - 1; ++t) load_a(t, t);

    // T0: position of the group's first step in the ring of activation fragments.  SUB: the zero point is taken off
    // every weight instead of off the sum.
    auto group = [&](int g, Grp (&w)[2], auto t0_tag, auto more_tag, auto sub_tag) {
      constexpr int T0 = decltype(t0_tag)::value;
      constexpr bool more = decltype(more_tag)::value, SUB = decltype(sub_tag)::value;
      uint32_t cw[2][C::ND], st[2][C::NW], z4[2];
      h2_t off[2], sh[2];                                           // -(BASE + zero), and the scale for !DEFER
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        if constexpr (C::WHOLE) {
#pragma unroll
          for (int i = 0; i < C::ND; ++i) cw[j][i] = w[j].raw[i];
        } else {
          skew_dwords<C::NL, C::ND, C::HB % 32 == 0>(w[j].raw, ((2u * (uint32_t)g + (uint32_t)half) * (uint32_t)C::HB) & 127u, cw[j]);
        }
        // the zero point in every byte, where a code has its bits
        z4[j] = perm(0, C::BASE == 64 ? w[j].z << 4 : C::BASE == 4 ? w[j].z | 0x44u : w[j].z, 0);
        const _Float16 n = (_Float16)(-(float)C::BASE - (float)w[j].z), f = __builtin_bit_cast(_Float16, (uint16_t)w[j].s);
        off[j] = h2_t{n, n}; sh[j] = h2_t{f, f};
      }
      uint4 sel[2][2];
      auto rank = [](uint32_t mw, int jj) { return (uint32_t)__builtin_popcount(mw & ((1u << (8 * jj)) - 1u)); };
      auto fetch = [&](int o, uint4 (&e)[2]) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
          if (BITMAP) {                                             // entry address: mask byte in byte 1, this lane's copy in byte 0
            const v4u v = *(const __attribute__((address_space(3))) v4u*)(uintptr_t)perm(w[j].m[BITMAP ? o >> 2 : 0], lut_lane, 0x0C0C0400u + ((uint32_t)(o & 3) << 8));
            e[j] = make_uint4(v[0], v[1], v[2], v[3]);
          }
      };
      // octet o of both rows -> the B operands of a step
      auto decode = [&](int o, const uint4 (&e)[2], v8h (&bf)[2]) {
        const int blk = o >> 2, jj = o & 3;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const uint32_t kb = C::BASE == 1024 ? 0x64646464u : 0x54545454u;
          // four bytes -> four halves
          auto widen = [&](uint32_t b, uint32_t& lo, uint32_t& hi) {
            if constexpr (C::BASE == 4) { lo = perm(0, b, 0x010C000Cu); hi = perm(0, b, 0x030C020Cu); }
            else { lo = perm(kb, b, 0x04010400u); hi = perm(kb, b, 0x04030402u); }
          };
          uint32_t h[4];
          if constexpr (C::B8) {
            const uint32_t b0 = cw[j][2 * o], b1 = cw[j][2 * o + 1];
            widen(b0, h[0], h[1]); widen(b1, h[2], h[3]);
          } else {
            if (jj == 0) {
#pragma unroll
              for (int k = 0; k < C::NW; ++k)
                st[j][k] = BITS == 3 ? expand3to4(get32<C::ND>(cw[j], blk * C::CB + 24 * k)) : get32<C::ND>(cw[j], blk * C::CB + 32 * k);
            }
            uint32_t win = BITMAP ? (jj == 0 ? st[j][0] : window<C::NW>(st[j], rank(w[j].m[BITMAP ? blk : 0], jj) * C::SB))
                                  : C::SB == 4 ? st[j][jj] : (st[j][jj >> 1] >> (16 * (jj & 1)));
            if (C::SB == 2) { win &= 0xFFFFu; win |= win << 14; }   // bytes c0 c4 c1 c5; four bits up c2 c6 c3 c7
            if (BITMAP) {
              // even and odd codes in the bits they have in a byte, the neighbour's bits beside them
              uint32_t q0 = C::BASE == 64 ? win << 4 : win, q1 = C::BASE == 64 ? win : win >> 4, b0, b1;
              if (C::HI2) {
                uint32_t h0, h1;
                hi2_pools(w[j].h2[C::HI2 ? blk : 0], jj == 0 ? 0u : rank(w[j].m[BITMAP ? blk : 0], jj), h0, h1);
                b0 = perm((q1 & 0x0F0F0F0Fu) | h1, (q0 & 0x0F0F0F0Fu) | h0, e[j].x) | (e[j].z & z4[j]);
                b1 = perm((q1 & 0x0F0F0F0Fu) | h1, (q0 & 0x0F0F0F0Fu) | h0, e[j].y) | (e[j].w & z4[j]);
              } else {                                              // a kept column's field, the zero point elsewhere (it has no bits there
                b0 = mask_select(e[j].z, z4[j], perm(q1, q0, e[j].x));   // in a kept column: it is a code itself)
                b1 = mask_select(e[j].w, z4[j], perm(q1, q0, e[j].y));
              }
              widen(b0, h[0], h[1]); widen(b1, h[2], h[3]);
            } else {                                                // columns in stream order (SkCfg::ORDER)
              const uint32_t q0 = C::BASE == 64 ? (win << 4) & 0xF0F0F0F0u : (win & 0x03030303u) | 0x44444444u;
              const uint32_t q1 = C::BASE == 64 ? win & 0xF0F0F0F0u : ((win >> 4) & 0x03030303u) | 0x44444444u;
              widen(q0, h[0], h[1]); widen(q1, h[2], h[3]);
            }
          }
          if constexpr (!DEFER || SUB) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              h2_t v = __builtin_bit_cast(h2_t, h[i]) + off[j];
              if constexpr (!DEFER) v = v * sh[j];
              h[i] = __builtin_bit_cast(uint32_t, v);
            }
          }
          const uint4 hv = make_uint4(h[0], h[1], h[2], h[3]);
          bf[j] = __builtin_bit_cast(v8h, hv);
        }
      };
      v8h bf[2][2];
      fetch(0, sel[0]);
      if (ST > 1) fetch(1, sel[1]);
      // -(BASE + zero) against the sum of this lane's half of the group (as two halfs)
      v16f part[DEFER ? TI : 1][2];
      if constexpr (DEFER) {
        v8h bz[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const uint32_t nn = perm(0, (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)off[j][0]), 0x01000100u);
          bz[j] = __builtin_bit_cast(v8h, make_uint4(nn, 0, 0, 0));
        }
#pragma unroll
        for (int i = 0; i < TI; ++i) {
          const v8h az = __builtin_bit_cast(v8h, make_uint4(xs[i], 0, 0, 0));
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            v16f zero16;
#pragma unroll
            for (int e = 0; e < 16; ++e) zero16[e] = 0.f;
            if constexpr (SUB) part[i][j] = zero16;
            else part[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(az, bz[j], zero16, 0, 0, 0);
          }
        }
        if constexpr (!SUB) load_sums(g - g0 + 1);
      }
      decode(0, sel[0], bf[0]);
      __builtin_amdgcn_sched_barrier(0);
      // Step o multiplies octet o while octet o + 1 is decoded and the selectors of octet o + 2 are fetched
      const int t0 = (g - g0) * ST;
#pragma unroll
      for (int o = 0; o < ST; ++o) {
        load_a(t0 + o + NA - 1, (T0 + o + NA - 1) % NA);
        if (o + 2 < ST) fetch(o + 2, sel[o & 1]);
        if (o + 1 < ST) decode(o + 1, sel[(o + 1) & 1], bf[(o + 1) & 1]);
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            v16f& d = DEFER ? part[DEFER ? i : 0][j] : tot[i][j];
            d = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[(T0 + o) % NA][i], bf[o & 1][j], d, 0, 0, 0);
          }
#pragma unroll
        for (int k = 0; k < 2 * TI; ++k) {                          // a matrix instruction, then a slice of the decode
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, DEFER ? 18 / TI : 8, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      float sc[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        sc[j] = h2f((uint16_t)w[j].s);
        asm("" : "+v"(sc[j]));                                      // (or the conversion is folded into v_fma_mix_f32, see below)
      }
      if (more) load_group(g + NG, w);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (DEFER) {
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) tot[i][j][e] = fmaf(part[i][j][e], sc[j], tot[i][j][e]);
      }
    };
    build_table();
    // No branch between the groups of a trip: where paths join, the compiler waits for every load in
    // flight.  A trip is UG groups: whole turns of both rings.
    constexpr int UG = NG == 3 && ST % NA ? 6 : NG;
    static_assert(UG % NG == 0 && UG * ST % NA == 0, "both rings turn a whole number of times per trip");
    using Yes = std::true_type; using No = std::false_type;
    int g = g0;
    if constexpr (DEFER) {
      // An infinity: its code times X' and the sum of the group are infinite too, and their difference is NaN where the
      // weight times it is not.  Such a wavefront takes its groups one at a time with the zero point off every weight.
      if (__builtin_expect(__ballot(rs == SK_INFINITE && rtok < a.M) != 0, 0)) {
        for (int h = g0; h < g1; ++h) {
          load_group(h, ring[0]);
#pragma unroll
          for (int t = 0; t < NA - 1; ++t) load_a((h - g0) * ST + t, t);
          group(h, ring[0], std::integral_constant<int, 0>{}, No{}, Yes{});
        }
        g = g1;
      }
    }
    for (; g + UG <= g1; g += UG) {
      group(g, ring[0], std::integral_constant<int, 0>{}, Yes{}, No{});
      group(g + 1, ring[1 % NG], std::integral_constant<int, ST % NA>{}, Yes{}, No{});
      if constexpr (UG > 2) group(g + 2, ring[2 % NG], std::integral_constant<int, 2 * ST % NA>{}, Yes{}, No{});
      if constexpr (UG > 3) {
        group(g + 3, ring[3 % NG], std::integral_constant<int, 3 * ST % NA>{}, Yes{}, No{});
        group(g + 4, ring[4 % NG], std::integral_constant<int, 4 * ST % NA>{}, Yes{}, No{});
        group(g + 5, ring[5 % NG], std::integral_constant<int, 5 * ST % NA>{}, Yes{}, No{});
      }
    }
    if (g < g1) group(g, ring[0], std::integral_constant<int, 0>{}, Yes{}, No{});
    if constexpr (UG > 2) {
      if (g + 1 < g1) group(g + 1, ring[1 % NG], std::integral_constant<int, ST % NA>{}, Yes{}, No{});
    }
    if constexpr (UG > 3) {
      if (g + 2 < g1) group(g + 2, ring[2 % NG], std::integral_constant<int, 2 * ST % NA>{}, Yes{}, No{});
      if (g + 3 < g1) group(g + 3, ring[3 % NG], std::integral_constant<int, 3 * ST % NA>{}, Yes{}, No{});
      if (g + 4 < g1) group(g + 4, ring[4 % NG], std::integral_constant<int, 4 * ST % NA>{}, No{}, No{});
    }
  }

  // ---- the four column parts through LDS, 32 tokens at a time.  D[r] of lane l: token 8 (r / 4) + 4 (l / 32) +
  // r % 4 of the block, weight row l % 32 of the 32.  Then a thread owns four rows of both row groups of one token.
  const int tok0 = tt * 32 * TI;
  const int et = tid >> 4, eq = (tid & 15) * 4;
  const size_t esz = a.ydt == CBK_F32 ? 4 : 2;
  const int rg0 = tr * (SK_ROWS * SK_WR), rg1 = rg0 + SK_ROWS;
  const int xg[2] = {a.par ? 0 : (rg0 >= a.vs0 ? 1 : 0) + (rg0 >= a.vs1 ? 1 : 0),       // vectors of the two row groups
                     a.par ? 1 : (rg1 >= a.vs0 ? 1 : 0) + (rg1 >= a.vs1 ? 1 : 0)};
#pragma unroll
  for (int i = 0; i < TI; ++i) {
    __syncthreads();                                                // the tile of the block before has been read
    float* mine = red + (size_t)(wc * SK_WR + wr) * 32 * SK_PITCH;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        mine[(8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)) * SK_PITCH + 32 * j + (lane & 31)] = tot[i][j][r];
    __syncthreads();
    const int tok = tok0 + 32 * i + et;
    if (tok >= a.M) continue;                                       // (no barrier is skipped: the next one is reached by all)
    float v[2][4];
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const float* s = a.row_scale + (size_t)xg[g] * a.rvs + (size_t)sp * SK_WC * a.rss + tok;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[g][e] = 0.f;
#pragma unroll
      for (int c = 0; c < SK_WC; ++c) {
        const float4 f = *(const float4*)(red + (size_t)(c * SK_WR + g) * 32 * SK_PITCH + et * SK_PITCH + eq);
        const float k = s[(size_t)c * a.rss];
        v[g][0] = fmaf(f.x, k, v[g][0]); v[g][1] = fmaf(f.y, k, v[g][1]);
        v[g][2] = fmaf(f.z, k, v[g][2]); v[g][3] = fmaf(f.w, k, v[g][3]);
      }
    }
    const bool part = a.nsplit > 1;
    void* y = part ? (void*)(a.part + (size_t)sp * a.part_stride) : a.y;
    const int ydt = part ? (int)CBK_F32 : a.ydt;
    const int64_t ld = part ? a.part_ld : a.ldy;
    const size_t es = part ? 4 : esz;
    if (!part && a.bias) {
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int k = a.par ? rg0 + 2 * (eq + e) + g : rg0 + SK_ROWS * g + eq + e;
          if (k < m.K) v[g][e] += a.ydt == CBK_F32 ? ((const float*)a.bias)[k] : a.ydt == CBK_F16 ? h2f(((const uint16_t*)a.bias)[k]) : bf2f(((const uint16_t*)a.bias)[k]);
        }
    }
    const bool vec = ((((uintptr_t)y) | (uintptr_t)(ld * (int64_t)es)) & (4 * es - 1)) == 0;
    if (!a.par) {
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const int k = rg0 + SK_ROWS * g + eq;
        sk_store4(y, ydt, (size_t)tok * ld + k, v[g], m.K - k, vec);
      }
    } else if (a.act >= 0 && !part) {
      float o[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = sk_act(a.act, v[0][e]) * v[1][e];
      const int k = (rg0 >> 1) + eq;
      sk_store4(y, ydt, (size_t)tok * ld + k, o, (m.K >> 1) - k, vec);
    } else {
      const int k = rg0 + 2 * eq;
      const float lo[4] = {v[0][0], v[1][0], v[0][1], v[1][1]}, hi[4] = {v[0][2], v[1][2], v[0][3], v[1][3]};
      sk_store4(y, ydt, (size_t)tok * ld + k, lo, m.K - k, vec);
      sk_store4(y, ydt, (size_t)tok * ld + k + 4, hi, m.K - k - 4, vec);
    }
  }
}

template <int BITS, int KEEP, int GRP, int TI>
static int launch_skinny_ti(const SkArgs& a, int blocks, hipStream_t st) {
  auto kern = gemm_skinny_kernel<BITS, KEEP, GRP, TI>;
  static std::atomic<int> configured{0};
  if (!configured.load(std::memory_order_acquire)) {
    if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024) != hipSuccess)
      return CBK_ERR_HIP;
    configured.store(1, std::memory_order_release);
  }
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(512), SK_LDS, st, a);
  return hipGetLastError() == hipSuccess ? CBK_OK : CBK_ERR_HIP;
}
template <int BITS, int KEEP, int GRP>
static int launch_skinny_cfg(const SkArgs& a, int ti, int blocks, hipStream_t st) {
  return ti == 1 ? launch_skinny_ti<BITS, KEEP, GRP, 1>(a, blocks, st)
       : ti == 2 ? launch_skinny_ti<BITS, KEEP, GRP, 2>(a, blocks, st)
       : ti == 3 ? launch_skinny_ti<BITS, KEEP, GRP, 3>(a, blocks, st) : CBK_ERR_UNSUPPORTED;
}
template <int BITS>
static int launch_skinny_bits(const SkArgs& a, int keep, int group, int ti, int blocks, hipStream_t st) {
#define CBK_SK_CASE(KEEP)                                                             \
  case KEEP: return group == 64 ? launch_skinny_cfg<BITS, KEEP, 64>(a, ti, blocks, st) \
                                : launch_skinny_cfg<BITS, KEEP, 128>(a, ti, blocks, st);
  switch (keep) {
    CBK_SK_CASE(0) CBK_SK_CASE(10) CBK_SK_CASE(16) CBK_SK_CASE(23)
    default: return CBK_ERR_UNSUPPORTED;
  }
#undef CBK_SK_CASE
}

}  // namespace cbk
