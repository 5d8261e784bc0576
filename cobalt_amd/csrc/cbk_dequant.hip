// Packed bytes -> dense W_hat, bit-exact float32 evaluation of
//   ((q - zero) * scale) * keep * col_scale
// in that order (reference: src/cobaltkernel/dequant_ref.py:69-82), then one RN-even cast.
//
// Bound: the write of the dense matrix.  A thread owns eight columns (16 bytes of 16-bit output) of
// sixteen consecutive rows: the stores of a wavefront are 1 KB runs, the column scales stay in
// registers over the rows, and in the tiled byte order the sixteen rows share the cache lines of
// their units.  One thread per 32-column block with single-element stores, the form before, was
// bound by those stores: 14336 x 4096 to fp16 300 us, now 28 us (5.1 TB/s).
#include "cbk_octet.h"

namespace cbk {

constexpr int DQ_ROWS = 16;                                         // rows per thread

template <int ODT>
__device__ inline void store8(void* out, size_t at, const float (&w)[8], bool vec) {
  constexpr int ESZ = ODT == CBK_F32 ? 4 : 2;
  if (!vec) {
#pragma unroll
    for (int i = 0; i < 8; ++i) store_out<ODT>(out, at + i, w[i]);
    return;
  }
  // Non-temporal: the output is larger than what the caches keep, and left to them its lines push
  // out each other (two outputs of 117 MB in turn: 43 us a pass, 28 us past the caches).
  typedef uint32_t u4 __attribute__((ext_vector_type(4)));
  u4* d = (u4*)((uint8_t*)out + at * ESZ);
  if (ODT == CBK_F32) {
    const u4 a = {__float_as_uint(w[0]), __float_as_uint(w[1]), __float_as_uint(w[2]), __float_as_uint(w[3])};
    const u4 b = {__float_as_uint(w[4]), __float_as_uint(w[5]), __float_as_uint(w[6]), __float_as_uint(w[7])};
    __builtin_nontemporal_store(a, d);
    __builtin_nontemporal_store(b, d + 1);
  } else {
    uint32_t p[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (ODT == CBK_F16) p[i] = (uint32_t)f2h(w[2 * i]) | ((uint32_t)f2h(w[2 * i + 1]) << 16);
      else {
        typedef __bf16 b2 __attribute__((ext_vector_type(2)));
        const b2 v = {(__bf16)w[2 * i], (__bf16)w[2 * i + 1]};      // round to nearest even
        p[i] = __builtin_bit_cast(uint32_t, v);
      }
    }
    const u4 v = {p[0], p[1], p[2], p[3]};
    __builtin_nontemporal_store(v, d);
  }
}

// ((q - z) * s) * keep * cs of an octet.  MASKED: a pruned column is multiplied by 0 (it keeps the
// sign of (0 - z) * s, as the reference's product does).
template <bool MASKED>
__device__ inline void octet_values(const Octet& o, float z, float s, const float (&cs)[8], float (&w)[8]) {
  const uint32_t k0 = bits_to_bytes(o.keep), k1 = bits_to_bytes(o.keep >> 4);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const uint32_t q = ((i < 4 ? o.lo : o.hi) >> (8 * (i & 3))) & 0xFFu;
    float v = __fmul_rn(__fsub_rn((float)q, z), s);
    if (MASKED) v = __fmul_rn(v, (float)(((i < 4 ? k0 : k1) >> (8 * (i & 3))) & 0xFFu));
    w[i] = __fmul_rn(v, cs[i]);
    asm("" : "+v"(w[i]));                                           // a float32 before the cast: one mixed-precision multiply-and-
  }                                                                 // convert instruction in its place would round once instead of twice
}

__device__ inline void load_cs8(const uint16_t* cs, uint32_t j8, float (&c)[8]) {
  const uint4 v = cs ? *(const uint4*)(cs + 8 * (size_t)j8) : make_uint4(0x3c003c00u, 0x3c003c00u, 0x3c003c00u, 0x3c003c00u);
  const uint32_t u[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) { c[2 * i] = h2f((uint16_t)(u[i] & 0xffffu)); c[2 * i + 1] = h2f((uint16_t)(u[i] >> 16)); }
}

// ONE_CS: at most one column-scale vector (none multiplies by 1, which changes nothing)
template <int FAM, int BITS, int ODT, bool ONE_CS>
__global__ __launch_bounds__(256) void dequant_fixed_kernel(DMat m, int row0, int nrows, int with_cs, void* out,
                                                            int64_t ld, int vec) {
  __shared__ uint2 lut[256 * OCT_LUT_LANES];
  if (FAM != FAM_DENSE) { octet_table(lut); __syncthreads(); }
  const uint32_t n8 = (uint32_t)m.N >> 3;
  const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int rb = (int)(id / n8);
  const uint32_t j8 = (uint32_t)(id % n8);
  const int r_begin = rb * DQ_ROWS;
  if (r_begin >= nrows) return;
  const int r_end = nrows - r_begin < DQ_ROWS ? nrows : r_begin + DQ_ROWS;
  const int g = (int)(j8 * 8) / m.group;
  const uint16_t* csv = with_cs ? m.cs : nullptr;
  float cs[8];
  load_cs8(csv, j8, cs);
  constexpr int U = 4;                                              // rows whose loads are in flight together
  for (int r = r_begin; r < r_end; r += U) {
    Octet o[U];
    float z[U], sc[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = row0 + (r + u < r_end ? r + u : r_end - 1);
      o[u] = octet_fixed<FAM, BITS>(m, row_view(m, k), j8, lut);
      const size_t mi = meta_index(m, k, g);
      z[u] = (float)m.zero[mi];
      sc[u] = h2f(m.scale[mi]);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (r + u >= r_end) break;
      if (!ONE_CS && csv) load_cs8(csv + (size_t)cs_row_of(m, row0 + r + u) * m.N, j8, cs);
      float w[8];
      octet_values<FAM != FAM_DENSE>(o[u], z[u], sc[u], cs, w);
      store8<ODT>(out, (size_t)(r + u) * ld + 8 * (size_t)j8, w, vec);
    }
  }
}

// Survivor streams: a workgroup takes ST_DQ_ROWS rows one after the other (the group offsets of a
// SPARSE4 row are summed once per row).
constexpr int ST_DQ_ROWS = 4;
template <int ODT>
__global__ __launch_bounds__(256) void dequant_sparse_kernel(DMat m, int row0, int nrows, int with_cs, void* out,
                                                             int64_t ld, int vec, int summed) {
  extern __shared__ uint32_t goff[];                                // [G] if summed (SPARSE4)
  __shared__ uint2 lut[256 * OCT_LUT_LANES];
  octet_table(lut);
  const uint32_t hdr = stream_header(m), n8 = (uint32_t)m.N >> 3;
  const int r0 = blockIdx.x * ST_DQ_ROWS, r1 = nrows - r0 < ST_DQ_ROWS ? nrows : r0 + ST_DQ_ROWS;
  for (int r = r0; r < r1; ++r) {
    const int k = row0 + r;
    const uint8_t* row = m.data + m.row_off[k];
    __syncthreads();                                                // the table; the offsets of the row before
    if (summed) {
      if (threadIdx.x < 64) stream_offsets(m, row, goff);
      __syncthreads();
    }
    const uint16_t* csv = with_cs && m.cs ? m.cs + (size_t)cs_row_of(m, k) * m.N : nullptr;
    for (uint32_t j8 = threadIdx.x; j8 < n8; j8 += 256) {
      const Octet o = octet_stream(m, row, hdr, summed ? goff : nullptr, j8, lut);
      const size_t mi = (size_t)k * m.G + (j8 >> 4);
      float cs[8], w[8];
      load_cs8(csv, j8, cs);
      octet_values<false>(o, (float)m.zero[mi], h2f(m.scale[mi]), cs, w);
#pragma unroll
      for (int i = 0; i < 8; ++i) w[i] = (o.keep >> i) & 1u ? w[i] : 0.f;
      store8<ODT>(out, (size_t)r * ld + 8 * (size_t)j8, w, vec);
    }
  }
}

template <int FAM, int BITS>
static void launch_fixed(const DMat& m, int row0, int nrows, int with_cs, void* out, int odt, int64_t ld, int vec,
                         hipStream_t st) {
  const int64_t items = (int64_t)((nrows + DQ_ROWS - 1) / DQ_ROWS) * (m.N / 8);
  const dim3 grid((unsigned)((items + 255) / 256)), blk(256);
  const bool one = !with_cs || m.cs_rows <= 1;
#define CBK_LAUNCH(ODT)                                                                                                   \
  do {                                                                                                                    \
    if (one) hipLaunchKernelGGL((dequant_fixed_kernel<FAM, BITS, ODT, true>), grid, blk, 0, st, m, row0, nrows, with_cs,  \
                                out, ld, vec);                                                                            \
    else hipLaunchKernelGGL((dequant_fixed_kernel<FAM, BITS, ODT, false>), grid, blk, 0, st, m, row0, nrows, with_cs,     \
                            out, ld, vec);                                                                                \
  } while (0)
  if (odt == CBK_F32) CBK_LAUNCH(CBK_F32);
  else if (odt == CBK_F16) CBK_LAUNCH(CBK_F16);
  else CBK_LAUNCH(CBK_BF16T);
#undef CBK_LAUNCH
}

int launch_dequant(const DMat& m, int row0, int nrows, int with_cs, void* out, int odt, int64_t ld,
                   hipStream_t st) {
  if (nrows == 0) return CBK_OK;
  if (odt != CBK_F32 && odt != CBK_F16 && odt != CBK_BF16T) return CBK_ERR_DTYPE;
  const int fam = family_of(m.layout);
  const int vec = (((uintptr_t)out | (uintptr_t)(ld * (odt == CBK_F32 ? 4 : 2))) & 15) == 0;   // whole 16-byte stores
  if (fam == FAM_SPARSE) {
    const dim3 grid((unsigned)((nrows + ST_DQ_ROWS - 1) / ST_DQ_ROWS)), blk(256);
    const int summed = stream_sums(m) ? 1 : 0;
    const size_t lds = summed ? (size_t)m.G * 4 : 0;
    if (odt == CBK_F32) hipLaunchKernelGGL(dequant_sparse_kernel<CBK_F32>, grid, blk, lds, st, m, row0, nrows, with_cs, out, ld, vec, summed);
    else if (odt == CBK_F16) hipLaunchKernelGGL(dequant_sparse_kernel<CBK_F16>, grid, blk, lds, st, m, row0, nrows, with_cs, out, ld, vec, summed);
    else hipLaunchKernelGGL(dequant_sparse_kernel<CBK_BF16T>, grid, blk, lds, st, m, row0, nrows, with_cs, out, ld, vec, summed);
  } else if (fam == FAM_BLK6) {
    launch_fixed<FAM_BLK6, 6>(m, row0, nrows, with_cs, out, odt, ld, vec, st);
  } else if (fam == FAM_DENSE) {
    if (m.bits == 2) launch_fixed<FAM_DENSE, 2>(m, row0, nrows, with_cs, out, odt, ld, vec, st);
    else if (m.bits == 3) launch_fixed<FAM_DENSE, 3>(m, row0, nrows, with_cs, out, odt, ld, vec, st);
    else if (m.bits == 4) launch_fixed<FAM_DENSE, 4>(m, row0, nrows, with_cs, out, odt, ld, vec, st);
    else launch_fixed<FAM_DENSE, 8>(m, row0, nrows, with_cs, out, odt, ld, vec, st);
  } else {
    if (m.bits == 2) launch_fixed<FAM_BLK, 2>(m, row0, nrows, with_cs, out, odt, ld, vec, st);
    else if (m.bits == 3) launch_fixed<FAM_BLK, 3>(m, row0, nrows, with_cs, out, odt, ld, vec, st);
    else launch_fixed<FAM_BLK, 4>(m, row0, nrows, with_cs, out, odt, ld, vec, st);
  }
  return hipGetLastError() == hipSuccess ? CBK_OK : CBK_ERR_HIP;
}

}  // namespace cbk
