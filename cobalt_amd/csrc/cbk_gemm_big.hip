// Prefill GEMM: activation pre-scaling kernel, the generic-reader instantiation
// and the dispatch over the per-code-width instantiations (cbk_gemm_big_b2/3/4.hip).  The
// kernel itself is in cbk_gemm_big.h.
#include "cbk_gemm_big.h"
#include "cbk_gemm_plan.h"
#include "cbk_prep.h"

namespace cbk {

int launch_gemm_big_b2(const GbArgs&, int keep, int group, int blocks, hipStream_t);
int launch_gemm_big_b3(const GbArgs&, int keep, int group, int blocks, hipStream_t);
int launch_gemm_big_b4(const GbArgs&, int keep, int group, int blocks, hipStream_t);
int launch_gemm_big_b6(const GbArgs&, int blocks, hipStream_t);

// ---- X' = fp16(x * col_scale / s_row), [Mpad, Npad] row-major, and s_row, one workgroup per row.
// s_row is the power of two that brings the row's largest |x * col_scale| below 2^15 (1 for
// nearly every row: only magnitudes beyond fp16's range need it); the GEMM kernel multiplies the
// row's outputs by it.  Rows M..Mpad-1 and columns N..Npad-1 are zero.
// One workgroup of T threads per row.  CH: 16-byte pieces of the row a thread keeps in
// registers between the two passes (the row is read from memory once); 0 = any row length, the
// second pass reads the row again.  Bound: reading x and writing X'.  The type of x is compiled in and no load stands behind a
// condition of its own (a wavefront waited for each piece before it asked for the next); long rows take 512 threads and
// six pieces rather than 1024 and three (four workgroups on a CU, so one's loads run beside another's stores); stores go on to
// memory (store16_through).  2048 rows of 21504 columns (176 MB moved) 40.0 -> 32.7 us, 2 x 2048 of 5376 17.9 -> 15.5.
template <int CH, int T, int XDT>
__global__ __launch_bounds__(T) void gemm_prep_kernel(const uint16_t* x, int64_t ldx, const uint16_t* cs, int M, int N, int Npad,
                                                      uint16_t* out, size_t out_vs, float* row_scale, int scale_vs) {
  __shared__ float red[T / 64];
  const int row = blockIdx.x, tid = threadIdx.x;
  const int n8 = Npad >> 3, nv = N >> 3;                           // N is a multiple of 128
  cs = cs ? cs + (size_t)blockIdx.y * N : nullptr;                  // one column-scale vector per blockIdx.y
  row_scale += (size_t)blockIdx.y * scale_vs;
  uint16_t* orow = out + (size_t)blockIdx.y * out_vs + (size_t)row * Npad;
  if (row >= M) {
    for (int c8 = tid; c8 < n8; c8 += T) *(uint4*)(orow + c8 * 8) = make_uint4(0, 0, 0, 0);
    if (tid == 0) row_scale[row] = 1.f;
    return;
  }
  const uint16_t* xr = x + (size_t)row * ldx;
  const uint4 one = make_uint4(0x3c003c00u, 0x3c003c00u, 0x3c003c00u, 0x3c003c00u);
  float a[CH ? CH : 1][8];
  float mx = 0.f;
  auto range = [&](const float (&f)[8]) {
#pragma unroll
    for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(f[e]));
  };
  if (CH) {
    // Pieces past the row: its last one again.  No load behind a condition of its own, which would wait for the one before.
    uint4 xv[CH ? CH : 1], cv[CH ? CH : 1];
#pragma unroll
    for (int i = 0; i < CH; ++i) { xv[i] = *(const uint4*)(xr + (tid + T * i < nv ? tid + T * i : nv - 1) * 8); cv[i] = one; }
    if (cs)
#pragma unroll
      for (int i = 0; i < CH; ++i) cv[i] = *(const uint4*)(cs + (tid + T * i < nv ? tid + T * i : nv - 1) * 8);
#pragma unroll
    for (int i = 0; i < CH; ++i) { prep8(xv[i], cv[i], XDT, a[i]); range(a[i]); }
  } else {
    for (int c8 = tid; c8 < nv; c8 += T) {
      prep8(*(const uint4*)(xr + c8 * 8), cs ? *(const uint4*)(cs + c8 * 8) : one, XDT, a[0]);
      range(a[0]);
    }
  }
#pragma unroll
  for (int o = 32; o; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
  if ((tid & 63) == 0) red[tid >> 6] = mx;
  __syncthreads();
  float all = red[0];
#pragma unroll
  for (int w = 1; w < T / 64; ++w) all = fmaxf(all, red[w]);
  const float s = token_scale(all);
  const float inv = 1.f / s;                                       // a power of two: exact
  if (tid == 0) row_scale[row] = s;
  const auto dst = through_buffer(orow);
  auto emit = [&](int c8, const float (&f)[8]) {
    uint32_t o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = (uint32_t)f2h(f[2 * e] * inv) | ((uint32_t)f2h(f[2 * e + 1] * inv) << 16);
    const bool in = c8 < nv;
    store16_through(dst, (uint32_t)c8 * 16u, make_uint4(in ? o[0] : 0u, in ? o[1] : 0u, in ? o[2] : 0u, in ? o[3] : 0u));
  };
  if (CH) {
#pragma unroll
    for (int i = 0; i < CH; ++i)
      if (tid + T * i < n8) emit(tid + T * i, a[i]);
  } else {
    for (int c8 = tid; c8 < n8; c8 += T) {
      const int c = c8 < nv ? c8 : nv - 1;
      prep8(*(const uint4*)(xr + c * 8), cs ? *(const uint4*)(cs + c * 8) : one, XDT, a[0]);
      emit(c8, a[0]);
    }
  }
}

typedef decltype(&gemm_prep_kernel<1, 256, CBK_F16>) PrepKernel;
template <int XDT>
static PrepKernel prep_of(int p8, int* threads) {                  // p8: 16-byte pieces of a row
  if (p8 <= 1024) {
    *threads = 256;
    return p8 <= 256 ? gemm_prep_kernel<1, 256, XDT> : p8 <= 512 ? gemm_prep_kernel<2, 256, XDT>
         : p8 <= 768 ? gemm_prep_kernel<3, 256, XDT> : gemm_prep_kernel<4, 256, XDT>;
  }
  *threads = 512;
  return p8 <= 2048 ? gemm_prep_kernel<4, 512, XDT> : p8 <= 3072 ? gemm_prep_kernel<6, 512, XDT>
       : p8 <= 4096 ? gemm_prep_kernel<8, 512, XDT> : gemm_prep_kernel<0, 512, XDT>;
}

static inline int gb_npad(int N) { return (N + 255) / 256 * 256; }

// ---- y = sum of the float32 partial tiles (+ bias), eight outputs per thread
__global__ __launch_bounds__(256) void gemm_split_reduce_kernel(const float* part, size_t part_stride, int64_t part_ld,
                                                               int nsplit, int M, int K, const void* bias, void* y,
                                                               int ydt, int64_t ldy) {
  const int k8 = (K + 7) >> 3;
  const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (id >= (int64_t)M * k8) return;
  const int tok = (int)(id / k8), k0 = (int)(id % k8) * 8;
  float v[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = 0.f;
  for (int p = 0; p < nsplit; ++p) {                                // fixed order: run-to-run identical
    const float* src = part + (size_t)p * part_stride + (size_t)tok * part_ld + k0;
    const float4 a = ((const float4*)src)[0], b = ((const float4*)src)[1];
    v[0] += a.x; v[1] += a.y; v[2] += a.z; v[3] += a.w; v[4] += b.x; v[5] += b.y; v[6] += b.z; v[7] += b.w;
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int k = k0 + e;
    if (k >= K) break;
    float o = v[e];
    if (bias) o += ydt == CBK_F32 ? ((const float*)bias)[k] : ydt == CBK_F16 ? h2f(((const uint16_t*)bias)[k]) : bf2f(((const uint16_t*)bias)[k]);
    const size_t at = (size_t)tok * ldy + k;
    if (ydt == CBK_F32) ((float*)y)[at] = o;
    else if (ydt == CBK_F16) ((uint16_t*)y)[at] = f2h(o);
    else ((uint16_t*)y)[at] = f2bf(o);
  }
}

// the matrices the byte-permute instantiations take (the others go through the generic reader,
// whose launches are never split)
static bool gb_fast(const DMat& m) {
  const int fam = family_of(m.layout);
  if (!(m.flags & CBK_FLAG_ZERO_LE_128) || (m.group != 64 && m.group != 128)) return false;
  if (fam == FAM_BLK6) return m.bits == 6 && m.keep == 16 && m.group == 128;
  if (m.bits < 2 || m.bits > 4) return false;
  if (fam == FAM_BLK) return m.keep == 10 || m.keep == 16 || m.keep == 23;
  return fam == FAM_DENSE;
}

// Token tile and split of the column range of a call.
//  * A launch of fewer tiles than a multiple of the 256 CUs leaves CUs idle for a whole tile
//    time; cutting the column range over several workgroups per output tile gives them work at
//    the price of the float32 partial tiles (written and read once).
//  * Calls of at most 64 / 128 activation rows take the 64- / 128-token tile.  Larger calls
//    take the 256-token tile unless the model below gives the 128-token tile the shorter time,
//    which it does for small matrices (4096 x 4096 at 256 to 2048 rows: 16 to 128 tiles of 256
//    tokens): twice the tiles, each 0.8 of the time.
// Times in microseconds, as measured when the kernel had 32 x 32 x 16 instructions: per 64-column stage 1.1 / 1.35 / 1.7
// for the three tiles, 8 - 10 per workgroup outside the stage loop, 4 TB/s for the partial tiles, 5 for the reduction kernel.  (With 1.25 and
// 7 TB/s, which fit a few small calls better, 4096 x 4096 at 2048 rows went from 92 to 104 us, 3840 x 7424 at 1024 from 89 to
// 98.)  Over 24 calls measured then
// (eight shapes, 256 / 512 / 2048 rows) the choice was within 2 % of the faster tile; always
// taking the 256-token tile lost 6 % on average and up to 34 %.
// The present kernel, a tile on every CU without a pause: 4-bit, 16 of 32 0.84 / 1.09 / 1.77; dense 0.73 - 0.89 / 1.00 - 1.22 /
// 1.52 - 1.95; 3-bit, 23 of 32 1.09 / 1.31 / 1.94; 6-bit 1.04 / 1.32 / 1.98; outside the loop 5 - 14.  So the model takes the
// smaller tiles for up to a third slower than they are and knows no code width.
static inline double gb_t_stage(int ti) { return ti == 1 ? 1.1 : ti == 2 ? 1.35 : 1.7; }
static inline double gb_t_wg(int ti) { return ti == 1 ? 8.0 : 10.0; }
static inline size_t gb_kpad(int K) { return (size_t)(K + 7) / 8 * 8; }
static size_t gb_space(const DMat& m, int M, int ti, int nsplit) {
  const size_t T = 64 * ti, mpad = (size_t)(M + T - 1) / T * T;
  const size_t nv = m.cs_rows > 1 ? m.cs_rows : 1;
  size_t b = (nv * mpad * gb_npad(m.N) * 2 + 255) & ~(size_t)255;     // X', one per col_scale vector
  b += (nv * mpad * 4 + 255) & ~(size_t)255;                          // and its row scales
  if (nsplit > 1) b += ((size_t)nsplit * M * gb_kpad(m.K) * 4 + 255) & ~(size_t)255;
  return b;
}
// stages per part, a multiple of 4; 0: a part would be empty
static int gb_part(const DMat& m, int nsplit) {
  const int nst = gb_npad(m.N) / GB_K, per = ((nst + nsplit - 1) / nsplit + 3) / 4 * 4;
  return nsplit > 1 && (nsplit - 1) * per >= nst ? 0 : per;
}
// The parts of a launch whose plan is `nsplit` parts of `tiles` tiles.  They are equal, but where a plan cuts 129 to 192 tiles
// in n >= 3 parts to fill n - 1 rounds: there two parts may do, the first ones, a workgroup each on its CU from the start,
// so long that the CUs without one need as long for all the second ones.  The same CU time with fewer partial tiles, and a
// workgroup's start and end less for most.  Workgroups go to the eight XCDs in turn and to the four shader engines of one in turn, and stay there:
// it is the eight CUs of an engine that share its second parts (168 tiles, 228 + 108 stages, as 256 CUs would
// share them: three turns instead of two, 5376 x 21504 at 2048 tokens 447 -> 574 us).  Equal and unequal parts, us, with preparation
// and reduction: 160 tiles 5120 x 20480 426 -> 408, 4096 x 14336 320 -> 307; 144 tiles 4608 x 18432 374 -> 360; 192 tiles
// 6144 x 24576 578 -> 552.  Above 192 tiles one CU of an engine would run seven second parts in turn: equal parts.
// (The plan does not count it: calls keep their kernel and room.)
static GbCut gb_cut(const DMat& m, int tiles, int ti, int nsplit) {
  const int per = gb_part(m, nsplit), nst = gb_npad(m.N) / GB_K;
  GbCut c = {nsplit, per, per};
  const int held = ((tiles + 7) / 8 + 3) / 4, left = 8 - held;      // CUs of a shader engine with and without a first part
  if (nsplit < 3 || tiles <= 128 || left < 2) return c;
  const double t_stage = gb_t_stage(ti), t_wg = gb_t_wg(ti);
  const int turns = (held + left - 1) / left;                       // second parts of a CU without a first one
  double best = (double)((tiles * nsplit + 255) / 256) * (per * t_stage + t_wg);
  for (int s = 4; 2 * s < nst; s += 4) {
    const double first = (nst - s) * t_stage + t_wg, rest = turns * (s * t_stage + t_wg), t = first > rest ? first : rest;
    if (t < best) { best = t; c = {2, nst - s, s}; }
  }
  return c;
}
static GemmPlan gb_plan_ti(const DMat& m, int M, int ti, int max_split, size_t room) {
  const int T = 64 * ti;
  const int tiles = ((M + T - 1) / T) * ((m.K + GB_R - 1) / GB_R);
  const double t_stage = gb_t_stage(ti), t_wg = gb_t_wg(ti);
  GemmPlan best, one;
  const bool may_split = max_split > 1 && m.cs_rows != 2 && gb_fast(m);
  for (int s = 1; s <= (may_split ? max_split : 1); ++s) {
    const int per = gb_part(m, s);
    if (!per) continue;
    const size_t bytes = gb_space(m, M, ti, s);
    if (bytes > room) continue;
    const double rounds = (double)((tiles * s + 255) / 256);
    double t = rounds * (per * t_stage + t_wg);
    if (s > 1) t += 2.0 * s * (double)M * m.K * 4 / 4.0e6 + 5.0;
    if (s == 1) best = one = {GEMM_TILE, ti, 1, t, bytes};
    else if (t < best.t) best = {GEMM_TILE, ti, s, t, bytes};
  }
  return best.t > 0.93 * one.t ? one : best;                        // (not worth a second kernel)
}
static GemmPlan gb_plan(const DMat& m, int M, int max_split, size_t room) {
  if (M <= 64) return gb_plan_ti(m, M, 1, max_split, room);
  if (M <= 128) return gb_plan_ti(m, M, 2, max_split, room);
  const GemmPlan p4 = gb_plan_ti(m, M, 4, max_split, room), p2 = gb_plan_ti(m, M, 2, max_split, room);
  return !p4.kernel || (p2.kernel && p2.t < p4.t) ? p2 : p4;
}
// the q|k|v matrices it takes whole: ranges that start on its row tiles
static bool gb_takes(const DMat& m, int M) {
  if (M < 1 || family_of(m.layout) == FAM_SPARSE) return false;
  return m.cs_rows <= 2 || (m.cs_split0 % GB_R == 0 && (m.cs_split0 + m.cs_split1) % GB_R == 0);
}
size_t big_unsplit_space(const DMat& m, int M) { return gb_plan(m, M, m.cs_rows <= 1 ? 16 : 1, ANY_ROOM).bytes; }
GemmPlan fixed_plan_big(const DMat& m, int M, int ti, int nsplit) {
  GemmPlan p;
  if (!gb_takes(m, M) || (ti != 1 && ti != 2 && ti != 4) || nsplit < 1 || nsplit > 16 || !gb_part(m, nsplit) ||
      (nsplit > 1 && (m.cs_rows == 2 || !gb_fast(m))))
    return p;
  p.kernel = GEMM_TILE; p.ti = ti; p.nsplit = nsplit; p.bytes = gb_space(m, M, ti, nsplit);
  return p;
}

// `t` is what a call takes, for the choice between this kernel and the one in cbk_gemm_skinny.h: the tile's and
// split's time, 5 us for the preparation kernel and the launch.  Partial tiles count at 6.5 TB/s here: 4 is what keeps the plan from
// splitting where it does not pay, calls that are split measure faster (14336 x 4096 at 256 rows 61 us, 3840 x 7424 at
// 1024 rows 89).  Layouts without a decoder of their own are read at a
// tenth of the rate.
GemmPlan plan_big(const DMat& m, int M, size_t room) {
  if (!gb_takes(m, M)) return GemmPlan();
  GemmPlan p = gb_plan(m, M, 16, room);
  const double parts = p.nsplit > 1 ? 2.0 * p.nsplit * (double)M * m.K * 4 : 0.0;
  p.t = (p.t - parts * (1 / 4.0e6 - 1 / 6.5e6)) * (gb_fast(m) ? 1.0 : 10.0) + 5.0;
  return p;
}

// Last round of a launch of 256-token tiles.  Tiles beyond a whole number of rounds over the 256 CUs keep a few CUs busy
// for a whole tile time; the row tiles that hold them go into a second launch of 64- or 128-token tiles if those fit one
// round.  Every output is the same sum in the same order whatever its tile.  Measured, N = 5376 at 2048 tokens, with the
// preparation: 64 tiles of 256 tokens 134 us, as 128 of 128 103, as 256 of 64 88; 128 tiles 135, as 256 of 128 109, as
// 512 of 64 162 (two rounds: not taken).
// The plan does not count it: a share of a tile time taken off the unsplit 256-token plan moved calls onto it that ran
// faster where they were (us before / after: 38323 x 256 at 294 tokens, 128-token tile, 44 / 54; 30878 x 7680 at 587,
// 96-token rows, 351 / 380; 5376 x 21504 at 3600, three parts, 923 / 946), off the 64-token rows kernel, which does not
// round weights, and within the room of cbk_gemm_static.
static int gb_row_tiles(const DMat& m) {                            // (gate/up: both parities of each range of rows)
  return m.cs_rows == 2 ? 2 * ((m.K + 2 * GB_R - 1) / (2 * GB_R)) : (m.K + GB_R - 1) / GB_R;
}
LastRound last_round_big(const DMat& m, const GemmPlan& p, int M) {
  if (p.kernel != GEMM_TILE || p.ti != 4 || p.nsplit != 1 || !gb_fast(m)) return LastRound();
  const int tiles_r = gb_row_tiles(m), tiles_t = (M + GB_T - 1) / GB_T;
  const int full = tiles_t * tiles_r / 256, left = tiles_t * tiles_r - 256 * full;
  if (!full || !left) return LastRound();
  int rows = (left + tiles_t - 1) / tiles_t;
  if (m.cs_rows == 2) rows += rows & 1;
  if (rows >= tiles_r) return LastRound();
  for (int ti = 1; ti <= 2; ++ti)
    if ((M + 64 * ti - 1) / (64 * ti) * rows <= 256) return {rows, ti};
  return LastRound();
}

GbCut cut_big(const DMat& m, const GemmPlan& p, int M) {            // (only unsplit plans have a last round of their own)
  return gb_cut(m, (M + 64 * p.ti - 1) / (64 * p.ti) * gb_row_tiles(m), p.ti, p.nsplit);
}

static int gb_launch(const GbArgs& a, hipStream_t st) {
  const DMat& m = a.m;
  const int tiles = a.tiles_t * a.tiles_r;
  const int blocks = a.nst_first == a.nst_part ? (tiles * a.nsplit + 7) / 8 * 8 : (tiles + 7) / 8 * 8 * a.nsplit;
  const bool le128 = (m.flags & CBK_FLAG_ZERO_LE_128) != 0;
  const int fam = family_of(m.layout);
  int rc = CBK_ERR_UNSUPPORTED;
  if (le128 && (fam == FAM_BLK || fam == FAM_DENSE)) {
    const int keep = fam == FAM_DENSE ? 0 : m.keep;
    if (m.bits == 2) rc = launch_gemm_big_b2(a, keep, m.group, blocks, st);
    else if (m.bits == 3) rc = launch_gemm_big_b3(a, keep, m.group, blocks, st);
    else if (m.bits == 4) rc = launch_gemm_big_b4(a, keep, m.group, blocks, st);
  } else if (le128 && fam == FAM_BLK6 && m.bits == 6 && m.keep == 16 && m.group == 128) {
    rc = launch_gemm_big_b6(a, blocks, st);
  }
  if (rc == CBK_ERR_UNSUPPORTED) {
    if (a.nsplit > 1) return CBK_ERR_UNSUPPORTED;                   // (only what the cases above take is ever split)
    rc = launch_big_cfg<0, 0, 128>(a, blocks, st);                  // generic reader
  }
  return rc;
}

int launch_gemm_big(const DMat& m, const GemmPlan& plan, const void* x, int xdt, int M, int64_t ldx, void* y, int ydt,
                    int64_t ldy, const void* bias, void* ws, size_t ws_bytes, hipStream_t st, bool halves) {
  if (halves && (m.cs_rows != 2 || (m.K & 1) || bias)) return CBK_ERR_UNSUPPORTED;
  // (q|k|v ranges off the row-tile grid: the caller passes them one by one)
  if (plan.kernel != GEMM_TILE || !gb_takes(m, M)) return CBK_ERR_UNSUPPORTED;
  if (ydt != CBK_F32 && ydt != CBK_F16 && ydt != CBK_BF16T) return CBK_ERR_DTYPE;
  if (!ws || ws_bytes < gb_space(m, M, plan.ti, plan.nsplit)) return CBK_ERR_WORKSPACE;
  if ((uintptr_t)ws & 255) return CBK_ERR_ALIGN;
  const int T = 64 * plan.ti;
  const int Mpad = (M + T - 1) / T * T;
  const int Npad = gb_npad(m.N);
  const int par = m.cs_rows == 2 ? 1 : 0;
  const int nv = m.cs_rows > 1 ? m.cs_rows : 1;
  const size_t xbytes = ((size_t)nv * Mpad * Npad * 2 + 255) & ~(size_t)255;
  const size_t sbytes = ((size_t)nv * Mpad * 4 + 255) & ~(size_t)255;
  float* row_scale = (float*)((uint8_t*)ws + xbytes);
  int threads;
  const PrepKernel prep = xdt == CBK_F16 ? prep_of<CBK_F16>(Npad / 8, &threads) : prep_of<CBK_BF16T>(Npad / 8, &threads);
  hipLaunchKernelGGL(prep, dim3((unsigned)Mpad, (unsigned)nv), dim3(threads), 0, st, (const uint16_t*)x, ldx, m.cs, M, m.N, Npad,
                     (uint16_t*)ws, (size_t)Mpad * Npad, row_scale, Mpad);   // one X' per col_scale vector
  GbArgs a;
  a.m = m; a.xp = (const uint16_t*)ws; a.M = M; a.Npad = Npad; a.y = y; a.ydt = ydt; a.ldy = ldy; a.bias = bias;
  a.par = par; a.xps = (size_t)Mpad * Npad;
  a.halves = halves ? 1 : 0;
  a.row_scale = row_scale; a.rss = Mpad;
  a.vs0 = m.cs_rows == 3 ? m.cs_split0 : 0x7fffffff;
  a.vs1 = m.cs_rows == 3 ? m.cs_split0 + m.cs_split1 : 0x7fffffff;
  a.part_ld = (int64_t)gb_kpad(m.K);
  a.part_stride = (size_t)M * gb_kpad(m.K);
  a.part = (float*)((uint8_t*)ws + xbytes + sbytes);
  a.ti = plan.ti;
  a.tr0 = 0;
  a.tiles_t = (M + T - 1) / T;
  const LastRound tail = last_round_big(m, plan, M);
  a.tiles_r = gb_row_tiles(m) - tail.rows;
  const GbCut cut = cut_big(m, plan, M);
  a.nsplit = cut.nsplit; a.nst_first = cut.first; a.nst_part = cut.part;
  int rc = gb_launch(a, st);
  if (rc == CBK_OK && tail.rows) {
    a.tr0 = a.tiles_r;
    a.tiles_r = tail.rows;
    a.ti = tail.ti;
    a.tiles_t = (M + 64 * a.ti - 1) / (64 * a.ti);
    rc = gb_launch(a, st);
  }
  if (rc == CBK_OK && a.nsplit > 1) {
    const int64_t items = (int64_t)M * ((m.K + 7) / 8);
    hipLaunchKernelGGL(gemm_split_reduce_kernel, dim3((unsigned)((items + 255) / 256)), dim3(256), 0, st,
                       (const float*)a.part, a.part_stride, a.part_ld, a.nsplit, M, m.K, bias, y, ydt, ldy);
    if (hipGetLastError() != hipSuccess) rc = CBK_ERR_HIP;
  }
  return rc;
}

}  // namespace cbk
