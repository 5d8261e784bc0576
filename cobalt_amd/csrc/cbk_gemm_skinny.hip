// Preparation kernel, reduction kernels, plan and dispatch of the GEMM in cbk_gemm_skinny.h.
#include "cbk_gemm_skinny.h"
#include "cbk_gemm_plan.h"
#include "cbk_prep.h"

namespace cbk {

int launch_skinny_b2(const SkArgs&, int keep, int group, int ti, int blocks, hipStream_t);
int launch_skinny_b3(const SkArgs&, int keep, int group, int ti, int blocks, hipStream_t);
int launch_skinny_b4(const SkArgs&, int keep, int group, int ti, int blocks, hipStream_t);
int launch_skinny_b68(const SkArgs&, int bits, int group, int ti, int blocks, hipStream_t);

// X' = fp16(x * col_scale / s_row) in fragment order and the sums of X' over the quantisation groups
// (see cbk_gemm_skinny.h), for every column-scale vector (blockIdx.z) and every part of the column range
// (blockIdx.y): a part is what one wavefront of the GEMM sums, so it has a scale per token of its own and
// no workgroup needs to see a whole row.  A workgroup takes eight tokens, whose 16-byte pieces of the
// same eight columns are a whole 128-byte line in that order.  Tokens past M are left unwritten, their
// outputs are never stored.  CH: pieces of the part a thread keeps in registers between the range pass
// and the write; 0 = any length, read twice.  (A scale per token over the whole row, found by one workgroup per
// four tokens or by every workgroup again, and half lines: 48 rows of 14336 columns 9 us, 512 rows 31.)
// Bound: latency at 48 rows, the write of X' at hundreds: without its stores the launch of 333 rows of 4096 columns and three
// vectors (8.2 MB) takes 4.9 us, with them 10.4, most of it the write-back of the L2s at its end, so the stores go on to
// memory (store16_through; non-temporal ones take 9.1, but the GEMM then reads X' 2 us slower).  The type of x and the
// order are compiled in, no load stands behind a condition of its own, sums go over lanes in registers: 333 rows 11.8 -> 9.7 us,
// 512 rows of 14336 columns 12.8 -> 9.0, 48 rows 5.9 -> 4.8.  Sixteen tokens per workgroup, stores of 256 bytes: 10.1, 13.6, 5.2.
__device__ inline float skinny_scale(float mx) {                   // the power of two that brings mx into [128, 256)
  if (!(mx > 0.f)) return 1.f;
  if (!(mx <= 3.4028234663852886e38f)) return SK_INFINITE;          // (mx is no NaN: fmaxf passes those over)
  int e = (int)((__float_as_uint(mx) >> 23) & 0xffu) - 7;          // its biased exponent
  e = e < 1 ? 1 : e;
  return __uint_as_float((uint32_t)e << 23);
}
// f of a lane's value and that of lane ^ 8, ^ 16, ^ 32, without a trip through LDS; f is commutative
template <typename F>
__device__ inline float lanes8(float v, F f) {                      // (a row of sixteen lanes turned by eight)
  return f(v, __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(v), 0x128, 0xf, 0xf, false)));
}
template <typename F>
__device__ inline float lanes16(float v, F f) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return f(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
template <typename F>
__device__ inline float lanes32(float v, F f) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return f(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
template <int CH, int XDT, int ORDER>
__global__ __launch_bounds__(1024) void skinny_prep_kernel(const uint16_t* x, int64_t ldx, const uint16_t* cs, int M, int N,
                                                           int lg, int ti, uint32_t inv_nq, uint16_t* out, size_t xps,
                                                           uint32_t* sums, size_t xcs, float* scale, int rss) {
  __shared__ float red[16][8];
  const int tid = threadIdx.x, tl = tid & 7, v = blockIdx.z, q = blockIdx.y, nq = gridDim.y;
  const int tok = blockIdx.x * 8 + tl;
  const bool ok = tok < M;
  // groups of 1 << lg columns; nothing is divided here (the part's bounds by the host's reciprocal)
  const int G = N >> lg, T8 = blockDim.x >> 3;
  const int b8 = (int)__umulhi((uint32_t)(G * q), inv_nq) << (lg - 3), e8 = (int)__umulhi((uint32_t)(G * (q + 1)), inv_nq) << (lg - 3);
  if (b8 == e8) {                                                   // (more parts than groups)
    if (ok && tid < 8) scale[((size_t)v * nq + q) * rss + tok] = 1.f;
    return;
  }
  const uint16_t* xr = x + (size_t)(ok ? tok : M - 1) * ldx;
  const uint16_t* cv = cs ? cs + (size_t)v * N : nullptr;
  const uint4 one = make_uint4(0x3c003c00u, 0x3c003c00u, 0x3c003c00u, 0x3c003c00u);
  float a[CH ? CH : 1][8];
  float mx = 0.f;
  auto range = [&](const float (&f)[8]) {
#pragma unroll
    for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(f[e]));
  };
  const int c0 = b8 + (tid >> 3);
  if (CH) {
    uint4 xk[CH ? CH : 1], ck[CH ? CH : 1];
#pragma unroll
    for (int i = 0; i < CH; ++i) {                                  // pieces past the part: its last one again
      const int c8 = c0 + T8 * i < e8 ? c0 + T8 * i : e8 - 1;
      xk[i] = *(const uint4*)(xr + c8 * 8);
      ck[i] = one;
    }
    if (cv)
#pragma unroll
      for (int i = 0; i < CH; ++i) ck[i] = *(const uint4*)(cv + (c0 + T8 * i < e8 ? c0 + T8 * i : e8 - 1) * 8);
#pragma unroll
    for (int i = 0; i < CH; ++i) { prep8(xk[i], ck[i], XDT, a[i]); range(a[i]); }
  } else {
    for (int c8 = c0; c8 < e8; c8 += T8) {
      prep8(*(const uint4*)(xr + c8 * 8), cv ? *(const uint4*)(cv + c8 * 8) : one, XDT, a[0]);
      range(a[0]);
    }
  }
  auto larger = [](float l, float r) { return fmaxf(l, r); };
  auto plus = [](float l, float r) { return l + r; };
  mx = lanes32(lanes16(lanes8(mx, larger), larger), larger);
  if ((tid & 63) < 8) red[tid >> 6][tl] = mx;
  __syncthreads();
  const int nw = blockDim.x >> 6;
  float all = red[0][tl];
#pragma unroll
  for (int w = 1; w < 16; ++w) all = fmaxf(all, red[w < nw ? w : 0][tl]);
  const float s = skinny_scale(all), inv = 1.f / s;                 // powers of two
  if (ok && tid < 8) scale[((size_t)v * nq + q) * rss + tok] = s;
  const uint32_t t32 = blockIdx.x >> 2, tile = ti == 1 ? t32 : ti == 2 ? t32 >> 1 : __umulhi(t32, 0xAAAAAAABu) >> 1;
  const uint32_t i32 = t32 - tile * ti, l = tok & 31;
  const auto o0 = through_buffer(out + (size_t)v * xps + ((size_t)tile * (N >> 4) * ti + i32) * 512);
  uint32_t* s0 = sums + (size_t)v * xcs + (size_t)tile * G * 2 * ti * 32 + i32 * 32 + l;
  auto emit = [&](int c8, const float (&f)[8]) {                    // (the pieces of half a group emit together: its sum needs all of them)
    uint16_t h[8];
    float sum = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) { h[e] = f2h(f[e] * inv); sum += h2f(h[e]); }
    uint32_t o[4];
    auto pair = [&](int lo, int hi) { return (uint32_t)h[lo] | ((uint32_t)h[hi] << 16); };
#pragma unroll
    for (int e = 0; e < 4; ++e)                                     // SkCfg::ORDER: as they are; even columns, then odd ones; 0 4 1 5 2 6 3 7
      o[e] = ORDER == 0 ? pair(2 * e, 2 * e + 1) : ORDER == 1 ? pair((4 * e + (e >> 1)) & 7, (4 * e + (e >> 1) + 2) & 7) : pair(e, e + 4);
    sum = lanes16(lanes8(sum, plus), plus);                         // the pieces of half a group: 32 or 64 columns
    const float both = lanes32(sum, plus);
    if (lg == 7) sum = both;
    const uint32_t run = (uint32_t)c8 >> (lg - 4), t = c8 & ((1 << (lg - 4)) - 1);   // half group, step in it
    if (ok && c8 < e8) {
      store16_through(o0, ((run >> 1 << (lg - 4)) + t) * (uint32_t)ti * 1024u + (run & 1) * 512u + l * 16u, make_uint4(o[0], o[1], o[2], o[3]));
      if (t == 0) {
        const uint16_t hi = f2h(sum), lo = f2h(sum - h2f(hi));
        s0[(size_t)run * ti * 32] = (uint32_t)hi | ((uint32_t)lo << 16);
      }
    }
  };
  if (CH) {
#pragma unroll
    for (int i = 0; i < CH; ++i) emit(c0 + T8 * i, a[i]);
  } else {
    // (no wavefront has both pieces of the part and pieces past it in one half group)
    for (int c8 = c0; c8 < e8; c8 += T8) {
      prep8(*(const uint4*)(xr + c8 * 8), cv ? *(const uint4*)(cv + c8 * 8) : one, XDT, a[0]);
      emit(c8, a[0]);
    }
  }
}

template <int CH, int XDT>
static auto skinny_prep_of(int order) {
  return order == 0 ? skinny_prep_kernel<CH, XDT, 0> : order == 1 ? skinny_prep_kernel<CH, XDT, 1> : skinny_prep_kernel<CH, XDT, 2>;
}
template <int XDT>
static auto skinny_prep_of(int ch, int order) {
  return ch <= 4 ? skinny_prep_of<4, XDT>(order) : ch <= 8 ? skinny_prep_of<8, XDT>(order) : skinny_prep_of<0, XDT>(order);
}

// y = sum of the float32 partial tiles in part order (+ bias); ACT: act(gate) * up of the interleaved
// gate / up sums.  Four outputs per thread.
template <bool ACT>
__global__ __launch_bounds__(256) void skinny_reduce_kernel(const float* part, size_t part_stride, int64_t part_ld, int nsplit,
                                                            int M, int K, const void* bias, void* y, int ydt, int64_t ldy,
                                                            int act) {
  constexpr int W = ACT ? 8 : 4;                                    // sums per thread
  const int Ko = ACT ? K >> 1 : K, k4 = (Ko + 3) >> 2;
  const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (id >= (int64_t)M * k4) return;
  const int tok = (int)(id / k4), o0 = (int)(id % k4) * 4, k0 = ACT ? 2 * o0 : o0;
  float v[W];
#pragma unroll
  for (int e = 0; e < W; ++e) v[e] = 0.f;
  const float* src = part + (size_t)tok * part_ld + k0;
  for (int p = 0; p < nsplit; ++p)
#pragma unroll
    for (int h = 0; h < W / 4; ++h) {
      const float4 f = ((const float4*)(src + (size_t)p * part_stride))[h];
      v[4 * h] += f.x; v[4 * h + 1] += f.y; v[4 * h + 2] += f.z; v[4 * h + 3] += f.w;
    }
  if (bias)
#pragma unroll
    for (int e = 0; e < W; ++e)
      if (k0 + e < K) v[e] += ydt == CBK_F32 ? ((const float*)bias)[k0 + e] : ydt == CBK_F16 ? h2f(((const uint16_t*)bias)[k0 + e]) : bf2f(((const uint16_t*)bias)[k0 + e]);
  float o[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = ACT ? sk_act(act, v[ACT ? 2 * e : e]) * v[ACT ? 2 * e + 1 : e] : v[e];
  const int esz = ydt == CBK_F32 ? 4 : 2;
  const bool vec = (((uintptr_t)y | (uintptr_t)(ldy * esz)) & (4 * esz - 1)) == 0;
  sk_store4(y, ydt, (size_t)tok * ldy + o0, o, Ko - o0, vec);
}

// ------------------------------------------------------------------ plan
static inline size_t sk_up(size_t v) { return (v + 255) & ~(size_t)255; }

// the matrices this kernel has a decoder for
bool gemm_skinny_takes(const DMat& m) {
  const int fam = family_of(m.layout);
  if (fam == FAM_SPARSE || (m.group != 64 && m.group != 128)) return false;
  if (m.cs_rows == 3 && (m.cs_split0 % SK_ROWS || (m.cs_split0 + m.cs_split1) % SK_ROWS)) return false;
  // 32-bit offsets inside a wavefront's 128 rows
  if ((uint64_t)m.stride * 160 >= (1ull << 32)) return false;
  if (fam == FAM_DENSE) return true;
  if (!(m.flags & CBK_FLAG_ZERO_ON_GRID)) return false;             // (a pruned column's zero point is decoded as a code)
  if (fam == FAM_BLK6) return m.bits == 6 && m.keep == 16 && m.group == 128;
  return m.keep == 10 || m.keep == 16 || m.keep == 23;
}

struct SkSpace { size_t x, sums, scale, part; int mpad; };
static SkSpace sk_space(const DMat& m, int M, int ti, int nsplit) {
  SkSpace s;
  s.mpad = (M + 32 * ti - 1) / (32 * ti) * (32 * ti);
  const size_t nv = m.cs_rows > 1 ? m.cs_rows : 1;
  s.x = sk_up(nv * s.mpad * m.N * 2);
  s.sums = sk_up(nv * s.mpad * m.G * 8);
  s.scale = sk_up(nv * s.mpad * nsplit * SK_WC * 4);                // one per part of the column range
  s.part = nsplit > 1 ? sk_up((size_t)nsplit * M * ((m.K + 7) / 8 * 8) * 4) : 0;
  return s;
}
static inline size_t sk_sum(const SkSpace& s) { return s.x + s.sums + s.scale + s.part; }
// Times in microseconds, fitted to calls of ten shapes (1024 x 4096 to 43008 x 5376) at 16 to 1700 rows,
// within a tenth of the measured ones: a group of a wavefront with two wavefronts per SIMD, by token tile
// (codes that do not start on 16-byte units take a fifth longer, 6-bit codes with their second plane
// 1.35, 1.27 and 1.07 times on the three tiles: 21504 x 5376 at 32, 64 and 96 rows 38.0, 45.7 and 50.3), 5.5 to 10 per workgroup outside the loop, 7.4 for the preparation kernel and the launches and 0.5 per megabyte of X' beyond four (written, and
// fetched by every XCD: 1024 x 5376 at 4096 rows, 44 MB, took 25 more than without that term), 5.5 and the
// partial tiles at 4 TB/s for the reduction kernel.
static GemmPlan sk_plan_ti(const DMat& m, int M, int ti, size_t room) {
  const int tiles = ((M + 32 * ti - 1) / (32 * ti)) * ((m.K + SK_ROWS * SK_WR - 1) / (SK_ROWS * SK_WR));
  static const double g128[3] = {1.7, 2.2, 2.8}, g64[3] = {1.17, 1.45, 1.53}, wg[3] = {5.5, 7.6, 10.0}, six[3] = {1.35, 1.27, 1.07};
  const bool skewed = family_of(m.layout) == FAM_BLK && (m.keep * m.bits * (m.group / 64)) % 32 != 0;
  const double two = m.cs_rows == 2 ? 1.12 : 1.0;                   // (two sets of X' compete for L2)
  const double t_group = (m.group == 128 ? g128 : g64)[ti - 1] * (skewed ? 1.2 : m.bits == 6 ? six[ti - 1] : 1.0) * two, t_wg = wg[ti - 1] * two;
  const double xmb = 2e-6 * (m.cs_rows > 1 ? m.cs_rows : 1) * (double)M * m.N, t_prep = 7.4 + (xmb > 4.0 ? 0.5 * (xmb - 4.0) : 0.0);
  GemmPlan best;
  for (int s = 1; s <= 16; ++s) {
    const size_t bytes = sk_sum(sk_space(m, M, ti, s));
    if (bytes > room) break;                                        // (more parts take more)
    const int per = (m.G + SK_WC * s - 1) / (SK_WC * s);
    double t = t_prep + (double)((tiles * s + 255) / 256) * (per * t_group + t_wg);
    if (s > 1) t += 2.0 * s * (double)M * m.K * 4 / 4.0e6 + 5.5;
    if (s == 1 || t < best.t) best = {GEMM_ROWS, ti, s, t, bytes};
    if (SK_WC * s >= m.G) break;
  }
  return best;
}
GemmPlan plan_skinny(const DMat& m, int M, size_t room) {
  GemmPlan best;
  if (M < 1 || !gemm_skinny_takes(m)) return best;
  for (int ti = 1; ti <= 3; ++ti) {
    const GemmPlan p = sk_plan_ti(m, M, ti, room);
    if (p.kernel && (!best.kernel || p.t < best.t)) best = p;
  }
  return best;
}
GemmPlan fixed_plan_skinny(const DMat& m, int M, int ti, int nsplit) {
  GemmPlan p;
  if (M < 1 || !gemm_skinny_takes(m) || ti < 1 || ti > 3 || nsplit < 1 || nsplit > 16 || SK_WC * (nsplit - 1) >= m.G) return p;
  p.kernel = GEMM_ROWS; p.ti = ti; p.nsplit = nsplit; p.bytes = sk_sum(sk_space(m, M, ti, nsplit));
  return p;
}

int launch_gemm_skinny(const DMat& m, const GemmPlan& plan, const void* x, int xdt, int M, int64_t ldx, void* y, int ydt,
                       int64_t ldy, const void* bias, int act, void* ws, size_t ws_bytes, hipStream_t st) {
  if (plan.kernel != GEMM_ROWS || !gemm_skinny_takes(m) || (act >= 0 && ((m.K & 1) || m.cs_rows == 3))) return CBK_ERR_UNSUPPORTED;
  const SkSpace sp = sk_space(m, M, plan.ti, plan.nsplit);
  if (!ws || ws_bytes < sk_sum(sp)) return CBK_ERR_WORKSPACE;
  if ((uintptr_t)ws & 255) return CBK_ERR_ALIGN;
  const int nv = m.cs_rows > 1 ? m.cs_rows : 1;
  SkArgs a;
  a.m = m; a.M = M; a.y = y; a.ydt = ydt; a.ldy = ldy; a.bias = bias;
  a.xp = (const uint16_t*)ws;
  a.xc = (const uint32_t*)((uint8_t*)ws + sp.x);
  a.row_scale = (const float*)((uint8_t*)ws + sp.x + sp.sums);
  a.par = m.cs_rows == 2 || act >= 0 ? 1 : 0;
  a.act = act;
  // (a gate/up matrix with one vector: both parities read the same X')
  a.xps = nv > 1 ? (size_t)sp.mpad * m.N : 0;
  a.xcs = nv > 1 ? (size_t)sp.mpad * m.G * 2 : 0;
  a.rss = sp.mpad;
  a.rvs = nv > 1 ? a.rss * plan.nsplit * SK_WC : 0;
  a.vs0 = m.cs_rows == 3 ? m.cs_split0 : 0x7fffffff;
  a.vs1 = m.cs_rows == 3 ? m.cs_split0 + m.cs_split1 : 0x7fffffff;
  a.nsplit = plan.nsplit;
  a.part = (float*)((uint8_t*)ws + sp.x + sp.sums + sp.scale);
  a.part_ld = (m.K + 7) / 8 * 8;
  a.part_stride = (size_t)M * a.part_ld;
  a.tiles_t = sp.mpad / (32 * plan.ti);
  a.tiles_r = (m.K + SK_ROWS * SK_WR - 1) / (SK_ROWS * SK_WR);
  const int order = family_of(m.layout) != FAM_DENSE || m.bits == 8 ? 0 : m.bits == 2 ? 2 : 1;   // SkCfg::ORDER
  const int nq = plan.nsplit * SK_WC, p8 = (m.G + nq - 1) / nq * (m.group / 8);   // parts, 16-byte pieces of the longest
  const int want = (2 * p8 + 63) / 64 * 64;                         // four pieces per thread
  const int threads = want > 1024 ? 1024 : want, ch = (8 * p8 + threads - 1) / threads;
  auto prep = xdt == CBK_F16 ? skinny_prep_of<CBK_F16>(ch, order) : skinny_prep_of<CBK_BF16T>(ch, order);
  hipLaunchKernelGGL(prep, dim3((unsigned)((M + 7) / 8), (unsigned)nq, (unsigned)nv), dim3(threads), 0, st, (const uint16_t*)x,
                     ldx, m.cs, M, m.N, m.group == 64 ? 6 : 7, plan.ti, (uint32_t)(((1ull << 32) + nq - 1) / nq), (uint16_t*)ws, a.xps,
                     (uint32_t*)a.xc, a.xcs, (float*)a.row_scale, a.rss);
  const int nb = a.tiles_t * a.tiles_r * a.nsplit, blocks = (nb + 7) / 8 * 8;
  const int fam = family_of(m.layout), keep = fam == FAM_DENSE ? 0 : m.keep;
  int rc;
  if (m.bits == 8 || fam == FAM_BLK6) rc = launch_skinny_b68(a, m.bits, m.group, plan.ti, blocks, st);
  else rc = m.bits == 2 ? launch_skinny_b2(a, keep, m.group, plan.ti, blocks, st)
          : m.bits == 3 ? launch_skinny_b3(a, keep, m.group, plan.ti, blocks, st) : launch_skinny_b4(a, keep, m.group, plan.ti, blocks, st);
  if (rc == CBK_OK && a.nsplit > 1) {
    const int Ko = act >= 0 ? m.K / 2 : m.K;
    const int64_t items = (int64_t)M * ((Ko + 3) / 4);
    const dim3 grid((unsigned)((items + 255) / 256));
    if (act >= 0) hipLaunchKernelGGL(skinny_reduce_kernel<true>, grid, dim3(256), 0, st, (const float*)a.part, a.part_stride,
                                     a.part_ld, a.nsplit, M, m.K, bias, y, ydt, ldy, act);
    else hipLaunchKernelGGL(skinny_reduce_kernel<false>, grid, dim3(256), 0, st, (const float*)a.part, a.part_stride,
                            a.part_ld, a.nsplit, M, m.K, bias, y, ydt, ldy, act);
    if (hipGetLastError() != hipSuccess) rc = CBK_ERR_HIP;
  }
  return rc;
}

}  // namespace cbk
