// Entry points of the many-rows linears (kernels: qgemm_rows.h, qgemm_tall.hip).
#include "qgemm_rows.h"

#define X(F) int tga_rows_launch_##F(const RowsArgs& a, int tt, unsigned grid, hipStream_t s);
ROWS_FORMATS(X)
#undef X

// format id of a block type with rows of K values, -1: not taken (K a multiple of 128 and of the superblock; the pair formats read 4-byte aligned rows)
int tga_rows_fmt(int ggml_type, int64_t K) {
  const bool k256 = K % 256 == 0;
  if (K < 128 || K % 128) return -1;
  switch (ggml_type) {
    case GGML_Q4_0: return F_Q4_0P;
    case GGML_Q8_0: return F_Q8_0P;
    case GGML_F16: case GGML_MXFP4: case GGML_Q4_1: case GGML_Q5_0: case GGML_Q5_1: return ggml_type;
    case GGML_Q4_K: case GGML_Q5_K: case GGML_Q6_K: case GGML_IQ4_XS: return k256 ? ggml_type : -1;
  }
  return -1;
}
int64_t tga_rows_row_bytes(int fmt, int64_t K) {
  switch (fmt) {
    case F_Q4_0P: return K / 32 * 18;
    case F_Q8_0P: return K / 32 * 34;
    case GGML_F16: return K * 2;
    case GGML_MXFP4: return K / 32 * 17;
    case GGML_Q4_1: return K / 32 * 20;
    case GGML_Q5_0: return K / 32 * 22;
    case GGML_Q5_1: return K / 32 * 24;
    case GGML_Q4_K: return K / 256 * 144;
    case GGML_Q5_K: return K / 256 * 176;
    case GGML_Q6_K: return K / 256 * 210;
    case GGML_IQ4_XS: return K / 256 * 136;
  }
  return 0;
}
int tga_rows_tall(int fmt, const RowsArgs& a, unsigned grid, hipStream_t s);             // qgemm_tall.hip
#define ROWS_TALL 512             // the tile height that asks for it
#define TALL_K_MIN 1024
int tga_rows_dispatch(int fmt, const RowsArgs& a, int tt, unsigned grid, hipStream_t s) {
  if (tt == ROWS_TALL) return tga_rows_tall(fmt, a, grid, s);
  switch (fmt) {
#define X(F) case F: return tga_rows_launch_##F(a, tt, grid, s);
    ROWS_FORMATS(X)
#undef X
  }
  return tga_set_error("tga_qlinear_many: no kernel for format %d", fmt);
}

// y = [residual +] the partial sums of a split K in its order; 4 neighbouring weight rows per thread
__global__ __launch_bounds__(256) void rows_reduce_kernel(const RowsArgs a) {
  const long long q4 = a.ntot / 4, total = (long long)a.M * q4, plane = (long long)a.M * a.ntot;
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < total; i += (long long)gridDim.x * 256) {
    const long long t = i / q4; long long row = (i - t * q4) * 4;
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
    const float* p = a.part + t * a.ntot + row;
    for (int k = 0; k < a.ks; k++) { const f32x4 v = *(const f32x4*)(p + k * plane); o.x += v.x; o.y += v.y; o.z += v.z; o.w += v.w; }
    int sg = 0;
    if (a.nseg > 1 && row >= a.n[0]) { row -= a.n[0]; sg = 1; if (a.nseg > 2 && row >= a.n[1]) { row -= a.n[1]; sg = 2; } }
    void* yb = sg == 0 ? a.y[0] : sg == 1 ? a.y[1] : a.y[2];
    const long long at = t * (sg == 0 ? a.n[0] : sg == 1 ? a.n[1] : a.n[2]) + row;
    if (a.epi == ROWS_RESID) { const f32x4 r = *(const f32x4*)(a.resid + at); o.x += r.x; o.y += r.y; o.z += r.z; o.w += r.w; }
    if (a.y_f32) *(f32x4*)((float*)yb + at) = o;
    else *(u32x2*)((uint16_t*)yb + at) = u32x2{f2h_bits(o.x) | (f2h_bits(o.y) << 16), f2h_bits(o.z) | (f2h_bits(o.w) << 16)};
  }
}

// The norm of the residual stream, with the sums of a split K completed on the way (ks > 1: x += partial sums in their order, what rows_reduce_kernel does): a workgroup per row, which
// stays in registers between its sum and its norm, 16-byte requests.  In place of a reduce launch and a norm launch that reads the row again: 1023 rows of 4096, four and two partial sums, 14 + 10.9 -> 14 us a time.
template <int V>
__global__ __launch_bounds__(512) void rows_norm_kernel(const float* __restrict__ part, int ks, float* x, const float* __restrict__ w, int n, float eps, uint16_t* __restrict__ xn) {
  __shared__ float red[8];
  const int tid = threadIdx.x, n4 = n / 4;
  const size_t row = (size_t)blockIdx.x * n, plane = (size_t)gridDim.x * n;
  f32x4 v[V], g[V];
#pragma unroll
  for (int j = 0; j < V; j++) { const int i = min(tid + 512 * j, n4 - 1); v[j] = *(const f32x4*)(x + row + 4 * i); g[j] = *(const f32x4*)(w + 4 * i); }
  if (ks > 1) {
    f32x4 o[V];
#pragma unroll
    for (int j = 0; j < V; j++) o[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int k = 0; k < ks; k++) {
#pragma unroll
      for (int j = 0; j < V; j++) {
        const f32x4 t = *(const f32x4*)(part + k * plane + row + 4 * min(tid + 512 * j, n4 - 1));
        o[j].x += t.x; o[j].y += t.y; o[j].z += t.z; o[j].w += t.w;
      }
    }
#pragma unroll
    for (int j = 0; j < V; j++) {
      v[j].x += o[j].x; v[j].y += o[j].y; v[j].z += o[j].z; v[j].w += o[j].w;
      if (tid + 512 * j < n4) *(f32x4*)(x + row + 4 * (tid + 512 * j)) = v[j];
    }
  }
  float s = 0.f;
#pragma unroll
  for (int j = 0; j < V; j++) if (tid + 512 * j < n4) s += v[j].x * v[j].x + v[j].y * v[j].y + v[j].z * v[j].z + v[j].w * v[j].w;
  s = wave_sum(s);
  if ((tid & 63) == 0) red[tid >> 6] = s;
  __syncthreads();
  float tot = 0.f;
#pragma unroll
  for (int i = 0; i < 8; i++) tot += red[i];
  const float sc = 1.0f / sqrtf(tot / (float)n + eps);
#pragma unroll
  for (int j = 0; j < V; j++) {
    if (tid + 512 * j < n4) *(u32x2*)(xn + row + 4 * (tid + 512 * j)) = u32x2{f2h_bits((v[j].x * sc) * g[j].x) | (f2h_bits((v[j].y * sc) * g[j].y) << 16),
                                                                             f2h_bits((v[j].z * sc) * g[j].z) | (f2h_bits((v[j].w * sc) * g[j].w) << 16)};
  }
}
#define ROWS_NORM_MAX 8192
// xn = norm(x [+ the ks partial sums behind part]) of M rows of n values, n a multiple of 4, at most ROWS_NORM_MAX
static int rows_norm(const float* part, int ks, float* x, const float* w, int M, int n, float eps, void* xn, hipStream_t s) {
  const int v = (n / 4 + 511) / 512;
  if (v == 1) rows_norm_kernel<1><<<M, 512, 0, s>>>(part, ks, x, w, n, eps, (uint16_t*)xn);
  else if (v == 2) rows_norm_kernel<2><<<M, 512, 0, s>>>(part, ks, x, w, n, eps, (uint16_t*)xn);
  else rows_norm_kernel<4><<<M, 512, 0, s>>>(part, ks, x, w, n, eps, (uint16_t*)xn);
  TGA_LAUNCH_CHECK();
  return 0;
}

// How a set of matrices is cut: tiles (tt: ROWS_WIDE or the activation rows of a tile of ROWS_WT weight rows) and the split of K, which is cut while the tiles leave CUs with fewer than
// two workgroups and a part keeps at least `least` values of it.
static int rows_split(const RowsArgs& a, bool may_split, size_t part_bytes, int least) {
  if (!may_split) return 1;
  int k = (int)(512 / ((long long)a.row_tiles * a.tok_tiles));
  if (k > a.K / least) k = a.K / least;
  while (k > 1 && (size_t)k * a.M * a.ntot * 4 > part_bytes) k--;
  return k < 1 ? 1 : k;
}
// The 256 x 128 tiles: a workgroup's start and end cost about 4 us more than the smaller tile's, so it takes them where a workgroup has twelve steps of 256 or more and at least 320 of
// them are running (4096 -> 6144 of 1023 rows, eight steps each: 87 us, the smaller tiles 83; 2047 rows, sixteen steps: 141 and 144; 4096 -> 2 x 14336 of 300 rows, 336 workgroups: 140 and 146,
// of 128 rows, 112 workgroups: 79 and 62).
static bool rows_wide(RowsArgs& a, int fmt, bool swiglu, bool may_split, size_t part_bytes) {
  if (fmt != F_Q4_0P || a.M <= 64 || a.K % 256 || a.K > (1 << 20) || a.ntot >= (1ll << 30)) return false;
  const int wt = swiglu ? WIDE_WT / 2 : WIDE_WT;
  a.row_tiles = (int)((a.ntot + wt - 1) / wt); a.tok_tiles = (a.M + WIDE_TT - 1) / WIDE_TT;
  a.ks = rows_split(a, may_split, part_bytes, 512);
  return a.K / 256 / a.ks >= 12 && (long long)a.row_tiles * a.tok_tiles * a.ks >= 320;
}
static int rows_plan_small(RowsArgs& a, int fmt, bool swiglu, bool may_split, size_t part_bytes) {
  if (rows_wide(a, fmt, swiglu, may_split, part_bytes)) return ROWS_WIDE;
  const int wt = swiglu ? ROWS_WT / 2 : ROWS_WT;
  a.row_tiles = (int)((a.ntot + wt - 1) / wt);
  // A product of few 128 x 128 x 128 steps takes tiles of fewer rows: more workgroups, each done sooner.  us with 128 / 64 / 32 rows a tile: 16 steps (Q4_0 512 -> 512, 100 rows) 11.4 / 7.9 / 7.0,
  // 224 (Q8_0 3584 -> 1024, 100) 15.9 / 12.6 / 11.4, 512 (fp16 2048 -> 2048, 200) 17.3 / 14.5 / 14.6, 1536 (Q4_0 4096 -> 6144, 100) 25.9 / 23.9 / 27.3, 1792 (Q8_0 3584 -> 1024, 1000) 27.6 / 23.9 / 27.0,
  // 3072 (Q4_0 4096 -> 6144, 200) 31.0 / 33.7 / 40.4, 3584 (Q4_K 14336 -> 4096, 100) 36.2 / 38.9 / 54.1; fp16, which decodes nothing: 3072 (2048 -> 6144, 511) 34.7 / 30.7 / 30.2, 6144 (1000) 46.4 / 40.8 / 54.7;
  // Q6_K, whose decode is the longest, 64 / 128 rows a tile: 768 steps 21.4 / 20.8 and 21.9 / 21.5, 1024 (five products, K 2048 .. 8192) 23.9 / 23.8, 22.1 / 22.1, 24.5 / 23.7, 24.2 / 22.9, 21.4 / 21.0,
  // 1152 (3072 -> 3072, 200) 25.2 / 28.0, 1536 30.9 / 28.3, 28.4 / 28.0, 26.9 / 28.3, 2048 31.6 / 30.0, 31.3 / 28.9, 4096 50.7 / 41.5: alike up to 1536 steps, 128 rows from there on.
  const long long steps = (long long)a.row_tiles * ((a.M + 127) / 128) * (a.K / ROWS_KS);
  const int tt = a.M <= 32 || steps < 512 ? 32 : a.M <= 64 || steps <= (fmt == GGML_F16 ? 6144 : fmt == GGML_Q6_K ? 1023 : 2048) ? 64 : 128;
  a.tok_tiles = (a.M + tt - 1) / tt;
  a.ks = rows_split(a, may_split, part_bytes, 4 * ROWS_KS);
  return tt;
}

// The 512 x 128 tiles of qgemm_tall.hip (one workgroup per CU) against the plan above (two): the choice falls by the time either takes, us, as measured on products of K 1024 .. 14336, 64 .. 2047 rows and
// 1024 .. 28672 outputs: a round of tall tiles 9 + 5.1 a step of 256, up to 6.3 where all CUs have one (the clock falls with the power), of 256 x 128 tiles 8 + 7.8, of 128 rows 6 + 2.1 a step of 128
// (1.65 where CUs have only one workgroup), of 64 rows 5 + 1.25 (1.05); Q4_K a sixth more in tall tiles; a split of K writes its sums and reads them.  A last round that is nearly empty costs tall tiles more
// than it costs small ones.  us, the plan above / tall tiles: Q4_0 4096 -> 2 x 14336 (SwiGLU), 300, 508, 640, 1023, 2047 rows 128 / 92, 131 / 106, 197 / 197 (not taken), 260 / 209, 488 / 448, Q4_K
// 135 / 106, 148 / 120, 215 / 230 (not taken), 291 / 237, 606 / 511; Q4_0 14336 -> 4096, 300, 508, 1023, 2047 rows 69 / 61, 86 / 77, 142 / 124, 257 / 217; 4096 -> 6144 of 768, 1023, 2047 rows 77 / 60, 76 / 70,
// 134 / 100; 4096 -> 4096 of 1023 rows 57 / 59 (not taken); 2048 -> 2 x 5632 of 1023 rows 65 / 53, of 640 43 / 52 (not taken); 3072 -> 2 x 8448 of 1280 rows,
// two rounds two thirds full, 146 / 156 (not taken); 14336 -> 4096 of 150 rows 45 / 47 (not taken).
// Several rounds of few steps pay each round's ramp (5 us above the estimate) and need a fuller last one: Q4_0, fewer than six steps, 71 % full 1280 -> 2 x 17312 of 1023 rows 119 / 125 (not taken), 77 % 1024 -> 2 x 12464 of
// 1024 rows 77 / 73; from six on 73 % 1536 -> 2 x 8784 of 2047 rows 146 / 143; Q4_K, fewer than eight, 77 % 1024 -> 2 x 18896 of 1024 rows 114 / 123, 74 % 1536 -> 2 x 24288 of 768 rows 152 / 161 (not taken), 81 %
// 1536 of 2 rounds 117 / 108; from eight on 76 % 2048 -> 2 x 18672 of 1024 rows 213 / 206.
static double rows_split_us(const RowsArgs& a) { return a.ks == 1 ? 0. : 2. + (double)a.ks * a.M * a.ntot * 8e-6 / 6.5; }
static double rows_us(const RowsArgs& a, int tt) {
  const long long wg = (long long)a.row_tiles * a.tok_tiles * a.ks;
  const double steps = (double)a.K / ROWS_KS / a.ks;
  if (tt == ROWS_WIDE) return (double)((wg + 511) / 512) * (8. + 3.9 * steps) + rows_split_us(a);
  if (tt == 128) return (double)((wg + 511) / 512) * (6. + (wg > 256 ? 2.1 : 1.65) * steps) + rows_split_us(a);
  return tt == 64 ? (double)((wg + 767) / 768) * (5. + (wg > 256 ? 1.25 : 1.05) * steps) + rows_split_us(a) : 0.;
}
static int rows_plan(RowsArgs& a, int fmt, bool swiglu, bool may_split, size_t part_bytes) {
  const int tt = rows_plan_small(a, fmt, swiglu, may_split, part_bytes);
  // (whole sub-tiles of sixteen rows, requests of sixteen bytes; below TALL_K_MIN nothing is measured, and the kernel's touches take two steps)
  if ((fmt != F_Q4_0P && fmt != GGML_Q4_K) || tt == 32 || a.K % 256 || a.K < TALL_K_MIN || a.K > (1 << 20) || a.ntot >= (1ll << 30)) return tt;
  for (int i = 0; i < (swiglu ? 2 : a.nseg); i++) if (a.n[i] % 16 || ((uintptr_t)a.w[i] & 15)) return tt;
  RowsArgs t = a, best = a;
  double us = rows_us(a, tt);
  const int wt = swiglu ? ROWS_TALL / 2 : ROWS_TALL;
  t.row_tiles = (int)((a.ntot + wt - 1) / wt); t.tok_tiles = (a.M + 127) / 128;
  const int steps = a.K / 256;
  const long long tiles = (long long)t.row_tiles * t.tok_tiles, per = (tiles + 7) / 8;       // (of the 32 CUs of an XCD)
  bool taken = false;
  for (int least = 5; least <= 7; least += 2) {
    t.ks = 1;
    if (may_split && per <= 32) {
      t.ks = (int)(32 / per);
      if (t.ks > steps / least) t.ks = steps / least;
      while (t.ks > 1 && (size_t)t.ks * a.M * a.ntot * 4 > part_bytes) t.ks--;
      if (t.ks < 1) t.ks = 1;
    }
    const long long rounds = (per * t.ks + 31) / 32;
    const double full = (double)(tiles * t.ks) / (double)(256 * rounds);
    const bool q4_k = fmt == GGML_Q4_K;
    if (full < (rounds == 1 ? 0.5 : steps / t.ks >= (q4_k ? 8 : 6) ? 0.7 : q4_k ? 0.78 : 0.75)) continue;
    const double step = (5.1 + (full > 0.6 ? 3. * (full - 0.6) : 0.)) * (q4_k ? 1.16 : 1.);
    const double e = (double)rounds * (9. + step * steps / t.ks) + rows_split_us(t);
    if (e < us) { us = e; best = t; taken = true; }
  }
  if (!taken) return tt;
  a = best;
  return ROWS_TALL;
}

// tga_qlinear_many; norm_w != nullptr (one matrix, epilogue 1 in place, fp32): also xn = fp16 RMSNorm of the result's rows; parts != nullptr (epilogue 0): the sums of a split K stay in the workspace,
// [parts][M][outputs of all matrices], for the caller to complete in their order (parts 1: they are in y)
int tga_rows_linear(int ggml_type, int nseg, const void* const* w, void* const* y, const int64_t* n, const void* x_f16, int y_dtype, int64_t M, int64_t K, int epilogue, const float* resid,
                    void* workspace, int64_t workspace_bytes, const float* norm_w, float norm_eps, void* xn, int* parts, void* stream) {
  TGA_REQUIRE(w && y && n && x_f16 && nseg >= 1 && nseg <= 3, "tga_qlinear_many: null pointer or %d matrices", nseg);
  TGA_REQUIRE(epilogue >= 0 && epilogue <= 2 && (epilogue != 2 || nseg == 2) && (epilogue != 1 || (nseg == 1 && resid)), "tga_qlinear_many: epilogue %d with %d matrices", epilogue, nseg);
  TGA_REQUIRE(y_dtype == TGA_F32 || y_dtype == TGA_F16, "tga_qlinear_many: y_dtype must be TGA_F16 or TGA_F32");
  const int fmt = tga_rows_fmt(ggml_type, K);
  TGA_REQUIRE(fmt >= 0 && M >= 1 && M * K < (1ll << 32) && M < (1 << 24), "tga_qlinear_many: type %d with K=%lld, M=%lld is outside the range", ggml_type, (long long)K, (long long)M);
  RowsArgs a = {};
  const int segs = epilogue == 2 ? 1 : nseg;
  for (int i = 0; i < nseg; i++) {
    TGA_REQUIRE(w[i] && n[i] > 0 && (i >= segs || y[i]), "tga_qlinear_many: null pointer in matrix %d", i);
    TGA_REQUIRE(((uintptr_t)w[i] & (ggml_type == GGML_F16 ? 15 : ggml_type == GGML_MXFP4 ? 0 : 3)) == 0, "tga_qlinear_many: weights must be 4-byte aligned (fp16: 16-byte)");
    TGA_REQUIRE(i + 1 >= segs || n[i] % 16 == 0, "tga_qlinear_many: matrices that share a launch need a multiple of 16 rows");
    a.w[i] = (const uint8_t*)w[i]; a.n[i] = n[i];
    if (i < segs) { a.y[i] = y[i]; a.ntot += n[i]; TGA_REQUIRE(((uintptr_t)y[i] & 15) == 0, "tga_qlinear_many: results must be 16-byte aligned"); }
  }
  TGA_REQUIRE(epilogue != 2 || n[0] == n[1], "tga_qlinear_many: gate and up differ in rows");
  TGA_REQUIRE((((uintptr_t)x_f16 | (uintptr_t)resid | (uintptr_t)workspace) & 15) == 0, "tga_qlinear_many: activations must be 16-byte aligned");
  a.row_bytes = tga_rows_row_bytes(fmt, K); a.x = (const uint16_t*)x_f16; a.resid = resid; a.part = (float*)workspace; a.nseg = segs; a.epi = epilogue; a.y_f32 = y_dtype == TGA_F32;
  a.M = (int)M; a.K = (int)K;
  bool split = epilogue != 2 && workspace && a.ntot % 4 == 0;
  for (int i = 0; i < segs; i++) split = split && n[i] % 4 == 0;
  const int tt = rows_plan(a, fmt, epilogue == 2, split, (size_t)workspace_bytes);
  if (a.ks > 1) a.epi = ROWS_PART;
  const unsigned grid = (unsigned)(((long long)a.row_tiles * a.tok_tiles + 7) / 8 * 8);
  if (const int rc = tga_rows_dispatch(fmt, a, tt, grid, (hipStream_t)stream)) return rc;
  const bool norm_here = norm_w && a.ntot <= ROWS_NORM_MAX && a.ntot % 4 == 0;
  if (norm_here) return rows_norm(a.part, a.ks, (float*)y[0], norm_w, (int)M, (int)a.ntot, norm_eps, xn, (hipStream_t)stream);
  if (parts) { *parts = a.ks; return 0; }
  if (a.ks > 1) {
    a.epi = epilogue;
    const long long total = M * (a.ntot / 4), wg = (total + 255) / 256;
    rows_reduce_kernel<<<(unsigned)(wg < 4096 ? wg : 4096), 256, 0, (hipStream_t)stream>>>(a);
    TGA_LAUNCH_CHECK();
  }
  return norm_w ? tga_rmsnorm_rows((const float*)y[0], norm_w, (int)M, (int)a.ntot, norm_eps, xn, nullptr, 0, stream) : 0;
}
// xn = fp16 RMSNorm of M rows of n values
int tga_rows_norm(float* x, const float* w, int M, int n, float eps, void* xn, void* stream) {
  if (n <= ROWS_NORM_MAX && n % 4 == 0) return rows_norm(nullptr, 1, x, w, M, n, eps, xn, (hipStream_t)stream);
  return tga_rmsnorm_rows(x, w, M, n, eps, xn, nullptr, 0, stream);
}

extern "C" {

int tga_qlinear_many(int ggml_type, int nseg, const void* const* w, void* const* y, const int64_t* n, const void* x_f16, int y_dtype, int64_t M, int64_t K, int epilogue,
                     const float* resid, void* workspace, int64_t workspace_bytes, void* stream) {
  return tga_rows_linear(ggml_type, nseg, w, y, n, x_f16, y_dtype, M, K, epilogue, resid, workspace, workspace_bytes, nullptr, 0.f, nullptr, nullptr, stream);
}

int tga_qlinear_many_tile(int ggml_type, int nseg, const int64_t* n, int64_t M, int64_t K, int epilogue, int64_t workspace_bytes, int* weight_rows, int* x_rows, int* parts) {
  const int fmt = tga_rows_fmt(ggml_type, K);
  TGA_REQUIRE(n && weight_rows && x_rows && parts && nseg >= 1 && nseg <= 3 && (epilogue != 2 || nseg == 2) && fmt >= 0 && M >= 1 && M * K < (1ll << 32) && M < (1 << 24) && workspace_bytes >= 0,
              "tga_qlinear_many_tile: null pointer, or a linear outside the range");
  RowsArgs a = {};
  a.nseg = epilogue == 2 ? 1 : nseg; a.M = (int)M; a.K = (int)K;
  bool split = epilogue != 2 && workspace_bytes > 0;
  for (int i = 0; i < nseg; i++) {
    TGA_REQUIRE(n[i] > 0, "tga_qlinear_many_tile: matrix %d has no rows", i);
    a.n[i] = n[i];
    if (i < a.nseg) { a.ntot += n[i]; split = split && n[i] % 4 == 0; }
  }
  const int tt = rows_plan(a, fmt, epilogue == 2, split, (size_t)workspace_bytes);
  *weight_rows = tt == ROWS_TALL ? 512 : tt == ROWS_WIDE ? WIDE_WT : ROWS_WT; *x_rows = tt == ROWS_TALL ? 128 : tt == ROWS_WIDE ? WIDE_TT : tt; *parts = a.ks;
  return 0;
}

}  // extern "C"
