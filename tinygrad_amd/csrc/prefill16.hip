// Prefill steps of many rows whose sums run in the order of the steps of sixteen rows (and of eight and four): every row of the keys, values and residuals has the bits those steps give it.
// An MoE model's expert choices at near-ties turn with the last bit of a sum, so its prompts keep that order (model.py:110-135, 464); what changes is that a weight matrix is read once for all rows
// of the prompt and not once for every sixteen (or, the experts', once for every token and slot).  Served: dense fp16 weights, MXFP4 experts, whole-row q / k norms, at most 4096 values in a row
// of the dense linears and 2048 in one of the experts' (prefill16_ok below); other models take the steps of sixteen.
// Orders that are kept, per output of a row:
//   dense linears (qgemm_wp.hip, qgemm_dma.hip, qgemm.hip)  steps of 256 values dealt to 8 (K a multiple of 1024) or 4 waves, two chains of matrix-core products per wave, waves summed in order
//   attention     (attn_decode_kernel, norm over whole rows) float32, partials per 64 positions from runs of lanes, merged in order
//   router        (moe_router_kernel)                        lanes' chains of dot2 over 16-byte pieces, then the tree over the wave
//   experts       (qgemv1.h)                                 a chain of sixteen dot2 per unit of 32 weights, its scale, then the tree over the units of the row
#include "qfmt.h"
#include "prefill.h"
#include "decode.h"
#include <utility>

typedef _Float16 v8f16 __attribute__((ext_vector_type(8)));
typedef _Float16 v4f16 __attribute__((ext_vector_type(4)));
typedef float v4f32 __attribute__((ext_vector_type(4)));
typedef float v16f32 __attribute__((ext_vector_type(16)));

// ------------------------------------------------------------------------------------------------ the dense linears
// 64 weight rows x 64 activation rows per workgroup, wave = 32 x 32.  K in steps of 256 values, staged whole by requests that write LDS themselves (two workgroups of 64 KB per CU: one loads while
// the other multiplies); row pieces of 16 bytes XORed with the row.  A step's operands are those of the sixteen-row kernels: lane 16 g + r holds the values 64 g + 8 v .. + 7 of row r for product v;
// products of even and odd v form two chains per part, parts (the steps of one wave there: p, p + nw, ...) are summed in order.
struct X16Gemm { const uint16_t* w[3]; float* y[3]; const float* resid; const uint16_t* x; int n[3]; int nseg, M, K, nw, ntiles; };
__global__ __launch_bounds__(256, 2) void x16_gemm_kernel(const X16Gemm a) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[65536];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4, r = lane & 15;
  const int mt = (a.M + 63) >> 6, xcd = blockIdx.x & 7, idx = blockIdx.x >> 3;
  int nt = (idx / mt) * 8 + xcd;                                          // (the row tiles of a weight tile on one XCD)
  const int m0 = (idx % mt) * 64;
  if (nt >= a.ntiles) return;
  int seg = 0;
  if (a.nseg > 1 && nt >= (a.n[0] >> 6)) { nt -= a.n[0] >> 6; seg = 1; if (nt >= (a.n[1] >> 6)) { nt -= a.n[1] >> 6; seg = 2; } }
  const uint16_t* w = (seg == 0 ? a.w[0] : seg == 1 ? a.w[1] : a.w[2]) + (size_t)nt * 64 * a.K;
  const int n = seg == 0 ? a.n[0] : seg == 1 ? a.n[1] : a.n[2];
  float* y = seg == 0 ? a.y[0] : seg == 1 ? a.y[1] : a.y[2];
  // request i of a wave fills 1 KB: rows 2 (wave + 4 i), + 1 of a 64-row tile
  const uint16_t* src[16];
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const int row = 2 * (wave + 4 * (i & 7)) + (lane >> 5), piece = (lane & 31) ^ (row & 15);
    const int xr = min(m0 + row, a.M - 1);
    src[i] = (i < 8 ? w + (size_t)row * a.K : a.x + (size_t)xr * a.K) + 8 * piece;
  }
  const int wr0 = (wave & 1) * 32, xr0 = (wave >> 1) * 32, nsteps = a.K >> 8;
  v4f32 c0[2][2], c1[2][2], tot[2][2];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) { c0[i][j] = c1[i][j] = tot[i][j] = v4f32{0.f, 0.f, 0.f, 0.f}; }
  for (int p = 0; p < a.nw && p < nsteps; p++) {
    for (int s = p; s < nsteps; s += a.nw) {
      __syncthreads();                                                    // everyone is done with the step before
#pragma unroll
      for (int i = 0; i < 16; i++)
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src[i] + 256 * s), (__attribute__((address_space(3))) void*)(lds + (i < 8 ? 0 : 32768) + (wave + 4 * (i & 7)) * 1024), 16, 0, 0);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
#pragma unroll
      for (int v = 0; v < 8; v++) {
        v8f16 wa[2], xb[2];
#pragma unroll
        for (int i = 0; i < 2; i++) {
          wa[i] = *(const v8f16*)(lds + (wr0 + 16 * i + r) * 512 + (((8 * g + v) ^ r) << 4));
          xb[i] = *(const v8f16*)(lds + 32768 + (xr0 + 16 * i + r) * 512 + (((8 * g + v) ^ r) << 4));
        }
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
          for (int j = 0; j < 2; j++) {
            if (v & 1) c1[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wa[i], xb[j], c1[i][j], 0, 0, 0);
            else c0[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wa[i], xb[j], c0[i][j], 0, 0, 0);
          }
      }
    }
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int j = 0; j < 2; j++) { const v4f32 part = c0[i][j] + c1[i][j]; tot[i][j] += part; c0[i][j] = c1[i][j] = v4f32{0.f, 0.f, 0.f, 0.f}; }
  }
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) {
      const int row = m0 + xr0 + 16 * j + r;
      if (row >= a.M) continue;
      const size_t o = (size_t)row * n + nt * 64 + wr0 + 16 * i + 4 * g;
      v4f32 v = tot[i][j];
      if (a.resid) v += *(const v4f32*)(a.resid + o);
      *(v4f32*)(y + o) = v;
    }
}

// ------------------------------------------------------------------------------------------------ the first norm of the steps of eight and four rows
// Those steps fold the first block's attn_norm into their q / k / v launch (qgemm_wp.hip / qgemm_dma.hip), whose waves sum the squares of 256 values each: lane l of wave w the values 256 w + 4 l .. + 3
__global__ __launch_bounds__(1024) void x16_fold_norm_kernel(const float* __restrict__ x, const float* __restrict__ w, int K, float eps, uint16_t* __restrict__ out) {
  __shared__ float nsum[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nw = K >> 8;
  x += (size_t)blockIdx.x * K; out += (size_t)blockIdx.x * K;
  f32x4 f = {0.f, 0.f, 0.f, 0.f}, nw4 = {0.f, 0.f, 0.f, 0.f};
  if (wave < nw) { f = ((const f32x4*)x)[tid]; nw4 = ((const f32x4*)w)[tid]; }
  float ps = 0.f;
  ps += f.x * f.x + f.y * f.y + f.z * f.z + f.w * f.w;
  ps = wave_sum(ps);
  if (lane == 0) nsum[wave] = ps;
  __syncthreads();
  float t = 0.f;
  for (int i = 0; i < nw; i++) t += nsum[i];
  const float sc = 1.0f / sqrtf(t / (float)K + eps);
  if (wave < nw) {
    f.x = (f.x * sc) * nw4.x; f.y = (f.y * sc) * nw4.y; f.z = (f.z * sc) * nw4.z; f.w = (f.w * sc) * nw4.w;
    ((u32x2*)out)[tid] = u32x2{f2h_bits(f.x) | (f2h_bits(f.y) << 16), f2h_bits(f.z) | (f2h_bits(f.w) << 16)};
  }
}

// ------------------------------------------------------------------------------------------------ q / k norm over whole rows, rotation, append
// One workgroup per row; the sums of squares as attn_decode_kernel forms them (four 16-byte pieces per thread of four waves, waves in order); eight waves rotate (four: 508 rows 9.0 us, eight 7.3).  q leaves rotated in float32.
__device__ __forceinline__ float x16_rope_lo(float x1, float x2, float c, float s) { return __builtin_fmaf(x1, c, -(x2 * s)); }
__device__ __forceinline__ float x16_rope_hi(float x1, float x2, float c, float s) { return __builtin_fmaf(x2, c, x1 * s); }
struct X16Rope { const float* q; const float* k; const float* v; const float* qn; const float* kn; const float* rope; float* qr; uint16_t* ck; uint16_t* cv; int* zero; int H, KV, hd, max_ctx, pos0, n_zero; float eps; };
__global__ __launch_bounds__(512) void x16_rope_kernel(const X16Rope a) {
  __shared__ float red[8];
  const int row = blockIdx.x, pos = a.pos0 + row, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, half = a.hd >> 1;
  const int nq = a.H * a.hd, nk = a.KV * a.hd;
  if (row == 0) for (int i = tid; i < a.n_zero; i += 512) a.zero[i] = 0;
  const float* q = a.q + (size_t)row * nq; const float* k = a.k + (size_t)row * nk; const float* v = a.v + (size_t)row * nk;
  const int n4q = nq >> 2, n4k = nk >> 2;
  if (wave < 4) {
    f32x4 nq4[4], nk4[4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
      const int i = tid + 256 * t;
      nq4[t] = ((const f32x4*)q)[i < n4q ? i : n4q - 1]; nk4[t] = ((const f32x4*)k)[i < n4k ? i : n4k - 1];
    }
    float s0 = 0.f, s1 = 0.f;
#pragma unroll
    for (int t = 0; t < 4; t++) {
      const int i = tid + 256 * t;
      const f32x4 x = nq4[t], y = nk4[t];
      s0 += i < n4q ? x.x * x.x + x.y * x.y + x.z * x.z + x.w * x.w : 0.f;
      s1 += i < n4k ? y.x * y.x + y.y * y.y + y.z * y.z + y.w * y.w : 0.f;
    }
    s0 = wave_sum(s0); s1 = wave_sum(s1);
    if (lane == 0) { red[wave] = s0; red[4 + wave] = s1; }
  }
  __syncthreads();
  const float qscale = 1.0f / sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)(a.H * a.hd) + a.eps);
  const float kscale = 1.0f / sqrtf((red[4] + red[5] + red[6] + red[7]) / (float)(a.KV * a.hd) + a.eps);
  const size_t cstep = (size_t)a.max_ctx * a.hd, crow = (size_t)pos * a.hd;
  for (int e = 4 * tid; e < nk; e += 2048) {
    const int hh = e / a.hd;
    const f32x4 x = *(const f32x4*)(v + e);
    *(u32x2*)(a.cv + crow + hh * cstep + (e - hh * a.hd)) = u32x2{f2h_bits(x.x) | (f2h_bits(x.y) << 16), f2h_bits(x.z) | (f2h_bits(x.w) << 16)};
  }
  const bool live = lane < half;
  const int i = live ? lane : half - 1;
  const float c = a.rope[(size_t)pos * a.hd + i], s = a.rope[(size_t)pos * a.hd + half + i];
#pragma unroll 4
  for (int h = wave; h < a.H + a.KV; h += 8) {
    const bool isq = h < a.H;
    const int o = (isq ? h : h - a.H) * a.hd;
    const float* src = isq ? q + o : k + o; const float* wn = isq ? a.qn + o : a.kn + o;
    const float sc = isq ? qscale : kscale;
    const float x1 = (src[i] * sc) * wn[i], x2 = (src[half + i] * sc) * wn[half + i];
    float lo = x16_rope_lo(x1, x2, c, s), hi = x16_rope_hi(x1, x2, c, s);
    asm volatile("" : "+v"(lo), "+v"(hi));                                // (float32 values before they are rounded to fp16, as there)
    if (!live) continue;
    if (isq) { float* d = a.qr + (size_t)row * nq + o; d[i] = lo; d[half + i] = hi; }
    else { uint16_t* d = a.ck + crow + (h - a.H) * cstep; d[i] = (uint16_t)f2h_bits(lo); d[half + i] = (uint16_t)f2h_bits(hi); }
  }
}

// ------------------------------------------------------------------------------------------------ attention
// The arithmetic of attn_decode_kernel (float32 products and sums, runs of HD8 lanes per row of keys, partials of 64 positions), with a workgroup's 64 keys and values in registers for the rows of a
// chunk: workgroup = (kv head, 64 positions, X16_ROWS rows); four (row, query head) pairs at a time.  Three workgroups fit a CU (153 registers; with
// 128 they spill: 78 us): of 512 rows and 16 heads 1152 workgroups of 32 rows, 1.5 rounds of the chip, or 2304 of 16, three: 60.5 -> 56.7 us.  Values behind a row's position are dropped by selects:
// 57.4 -> 62.5 us; a path of its own for tiles that hold a value that is not finite takes registers or hoisted conversions from the other one (61.5 .. 70.9 us).
// Bound by vector instructions, 170 a pair and wave.  Pairs counted on instead of divided, 62.8 -> 61.2, and without a branch per pair 59.7 us; two pairs step by step, or a loop without masks for tiles
// whose rows see all 64 positions (217 registers, or 168 with spills), were 62.8 and 62.8 .. 64.3.
#define X16_ROWS 16
struct X16Attn { const float* qr; const uint16_t* ck; const uint16_t* cv; float* part; uint16_t* out; int H, KV, max_ctx, P, pos0, nsplit; float scale; };

template <int HD8>
__device__ __forceinline__ float x16_run_sum(float v) {
  v = dpp_add<0xB1>(v); v = dpp_add<0x4E>(v); v = dpp_add<0x141>(v);
  if constexpr (HD8 >= 16) v = dpp_add<0x140>(v);
  return v;
}

template <int HD8>
__global__ __launch_bounds__(256) void x16_attn_kernel(const X16Attn a) {
  constexpr int HD = HD8 * 8, RPI = 64 / HD8, NVI = 16 / RPI, NGRP = 4 * RPI, CSTR = HD + 4;
  __shared__ float comb[4 * NGRP * CSTR];
  const int kvh = blockIdx.x, split = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int group = a.H / a.KV, vr = lane / HD8, vp = lane % HD8;
  const int row_end = min((int)(blockIdx.z + 1) * X16_ROWS, a.P), row_first = max((int)blockIdx.z * X16_ROWS, split * 64 - a.pos0);      // (rows that see a position of the split)
  if (row_first >= row_end) return;
  const int p0 = split * 64 + wave * 16, last = a.pos0 + a.P - 1;
  u32x4 kt[NVI], vt[NVI];
  {
    const uint16_t* kb = a.ck + (size_t)kvh * a.max_ctx * HD + vp * 8; const uint16_t* vb = a.cv + (size_t)kvh * a.max_ctx * HD + vp * 8;
#pragma unroll
    for (int i = 0; i < NVI; i++) {
      const int rc = min(p0 + i * RPI + vr, last);                         // (beyond the rows appended so far: masked below, but 0 times what lies there has to be 0)
      kt[i] = *(const u32x4*)(kb + (size_t)rc * HD); vt[i] = *(const u32x4*)(vb + (size_t)rc * HD);
    }
  }
  const int np = (row_end - row_first) * group;
  f32x4 qa[4], qb[4];
  int fp = 0, fh = 0;                                                      // the next pair to fetch: number, head in its group
  const float* fs = a.qr + ((size_t)row_first * a.H + kvh * group) * HD + vp * 8;
  const int to_row = (a.H - group + 1) * HD;
  auto fetch = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int hh = 0; hh < 4; hh++) {
      qa[hh] = *(const f32x4*)fs; qb[hh] = *(const f32x4*)(fs + 4);
      if (++fp < np) { fh++; const bool turn = fh == group; fs += turn ? to_row : HD; fh = turn ? 0 : fh; }      // (past the end: the last pair again)
    }
  };
  fetch();
  int pos = a.pos0 + row_first, ph = 0;                                    // the next pair's position, head in its group
  int or_ = row_first + wave / group, oh = wave % group;                   // row, head in its group of the pair whose partials this wave folds; four pairs further: + (4 / group, 4 % group)
  const int or4 = 4 / group, oh4 = 4 % group;
  for (int b = 0; b < np; b += 4) {
    f32x4 q0[4], q1[4];
#pragma unroll
    for (int hh = 0; hh < 4; hh++) { q0[hh] = qa[hh]; q1[hh] = qb[hh]; }
    fetch();
#pragma unroll
    for (int hh = 0; hh < 4; hh++) {                                       // (pairs past the end repeat the last one, nothing reads their sums: without a branch per pair the steps of one run beside those of the next)
      const float qq[8] = {q0[hh].x, q0[hh].y, q0[hh].z, q0[hh].w, q1[hh].x, q1[hh].y, q1[hh].z, q1[hh].w};
      float sc[NVI];
      float m = -INFINITY;
#pragma unroll
      for (int i = 0; i < NVI; i++) {
        const u32x4 kk = kt[i];
        const half2_t k0 = as_h2(kk.x), k1 = as_h2(kk.y), k2 = as_h2(kk.z), k3 = as_h2(kk.w);
        float t = qq[0] * (float)k0.x; t += qq[1] * (float)k0.y; t += qq[2] * (float)k1.x; t += qq[3] * (float)k1.y;
        t += qq[4] * (float)k2.x; t += qq[5] * (float)k2.y; t += qq[6] * (float)k3.x; t += qq[7] * (float)k3.y;
        t = x16_run_sum<HD8>(t);
        sc[i] = (p0 + i * RPI + vr <= pos) ? t * a.scale : -INFINITY;
        m = fmaxf(m, sc[i]);
      }
      float l = 0.f;
      f32x4 o0 = {0.f, 0.f, 0.f, 0.f}, o1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < NVI; i++) {
        const float pj = (p0 + i * RPI + vr <= pos) ? __expf(sc[i] - m) : 0.f;
        l += pj;
        u32x4 vv = vt[i];
        if (p0 + i * RPI + vr > pos) vv = u32x4{0u, 0u, 0u, 0u};         // (a later position's: 0 times a value that is not finite would reach this row)
        const half2_t v0 = as_h2(vv.x), v1 = as_h2(vv.y), v2 = as_h2(vv.z), v3 = as_h2(vv.w);
        o0.x += pj * (float)v0.x; o0.y += pj * (float)v0.y; o0.z += pj * (float)v1.x; o0.w += pj * (float)v1.y;
        o1.x += pj * (float)v2.x; o1.y += pj * (float)v2.y; o1.z += pj * (float)v3.x; o1.w += pj * (float)v3.y;
      }
      float* cw = comb + (size_t)(hh * NGRP + wave * RPI + vr) * CSTR;
      *(f32x4*)(cw + vp * 8) = o0; *(f32x4*)(cw + vp * 8 + 4) = o1;
      if (vp == 0) { cw[HD] = m; cw[HD + 1] = l; }
      if (++ph == group) { ph = 0; pos++; }
    }
    __syncthreads();
    if (b + wave < np) {
      const int row = or_, head = kvh * group + oh;
      const float* cb = comb + (size_t)wave * NGRP * CSTR;
      float m = -INFINITY;
#pragma unroll
      for (int g = 0; g < NGRP; g++) m = fmaxf(m, cb[g * CSTR + HD]);
      float l = 0.f, od[HD / 64];
#pragma unroll
      for (int j = 0; j < HD / 64; j++) od[j] = 0.f;
#pragma unroll
      for (int g = 0; g < NGRP; g++) {
        const float mg = cb[g * CSTR + HD];
        const float wg = mg == -INFINITY ? 0.f : __expf(mg - m);
        l += wg * cb[g * CSTR + HD + 1];
#pragma unroll
        for (int j = 0; j < HD / 64; j++) od[j] += wg * cb[g * CSTR + lane + 64 * j];
      }
      float* po = a.part + (((size_t)row * a.H + head) * a.nsplit + split) * (HD + 2);
#pragma unroll
      for (int j = 0; j < HD / 64; j++) po[lane + 64 * j] = od[j];
      if (lane == 0) { po[HD] = m; po[HD + 1] = l; }
    }
    or_ += or4; oh += oh4;
    if (oh >= group) { oh -= group; or_++; }
    __syncthreads();
  }
}

// The partials of a (row, head) merged as attn_merge_kernel does (at most HD splits)
template <int HD>
__global__ __launch_bounds__(HD) void x16_merge_kernel(const X16Attn a) {
  constexpr int FB = 24, NB = 16;
  const int head = blockIdx.x, row = blockIdx.y, d = threadIdx.x;
  __shared__ float sw[HD];
  __shared__ float red[2 * (HD / 64)];
  const float* ph = a.part + ((size_t)row * a.H + head) * a.nsplit * (HD + 2);
  const int ns = ((a.pos0 + row) >> 6) + 1;                                // (at most nsplit)
  const int spc = d < ns ? d : ns - 1;
  const float mv = ph[(size_t)spc * (HD + 2) + HD], lv = ph[(size_t)spc * (HD + 2) + HD + 1];
  float v[FB];
#pragma unroll
  for (int j = 0; j < FB; j++) v[j] = ph[(size_t)(j < ns ? j : ns - 1) * (HD + 2) + d];
  float m = wave_max(d < ns ? mv : -INFINITY), l = 0.f;
  if constexpr (HD > 64) {
    if ((d & 63) == 0) red[d >> 6] = m;
    __syncthreads();
    m = red[0];
#pragma unroll
    for (int i = 1; i < HD / 64; i++) m = fmaxf(m, red[i]);
  }
  const float e = d < ns ? __expf(mv - m) : 0.f;
  if (d < ns) sw[d] = e;
  l = d < ns ? lv * e : 0.f;
  l = wave_sum(l);
  if constexpr (HD > 64) {
    if ((d & 63) == 0) red[HD / 64 + (d >> 6)] = l;
    __syncthreads();
    l = 0.f;
#pragma unroll
    for (int i = 0; i < HD / 64; i++) l += red[HD / 64 + i];
  } else __syncthreads();
  float o = 0.f;
#pragma unroll
  for (int j = 0; j < FB; j++) o += j < ns ? v[j] * sw[j] : 0.f;
  for (int s0 = FB; s0 < ns; s0 += NB) {
    float w[NB];
#pragma unroll
    for (int j = 0; j < NB; j++) w[j] = ph[(size_t)min(s0 + j, ns - 1) * (HD + 2) + d];
#pragma unroll
    for (int j = 0; j < NB; j++) o += s0 + j < ns ? w[j] * sw[s0 + j] : 0.f;
  }
  o *= 1.0f / l;
  asm volatile("" : "+v"(o));                                             // (a float32 value before it is rounded to fp16, as there)
  a.out[((size_t)row * a.H + head) * HD + d] = (uint16_t)f2h_bits(o);
}

// ------------------------------------------------------------------------------------------------ ffn_norm and router logits
// The arithmetic of moe_router_kernel, RT rows per workgroup: normalised once, the router's rows read once for all of them.  The normalised rows leave as the experts read them: the sixteen pairs
// (value j, value j + 16) of a unit of 32 behind each other, those of j = g, g + 4, g + 8, g + 12 as a piece of sixteen bytes.
struct X16Router { const float* x; const float* nw; const uint16_t* wr; uint16_t* xs; float* logits; int R, dim, E; float eps; };
// Bound by the latency of the router's rows, which come from the L2s: sixteen waves share them, four of which form the norm (512 rows, 64 experts of 2048 values: 17.6 -> 9.1 us with sixteen waves instead of four).
template <int RT>
__global__ __launch_bounds__(1024) void x16_router_kernel(const X16Router a) {
  __shared__ __attribute__((aligned(16))) uint16_t xn[RT][2048];
  __shared__ float red[RT][4];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), np = a.dim >> 3, r0 = blockIdx.x * RT;
  const bool have = tid < np;                                              // (dim <= 2048: a piece of 8 values per thread of the first four waves)
  const int p = have ? tid : np - 1;
  f32x4 xa[RT][2];
#pragma unroll
  for (int t = 0; t < RT; t++) { const float* x = a.x + (size_t)min(r0 + t, a.R - 1) * a.dim; xa[t][0] = ((const f32x4*)x)[2 * p]; xa[t][1] = ((const f32x4*)x)[2 * p + 1]; }
  const f32x4 w0 = ((const f32x4*)a.nw)[2 * p], w1 = ((const f32x4*)a.nw)[2 * p + 1];
#pragma unroll
  for (int t = 0; t < RT; t++) {
    float s = 0.f;
    if (have) {
#pragma unroll
      for (int h = 0; h < 2; h++) s += xa[t][h].x * xa[t][h].x + xa[t][h].y * xa[t][h].y + xa[t][h].z * xa[t][h].z + xa[t][h].w * xa[t][h].w;
    }
    if (wave < 4) { s = wave_sum(s); if (lane == 0) red[t][wave] = s; }
  }
  __syncthreads();
#pragma unroll
  for (int t = 0; t < RT; t++) {
    const float nscale = 1.0f / sqrtf((red[t][0] + red[t][1] + red[t][2] + red[t][3]) / (float)a.dim + a.eps);
    if (have) {
      float v[8] = {xa[t][0].x, xa[t][0].y, xa[t][0].z, xa[t][0].w, xa[t][1].x, xa[t][1].y, xa[t][1].z, xa[t][1].w};
      const float w[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
#pragma unroll
      for (int i = 0; i < 8; i++) { v[i] = (v[i] * nscale) * w[i]; asm volatile("" : "+v"(v[i])); }      // (a float32 value before it is rounded to fp16, as there: one instruction would round once)
      *(u32x4*)(&xn[t][8 * p]) = u32x4{f2h_bits(v[0]) | (f2h_bits(v[1]) << 16), f2h_bits(v[2]) | (f2h_bits(v[3]) << 16), f2h_bits(v[4]) | (f2h_bits(v[5]) << 16), f2h_bits(v[6]) | (f2h_bits(v[7]) << 16)};
    }
  }
  __syncthreads();
#pragma unroll
  for (int t = 0; t < RT; t++)
    if (r0 + t < a.R)
      for (int d = tid; d < (a.dim >> 1); d += 1024) {
        const int e = 32 * (d >> 4) + 4 * (d & 3) + ((d >> 2) & 3);
        const uint32_t lo = xn[t][e], hi = xn[t][e + 16];
        ((uint32_t*)(a.xs + (size_t)(r0 + t) * a.dim))[d] = lo | (hi << 16);
      }
  for (int e = wave; e < a.E; e += 16) {
    const uint16_t* wrow = a.wr + (size_t)e * a.dim;
    u32x4 wv[4];
#pragma unroll
    for (int j = 0; j < 4; j++) { const int q = lane + 64 * j; wv[j] = *(const u32x4*)(wrow + 8 * (q < np ? q : np - 1)); }
#pragma unroll
    for (int t = 0; t < RT; t++) {
      float acc = 0.f;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int q = lane + 64 * j;
        if (q < np) { const u32x4 xv = *(const u32x4*)(&xn[t][8 * q]); acc = dot2(wv[j].w, xv.w, dot2(wv[j].z, xv.z, dot2(wv[j].y, xv.y, dot2(wv[j].x, xv.x, acc)))); }
      }
      acc = wave_sum(acc);
      if (lane == 0 && r0 + t < a.R) a.logits[(size_t)(r0 + t) * a.E + e] = acc;
    }
  }
}

// ------------------------------------------------------------------------------------------------ the experts
// An expert's MXFP4 weights against the rows of all its assignments, each result with the bits of the expert GEMV (qgemv1.h): per unit of 32 weights a chain of sixteen dot2 from zero, times the
// block's scale, then the tree over the units (pairs of neighbours first).  v_dot2_f32_f16 rounds the sum of two products and the addend once, and so does a matrix-core product whose other products
// are zeros: v_mfma_f32_16x16x4_4b_f16 with two of its four values zero is 1024 dot2 in 32 cycles where the vector unit takes 93 (16 instructions, 5.8 cycles each in a loop of nothing else; bits compared over
// normal, subnormal and huge values, sums from zero and not; with all four values in use they differ, so the matrix cores run at an eighth of their fp16 rate here).
// An item is 64 weight rows of one expert (SwiGLU: 32 of gate and the same 32 of up) and all of the expert's rows, in tiles of sixteen.  Workgroups stay for the whole launch and share the tiles of all
// items evenly, each a contiguous run of them (an item may be cut); wave w holds units 8 w .. of the item's weight rows in registers, so weights are read once per item, and touches those of the next item at
// the first tile of this one (they wait in the XCD's L2; a second set of registers does not fit).  Lane 16 b + c supplies column c of block b; the sixteen rows of the tile are the other operand, the same for the four blocks, brought to LDS by requests of the wave itself,
// two runs of four units ahead, across items.  The waves' partial sums meet in LDS, where the upper levels of the tree are formed.
// The zeros sit in the weight operand (the pair beside a weight pair), so where a row holds an infinity its results are NaN, which the expert GEMV's are from the first zero weight on: of 2048 values
// and more, behind the next norm the whole row is NaN either way.
#define X16_RUN 4096                     // bytes of LDS for four units of a tile's sixteen rows
struct X16Expert { const uint8_t* w[2]; const uint16_t* x; void* y; const int* off; const int2* tiles; const int* n_tiles; long long estride, row_bytes; int K, N, ngroups; };

// (units as calls with constants: a loop is unrolled too late for its arrays to become registers)
template <class F, int... I> __device__ __forceinline__ void x16_each(F& f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }

// NS: subtrees of eight units, the waves of a workgroup at most (a tree of 32 or 64 leaves)
template <bool SW, int NS>
__global__ __launch_bounds__(64 * NS, 2) void x16_expert_kernel(const X16Expert a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t ring[];           // [wave][3 runs][16 rows of 256 bytes]
  __shared__ float part[NS][16][64];
  __shared__ uint32_t touched[NS][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), blk = lane >> 4, c = lane & 15;
  const int nw = blockDim.x >> 6;                                          // (K = 256 nw)
  const int ntiles = *a.n_tiles;
  // this workgroup's tiles: of the sequence (expert, item, tile) those from s0 on, neighbouring runs on one XCD
  const long long total = (long long)ntiles * a.ngroups;
  const unsigned nwg = gridDim.x, turn = (blockIdx.x & 7) * (nwg >> 3) + (blockIdx.x >> 3);      // (nwg is a multiple of 8)
  const int s0 = (int)(total * turn / nwg);
  int left = (int)(total * (turn + 1) / nwg) - s0;
  if (left <= 0) return;
  struct Item { int e, grp, tf, nt, first, cnt; };                         // tf: the expert's first tile in the list
  auto expert_at = [&](int tile, Item& it) __attribute__((always_inline)) {
    it.e = a.tiles[tile].x; it.tf = tile - (a.tiles[tile].y >> 4); it.first = a.off[it.e]; it.cnt = a.off[it.e + 1] - it.first; it.nt = (it.cnt + 15) >> 4;
  };
  auto item_behind = [&](const Item& it) __attribute__((always_inline)) {
    Item n = it;
    if (it.grp + 1 < a.ngroups) n.grp = it.grp + 1;
    else if (it.tf + it.nt < ntiles) { expert_at(it.tf + it.nt, n); n.grp = 0; }
    return n;                                                              // (behind the last: the last again)
  };
  Item it, nx;
  expert_at(s0 / a.ngroups, it);
  int t = s0 - it.tf * a.ngroups;
  it.grp = t / it.nt; t -= it.grp * it.nt;
  nx = item_behind(it);
  // this wave's eight units of the item's 64 columns: cw[u][t] holds, of column c of block t, the bytes g, g + 4, g + 8, g + 12 (g = blk) of unit u's sixteen - the weights of the four products that this
  // lane's group of a matrix product takes -; sc the scale bytes of this lane's own column
  uint32_t cw[8][4], sc[2];
  auto weights_of = [&](const Item& i) __attribute__((always_inline)) {
    const int col = SW ? i.grp * 32 + (blk & 1) * 16 + c : i.grp * 64 + lane;
    return (SW && blk >= 2 ? a.w[1] : a.w[0]) + i.e * a.estride + (long long)col * a.row_bytes + 136 * wave;      // (4-byte aligned: K is a multiple of 256)
  };
  auto load = [&](const Item& i) __attribute__((always_inline)) {
    const uint8_t* p = weights_of(i);
    uint32_t raw[34];
#pragma unroll
    for (int q = 0; q < 8; q++) { const u32x4 v = ld16(p + 16 * q); raw[4 * q] = v.x; raw[4 * q + 1] = v.y; raw[4 * q + 2] = v.z; raw[4 * q + 3] = v.w; }
    u32x2 v; __builtin_memcpy(&v, p + 128, 8); raw[32] = v.x; raw[33] = v.y;
    __builtin_amdgcn_s_waitcnt(0x0f70);                                    // (vmcnt 0: what is counted behind it are requests into LDS and stores)
    // a lane's own column, bytes transposed within the unit, then across the four lanes that share c
    sc[0] = sc[1] = 0;
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const int o = 17 * u;
      sc[u >> 2] |= ((raw[o >> 2] >> (8 * (o & 3))) & 0xffu) << (8 * (u & 3));
      uint32_t d[4];
#pragma unroll
      for (int q = 0; q < 4; q++) { const int at = o + 1 + 4 * q; d[q] = (at & 3) ? __builtin_amdgcn_alignbit(raw[(at >> 2) + 1], raw[at >> 2], 8 * (at & 3)) : raw[at >> 2]; }
      const uint32_t e0 = __builtin_amdgcn_perm(d[1], d[0], 0x05010400u), e1 = __builtin_amdgcn_perm(d[1], d[0], 0x07030602u), e2 = __builtin_amdgcn_perm(d[3], d[2], 0x05010400u), e3 = __builtin_amdgcn_perm(d[3], d[2], 0x07030602u);
      const uint32_t t0 = __builtin_amdgcn_perm(e2, e0, 0x05040100u), t1 = __builtin_amdgcn_perm(e2, e0, 0x07060302u), t2 = __builtin_amdgcn_perm(e3, e1, 0x05040100u), t3 = __builtin_amdgcn_perm(e3, e1, 0x07060302u);
      const auto h02 = __builtin_amdgcn_permlane32_swap(t0, t2, false, false), h13 = __builtin_amdgcn_permlane32_swap(t1, t3, false, false);
      const auto a01 = __builtin_amdgcn_permlane16_swap(h02[0], h13[0], false, false), a23 = __builtin_amdgcn_permlane16_swap(h02[1], h13[1], false, false);
      cw[u][0] = a01[0]; cw[u][1] = a01[1]; cw[u][2] = a23[0]; cw[u][3] = a23[1];
    }
  };
  load(it);
  uint8_t* rw = ring + wave * (3 * X16_RUN);
  for (int w = nw + wave; w < NS; w += nw) {                               // (units beyond the row are zeros of the tree)
#pragma unroll
    for (int i = 0; i < 16; i++) part[w][i][lane] = 0.f;
  }
  // a wave's request: its values of four units, 256 bytes of each of the tile's sixteen rows, four rows per instruction, pieces of 16 bytes XORed with the row
  uint32_t src[4];
  auto point = [&](const Item& i, int tile) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < 4; q++) src[q] = (uint32_t)(i.first + min(16 * tile + 4 * q + blk, i.cnt - 1)) * (uint32_t)(2 * a.K) + 512 * wave + (((c ^ blk) ^ (4 * q)) << 4);
  };
  auto request = [&](int half, int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < 4; q++)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)((const char*)a.x + (src[q] + 256 * half)), (__attribute__((address_space(3))) void*)(rw + slot * X16_RUN + q * 1024), 16, 0, 0);
  };
  point(it, t);
  request(0, 0); request(1, 1);
  u32x4 x[2];
  auto read_x = [&](u32x4& d, int slot, int u) __attribute__((always_inline)) {
    d = *(const u32x4*)(ring + (((uint32_t)(wave * 3 + slot) * X16_RUN + c * 272) ^ (64 * u + 16 * blk)));      // (c * 256 + 16 c: the low eight bits are the row's)
  };
  asm volatile("s_waitcnt vmcnt(4)" ::: "memory");                        // run 0 has landed
  read_x(x[0], 0, 0);
  // weight operands with their zeros in place: pair i of a lane's four, for two blocks
  u32x4 wz[2][4];
#pragma unroll
  for (int z = 0; z < 2; z++)
#pragma unroll
    for (int i = 0; i < 4; i++) { wz[z][i] = u32x4{0u, 0u, 0u, 0u}; asm volatile("" : "+v"(wz[z][i])); }
  int slot = 0;
  bool fresh = true;                                                       // the first tile on these weights: the next item's are touched
  for (;;) {
    const bool same = t + 1 < it.nt;
    float st[3][16], leaf[16];                                             // sums of 1, 2 and 4 units that wait for their neighbour
    auto unit = [&](auto u_) __attribute__((always_inline)) {
      constexpr int u = decltype(u_)::value;
      const int nslot = slot == 2 ? 0 : slot + 1;
      if constexpr (u == 0) { if (same) point(it, t + 1); else point(nx, 0); }
      if constexpr (u % 4 == 0) request(u / 4, slot == 0 ? 2 : slot - 1);  // (the run after the next one goes where the one before this was read from)
      if constexpr (u == 0) {
        if (fresh) {                                                       // both ends of the lane's run, into LDS that nobody reads
          const uint8_t* p = weights_of(nx);
#pragma unroll
          for (int z = 0; z < 2; z++) __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(p + 132 * z), (__attribute__((address_space(3))) void*)touched[wave], 4, 0, 0);
        }
      }
      if constexpr (u % 4 == 3) {
        // the next run has landed; behind it the run requested last and, at a first tile, the two touches may be on their way
        if (fresh) asm volatile("s_waitcnt vmcnt(6)" ::: "memory"); else asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
        read_x(x[(u + 1) & 1], nslot, 0);
      } else read_x(x[(u + 1) & 1], slot, (u & 3) + 1);
#pragma unroll
      for (int i = 0; i < 4; i++) asm volatile("" : "+v"(cw[u][i]));       // (decoded here and anew for every tile: decoded ahead, they do not fit the registers)
      asm volatile("" : "+v"(sc[u >> 2]));
      const uint32_t eb = (sc[u >> 2] >> (8 * (u & 3))) & 0xffu;
      const uint32_t s02 = eb ? (eb << 23) : 0x00400000u;
      v4f32 acc[4];
#pragma unroll
      for (int b = 0; b < 4; b++) acc[b] = v4f32{0.f, 0.f, 0.f, 0.f};
      auto product = [&](auto i_) __attribute__((always_inline)) {         // four dot2 of every chain: those of pairs 4 i .. 4 i + 3
        constexpr int i = decltype(i_)::value;
#pragma unroll
        for (int b = 0; b < 4; b++) {
          wz[b & 1][i][i] = as_u32(__builtin_amdgcn_cvt_scalef32_pk_f16_fp4(cw[u][b], 1.0f, i));
          acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8f16, x[u & 1]), __builtin_bit_cast(v8f16, wz[b & 1][i]), acc[b], 0, 0, 0);
          asm volatile("" : "+v"(wz[b & 1][i]));                           // (its other pairs are no constants to the compiler, which set them anew for every product)
        }
      };
      x16_each(product, std::make_integer_sequence<int, 4>{});
      // the scales of the four blocks' column c
      const auto h = __builtin_amdgcn_permlane32_swap(s02, s02, false, false);
      const auto l0 = __builtin_amdgcn_permlane16_swap(h[0], h[0], false, false), l1 = __builtin_amdgcn_permlane16_swap(h[1], h[1], false, false);
      const uint32_t su[4] = {l0[0], l0[1], l1[0], l1[1]};                // (a bit cast of an element of such a pair takes the first)
      const float sb[4] = {__builtin_bit_cast(float, su[0]), __builtin_bit_cast(float, su[1]), __builtin_bit_cast(float, su[2]), __builtin_bit_cast(float, su[3])};
#pragma unroll
      for (int i = 0; i < 16; i++) {
        float v = __builtin_fmaf(sb[i >> 2], acc[i >> 2][i & 3], 0.f);
        if constexpr (u & 1) { v = st[0][i] + v; if constexpr (u & 2) { v = st[1][i] + v; if constexpr (u & 4) leaf[i] = st[2][i] + v; else st[2][i] = v; } else st[1][i] = v; }
        else st[0][i] = v;
      }
      if constexpr (u % 4 == 3) slot = nslot;
    };
    x16_each(unit, std::make_integer_sequence<int, 8>{});
    // (barriers of their own: __syncthreads would wait for the requests in flight)
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");         // everyone has summed the tile before
#pragma unroll
    for (int i = 0; i < 16; i++) part[wave][i][lane] = leaf[i];
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    // register 4 b + i of lane l is row 4 (l / 16) + i of column l % 16 of block b
    for (int o = tid; o < 512; o += blockDim.x) {
      const int l = o & 63, h = (o >> 6) & 1, i = o >> 7, row = 16 * t + 4 * (l >> 4) + i, cc = l & 15;
      if (row >= it.cnt) continue;
      float s[2];
#pragma unroll
      for (int z = 0; z < 2; z++) {
        const int rg = 4 * (h + 2 * z) + i;
        s[z] = (part[0][rg][l] + part[1][rg][l]) + (part[2][rg][l] + part[3][rg][l]);
        if constexpr (NS == 8) s[z] += (part[4][rg][l] + part[5][rg][l]) + (part[6][rg][l] + part[7][rg][l]);
      }
      if constexpr (SW) {
        float v = silu_f(s[0]) * s[1];
        asm volatile("" : "+v"(v));                                       // (rounded to float32 first, as there)
        ((uint16_t*)a.y)[(size_t)(it.first + row) * a.N + it.grp * 32 + 8 * (cc & 3) + 2 * (cc >> 2) + h] = (uint16_t)f2h_bits(v);
      } else {
        float* y = (float*)a.y + (size_t)(it.first + row) * a.N + it.grp * 64 + cc;
        y[16 * h] = s[0]; y[16 * (h + 2)] = s[1];
      }
    }
    if (--left == 0) break;
    if (same) { t++; fresh = false; continue; }
    t = 0; fresh = true; it = nx; nx = item_behind(it);
    load(it);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                        // (the last requests are read by nobody: they have arrived before the workgroup's LDS is given to another)
}

// Offsets of the experts' rows, the list of their tiles of sixteen (the first workgroup), and the normalised rows in the order of the experts' rows: two rows a workgroup, each read once, while the counts
// are scanned, and written for each of its experts (a launch for the lists and one that read a row for each of its experts, 508 rows, top 8: 4.7 + 5.9 us)
__global__ __launch_bounds__(512) void x16_group_kernel(const int* __restrict__ counts, const int* __restrict__ sel, const int* __restrict__ place, const uint16_t* __restrict__ xs, int R, int E, int k, int dim,
                                                        int* __restrict__ off, int2* __restrict__ tiles, int* __restrict__ n_tiles, uint16_t* __restrict__ xe) {
  __shared__ int s_off[512], s_row[128], s_t[8], s_o[8];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, half = tid >> 8, p = tid & 255, t = blockIdx.x * 2 + half, np = dim >> 3;
  const u32x4 v = *(const u32x4*)(xs + (size_t)min(t, R - 1) * dim + 8 * min(p, np - 1));
  const int j = blockIdx.x * 2 * k + tid;                                  // (an assignment per thread: k <= 64)
  const bool mine = tid < 2 * k && j < R * k;
  const int se = mine ? sel[j] : 0, at = mine ? place[j] : 0;
  const int c = tid < E ? counts[tid] : 0, nt = (c + 15) >> 4;
  int io = c, it = nt;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) { const int uo = __shfl_up(io, o), ut = __shfl_up(it, o); if (lane >= o) { io += uo; it += ut; } }
  if (lane == 63) { s_o[wave] = io; s_t[wave] = it; }
  __syncthreads();
  for (int w = 0; w < wave; w++) { io += s_o[w]; it += s_t[w]; }
  s_off[tid] = io - c;
  __syncthreads();
  if (mine) s_row[tid] = s_off[se] + at;
  __syncthreads();
  if (t < R && p < np) for (int i = 0; i < k; i++) *(u32x4*)(xe + (size_t)s_row[half * k + i] * dim + 8 * p) = v;
  if (blockIdx.x == 0 && tid < E) {
    off[tid] = io - c;
    for (int i = 0; i < nt; i++) tiles[it - nt + i] = int2{tid, 16 * i};
    if (tid == E - 1) { off[E] = io; *n_tiles = it; }
  }
}

// The weighted sum of a row's experts + residual and the norm behind it, as rmsnorm_kernel<true> (rows of at most 2048 values), over results in the order of the experts' rows
__global__ __launch_bounds__(1024) void x16_combine_kernel(float* __restrict__ x, const float* __restrict__ y, const float* __restrict__ probs, const int* __restrict__ sel, const int* __restrict__ place,
                                                           const int* __restrict__ off, const float* __restrict__ w, int k, int dim, float eps, uint16_t* __restrict__ out) {
  __shared__ float red[16];
  __shared__ float pp[64]; __shared__ int at[64];
  const int row = blockIdx.x, tid = threadIdx.x;
  if (tid < k) { pp[tid] = probs[(size_t)row * k + tid]; at[tid] = off[sel[(size_t)row * k + tid]] + place[(size_t)row * k + tid]; }
  __syncthreads();
  x += (size_t)row * dim; out += (size_t)row * dim;
  const int e0 = tid, e1 = tid + 1024;
  auto value = [&](int e) {
    float v = x[e];
    for (int j0 = 0; j0 < k; j0 += 8) {
      float yy[8];
#pragma unroll
      for (int i = 0; i < 8; i++) yy[i] = y[(size_t)at[j0 + i < k ? j0 + i : k - 1] * dim + e];
#pragma unroll
      for (int i = 0; i < 8; i++) if (j0 + i < k) v += pp[j0 + i] * yy[i];
    }
    x[e] = v;
    return v;
  };
  float v0 = 0.f, v1 = 0.f, w0 = 0.f, w1 = 0.f;
  if (e0 < dim) { v0 = value(e0); w0 = w[e0]; }
  if (e1 < dim) { v1 = value(e1); w1 = w[e1]; }
  float s = v0 * v0 + v1 * v1;
  s = wave_sum(s);
  if ((tid & 63) == 0) red[tid >> 6] = s;
  __syncthreads();
  float tot = 0.f;
  for (int i = 0; i < 16; i++) tot += red[i];
  const float scale = 1.0f / sqrtf(tot / (float)dim + eps);
  float o0 = (v0 * scale) * w0, o1 = (v1 * scale) * w1;
  asm volatile("" : "+v"(o0), "+v"(o1));
  if (e0 < dim) out[e0] = (uint16_t)f2h_bits(o0);
  if (e1 < dim) out[e1] = (uint16_t)f2h_bits(o1);
}

// ------------------------------------------------------------------------------------------------ the step
struct X16Ws { size_t x, xn, q, k, v, qr, attn, part, logits, sel, probs, place, counts, off, tiles, ntiles, xs, xe, act, y, total; };
static X16Ws x16_layout(const int64_t* m, int64_t R, int64_t nsplit) {
  X16Ws w = {}; size_t o = 0;
  auto take = [&](size_t n) { const size_t at = o; o += (n + 255) & ~(size_t)255; return at; };
  const int64_t dim = m[PM_DIM], nq = m[PM_HEADS] * m[PM_HD], nk = m[PM_KV] * m[PM_HD], E = m[PM_EXPERTS], k = m[PM_TOPK];
  w.x = take(R * dim * 4); w.xn = take(R * dim * 2); w.q = take(R * nq * 4); w.k = take(R * nk * 4); w.v = take(R * nk * 4); w.qr = take(R * nq * 4); w.attn = take(R * nq * 2);
  w.part = take(R * m[PM_HEADS] * nsplit * (m[PM_HD] + 2) * 4);
  w.logits = take(R * E * 4); w.sel = take(R * k * 4); w.probs = take(R * k * 4); w.place = take(R * k * 4); w.counts = take(E * 4); w.off = take((E + 1) * 4);
  w.tiles = take((R * k / 16 + E + 1) * 8); w.ntiles = take(4); w.xs = take(R * dim * 2); w.xe = take(R * k * dim * 2);
  w.act = take(R * k * m[PM_HIDDEN] * 2); w.y = take(R * k * dim * 4);
  w.total = o;
  return w;
}

// steps of 256 values go to eight waves in qgemm_wp.hip and qgemm_dma.hip (K a multiple of 1024), to four in qgemm.hip
static int x16_waves(int64_t K) { return K % 1024 == 0 ? 8 : 4; }
static bool x16_dense(int64_t type, int64_t w, int64_t n, int64_t K) { return type == GGML_F16 && w % 16 == 0 && n > 0 && n % 64 == 0 && K >= 512 && K <= 4096 && K % 256 == 0; }
static bool prefill16_ok(const int64_t* m, const int64_t* blocks) {
  const int64_t dim = m[PM_DIM], H = m[PM_HEADS], KV = m[PM_KV], hd = m[PM_HD], E = m[PM_EXPERTS], k = m[PM_TOPK], hid = m[PM_HIDDEN];
  if (!(hd == 64 || hd == 128) || KV <= 0 || H % KV || H * hd > 4096 || m[PM_QKNORM] != H * hd || m[PM_QKNORM] == hd || E < 1 || E > 512 || k < 1 || k > 64 || k > E || m[PM_GATING] < 1 || m[PM_GATING] > 4) return false;
  if (dim > 2048 || dim % 256 || hid > 2048 || hid % 256 || hid < 256 || (m[PM_MAXCTX] + 63) / 64 > hd) return false;
  for (int64_t i = 0; i < m[PM_NBLOCKS]; i++) {
    const int64_t* b = blocks + i * PB_COUNT;
    if (!b[PB_MOE] || !b[PB_QN] || !b[PB_KN] || b[PB_TGATE] != GGML_MXFP4 || b[PB_TDOWN] != GGML_MXFP4) return false;
    if (!x16_dense(b[PB_TQ], b[PB_WQ], H * hd, dim) || !x16_dense(b[PB_TK], b[PB_WK], KV * hd, dim) || !x16_dense(b[PB_TV], b[PB_WV], KV * hd, dim) || !x16_dense(b[PB_TO], b[PB_WO], dim, H * hd)) return false;
    if ((b[PB_GATE] | b[PB_UP] | b[PB_DOWN]) % 4 || (b[PB_ROUTER] | b[PB_ATTN_NORM] | b[PB_FFN_NORM] | b[PB_QN] | b[PB_KN] | b[PB_CK] | b[PB_CV]) % 16) return false;
  }
  return true;
}

static int x16_linear(int nseg, const int64_t* w, float* const* y, const int64_t* n, const uint16_t* x, int64_t M, int64_t K, const float* resid, hipStream_t s) {
  X16Gemm a = {};
  for (int i = 0; i < nseg; i++) { a.w[i] = (const uint16_t*)w[i]; a.y[i] = y[i]; a.n[i] = (int)n[i]; a.ntiles += (int)(n[i] / 64); }
  a.resid = resid; a.x = x; a.nseg = nseg; a.M = (int)M; a.K = (int)K; a.nw = x16_waves(K);
  x16_gemm_kernel<<<(unsigned)((a.ntiles + 7) / 8 * 8 * ((M + 63) / 64)), 256, 0, s>>>(a);
  TGA_LAUNCH_CHECK();
  return 0;
}

template <bool SW>
static int x16_experts(const X16Expert& e, int64_t K, int64_t N, hipStream_t s) {
  X16Expert a = e;
  a.row_bytes = K / 32 * 17; a.estride = a.row_bytes * N; a.K = (int)K; a.N = (int)N; a.ngroups = (int)(SW ? N / 32 : N / 64);
  // The tree has 64 leaves for rows of more than 32 units (qgemv1.h: a wave), else 32 (half a wave).  Two workgroups of four waves per CU or one of eight
  const int nw = (int)(K / 256), ns = nw > 4 ? 8 : 4;
  auto kern = ns == 4 ? x16_expert_kernel<SW, 4> : x16_expert_kernel<SW, 8>;
  static const hipError_t configured = [] {
    const hipError_t r = hipFuncSetAttribute((const void*)x16_expert_kernel<SW, 4>, hipFuncAttributeMaxDynamicSharedMemorySize, 4 * 3 * X16_RUN);
    return r != hipSuccess ? r : hipFuncSetAttribute((const void*)x16_expert_kernel<SW, 8>, hipFuncAttributeMaxDynamicSharedMemorySize, 8 * 3 * X16_RUN);
  }();
  TGA_HIP(configured);
  kern<<<ns == 4 ? 512 : 256, 64 * nw, nw * 3 * X16_RUN, s>>>(a);
  TGA_LAUNCH_CHECK();
  return 0;
}

// The last one to three positions of a prompt: rows with the bits of single steps, whose kernels these are, with a job per row - a weight matrix comes from HBM once for all of them - and without
// the last block's feed-forward, which nothing reads.  A block of three rows of the OLMoE architecture: q / k / v 12.9 us (9.1 for one row), appending 4.6, attention 5.4 (5.7), attn_output 8.2 (5.1),
// router 4, gate / up 19.1 (11.1), down 8.9 (5.2): 63 us against 119 in three steps.  A prompt and its first logits, 508 positions and 1 / 2 / 3 more, together / as single steps: 8000 / 8010, 8120 / 8650,
// 8290 / 9380 us; six blocks of D 1024: 1355 / 1405, 1378 / 1585, 1395 / 1800.
template <int T> int qgemv1_launch_format(QArgs a, hipStream_t s);       // qgemv1.h
#define X16_TAIL 3
struct X16TailWs { size_t x, x2, qkv, part, xn, logits, sel, probs, act, y, total; };
static X16TailWs x16_tail_layout(const int64_t* m, int64_t nsplit) {
  X16TailWs w = {}; size_t o = 0;
  auto take = [&](size_t n) { const size_t at = o; o += (X16_TAIL * n + 255) & ~(size_t)255; return at; };
  const int64_t dim = m[PM_DIM], H = m[PM_HEADS], KV = m[PM_KV], hd = m[PM_HD], k = m[PM_TOPK];
  w.x = take(dim * 4); w.x2 = take(dim * 4); w.qkv = take((H + 2 * KV) * hd * 4); w.part = take(H * (nsplit * hd + 16) * 4); w.xn = take(dim * 2);
  w.logits = take(m[PM_EXPERTS] * 4); w.sel = take(k * 4); w.probs = take(k * 4); w.act = take(k * m[PM_HIDDEN] * 2); w.y = take(k * dim * 4);
  w.total = o;
  return w;
}
// (a single step of such a model: the one-launch attention, its partials merged by attn_output, the weighted sum of at most eight experts completed by the next block's q / k / v)
static bool prefill16_tail_ok(const int64_t* m, const int64_t* blocks) {
  return prefill16_ok(m, blocks) && m[PM_TOPK] <= 8 && m[PM_HEADS] * m[PM_HD] >= 512 && attn_split_rows_splits((int)m[PM_MAXCTX]) > 0;
}

extern "C" {

int tga_prefill16_tail_plan(const int64_t* m, const int64_t* blocks, int* ok, int64_t* nbytes) {
  TGA_REQUIRE(m && blocks && ok && nbytes, "tga_prefill16_tail_plan: null pointer");
  *ok = prefill16_tail_ok(m, blocks);
  *nbytes = *ok ? (int64_t)x16_tail_layout(m, attn_split_rows_splits((int)m[PM_MAXCTX])).total : 0;
  return 0;
}

int tga_prefill16_tail(const int64_t* m, const int64_t* blocks, const int32_t* tokens, int64_t rows, int64_t pos0, void* workspace, void* state, void* stream) {
  TGA_REQUIRE(m && blocks && tokens && workspace && state && rows >= 1 && rows <= X16_TAIL && pos0 >= 0 && pos0 + rows <= m[PM_MAXCTX], "tga_prefill16_tail: null pointer, or rows beyond the cache or more than %d", X16_TAIL);
  TGA_REQUIRE(prefill16_tail_ok(m, blocks), "tga_prefill16_tail: a model outside the range (tga_prefill16_tail_plan says which are inside)");
  const int R = (int)rows, dim = (int)m[PM_DIM], H = (int)m[PM_HEADS], KV = (int)m[PM_KV], hd = (int)m[PM_HD], nq = H * hd, nk = KV * hd, E = (int)m[PM_EXPERTS], k = (int)m[PM_TOPK], hid = (int)m[PM_HIDDEN];
  const int nsplit = attn_split_rows_splits((int)m[PM_MAXCTX]);
  const X16TailWs w = x16_tail_layout(m, nsplit);
  uint8_t* ws = (uint8_t*)workspace;
  float* x = (float*)(ws + w.x); float* x_new = (float*)(ws + w.x2); float* qkv = (float*)(ws + w.qkv); float* part = (float*)(ws + w.part); float* logits = (float*)(ws + w.logits);
  float* probs = (float*)(ws + w.probs); float* y = (float*)(ws + w.y); int* sel = (int*)(ws + w.sel);
  void* xn = ws + w.xn; void* act = ws + w.act;
  hipStream_t s = (hipStream_t)stream;
  const float eps = bits_f(m[PM_EPS_BITS]);
  int rc;
#define PF_DO(call) do { if ((rc = (call))) return rc; } while (0)
  PF_DO(tga_embed_rows((const void*)m[PM_EMB], (int)m[PM_EMB_TYPE], dim, tokens, R, state, x, stream));
  QArgs j = {};                                                           // a job per row over one matrix: whatever sel holds, its experts lie 0 bytes apart
  j.sel = sel; j.xdiv = 1; j.xdiv_jobs = R; j.x_f32 = j.y_f32 = 1;
  for (int64_t bi = 0; bi < m[PM_NBLOCKS]; bi++) {
    const int64_t* b = blocks + bi * PB_COUNT;
    QArgs a = j;
    a.nseg = 3; a.K = dim; a.x = x; a.norm_w = (const float*)b[PB_ATTN_NORM]; a.norm_eps = eps; a.ystride = nq + 2 * nk; a.ntot = nq + 2 * nk;
    a.w[0] = (const uint8_t*)b[PB_WQ]; a.w[1] = (const uint8_t*)b[PB_WK]; a.w[2] = (const uint8_t*)b[PB_WV];
    a.y[0] = qkv; a.y[1] = qkv + nq; a.y[2] = qkv + nq + nk; a.n[0] = nq; a.n[1] = a.n[2] = nk;
    if (bi) { a.comb_y = y; a.comb_p = probs; a.comb_k = k; a.comb_x_out = x_new; }
    PF_DO(qgemv1_launch_format<GGML_F16>(a, s));
    if (bi) { float* t = x; x = x_new; x_new = t; }
    const bool last = bi + 1 == m[PM_NBLOCKS];
    PF_DO(attn_split_rows(qkv, qkv + nq, qkv + nq + nk, nq + 2 * nk, (const float*)b[PB_QN], (const float*)b[PB_KN], eps, (void*)b[PB_CK], (void*)b[PB_CV], part, R, (int)pos0, H, KV, hd, (int)m[PM_MAXCTX],
                          (const float*)m[PM_ROPE], last, s));
    if (last) break;
    a = j;
    a.nseg = 1; a.K = nq; a.x = part; a.epilogue = 1; a.attn_S = nsplit; a.attn_hd_log2 = hd == 64 ? 6 : 7; a.ystride = dim; a.ntot = dim;
    a.w[0] = (const uint8_t*)b[PB_WO]; a.y[0] = x; a.resid[0] = x; a.n[0] = dim;
    PF_DO(qgemv1_launch_format<GGML_F16>(a, s));
    PF_DO(tga_moe_router_rows(x, (const float*)b[PB_FFN_NORM], eps, (const void*)b[PB_ROUTER], R, dim, E, xn, logits, stream));
    PF_DO(tga_qlinear_experts_routed_rows(GGML_MXFP4, (const void*)b[PB_GATE], (const void*)b[PB_UP], E, logits, R, k, (int)m[PM_GATING], (int)m[PM_NORM_TOPK], bits_f(m[PM_SCALE_BITS]), sel, probs,
                                          xn, act, TGA_F16, hid, dim, stream));
    PF_DO(tga_qlinear_experts(GGML_MXFP4, (const void*)b[PB_DOWN], nullptr, E, sel, R * k, 1, act, TGA_F16, y, TGA_F32, dim, hid, stream));
  }
#undef PF_DO
  return 0;
}

int tga_prefill16_plan(const int64_t* m, const int64_t* blocks, int64_t rows, int64_t end, int* ok, int64_t* nbytes) {
  TGA_REQUIRE(m && blocks && ok && nbytes && rows >= 1 && end >= rows, "tga_prefill16_plan: null pointer or no rows");
  *ok = prefill16_ok(m, blocks);
  *nbytes = *ok ? (int64_t)x16_layout(m, rows, (end + 63) / 64).total : 0;
  return 0;
}

int tga_prefill16_step(const int64_t* m, const int64_t* blocks, const int32_t* tokens, int64_t P, int64_t tail, int64_t pos0, void* workspace, void* state, void* stream) {
  TGA_REQUIRE(m && blocks && tokens && workspace && state && P >= 1 && tail >= 0 && tail <= P && pos0 >= 0 && pos0 + P <= m[PM_MAXCTX], "tga_prefill16_step: null pointer or rows beyond the cache");
  TGA_REQUIRE(prefill16_ok(m, blocks), "tga_prefill16_step: a model outside the range (tga_prefill16_plan says which are inside)");
  const int64_t R = P, dim = m[PM_DIM], H = m[PM_HEADS], KV = m[PM_KV], hd = m[PM_HD], nq = H * hd, nk = KV * hd, E = m[PM_EXPERTS], k = m[PM_TOPK], hid = m[PM_HIDDEN], nsplit = (pos0 + P + 63) / 64;
  TGA_REQUIRE(R <= 4096 && R * k <= 65536, "tga_prefill16_step: %lld rows are more than a step takes", (long long)R);
  const X16Ws w = x16_layout(m, R, nsplit);
  uint8_t* ws = (uint8_t*)workspace;
  float* x = (float*)(ws + w.x); uint16_t* xn = (uint16_t*)(ws + w.xn); float* q = (float*)(ws + w.q); float* kk = (float*)(ws + w.k); float* v = (float*)(ws + w.v); uint16_t* attn = (uint16_t*)(ws + w.attn);
  float* logits = (float*)(ws + w.logits); float* probs = (float*)(ws + w.probs); float* ye = (float*)(ws + w.y); int* off = (int*)(ws + w.off);
  int* sel = (int*)(ws + w.sel); int* place = (int*)(ws + w.place); int2* tiles = (int2*)(ws + w.tiles); int* nt = (int*)(ws + w.ntiles);
  hipStream_t s = (hipStream_t)stream;
  const float eps = bits_f(m[PM_EPS_BITS]);
  int rc;
#define PF_DO(call) do { if ((rc = (call))) return rc; } while (0)
  PF_DO(tga_embed_rows((const void*)m[PM_EMB], (int)m[PM_EMB_TYPE], (int)dim, tokens, (int)R, state, x, stream));
  for (int64_t bi = 0; bi < m[PM_NBLOCKS]; bi++) {
    const int64_t* b = blocks + bi * PB_COUNT;
    const float* an = (const float*)b[PB_ATTN_NORM];
    if (bi) { x16_combine_kernel<<<(unsigned)R, 1024, 0, s>>>(x, ye, probs, sel, place, off, an, (int)k, (int)dim, eps, xn); TGA_LAUNCH_CHECK(); }
    else {
      const int64_t folded = dim % 1024 == 0 ? tail : 0;
      if (R > folded) PF_DO(tga_rmsnorm_rows(x, an, (int)(R - folded), (int)dim, eps, xn, nullptr, 0, stream));
      if (folded) { x16_fold_norm_kernel<<<(unsigned)folded, 1024, 0, s>>>(x + (R - folded) * dim, an, (int)dim, eps, xn + (R - folded) * dim); TGA_LAUNCH_CHECK(); }
    }
    { const int64_t wt[3] = {b[PB_WQ], b[PB_WK], b[PB_WV]}, n[3] = {nq, nk, nk}; float* const y[3] = {q, kk, v}; PF_DO(x16_linear(3, wt, y, n, xn, R, dim, nullptr, s)); }
    X16Rope ra;
    ra.q = q; ra.k = kk; ra.v = v; ra.qn = (const float*)b[PB_QN]; ra.kn = (const float*)b[PB_KN]; ra.rope = (const float*)m[PM_ROPE]; ra.qr = (float*)(ws + w.qr); ra.ck = (uint16_t*)b[PB_CK]; ra.cv = (uint16_t*)b[PB_CV];
    ra.zero = (int*)(ws + w.counts); ra.n_zero = (int)E; ra.H = (int)H; ra.KV = (int)KV; ra.hd = (int)hd; ra.max_ctx = (int)m[PM_MAXCTX]; ra.pos0 = (int)pos0; ra.eps = eps;
    x16_rope_kernel<<<(unsigned)R, 512, 0, s>>>(ra);
    TGA_LAUNCH_CHECK();
    if (bi + 1 == m[PM_NBLOCKS]) break;                                   // the last block's keys and values are in the cache; what follows them there is read by nobody
    X16Attn aa;
    aa.qr = ra.qr; aa.ck = ra.ck; aa.cv = ra.cv; aa.part = (float*)(ws + w.part); aa.out = attn; aa.H = (int)H; aa.KV = (int)KV; aa.max_ctx = ra.max_ctx; aa.P = (int)P; aa.pos0 = (int)pos0; aa.nsplit = (int)nsplit;
    aa.scale = 1.0f / sqrtf((float)hd);
    const dim3 ag((unsigned)KV, (unsigned)nsplit, (unsigned)((P + X16_ROWS - 1) / X16_ROWS)), mg((unsigned)H, (unsigned)R);
    if (hd == 64) x16_attn_kernel<8><<<ag, 256, 0, s>>>(aa); else x16_attn_kernel<16><<<ag, 256, 0, s>>>(aa);
    TGA_LAUNCH_CHECK();
    if (hd == 64) x16_merge_kernel<64><<<mg, 64, 0, s>>>(aa); else x16_merge_kernel<128><<<mg, 128, 0, s>>>(aa);
    TGA_LAUNCH_CHECK();
    { const int64_t wt[1] = {b[PB_WO]}, n[1] = {dim}; float* const y[1] = {x}; PF_DO(x16_linear(1, wt, y, n, attn, R, nq, x, s)); }
    X16Router rt;
    rt.x = x; rt.nw = (const float*)b[PB_FFN_NORM]; rt.wr = (const uint16_t*)b[PB_ROUTER]; rt.xs = (uint16_t*)(ws + w.xs); rt.logits = logits; rt.R = (int)R; rt.dim = (int)dim; rt.E = (int)E; rt.eps = eps;
    x16_router_kernel<2><<<(unsigned)((R + 1) / 2), 1024, 0, s>>>(rt);
    TGA_LAUNCH_CHECK();
    PF_DO(pf_gate(logits, (int)R, (int)E, (int)k, (int)m[PM_GATING], (int)m[PM_NORM_TOPK], bits_f(m[PM_SCALE_BITS]), sel, probs, (int*)(ws + w.counts), place, s));
    uint16_t* xe = (uint16_t*)(ws + w.xe);
    x16_group_kernel<<<(unsigned)((R + 1) / 2), 512, 0, s>>>((const int*)(ws + w.counts), sel, place, rt.xs, (int)R, (int)E, (int)k, (int)dim, off, tiles, nt, xe);
    TGA_LAUNCH_CHECK();
    X16Expert ea = {};
    ea.off = off; ea.tiles = tiles; ea.n_tiles = nt;
    ea.w[0] = (const uint8_t*)b[PB_GATE]; ea.w[1] = (const uint8_t*)b[PB_UP]; ea.x = xe; ea.y = ws + w.act;
    PF_DO(x16_experts<true>(ea, dim, hid, s));
    ea.w[0] = (const uint8_t*)b[PB_DOWN]; ea.w[1] = nullptr; ea.x = (const uint16_t*)(ws + w.act); ea.y = ye;
    PF_DO(x16_experts<false>(ea, hid, dim, s));
  }
#undef PF_DO
  return 0;
}

}  // extern "C"
