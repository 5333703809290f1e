// Many activation rows against GGUF blocks on the matrix cores: y = x . W^T for the rows of a prefill step of any length, of several sequences, or of the tokens routed to
// each expert (tinygrad/llm/model.py:464, 476-481, 21-27: T > 1 calls of the same linears over the lazily dequantized weight).  Kernel template; the per-format
// instantiations are in qgemm_rows_*.hip, the entry points in qgemm_rows.hip.
//
// A workgroup of four waves owns 128 weight rows x TT activation rows (128, 64 or 32) and walks K in steps of 128.  Per step every thread decodes ONE unit of 64 weights
// into fp16 - (pattern - bias) * scale with one rounding, the reference's own fp16 weight cast (model.py:376) - and copies its share of the activation rows; both
// operands go through LDS as plain [row][64 values] lines whose 16-byte pieces are XORed with the row and the unit (conflict-free for the writers and
// for the readers, 16 rows of one piece), and 64 v_mfma_f32_16x16x32_f16 per wave (TT = 128) follow.  One LDS stage of 64 KB and two barriers per step: TWO workgroups share
// a CU, one decodes and writes while the other multiplies, which two stages in one workgroup of eight waves would have to be scheduled into.  The loads of the next
// step are issued before the multiplication and are consumed behind it.
// The decoded unit is put into natural order (pairs picked from the format's decode order with at most one v_perm_b32 each), so the activations are plain fp16 rows for
// every format and nothing is staged by a launch of its own.
#pragma once
#include "qfmt.h"
#include "qfmt_cb.h"

typedef _Float16 v8f16 __attribute__((ext_vector_type(8)));
typedef float v4f32 __attribute__((ext_vector_type(4)));

#define ROWS_WT 128               // weight rows of a workgroup
#define ROWS_KS 128               // K step

enum { ROWS_PLAIN = 0, ROWS_RESID = 1, ROWS_SWIGLU = 2, ROWS_PART = 3 };

struct RowsArgs {
  const uint8_t* w[3]; void* y[3]; long long n[3];      // matrices that share the activation rows (SwiGLU: w[0] gate, w[1] up, one output); every n but the last a multiple of 16
  long long ntot, row_bytes;                            // weight rows over all matrices (SwiGLU: of one), bytes per weight row
  const uint16_t* x;                                    // fp16 activation rows [.][K]
  const float* resid; float* part;                      // resid: added to y[0] (same shape; may be y[0]); part: [ks][M][ntot] partial sums of a split K
  int nseg, epi, y_f32, M, K, ks;
  int row_tiles, tok_tiles;
  // routed rows: tiles[t] = {expert, first row of the tile among that expert's rows}; rows of expert e are off[e] .. off[e + 1] - 1; activation row = row_tok[row] (nullptr: row),
  // output row = row_dst[row] (nullptr: row)
  const int2* tiles; const int* n_tiles; const int* off; const int* row_tok; const int* row_dst; long long estride;
};

// A unit of 64 weights of one row: load and decode into eight 16-byte pieces of natural neighbours, piece v = elements elem(u, v) .. + 7 of the row
template <int T> struct RowsFmt {
  using F = Fmt<T>;
  typedef typename F::Raw Raw;
  static constexpr int NKC = F::NKC;
  static __device__ __forceinline__ Raw load(const uint8_t* row, int u) { return F::load(row, u); }
  static __device__ __forceinline__ int elem(int u, int v) { return F::xoff(u, 4 * v); }
  static __device__ __forceinline__ void nat(const Raw& r, const uint32_t* kc, u32x4* out) {
    uint32_t wv[F::NWV];
    F::decode(r, wv, kc);
    F::to_f16(r, wv);
#pragma unroll
    for (int k = 0; k < 32; k++) {                      // pair k = elements xoff(0, k), + 1: where the decode order keeps its halves (compile-time positions)
      const int e = F::xoff(0, k), p0 = F::spos(e, 4), p1 = F::spos(e + 1, 4);
      const int d0 = 4 * ((p0 >> 3) >> 2) + ((p0 >> 1) & 3), d1 = 4 * ((p1 >> 3) >> 2) + ((p1 >> 1) & 3);
      const uint32_t sel = ((p0 & 1) ? 0x0302u : 0x0100u) | (((p1 & 1) ? 0x0706u : 0x0504u) << 16);
      out[k >> 2][k & 3] = (d0 == d1 && !(p0 & 1) && (p1 & 1)) ? wv[d0] : __builtin_amdgcn_perm(wv[d1], wv[d0], sel);
    }
  }
};
template <> struct RowsFmt<GGML_MXFP4> {                // two blocks of 32
  using F = Fmt<GGML_MXFP4>;
  struct Raw { F::Raw b[2]; };
  static constexpr int NKC = F::NKC;
  static __device__ __forceinline__ Raw load(const uint8_t* row, int u) { Raw r; r.b[0] = F::load(row, 2 * u); r.b[1] = F::load(row, 2 * u + 1); return r; }
  static __device__ __forceinline__ int elem(int u, int v) { return 64 * u + 8 * v; }
  static __device__ __forceinline__ void nat(const Raw& r, const uint32_t*, u32x4* out) {
#pragma unroll
    for (int h = 0; h < 2; h++) {
      uint32_t wv[F::NWV];
      F::to_f16(r.b[h], wv);                            // dword q: (element q, element q + 16)
#pragma unroll
      for (int k = 0; k < 8; k++) {
        out[4 * h + (k >> 2)][k & 3] = pack_even(wv[2 * k], wv[2 * k + 1]);
        out[4 * h + 2 + (k >> 2)][k & 3] = pack_odd(wv[2 * k], wv[2 * k + 1]);
      }
    }
  }
};

__device__ __forceinline__ float rows_silu(float x) { return silu_f(x); }

// Epilogue of a wave: sub-tiles of 16 x 16 results, IS from weight sub-tile wsub (SwiGLU: pairs gate / up) x JN from activation sub-tile tsub (acc column J0) of a tile of cnt rows from
// row0 on.  A lane's accumulator holds the weight rows 4 g .. 4 g + 3 of activation row r16; they go through the wave's own part of LDS (16-byte pieces XORed with the row) so that
// neighbouring lanes store neighbouring results of a row, and in a loop instead of IS x JN copies of the code for every kind of result; the residual rows of four passes are requested
// together.  272 x 256 weights, 200 rows, + residual: 10.8 -> 8.6 us a call.
template <int IS, int JT, int J0, int JN, bool SW, bool MOE>
__device__ __forceinline__ void rows_store(const RowsArgs& a, v4f32 (&acc)[IS][JT], uint8_t* lds, int wsub, int tsub, int lane, int cnt, int row0) {
  constexpr int PC = (SW ? IS / 2 : IS) * 4, TI = 64 / PC;                              // 16-byte pieces of an activation row, rows per pass
  const int r16 = lane & 15, g = lane >> 4;
#pragma unroll
  for (int j = 0; j < JN; j++) {
    uint8_t* const d = lds + (j * 16 + r16) * (PC * 16);
#pragma unroll
    for (int i = 0; i < IS; i += SW ? 2 : 1) {
      f32x4 o;
#pragma unroll
      for (int c = 0; c < 4; c++) { if constexpr (SW) o[c] = rows_silu(acc[i][J0 + j][c]) * acc[i + 1][J0 + j][c]; else o[c] = acc[i][J0 + j][c]; }
      *(f32x4*)(d + ((((SW ? i / 2 : i) * 4 + g) ^ (r16 & (PC - 1))) << 4)) = o;
    }
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  // What a lane stores lies in the same four weight rows of every activation row: matrix, column and address are settled once, a pass adds a step to the address
  const int tl0 = lane / PC, pc = lane & (PC - 1);
  long long row = (long long)wsub * (SW ? 8 : 16) + 4 * pc;
  if (row >= a.ntot) return;
  const bool part = !SW && a.epi == ROWS_PART, res = !SW && a.epi == ROWS_RESID, f32 = part || a.y_f32;
  long long n = a.ntot;
  void* yb = a.y[0];
  if (part) yb = a.part + (size_t)blockIdx.y * a.M * a.ntot;
  else if (!SW) {                                                                       // (a sub-tile lies in one matrix)
    n = a.n[0];
    if (a.nseg > 1 && row >= a.n[0]) { row -= a.n[0]; yb = a.y[1]; n = a.n[1]; if (a.nseg > 2 && row >= n) { row -= n; yb = a.y[2]; n = a.n[2]; } }
  }
  const bool whole = row + 3 < n && (n & 3) == 0;
  const uint32_t left = whole ? 4 : (uint32_t)min(4ll, n - row);
  const int t0 = tsub * 16 + tl0;
  const int* dst = nullptr;
  if constexpr (MOE) dst = a.row_dst;
  constexpr int NB = JN * 16 / TI < 4 ? JN * 16 / TI : 4;                               // passes whose loads are requested together (rows beyond the tile's repeat its last one)
#pragma unroll 1
  for (int it = 0; it < JN * 16 / TI; it += NB) {
    if (tsub * 16 + it * TI >= cnt) break;
    f32x4 o[NB], q[NB]; size_t e[NB];
#pragma unroll
    for (int k = 0; k < NB; k++) {
      const int tl = (it + k) * TI + tl0, t = row0 + min(t0 + (it + k) * TI, cnt - 1);
      o[k] = *(const f32x4*)(lds + tl * (PC * 16) + ((pc ^ (tl & (PC - 1))) << 4));
      e[k] = (size_t)(uint32_t)((MOE && dst) ? dst[t] : t) * (size_t)n + (size_t)row;
    }
    if (whole) {
      if (res) {
#pragma unroll
        for (int k = 0; k < NB; k++) q[k] = *(const f32x4*)(a.resid + e[k]);
#pragma unroll
        for (int k = 0; k < NB; k++) { o[k][0] += q[k].x; o[k][1] += q[k].y; o[k][2] += q[k].z; o[k][3] += q[k].w; }
      }
#pragma unroll
      for (int k = 0; k < NB; k++) {
        if (t0 + (it + k) * TI >= cnt) continue;
        if (f32) *(f32x4*)((float*)yb + e[k]) = o[k];
        else *(u32x2*)((uint16_t*)yb + e[k]) = u32x2{f2h_bits(o[k][0]) | (f2h_bits(o[k][1]) << 16), f2h_bits(o[k][2]) | (f2h_bits(o[k][3]) << 16)};
      }
    } else {
#pragma unroll
      for (int k = 0; k < NB; k++) {
        if (t0 + (it + k) * TI >= cnt) continue;
        for (uint32_t c = 0; c < left; c++) {
          const float v = c == 0 ? o[k][0] : c == 1 ? o[k][1] : c == 2 ? o[k][2] : o[k][3], u = res ? v + a.resid[e[k] + c] : v;
          if (f32) ((float*)yb)[e[k] + c] = u; else ((uint16_t*)yb)[e[k] + c] = (uint16_t)f2h_bits(u);
        }
      }
    }
  }
}

template <int T, int TT, bool SW, bool MOE>
__global__ __launch_bounds__(256, 2) void qgemm_rows_kernel(const RowsArgs a) {
  constexpr bool F16 = T == GGML_F16;
  using RF = RowsFmt<T>;
  constexpr int WW = TT == 128 ? 2 : 4, IS = ROWS_WT / WW / 16, JS = TT / (4 / WW) / 16;   // waves along the weight rows; 16-row sub-tiles of a wave: weights, activations
  constexpr int PX = TT * 16 / 256, PW = ROWS_WT * 16 / 256;                            // 16-byte pieces per thread and step: activations, fp16 weights
  constexpr int XU = TT * 128, WU = ROWS_WT * 128;                                      // bytes of one unit column block in LDS
  __shared__ __attribute__((aligned(16))) uint8_t lds[2 * (XU + WU)];                   // [weights: 2 units x 128 rows x 128 bytes | activations: 2 units x TT rows x 128 bytes]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g = lane >> 4, ww = wave & (WW - 1), wt = wave / WW;
  uint8_t* const ldw = lds; uint8_t* const ldx = lds + 2 * WU;
  // ---- tile.  The workgroups of an XCD (b % 8) take a contiguous run of tiles, activation tiles innermost: a weight tile is fetched into one L2
  const int nwg = a.row_tiles * (MOE ? *a.n_tiles : a.tok_tiles);
  const int per = (nwg + 7) >> 3, b = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
  if (((int)blockIdx.x >> 3) >= per || b >= nwg) return;
  int rt, t0, cnt, erow = 0;
  const uint8_t* wbase0 = a.w[0]; const uint8_t* wbase1 = a.w[1];
  if constexpr (MOE) {
    const int ti = b / a.row_tiles; rt = b - ti * a.row_tiles;                          // (the row tiles of an expert's tile innermost: its few activation rows stay near)
    const int2 te = a.tiles[ti];
    erow = a.off[te.x]; t0 = te.y; cnt = min(a.off[te.x + 1] - erow - t0, TT); erow += t0;
    wbase0 += te.x * a.estride; if (SW) wbase1 += te.x * a.estride;
  } else {
    rt = b / a.tok_tiles; t0 = (b - rt * a.tok_tiles) * TT; cnt = min(a.M - t0, TT);
  }
  // ---- this thread's weight row: LDS row tid >> 1, unit tid & 1 of the step.  The requests for weights are bound by the cache lines they touch, not by their bytes: neighbouring lanes
  // read neighbouring units of a row, half the lines of a request that takes 64 rows (1023 rows x 4096 -> 2 x 14336, gate / up: Q4_0 318 -> 301 us, Q8_0 352 -> 311, Q6_K 427 -> 386).
  // SwiGLU: sub-tiles alternate gate / up, so partner values meet in one lane
  const int lr = tid >> 1, un = tid & 1;
  auto wrow_ptr = [&](int R) __attribute__((always_inline)) {
    if constexpr (SW) {
      long long row = (long long)rt * (ROWS_WT / 2) + (R >> 5) * 16 + (R & 15);
      row = row < a.ntot ? row : a.ntot - 1;
      return ((R & 16) ? wbase1 : wbase0) + row * a.row_bytes;
    } else {
      long long row = (long long)rt * ROWS_WT + R;
      row = row < a.ntot ? row : a.ntot - 1;
      const uint8_t* wb = wbase0;
      if (a.nseg > 1 && row >= a.n[0]) { row -= a.n[0]; wb = a.w[1]; if (a.nseg > 2 && row >= a.n[1]) { row -= a.n[1]; wb = a.w[2]; } }
      return wb + row * a.row_bytes;
    }
  };
  const int nsteps = a.K / ROWS_KS, s0 = (int)((long long)blockIdx.y * nsteps / a.ks), s1 = (int)((long long)(blockIdx.y + 1) * nsteps / a.ks);
  const uint8_t* wp = nullptr; const uint8_t* wpp[F16 ? PW : 1];
  uint32_t kc[RF::NKC];
  if constexpr (F16) {
#pragma unroll
    for (int j = 0; j < PW; j++) wpp[j] = wrow_ptr((tid >> 4) + 16 * j) + (tid & 15) * 16;
  } else { wp = wrow_ptr(lr); RF::F::consts(kc); }
  // ---- this thread's activation pieces: rows (tid >> 4) + 16 j, piece tid & 15 of the step's 256 bytes
  const int xu = (tid >> 3) & 1, xv = tid & 7;
  uint32_t xoff[PX];
#pragma unroll
  for (int j = 0; j < PX; j++) {
    int r = min((tid >> 4) + 16 * j, cnt - 1);                                          // (rows beyond the tile's repeat its last one; their results are dropped)
    if constexpr (MOE) { r += erow; if (a.row_tok) r = a.row_tok[r]; } else r += t0;
    xoff[j] = (uint32_t)r * (uint32_t)a.K;
  }
  typename RF::Raw raw; u32x4 wq[F16 ? PW : 1]; u32x4 xq[PX];
  auto fetch = [&](int s) __attribute__((always_inline)) {
    if constexpr (F16) {
#pragma unroll
      for (int j = 0; j < PW; j++) wq[j] = gld16(wpp[j] + (size_t)s * (2 * ROWS_KS));
    } else raw = RF::load(wp, 2 * s + un);
    const int e = RF::elem(2 * s + xu, xv);
#pragma unroll
    for (int j = 0; j < PX; j++) xq[j] = gld16(a.x + (size_t)(xoff[j] + (uint32_t)e));
  };
  auto put = [&]() __attribute__((always_inline)) {
    if constexpr (F16) {
#pragma unroll
      for (int j = 0; j < PW; j++) { const int R = (tid >> 4) + 16 * j; *(u32x4*)(ldw + xu * WU + R * 128 + ((xv ^ (R & 7) ^ (xu << 2)) << 4)) = wq[j]; }
    } else {
      u32x4 o[8];
      RF::nat(raw, kc, o);
#pragma unroll
      for (int v = 0; v < 8; v++) *(u32x4*)(ldw + un * WU + lr * 128 + ((v ^ (lr & 7) ^ (un << 2)) << 4)) = o[v];
    }
#pragma unroll
    for (int j = 0; j < PX; j++) { const int R = (tid >> 4) + 16 * j; *(u32x4*)(ldx + xu * XU + R * 128 + ((xv ^ (R & 7)) << 4)) = xq[j]; }
  };
  v4f32 acc[IS][JS];
#pragma unroll
  for (int i = 0; i < IS; i++)
#pragma unroll
    for (int j = 0; j < JS; j++) acc[i][j] = v4f32{0.f, 0.f, 0.f, 0.f};
  const uint8_t* const fw = ldw + (ww * IS * 16 + r16) * 128; const uint8_t* const fx = ldx + (wt * JS * 16 + r16) * 128;
  fetch(s0);
  for (int s = s0; s < s1; s++) {
    put();
    if (s + 1 < s1) fetch(s + 1);
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < 4; kk++) {
      const int slot = ((4 * (kk & 1) + g) ^ (r16 & 7)) << 4;
      v8f16 aw[IS], bx[JS];
#pragma unroll
      for (int i = 0; i < IS; i++) aw[i] = *(const v8f16*)(fw + (kk >> 1) * WU + i * 2048 + (slot ^ ((kk >> 1) << 6)));
#pragma unroll
      for (int j = 0; j < JS; j++) bx[j] = *(const v8f16*)(fx + (kk >> 1) * XU + j * 2048 + slot);
#pragma unroll
      for (int i = 0; i < IS; i++)
#pragma unroll
        for (int j = 0; j < JS; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(aw[i], bx[j], acc[i][j], 0, 0, 0);
    }
    __syncthreads();
  }
  // (a wave's results, 64 x 64, 32 x 64 or 32 x 32, fit its quarter of LDS; every wave is behind the last barrier)
  rows_store<IS, JS, 0, JS, SW, MOE>(a, acc, lds + wave * ((XU + WU) / 2), rt * (ROWS_WT / 16) + ww * IS, wt * JS, lane, cnt, MOE ? erow : t0);
}

template <int T, bool MOE> int rows_launch_tt(const RowsArgs& a, int tt, unsigned grid, hipStream_t s) {
  const dim3 g(grid, a.ks);
  const bool sw = a.epi == ROWS_SWIGLU;
  if (tt == 128) { if (sw) qgemm_rows_kernel<T, 128, true, MOE><<<g, 256, 0, s>>>(a); else qgemm_rows_kernel<T, 128, false, MOE><<<g, 256, 0, s>>>(a); }
  else if (tt == 64) { if (sw) qgemm_rows_kernel<T, 64, true, MOE><<<g, 256, 0, s>>>(a); else qgemm_rows_kernel<T, 64, false, MOE><<<g, 256, 0, s>>>(a); }
  else { if (sw) qgemm_rows_kernel<T, 32, true, MOE><<<g, 256, 0, s>>>(a); else qgemm_rows_kernel<T, 32, false, MOE><<<g, 256, 0, s>>>(a); }
  TGA_LAUNCH_CHECK();
  return 0;
}
template <int T> int rows_launch(const RowsArgs& a, int tt, unsigned grid, hipStream_t s) { return a.tiles ? rows_launch_tt<T, true>(a, tt, grid, s) : rows_launch_tt<T, false>(a, tt, grid, s); }
// one function per format, defined in qgemm_rows_*.hip
#define ROWS_FORMATS(X) X(F_Q4_0P) X(F_Q8_0P) X(GGML_F16) X(GGML_MXFP4) X(GGML_Q4_K) X(GGML_Q5_K) X(GGML_Q6_K) X(GGML_IQ4_XS) X(GGML_Q4_1) X(GGML_Q5_0) X(GGML_Q5_1)
