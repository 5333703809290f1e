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

// Eight 16-byte pieces of natural neighbours from a unit in a format's decode order
template <int T> __device__ __forceinline__ void rows_natural(const typename Fmt<T>::Raw& r, const uint32_t* kc, u32x4* out) {
  using F = Fmt<T>;
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

// A unit of 64 weights of one row: load and decode into eight 16-byte pieces of natural neighbours, piece v = elements elem(u, v) .. + 7 of the row
template <int T> struct RowsFmt {
  using F = Fmt<T>;
  typedef typename F::Raw Raw;
  static constexpr int NKC = F::NKC;
  static __device__ __forceinline__ Raw load(const uint8_t* row, int u) { return F::load(row, u); }
  static __device__ __forceinline__ int elem(int u, int v) { return F::xoff(u, 4 * v); }
  static __device__ __forceinline__ void nat(const Raw& r, const uint32_t* kc, u32x4* out) { rows_natural<T>(r, kc, out); }
};
template <> struct RowsFmt<GGML_MXFP4> {                // two blocks of 32
  using F = Fmt<GGML_MXFP4>;
  // The 34 bytes start anywhere in a dword.  The requested dwords are kept as they arrive and shifted where they are used: a shift behind the request would wait for it
  struct Raw { u32x4 v[2]; uint32_t t[2], o; };
  static constexpr int NKC = F::NKC;
  static __device__ __forceinline__ Raw load(const uint8_t* row, int u) {
    const uintptr_t a = (uintptr_t)(row + 34 * u); const uint8_t* q0 = (const uint8_t*)(a & ~(uintptr_t)3); const uint8_t* q1 = (const uint8_t*)((a + 17) & ~(uintptr_t)3);
    Raw r; r.o = (uint32_t)(a & 3); r.v[0] = ld16_a4(q0); r.t[0] = ld4_a4(q0 + 16); r.v[1] = ld16_a4(q1); r.t[1] = ld4_a4(q1 + 16); return r;
  }
  static __device__ __forceinline__ int elem(int u, int v) { return 64 * u + 8 * v; }
  // A byte of a block holds weights e and e + 16: two neighbours are put into one byte first (shifts and a bit-field insert for two pairs), so that the conversions give natural pairs and
  // nothing is packed behind them (150 -> 118 operations for 32 products of a wave at 64 rows; 108 -> 104.5 us for the gate / up experts of 512 tokens)
  static __device__ __forceinline__ void nat(const Raw& r, const uint32_t*, u32x4* out) {
    const uint32_t M = vgpr_const(0x000F000Fu);         // (a register: of a constant mask the compiler makes two operations instead of v_bfi)
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const uint32_t o = h ? (r.o + 1) & 3 : r.o, sh = 8 * (o + 1), e = (r.v[h].x >> (8 * o)) & 0xFFu;      // the block: a scale byte, then sixteen of codes
      const uint32_t d[5] = {r.v[h].x, r.v[h].y, r.v[h].z, r.v[h].w, r.t[h]};
      const float sc = __builtin_bit_cast(float, e ? (e << 23) : 0x00400000u);
#pragma unroll
      for (int t = 0; t < 4; t++) {
        const uint32_t w = (uint32_t)((((uint64_t)d[t + 1] << 32) | d[t]) >> sh), s4 = w >> 4, s8 = w >> 8, lo = (M & w) | (~M & s4), hi = (M & s4) | (~M & s8);
        out[4 * h + (t >> 1)][2 * (t & 1)] = as_u32(__builtin_amdgcn_cvt_scalef32_pk_f16_fp4(lo, sc, 0)); out[4 * h + (t >> 1)][2 * (t & 1) + 1] = as_u32(__builtin_amdgcn_cvt_scalef32_pk_f16_fp4(lo, sc, 2));
        out[4 * h + 2 + (t >> 1)][2 * (t & 1)] = as_u32(__builtin_amdgcn_cvt_scalef32_pk_f16_fp4(hi, sc, 0)); out[4 * h + 2 + (t >> 1)][2 * (t & 1) + 1] = as_u32(__builtin_amdgcn_cvt_scalef32_pk_f16_fp4(hi, sc, 2));
      }
    }
  }
};

template <> struct RowsFmt<GGML_Q6_K> {                 // Fmt's units, but the dwords around each piece are kept as they arrive (superblocks lie at even addresses; see MXFP4)
  using F = Fmt<GGML_Q6_K>;
  struct Raw { u32x4 v[3]; uint32_t e[3]; u32x2 sc; uint32_t se, d, m; };
  static constexpr int NKC = F::NKC;
  typedef uint32_t u32_a2 __attribute__((aligned(2)));
  static __device__ __forceinline__ Raw load(const uint8_t* row, int u) {
    const uint8_t* p = row + 210 * (u >> 2); const int h = (u >> 1) & 1, g = u & 1;
    const uintptr_t a = (uintptr_t)p; const uint8_t* q = (const uint8_t*)(a & ~(uintptr_t)3);
    const int at[3] = {64 * h + 16 * g, 64 * h + 32 + 16 * g, 128 + 32 * h + 16 * g};
    Raw r; r.m = (uint32_t)(a & 2) * 8 | (uint32_t)g;
#pragma unroll
    for (int i = 0; i < 3; i++) { r.v[i] = ld16_a4(q + at[i]); r.e[i] = ld4_a4(q + at[i] + 16); }
    r.sc = *(const TGA_GLOBAL u32x2_a4*)(q + 192 + 8 * h); r.se = ld4_a4(q + 200 + 8 * h); r.d = *(const TGA_GLOBAL uint16_t*)(p + 208);
    return r;
  }
  static __device__ __forceinline__ int elem(int u, int v) { return F::xoff(u, 4 * v); }
  static __device__ __forceinline__ void nat(const Raw& r, const uint32_t* kc, u32x4* out) {
    const uint32_t sh = r.m & 16;
    F::Raw f; u32x4 q[3];
#pragma unroll
    for (int i = 0; i < 3; i++)
      q[i] = u32x4{__builtin_amdgcn_alignbit(r.v[i].y, r.v[i].x, sh), __builtin_amdgcn_alignbit(r.v[i].z, r.v[i].y, sh), __builtin_amdgcn_alignbit(r.v[i].w, r.v[i].z, sh), __builtin_amdgcn_alignbit(r.e[i], r.v[i].w, sh)};
    f.a = q[0]; f.b = q[1]; f.h = q[2];
    f.sc0 = __builtin_amdgcn_alignbit(r.sc.y, r.sc.x, sh); f.sc1 = __builtin_amdgcn_alignbit(r.se, r.sc.y, sh); f.d = (r.m & 1) | (r.d << 16);
    rows_natural<GGML_Q6_K>(f, kc, out);
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
  // Requests: activations (from L2) one step ahead, weights (from HBM) two, in two register sets; fp16 weights, four times the registers, one.  OLMoE-arch experts of 64 rows each, MXFP4:
  // gate / up 104.5 -> 92.4 us, down 57.1 -> 52.8 (with the shifts of a unit's bytes moved behind the wait); 1023 rows, gate / up: Q6_K 383 -> 357 us, Q4_K 301 -> 296; 60 rows: Q8_0 45 -> 40
  constexpr int ND = F16 ? 1 : 2;
  typename RF::Raw raw[ND]; u32x4 wq[F16 ? PW : 1]; u32x4 xq[PX];
  auto wfetch = [&](int s, int q) __attribute__((always_inline)) {
    if constexpr (F16) {
#pragma unroll
      for (int j = 0; j < PW; j++) wq[j] = gld16(wpp[j] + (size_t)s * (2 * ROWS_KS));
    } else raw[q] = RF::load(wp, 2 * s + un);
  };
  auto xfetch = [&](int s) __attribute__((always_inline)) {
    const int e = RF::elem(2 * s + xu, xv);
#pragma unroll
    for (int j = 0; j < PX; j++) xq[j] = gld16(a.x + (size_t)(xoff[j] + (uint32_t)e));
  };
  auto put = [&](int q) __attribute__((always_inline)) {
    if constexpr (F16) {
#pragma unroll
      for (int j = 0; j < PW; j++) { const int R = (tid >> 4) + 16 * j; *(u32x4*)(ldw + xu * WU + R * 128 + ((xv ^ (R & 7) ^ (xu << 2)) << 4)) = wq[j]; }
    } else {
      u32x4 o[8];
      RF::nat(raw[q], kc, o);
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
  auto step = [&](int s, int q) __attribute__((always_inline)) {
    put(q);
    if (s + 1 < s1) xfetch(s + 1);
    if (s + ND < s1) wfetch(s + ND, q);
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
  };
  wfetch(s0, 0); xfetch(s0);
  if constexpr (ND == 2) {
    if (s0 + 1 < s1) wfetch(s0 + 1, ND - 1);
    for (int s = s0; s < s1; s += 2) { step(s, 0); if (s + 1 < s1) step(s + 1, ND - 1); }
  } else { for (int s = s0; s < s1; s++) step(s, 0); }
  // (a wave's results, 64 x 64, 32 x 64 or 32 x 32, fit its quarter of LDS; every wave is behind the last barrier)
  rows_store<IS, JS, 0, JS, SW, MOE>(a, acc, lds + wave * ((XU + WU) / 2), rt * (ROWS_WT / 16) + ww * IS, wt * JS, lane, cnt, MOE ? erow : t0);
}

// ------------------------------------------------------------------------------------------------ 256 weight rows x 128 activation rows
// Long runs of Q4_0 (the rule: rows_wide, qgemm_rows.hip).  In the kernel above both operands of every product go through LDS: 64 x 64 results per wave read 16 KB for 16 KB of written
// tile and step, and LDS is busy longer than the matrix cores.  Here a wave owns 64 weight rows for itself and decodes them straight into its A operands: lane (r16, g) of sub-tile i
// holds the weights of row 16 i + r16 at K position group g of the products, half a unit of 64 at a time, so no weight passes through LDS and none is decoded twice.
// Only the activations are shared: two halves of 128 rows x 128 values, filled by requests that write LDS themselves, one barrier per half step (128 products of a wave); they are read
// as 16-byte pieces in the order in which the weights fall out of their blocks (elem).  Twice the results per byte read from LDS, half of its writes.
// 254 registers at two waves per SIMD are what bounds the formats: Q8_0 and Q4_K, whose half units take twice the registers, were built the same way and were no faster than above (the loop
// of Q4_K spilled; the plain Q4_0 variant keeps five registers in scratch from before its loop to behind it, none inside).
// 1023 rows x 4096 -> 2 x 14336 (gate / up) 301 -> 268 us, x 14336 -> 4096 (down) 158 -> 145 us, 2047 rows 603 -> 505 us and 304 -> 271 us.
#define WIDE_WT 256
#define WIDE_TT 128
#define ROWS_WIDE 256             // the tile height that asks a launcher for this kernel

// Natural pairs (b0, b1), (b2, b3) of the four bytes of w, one byte per halfword
__device__ __forceinline__ uint32_t bytes01(uint32_t w) { return __builtin_amdgcn_perm(0u, w, 0x0c010c00u); }
__device__ __forceinline__ uint32_t bytes23(uint32_t w) { return __builtin_amdgcn_perm(0u, w, 0x0c030c02u); }

// A buffer descriptor on a wave-uniform address: a request is descriptor + 32-bit lane offset + scalar offset, so that the loop keeps one register per sub-tile where 64-bit lane addresses
// would take two per load.  Nothing relies on its range check: rows are clamped.
typedef __amdgpu_buffer_rsrc_t wide_rsrc;
__device__ __forceinline__ wide_rsrc wide_desc(const void* p) { return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, -1, 0x00027000); }
struct WideRow { wide_rsrc r; uint32_t off; };          // sixteen weight rows and the lane's offset in them
__device__ __forceinline__ u32x4 bld16(const WideRow& w, uint32_t at) { return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(w.r, w.off, at, 0)); }
__device__ __forceinline__ uint32_t bld4(const WideRow& w, uint32_t at) { return __builtin_amdgcn_raw_buffer_load_b32(w.r, w.off, at, 0); }

// Half a unit per lane: 32 weights of a row at K positions elem(g, h, v) .. + 7 of the 256 of a step, v = 0 .. 3.  prep: behind the arrival;
// pair(v, t): weights 4 t .. 4 t + 3 of eight, as fp16 rounded like Fmt::to_f16.
template <int T> struct WideFmt { static constexpr bool ok = false; };
template <> struct WideFmt<F_Q4_0P> {                   // block 2 (4 s + g) + h
  static constexpr bool ok = true;
  static constexpr uint32_t K0 = 0x64006400u, K1 = 0x54005400u;
  struct Raw { u32x4 q; uint32_t d; };
  static __device__ __forceinline__ int elem(int g, int h, int v) { return 64 * g + 32 * h + 8 * v; }
  static __device__ __forceinline__ uint32_t lane_off(int g) { return 36 * g; }
  static __device__ __forceinline__ void load(Raw& r, const WideRow& w, int s, int h) { r.q = bld16(w, 144 * s + (h ? 20 : 0)); r.d = bld4(w, 144 * s + 16); }
  static __device__ __forceinline__ void prep(Raw& r, int h) {
    if (h) { r.d >>= 16; return; }
    const uint32_t d = r.q.x & 0xFFFFu;
    r.q = u32x4{__builtin_amdgcn_alignbit(r.q.y, r.q.x, 16), __builtin_amdgcn_alignbit(r.q.z, r.q.y, 16), __builtin_amdgcn_alignbit(r.q.w, r.q.z, 16), __builtin_amdgcn_alignbit(r.d, r.q.w, 16)};
    r.d = d;
  }
  static __device__ __forceinline__ u32x2 pair(const Raw& r, const uint32_t* kc, int v, int t) {
    const half2_t d = h2_splat_bits(r.d & 0xFFFFu);
    uint32_t w = r.q[2 * (v & 1) + t];
    if (v >= 2) w = vgpr_const(w);                      // (the byte pairs are formed again: kept from v - 2 on they would take sixteen registers)
    const uint32_t a = bytes01(w), b = bytes23(w);
    if (v < 2) return u32x2{h2_unbias_scale(and_or(a, 0x000F000Fu, kc[0]), 1032.f, d), h2_unbias_scale(and_or(b, 0x000F000Fu, kc[0]), 1032.f, d)};
    return u32x2{h2_unbias_scale(and_or(a, 0x00F000F0u, kc[1]), 72.f, d), h2_unbias_scale(and_or(b, 0x00F000F0u, kc[1]), 72.f, d)};
  }
};

template <int T, bool SW>
__global__ __launch_bounds__(256, 2) void qgemm_wide_kernel(const RowsArgs a) {
  using WF = WideFmt<T>;
  constexpr int HB = WIDE_TT * 256;                                                     // bytes of one half: 128 rows x 128 values
  // (two variables, so that the compiler knows a read of one half from the requests that fill the other and places no wait between them)
  __shared__ __attribute__((aligned(16))) uint8_t half0[HB];
  __shared__ __attribute__((aligned(16))) uint8_t half1[HB];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, g = lane >> 4;
  const int nwg = a.row_tiles * a.tok_tiles, per = (nwg + 7) >> 3, b = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
  if (((int)blockIdx.x >> 3) >= per || b >= nwg) return;
  const int rt = b / a.tok_tiles, t0 = (b - rt * a.tok_tiles) * WIDE_TT, cnt = min(a.M - t0, WIDE_TT);
  const int nsteps = a.K / 256, s0 = (int)((long long)blockIdx.y * nsteps / a.ks), s1 = (int)((long long)(blockIdx.y + 1) * nsteps / a.ks);
  // This lane's rows.  A sub-tile of sixteen lies in one matrix (its descriptor is wave-uniform); rows beyond the last repeat it, their results are dropped
  wide_rsrc wr[4]; int wlast[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int last = (int)a.ntot - 1;
    int row0 = SW ? rt * (WIDE_WT / 2) + wave * 32 + (i >> 1) * 16 : rt * WIDE_WT + wave * 64 + i * 16;
    row0 = min(row0, last & ~15);
    wlast[i] = last - row0;
    const uint8_t* wb = a.w[0];
    if constexpr (SW) { if (i & 1) wb = a.w[1]; }                                       // (sub-tiles alternate gate / up, so partner values meet in one lane)
    else if (a.nseg > 1 && row0 >= a.n[0]) { row0 -= (int)a.n[0]; wb = a.w[1]; if (a.nseg > 2 && row0 >= a.n[1]) { row0 -= (int)a.n[1]; wb = a.w[2]; } }
    wr[i] = wide_desc(wb + (size_t)row0 * a.row_bytes);
  }
  // Activations: thread = slot tid & 15 of rows (tid >> 4) + 16 j; slot = piece ^ row, piece 4 v + g = K positions elem(g, h, v) .. + 7
  const int xr = tid >> 4, piece = (tid & 15) ^ xr, pg = piece & 3, pv = piece >> 2;
  const wide_rsrc xd = wide_desc(a.x + (size_t)t0 * a.K);
  const uint32_t xe = (uint32_t)WF::elem(pg, 0, pv) * 2, row_bytes = (uint32_t)a.row_bytes, K2 = (uint32_t)a.K * 2;
  const int xh = WF::elem(0, 1, 0);                                                     // (the second half lies a constant behind the first)
  // (lane offsets are formed at each request: eleven registers that the loop has no room for)
  auto xrequest = [&](uint8_t* buf, int s, int h, int j) __attribute__((always_inline)) {     // piece of lane l of wave w, row group j: LDS byte 4096 j + 1024 w + 16 l
    int row = xr; asm volatile("" : "+v"(row));
    const uint32_t off = __umul24((uint32_t)min(row + 16 * j, cnt - 1), K2) + xe;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(xd, (__attribute__((address_space(3))) void*)(buf + j * 4096 + wave * 1024), 16, off, 512 * s + 2 * h * xh, 0, 0);
  };
  auto wrow = [&](int i) __attribute__((always_inline)) {
    int row = r16; asm volatile("" : "+v"(row));
    return WideRow{wr[i], __umul24((uint32_t)min(row, wlast[i]), row_bytes) + WF::lane_off(g)};
  };
  uint32_t kc[2] = {vgpr_const(WF::K0), vgpr_const(WF::K1)};
  v4f32 acc[4][8];
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = 0; j < 8; j++) acc[i][j] = v4f32{0.f, 0.f, 0.f, 0.f};
  typename WF::Raw raw[4], nxt[4];
#pragma unroll
  for (int j = 0; j < 8; j++) xrequest(half0, s0, 0, j);
#pragma unroll
  for (int i = 0; i < 4; i++) WF::load(nxt[i], wrow(i), s0, 0);
  asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  for (int s = s0; s < s1; s++) {
    const int sn = min(s + 1, s1 - 1);                                                  // (behind the last step the requests repeat it; nothing reads what they bring)
#pragma unroll
    for (int h = 0; h < 2; h++) {
      uint8_t* const here = h ? half1 : half0; uint8_t* const there = h ? half0 : half1;
      const int st = h ? sn : s;                                                        // step of the next half
      u32x4 w[2][4]; v8f16 x[3];
      auto xread = [&](int n) __attribute__((always_inline)) { return *(const v8f16*)(here + r16 * 256 + (((4 * (n >> 3) + g) ^ r16) << 4) + (n & 7) * 4096); };
      x[0] = xread(0); x[1] = xread(1);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        raw[i] = nxt[i];
        WF::prep(raw[i], h);
        const u32x2 p = WF::pair(raw[i], kc, 0, 0), q = WF::pair(raw[i], kc, 0, 1);
        w[0][i] = u32x4{p.x, p.y, q.x, q.y};
      }
      // 32 groups of four products, in this order: with each, the activations of two groups further are read, four weights of the next eight of a sub-tile are decoded, and one
      // request of the next half is made
#pragma unroll
      for (int n = 0; n < 32; n++) {
        const int v = n >> 3, j = n & 7;
        if (n + 2 < 32) x[(n + 2) % 3] = xread(n + 2);
        if (v == 0) xrequest(there, st, h ^ 1, j);
        if (v == 1 && j < 4) WF::load(nxt[j], wrow(j), st, h ^ 1);
        if (v < 3) {
          const u32x2 p = WF::pair(raw[j >> 1], kc, v + 1, j & 1);
          u32x4& d = w[(v + 1) & 1][j >> 1];
          if (j & 1) { d.z = p.x; d.w = p.y; } else { d.x = p.x; d.y = p.y; }
        }
#pragma unroll
        for (int i = 0; i < 4; i++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8f16, w[v & 1][i]), x[n % 3], acc[i][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");          // what this half has requested is there; every wave has read its own
    }
  }
  // (a wave's results in two halves of 64 rows, 16 KB each: its quarter of LDS; every wave is behind the last barrier)
  rows_store<4, 8, 0, 4, SW, false>(a, acc, (wave < 2 ? half0 : half1) + (wave & 1) * (HB / 2), rt * (WIDE_WT / 16) + wave * 4, 0, lane, cnt, t0);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  rows_store<4, 8, 4, 4, SW, false>(a, acc, (wave < 2 ? half0 : half1) + (wave & 1) * (HB / 2), rt * (WIDE_WT / 16) + wave * 4, 4, lane, cnt, t0);
}

template <int T, bool MOE> int rows_launch_tt(const RowsArgs& a, int tt, unsigned grid, hipStream_t s) {
  const dim3 g(grid, a.ks);
  const bool sw = a.epi == ROWS_SWIGLU;
  if constexpr (!MOE && WideFmt<T>::ok) {
    if (tt == ROWS_WIDE) { if (sw) qgemm_wide_kernel<T, true><<<g, 256, 0, s>>>(a); else qgemm_wide_kernel<T, false><<<g, 256, 0, s>>>(a); TGA_LAUNCH_CHECK(); return 0; }
  }
  if (tt == 128) { if (sw) qgemm_rows_kernel<T, 128, true, MOE><<<g, 256, 0, s>>>(a); else qgemm_rows_kernel<T, 128, false, MOE><<<g, 256, 0, s>>>(a); }
  else if (tt == 64) { if (sw) qgemm_rows_kernel<T, 64, true, MOE><<<g, 256, 0, s>>>(a); else qgemm_rows_kernel<T, 64, false, MOE><<<g, 256, 0, s>>>(a); }
  else { if (sw) qgemm_rows_kernel<T, 32, true, MOE><<<g, 256, 0, s>>>(a); else qgemm_rows_kernel<T, 32, false, MOE><<<g, 256, 0, s>>>(a); }
  TGA_LAUNCH_CHECK();
  return 0;
}
template <int T> int rows_launch(const RowsArgs& a, int tt, unsigned grid, hipStream_t s) { return a.tiles ? rows_launch_tt<T, true>(a, tt, grid, s) : rows_launch_tt<T, false>(a, tt, grid, s); }
// one function per format, defined in qgemm_rows_*.hip
#define ROWS_FORMATS(X) X(F_Q4_0P) X(F_Q8_0P) X(GGML_F16) X(GGML_MXFP4) X(GGML_Q4_K) X(GGML_Q5_K) X(GGML_Q6_K) X(GGML_IQ4_XS) X(GGML_Q4_1) X(GGML_Q5_0) X(GGML_Q5_1)
