// Many activation rows against Q4_0 and Q4_K blocks in tiles of 512 weight rows x 128 activation rows: the linears of qgemm_rows.hip where such tiles fill the chip (the rule: rows_tall there).
//
// What bounds the 256 x 128 tiles of qgemm_rows.h (1023 rows x 4096 -> 2 x 14336, gate / up, 270 us) are the cache lines that a CU receives, not the matrix cores: a lane fetches its half units from
// rows 2304 bytes apart, so a step of 256 values touches every line of 144 bytes of a row four times over (with requests for whole lines the same kernel took 210 us, with no weight requests 205).
// Here a wave brings the 144 bytes that a step takes of each of its 64 rows into LDS by requests that write it themselves - 1 KB each, contiguous pieces, every line once - and reads its units from
// there.  Weights and decode stay private to the wave, so no barrier concerns them: a wave decodes 64 rows straight into its A operands (lane (r16, g) of sub-tile i: row 16 i + r16, K position
// group g), eight weights of each sub-tile per 32 products.  Eight waves share the activations: a ring of four quarter steps of 64 values, requested two quarters ahead, one barrier per quarter
// in front of its last products, so that the first operands of the next quarter are read behind this one's.  Requests are inline assembly: the compiler would wait for all of them at every read of LDS;
// the waits below are counted by hand and none of the compiler's own is in the loop.  Weights that come from HBM arrive later than the two quarters for which their requests are under way, so every wave
// touches the lines of 32 of its rows two and three steps ahead (the workgroups of neighbouring activation tiles the other 32): weights not in the caches behind the L2s, gate / up of 508 / 1023 / 2047 rows
// 127 -> 120, 235 -> 227, 471 -> 450 us.
// 1023 rows: gate / up 270 -> 217 us, at 2048 rows 495 -> 436; the loop keeps the matrix pipe busy in 70 % of its cycles, at a clock that its power brings down to 1.8 GHz (2.2 in the kernel above).
#include "qgemm_rows.h"

#define TALL_WT 512
#define TALL_TT 128

// A unit of 64 weights of a row per lane and step of 256, read from LDS: unit g of the row's CH bytes.  prep: behind its arrival; pair(v, t): weights 8 v + 4 t .. + 3 as fp16 rounded like Fmt::to_f16
template <int T> struct TallFmt;
template <> struct TallFmt<F_Q4_0P> {
  static constexpr int CH = 144;                        // bytes of 256 weights
  struct Unit { uint32_t a[4], b[4], d; };              // codes of either block, both scales
  static __device__ __forceinline__ Unit unit(const uint8_t* row, int g) {
    const uint32_t* p = (const uint32_t*)(row + 36 * g);
    Unit u;
#pragma unroll
    for (int i = 0; i < 4; i++) { u.a[i] = p[i]; u.b[i] = p[5 + i]; }
    u.d = p[4];
    return u;
  }
  static __device__ __forceinline__ void prep(Unit& u) {
    const uint32_t d = __builtin_amdgcn_perm(u.d, u.a[0], 0x07060100u);
#pragma unroll
    for (int i = 0; i < 3; i++) u.a[i] = __builtin_amdgcn_alignbit(u.a[i + 1], u.a[i], 16);
    u.a[3] = __builtin_amdgcn_alignbit(u.d, u.a[3], 16); u.d = d;
  }
  static __device__ __forceinline__ u32x2 pair(const Unit& u, const uint32_t* kc, int v, int t) {
    const half2_t d = h2_splat_bits(v >= 4 ? u.d >> 16 : u.d & 0xFFFFu);
    uint32_t w = v >= 4 ? u.b[2 * (v & 1) + t] : u.a[2 * (v & 1) + t];
    if (v & 2) w = vgpr_const(w);                       // (the byte pairs are formed again: kept from v - 2 on they would take sixteen registers)
    const uint32_t p = __builtin_amdgcn_perm(0u, w, kc[2]), q = __builtin_amdgcn_perm(0u, w, kc[3]);
    if (!(v & 2)) return u32x2{h2_unbias_scale(and_or(p, 0x000F000Fu, kc[0]), 1032.f, d), h2_unbias_scale(and_or(q, 0x000F000Fu, kc[0]), 1032.f, d)};
    return u32x2{h2_unbias_scale(and_or(p, 0x00F000F0u, kc[1]), 72.f, d), h2_unbias_scale(and_or(q, 0x00F000F0u, kc[1]), 72.f, d)};
  }
};
template <> struct TallFmt<GGML_Q4_K> {                 // low nibbles of 32 bytes are sub-block 2 g, high nibbles 2 g + 1
  static constexpr int CH = 144;
  struct Unit { uint32_t q[8], h[4]; };                 // h: the superblock's header; behind prep scale and offset of either sub-block as float32
  static __device__ __forceinline__ Unit unit(const uint8_t* row, int g) {
    const u32x4 h = *(const u32x4*)row, a = *(const u32x4*)(row + 16 + 32 * g), b = *(const u32x4*)(row + 32 + 32 * g);
    Unit u;
#pragma unroll
    for (int i = 0; i < 4; i++) { u.h[i] = h[i]; u.q[i] = a[i]; u.q[4 + i] = b[i]; }
    return u;
  }
  static __device__ __forceinline__ void prep(Unit& u) {
    uint32_t t = threadIdx.x; asm volatile("" : "+v"(t));                                // (formed at each use: registers that the loop has no room for)
    const uint32_t sh = t & 16, lm = ((t >> 5) & 1) - 1;                                 // get_scale_min_k4 as in Fmt::decode; lm: all ones for sub-blocks 0 .. 3
    const uint32_t y = u.h[1] >> sh, z = u.h[2] >> sh, w = u.h[3] >> sh;
    const uint32_t sc = (y & 0x3F3Fu & lm) | (((w & 0x0F0Fu) | ((y >> 2) & 0x3030u)) & ~lm), mn = (z & 0x3F3Fu & lm) | ((((w >> 4) & 0x0F0Fu) | ((z >> 2) & 0x3030u)) & ~lm);
    const float d = h2f_bits(u.h[0] & 0xFFFFu), dmin = h2f_bits(u.h[0] >> 16);
    const float s0 = d * (float)(sc & 0xFFu), s1 = d * (float)((sc >> 8) & 0xFFu);
    const float m0 = dmin * (float)(mn & 0xFFu) * (1.0f / 1024.0f), m1 = dmin * (float)((mn >> 8) & 0xFFu) * (1.0f / 64.0f);
    u.h[0] = __builtin_bit_cast(uint32_t, s0); u.h[1] = __builtin_bit_cast(uint32_t, s1);
    u.h[2] = __builtin_bit_cast(uint32_t, -1024.f * s0 - 1024.f * m0); u.h[3] = __builtin_bit_cast(uint32_t, -64.f * s1 - 64.f * m1);
  }
  static __device__ __forceinline__ u32x2 pair(const Unit& u, const uint32_t* kc, int v, int t) {
    uint32_t w = u.q[2 * (v & 3) + t];
    if (v & 4) w = vgpr_const(w);
    const uint32_t p = __builtin_amdgcn_perm(0u, w, kc[2]), q = __builtin_amdgcn_perm(0u, w, kc[3]);
    const float s = __builtin_bit_cast(float, u.h[v >> 2]), c = __builtin_bit_cast(float, u.h[2 + (v >> 2)]);
    if (!(v & 4)) return u32x2{h2_unbias_scale_f32(and_or(p, 0x000F000Fu, kc[0]), s, c), h2_unbias_scale_f32(and_or(q, 0x000F000Fu, kc[0]), s, c)};
    return u32x2{h2_unbias_scale_f32(and_or(p, 0x00F000F0u, kc[1]), s, c), h2_unbias_scale_f32(and_or(q, 0x00F000F0u, kc[1]), s, c)};
  }
};

// A request of the wave: lane l's sixteen bytes at descriptor + off + at land at LDS byte dst + 16 l (m0; one wait state between its write and the request, which the compiler does not add inside an asm statement; m0
// is no clobber, as the compiler calls that undefined: it uses none of its own in this kernel)
__device__ __forceinline__ void tall_request(u32x4 r, uint32_t dst, uint32_t off, int at) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" :: "s"(dst), "v"(off), "s"(r), "s"(at) : "memory");
}
// ... four bytes a lane: what brings a line nearer
__device__ __forceinline__ void tall_touch(u32x4 r, uint32_t dst, uint32_t off) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, 0 offen lds" :: "s"(dst), "v"(off), "s"(r) : "memory");
}
__device__ __forceinline__ u32x4 tall_desc(const void* p) {                             // (as wide_desc: no request relies on its range check; a touch near the end of a matrix does, with a range of its own)
  const uint64_t v = (uint64_t)(uintptr_t)p;
  return u32x4{(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)v), (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(v >> 32)) & 0xFFFFu, 0xFFFFFFFFu, 0x00027000u};
}

template <int T, bool SW>
__global__ __launch_bounds__(512, 1) void qgemm_tall_kernel(const RowsArgs a) {
  using WF = TallFmt<T>;
  constexpr int QB = TALL_TT * 128, SB = 16 * WF::CH, PC = WF::CH / 16, WB = 4 * SB;    // bytes: activations of a quarter, weights of a sub-tile; pieces of a row; bytes of a wave's weights
  static_assert(SB > 2048 && SB <= 3072 && 4 * QB >= 4 * 16384 && 8 * WB >= 4 * 16384, "three requests a sub-tile; 16 KB a wave for its results");
  __shared__ __attribute__((aligned(16))) uint8_t lds[4 * QB + 8 * WB + 256];           // [four quarters: 128 rows of 64 values | eight waves: 64 rows of CH bytes | what touches bring]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, g = lane >> 4;
  // ---- tile: as in qgemm_rows_kernel, the workgroups of an XCD take a contiguous run, activation tiles innermost
  const int nwg = a.row_tiles * a.tok_tiles, per = (nwg + 7) >> 3, b = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
  if (((int)blockIdx.x >> 3) >= per || b >= nwg) return;
  const int rt = b / a.tok_tiles, t0 = (b - rt * a.tok_tiles) * TALL_TT, cnt = min(a.M - t0, TALL_TT);
  const int nsteps = a.K / 256, s0 = (int)((long long)blockIdx.y * nsteps / a.ks), s1 = (int)((long long)(blockIdx.y + 1) * nsteps / a.ks);
  // ---- this wave's rows: sub-tiles of sixteen, each in one matrix (SwiGLU: they alternate gate / up, so partner values meet in one lane); those beyond the last repeat it, their results are dropped
  u32x4 wr[4], tr = {};
  const int ti = SW ? b & 1 : (b & 1) * 2;                                              // (sub-tile from which on this workgroup's touches bring 32 rows)
#pragma unroll
  for (int i = 0; i < 4; i++) {
    int row0 = min(SW ? rt * (TALL_WT / 2) + wave * 32 + (i >> 1) * 16 : rt * TALL_WT + wave * 64 + i * 16, (int)a.ntot - 16);
    const uint8_t* wb = a.w[0]; int n = (int)a.n[0];
    if constexpr (SW) { if (i & 1) wb = a.w[1]; }
    else if (a.nseg > 1 && row0 >= n) { row0 -= n; wb = a.w[1]; n = (int)a.n[1]; if (a.nseg > 2 && row0 >= n) { row0 -= n; wb = a.w[2]; n = (int)a.n[2]; } }
    wr[i] = tall_desc(wb + (size_t)row0 * a.row_bytes);
    if (i == ti) { tr = wr[i]; tr.z = (uint32_t)min((long long)(n - row0) * a.row_bytes, 0xFFFFFFFFll); }      // (its range ends with the matrix: 32 rows may not)
  }
  // ---- weights: a sub-tile's 16 PC pieces by three requests, the last one from its end (pieces that two of them bring are the same bytes)
  const uint32_t lbase = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint8_t*)lds, wbase = lbase + 4 * QB + wave * WB;
  auto woffset = [&](int k) __attribute__((always_inline)) {                            // (formed where it is used: the loop has no room for three registers)
    int l = lane; asm volatile("" : "+v"(l));
    const int p = (k < 2 ? 64 * k : 16 * PC - 64) + l, r = p / PC;
    return __umul24((uint32_t)r, (uint32_t)a.row_bytes) + (uint32_t)(p - r * PC) * 16;
  };
  uint32_t woff;
  auto wrequest = [&](int s, int n) __attribute__((always_inline)) {
    const int k = n >> 2, i = n & 3;
    if (i == 0) woff = woffset(k);
    tall_request(wr[i], wbase + i * SB + (k < 2 ? 1024 * k : SB - 1024), woff, WF::CH * s);
  };
  auto touch = [&](int s) __attribute__((always_inline)) {
    int l = lane; asm volatile("" : "+v"(l));
    const uint32_t at = (uint32_t)min(WF::CH * (s & ~1), (int)a.row_bytes - 2 * WF::CH);
    tall_touch(tr, lbase + 4 * QB + 8 * WB, __umul24((uint32_t)((l & 15) + 16 * (s & 1)), (uint32_t)a.row_bytes) + (uint32_t)min((l >> 4) * 96, 2 * WF::CH - 4) + at);
  };
  // ---- activations: quarter c of a step = values 64 g + 16 c .. + 15 of every group g; thread: slot tid & 7 of rows tid >> 3 and + 64; slot = piece ^ row, piece 4 e + g = values 64 g + 16 c + 8 e .. + 7
  const int xr = tid >> 3, piece = (tid & 7) ^ (xr & 7);
  const u32x4 xd = tall_desc(a.x + (size_t)t0 * a.K);
  uint32_t xo[2];
#pragma unroll
  for (int j = 0; j < 2; j++) xo[j] = (uint32_t)min(xr + 64 * j, cnt - 1) * ((uint32_t)a.K * 2) + (uint32_t)(128 * (piece & 3) + 16 * (piece >> 2));      // (rows beyond the tile's repeat its last one)
  auto xrequest = [&](int c, int s, int j) __attribute__((always_inline)) { tall_request(xd, lbase + c * QB + j * 8192 + wave * 1024, xo[j], 512 * s + 32 * c); };
  // ---- reads (addresses kept from the compiler, which would form each of a step's 64 in front of the loop)
  uint32_t xl[2] = {(uint32_t)(r16 * 128 + ((g ^ (r16 & 7)) << 4)), (uint32_t)(r16 * 128 + (((4 + g) ^ (r16 & 7)) << 4))}, ub = 4 * QB + wave * WB + r16 * WF::CH;
  asm volatile("" : "+v"(xl[0]), "+v"(xl[1]), "+v"(ub));
  auto xread = [&](int c, int n) __attribute__((always_inline)) { return *(const v8f16*)(lds + xl[n >> 3] + c * QB + (n & 7) * 2048); };
  uint32_t kc[4] = {vgpr_const(0x64006400u), vgpr_const(0x54005400u), 0x0c010c00u, 0x0c030c02u};      // (kc[2], kc[3]: natural pairs of a dword's four bytes)
  asm("" : "+s"(kc[2]), "+s"(kc[3]));
  v4f32 acc[4][8];
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = 0; j < 8; j++) acc[i][j] = v4f32{0.f, 0.f, 0.f, 0.f};
  typename WF::Unit u[4];
  u32x4 w[2][4]; v8f16 x[3];
  auto uread = [&](int i) __attribute__((always_inline)) { u[i] = WF::unit(lds + ub + i * SB, g); };
  auto decode = [&](int v, int j) __attribute__((always_inline)) {                      // half of weights 8 v .. + 7 of sub-tile j / 2
    const u32x2 p = WF::pair(u[j >> 1], kc, v, j & 1);
    u32x4& d = w[v & 1][j >> 1];
    if (j & 1) { d.z = p.x; d.w = p.y; } else { d.x = p.x; d.y = p.y; }
  };
#pragma unroll
  for (int n = 0; n < 12; n++) wrequest(s0, n);
#pragma unroll
  for (int c = 0; c < 3; c++) { xrequest(c, s0, 0); xrequest(c, s0, 1); }
  touch((s0 + 1) & ~1); touch((s0 + 1) | 1);
  asm volatile("s_waitcnt vmcnt(2)\n\ts_barrier" ::: "memory");
#pragma unroll
  for (int i = 0; i < 4; i++) uread(i);
#pragma unroll
  for (int i = 0; i < 4; i++) { WF::prep(u[i]); decode(0, 2 * i); decode(0, 2 * i + 1); }
  x[0] = xread(0, 0); x[1] = xread(0, 1);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                                    // (the first step's units are in registers: the next one's requests may land)
  for (int s = s0; s < s1; s++) {
    const int sn = min(s + 1, s1 - 1);                                                  // (behind the last step the requests repeat it; nothing reads what they bring)
    // 64 groups of four products, in this order.  With each: the activations of two groups further are read and four weights of the next eight of a sub-tile are decoded.  Requests: next step's weights
    // in the first quarter (its units are read in the last one, when each sub-tile's are used up), a quarter's activations at the end of the one three before it, behind a barrier that every wave
    // reaches when it has used the quarter which they replace, and a touch last in the first quarter, so that only the last barrier's wait has it in front.
#pragma unroll
    for (int c = 0; c < 4; c++) {
#pragma unroll
      for (int n = 0; n < 16; n++) {
        const int v = 2 * c + (n >> 3), j = n & 7, m = 16 * c + n;
        if (n == 12) {                                                                  // the next quarter's activations are there; younger are the two requests of the quarter behind it, twelve for weights, a touch
          if (c == 0) asm volatile("s_waitcnt vmcnt(14)\n\ts_barrier" ::: "memory");
          else if (c == 1) asm volatile("s_waitcnt vmcnt(15)\n\ts_barrier" ::: "memory");
          else if (c == 2) asm volatile("s_waitcnt vmcnt(3)\n\ts_barrier" ::: "memory");
          else asm volatile("s_waitcnt vmcnt(2)\n\ts_barrier" ::: "memory");
        }
        x[(m + 2) % 3] = n < 14 ? xread(c, n + 2) : xread((c + 1) & 3, n - 14);
        if (c == 0 && n < 12) wrequest(sn, n);
        if (n >= 14) xrequest((c + 3) & 3, c == 0 ? s : sn, n - 14);
        if (c == 0 && n == 15) touch(s + 3);
        if (v == 6 && j >= 2 && !(j & 1)) uread(j / 2 - 1);
        if (v == 7 && j == 0) uread(3);
        if (v < 7) decode(v + 1, j);
        else { if (!(j & 1)) WF::prep(u[j >> 1]); decode(0, j); }
#pragma unroll
        for (int i = 0; i < 4; i++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8f16, w[v & 1][i]), x[m % 3], acc[i][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    x[0] = x[1]; x[1] = x[2];                                                           // (64 groups, three operands)
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  // (a wave's results in two halves of 64 rows, 16 KB each; every wave is behind the last barrier and no request is under way)
  rows_store<4, 8, 0, 4, SW, false>(a, acc, lds + wave * 16384, rt * (TALL_WT / 16) + wave * 4, 0, lane, cnt, t0);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  rows_store<4, 8, 4, 4, SW, false>(a, acc, lds + wave * 16384, rt * (TALL_WT / 16) + wave * 4, 4, lane, cnt, t0);
}

int tga_rows_tall(int fmt, const RowsArgs& a, unsigned grid, hipStream_t s) {
  TGA_REQUIRE(a.K >= 512 && a.K % 256 == 0, "tga_rows_tall: rows of %d values", a.K);    // (a touch brings two steps of a row)
  const dim3 g(grid, a.ks);
  const bool sw = a.epi == ROWS_SWIGLU;
  if (fmt == F_Q4_0P) { if (sw) qgemm_tall_kernel<F_Q4_0P, true><<<g, 512, 0, s>>>(a); else qgemm_tall_kernel<F_Q4_0P, false><<<g, 512, 0, s>>>(a); }
  else { if (sw) qgemm_tall_kernel<GGML_Q4_K, true><<<g, 512, 0, s>>>(a); else qgemm_tall_kernel<GGML_Q4_K, false><<<g, 512, 0, s>>>(a); }
  TGA_LAUNCH_CHECK();
  return 0;
}
