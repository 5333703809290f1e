// A prefill step of any number of rows: the positions pos0 .. pos0 + P - 1 of one or more sequences go through all blocks together (the reference's chunked prefill,
// tinygrad/llm/model.py:464, 476-481, with the prompt as one chunk), every linear as ONE pass over its weights (qgemm_rows.h).  Per block: q / k / v -> rotation +
// append -> attention -> attn_output (+ residual, norm) -> gate / up + SwiGLU -> down (+ residual, the next block's norm): eight launches, or for a MoE block norm -> router logits -> gating ->
// grouping -> selected experts' gate / up + SwiGLU -> down -> weighted sum (+ residual), model.py:110-135.  The launches are issued by one native call.
// MI355X, prompt to first logits: 8B-arch Q4_0 of 1024 tokens 42.4 ms (steps of 128 rows, qgemm64.hip) -> 18.0; OLMoE-arch of 512 tokens, where its user asks for it, 64.0 (steps of 16 rows, an
// expert GEMV per token and slot) -> 5.0; four 8B-arch Q4_K_M sequences of 128 tokens 333 (one lockstep step per position) -> 13.3.
#include "qgemm_rows.h"
#include "decode.h"
#include "moe_gate.h"
#include "prefill.h"

int tga_rows_fmt(int ggml_type, int64_t K);                                              // qgemm_rows.hip
int64_t tga_rows_row_bytes(int fmt, int64_t K);
int tga_rows_dispatch(int fmt, const RowsArgs& a, int tt, unsigned grid, hipStream_t s);
int tga_rows_linear(int ggml_type, int nseg, const void* const* w, void* const* y, const int64_t* n, const void* x_f16, int y_dtype, int64_t M, int64_t K, int epilogue, const float* resid,
                    void* workspace, int64_t workspace_bytes, const float* norm_w, float norm_eps, void* xn, int* parts, void* stream);
int tga_rows_norm(float* x, const float* w, int M, int n, float eps, void* xn, void* stream);

// ------------------------------------------------------------------------------------------------ rotation + append
// One workgroup per row.  q is rotated (after its norm) and leaves as TWO fp16 values per element, the rounded value and what the rounding left over, for matrix-core
// scores of the float32 query (rows_attn_kernel); k is rotated into the cache, v copied.  The rotation is apply_rope's (model.py:29-33) written as one rounded product and one fused multiply-add,
// like every kernel that rotates, so a cache row has the same bits whichever path appended it.  norm: 0 none, 1 RMSNorm over the whole q / k rows (model.py:169), 2 per head (:180).
// Rows come as the linears leave them: whole (ks 1), or as the sums of a split K, plane values apart, which are completed here in their order.  A launch that completes them and a rotation of whole rows / here, us:
// 4096 + 2 x 1024 values, 1023 and 508 rows of two parts 12.0 + 8.9 / 12.0, 7.0 + 5.8 / 7.2, 256 and 129 of five 7.2 + 5.1 / 8.0, 5.0 + 4.8 / 6.2, 26 of eight 4.6 + 4.4 / 6.2; 2048 + 2 x 512, 699 rows of three
// 7.1 + 5.2 / 6.8, 97 and 22 of four 4.1 + 3.7 / 4.1, 2.8 + 3.7 / 4.0; 1024 + 2 x 256, 1099 of two 5.2 + 5.2 / 5.5.  Few rows are a chain of trips to memory: with a trip per part the 22 rows took 10.9.
struct RopeSrc { const float* p; size_t plane; int stride, ks; };
struct RopeArgs {
  RopeSrc q, k, v; const float* qn; const float* kn; const float* rope;
  uint16_t* qh; uint16_t* ql; uint16_t* ck; uint16_t* cv; int* zero;      // zero: n_zero counters cleared for the launches behind this one
  int H, KV, hd, max_ctx, P, pos0, norm, n_zero; float eps;
};
// RU: heads of a wave whose values are requested together, and with them up to four parts of each: a head or a part at a time, each is a trip to memory.  PARTS: ks of q and k, 5: more than four (kernels of
// their own: one that holds them all takes 224 registers, whole rows 50, and half as many workgroups share a CU)
template <int RU, int PARTS>
__global__ __launch_bounds__(512) void rows_rope_kernel(const RopeArgs a) {
  __shared__ float red[8];
  const int r = blockIdx.x, z = r / a.P, pos = a.pos0 + r % a.P, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, half = a.hd >> 1;
  const int nq = a.H * a.hd, nk = a.KV * a.hd;
  if (r == 0) for (int i = tid; i < a.n_zero; i += 512) a.zero[i] = 0;
  const float* q = a.q.p + (size_t)r * a.q.stride; const float* k = a.k.p + (size_t)r * a.k.stride; const float* v = a.v.p + (size_t)r * a.v.stride;
  const size_t crow = ((size_t)z * a.KV * a.max_ctx + pos) * a.hd, cstep = (size_t)a.max_ctx * a.hd;
  for (int e = 4 * (511 - tid); e < nk; e += 2048) {                      // (the last waves first: they have the fewest heads)
    const int hh = e / a.hd;
    f32x4 x = *(const f32x4*)(v + e);
    for (int p = 1; p < a.v.ks; p += 3) {                                 // (the last part again behind it, and not added)
      f32x4 y[3];
#pragma unroll
      for (int j = 0; j < 3; j++) y[j] = *(const f32x4*)(v + min(p + j, a.v.ks - 1) * a.v.plane + e);
#pragma unroll
      for (int j = 0; j < 3; j++) if (p + j < a.v.ks) { x.x += y[j].x; x.y += y[j].y; x.z += y[j].z; x.w += y[j].w; }
    }
    *(u32x2*)(a.cv + crow + hh * cstep + (e - hh * a.hd)) = u32x2{f2h_bits(x.x) | (f2h_bits(x.y) << 16), f2h_bits(x.z) | (f2h_bits(x.w) << 16)};
  }
  float qs = 1.f, ks = 1.f;
  if (a.norm == 1) {
    float s0 = 0.f, s1 = 0.f;
    for (int i = tid & 255; wave < 4 && i < (nq >> 2); i += 256) { const f32x4 x = ((const f32x4*)q)[i]; s0 += x.x * x.x + x.y * x.y + x.z * x.z + x.w * x.w; }
    for (int i = tid & 255; wave < 4 && i < (nk >> 2); i += 256) { const f32x4 x = ((const f32x4*)k)[i]; s1 += x.x * x.x + x.y * x.y + x.z * x.z + x.w * x.w; }
    s0 = wave_sum(s0); s1 = wave_sum(s1);
    if (lane == 0 && wave < 4) { red[wave] = s0; red[4 + wave] = s1; }
    __syncthreads();
    qs = 1.0f / sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)nq + a.eps);
    ks = 1.0f / sqrtf((red[4] + red[5] + red[6] + red[7]) / (float)nk + a.eps);
  }
  const float* rr = a.rope + (size_t)pos * a.hd;
  const bool live = lane < half;                                          // (half is 32 or 64)
  const int i = live ? lane : half - 1;
  const float c = rr[i], s = rr[half + i];
  const int nh = a.H + a.KV;
  for (int h0 = wave; h0 < nh; h0 += 8 * RU) {
    constexpr int N = PARTS < 5 ? PARTS : 4;
    float xa[RU], xb[RU], ya[N][RU], yb[N][RU];
    auto request = [&](int p) __attribute__((always_inline)) {              // parts p .. p + N - 1 (q and k are of one launch where they are split); behind the last one that one again
#pragma unroll
      for (int j = 0; j < N; j++)
#pragma unroll
        for (int u = 0; u < RU; u++) {
          const int h = min(h0 + 8 * u, nh - 1);
          const float* src = (h < a.H ? q + h * a.hd : k + (h - a.H) * a.hd) + (PARTS < 5 ? j : min(p + j, a.q.ks - 1)) * a.q.plane;
          ya[j][u] = src[i]; yb[j][u] = src[half + i];
        }
    };
    request(0);
#pragma unroll
    for (int u = 0; u < RU; u++) {
      xa[u] = ya[0][u]; xb[u] = yb[0][u];
#pragma unroll
      for (int j = 1; j < N; j++) { xa[u] += ya[j][u]; xb[u] += yb[j][u]; }
    }
    if constexpr (PARTS == 5) {
#pragma clang loop unroll(disable)
      for (int p = 4; p < a.q.ks; p += 4) {
        request(p);
#pragma unroll
        for (int j = 0; j < N; j++)
          if (p + j < a.q.ks)
#pragma unroll
            for (int u = 0; u < RU; u++) { xa[u] += ya[j][u]; xb[u] += yb[j][u]; }
      }
    }
#pragma unroll
    for (int u = 0; u < RU; u++) {
      const int h = h0 + 8 * u;
      if (h >= nh) break;
      const bool isq = h < a.H;
      const int hh = isq ? h : h - a.H;
      float x1 = xa[u], x2 = xb[u];
      if (a.norm) {
        float sc = isq ? qs : ks;
        if (a.norm == 2) sc = 1.0f / sqrtf(wave_sum(live ? x1 * x1 + x2 * x2 : 0.f) / (float)a.hd + a.eps);
        const float* w = isq ? a.qn : a.kn;
        const int wo = a.norm == 2 ? 0 : hh * a.hd;
        x1 = (x1 * sc) * w[wo + i]; x2 = (x2 * sc) * w[wo + half + i];
      }
      float lo = __builtin_fmaf(x1, c, -(x2 * s)), hi = __builtin_fmaf(x2, c, x1 * s);
      asm volatile("" : "+v"(lo), "+v"(hi));                            // (float32 values: folded with the conversion into v_fma_mixlo_f16 they round once, and some cache rows had other bits)
      if (!live) continue;
      if (isq) {
        const size_t o = (size_t)r * nq + hh * a.hd + i;
        const _Float16 l16 = (_Float16)lo, h16 = (_Float16)hi;
        a.qh[o] = __builtin_bit_cast(uint16_t, l16); a.qh[o + half] = __builtin_bit_cast(uint16_t, h16);
        a.ql[o] = (uint16_t)f2h_bits(lo - (float)l16); a.ql[o + half] = (uint16_t)f2h_bits(hi - (float)h16);
      } else {
        uint16_t* d = a.ck + crow + hh * cstep;
        d[i] = (uint16_t)f2h_bits(lo); d[half + i] = (uint16_t)f2h_bits(hi);
      }
    }
  }
}

// (heads of a wave dealt evenly to as few groups of five as hold them)
static void rows_rope_launch(const RopeArgs& a, unsigned rows, hipStream_t s) {
  const int n = (a.H + a.KV + 7) / 8, groups = (n + 4) / 5, ru = (n + groups - 1) / groups, parts = a.q.ks < 5 ? a.q.ks : 5;
#define ROPE_P(RU, PARTS) if (parts == PARTS) rows_rope_kernel<RU, PARTS><<<rows, 512, 0, s>>>(a)
#define ROPE(RU) do { ROPE_P(RU, 1); ROPE_P(RU, 2); ROPE_P(RU, 3); ROPE_P(RU, 4); ROPE_P(RU, 5); } while (0)
  if (ru <= 2) ROPE(2); else if (ru == 3) ROPE(3); else ROPE(5);
#undef ROPE
#undef ROPE_P
}

// ------------------------------------------------------------------------------------------------ attention
// Causal attention of the rows over the cache (their own keys included): workgroup = 64 rows of one query head, wave = 16 of them, tiles of 64 keys with a running maximum.
// S^T = K Q^T: keys as A operand from LDS (rows of head_dim values, 16-byte pieces XORed with the key), the rotated queries as two fp16 B operands held in registers.
// O^T = V^T P^T: the probabilities likewise as a rounded value and its remainder (each product once more on matrix cores that are far from busy here); the eight keys a lane holds after the first product are taken as they are, and V is written to LDS transposed with its keys in that order, two keys
// per dword, pieces XORed with the dimension.  The next tile is fetched while this one is multiplied.  flattened workgroup = (kv head, sequence) innermost: with eight
// kv heads all readers of a head's rows run on one XCD and share its L2; the longest row tiles come first, in runs of as many tiles as give every CU a workgroup (cus), every second run
// the other way round: the workgroups that share a CU have long and short tiles (1023 rows, 32 heads, two workgroups a CU: 41.4 -> 39.5 us).
// NG = 2: eight waves, of which four take the even tiles of keys and four the odd ones; their sums meet in LDS.  A workgroup is a chain of tiles, 2.4 us each where it has a CU to itself and little less
// where two share one, and registers leave room for eight waves a CU: for as many workgroups as CUs from four tiles on (heads of 128, 192 / 256 workgroups of up to 6 / 8 tiles 16.4 -> 15.5 / 20.4 ->
// 18.1 us; of 64, 128 / 256 of up to 16 / 32 28.8 -> 20.5 / 55 -> 37), and for twice as many where chains are long (heads of 128, 288 of up to 12 tiles 28.0 -> 23.5, 384 of up to 16
// 36.7 -> 30.7, 448 / 512 of up to 16 36.8 -> 36.0 / 39.2 -> 38.1 in the Q4_0 8B model, 512 of up to 32 67 -> 62; of 64, 512 of up to 16 / 32 29.2 -> 24.3, 54.4 -> 41.6; not
// taken: 192 of 3 tiles 10.9 / 11.7, 384 of 3 12.9 / 17.2, 512 of 4 / 8 16.9 / 21.0, 24 / 26, 768 of up to 24 71 / 82, 1024 of up to 32 114 / 129).
// Two fp16 values hold 22 bits and more of a query or probability, and sums are formed in few additions at their full size (remainders first, two chains per score, a tile's products from
// zero).  Share of fp16 results that are not the rounded float64 attention, 64 and 1024 positions, heads of 64 and 128, scores of standard deviation 0.03 .. 5: 1.8e-4 .. 2.2e-3; the float32
// kernel of eight rows and fewer: 2.4e-4 .. 2.4e-3.  (Queries beyond 65504 have no such pair, as keys beyond have no cache row.)
#define PSCALE 32768.0f             // of probabilities on their way to two fp16 values (the remainder of 0.2 is a subnormal number already: the absolute step 2^-24)
struct RowsAttnArgs { const uint16_t* qh; const uint16_t* ql; const uint16_t* ck; const uint16_t* cv; uint16_t* out; int H, KV, max_ctx, P, pos0, nseq, qtiles, cus; float scale; };

template <int HD, int NG>
__global__ __launch_bounds__(256 * NG) void rows_attn_kernel(const RowsAttnArgs a) {
  constexpr int NJ = HD / 32, NH = HD / 16, PC = HD / 8, IK = HD / 32, IV = HD / 64;     // 16-byte pieces per row; loads per thread and tile
  __shared__ __attribute__((aligned(16))) uint8_t kl_[NG][64 * HD * 2];
  __shared__ __attribute__((aligned(16))) uint8_t vl_[NG][HD * 128];
  const int part_ = NG > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0, tid = NG > 1 ? threadIdx.x & 255 : threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 4, c = lane & 15;
  uint8_t* const kl = kl_[part_]; uint8_t* const vl = vl_[part_];
  const int group = a.H / a.KV, kz = a.KV * a.nseq;
  int b = blockIdx.x;
  const int kvz = b % kz; b /= kz;
  const int hh = b % group, rank = b / group, part = rank / a.cus, qt = a.qtiles - 1 - ((part & 1) ? min((part + 1) * a.cus, a.qtiles) - 1 - (rank - part * a.cus) : rank);
  const int kvh = kvz % a.KV, z = kvz / a.KV, head = kvh * group + hh;
  const int row_first = qt * 64, nq = a.H * HD;
  const int wrow = row_first + wave * 16;                                 // first row of this wave
  const int row = min(wrow + c, a.P - 1), pos = a.pos0 + row;
  const uint16_t* ck = a.ck + ((size_t)z * a.KV + kvh) * a.max_ctx * HD; const uint16_t* cv = a.cv + ((size_t)z * a.KV + kvh) * a.max_ctx * HD;
  u32x4 qb[NJ], qr[NJ];
  const size_t qo = ((size_t)z * a.P + row) * nq + head * HD + 8 * g;
#pragma unroll
  for (int j = 0; j < NJ; j++) { qb[j] = *(const u32x4*)(a.qh + qo + 32 * j); qr[j] = *(const u32x4*)(a.ql + qo + 32 * j); }
  const int last_wg = a.pos0 + min(row_first + 63, a.P - 1), ntiles = last_wg / 64 + 1;      // keys 0 .. last_wg are visible to some row of the workgroup
  const int last_wave = a.pos0 + min(wrow + 15, a.P - 1), first_wave = a.pos0 + min(wrow, a.P - 1);
  u32x4 kq[IK], vq[IV][2];
  const int vchunk = tid % PC, vpair = tid / PC;                          // V: dimensions 8 vchunk .. + 7 of keys 2 pair, 2 pair + 1
  auto fetch = [&](int t) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < IK; i++) {
      const int it = tid + 256 * i, key = min(64 * t + it / PC, last_wg);                     // (rows that no position here sees are masked, but 0 times what an earlier prompt left there would be NaN if that is not finite)
      kq[i] = *(const u32x4*)(ck + (size_t)key * HD + (it % PC) * 8);
    }
#pragma unroll
    for (int i = 0; i < IV; i++)
#pragma unroll
      for (int h = 0; h < 2; h++) { const int key = min(64 * t + 2 * (vpair + i * (256 / PC)) + h, last_wg); vq[i][h] = *(const u32x4*)(cv + (size_t)key * HD + vchunk * 8); }
  };
  auto put = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < IK; i++) { const int it = tid + 256 * i, key = it / PC; *(u32x4*)(kl + key * HD * 2 + (((it % PC) ^ (key & 7)) << 4)) = kq[i]; }
#pragma unroll
    for (int i = 0; i < IV; i++) {
      const int j = 2 * (vpair + i * (256 / PC)), slot = (j & 32) + 8 * ((j & 15) >> 2) + 4 * ((j >> 4) & 1) + (j & 3);
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const uint32_t lo = vq[i][0][e >> 1], hi = vq[i][1][e >> 1];
        const int d = vchunk * 8 + e;
        *(uint32_t*)(vl + d * 128 + (((slot >> 3) ^ ((d ^ (d >> 3)) & 7)) << 4) + (slot & 7) * 2) = (e & 1) ? pack_odd(lo, hi) : pack_even(lo, hi);
      }
    }
  };
  v4f32 O[NH];
#pragma unroll
  for (int h = 0; h < NH; h++) O[h] = v4f32{0.f, 0.f, 0.f, 0.f};
  float M = -INFINITY, L = 0.f;
  fetch(part_);
  for (int t = part_; t - part_ < ntiles; t += NG) {                       // (every part as often: a tile behind the last one is skipped below)
    put();
    if (t - part_ + NG < ntiles) fetch(t + NG);
    __syncthreads();
    if (64 * t <= last_wave) {
      v4f32 sc[4];
#pragma unroll
      for (int k = 0; k < 4; k++) {
        sc[k] = v4f32{0.f, 0.f, 0.f, 0.f};
        const int key = 16 * k + c;
        v8f16 ka[NJ];
#pragma unroll
        for (int j = 0; j < NJ; j++) ka[j] = *(const v8f16*)(kl + key * HD * 2 + (((4 * j + g) ^ (key & 7)) << 4));
        // (the remainders' products first, then two chains: fewer additions at the size of the whole sum)
#pragma unroll
        for (int j = 0; j < NJ; j++) sc[k] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ka[j], __builtin_bit_cast(v8f16, qr[j]), sc[k], 0, 0, 0);
        v4f32 s2 = v4f32{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < NJ / 2; j++) {
          sc[k] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ka[j], __builtin_bit_cast(v8f16, qb[j]), sc[k], 0, 0, 0);
          s2 = __builtin_amdgcn_mfma_f32_16x16x32_f16(ka[NJ / 2 + j], __builtin_bit_cast(v8f16, qb[NJ / 2 + j]), s2, 0, 0, 0);
        }
        sc[k] += s2;
      }
      float m = -INFINITY;
      const bool mask = 64 * t + 63 > first_wave;
#pragma unroll
      for (int k = 0; k < 4; k++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          float s = sc[k][i];
          if (mask) s = 64 * t + 16 * k + 4 * g + i <= pos ? s : -INFINITY;
          sc[k][i] = s; m = fmaxf(m, s);
        }
      m = fmaxf(m, __shfl_xor(m, 16)); m = fmaxf(m, __shfl_xor(m, 32));
      const float mt = fmaxf(M, m * a.scale);                              // (log2(e) folded into the scale)
      const float mn = NG > 1 && mt == -INFINITY ? 0.f : mt;              // (key 0 is visible to every row, but none of the other part's may be)
      const float alpha = __builtin_amdgcn_exp2f(M - mn);
      float l = 0.f;
      u32x4 ph[2], pl[2];
#pragma unroll
      for (int u = 0; u < 2; u++)
#pragma unroll
        for (int w = 0; w < 4; w++) {
          const int k = 2 * u + (w >> 1), i = 2 * (w & 1);
          const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[k][i], a.scale, -mn)), p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[k][i + 1], a.scale, -mn));
          l += p0 + p1;
          const float q0 = p0 * PSCALE, q1 = p1 * PSCALE;
          const _Float16 h0 = (_Float16)q0, h1 = (_Float16)q1;
          ph[u][w] = (uint32_t)__builtin_bit_cast(uint16_t, h0) | ((uint32_t)__builtin_bit_cast(uint16_t, h1) << 16);
          pl[u][w] = f2h_bits(q0 - (float)h0) | (f2h_bits(q1 - (float)h1) << 16);
        }
      l += __shfl_xor(l, 16); l += __shfl_xor(l, 32);
      L = L * alpha + l; M = mt;
#pragma unroll
      for (int h = 0; h < NH; h++) {
        // (the tile's products sum from zero, remainders first: one addition at the size of the whole sum)
        v8f16 va[2]; v4f32 o = v4f32{0.f, 0.f, 0.f, 0.f};
        const int d = 16 * h + c;
#pragma unroll
        for (int u = 0; u < 2; u++) va[u] = *(const v8f16*)(vl + d * 128 + (((4 * u + g) ^ ((d ^ (d >> 3)) & 7)) << 4));
#pragma unroll
        for (int u = 0; u < 2; u++) o = __builtin_amdgcn_mfma_f32_16x16x32_f16(va[u], __builtin_bit_cast(v8f16, pl[u]), o, 0, 0, 0);
#pragma unroll
        for (int u = 0; u < 2; u++) o = __builtin_amdgcn_mfma_f32_16x16x32_f16(va[u], __builtin_bit_cast(v8f16, ph[u]), o, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; i++) O[h][i] = __builtin_fmaf(O[h][i], alpha, o[i]);
      }
    }
    __syncthreads();
  }
  if constexpr (NG > 1) {                                                 // the other part's sums, by way of LDS
    f32x4* const so = (f32x4*)kl_ + wave * NH * 64 + lane; float* const sm = (float*)vl_ + tid * 2;
    if (part_) {
#pragma unroll
      for (int h = 0; h < NH; h++) so[h * 64] = f32x4{O[h][0], O[h][1], O[h][2], O[h][3]};
      sm[0] = M; sm[1] = L;
    }
    __syncthreads();
    if (part_) return;
    const float mt = fmaxf(M, sm[0]), f0 = __builtin_amdgcn_exp2f(M - mt), f1 = __builtin_amdgcn_exp2f(sm[0] - mt);
    L = L * f0 + sm[1] * f1;
#pragma unroll
    for (int h = 0; h < NH; h++) {
      const f32x4 o = so[h * 64];
#pragma unroll
      for (int i = 0; i < 4; i++) O[h][i] = __builtin_fmaf(O[h][i], f0, o[i] * f1);
    }
  }
  if (wrow + c < a.P) {
    const float inv = (1.0f / PSCALE) / L;
    uint16_t* o = a.out + ((size_t)z * a.P + wrow + c) * nq + head * HD + 4 * g;
#pragma unroll
    for (int h = 0; h < NH; h++) *(u32x2*)(o + 16 * h) = u32x2{f2h_bits(O[h][0] * inv) | (f2h_bits(O[h][1] * inv) << 16), f2h_bits(O[h][2] * inv) | (f2h_bits(O[h][3] * inv) << 16)};
  }
}

// ------------------------------------------------------------------------------------------------ grouping of the routed rows by expert
#define PF_MAX_E 512
// One wave per token: selection and weights (gate_topk_wave), and this assignment's place among the rows of its expert.  The order of places is that of arrival: a row's
// values do not depend on its place, and the weighted sum of a token runs over its slots in order.  A workgroup counts its tokens' assignments in LDS and adds them up in one go (an addition per
// assignment: the two lines that 64 counts are in were what all waves waited for; 508 rows of 64 experts, top 8: 11.6 -> 4.8 us).  T tokens a workgroup: sixteen where a wave gates in registers; by way of LDS its
// reads are what bounds it - all waves of a CU share them - and fewer tokens a workgroup spread them.  us with 4 / 8 / 16 tokens a workgroup, 100 and 1024 rows: 64 experts, 24 taken 5.8 / 5.9 / 7.1, 9.9 / 7.6 / 7.4;
// 96, 8 taken 8.7 / 9.6 / 12.1, 13.1 / 11.0 / 12.3; 128, 8 taken 10.8 / 11.1 / 14.4, 14.5 / 12.7 / 14.6; 160, 6 taken 16.8 / 17.6 / 22.8, 20.0 / 19.0 / 23.1; 256, 8 taken 30.4 / 32.0 / 42.5, 33.3 / 33.2 / 42.9;
// 512, 10 taken 106.5 / 114.0 / 153.5, 107.3 / 114.4 / 153.2.
template <int T>
__global__ __launch_bounds__(64 * T) void rows_gate_kernel(const float* __restrict__ logits, int R, int E, int k, int gating, int norm_topk, float scale, int* __restrict__ sel,
                                                        float* __restrict__ probs, int* __restrict__ counts, int* __restrict__ place) {
  __shared__ float sc[T][PF_MAX_E]; __shared__ float tmp[T][192];
  __shared__ int s_count[PF_MAX_E];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, t = blockIdx.x * T + wave;
  for (int i = tid; i < E; i += 64 * T) s_count[i] = 0;
  if (t < R) gate_topk_wave(logits + (size_t)t * E, E, k, gating, norm_topk, scale, sel + (size_t)t * k, probs + (size_t)t * k, sc[wave], tmp[wave], lane);
  __syncthreads();
  const bool has = t < R && lane < k;
  int e = 0, at = 0;
  if (has) { e = ((const int*)tmp[wave])[lane]; at = atomicAdd(&s_count[e], 1); }
  __syncthreads();
  for (int i = tid; i < E; i += 64 * T) if (s_count[i]) s_count[i] = atomicAdd(&counts[i], s_count[i]);
  __syncthreads();
  if (has) place[(size_t)t * k + lane] = s_count[e] + at;
}
// Offsets of the experts' rows, the list of tiles of tt rows, and every row's token and assignment; each workgroup scans the counts for itself, the first writes the lists
__global__ __launch_bounds__(512) void rows_group_kernel(const int* __restrict__ counts, const int* __restrict__ sel, const int* __restrict__ place, int R, int E, int k, int tt,
                                                         int* __restrict__ off, int2* __restrict__ tiles, int* __restrict__ n_tiles, int* __restrict__ row_tok, int* __restrict__ row_dst) {
  __shared__ int s_off[PF_MAX_E + 1], s_t[8], s_o[8];
  const int e = threadIdx.x, lane = e & 63, wave = e >> 6;
  const int c = e < E ? counts[e] : 0, nt = (c + tt - 1) / tt;
  int io = c, it = nt;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) { const int uo = __shfl_up(io, o), ut = __shfl_up(it, o); if (lane >= o) { io += uo; it += ut; } }
  if (lane == 63) { s_o[wave] = io; s_t[wave] = it; }
  __syncthreads();
  for (int w = 0; w < wave; w++) { io += s_o[w]; it += s_t[w]; }
  if (e < E) s_off[e] = io - c;
  __syncthreads();
  if (blockIdx.x == 0) {
    if (e < E) {
      off[e] = io - c;
      for (int i = 0; i < nt; i++) tiles[it - nt + i] = int2{e, i * tt};
      if (e == E - 1) { off[E] = io; *n_tiles = it; }
    }
  }
  const int n = R * k;
  for (int j = blockIdx.x * 512 + threadIdx.x; j < n; j += gridDim.x * 512) {
    const int row = s_off[sel[j]] + place[j];
    row_tok[row] = j / k; row_dst[row] = j;
  }
}

int pf_gate(const float* logits, int R, int E, int k, int gating, int norm_topk, float scale, int* sel, float* probs, int* counts, int* place, hipStream_t s) {
#define PF_GATE(T) rows_gate_kernel<T><<<(unsigned)((R + T - 1) / T), 64 * T, 0, s>>>(logits, R, E, k, gating, norm_topk, scale, sel, probs, counts, place)
  if (gate_in_lanes(E, k)) PF_GATE(16); else if (E <= 64) PF_GATE(8); else PF_GATE(4);
#undef PF_GATE
  TGA_LAUNCH_CHECK();
  return 0;
}
static int pf_group(const int* counts, const int* sel, const int* place, int R, int E, int k, int tt, int* off, int2* tiles, int* n_tiles, int* row_tok, int* row_dst, hipStream_t s) {
  const int64_t gb = ((int64_t)R * k + 511) / 512;
  rows_group_kernel<<<(unsigned)(gb < 64 ? gb : 64), 512, 0, s>>>(counts, sel, place, R, E, k, tt, off, tiles, n_tiles, row_tok, row_dst);
  TGA_LAUNCH_CHECK();
  return 0;
}

// ------------------------------------------------------------------------------------------------ the step
#define PF_PART ((size_t)64 << 20)            // partial tiles of a split K

struct PfWs { size_t x, xn, q, k, v, qh, ql, attn, act, part, logits, sel, probs, place, counts, off, tiles, ntiles, row_tok, row_dst, act_e, y_e, total; };
static PfWs pf_layout(const int64_t* m, int64_t R) {
  PfWs w = {}; size_t o = 0;
  auto take = [&](size_t n) { const size_t at = o; o += (n + 255) & ~(size_t)255; return at; };
  const int64_t dim = m[PM_DIM], nq = m[PM_HEADS] * m[PM_HD], nk = m[PM_KV] * m[PM_HD], E = m[PM_EXPERTS], k = m[PM_TOPK];
  const int64_t h = E ? m[PM_DENSE_HIDDEN] : m[PM_HIDDEN];
  w.x = take(R * dim * 4); w.xn = take(R * dim * 2); w.q = take(R * nq * 4); w.k = take(R * nk * 4); w.v = take(R * nk * 4); w.qh = take(R * nq * 2); w.ql = take(R * nq * 2);
  w.attn = take(R * nq * 2); w.act = take(R * (h > 0 ? h : 1) * 2);
  w.part = take(PF_PART);
  if (E) {
    w.logits = take(R * E * 4); w.sel = take(R * k * 4); w.probs = take(R * k * 4); w.place = take(R * k * 4); w.counts = take(E * 4); w.off = take((E + 1) * 4);
    w.tiles = take((R * k / 32 + E + 1) * 8); w.ntiles = take(4); w.row_tok = take(R * k * 4); w.row_dst = take(R * k * 4);
    w.act_e = take(R * k * m[PM_HIDDEN] * 2); w.y_e = take(R * k * dim * 4);
  }
  w.total = o;
  return w;
}

// one expert-grouped product over the tiles rows_group_kernel listed; up != nullptr: silu(gate) * up
static int pf_experts(int type, const void* wgt, const void* up, int64_t N, int64_t K, const uint16_t* x, void* y, int y_f32, int tt, int64_t max_tiles, const int2* tiles, const int* n_tiles,
                      const int* off, const int* row_tok, const int* row_dst, hipStream_t s) {
  RowsArgs a = {};
  const int fmt = tga_rows_fmt(type, K);
  a.w[0] = (const uint8_t*)wgt; a.w[1] = (const uint8_t*)up; a.y[0] = y; a.n[0] = N; a.n[1] = N; a.ntot = N; a.row_bytes = tga_rows_row_bytes(fmt, K); a.estride = a.row_bytes * N;
  a.x = x; a.nseg = 1; a.epi = up ? ROWS_SWIGLU : ROWS_PLAIN; a.y_f32 = y_f32; a.K = (int)K; a.ks = 1;
  const int per = up ? ROWS_WT / 2 : ROWS_WT;
  a.row_tiles = (int)((N + per - 1) / per);
  a.tiles = tiles; a.n_tiles = n_tiles; a.off = off; a.row_tok = row_tok; a.row_dst = row_dst;
  return tga_rows_dispatch(fmt, a, tt, (unsigned)((max_tiles * a.row_tiles + 7) / 8 * 8), s);
}

extern "C" {

int tga_prefill_plan(const int64_t* model, int64_t rows, int64_t* nbytes) {
  TGA_REQUIRE(model && nbytes && rows >= 1, "tga_prefill_plan: null pointer or no rows");
  *nbytes = (int64_t)pf_layout(model, rows).total;
  return 0;
}

int tga_rows_format_ok(int ggml_type, int64_t K, int* ok) { TGA_REQUIRE(ok, "tga_rows_format_ok: null pointer"); *ok = tga_rows_fmt(ggml_type, K) >= 0; return 0; }

int tga_prefill_step(const int64_t* m, const int64_t* blocks, const int32_t* tokens, int64_t nseq, int64_t P, int64_t pos0, void* workspace, void* state, void* stream) {
  TGA_REQUIRE(m && blocks && tokens && workspace && state && nseq >= 1 && P >= 1 && pos0 >= 0 && pos0 + P <= m[PM_MAXCTX], "tga_prefill_step: null pointer or rows beyond the cache");
  const int64_t R = nseq * P, dim = m[PM_DIM], H = m[PM_HEADS], KV = m[PM_KV], hd = m[PM_HD], nq = H * hd, nk = KV * hd, E = m[PM_EXPERTS], k = m[PM_TOPK];
  TGA_REQUIRE((hd == 64 || hd == 128) && KV > 0 && H % KV == 0 && E <= PF_MAX_E && k <= 64 && R < (1 << 20), "tga_prefill_step: geometry outside the range");
  // (the kernels form the place of an activation row, row * values, in 32 bits)
  const int64_t hidden = m[PM_HIDDEN];
  TGA_REQUIRE(R * dim < (1ll << 32) && R * nq < (1ll << 32) && R * (E ? m[PM_DENSE_HIDDEN] : hidden) < (1ll << 32), "tga_prefill_step: %lld rows of that model are more than a step takes", (long long)R);
  TGA_REQUIRE(!E || (k >= 1 && k <= E && hidden >= 1 && R * k * hidden < (1ll << 32)), "tga_prefill_step: %lld rows of %lld of %lld experts are more than a step takes", (long long)R, (long long)k, (long long)E);
  TGA_REQUIRE(!E || (m[PM_GATING] >= 1 && m[PM_GATING] <= 4), "tga_prefill_step: unknown ExpertGating %lld", (long long)m[PM_GATING]);
  for (int64_t bi = 0; bi < m[PM_NBLOCKS]; bi++) {
    const int64_t* b = blocks + bi * PB_COUNT;
    TGA_REQUIRE(!b[PB_MOE] || (E && tga_rows_fmt((int)b[PB_TGATE], dim) >= 0 && tga_rows_fmt((int)b[PB_TDOWN], hidden) >= 0), "tga_prefill_step: the experts of block %lld are outside the range", (long long)bi);
  }
  const PfWs w = pf_layout(m, R);
  uint8_t* ws = (uint8_t*)workspace;
  float* x = (float*)(ws + w.x); uint16_t* xn = (uint16_t*)(ws + w.xn); float* q = (float*)(ws + w.q); float* kk = (float*)(ws + w.k); float* v = (float*)(ws + w.v);
  uint16_t* attn = (uint16_t*)(ws + w.attn); uint16_t* act = (uint16_t*)(ws + w.act);
  hipStream_t s = (hipStream_t)stream;
  const float eps = bits_f(m[PM_EPS_BITS]);
  int rc;
#define PF_DO(call) do { if ((rc = (call))) return rc; } while (0)
  auto linear = [&](int type, int nseg, const void* const* wt, void* const* y, const int64_t* n, const void* in, int ydt, int64_t K, int epi, const float* resid) {
    return tga_qlinear_many(type, nseg, wt, y, n, in, ydt, R, K, epi, resid, ws + w.part, (int64_t)PF_PART, stream);
  };
  // x += in . W^T, and xn = the norm that follows (norm nullptr: nothing follows)
  auto linear_norm = [&](int type, int64_t wp, const void* in, int64_t K, const float* norm) {
    const void* wt[1] = {(const void*)wp}; void* y[1] = {x}; const int64_t n[1] = {dim};
    return tga_rows_linear(type, 1, wt, y, n, in, TGA_F32, R, K, 1, x, ws + w.part, (int64_t)PF_PART, norm, eps, xn, nullptr, stream);
  };
  PF_DO(tga_embed_rows((const void*)m[PM_EMB], (int)m[PM_EMB_TYPE], (int)dim, tokens, (int)R, state, x, stream));
  for (int64_t bi = 0; bi < m[PM_NBLOCKS]; bi++) {
    const int64_t* b = blocks + bi * PB_COUNT;
    const bool pending = bi > 0 && blocks[(bi - 1) * PB_COUNT + PB_MOE];  // the block before left its weighted expert sum to this norm
    if (pending) PF_DO(tga_moe_combine_rmsnorm_rows((float*)(ws + w.y_e), (float*)(ws + w.probs), x, (const float*)b[PB_ATTN_NORM], (int)R, (int)k, (int)dim, eps, xn, nullptr, stream));
    else if (bi == 0) PF_DO(tga_rows_norm(x, (const float*)b[PB_ATTN_NORM], (int)R, (int)dim, eps, xn, stream));      // (later ones come behind the block before)
    const void* wt[3] = {(const void*)b[PB_WQ], (const void*)b[PB_WK], (const void*)b[PB_WV]};
    void* y[3] = {q, kk, v}; const int64_t n[3] = {nq, nk, nk};
    RopeArgs ra;
    ra.norm = !b[PB_QN] ? 0 : m[PM_QKNORM] == hd ? 2 : 1;
    RopeSrc* const src[3] = {&ra.q, &ra.k, &ra.v};
    int64_t used = 0;
    for (int i = 0; i < 3;) {                                             // one launch per run of equal block types
      int j = i + 1, ks = 1;
      while (j < 3 && b[PB_TQ + j] == b[PB_TQ + i]) j++;
      int64_t run = 0, at = 0;
      for (int l = i; l < j; l++) run += n[l];
      // (the rotation completes the sums itself where q and k are of one launch, and needs no norm over whole rows first)
      const bool leave = ra.norm != 1 && (i == 2 || (i == 0 && j >= 2));
      PF_DO(tga_rows_linear((int)b[PB_TQ + i], j - i, wt + i, y + i, n + i, xn, TGA_F32, R, dim, 0, nullptr, ws + w.part + used, (int64_t)PF_PART - used, nullptr, 0.f, nullptr, leave ? &ks : nullptr, stream));
      for (int l = i; l < j; at += n[l++]) *src[l] = ks > 1 ? RopeSrc{(const float*)(ws + w.part + used) + at, (size_t)(R * run), (int)run, ks} : RopeSrc{(const float*)y[l], 0, (int)n[l], 1};
      if (ks > 1) used += (ks * R * run * 4 + 255) & ~(int64_t)255;
      i = j;
    }
    ra.qn = (const float*)b[PB_QN]; ra.kn = (const float*)b[PB_KN]; ra.rope = (const float*)m[PM_ROPE];
    ra.qh = (uint16_t*)(ws + w.qh); ra.ql = (uint16_t*)(ws + w.ql); ra.ck = (uint16_t*)b[PB_CK]; ra.cv = (uint16_t*)b[PB_CV];
    ra.zero = b[PB_MOE] ? (int*)(ws + w.counts) : nullptr; ra.n_zero = b[PB_MOE] ? (int)E : 0;
    ra.H = (int)H; ra.KV = (int)KV; ra.hd = (int)hd; ra.max_ctx = (int)m[PM_MAXCTX]; ra.P = (int)P; ra.pos0 = (int)pos0; ra.eps = eps;
    rows_rope_launch(ra, (unsigned)R, s);
    TGA_LAUNCH_CHECK();
    // The last block's keys and values are in the cache, and the first logits come from the decode step behind the prompt: its rows go no further (8B-arch, 1024 tokens: 0.5 ms of 21).  A model of one
    // block takes the whole step: its workspace is where single blocks are compared with the reference
    if (bi > 0 && bi + 1 == m[PM_NBLOCKS]) break;
    RowsAttnArgs aa;
    aa.qh = ra.qh; aa.ql = ra.ql; aa.ck = ra.ck; aa.cv = ra.cv; aa.out = attn; aa.H = (int)H; aa.KV = (int)KV; aa.max_ctx = ra.max_ctx; aa.P = (int)P; aa.pos0 = (int)pos0; aa.nseq = (int)nseq;
    aa.qtiles = (int)((P + 63) / 64); aa.cus = (int)(H * nseq < 256 ? 256 / (H * nseq) : 1); aa.scale = (float)(1.4426950408889634 / sqrt((double)hd));
    const unsigned ag = (unsigned)(aa.qtiles * H * nseq);
    if (ag <= 256 ? (pos0 + P + 63) / 64 >= 4 : ag <= 512 && (pos0 + P + 63) / 64 >= 12) {
      aa.cus = aa.qtiles;                                                 // (one workgroup per CU: the longest first)
      if (hd == 64) rows_attn_kernel<64, 2><<<ag, 512, 0, s>>>(aa); else rows_attn_kernel<128, 2><<<ag, 512, 0, s>>>(aa);
    } else if (hd == 64) rows_attn_kernel<64, 1><<<ag, 256, 0, s>>>(aa); else rows_attn_kernel<128, 1><<<ag, 256, 0, s>>>(aa);
    TGA_LAUNCH_CHECK();
    PF_DO(linear_norm((int)b[PB_TO], b[PB_WO], attn, nq, (const float*)b[PB_FFN_NORM]));
    if (!b[PB_MOE]) {
      const int64_t h = E ? m[PM_DENSE_HIDDEN] : m[PM_HIDDEN];
      const void* wg[2] = {(const void*)b[PB_GATE], (const void*)b[PB_UP]}; void* yg[2] = {act, nullptr}; const int64_t ng[2] = {h, h};
      PF_DO(linear((int)b[PB_TGATE], 2, wg, yg, ng, xn, TGA_F16, dim, 2, nullptr));
      PF_DO(linear_norm((int)b[PB_TDOWN], b[PB_DOWN], act, h, bi + 1 < m[PM_NBLOCKS] ? (const float*)blocks[(bi + 1) * PB_COUNT + PB_ATTN_NORM] : nullptr));
      continue;
    }
    float* logits = (float*)(ws + w.logits); int* counts = (int*)(ws + w.counts); int* sel = (int*)(ws + w.sel); int* place = (int*)(ws + w.place);
    { const void* wr[1] = {(const void*)b[PB_ROUTER]}; void* yr[1] = {logits}; const int64_t nr[1] = {E}; PF_DO(linear(TGA_F16, 1, wr, yr, nr, xn, TGA_F32, dim, 0, nullptr)); }
    // Rows of an expert's tile, us a block with 32 / 64 / 128 (D 2048, H 1024, 64 experts, top 8 | H 1024, 16, top 8 | H 1536, 32, top 8): 24 rows per expert 189 / 185 / 226 | 107 / 112 / 125 | 159 / 152 / 186,
    // 32: 213 / 196 / 236 | 119 / 114 / 127 | 174 / 157 / 191, 80: 319 / 307 / 285 | 142 / 140 / 140 | 245 / 236 / 218, 104: 373 / 338 / 344 | 162 / 146 / 147 | 279 / 243 / 231, 160: 496 / 447 / 474 | 194 / 174 / 183 |
    // 350 / 314 / 332, 255: 712 / 632 / 630 | 243 / 222 / 232 | 484 / 426 / 427, 510: - | 377 / 338 / 337 | 860 / 738 / 712, 1000: - | 660 / 578 / 561; D 1024, H 512, 8 experts, top 4: 128 rows
    // 8 .. 14 % slower from 104 to 160, alike from 255 on.  At either line the sides are about a tenth apart, one way or the other.
    const int64_t avg = R * k / E;
    const int tt = avg <= 32 ? 32 : avg <= 96 ? 64 : 128;
    const int64_t max_tiles = R * k / tt + (R * k < E ? R * k : E);
    int2* tiles = (int2*)(ws + w.tiles); int* nt = (int*)(ws + w.ntiles); int* off = (int*)(ws + w.off); int* row_tok = (int*)(ws + w.row_tok); int* row_dst = (int*)(ws + w.row_dst);
    PF_DO(pf_gate(logits, (int)R, (int)E, (int)k, (int)m[PM_GATING], (int)m[PM_NORM_TOPK], bits_f(m[PM_SCALE_BITS]), sel, (float*)(ws + w.probs), counts, place, s));
    PF_DO(pf_group(counts, sel, place, (int)R, (int)E, (int)k, tt, off, tiles, nt, row_tok, row_dst, s));
    const int64_t hid = m[PM_HIDDEN];
    PF_DO(pf_experts((int)b[PB_TGATE], (const void*)b[PB_GATE], (const void*)b[PB_UP], hid, dim, xn, ws + w.act_e, 0, tt, max_tiles, tiles, nt, off, row_tok, nullptr, s));
    PF_DO(pf_experts((int)b[PB_TDOWN], (const void*)b[PB_DOWN], nullptr, dim, hid, (const uint16_t*)(ws + w.act_e), ws + w.y_e, 1, tt, max_tiles, tiles, nt, off, nullptr, row_dst, s));
  }
#undef PF_DO
  return 0;
}

}  // extern "C"
