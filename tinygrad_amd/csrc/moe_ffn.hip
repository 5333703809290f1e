// The grouped MoE feed-forward of an MXFP8 model (examples/mlperf/models/gpt_oss.py:213-226) as five launches over compact rows:
//   1. moe_prep_kernel      quantises the T input rows once (a token's row serves all of its experts) and, in other workgroups, picks each token's experts and gives every
//                           assignment its place among the rows of its expert
//   2. ffn_gemm_kernel<..., gate/up>   gathers the quantised rows by token, multiplies, adds the bias, applies the clamped interleaved SwiGLU and quantises the result
//   3. ffn_gemm_kernel<..., down>      multiplies and adds the bias; rows stay in expert order
//   4. moe_combine_kernel   weighs and sums the k rows of every token
// (+ a fill of the expert counters in front when more than one workgroup routes).  The values are those of route -> dispatch -> quantize_mxfp8 -> grouped_mx_gemm ->
// add_expert_bias -> swiglu -> quantize_mxfp8 -> grouped_mx_gemm -> add_expert_bias -> combine: every rounding to bf16 and to E4M3 sits where it sits there.  What
// is gone are the passes between them (T = 4096, k = 8, E = 128, D = 2048, I = 768: dispatch, two quantisations, two bias adds, SwiGLU over 65536 padded rows) and the
// padding of every expert's rows to 256, and the host work of eleven entry points.  MI355X, back to back: T = 2000, k = 8, E = 64, D = 2048, I = 512, popularity
// by 1 / rank^1.1: 2480 (single passes: 810) -> 182 -> 150 us; T = 32, k = 8, E = 64, I = 768: 840 (single) -> 77 -> 62 us; T = 4096, E = 128, I = 768: 1340 (single) -> 406 -> 370 us.  The second step of
// each: operands by direct-to-LDS loads instead of through registers, scales sixteen bytes a row, lower tiles, routing workgroups of 16 tokens.
#include "mxfp8.h"
#include "host.h"
#include <type_traits>

#define FFN_MAX_E 512             // experts (their counts and offsets sit in LDS)
#define FFN_MAX_K 64              // experts per token
#define FFN_TALL_STAGE (512 * 132)

struct FfnArgs {
  const uint16_t* x; const float* logits; const uint8_t* w[2]; const uint8_t* we8[2]; const float* bias[2];
  int T, D, I, E, k; float limit;
  // workspace
  uint8_t* xq; uint8_t* xe8; uint8_t* yq; uint8_t* ye8; uint16_t* z;
  int* counts;                    // [E] rows of each expert
  int* row_tok;                   // [E][T] the token of each row of each expert
  int* place_e; int* place;       // [T][k] expert of each assignment and its row among that expert's
  float* weights;                 // [T][k]
  uint16_t* out;
  int nq_blocks;                  // workgroups of moe_prep_kernel that quantise
  int prep_tokens;                // tokens of a routing workgroup
  int one_route_block;
};

// ---------------------------------------------------------------------------------------------------- routing + quantisation of the input
#define PREP_TOKENS 64            // most tokens of a routing workgroup of sixteen waves

template <int CTRL, int ROW_MASK> __device__ __forceinline__ uint32_t dpp_umax(uint32_t v) {
  const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROW_MASK, 0xF, false);
  return v > o ? v : o;
}
__device__ __forceinline__ uint32_t wave_umax(uint32_t v) {             // over the 64 lanes, uniform
  v = dpp_umax<0xB1, 0xF>(v); v = dpp_umax<0x4E, 0xF>(v); v = dpp_umax<0x141, 0xF>(v); v = dpp_umax<0x140, 0xF>(v); v = dpp_umax<0x142, 0xA>(v); v = dpp_umax<0x143, 0xC>(v);
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// Routing of one token by one wave: descending logits, the lower index first among equals (Tensor.topk's order), then the softmax over the k picked ones.  Lane l holds
// the logits l, l + 64, ... as order-preserving integers; a pick is one wave maximum of the values and one of the complemented indices (12 DPP steps).
template <int NV>
__device__ __forceinline__ void route_token(const FfnArgs& a, const int t, const int lane, int* ids) {
  uint32_t key[NV];
#pragma unroll
  for (int j = 0; j < NV; j++) {
    const int i = lane + 64 * j;
    const float x = i < a.E ? a.logits[(size_t)t * a.E + i] + 0.0f : 0.0f;     // (-0 becomes +0: equal values)
    const uint32_t u = __builtin_bit_cast(uint32_t, x);
    key[j] = i >= a.E ? 0u : x != x ? 1u : (u & 0x80000000u) ? ~u : u | 0x80000000u;   // 0: cannot be picked; a NaN ranks last
  }
  uint32_t mine = 0; int my_id = 0;                                     // lane s keeps pick s
  for (int s = 0; s < a.k; s++) {
    uint32_t m = 0;
#pragma unroll
    for (int j = 0; j < NV; j++) m = m > key[j] ? m : key[j];
    m = wave_umax(m);
    uint32_t ci = 0;                                                    // complement of the lowest index that holds the maximum
#pragma unroll
    for (int j = NV - 1; j >= 0; j--) if (key[j] == m) ci = 0x7fffffffu - (lane + 64 * j);
    const int id = (int)(0x7fffffffu - wave_umax(ci));
#pragma unroll
    for (int j = 0; j < NV; j++) if (lane + 64 * j == id) key[j] = 0;
    if (lane == s) { mine = m; my_id = id; }
  }
  const float v = __builtin_bit_cast(float, (mine & 0x80000000u) ? mine & 0x7fffffffu : ~mine);
  const float top = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v)));
  const float ex = expf(v - top);
  float z = 0.f;
  for (int j = 0; j < a.k; j++) z += __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, ex), j));
  if (lane < a.k) { a.weights[(size_t)t * a.k + lane] = ex * (1.0f / z); ids[lane] = my_id; }
}

template <int NV>
__global__ __launch_bounds__(1024) void moe_prep_kernel(const FfnArgs a) {
  if ((int)blockIdx.x < a.nq_blocks) {                                  // four lanes per block of 32 values, as quantize_mxfp8_kernel<1>
    const long long n8 = (long long)a.T * (a.D / 8);
    for (long long p = (long long)blockIdx.x * 1024 + threadIdx.x; p < n8; p += (long long)a.nq_blocks * 1024) {
      const u32x4 w = ((const u32x4*)a.x)[p];
      float v[8], amax = 0.f;
#pragma unroll
      for (int i = 0; i < 4; i++) { v[2 * i] = bf16_lo(w[i]); v[2 * i + 1] = bf16_hi(w[i]); }
#pragma unroll
      for (int i = 0; i < 8; i++) amax = fmaxf(amax, fabsf(v[i]));
      const int e = mx_e8(quad_max(amax));
      const float s = mx_scale(e);
      ((u32x2*)a.xq)[p] = u32x2{e4m3x4(v[0] * s, v[1] * s, v[2] * s, v[3] * s), e4m3x4(v[4] * s, v[5] * s, v[6] * s, v[7] * s)};
      if ((threadIdx.x & 3) == 0) a.xe8[p >> 2] = (uint8_t)e;
    }
    return;
  }
  __shared__ int ids[PREP_TOKENS * FFN_MAX_K];
  __shared__ int hist[FFN_MAX_E], base[FFN_MAX_E];
  const int t0 = ((int)blockIdx.x - a.nq_blocks) * a.prep_tokens, nt = min(a.prep_tokens, a.T - t0), n = nt * a.k;
  for (int e = threadIdx.x; e < a.E; e += 1024) hist[e] = 0;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  for (int i = wave; i < nt; i += 16) route_token<NV>(a, t0 + i, lane, ids + i * a.k);
  __syncthreads();
  int rank[PREP_TOKENS * FFN_MAX_K / 1024];
#pragma unroll
  for (int u = 0; u < PREP_TOKENS * FFN_MAX_K / 1024; u++) { const int i = threadIdx.x + 1024 * u; if (i < n) rank[u] = atomicAdd(&hist[ids[i]], 1); }
  __syncthreads();
  // places of one expert are taken in the order the workgroups arrive: which row a token gets does not change its values, and every token sums its rows in slot order
  for (int e = threadIdx.x; e < a.E; e += 1024) {
    const int c = hist[e];
    if (a.one_route_block) { a.counts[e] = c; base[e] = 0; }
    else if (c) base[e] = atomicAdd(&a.counts[e], c);
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < PREP_TOKENS * FFN_MAX_K / 1024; u++) {
    const int i = threadIdx.x + 1024 * u;
    if (i < n) {
      const int e = ids[i], r = base[e] + rank[u];
      a.row_tok[(size_t)e * a.T + r] = t0 + i / a.k;
      a.place_e[(size_t)t0 * a.k + i] = e; a.place[(size_t)t0 * a.k + i] = r;
    }
  }
}
__global__ __launch_bounds__(512) void moe_zero_counts_kernel(int* counts, int E) { if ((int)threadIdx.x < E) counts[threadIdx.x] = 0; }

// Exclusive prefix sums over the experts' counts and over their tiles of bm rows, by the first wave of a workgroup: off[e] = first row, tile[e] = first tile (off[E], tile[E]: the totals).
// tall: tiles of 256 rows instead, and *tall = 1, where their rounds of a launch of `grid` workgroups are at most five ninths of those of bm rows (see the dispatch); otherwise *tall = 0.
__device__ __forceinline__ void ffn_offsets(const int* __restrict__ counts, int E, int bm, int tiles_n, int* off, int* tile, int* tall = nullptr, int grid = 1) {
  const int lane = threadIdx.x;
  if (lane < 64) {
    constexpr int PER = FFN_MAX_E / 64;
    int c[PER], so = 0, st = 0, st2 = 0;
#pragma unroll
    for (int i = 0; i < PER; i++) {                                       // (one wait for all of them)
      const int e = lane * PER + i, v = counts[min(e, E - 1)];
      c[i] = e < E ? v : 0;
    }
#pragma unroll
    for (int i = 0; i < PER; i++) { so += c[i]; st += (c[i] + bm - 1) / bm * tiles_n; if (tall) st2 += (c[i] + 255) / 256 * tiles_n; }
    int io = so, it = st, it2 = st2;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int uo = __shfl_up(io, o), ut = __shfl_up(it, o), u2 = tall ? __shfl_up(it2, o) : 0;
      if (lane >= o) { io += uo; it += ut; it2 += u2; }
    }
    if (tall) {
      const int n = __builtin_amdgcn_readlane(it, 63), n2 = __builtin_amdgcn_readlane(it2, 63);
      const bool take = 9 * ((n2 + grid - 1) / grid) <= 5 * ((n + grid - 1) / grid);
      if (take) { bm = 256; it = it2; st = st2; }
      if (lane == 0) *tall = take;
    }
    io -= so; it -= st;
#pragma unroll
    for (int i = 0; i < PER; i++) {
      const int e = lane * PER + i;
      if (e <= E) { off[e] = io; if (tile) tile[e] = it; }
      io += c[i]; it += (c[i] + bm - 1) / bm * tiles_n;
      if (e == E - 1) { off[E] = io; if (tile) tile[E] = it; }
    }
  }
}

// ---------------------------------------------------------------------------------------------------- the two products
// The tile of BM x BN that a workgroup is at: expert, rows [m0, m0 + valid) of it from compact row row0 on, columns [BN tn, ...), first weight row
struct FfnCur { uint32_t boff; int e, m0, tn, valid, row0; };
template <int BM, int BN>
__device__ __forceinline__ void ffn_find(int E, int N, int tiles_n, const int* s_off, const int* s_tile, int tile, FfnCur& c) {
  const int lane = threadIdx.x & 63;
  int n = 0;                                                             // the expert whose tiles hold this one: the last that starts at or in front of it
  for (int e = 0; e < E; e += 64) n += __popcll(__ballot(e + lane < E && s_tile[e + lane] <= tile));
  const int lo = n - 1;
  const int i = tile - __builtin_amdgcn_readfirstlane(s_tile[lo]), tm = i / tiles_n, off = __builtin_amdgcn_readfirstlane(s_off[lo]);
  c.e = lo; c.tn = i - tm * tiles_n; c.m0 = tm * BM; c.valid = min(__builtin_amdgcn_readfirstlane(s_off[lo + 1]) - off - c.m0, BM);
  c.row0 = off + c.m0;
  c.boff = ((uint32_t)lo * (uint32_t)N + (uint32_t)c.tn * BN);
}

// fminf / fmaxf of values that are no signalling NaN (bf16 results of a conversion): one instruction, where the functions quieten their arguments first
__device__ __forceinline__ float min_q(float a, float b) { float o; asm("v_min_f32 %0, %1, %2" : "=v"(o) : "v"(a), "v"(b)); return o; }
__device__ __forceinline__ float max_q(float a, float b) { float o; asm("v_max_f32 %0, %1, %2" : "=v"(o) : "v"(a), "v"(b)); return o; }
__device__ __forceinline__ float max3_abs(float m, float a, float b) { float o; asm("v_max3_f32 %0, %1, |%2|, |%3|" : "=v"(o) : "v"(m), "v"(a), "v"(b)); return o; }

__device__ __forceinline__ float lanes_max(float v) {                     // over lanes l, l ^ 16, l ^ 32, l ^ 48; no signalling NaN
  const uint32_t u = __builtin_bit_cast(uint32_t, v);
  const auto h = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  const uint32_t m = __builtin_bit_cast(uint32_t, max_q(__builtin_bit_cast(float, (uint32_t)h[0]), __builtin_bit_cast(float, (uint32_t)h[1])));
  const auto l = __builtin_amdgcn_permlane16_swap(m, m, false, false);
  return max_q(__builtin_bit_cast(float, (uint32_t)l[0]), __builtin_bit_cast(float, (uint32_t)l[1]));
}

// The result of a tile: lane = row r16 of sub-tile WM i + wm, columns 4 kg .. 4 kg + 3 of n sub-tile j. b: the bias of its 64 columns.
// The four lanes of a row exchange their results in registers (a pass through LDS, with a barrier in front of it and a wait for the requests in flight that the compiler puts before its stores, and the
// bias rounded by integer code: 84 + 45.5 us of the first size below, now 82.7 + 45.2).
template <int RS, int WM, int BN, bool UP>
__device__ __forceinline__ void ffn_epilogue(const FfnArgs& a, const FfnCur& c, const v4f32 (&acc)[RS][4], int nsub, int wm, int wn, const float* b) {
  const int lane = threadIdx.x & 63, r16 = lane & 15, kg = lane >> 4, row0 = c.row0;
  const float limit = __builtin_canonicalizef(a.limit);
  f32x4 bias[4];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    bias[j] = *(const f32x4*)(b + 16 * j + 4 * kg);
    const uint32_t b01 = pack_bf16x2(bias[j][0], bias[j][1]), b23 = pack_bf16x2(bias[j][2], bias[j][3]);
    bias[j] = f32x4{bf16_lo(b01), bf16_hi(b01), bf16_lo(b23), bf16_hi(b23)};
  }
#pragma unroll
  for (int i = 0; i < RS; i++) {
    if (i >= nsub) break;
    const int r0 = 16 * (WM * i + wm);                                // first row of the sub-tile
    if constexpr (UP) {
      float y[8], amax = 0.f;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        // h = bf16(acc); h = bf16(h + bf16(bias)); then gate and up are neighbouring columns
        const uint32_t h01 = pack_bf16x2(acc[i][j][0], acc[i][j][1]), h23 = pack_bf16x2(acc[i][j][2], acc[i][j][3]);
        const uint32_t g01 = pack_bf16x2(bf16_lo(h01) + bias[j][0], bf16_hi(h01) + bias[j][1]), g23 = pack_bf16x2(bf16_lo(h23) + bias[j][2], bf16_hi(h23) + bias[j][3]);
        const float gl0 = min_q(bf16_lo(g01), limit), gl1 = min_q(bf16_lo(g23), limit);
        const float li0 = min_q(max_q(bf16_hi(g01), -limit), limit), li1 = min_q(max_q(bf16_hi(g23), -limit), limit);
        const uint32_t ag = pack_bf16x2(1.702f * gl0, 1.702f * gl1);
        const uint32_t sg = pack_bf16x2(mx_sigmoid_bf16(bf16_lo(ag)), mx_sigmoid_bf16(bf16_hi(ag)));
        const uint32_t p = pack_bf16x2(gl0 * bf16_lo(sg), gl1 * bf16_hi(sg)), q = pack_bf16x2(li0 + 1.0f, li1 + 1.0f);
        const uint32_t o = pack_bf16x2(bf16_lo(p) * bf16_lo(q), bf16_hi(p) * bf16_hi(q));
        y[2 * j] = bf16_lo(o); y[2 * j + 1] = bf16_hi(o);
        amax = max3_abs(amax, y[2 * j], y[2 * j + 1]);
      }
      amax = lanes_max(amax);     // the wave's 64 columns are one block of 32 results
      const int e = mx_e8(amax);
      const float sc = mx_scale(e);
      // two bytes of each of four n sub-tiles a lane -> the eight of n sub-tile kg: the rows' four lanes change places
      const auto h = __builtin_amdgcn_permlane32_swap(e4m3x4(y[0] * sc, y[1] * sc, y[2] * sc, y[3] * sc), e4m3x4(y[4] * sc, y[5] * sc, y[6] * sc, y[7] * sc), false, false);
      const auto l = __builtin_amdgcn_permlane16_swap(__builtin_amdgcn_perm(h[1], h[0], 0x05040100u), __builtin_amdgcn_perm(h[1], h[0], 0x07060302u), false, false);
      const u32x2 o = {__builtin_amdgcn_perm(l[1], l[0], 0x05040100u), __builtin_amdgcn_perm(l[1], l[0], 0x07060302u)};
      if (r0 + r16 < c.valid) {
        const size_t row = (size_t)(row0 + r0 + r16);
        *(u32x2*)(a.yq + row * a.I + c.tn * (BN / 2) + wn * 32 + 8 * kg) = o;
        if (kg == 0) a.ye8[row * (a.I / 32) + c.tn * (BN / 64) + wn] = (uint8_t)e;
      }
    } else {
      u32x2 o[4];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const uint32_t h01 = pack_bf16x2(acc[i][j][0], acc[i][j][1]), h23 = pack_bf16x2(acc[i][j][2], acc[i][j][3]);
        o[j] = u32x2{pack_bf16x2(bf16_lo(h01) + bias[j][0], bf16_hi(h01) + bias[j][1]), pack_bf16x2(bf16_lo(h23) + bias[j][2], bf16_hi(h23) + bias[j][3])};
      }
      uint16_t* to = (uint16_t*)a.z + (size_t)(row0 + r0 + r16) * a.D + c.tn * BN + wn * 64 + 16 * (kg & 1) + 4 * (kg & 2);
      u32x4 q[2];
#pragma unroll
      for (int p = 0; p < 2; p++) {                                      // an even lane group: eight columns of sub-tile 2 p, its own and the next group's; an odd one: of 2 p + 1
        const auto x = __builtin_amdgcn_permlane16_swap(o[2 * p].x, o[2 * p + 1].x, false, false), y = __builtin_amdgcn_permlane16_swap(o[2 * p].y, o[2 * p + 1].y, false, false);
        q[p] = u32x4{x[0], y[0], x[1], y[1]};
      }
      if (r0 + r16 < c.valid) { *(u32x4*)to = q[0]; *(u32x4*)(to + 32) = q[1]; }
    }
  }
}

// Tiles of 256 x 256, two steps in LDS, the next one through registers: half as many tiles as above, each 1.6 times as long.
template <bool UP>
__device__ __forceinline__ void ffn_tall(const FfnArgs& a, uint8_t* smem, int* s_row, const int* s_off, const int* s_tile) {
  constexpr int BM = 256, BN = 256, WM = 2, NT = 512, RS = 8;            // threads, 16-row sub-tiles of a wave
  constexpr int PA = BM * 8 / NT, PB = BN * 8 / NT, NS = (BM + BN + NT - 1) / NT;   // 16-byte pieces and scale dwords per thread and step
  constexpr int STAGE = FFN_TALL_STAGE;
  constexpr int RPT = NT / 8;                                            // rows between a thread's pieces
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 2, wn = wave & 3, r16 = lane & 15, kg = lane >> 4;
  const int N = UP ? 2 * a.I : a.D, K = UP ? a.D : a.I, KB = K / 32, nsteps = K / 128, tiles_n = N / BN;
  const uint8_t* __restrict__ A = UP ? a.xq : a.yq; const uint8_t* __restrict__ Ae = UP ? a.xe8 : a.ye8;
  const uint8_t* __restrict__ B = a.w[UP ? 0 : 1]; const uint8_t* __restrict__ Be = a.we8[UP ? 0 : 1];
  const int ntiles = __builtin_amdgcn_readfirstlane(s_tile[a.E]);
  const int per = (ntiles + 7) >> 3;                                     // tiles of an XCD's run
  const int first = ((int)blockIdx.x & 7) * per, last = min(first + per, ntiles), step_wg = (int)(gridDim.x + 7 - (blockIdx.x & 7)) >> 3;
  int t = first + ((int)blockIdx.x >> 3);
  if (t >= last) return;

  const int cpy_c = tid & 7, cpy_r = tid >> 3, slot0 = gg_slot_off(cpy_r, cpy_c);     // (RPT rows further on: RPT * 128 bytes)
  const int f0 = ((16 * kg + (r16 ^ kg)) << 4), f1 = 1024 + ((16 * kg + (r16 ^ (kg + 4))) << 4);

  auto setup = [&](int tile, FfnCur& c, int which) __attribute__((always_inline)) {
    ffn_find<BM, BN>(a.E, N, tiles_n, s_off, s_tile, tile, c);
    if (tid < BM) { const int r = min(tid, c.valid - 1); s_row[which * BM + tid] = UP ? a.row_tok[(size_t)c.e * a.T + c.m0 + r] : c.row0 + r; }   // rows beyond the expert's repeat its last one (their results are dropped)
  };
  u32x4 va[PA], vb[PB]; uint32_t vs[NS];
  auto load_a = [&](int which, int s, int j) __attribute__((always_inline)) { va[j] = *(const u32x4*)(A + (size_t)(uint32_t)s_row[which * BM + cpy_r + RPT * j] * K + (uint32_t)(s * 128 + cpy_c * 16)); };
  auto load_b = [&](const FfnCur& c, int s, int j) __attribute__((always_inline)) {
    vb[j] = *(const u32x4*)(B + (size_t)(c.boff + RPT * j) * K + (uint32_t)cpy_r * (uint32_t)K + (uint32_t)(s * 128 + cpy_c * 16));
  };
  auto load_s = [&](const FfnCur& c, int which, int s) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NS; j++) {
      const int i = tid + NT * j;
      const uint8_t* p = i < BM ? Ae + (size_t)(uint32_t)s_row[which * BM + i] * KB : Be + (size_t)(c.boff + (uint32_t)min(i - BM, BN - 1)) * KB;
      vs[j] = *(const uint32_t*)(p + 4 * s);
    }
  };
  auto store_a = [&](uint8_t* st, int j) __attribute__((always_inline)) { *(u32x4*)(st + slot0 + RPT * 128 * j) = va[j]; };
  auto store_b = [&](uint8_t* st, int j) __attribute__((always_inline)) { *(u32x4*)(st + BM * 128 + slot0 + RPT * 128 * j) = vb[j]; };
  auto store_s = [&](uint8_t* st) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NS; j++) { const int i = tid + NT * j; if (i < BM + BN) ((uint32_t*)(st + (BM + BN) * 128))[i] = vs[j]; }
  };

  FfnCur cur, nxt;
  int which = 0;
  setup(t, cur, 0);
  __syncthreads();
  load_s(cur, 0, 0);
#pragma unroll
  for (int j = 0; j < PA; j++) load_a(0, 0, j);
#pragma unroll
  for (int j = 0; j < PB; j++) load_b(cur, 0, j);
#pragma unroll
  for (int j = 0; j < PA; j++) store_a(smem, j);
#pragma unroll
  for (int j = 0; j < PB; j++) store_b(smem, j);
  store_s(smem);
  __syncthreads();
  int par = 0;
  while (true) {
    const int tnext = t + step_wg;
    const bool more = tnext < last;
    nxt = cur;
    if (more) setup(tnext, nxt, which ^ 1);
    v4f32 acc[RS][4];
#pragma unroll
    for (int i = 0; i < RS; i++)
#pragma unroll
      for (int j = 0; j < 4; j++) acc[i][j] = v4f32{0.f, 0.f, 0.f, 0.f};
    const int nsub = (((cur.valid + 15) >> 4) - wm + WM - 1) / WM;        // sub-tiles wm, wm + WM, ... of this wave that hold rows
    for (int s = 0; s < nsteps; s++) {
      uint8_t* st = smem + ((par + s) & 1) * STAGE; uint8_t* st2 = smem + ((par + s + 1) & 1) * STAGE;
      const bool lastk = s + 1 == nsteps;
      const int ls = lastk ? (more ? 0 : s) : s + 1;
      FfnCur src = cur;
      if (lastk) src = nxt;                                               // (the barriers of the steps before lie between setup() and this; K has at least two steps)
      const int sw = lastk && more ? which ^ 1 : which;
      load_s(src, sw, ls);
#pragma unroll
      for (int j = 0; j < PA; j++) load_a(sw, ls, j);
#pragma unroll
      for (int j = 0; j < PB; j++) load_b(src, ls, j);
      __builtin_amdgcn_sched_barrier(0);
      const uint8_t* As = st; const uint8_t* Bs = st + BM * 128 + wn * 4 * 2048;
      const uint32_t* sA = (const uint32_t*)(st + (BM + BN) * 128) + r16; const uint32_t* sB = sA + BM + wn * 64;
      if (nsub > 0) {
        v8i32 bf[4]; int sb[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const u32x4 y0 = *(const u32x4*)(Bs + j * 2048 + f0), y1 = *(const u32x4*)(Bs + j * 2048 + f1);
          bf[j] = v8i32{(int)y0.x, (int)y0.y, (int)y0.z, (int)y0.w, (int)y1.x, (int)y1.y, (int)y1.z, (int)y1.w};
          sb[j] = (int)(sB[16 * j] >> (8 * kg));
        }
        auto frag = [&](int i, v8i32& af, int& sa) __attribute__((always_inline)) {
          const uint8_t* p = As + (WM * i + wm) * 2048;
          const u32x4 x0 = *(const u32x4*)(p + f0), x1 = *(const u32x4*)(p + f1);
          af = v8i32{(int)x0.x, (int)x0.y, (int)x0.z, (int)x0.w, (int)x1.x, (int)x1.y, (int)x1.z, (int)x1.w};
          sa = (int)sA[16 * (WM * i + wm)];
        };
        v8i32 af[2]; int sa[2];
        frag(0, af[0], sa[0]);
#pragma unroll
        for (int i = 0; i < RS; i++) {
          if (i + 1 < nsub) frag(i + 1, af[(i + 1) & 1], sa[(i + 1) & 1]);
          if (i < nsub) {
            const int sai = sa[i & 1] >> (8 * kg);
#pragma unroll
            for (int j = 0; j < 4; j++) acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(bf[j], af[i & 1], acc[i][j], 0, 0, 0, sb[j], 0, sai);
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < PA; j++) store_a(st2, j);
#pragma unroll
      for (int j = 0; j < PB; j++) store_b(st2, j);
      store_s(st2);
      __syncthreads();
    }
    ffn_epilogue<RS, WM, BN, UP>(a, cur, acc, nsub, wm, wn, a.bias[UP ? 0 : 1] + (size_t)cur.e * N + cur.tn * BN + wn * 64);
    if (!more) break;
    par = (par + nsteps) & 1; cur = nxt; t = tnext; which ^= 1;
  }
}

// Tile of BM rows x 64 WN weight rows, K steps of 128, WM x WN waves of (BM / WM) x 64, weights as the A operand of the scaled MFMA, so a lane holds four consecutive
// output columns of one row.  The 16-row sub-tiles are dealt to the WM waves alternately and only those that hold rows are multiplied.  A workgroup walks tiles b,
// b + gridDim.x, ...: consecutive tiles of an expert share its weight or activation rows, and the workgroups of an XCD (b % 8) take a contiguous run of tiles.
// Operands go to a ring of NB steps in LDS by direct-to-LDS loads, NB - 1 steps ahead of the multiplication and across tile borders: one barrier per step, no registers in between.
// A step's region: rows of 128 bytes, 16-byte chunk c of row R at chunk c ^ (R & 7) (a request covers eight whole rows, a read of sixteen rows meets each bank group once
// per eight lanes).  Scales come four steps at a time, sixteen bytes a row: a dword a row and step was 64 cache lines a request, a fifth of the time.  Rows beyond the expert's repeat its last one.
// UP: gate/up (rows gathered by token, epilogue bias + clamped interleaved SwiGLU + quantisation) or down (compact rows, epilogue bias).  ONCE: weights requested past the caches.
// In full tiles of 128 rows the requests of a step go out between its products (in front of them 82.7 -> 80.0 + 44.8), and the scales' position in the row's sixteen bytes is a selector of the
// byte permutation, not a branch per row (sixteen branches every four steps: -> 76.6 + 44.0).
// Measured (us, gate/up + down): 16000 rows of 64 experts skewed, D 2048, I 512, tiles of 128: 97.5 + 52.7 (tiles of 256 through registers) -> 76.6 + 44.0; 256 rows of 64 experts, I 768, tiles of 16:
// 42.1 + 23.3 -> 35.8 + 20.2, past the caches 31.5 + 19.1: 5.2 TB/s of weights.  What bounds the first: of 77 us, requests alone are 45 (14 TB/s out of L2), products and reads alone 44, the launch
// itself 10, the epilogue 11 (down: 11 of 44, most of it the 64 MB it writes); what overlaps is what the two waves of a SIMD leave each other.  Not kept: two groups of waves half a step apart with a
// barrier each half (77 + 44 where one was 79 + 42), the next step's weights read into registers while this one is multiplied (81 + 46.5), a last round of half tiles (78.4 + 44.6), tiles of 128 x 128
// by four waves, two a CU (115).
__device__ __forceinline__ const uint8_t* scalar_ptr(const uint8_t* p) {
  const uint64_t v = (uint64_t)(uintptr_t)p;
  uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v), hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
  asm("" : "+s"(lo), "+s"(hi));
  return (const uint8_t*)(uintptr_t)(((uint64_t)hi << 32) | lo);
}
template <int N> __device__ __forceinline__ void ffn_wait_vm() { asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory"); }

template <int BM, int WM, int WN, int NB, bool UP, bool ONCE>
__global__ __launch_bounds__(64 * WM * WN) void ffn_gemm_kernel(const FfnArgs a) {
  constexpr int NW = WM * WN, BN = 64 * WN, RS = BM / 16 / WM;          // waves, weight rows of a tile, 16-row sub-tiles of a wave
  constexpr int IA = BM / 8 / NW, IB = BN / 8 / NW, SI = (BM + BN + 63) / 64, IS = (SI + NW - 1) / NW, NI = IA + IB;   // requests of a wave: eight rows of operands a step, 64 rows' scales of four steps
  constexpr int STAGE = (BM + BN) * 128;
  constexpr bool SPREAD = RS == 4;                                       // a full tile's requests between its products
  static_assert(IA * 8 * NW == BM && IB * 8 * NW == BN && RS >= 1 && (NB == 2 || NB == 3), "tile shape");
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];        // NB steps, the scales of up to four steps, the experts' first rows and tiles
  __shared__ __attribute__((aligned(16))) float s_bias[2][BN];          // of the tile multiplied and the one requested
  __shared__ __attribute__((aligned(16))) int s_ids[UP ? NW : 1][UP ? 8 * IA + 64 * IS : 1];   // tokens of the rows this wave requests: operands, scales (its own: no barrier between their arrival and their use)
  uint8_t* const scales = smem + NB * STAGE;
  int* const s_off = (int*)(scales + (BM + BN) * 16); int* const s_tile = s_off + a.E + 1;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN, r16 = lane & 15, kg = lane >> 4;
  const int N = UP ? 2 * a.I : a.D, K = UP ? a.D : a.I, KB = K / 32, nsteps = K / 128, tiles_n = N / BN;
  const uint8_t* __restrict__ A = UP ? a.xq : a.yq; const uint8_t* __restrict__ Ae = UP ? a.xe8 : a.ye8;
  const uint8_t* __restrict__ B = a.w[UP ? 0 : 1]; const uint8_t* __restrict__ Be = a.we8[UP ? 0 : 1];
  if constexpr (BM == 128) {                                             // tall tiles where they nearly halve the rounds of the launch: see the dispatch
    __shared__ int s_tall;
    ffn_offsets(a.counts, a.E, BM, tiles_n, s_off, s_tile, &s_tall, (int)gridDim.x);
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(s_tall)) { ffn_tall<UP>(a, smem, (int*)(smem + 2 * FFN_TALL_STAGE), s_off, s_tile); return; }
  } else { ffn_offsets(a.counts, a.E, BM, tiles_n, s_off, s_tile); __syncthreads(); }
  const int ntiles = __builtin_amdgcn_readfirstlane(s_tile[a.E]);
  const int per = (ntiles + 7) >> 3;                                     // tiles of an XCD's run
  const int first = ((int)blockIdx.x & 7) * per, last = min(first + per, ntiles), step_wg = (int)(gridDim.x + 7 - (blockIdx.x & 7)) >> 3;
  int t = first + ((int)blockIdx.x >> 3);
  if (t >= last) return;
  const long long total = (long long)((last - t + step_wg - 1) / step_wg) * nsteps;   // steps of this workgroup

  auto find = [&](int tile, FfnCur& c) __attribute__((always_inline)) { ffn_find<BM, BN>(a.E, N, tiles_n, s_off, s_tile, tile, c); };

  // ---- the requesting side: where it is, and this lane's addresses in that tile
  int rt_ = t, rs_ = 0, rslot = 0, rn = 0;                               // tile, step, ring position, tiles begun
  FfnCur rc_;                                                            // the tile that begins next
  const uint8_t* pa[IA]; const uint8_t* ps[IS]; const uint8_t* pb = nullptr;
  uint32_t boff_lane[IB];
#pragma unroll
  for (int i = 0; i < IB; i++) boff_lane[i] = (uint32_t)(8 * i + (lane >> 3)) * (uint32_t)K + (uint32_t)(((lane & 7) ^ (lane >> 3)) << 4);
  // UP: the tokens of a tile's rows, requested when the tile before it begins (a load whose result is waited for would wait for everything requested in front of it)
  auto request_ids = [&]() __attribute__((always_inline)) {
    const int* tok = a.row_tok + (size_t)rc_.e * a.T + rc_.m0;
    int* to = &s_ids[UP ? wave : 0][0];
    if (lane < 8 * IA) __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(tok + min(8 * IA * wave + lane, rc_.valid - 1)), (__attribute__((address_space(3))) void*)to, 4, 0, 0);
#pragma unroll
    for (int i = 0; i < IS; i++)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(tok + min(64 * min(wave * IS + i, SI - 1) + lane, rc_.valid - 1)), (__attribute__((address_space(3))) void*)(to + 8 * IA + 64 * i), 4, 0, 0);
  };
  auto begin = [&]() __attribute__((always_inline)) {
    const FfnCur c = rc_;
    // (read by inline assembly, its wait with it: in front of a plain read the compiler would wait for all requests in flight.  At rn = 0 they are waited for; later the wait of a step
    // behind the one they were requested at is behind this wave: a tile has at least two steps.)
    if constexpr (UP) { if (rn == 0) ffn_wait_vm<0>(); }
    const uint32_t ids = (uint32_t)(uintptr_t)&s_ids[UP ? wave : 0][0];
    auto row_of = [&](int r, int at) __attribute__((always_inline)) {     // row r of the tile, entry `at` of the list
      int id = c.row0 + min(r, c.valid - 1);
      if constexpr (UP) asm volatile("ds_read_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=v"(id) : "v"(ids + 4u * (uint32_t)at) : "memory");
      return (size_t)(uint32_t)id;
    };
#pragma unroll
    for (int i = 0; i < IA; i++) pa[i] = A + row_of(8 * (wave * IA + i) + (lane >> 3), 8 * i + (lane >> 3)) * K + (((lane & 7) ^ (lane >> 3)) << 4);
    pb = B + ((size_t)c.boff + (size_t)(wave * IB) * 8) * K;
#pragma unroll
    for (int i = 0; i < IS; i++) {
      const int r = 64 * min(wave * IS + i, SI - 1) + lane;              // (the last waves repeat the last request)
      const uint8_t* in_a = Ae + row_of(r, 8 * IA + 64 * i + lane) * KB;
      const uint8_t* in_b = Be + ((size_t)c.boff + (size_t)min(max(r - BM, 0), BN - 1)) * KB;
      ps[i] = r < BM ? in_a : in_b;
    }
    if (wave < WN) __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(a.bias[UP ? 0 : 1] + (size_t)c.e * N + (size_t)c.tn * BN + 64 * wave + lane),
                                                    (__attribute__((address_space(3))) void*)&s_bias[rn & 1][64 * wave], 4, 0, 0);
    rn++;
    if (rt_ + step_wg < last) { find(rt_ + step_wg, rc_); if constexpr (UP) request_ids(); }
  };
  // The scales of steps q .. q + 3 (a tile's last steps may be two), sixteen bytes a row.  A row's last eight bytes come with the eight in front of them; rows of eight bytes (K = 256) as two dwords,
  // each in a plane of its own.
  auto request_scales = [&](int q) __attribute__((always_inline)) {
    const int at = min(4 * q, KB - 16);
#pragma unroll
    for (int i = 0; i < IS; i++) {
      const int u = min(wave * IS + i, SI - 1);
      if ((BM + BN) % 64 == 0 || 64 * u + lane < BM + BN) {
        if (at >= 0) __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(ps[i] + at), (__attribute__((address_space(3))) void*)(scales + u * 1024), 16, 0, 0);
        else {
          __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)ps[i], (__attribute__((address_space(3))) void*)(scales + u * 256), 4, 0, 0);
          __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(ps[i] + 4), (__attribute__((address_space(3))) void*)(scales + (BM + BN) * 4 + u * 256), 4, 0, 0);
        }
      }
    }
  };
  // a step of the tile that is requested; q >= 0: the scales from that step on in front of it
  auto request_front = [&](int q) __attribute__((always_inline)) {
    if (rs_ == 0) begin();
    if (q >= 0) request_scales(q);
    uint8_t* st = smem + rslot * STAGE;
#pragma unroll
    for (int i = 0; i < IA; i++) __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)pa[i], (__attribute__((address_space(3))) void*)(st + (wave * IA + i) * 1024), 16, 0, 0);
  };
  auto request_b = [&](int from, int to) __attribute__((always_inline)) {
    uint8_t* st = smem + rslot * STAGE;
#pragma unroll
    for (int i = from; i < to; i++)                                      // (scalar base + the lane's offset: no vector address arithmetic)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(scalar_ptr(pb) + boff_lane[i]), (__attribute__((address_space(3))) void*)(st + BM * 128 + (wave * IB + i) * 1024), 16, 0, ONCE ? 2 : 0);
  };
  auto request_end = [&]() __attribute__((always_inline)) {
    pb += 128;
#pragma unroll
    for (int i = 0; i < IA; i++) pa[i] += 128;
    rslot = rslot + 1 == NB ? 0 : rslot + 1;
    if (++rs_ == nsteps) { rs_ = 0; rt_ += step_wg; }
  };
  auto request = [&](int q) __attribute__((always_inline)) { request_front(q); request_b(0, IB); request_end(); };

  FfnCur cur;
  find(t, cur);
  rc_ = cur;
  if constexpr (UP) request_ids();
  for (int i = 0; i < NB - 1; i++) request(i == 0 ? 0 : -1);             // (a tile has at least two steps)
  const int f0 = r16 * 128 + ((kg ^ (r16 & 7)) << 4), f1 = f0 ^ 64;
  int slot = 0, cn = 0, stores = 0;                                      // stores: of the last tile's epilogue, at least
  const uint32_t pick = (uint32_t)(kg | (kg + 4) << 8) | 0x0C0C0000u;    // v_perm: byte kg of two dwords
  long long left = total;                                                // steps not yet multiplied
  while (true) {
    v4f32 acc[RS][4];
#pragma unroll
    for (int i = 0; i < RS; i++)
#pragma unroll
      for (int j = 0; j < 4; j++) acc[i][j] = v4f32{0.f, 0.f, 0.f, 0.f};
    const int nsub = (((cur.valid + 15) >> 4) - wm + WM - 1) / WM;        // sub-tiles wm, wm + WM, ... of this wave that hold rows
    uint8_t* st = smem;
    uint32_t sca[RS], scb[4];                                             // this lane's scale bytes of the steps ahead
    for (int s = 0; s < nsteps; s++) {
      // This wave's requests of the step have landed, and so have the others'.  What was requested behind it may be in flight: the next step (NB = 3), the scales in front of that one, the stores
      // of the tile before.
      left--;
      if (NB == 2 || left == 0) ffn_wait_vm<0>();
      else if (s < 2) { if (stores >= 8) ffn_wait_vm<NI + 8>(); else if (stores >= 6) ffn_wait_vm<NI + 6>(); else if (stores >= 4) ffn_wait_vm<NI + 4>(); else if (stores >= 2) ffn_wait_vm<NI + 2>(); else ffn_wait_vm<NI>(); }
      else if ((s & 3) == 3) ffn_wait_vm<NI + IS>();
      else ffn_wait_vm<NI>();
      asm volatile("s_barrier" ::: "memory");
      // Into the position of the step before, which every wave has read; the scales of the next four steps once every wave has those of this group (read at its first step)
      const int p4 = s & ~3, len = min(4, nsteps - p4), q = p4 + len;
      const bool req = left >= NB - 1;
      const int rq = s - p4 != max(1, len - (NB - 1)) ? -1 : q < nsteps ? q : t + step_wg < last ? 0 : -1;
      const bool spread = SPREAD && nsub == RS;
      if (req && !spread) request(rq);
      st = smem + slot * STAGE;
      slot = slot + 1 == NB ? 0 : slot + 1;
      if (s == p4) {
        // byte i: the scale of step s + i of this lane's block
        if (KB == 8) {
          const uint32_t* b8 = (const uint32_t*)scales + (BM + wn * 64 + r16); const uint32_t* a8 = (const uint32_t*)scales + (16 * wm + r16);
#pragma unroll
          for (int j = 0; j < 4; j++) scb[j] = __builtin_amdgcn_perm(b8[BM + BN + 16 * j], b8[16 * j], pick);
#pragma unroll
          for (int i = 0; i < RS; i++) sca[i] = __builtin_amdgcn_perm(a8[BM + BN + 16 * WM * i], a8[16 * WM * i], pick);
        } else {
          const uint32_t halves = len == 2 ? 0x0C0C0504u : 0x05040100u;  // (the last two steps of a row lie behind the two before them)
          auto bytes = [&](const u32x4& d) __attribute__((always_inline)) { return __builtin_amdgcn_perm(__builtin_amdgcn_perm(d.w, d.z, pick), __builtin_amdgcn_perm(d.y, d.x, pick), halves); };
          // (by inline assembly, their wait with them: in front of plain reads the compiler would wait for all requests in flight)
          const uint32_t at_b = (uint32_t)(uintptr_t)scales + (uint32_t)(BM + wn * 64 + r16) * 16u, at_a = (uint32_t)(uintptr_t)scales + (uint32_t)(16 * wm + r16) * 16u;
          u32x4 d0, d1, d2, d3;
          asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %4 offset:256\n\tds_read_b128 %2, %4 offset:512\n\tds_read_b128 %3, %4 offset:768\n\ts_waitcnt lgkmcnt(0)" : "=&v"(d0), "=&v"(d1), "=&v"(d2), "=&v"(d3) : "v"(at_b) : "memory");
          scb[0] = bytes(d0); scb[1] = bytes(d1); scb[2] = bytes(d2); scb[3] = bytes(d3);
          if constexpr (RS == 1) {
            asm volatile("ds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=&v"(d0) : "v"(at_a) : "memory");
            sca[0] = bytes(d0);
          } else {
#pragma unroll
            for (int i = 0; i < RS; i += 2) {
              asm volatile("ds_read_b128 %0, %2 offset:%3\n\tds_read_b128 %1, %2 offset:%4\n\ts_waitcnt lgkmcnt(0)" : "=&v"(d0), "=&v"(d1) : "v"(at_a), "n"(256 * WM * i), "n"(256 * WM * (i + 1)) : "memory");
              sca[i] = bytes(d0); sca[(i + 1) % RS] = bytes(d1);
            }
          }
        }
      }
      const uint8_t* As = st; const uint8_t* Bs = st + BM * 128 + wn * 4 * 2048;
      auto multiply = [&](auto full_tag) __attribute__((always_inline)) {
        constexpr bool FULL = decltype(full_tag)::value;                  // every sub-tile holds rows: no branches between the products
        v8i32 bf[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const u32x4 y0 = *(const u32x4*)(Bs + j * 2048 + f0), y1 = *(const u32x4*)(Bs + j * 2048 + f1);
          bf[j] = v8i32{(int)y0.x, (int)y0.y, (int)y0.z, (int)y0.w, (int)y1.x, (int)y1.y, (int)y1.z, (int)y1.w};
        }
        auto frag = [&](int i, v8i32& af) __attribute__((always_inline)) {
          const uint8_t* p = As + (WM * i + wm) * 2048;
          const u32x4 x0 = *(const u32x4*)(p + f0), x1 = *(const u32x4*)(p + f1);
          af = v8i32{(int)x0.x, (int)x0.y, (int)x0.z, (int)x0.w, (int)x1.x, (int)x1.y, (int)x1.z, (int)x1.w};
        };
        v8i32 af[2];
        frag(0, af[0]);
#pragma unroll
        for (int i = 0; i < RS; i++) {
          if (i + 1 < (FULL ? RS : nsub)) frag(i + 1, af[(i + 1) & 1]);
          if (FULL || i < nsub) {
#pragma unroll
            for (int j = 0; j < 4; j++) acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(bf[j], af[i & 1], acc[i][j], 0, 0, 0, (int)scb[j], 0, (int)sca[i]);
            if constexpr (FULL && SPREAD) {
              if (req) { if (i == 0) request_front(rq); else if (i == 1) request_b(0, IB / 2); else if (i == 2) { request_b(IB / 2, IB); request_end(); } }
            }
          }
        }
      };
      if (RS <= 4 && nsub == RS) multiply(std::true_type{}); else if (nsub > 0) multiply(std::false_type{});
#pragma unroll
      for (int j = 0; j < 4; j++) scb[j] >>= 8;
#pragma unroll
      for (int i = 0; i < RS; i++) sca[i] >>= 8;
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                  // every read of this position is done: behind the next barrier it is requested into
    }
    ffn_epilogue<RS, WM, BN, UP>(a, cur, acc, nsub, wm, wn, &s_bias[cn & 1][wn * 64]);
    stores = nsub > 0 ? 2 * nsub : 0;                                    // (every sub-tile stores at least its first row)
    t += step_wg; cn++;
    if (t >= last) break;
    find(t, cur);
  }
}

// out[t, :] = sum_s bf16(bf16(weight) * z[row of (t, s), :]), float32 sum in slot order, bf16 result: eight columns per thread, the rows of up to eight slots requested together
__global__ __launch_bounds__(256) void moe_combine_kernel(const FfnArgs a) {
  __shared__ int s_off[FFN_MAX_E + 1];
  __shared__ int s_row[FFN_MAX_K]; __shared__ float s_w[FFN_MAX_K];
  ffn_offsets(a.counts, a.E, 1, 1, s_off, nullptr);
  __syncthreads();
  for (int t = blockIdx.x; t < a.T; t += gridDim.x) {
    if ((int)threadIdx.x < a.k) {
      const size_t j = (size_t)t * a.k + threadIdx.x;
      s_row[threadIdx.x] = s_off[a.place_e[j]] + a.place[j]; s_w[threadIdx.x] = bf16_to_f(f_to_bf16(a.weights[j]));
    }
    __syncthreads();
    for (int d = threadIdx.x; d < a.D / 8; d += 256) {
      float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      for (int s0 = 0; s0 < a.k; s0 += 8) {
        u32x4 v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = *(const u32x4*)(a.z + (size_t)s_row[min(s0 + u, a.k - 1)] * a.D + 8 * d);
#pragma unroll
        for (int u = 0; u < 8; u++) {
          if (s0 + u < a.k) {
            const float w = s_w[s0 + u];
#pragma unroll
            for (int i = 0; i < 4; i++) { const uint32_t p = pack_bf16x2(bf16_lo(v[u][i]) * w, bf16_hi(v[u][i]) * w); acc[2 * i] += bf16_lo(p); acc[2 * i + 1] += bf16_hi(p); }
          }
        }
      }
      *(u32x4*)(a.out + (size_t)t * a.D + 8 * d) = u32x4{pack_bf16x2(acc[0], acc[1]), pack_bf16x2(acc[2], acc[3]), pack_bf16x2(acc[4], acc[5]), pack_bf16x2(acc[6], acc[7])};
    }
    __syncthreads();
  }
}

static size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }
struct FfnLayout { size_t xq, xe8, yq, ye8, z, counts, row_tok, place, place_e, weights, total; };
static FfnLayout ffn_layout(long long T, long long D, long long I, long long E, long long k) {
  FfnLayout l; size_t o = 0; const long long R = T * k;
  auto take = [&](size_t n) { const size_t at = o; o += align256(n); return at; };
  l.xq = take(T * D); l.xe8 = take(T * (D / 32)); l.yq = take(R * I); l.ye8 = take(R * (I / 32)); l.z = take(R * D * 2);
  l.counts = take(E * 4); l.row_tok = take(E * T * 4); l.place = take(R * 4); l.place_e = take(R * 4); l.weights = take(R * 4); l.total = o;
  return l;
}

// per_cu: workgroups of a CU, at most; each launch has as many as its LDS leaves room for (16-row tiles: three of gate/up, whose rows' tokens sit in LDS, and four of down up to 90 experts).  With four for
// both, a quarter of gate/up's tiles beyond 768 began when others had ended: 80 experts, I 768, 32 / 56 tokens 93.5 -> 90.7 / 97.7 -> 94.2 us, 128 experts (down: three), I 512 / 768, 64 tokens 110 -> 101 / 132 -> 123, up to 768 tiles the same.
template <int BM, int WM, int WN, int NB, bool ONCE>
static hipError_t launch_ffn(const FfnArgs& a, int n_cu, int per_cu, hipStream_t s) {
  constexpr int ring = (BM + 64 * WN) * (128 * NB + 16), most = ring + 8 * (FFN_MAX_E + 1);
  const int lds = ring + 8 * (a.E + 1);
  auto up = ffn_gemm_kernel<BM, WM, WN, NB, true, ONCE>; auto down = ffn_gemm_kernel<BM, WM, WN, NB, false, ONCE>;
  static int own[2];                                                     // LDS of the kernels' own
  static const hipError_t configured = [&] {
    const void* k[2] = {(const void*)up, (const void*)down};
    for (int i = 0; i < 2; i++) {
      hipFuncAttributes fa;
      hipError_t e = hipFuncGetAttributes(&fa, k[i]);
      if (e == hipSuccess) e = hipFuncSetAttribute(k[i], hipFuncAttributeMaxDynamicSharedMemorySize, most);
      if (e != hipSuccess) return e;
      own[i] = (int)fa.sharedSizeBytes;
    }
    return hipSuccess;
  }();
  if (configured != hipSuccess) return configured;
  auto grid = [&](int i) { const int fit = 160 * 1024 / ((lds + own[i] + 1279) / 1280 * 1280); return n_cu * (fit < 1 ? 1 : fit < per_cu ? fit : per_cu); };      // (LDS is handed out in pieces of 1280 bytes)
  up<<<grid(0), 64 * WM * WN, lds, s>>>(a);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  down<<<grid(1), 64 * WM * WN, lds, s>>>(a);
  return hipGetLastError();
}

extern "C" {

// bytes of workspace tga_moe_feed_forward needs; 0 when the sizes are outside its range (the caller then runs the single steps)
int tga_moe_feed_forward_plan(int64_t T, int64_t D, int64_t I, int n_experts, int k, int64_t* nbytes) {
  TGA_REQUIRE(nbytes, "tga_moe_feed_forward_plan: null pointer");
  *nbytes = 0;
  if (T < 1 || k < 1 || k > FFN_MAX_K || k > n_experts || n_experts > FFN_MAX_E || D < 256 || D % 256 || I < 256 || I % 256) return 0;
  if (T >= (1 << 24) || T * k >= (1ll << 31) || (int64_t)n_experts * 2 * I >= (1ll << 31) || (int64_t)n_experts * D >= (1ll << 31)) return 0;
  *nbytes = (int64_t)ffn_layout(T, D, I, n_experts, k).total;
  return 0;
}

int tga_moe_feed_forward(const void* x_bf16, const float* logits, int64_t T, int64_t D, int64_t I, int n_experts, int k, const void* w_gate_up, const void* e8_gate_up,
                         const float* b_gate_up, const void* w_down, const void* e8_down, const float* b_down, float limit, void* workspace, void* out_bf16, void* stream) {
  TGA_REQUIRE(x_bf16 && logits && w_gate_up && e8_gate_up && b_gate_up && w_down && e8_down && b_down && workspace && out_bf16, "tga_moe_feed_forward: null pointer");
  int64_t need = 0;
  tga_moe_feed_forward_plan(T, D, I, n_experts, k, &need);
  TGA_REQUIRE(need > 0, "tga_moe_feed_forward: sizes outside the range (T=%lld D=%lld I=%lld E=%d k=%d)", (long long)T, (long long)D, (long long)I, n_experts, k);
  TGA_REQUIRE((((uintptr_t)x_bf16 | (uintptr_t)w_gate_up | (uintptr_t)w_down | (uintptr_t)b_gate_up | (uintptr_t)b_down | (uintptr_t)workspace | (uintptr_t)out_bf16) & 15) == 0
              && (((uintptr_t)e8_gate_up | (uintptr_t)e8_down) & 3) == 0, "tga_moe_feed_forward: operands must be 16-byte aligned (scales 4-byte)");
  const FfnLayout l = ffn_layout(T, D, I, n_experts, k);
  uint8_t* ws = (uint8_t*)workspace;
  FfnArgs a;
  a.x = (const uint16_t*)x_bf16; a.logits = logits; a.w[0] = (const uint8_t*)w_gate_up; a.w[1] = (const uint8_t*)w_down; a.we8[0] = (const uint8_t*)e8_gate_up; a.we8[1] = (const uint8_t*)e8_down;
  a.bias[0] = b_gate_up; a.bias[1] = b_down; a.T = (int)T; a.D = (int)D; a.I = (int)I; a.E = n_experts; a.k = k; a.limit = limit;
  a.xq = ws + l.xq; a.xe8 = ws + l.xe8; a.yq = ws + l.yq; a.ye8 = ws + l.ye8; a.z = (uint16_t*)(ws + l.z); a.counts = (int*)(ws + l.counts); a.row_tok = (int*)(ws + l.row_tok);
  a.place = (int*)(ws + l.place); a.place_e = (int*)(ws + l.place_e); a.weights = (float*)(ws + l.weights); a.out = (uint16_t*)out_bf16;
  hipStream_t s = (hipStream_t)stream;
  const long long n8 = T * (D / 8), qb = (n8 + 1023) / 1024;
  a.nq_blocks = (int)(qb < 448 ? qb : 448);
  // one workgroup needs no shared counters; beyond, a token per wave, until there are so many workgroups that they queue for the counters (the whole call, T = 2000, 64 experts: 155 -> 150 us with
  // 16 tokens a workgroup instead of 64, 32: 150.3; 1600 tokens, 32 experts: 71.5 -> 65.4; 8000 tokens, 80 experts: 75.1 -> 77.9)
  a.prep_tokens = T <= 64 || T > 4096 ? 64 : T > 2048 ? 32 : 16;
  const int route_blocks = (int)((T + a.prep_tokens - 1) / a.prep_tokens);
  a.one_route_block = route_blocks == 1;
  if (!a.one_route_block) { moe_zero_counts_kernel<<<1, 512, 0, s>>>(a.counts, n_experts); TGA_LAUNCH_CHECK(); }
  const dim3 pg(a.nq_blocks + route_blocks);
  if (n_experts <= 64) moe_prep_kernel<1><<<pg, 1024, 0, s>>>(a);
  else if (n_experts <= 128) moe_prep_kernel<2><<<pg, 1024, 0, s>>>(a);
  else moe_prep_kernel<FFN_MAX_E / 64><<<pg, 1024, 0, s>>>(a);
  TGA_LAUNCH_CHECK();
  static const int n_cu = [] { int dev = 0, n = 0; return (hipGetDevice(&dev) == hipSuccess && hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0) ? n : 256; }();
  // Tile height by the rows per expert r, us of the call (heights 16 / 32 / 64 / 128; MI355X).  64 experts, D 2048, I 512, k 8, even popularity: r = 2 50.5 / 52.0 / 51.8 / 51.2, 8 61.4 / 62.4 / 62.7 / 61.9,
  // 32 86.6 / 69.5 / 68.4 / 69.5, 48 - / 87 / 80 / 73, 64 126 / 90 / 89 / 76, 128 199 / 125 / 119 / 112, 200 271 / 164 / 155 / 119; popularity by 1 / rank^1.1: 2 45.9 / 46.5 / 49.2 / 48.1, 16 82 / 67 / 84 / 73,
  // 32 89 / 83 / 83 / 94, 64 127 / 90 / 92 / 100, 128 202 / 127 / 119 / 115, 200 278 / 166 / 150 / 146.  16 experts, D 1536, I 768, k 4 (few tiles: lower ones fill the chip): 16 35.2 / 33.3 / 36.3 / 40.9,
  // 64 49.9 / 37.9 / 40.0 / 47.3, 128 66 / 53.7 / 43.1 / 51.5, 200 86 / 60.9 / 60.1 / 53.3.  Where 256 rows make at most five ninths of the rounds that 128 make, each launch takes them on the device, which has
  // the counts.  gate/up or down alone, rounds 128 / 256, us of 128 / 256: 2 / 1 rounds 57.1 / 45.3 (64 experts, r = 128), 58.0 / 55.5 (8, r = 1024), 56.0 / 52.8 (16, r = 512); 4 / 2 89.3 / 84.9 and 45.7 / 43.5
  // (16, r = 1000), 116 / 109 (8, r = 4096); 8 / 4 70.6 / 67.7 (8, r = 4096); 9 / 5 76.7 / 74.7 (16, r = 2048), 57.2 / 55.2 (32, r = 1024); 5 / 3 137 / 132 (16, r = 2048, even) but 141 / 151 (skewed), 134 / 148 (32),
  // 46.8 / 50.3 (64, r = 250); 3 / 2 82 / 101 (8, r = 2048), 50 / 64; 8 / 5 53.8 / 54.1.  Against tiles of 256 for all of them: the call of 16 experts, r = 2048, even, 232 -> 240, skewed 256 -> 243.
  // Low tiles read a weight about once.  Where the layer's weights are also more than half of the 256 MB behind the L2s, so that they are not there again at the next call, the requests pass them by:
  // 32 tokens of 64 experts, I 768 67.7 -> 61.9 us, r = 4, I 512 56.5 -> 51.1, r = 24 64.7 -> 61.7; of 57 MB that are still there 32.4 -> 36.1.
  const bool once = 3ll * n_experts * I * D >= (128ll << 20);
  if (T * k < 6ll * n_experts) {
    TGA_HIP((once ? launch_ffn<16, 1, 2, 2, true>(a, n_cu, 4, s) : launch_ffn<16, 1, 2, 2, false>(a, n_cu, 4, s)));
  } else if (T * k < 48ll * n_experts) {
    TGA_HIP((once ? launch_ffn<32, 2, 2, 2, true>(a, n_cu, 3, s) : launch_ffn<32, 2, 2, 2, false>(a, n_cu, 3, s)));
  } else if (4 * (n_experts * ((T * k + 128ll * n_experts - 1) / (128ll * n_experts)) * (2 * I / 256)) < 3 * n_cu) {
    TGA_HIP((launch_ffn<64, 2, 2, 2, false>(a, n_cu, 2, s)));
  } else {
    TGA_HIP((launch_ffn<128, 2, 4, 3, false>(a, n_cu, 1, s)));
  }
  moe_combine_kernel<<<(unsigned)(T < 2048 ? T : 2048), 256, 0, s>>>(a);
  TGA_LAUNCH_CHECK();
  return 0;
}

}  // extern "C"
