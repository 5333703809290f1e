// The grouped MoE feed-forward of an MXFP8 model (examples/mlperf/models/gpt_oss.py:213-226) as five launches over compact rows:
//   1. moe_prep_kernel      quantises the T input rows once (a token's row serves all of its experts) and, in other workgroups, picks each token's experts and gives every
//                           assignment its place among the rows of its expert
//   2. ffn_gemm_kernel<..., gate/up>   gathers the quantised rows by token, multiplies, adds the bias, applies the clamped interleaved SwiGLU and quantises the result
//   3. ffn_gemm_kernel<..., down>      multiplies and adds the bias; rows stay in expert order
//   4. moe_combine_kernel   weighs and sums the k rows of every token
// (+ a fill of the expert counters in front when more than one workgroup routes).  The values are those of route -> dispatch -> quantize_mxfp8 -> grouped_mx_gemm ->
// add_expert_bias -> swiglu -> quantize_mxfp8 -> grouped_mx_gemm -> add_expert_bias -> combine: every rounding to bf16 and to E4M3 sits where it sits there.  What
// is gone are the passes between them (T = 4096, k = 8, E = 128, D = 2048, I = 768: dispatch, two quantisations, two bias adds, SwiGLU over 65536 padded rows) and the
// padding of every expert's rows to 256, and the host work of eleven entry points.  MI355X, back to back: T = 2000, k = 8, E = 64, D = 2048, I = 512 2480 (single passes:
// 810) -> 186 us; T = 32, k = 8, E = 64, I = 768 840 (single) -> 81 us; the benchmark's T = 4096, E = 128, I = 768 1340 (single) -> 406 us.
#include "mxfp8.h"
#include "host.h"

#define FFN_MAX_E 512             // experts (their counts and offsets sit in LDS)
#define FFN_MAX_K 64              // experts per token
#define FFN_BN 256                // weight rows of a tile

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
  int one_route_block;
};

// ---------------------------------------------------------------------------------------------------- routing + quantisation of the input
#define PREP_TOKENS 64            // tokens of a routing workgroup: sixteen waves of four

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
  const int t0 = ((int)blockIdx.x - a.nq_blocks) * PREP_TOKENS, nt = min(PREP_TOKENS, a.T - t0), n = nt * a.k;
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

// Exclusive prefix sums over the experts' counts and over their tiles by the first wave of a workgroup: off[e] = first row, tile[e] = first tile (off[E], tile[E]: the totals)
__device__ __forceinline__ void ffn_offsets(const int* __restrict__ counts, int E, int bm, int tiles_n, int* off, int* tile) {
  const int lane = threadIdx.x;
  if (lane < 64) {
    constexpr int PER = FFN_MAX_E / 64;
    int c[PER], so = 0, st = 0;
#pragma unroll
    for (int i = 0; i < PER; i++) { const int e = lane * PER + i; c[i] = e < E ? counts[e] : 0; so += c[i]; st += (c[i] + bm - 1) / bm * tiles_n; }
    int io = so, it = st;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) { const int uo = __shfl_up(io, o), ut = __shfl_up(it, o); if (lane >= o) { io += uo; it += ut; } }
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
// Tile of BM rows x 256 weight rows, K steps of 128, WM x 4 waves of (BM / WM) x 64, operands in LDS in the order the scaled MFMA consumes (mxfp8.h), weights as the A
// operand, so a lane holds four consecutive output columns of one row.  The 16-row sub-tiles are dealt to the WM waves alternately and only those that hold rows are
// multiplied.  A workgroup walks tiles b, b + gridDim.x, ...: consecutive tiles of an expert share its weight or activation rows, and the workgroups of an XCD (b % 8) take a
// contiguous run of tiles.  The first step of the next tile is fetched during the last step of this one.
// UP: gate/up (rows gathered by token, epilogue bias + clamped interleaved SwiGLU + quantisation) or down (compact rows, epilogue bias).
struct FfnCur { uint32_t boff; int e, m0, tn, valid, row0; };

template <int BM, int WM, bool UP>
__global__ __launch_bounds__(256 * WM) void ffn_gemm_kernel(const FfnArgs a) {
  constexpr int NT = 256 * WM, RS = BM / 16 / WM;                        // threads, 16-row sub-tiles of a wave
  constexpr int PA = BM * 8 / NT, PB = FFN_BN * 8 / NT, NS = (BM + FFN_BN + NT - 1) / NT;   // 16-byte pieces and scale dwords per thread and step
  static_assert(PA >= 1 && RS >= 1, "tile too small");
  constexpr int STAGE = (BM + FFN_BN) * 132;
  constexpr int RPT = NT / 8;                                            // rows between a thread's pieces
  __shared__ __attribute__((aligned(16))) uint8_t smem[2 * STAGE];
  __shared__ int s_off[FFN_MAX_E + 1], s_tile[FFN_MAX_E + 1], s_row[2][BM];   // s_row: operand rows of the tile being multiplied and of the next one
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 2, wn = wave & 3, r16 = lane & 15, kg = lane >> 4;
  const int N = UP ? 2 * a.I : a.D, K = UP ? a.D : a.I, KB = K / 32, nsteps = K / 128, tiles_n = N / FFN_BN;
  const uint8_t* __restrict__ A = UP ? a.xq : a.yq; const uint8_t* __restrict__ Ae = UP ? a.xe8 : a.ye8;
  const uint8_t* __restrict__ B = a.w[UP ? 0 : 1]; const uint8_t* __restrict__ Be = a.we8[UP ? 0 : 1];
  ffn_offsets(a.counts, a.E, BM, tiles_n, s_off, s_tile);
  __syncthreads();
  const int ntiles = __builtin_amdgcn_readfirstlane(s_tile[a.E]);
  const int per = (ntiles + 7) >> 3;                                     // tiles of an XCD's run
  const int first = ((int)blockIdx.x & 7) * per, last = min(first + per, ntiles), step_wg = (int)(gridDim.x + 7 - (blockIdx.x & 7)) >> 3;
  int t = first + ((int)blockIdx.x >> 3);
  if (t >= last) return;

  const int cpy_c = tid & 7, cpy_r = tid >> 3;
  int lds_a[PA], lds_b[PB];
#pragma unroll
  for (int j = 0; j < PA; j++) lds_a[j] = gg_slot_off(cpy_r + RPT * j, cpy_c);
#pragma unroll
  for (int j = 0; j < PB; j++) lds_b[j] = BM * 128 + gg_slot_off(cpy_r + RPT * j, cpy_c);
  const int f0 = ((16 * kg + (r16 ^ kg)) << 4), f1 = 1024 + ((16 * kg + (r16 ^ (kg + 4))) << 4);

  auto setup = [&](int tile, FfnCur& c, int which) __attribute__((always_inline)) {
    int lo = 0, hi = a.E;                                                // the expert whose tiles hold this one
    while (hi - lo > 1) { const int mid = (lo + hi) >> 1; if (__builtin_amdgcn_readfirstlane(s_tile[mid]) <= tile) lo = mid; else hi = mid; }
    const int i = tile - __builtin_amdgcn_readfirstlane(s_tile[lo]), tm = i / tiles_n, off = __builtin_amdgcn_readfirstlane(s_off[lo]);
    c.e = lo; c.tn = i - tm * tiles_n; c.m0 = tm * BM; c.valid = min(__builtin_amdgcn_readfirstlane(s_off[lo + 1]) - off - c.m0, BM);
    c.row0 = off + c.m0;
    c.boff = ((uint32_t)lo * (uint32_t)N + (uint32_t)c.tn * FFN_BN);     // first weight row
    if (tid < BM) { const int r = min(tid, c.valid - 1); s_row[which][tid] = UP ? a.row_tok[(size_t)lo * a.T + c.m0 + r] : c.row0 + r; }   // rows beyond the expert's repeat its last one (their results are dropped)
  };
  u32x4 va[PA], vb[PB]; uint32_t vs[NS];
  auto load_a = [&](int which, int s, int j) __attribute__((always_inline)) { va[j] = *(const u32x4*)(A + (size_t)(uint32_t)s_row[which][cpy_r + RPT * j] * K + (uint32_t)(s * 128 + cpy_c * 16)); };
  auto load_b = [&](const FfnCur& c, int s, int j) __attribute__((always_inline)) {
    vb[j] = *(const u32x4*)(B + (size_t)(c.boff + RPT * j) * K + (uint32_t)cpy_r * (uint32_t)K + (uint32_t)(s * 128 + cpy_c * 16));
  };
  auto load_s = [&](const FfnCur& c, int which, int s) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NS; j++) {
      const int i = tid + NT * j;
      const uint8_t* p = i < BM ? Ae + (size_t)(uint32_t)s_row[which][i] * KB : Be + (size_t)(c.boff + (uint32_t)min(i - BM, FFN_BN - 1)) * KB;
      vs[j] = *(const uint32_t*)(p + 4 * s);
    }
  };
  auto store_a = [&](uint8_t* st, int j) __attribute__((always_inline)) { *(u32x4*)(st + lds_a[j]) = va[j]; };
  auto store_b = [&](uint8_t* st, int j) __attribute__((always_inline)) { *(u32x4*)(st + lds_b[j]) = vb[j]; };
  auto store_s = [&](uint8_t* st) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NS; j++) { const int i = tid + NT * j; if (i < BM + FFN_BN) ((uint32_t*)(st + (BM + FFN_BN) * 128))[i] = vs[j]; }
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
      const uint32_t* sA = (const uint32_t*)(st + (BM + FFN_BN) * 128) + r16; const uint32_t* sB = sA + BM + wn * 64;
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
    // ---- epilogue: lane = row r16 of sub-tile WM i + wm, columns 4 kg .. 4 kg + 3 of n sub-tile j.  The stage the last step was read from is idle: wave-private slabs.
    {
      uint8_t* slab = smem + ((par + nsteps - 1) & 1) * STAGE + wave * 2304;   // 16 rows of 144 bytes
      const int row0 = cur.row0;
      f32x4 bias[4];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        bias[j] = *(const f32x4*)(a.bias[UP ? 0 : 1] + (size_t)cur.e * N + cur.tn * FFN_BN + wn * 64 + 16 * j + 4 * kg);
#pragma unroll
        for (int c = 0; c < 4; c++) bias[j][c] = bf16_to_f(f_to_bf16(bias[j][c]));
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
            const float gl0 = fminf(bf16_lo(g01), a.limit), gl1 = fminf(bf16_lo(g23), a.limit);
            const float li0 = fminf(fmaxf(bf16_hi(g01), -a.limit), a.limit), li1 = fminf(fmaxf(bf16_hi(g23), -a.limit), a.limit);
            const uint32_t ag = pack_bf16x2(1.702f * gl0, 1.702f * gl1);
            const uint32_t sg = pack_bf16x2(mx_sigmoid_bf16(bf16_lo(ag)), mx_sigmoid_bf16(bf16_hi(ag)));
            const uint32_t p = pack_bf16x2(gl0 * bf16_lo(sg), gl1 * bf16_hi(sg)), q = pack_bf16x2(li0 + 1.0f, li1 + 1.0f);
            const uint32_t o = pack_bf16x2(bf16_lo(p) * bf16_lo(q), bf16_hi(p) * bf16_hi(q));
            y[2 * j] = bf16_lo(o); y[2 * j + 1] = bf16_hi(o);
            amax = fmaxf(amax, fmaxf(fabsf(y[2 * j]), fabsf(y[2 * j + 1])));
          }
          amax = fmaxf(amax, __shfl_xor(amax, 16)); amax = fmaxf(amax, __shfl_xor(amax, 32));     // the wave's 64 columns are one block of 32 results
          const int e = mx_e8(amax);
          const float sc = mx_scale(e);
#pragma unroll
          for (int j = 0; j < 4; j++) *(uint16_t*)(slab + r16 * 40 + 8 * j + 2 * kg) = (uint16_t)e4m3x2(y[2 * j] * sc, y[2 * j + 1] * sc);
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
          const u32x2 o = *(const u32x2*)(slab + r16 * 40 + 8 * kg);
          if (r0 + r16 < cur.valid) {
            const size_t row = (size_t)(row0 + r0 + r16);
            *(u32x2*)(a.yq + row * a.I + cur.tn * 128 + wn * 32 + 8 * kg) = o;
            if (kg == 0) a.ye8[row * (a.I / 32) + cur.tn * 4 + wn] = (uint8_t)e;
          }
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        } else {
#pragma unroll
          for (int j = 0; j < 4; j++) {
            const uint32_t h01 = pack_bf16x2(acc[i][j][0], acc[i][j][1]), h23 = pack_bf16x2(acc[i][j][2], acc[i][j][3]);
            *(u32x2*)(slab + r16 * 144 + 32 * j + 8 * kg) = u32x2{pack_bf16x2(bf16_lo(h01) + bias[j][0], bf16_hi(h01) + bias[j][1]), pack_bf16x2(bf16_lo(h23) + bias[j][2], bf16_hi(h23) + bias[j][3])};
          }
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
          const int rr = lane >> 3, rc = lane & 7;
#pragma unroll
          for (int p = 0; p < 2; p++) {
            const u32x4 o = *(const u32x4*)(slab + (rr + 8 * p) * 144 + 16 * rc);
            if (r0 + rr + 8 * p < cur.valid) *(u32x4*)(a.z + (size_t)(row0 + r0 + rr + 8 * p) * N + cur.tn * FFN_BN + wn * 64 + 8 * rc) = o;
          }
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
      }
    }
    if (!more) break;
    __syncthreads();                                                      // the slabs are free before any wave's next step writes that stage
    par = (par + nsteps) & 1; cur = nxt; t = tnext; which ^= 1;
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
  const int route_blocks = (int)((T + PREP_TOKENS - 1) / PREP_TOKENS);
  a.one_route_block = route_blocks == 1;
  if (!a.one_route_block) { moe_zero_counts_kernel<<<1, 512, 0, s>>>(a.counts, n_experts); TGA_LAUNCH_CHECK(); }
  const dim3 pg(a.nq_blocks + route_blocks);
  if (n_experts <= 64) moe_prep_kernel<1><<<pg, 1024, 0, s>>>(a);
  else if (n_experts <= 128) moe_prep_kernel<2><<<pg, 1024, 0, s>>>(a);
  else moe_prep_kernel<FFN_MAX_E / 64><<<pg, 1024, 0, s>>>(a);
  TGA_LAUNCH_CHECK();
  static const int n_cu = [] { int dev = 0, n = 0; return (hipGetDevice(&dev) == hipSuccess && hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0) ? n : 256; }();
  // Tiles of 32 or 256 rows by the rows per expert, us of the call (32 / 256): 64 experts, D 2048, I 512, even popularity: 16 rows 61.5 / 65.8, 24 71.3 / 67.1, 40 71.7 / 70.1, 48 90.0 / 72.3, 128 125 / 93,
  // 200 181 / 114; popularity by 1 / rank^1.1: 16 67.5 / 74.6, 48 73.2 / 110, 64 91.7 / 132, 128 126 / 150, 200 185 / 167.  128 experts, I 768: even 32 189 / 182, 48 221 / 192, 128 349 / 231; skewed 32
  // 191 / 219, 48 229 / 235, 64 238 / 242, 96 304 / 271.  16 experts, D 1536, I 768: 48 45.0 / 50.7, 128 53.2 / 64.9, 200 71.6 / 77.5 even, 46.0 / 68.0, 52.5 / 75.7, 72.1 / 78.5 skewed.  At 48 the even
  // popularity gains; where it is skewed, or the experts are few, 32 rows stay better up to 128 and more, but the host does not know the counts.
  const bool small = T * k < 48ll * n_experts;
  if (small) {
    ffn_gemm_kernel<32, 1, true><<<2 * n_cu, 256, 0, s>>>(a); TGA_LAUNCH_CHECK();
    ffn_gemm_kernel<32, 1, false><<<2 * n_cu, 256, 0, s>>>(a); TGA_LAUNCH_CHECK();
  } else {
    ffn_gemm_kernel<256, 2, true><<<n_cu, 512, 0, s>>>(a); TGA_LAUNCH_CHECK();
    ffn_gemm_kernel<256, 2, false><<<n_cu, 512, 0, s>>>(a); TGA_LAUNCH_CHECK();
  }
  moe_combine_kernel<<<(unsigned)(T < 2048 ? T : 2048), 256, 0, s>>>(a);
  TGA_LAUNCH_CHECK();
  return 0;
}

}  // extern "C"
