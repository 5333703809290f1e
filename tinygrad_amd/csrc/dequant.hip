// Block dequant kernels: bit-exact restatement of ggml_data_to_tensor (tinygrad/llm/gguf.py:23-119) for Q4_0 (:46), Q4_1 (:47-49), Q5_0 / Q5_1 (:50-55), Q8_0 (:56),
// Q4_K / Q5_K (:57-67), Q6_K (:68-72), IQ3_XXS / IQ3_S / IQ2_S (:73-95), IQ4_XS (:96-104), MXFP4 (:105-114) and Q1_0 (:115-118).  One thread produces the
// consecutive results of one 16-byte store: eight fp16, which share their sub-block's header, or four fp32.  What bounds it is the number of requests, not their bytes: one per header field and
// one per four codes, whatever the block's alignment, where a byte at a time took twice as many (14336 x 4096 to fp16, back to back into one buffer: Q4_K 43 -> 25 us; Q4_0 28.5 -> 22.7; MXFP4 50 -> 29;
// eight fp32 per thread are two stores with gaps between lanes: Q4_0 43 us, four 38).  Into memory that no cache holds, with stores past the caches: Q4_K 42.4 -> 24.7 us (6.1 TB/s), Q4_0 32.3 -> 21.7,
// Q6_K 36.1 -> 34.8, MXFP4 49.3 -> 41.6, Q4_K to fp32 70.6 -> 39.3.
#include "deq.h"
#include "host.h"

// The eight (fp16) or four (fp32) results from value e0 of block b on, as one store
template <int T, bool F16, bool PAST>
__device__ __forceinline__ void dequant_store(const uint8_t* b, int e0, uint8_t* out) {
  float o[F16 ? 8 : 4];
  Deq<T>::get4(b, e0, o);
  if constexpr (F16) {
    Deq<T>::get4(b, e0 | 4, o + 4);
    // keep the float32 result opaque: folding the multiply into v_fma_mixlo_f16 (product + 0) would turn -0.0 into +0.0
#pragma unroll
    for (int q = 0; q < 8; q++) asm volatile("" : "+v"(o[q]));
    const u32x4 v = {f2h_bits(o[0]) | (f2h_bits(o[1]) << 16), f2h_bits(o[2]) | (f2h_bits(o[3]) << 16), f2h_bits(o[4]) | (f2h_bits(o[5]) << 16), f2h_bits(o[6]) | (f2h_bits(o[7]) << 16)};
    typedef u32x4 any_u32x4 __attribute__((aligned(2)));                   // (a store that asks for no more alignment than two of four values did)
    store_result<PAST, any_u32x4>(v, (any_u32x4*)out);
  } else store_result<PAST>(f32x4{o[0], o[1], o[2], o[3]}, (f32x4*)out);
}

template <int T, bool F16, bool PAST>
__global__ __launch_bounds__(256) void dequant_kernel(const uint8_t* __restrict__ blocks, uint8_t* __restrict__ out, int64_t n) {
  constexpr int V = F16 ? 8 : 4;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n / V; i += (int64_t)gridDim.x * 256) {
    const int64_t e = i * V, blk = e / Deq<T>::NEL;
    dequant_store<T, F16, PAST>(blocks + blk * Deq<T>::NBY, (int)(e % Deq<T>::NEL), out + 16 * i);
  }
}

// The same with a workgroup's blocks brought to LDS first, as they lie in memory: sixteen bytes a request whatever the fields of a block are.  Two results a thread, cold, 14336 x 4096, us:
// to fp16 Q4_1 30.3 -> 25.5, Q5_0 33.5 -> 29.5, Q5_1 31.2 -> 26.5, Q4_K 24.0 -> 21.9, Q5_K 46.0 -> 26.2, Q6_K 34.8 -> 27.7, IQ3_XXS 26.4 -> 22.5, IQ3_S 25.1 -> 21.6, IQ4_XS 33.6 -> 30.0, MXFP4 42.7 -> 32.5;
// not Q4_0 21.7 -> 22.2, Q8_0 30.8 -> 31.1, IQ2_S 27.0 -> 28.8, Q1_0 18.3 -> 18.9.  To fp32 Q8_0 52.4 -> 46.6, Q4_K 39.2 -> 37.6, Q5_K 40.2 -> 38.5, IQ3_XXS 41.3 -> 38.9, IQ3_S 40.4 -> 38.5, IQ2_S 40.3 -> 34.4;
// not Q5_0 38.2 -> 53.2 nor the rest, within 2 us either way.
template <int T, bool F16> constexpr bool dequant_by_lds() {
  return F16 ? T != GGML_Q4_0 && T != GGML_Q8_0 && T != GGML_IQ2_S && T != GGML_Q1_0
             : T == GGML_Q8_0 || T == GGML_Q4_K || T == GGML_Q5_K || T == GGML_IQ3_XXS || T == GGML_IQ3_S || T == GGML_IQ2_S;
}
template <int T, bool F16, bool PAST>
__global__ __launch_bounds__(256) void dequant_lds_kernel(const uint8_t* __restrict__ blocks, uint8_t* __restrict__ out, int64_t n) {
  constexpr int V = F16 ? 8 : 4, VALS = 512 * V, BYTES = VALS / Deq<T>::NEL * Deq<T>::NBY;
  __shared__ __attribute__((aligned(16))) uint8_t in[(BYTES + 15) / 16 * 16];
  const int64_t first = (int64_t)blockIdx.x * VALS;
  const uint8_t* src = blocks + first / Deq<T>::NEL * Deq<T>::NBY;
  const int vals = n - first < VALS ? (int)(n - first) : VALS, bytes = vals / Deq<T>::NEL * Deq<T>::NBY;     // (n is whole blocks)
  for (int p = threadIdx.x; 16 * p + 16 <= bytes; p += 256) *(u32x4*)(in + 16 * p) = ld16(src + 16 * p);
  if ((int)threadIdx.x < (bytes & 15)) in[(bytes & ~15) + threadIdx.x] = src[(bytes & ~15) + threadIdx.x];
  __syncthreads();
#pragma unroll
  for (int u = 0; u < 2; u++) {
    const int e = (u * 256 + threadIdx.x) * V;
    if (e < vals) dequant_store<T, F16, PAST>(in + e / Deq<T>::NEL * Deq<T>::NBY, e % Deq<T>::NEL, out + 16 * (first / V + u * 256 + threadIdx.x));
  }
}

template <int T, bool F16> static void run_dequant(const void* blocks, int64_t n, void* out, hipStream_t s) {
  constexpr int V = F16 ? 8 : 4;
  const bool past = n * (F16 ? 2 : 4) >= TGA_PAST_BYTES;
  if constexpr (dequant_by_lds<T, F16>()) {
    auto kern = past ? dequant_lds_kernel<T, F16, true> : dequant_lds_kernel<T, F16, false>;
    kern<<<(unsigned)((n + 512 * V - 1) / (512 * V)), 256, 0, s>>>((const uint8_t*)blocks, (uint8_t*)out, n);
  } else {
    auto kern = past ? dequant_kernel<T, F16, true> : dequant_kernel<T, F16, false>;
    const int64_t full = (n / V + 255) / 256;
    kern<<<(unsigned)(full < 65536 ? full : 65536), 256, 0, s>>>((const uint8_t*)blocks, (uint8_t*)out, n);
  }
}

template <int T> static int launch_dequant(const void* blocks, int64_t n, void* out, int out_dtype, hipStream_t s) {
  TGA_REQUIRE(n % Deq<T>::NEL == 0, "tga_dequant: n=%lld is not a multiple of the block size %d", (long long)n, Deq<T>::NEL);
  if (n == 0) return 0;
  if (out_dtype == TGA_F32) run_dequant<T, false>(blocks, n, out, s); else run_dequant<T, true>(blocks, n, out, s);
  TGA_LAUNCH_CHECK();
  return 0;
}

extern "C" int tga_dequant(int ggml_type, const void* blocks, int64_t n, void* out, int out_dtype, void* stream) {
  TGA_REQUIRE(out_dtype == TGA_F32 || out_dtype == TGA_F16, "tga_dequant: out_dtype must be TGA_F32 or TGA_F16");
  TGA_REQUIRE(n >= 0 && (n == 0 || (blocks && out)), "tga_dequant: null pointer");
  hipStream_t s = (hipStream_t)stream;
  switch (ggml_type) {
    case GGML_Q4_0: return launch_dequant<GGML_Q4_0>(blocks, n, out, out_dtype, s);
    case GGML_Q4_1: return launch_dequant<GGML_Q4_1>(blocks, n, out, out_dtype, s);
    case GGML_Q5_0: return launch_dequant<GGML_Q5_0>(blocks, n, out, out_dtype, s);
    case GGML_Q5_1: return launch_dequant<GGML_Q5_1>(blocks, n, out, out_dtype, s);
    case GGML_Q8_0: return launch_dequant<GGML_Q8_0>(blocks, n, out, out_dtype, s);
    case GGML_Q4_K: return launch_dequant<GGML_Q4_K>(blocks, n, out, out_dtype, s);
    case GGML_Q5_K: return launch_dequant<GGML_Q5_K>(blocks, n, out, out_dtype, s);
    case GGML_Q6_K: return launch_dequant<GGML_Q6_K>(blocks, n, out, out_dtype, s);
    case GGML_MXFP4: return launch_dequant<GGML_MXFP4>(blocks, n, out, out_dtype, s);
    case GGML_IQ4_XS: return launch_dequant<GGML_IQ4_XS>(blocks, n, out, out_dtype, s);
    case GGML_IQ3_XXS: return launch_dequant<GGML_IQ3_XXS>(blocks, n, out, out_dtype, s);
    case GGML_IQ3_S: return launch_dequant<GGML_IQ3_S>(blocks, n, out, out_dtype, s);
    case GGML_IQ2_S: return launch_dequant<GGML_IQ2_S>(blocks, n, out, out_dtype, s);
    case GGML_Q1_0: return launch_dequant<GGML_Q1_0>(blocks, n, out, out_dtype, s);
  }
  return tga_set_error("GGML type '%d' is not supported!", ggml_type);   // message of tinygrad/llm/gguf.py:119
}
