// Device-resident decode bookkeeping shared by the decode-step kernels.
#pragma once
#include <stdint.h>
#include <hip/hip_runtime.h>

struct DecodeState {   // 16 int32
  int pos;             // position of the token being processed
  int token;           // current input token id
  int step;            // tokens generated so far
  int n_prompt;        // prompt length: while pos + 1 < n_prompt the next input token comes from the prompt, not from argmax
  int error;           // set by kernels that refuse their input instead of reading out of bounds: bit 0 token id outside the table, bit 1 position >= max_ctx
  int vocab;           // rows of the embedding table (0: unknown, token ids are then not checked)
  int pad[10];
};

// The one-launch attention of a decode step (whole-row q / k norms, heads of 64 or 128) for several rows of one sequence, positions pos0 .. pos0 + rows - 1, with its bits: a row's q, k and v `stride` floats
// behind the row's before; partials [rows][heads][splits x head_dim + 16].  append_only: their keys and values alone.  attn_split_rows_splits: splits of that attention, 0 where it has no such form
int attn_split_rows_splits(int max_ctx);
int attn_split_rows(const float* q, const float* k, const float* v, long long stride, const float* q_norm_weight, const float* k_norm_weight, float norm_eps, void* cache_k, void* cache_v, float* partials,
                    int rows, int pos0, int n_heads, int n_kv_heads, int head_dim, int max_ctx, const float* rope_table, bool append_only, hipStream_t s);
