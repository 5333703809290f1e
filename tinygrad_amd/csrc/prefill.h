// The tables a caller passes to the prefill steps (prefill.hip, prefill16.hip): indices of int64 values, pointers as integers.
#pragma once
#include <string.h>
#include "host.h"

enum { PM_NBLOCKS, PM_DIM, PM_HEADS, PM_KV, PM_HD, PM_MAXCTX, PM_EMB, PM_EMB_TYPE, PM_ROPE, PM_EXPERTS, PM_TOPK, PM_GATING, PM_NORM_TOPK, PM_QKNORM, PM_HIDDEN, PM_DENSE_HIDDEN, PM_EPS_BITS, PM_SCALE_BITS, PM_COUNT };
enum { PB_ATTN_NORM, PB_FFN_NORM, PB_QN, PB_KN, PB_CK, PB_CV, PB_MOE, PB_WQ, PB_WK, PB_WV, PB_WO, PB_GATE, PB_UP, PB_DOWN, PB_ROUTER, PB_TQ, PB_TK, PB_TV, PB_TO, PB_TGATE, PB_TDOWN, PB_COUNT };

static inline float bits_f(int64_t b) { uint32_t u = (uint32_t)b; float f; memcpy(&f, &u, 4); return f; }

// Gating of R rows of router logits (prefill.hip): selection and weights per row, the experts' counts (E zeros before) and each assignment's place among its expert's rows
int pf_gate(const float* logits, int R, int E, int k, int gating, int norm_topk, float scale, int* sel, float* probs, int* counts, int* place, hipStream_t s);
