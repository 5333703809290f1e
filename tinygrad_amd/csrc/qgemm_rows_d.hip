// Instantiations of qgemm_rows.h: GGML_Q6_K GGML_IQ4_XS
#include "qgemm_rows.h"
int tga_rows_launch_GGML_Q6_K(const RowsArgs& a, int tt, unsigned grid, hipStream_t s) { return rows_launch<GGML_Q6_K>(a, tt, grid, s); }
int tga_rows_launch_GGML_IQ4_XS(const RowsArgs& a, int tt, unsigned grid, hipStream_t s) { return rows_launch<GGML_IQ4_XS>(a, tt, grid, s); }
