// Instantiations of qgemm_rows.h: GGML_Q4_K GGML_Q5_K
#include "qgemm_rows.h"
int tga_rows_launch_GGML_Q4_K(const RowsArgs& a, int tt, unsigned grid, hipStream_t s) { return rows_launch<GGML_Q4_K>(a, tt, grid, s); }
int tga_rows_launch_GGML_Q5_K(const RowsArgs& a, int tt, unsigned grid, hipStream_t s) { return rows_launch<GGML_Q5_K>(a, tt, grid, s); }
