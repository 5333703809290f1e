// Instantiations of qgemm_rows.h: GGML_Q4_1 GGML_Q5_0 GGML_Q5_1
#include "qgemm_rows.h"
int tga_rows_launch_GGML_Q4_1(const RowsArgs& a, int tt, unsigned grid, hipStream_t s) { return rows_launch<GGML_Q4_1>(a, tt, grid, s); }
int tga_rows_launch_GGML_Q5_0(const RowsArgs& a, int tt, unsigned grid, hipStream_t s) { return rows_launch<GGML_Q5_0>(a, tt, grid, s); }
int tga_rows_launch_GGML_Q5_1(const RowsArgs& a, int tt, unsigned grid, hipStream_t s) { return rows_launch<GGML_Q5_1>(a, tt, grid, s); }
