// Instantiations of qgemm_rows.h: GGML_F16 GGML_MXFP4
#include "qgemm_rows.h"
int tga_rows_launch_GGML_F16(const RowsArgs& a, int tt, unsigned grid, hipStream_t s) { return rows_launch<GGML_F16>(a, tt, grid, s); }
int tga_rows_launch_GGML_MXFP4(const RowsArgs& a, int tt, unsigned grid, hipStream_t s) { return rows_launch<GGML_MXFP4>(a, tt, grid, s); }
