// Instantiations of qgemm_rows.h: F_Q4_0P F_Q8_0P
#include "qgemm_rows.h"
int tga_rows_launch_F_Q4_0P(const RowsArgs& a, int tt, unsigned grid, hipStream_t s) { return rows_launch<F_Q4_0P>(a, tt, grid, s); }
int tga_rows_launch_F_Q8_0P(const RowsArgs& a, int tt, unsigned grid, hipStream_t s) { return rows_launch<F_Q8_0P>(a, tt, grid, s); }
