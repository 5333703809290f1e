// M = 1 dequant-GEMV kernels of this weight format (template in qgemv1.h)
#include "qgemv1.h"

template int qgemv1_launch_format<F_F16_PAST>(QArgs, hipStream_t);
