// Split-BF16 products through zgemm_kernel, second half.
#include "gemm_zgemm.hpp"

ZGEMM_LAUNCH(CP_BF16X3, bfs, bfs, float, true, true)
ZGEMM_LAUNCH(CP_BF16X3, bfs, double, float, true, true)
ZGEMM_LAUNCH(CP_BF16X3, bfs, float, bfs, true, false)
ZGEMM_LAUNCH(CP_BF16X3, double, bfs, float, true, true)
ZGEMM_LAUNCH(CP_BF16X3, double, double, bfs, true, true)
ZGEMM_LAUNCH(CP_BF16X3, double, double, double, false, true)
ZGEMM_LAUNCH(CP_BF16X3, double, double, double, true, false)
