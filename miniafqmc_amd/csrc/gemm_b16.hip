// Split-BF16 products through zgemm_kernel, first half (gemm_b16b.hip holds the others).
#include "gemm_zgemm.hpp"

ZGEMM_LAUNCH(CP_BF16X3, bfs, bfs, bfs, true, true)
ZGEMM_LAUNCH(CP_BF16X3, bfs, bfs, double, true, true)
ZGEMM_LAUNCH(CP_BF16X3, bfs, double, float, true, false)
ZGEMM_LAUNCH(CP_BF16X3, double, double, double, false, false)
ZGEMM_LAUNCH(CP_BF16X3, double, double, double, true, true)
