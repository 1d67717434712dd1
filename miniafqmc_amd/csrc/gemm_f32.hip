// FP32 products.
#include "gemm_zgemm.hpp"

ZGEMM_LAUNCH(CP_F32, double, double, bfs, true, true)
ZGEMM_LAUNCH(CP_F32, double, double, double, false, false)
ZGEMM_LAUNCH(CP_F32, double, double, double, false, true)
ZGEMM_LAUNCH(CP_F32, double, double, double, true, false)
ZGEMM_LAUNCH(CP_F32, double, double, double, true, true)
ZGEMM_LAUNCH(CP_F32, double, double, float, true, true)
ZGEMM_LAUNCH(CP_F32, double, float, float, true, true)
ZGEMM_LAUNCH(CP_F32, float, double, float, true, false)
ZGEMM_LAUNCH(CP_F32, float, double, float, true, true)
ZGEMM_LAUNCH(CP_F32, float, float, double, true, true)
ZGEMM_LAUNCH(CP_F32, float, float, float, true, false)
ZGEMM_LAUNCH(CP_F32, float, float, float, true, true)
