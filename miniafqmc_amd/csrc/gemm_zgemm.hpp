// zgemm_kernel's launcher, for the files that instantiate it.
#pragma once
#include "gemm_launch.hpp"

template <int CP, class AT, class BT, class OT, bool AK, bool BK>
void zgemm_launch(hipStream_t st, const ZGemmArgs& a, unsigned tiles, int ci, int dma)
{
  auto go = [&](auto cic) {
    constexpr int CI = decltype(cic)::value;
    constexpr TileCfg t = CP == CP_F32 ? kCfgF32[CI < kNF32 ? CI : 0] : kCfgB16[CI];
    constexpr int BKC = (CP == CP_BF16X3) ? 16 : (t.WM * t.WN == 1 ? 16 : 8);
    const dim3 grid(tiles), block(64 * t.WM * t.WN);
    if constexpr (CP == CP_BF16X3 && std::is_same<AT, bfs>::value && AK) {
      if constexpr (std::is_same<BT, bfs>::value && BK) {
        if (dma == 2) {
          hipLaunchKernelGGL((zgemm_kernel<CP, AT, BT, OT, AK, BK, t.BM, t.BNC, BKC, t.WM, t.WN, true, true>), grid, block,
                             0, st, a);
          return;
        }
      }
      if (dma >= 1) {
        hipLaunchKernelGGL((zgemm_kernel<CP, AT, BT, OT, AK, BK, t.BM, t.BNC, BKC, t.WM, t.WN, true>), grid, block, 0,
                           st, a);
        return;
      }
    }
    hipLaunchKernelGGL((zgemm_kernel<CP, AT, BT, OT, AK, BK, t.BM, t.BNC, BKC, t.WM, t.WN>), grid, block, 0, st, a);
  };
  switch (ci) {
  case 1: return go(std::integral_constant<int, 1>());
  case 2: return go(std::integral_constant<int, 2>());
  case 3:
    if constexpr (CP == CP_BF16X3) return go(std::integral_constant<int, 3>());
    break;
  case 4:
    if constexpr (CP == CP_BF16X3) return go(std::integral_constant<int, 4>());
    break;
  }
  go(std::integral_constant<int, 0>());
}

#define ZGEMM_LAUNCH(CP, AT, BT, OT, AK, BK) \
  template void zgemm_launch<CP, AT, BT, OT, AK, BK>(hipStream_t, const ZGemmArgs&, unsigned, int, int);
