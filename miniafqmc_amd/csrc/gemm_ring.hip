// Split-BF16 and FP32 products through the staged-ring kernel.
#include "gemm_b16.hpp"
#include "gemm_launch.hpp"

namespace {
template <class OT, int NP, bool XD> void ring_go(hipStream_t st, const ZGemmArgs& a, unsigned tiles, int ri)
{
  auto go = [&](auto ric) {
    constexpr int RI = decltype(ric)::value;
    constexpr RingCfg t = ring_cfg<NP>(RI < ring_count<NP>() ? RI : 0);
    hipLaunchKernelGGL((zgemm_b16dma_kernel<OT, t.BM, t.BN, t.WM, t.WN, t.S, NP, XD>), dim3(tiles),
                       dim3(64 * t.WM * t.WN), 0, st, a);
  };
  switch (ri) {
  case 1: return go(std::integral_constant<int, 1>());
  case 2: return go(std::integral_constant<int, 2>());
  case 3:
    if constexpr (3 < ring_count<NP>()) return go(std::integral_constant<int, 3>());
    break;
  case 4:
    if constexpr (4 < ring_count<NP>()) return go(std::integral_constant<int, 4>());
    break;
  case 5:
    if constexpr (5 < ring_count<NP>() && !XD) return go(std::integral_constant<int, 5>());
    break;
  }
  go(std::integral_constant<int, 0>());
}
} // namespace

template <class OT, int NP> void ring_launch(hipStream_t st, const ZGemmArgs& a, unsigned tiles, int ri)
{
  ring_go<OT, NP, false>(st, a, tiles, ri);
}
template <int NP> void ring_exch_launch(hipStream_t st, const ZGemmArgs& a, unsigned tiles, int ri)
{
  ring_go<float, NP, true>(st, a, tiles, ri);
}
template void ring_exch_launch<0>(hipStream_t, const ZGemmArgs&, unsigned, int);
template void ring_exch_launch<2>(hipStream_t, const ZGemmArgs&, unsigned, int);
template void ring_exch_launch<4>(hipStream_t, const ZGemmArgs&, unsigned, int);
template void ring_exch_launch<3>(hipStream_t, const ZGemmArgs&, unsigned, int);

#define RING_LAUNCH(OT, NP) template void ring_launch<OT, NP>(hipStream_t, const ZGemmArgs&, unsigned, int);
RING_LAUNCH(float, 0)
RING_LAUNCH(double, 0)
RING_LAUNCH(bfs, 1)
RING_LAUNCH(bfs, 2)
RING_LAUNCH(float, 2)
RING_LAUNCH(double, 2)
RING_LAUNCH(bfs, 4)
RING_LAUNCH(float, 4)
RING_LAUNCH(double, 4)
RING_LAUNCH(bfs, 3)
RING_LAUNCH(float, 3)
RING_LAUNCH(double, 3)
