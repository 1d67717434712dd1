// FP64 products.
#include "gemm_launch.hpp"

template <class OZ> void f64_launch(hipStream_t st, const F64Args& a, unsigned tiles, int ci, bool dma)
{
  auto go = [&](auto cic, auto dmac) {
    constexpr F64Cfg t = kF64[decltype(cic)::value];
    hipLaunchKernelGGL((zgemm_f64_kernel<OZ, t.BM, t.BN, t.WM, t.WN, t.S, decltype(dmac)::value>), dim3(tiles),
                       dim3(64 * t.WM * t.WN), 0, st, a);
  };
  if (!dma) return go(std::integral_constant<int, 0>(), std::false_type());
  switch (ci) {
  case 1: return go(std::integral_constant<int, 1>(), std::true_type());
  case 2: return go(std::integral_constant<int, 2>(), std::true_type());
  default: return go(std::integral_constant<int, 0>(), std::true_type());
  }
}

#define F64_LAUNCH(OZ) template void f64_launch<OZ>(hipStream_t, const F64Args&, unsigned, int, bool);
F64_LAUNCH(zd)
F64_LAUNCH(zf)
F64_LAUNCH(zb)

void f64_exch_launch(hipStream_t st, const F64Args& a, unsigned tiles, int ci)
{
  auto go = [&](auto cic) {
    constexpr F64Cfg t = kF64[decltype(cic)::value];
    hipLaunchKernelGGL((zgemm_f64_kernel<zd, t.BM, t.BN, t.WM, t.WN, t.S, true, true>), dim3(tiles),
                       dim3(64 * t.WM * t.WN), 0, st, a);
  };
  switch (ci) {
  case 1: return go(std::integral_constant<int, 1>());
  case 2: return go(std::integral_constant<int, 2>());
  default: return go(std::integral_constant<int, 0>());
  }
}
