// The matrix-product kernels' tile candidates and launchers.  The launchers
// are instantiated in gemm_f32.hip, gemm_b16.hip, gemm_b16b.hip, gemm_ring.hip
// and gemm_f64.hip, so that the kernels compile side by side.
#pragma once
#include "gemm.hpp"
#include "gemm_f64.hpp"

// zgemm_kernel: FP32 (BKC 16 or 8 complex) and split-BF16 (BKC 16)
struct TileCfg {
  int BM, BNC, WM, WN;
};
constexpr TileCfg kCfgF32[] = {{32, 16, 1, 1}, {128, 64, 2, 2}, {128, 128, 2, 2}};
constexpr TileCfg kCfgB16[] = {{32, 16, 1, 1}, {128, 64, 2, 2}, {128, 128, 2, 2}, {256, 64, 4, 2}, {64, 64, 2, 2}};
constexpr int kNF32 = 3, kNB16 = 5;

// Split-BF16 products whose operands are both split-BF16 with k contiguous
// run zgemm_b16dma_kernel (both operands staged by direct loads through a
// ring of LDS stages); candidates (rows, complex columns, waves, stages):
struct RingCfg {
  int BM, BN, WM, WN, S;
};
constexpr RingCfg kRing[] = {
    {128, 128, 2, 2, 2}, {256, 128, 4, 2, 2}, {128, 256, 2, 4, 2}, {256, 128, 4, 2, 3}, {64, 64, 2, 2, 2}, {32, 32, 2, 2, 4}};
// three-piece operands take half as much LDS again per stage
constexpr RingCfg kRing3[] = {
    {128, 128, 2, 2, 2}, {256, 128, 4, 2, 2}, {128, 256, 2, 4, 2}, {128, 128, 2, 2, 3}, {64, 64, 2, 2, 2}};
constexpr int kNRing = 6, kNRing3 = 5, kNExch = 5;
// relative rates with the chip full, by pieces: the HS potential, the bias
// and the propagator products at 256 to 512 orbitals
// (the last tile is for long sums over few outputs, which leave most CUs idle
// in 64 x 64 tiles: its rate lets it win where those fill half the chip or less)
constexpr double kRingRate[] = {0.87, 1.0, 1.0, 1.02, 0.85, 0.42};
constexpr double kRingRate3[] = {0.95, 1.0, 1.0, 0.92, 0.93};
// FP32 operands, small tiles: three to five workgroups a CU cover each other's
// barriers (HS potential at 300 orbitals, 128 walkers, 1200 vectors: 111, 117
// and 111 TFLOP/s; 128 x 64 and 128 x 128 with eight waves 110 and 104, a third
// stage of 64 x 64 or a fourth of 32 x 32 no gain)
constexpr RingCfg kRingF[] = {{32, 32, 2, 2, 3}, {64, 64, 2, 2, 2}, {64, 32, 2, 2, 3}};
constexpr int kNRingF = 3;
constexpr double kRingRateF[] = {0.95, 1.0, 0.95};
template <int NP> constexpr int ring_count() { return NP == 0 ? kNRingF : NP == 3 ? kNRing3 : kNRing; }
template <int NP> constexpr RingCfg ring_cfg(int i) { return NP == 0 ? kRingF[i] : NP == 3 ? kRing3[i] : kRing[i]; }
template <int NP> constexpr double ring_rate(int i)
{
  return NP == 0 ? kRingRateF[i] : NP == 3 ? kRingRate3[i] : kRingRate[i];
}

// FP64 products (zgemm_f64_kernel): every operand order, tile candidates
// (rows, complex columns, waves, LDS stages).
struct F64Cfg {
  int BM, BN, WM, WN, S;
};
constexpr F64Cfg kF64[] = {{32, 32, 2, 2, 3}, {64, 64, 2, 2, 2}, {128, 64, 4, 2, 2}};
constexpr int kNF64 = 3;
// TFLOP/s with the chip full (2048 x 128 x 128 x 512)
constexpr double kF64Rate[] = {57.4, 62.7, 63.9};

// tiles: the grid; ci: the candidate; dma: split-BF16 operands staged by
// direct loads (0 none, 1 A, 2 both)
template <int CP, class AT, class BT, class OT, bool AK, bool BK>
void zgemm_launch(hipStream_t st, const ZGemmArgs& a, unsigned tiles, int ci, int dma);
template <class OT, int NP> void ring_launch(hipStream_t st, const ZGemmArgs& a, unsigned tiles, int ri);
template <class OZ> void f64_launch(hipStream_t st, const F64Args& a, unsigned tiles, int ci, bool dma);
// the exchange energy (a.x, grid from exch_grid)
template <int NP> void ring_exch_launch(hipStream_t st, const ZGemmArgs& a, unsigned tiles, int ri);
void f64_exch_launch(hipStream_t st, const F64Args& a, unsigned tiles, int ci);
