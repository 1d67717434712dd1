// Batched FP64 complex GEMM on v_mfma_f64_16x16x4_f64.
//
//   C(m,n) = alpha * sum_k opA(m,k) * opB(n,k) + F(m,n) + beta * C(m,n)
//
// opA / opB: the operand or its conjugate.  Operands may have any strides;
// rows (m) and columns (n) may be folded, index -> (index / inner) * outer
// stride + (index % inner) * stride, so that a batch that shares one operand
// runs as one tall product without a partial tile per batch item.
//
// Bound: the matrix cores.  One MFMA takes 64 cycles of its SIMD for 2048
// flops, so a 32 x 32 complex wave tile has 2048 cycles of MFMA per k-tile of
// 8 against 8 LDS reads of 16 bytes per lane (16 x 16, for outputs that would
// leave CUs idle: 512 against 4); what the kernel has to get right is that no
// wave ever waits on memory.  Each k-tile (8 complex = 128
// bytes per row) goes from global memory straight into LDS
// (global_load_lds_dwordx4, one complex per lane, any operand order since
// every lane has an address of its own), STAGES k-tiles in a ring: the loads
// of tile t + STAGES - 1 are issued after the barrier of tile t and waited
// for with a vmcnt that leaves the later tiles in flight.  Chunk c (one
// complex) of tile row R sits at c ^ swz(R), so that the 16 rows of a
// fragment read fall on distinct 16-byte bank groups.
//
// The real and imaginary parts of a 16 x 16 complex block have accumulators
// of their own: re += a_re b_re, re += a_im (-b_im), im += a_re b_im,
// im += a_im b_re per group of four k, ascending.  That order does not depend
// on the tile shape, so every shape gives the same bits.
//
// Measured (MI355X; before: one kernel for all precisions, B expanded to its
// real 2 x 2 form in registers and both operands staged through them):
// 2048 x (128 x 128 x 512) 3.76 -> 2.15 ms (64 TFLOP/s), 256 x (256 x 128 x
// 256) 0.51 -> 0.29 ms, 1024 x 256 x 32768 1.80 -> 1.07 ms; a plain FP64
// matrix product of the library reaches 72.8 TFLOP/s.  Four-wave tiles of
// 64 x 64 and eight-wave tiles of 128 x 64 (32 x 32 per wave) beat 64 x 32 per
// wave (53 TFLOP/s: half the waves to cover the LDS reads); a third stage
// gains nothing but for the 32 x 32 tile.
//
// Rows past m and columns past n read the last valid one (their results are
// not stored); k past the end reads the last valid k and both fragments are
// zeroed, so nothing outside the operands is touched or enters the sums.
#pragma once
#include "common.hpp"

struct F64Args {
  const void* A;
  const void* B;
  void* C;
  const void* F;              // added when not null (C's element type)
  int m, n, k;
  int mi, ni;                 // inner extents of folded rows and columns (m, n: not folded)
  long sam, samo, sak;        // A(row, k), complex elements
  long sbn, sbno, sbk;        // B(col, k)
  long scm, scmo, scn, scno;  // C(row, col)
  long sfm, sfmo, sfn, sfno;  // F(row, col)
  // batch b -> offset (b / bdiv) * s1 + (b % bdiv) * s2 (F: as C)
  int bdiv;
  long sa1, sa2, sb1, sb2, sc1, sc2;
  double ar, ai, br, bi;
  int conja, conjb;
  // lower-triangular B: B(n, k) = 0 for k > n, so a tile of columns
  // [n0, n0 + BN) stops its k loop at n0 + BN; heavy tiles run first
  int ktri;
  // k split over the batch: item b % bdiv covers k of ktot from (b % bdiv) * k
  // (0: every item covers k)
  long ktot;
  int MT, NT;                 // tile grid (filled by the launcher)
  // XD mode: A, B at the spin and chunk (0, 0), m walkers
  ExchArgs x;
};

namespace f64g {

__device__ __forceinline__ void put(zd* p, long o, double re, double im) { p[o] = zd{re, im}; }
__device__ __forceinline__ void put(zf* p, long o, double re, double im) { p[o] = zf{(float)re, (float)im}; }
__device__ __forceinline__ void put(zb* p, long o, double re, double im) { p[o] = split_z((float)re, (float)im); }

} // namespace f64g

// OZ: element of C and F (zd, zf; zb without F and beta).  DMA = false: the
// operands pass through registers (operands not aligned to 16 bytes).  XD:
// the exchange energy (ExchArgs), the tile's product dotted with G into one
// partial per walker instead of being stored.
template <class OZ, int BM, int BN, int WM, int WN, int STAGES, bool DMA = true, bool XD = false>
__global__ __launch_bounds__(64 * WM * WN) void zgemm_f64_kernel(F64Args p)
{
  constexpr int NT = 64 * WM * WN;
  constexpr int WTM = BM / WM, WTN = BN / WN;
  constexpr int TM = WTM / 16, TN = WTN / 16;
  constexpr int KT = 8;
  constexpr int AL = BM * KT / NT, BL = BN * KT / NT;  // 16-byte loads per thread per tile
  constexpr int LPT = AL + BL;
  static_assert(WTM % 16 == 0 && WTN % 16 == 0, "wave tile must be a multiple of 16");
  static_assert((BM * KT) % NT == 0 && (BN * KT) % NT == 0, "tiles must split evenly over the threads");
  static_assert(NT % 128 == 0, "a thread's loads must share one chunk");
  static_assert(STAGES >= 2 && STAGES <= 4 && LPT * (STAGES - 2) < 64, "stages");
  constexpr int STG = (BM + BN) * KT;
  __shared__ __align__(16) zd s0[STG];
  __shared__ __align__(16) zd s1[STG];
  __shared__ __align__(16) zd s2[STAGES > 2 ? STG : 1];
  __shared__ __align__(16) zd s3[STAGES > 3 ? STG : 1];

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int wm = wave % WM, wn = wave / WM;
  const int g = lane >> 4, r = lane & 15;

  // XCD-aware tile order (as zgemm_kernel): ids go round-robin over the 8
  // XCDs, so each gets a contiguous run of tiles; triangular products deal
  // their column tiles round-robin instead, heaviest first
  long lin = blockIdx.x;
  ExchTile xt{};
  if constexpr (XD) {
    if (!exch_tile(p.x, p.MT, BN, xt)) return;
  } else {
    const long T = gridDim.x, per = T / 8;
    if (p.ktri) {
      if ((p.NT & 7) == 0 && T == (long)p.MT * p.NT) {
        const long x = lin & 7, q = lin >> 3;
        lin = (x + 8 * (q / p.MT)) * p.MT + q % p.MT;
      }
    } else if (per > 0 && lin < per * 8) {
      lin = (lin % 8) * per + lin / 8;
    }
  }
  const int mt = XD ? xt.mt : (int)(lin % p.MT);
  const long rest = lin / p.MT;
  const int ntl = (int)(rest % p.NT);
  const int m0 = mt * BM, n0 = XD ? xt.n0 : (p.ktri ? p.NT - 1 - ntl : ntl) * BN;
  const int b = XD ? 0 : (int)(rest / p.NT);
  const long bq = XD ? 0 : b / p.bdiv, br_ = XD ? 0 : b % p.bdiv;
  const int pn = XD ? (int)(p.x.NM - xt.q0) : p.n;
  int kend = p.k;
  if constexpr (XD) {
    kend = (int)min(min(p.x.xch, p.x.NM - xt.q0), (long)(n0 + BN));
  } else {
    if (p.ktot) kend = (int)min((long)p.k, p.ktot - br_ * p.k);
    if (p.ktri) kend = min(kend, n0 + BN);
  }
  const zd* A = (const zd*)p.A + (XD ? xt.sp * p.x.NM + xt.q0 : bq * p.sa1 + br_ * p.sa2);
  const zd* B = (const zd*)p.B + (XD ? (xt.sp * p.x.NM + xt.q0) * p.x.NM + xt.q0 : bq * p.sb1 + br_ * p.sb2);

  // unit u = i * NT + tid of a tile is (row u / 8, slot u % 8) and holds the
  // row's k = slot ^ swz(row), which is the same for all of a thread's units
  const int kc = (tid & 7) ^ dma::swz(tid >> 3);
  const zd* pa[AL];
  const zd* pb[BL];
#pragma unroll
  for (int i = 0; i < AL; i++) {
    const int row = min(m0 + (i * NT + tid) / KT, p.m - 1);
    pa[i] = A + (XD ? (long)row * p.sam : (long)(row / p.mi) * p.samo + (long)(row % p.mi) * p.sam) + (long)kc * p.sak;
  }
#pragma unroll
  for (int i = 0; i < BL; i++) {
    const int col = min(n0 + (i * NT + tid) / KT, pn - 1);
    pb[i] = B + (XD ? (long)col * p.sbn : (long)(col / p.ni) * p.sbno + (long)(col % p.ni) * p.sbn) + (long)kc * p.sbk;
  }
  const int w0 = __builtin_amdgcn_readfirstlane(wave);
  const int klast = kend - 1 - kc;  // largest k0 whose chunk lies inside (may be negative)
  auto issue = [&](zd* st, int k0) __attribute__((always_inline)) {
    const int ko = min(k0, klast);
    const long oa = (long)ko * p.sak, ob = (long)ko * p.sbk;
    if constexpr (DMA) {
#pragma unroll
      for (int i = 0; i < AL; i++)
        __builtin_amdgcn_global_load_lds((const void*)(pa[i] + oa),
                                         (__attribute__((address_space(3))) void*)&st[i * NT + w0 * 64], 16, 0, 0);
#pragma unroll
      for (int i = 0; i < BL; i++)
        __builtin_amdgcn_global_load_lds((const void*)(pb[i] + ob),
                                         (__attribute__((address_space(3))) void*)&st[BM * KT + i * NT + w0 * 64], 16,
                                         0, 0);
    } else {
#pragma unroll
      for (int i = 0; i < AL; i++) st[i * NT + tid] = zd{pa[i][oa].re, pa[i][oa].im};
#pragma unroll
      for (int i = 0; i < BL; i++) st[BM * KT + i * NT + tid] = zd{pb[i][ob].re, pb[i][ob].im};
    }
  };

  doublex4 cr[TM][TN], ci[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int q = 0; q < 4; q++) cr[i][j][q] = ci[i][j][q] = 0.0;

  // fragment rows are 16-aligned blocks + r, so swz(row) = swz(r); lane group
  // g takes k = 4 kq + g
  const int sw = dma::swz(r);
  const int arow = wm * WTM + r, brow = BM + wn * WTN + r;
  const unsigned long long sa_ = p.conja ? 0x8000000000000000ull : 0ull, sb_ = p.conjb ? 0x8000000000000000ull : 0ull;
  auto flip = [](double x, unsigned long long s) __attribute__((always_inline)) {
    return __longlong_as_double((long long)((unsigned long long)__double_as_longlong(x) ^ s));
  };
  struct Frags {
    zd a[2][TM], b[2][TN];
  };
  auto read = [&](const zd* st, int k0, Frags& f) __attribute__((always_inline)) {
#pragma unroll
    for (int kq = 0; kq < 2; kq++) {
      const int c = (4 * kq + g) ^ sw;
      const bool in = k0 + 4 * kq + g < kend;
#pragma unroll
      for (int i = 0; i < TM; i++) {
        const zd v = st[(arow + 16 * i) * KT + c];
        f.a[kq][i] = zd{in ? v.re : 0.0, in ? flip(v.im, sa_) : 0.0};
      }
#pragma unroll
      for (int j = 0; j < TN; j++) {
        const zd v = st[(brow + 16 * j) * KT + c];
        f.b[kq][j] = zd{in ? v.re : 0.0, in ? flip(v.im, sb_) : 0.0};
      }
    }
  };
  auto mfmas = [&](const Frags& f) __attribute__((always_inline)) {
#pragma unroll
    for (int kq = 0; kq < 2; kq++) {
      // the two MFMAs of one accumulator are 2 TM TN apart
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) {
          cr[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(f.a[kq][i].re, f.b[kq][j].re, cr[i][j], 0, 0, 0);
          ci[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(f.a[kq][i].re, f.b[kq][j].im, ci[i][j], 0, 0, 0);
        }
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) {
          cr[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(f.a[kq][i].im, -f.b[kq][j].im, cr[i][j], 0, 0, 0);
          ci[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(f.a[kq][i].im, f.b[kq][j].re, ci[i][j], 0, 0, 0);
        }
    }
  };

  const int nk = (kend + KT - 1) / KT;
  // Step j issues tile j into stage j % STAGES and computes tile
  // c = j - (STAGES - 1): wait until tile c has landed (the later ones stay
  // in flight), barrier (every wave has also finished reading tile c - 1,
  // whose stage tile j refills), read the fragments, issue tile j, multiply.
  auto step = [&](auto stc, int j) __attribute__((always_inline)) {
    constexpr int ST = decltype(stc)::value;
    constexpr int SC = (ST + 1) % STAGES;
    zd* in_ = ST == 0 ? s0 : ST == 1 ? s1 : ST == 2 ? s2 : s3;
    const zd* cs = SC == 0 ? s0 : SC == 1 ? s1 : SC == 2 ? s2 : s3;
    const int c = j - (STAGES - 1);
    Frags f;
    if (c >= 0) {
      if constexpr (DMA) {
        const int ahead = min(nk - 1 - c, STAGES - 2);  // tiles issued after c
        if (ahead >= 2) dma::wait_vmcnt<(STAGES > 3 ? 2 * LPT : 0)>();
        else if (ahead == 1) dma::wait_vmcnt<(STAGES > 2 ? LPT : 0)>();
        else dma::wait_vmcnt<0>();
        __builtin_amdgcn_s_barrier();
      } else {
        __syncthreads();
      }
      read(cs, c * KT, f);
    }
    if (j < nk) issue(in_, j * KT);
    if (c >= 0) mfmas(f);
  };
  for (int j = 0; j < nk + STAGES - 1; j += STAGES) {
    step(std::integral_constant<int, 0>(), j);
    if (j + 1 < nk + STAGES - 1) step(std::integral_constant<int, 1>(), j + 1);
    if constexpr (STAGES > 2)
      if (j + 2 < nk + STAGES - 1) step(std::integral_constant<int, 2>(), j + 2);
    if constexpr (STAGES > 3)
      if (j + 3 < nk + STAGES - 1) step(std::integral_constant<int, 3>(), j + 3);
  }

  if constexpr (XD) {
    // lane: element (walker 4q + g, row r) of each block; the tile's dot per
    // walker over the lane's rows, the 16 lanes of a group, then the WN waves
    __shared__ zd red[WN][BM];
    const zd* G = p.x.G + xt.sp * p.x.NM + xt.q0 + n0 + wn * WTN + r;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int lw = wm * WTM + 16 * i + 4 * q + g;
        const zd* Gw = G + (long)min(m0 + lw, p.m - 1) * 2 * p.x.NM;
        zd a{0.0, 0.0};
#pragma unroll
        for (int j = 0; j < TN; j++) {
          if (n0 + wn * WTN + 16 * j + r >= pn) continue;
          const double y_r = p.ar * cr[i][j][q], y_i = p.ar * ci[i][j][q];
          const zd gv = Gw[16 * j];
          a.re += gv.re * y_r - gv.im * y_i;
          a.im += gv.re * y_i + gv.im * y_r;
        }
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) {
          a.re += __shfl_xor(a.re, o);
          a.im += __shfl_xor(a.im, o);
        }
        if (r == 0) red[wn][lw] = a;
      }
    __syncthreads();
    for (int lw = tid; lw < BM; lw += NT) {
      if (m0 + lw >= p.m) continue;
      zd a = red[0][lw];
#pragma unroll
      for (int v = 1; v < WN; v++) a = zadd(a, red[v][lw]);
      p.x.part[((long)xt.sp * p.x.xt + xt.t) * p.m + m0 + lw] = a;
    }
    return;
  }
  // epilogue: the lane holds complex element (row 4q + g, column r) of each
  // 16 x 16 block
  const long coff = bq * p.sc1 + br_ * p.sc2;
  OZ* C = (OZ*)p.C + coff;
  const OZ* F = p.F ? (const OZ*)p.F + coff : nullptr;
  const bool has_beta = (p.br != 0.0 || p.bi != 0.0);
  long co[TN], fo[TN];
#pragma unroll
  for (int j = 0; j < TN; j++) {
    const int col = min(n0 + wn * WTN + 16 * j + r, p.n - 1);
    co[j] = (long)(col / p.ni) * p.scno + (long)(col % p.ni) * p.scn;
    fo[j] = (long)(col / p.ni) * p.sfno + (long)(col % p.ni) * p.sfn;
  }
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int row = m0 + wm * WTM + 16 * i + 4 * q + g;
      if (row >= p.m) continue;
      const long ro = (long)(row / p.mi) * p.scmo + (long)(row % p.mi) * p.scm;
      const long rf = (long)(row / p.mi) * p.sfmo + (long)(row % p.mi) * p.sfm;
      zd fv[TN], cv[TN];
      if constexpr (!std::is_same<OZ, zb>::value) {
#pragma unroll
        for (int j = 0; j < TN; j++) {
          fv[j] = F ? to_zd(F[rf + fo[j]]) : zd{0.0, 0.0};
          cv[j] = has_beta ? to_zd(C[ro + co[j]]) : zd{0.0, 0.0};
        }
      }
#pragma unroll
      for (int j = 0; j < TN; j++) {
        if (n0 + wn * WTN + 16 * j + r >= p.n) continue;
        const double re = cr[i][j][q], im = ci[i][j][q];
        double ore = p.ar * re - p.ai * im, oim = p.ar * im + p.ai * re;
        if constexpr (!std::is_same<OZ, zb>::value) {
          if (has_beta) {
            ore += p.br * cv[j].re - p.bi * cv[j].im;
            oim += p.br * cv[j].im + p.bi * cv[j].re;
          }
          ore += fv[j].re;
          oim += fv[j].im;
        }
        f64g::put(C, ro + co[j], ore, oim);
      }
    }
}
