// The propagator of small systems, one kernel per substep (prop_small.hpp).
//
// A block of columns of each product P W, V U_k, P U_1 needs only the same
// columns of its right operand, so a workgroup takes one walker and NB of its
// 2N columns (both spins side by side) through all eight products.  Wave i
// owns rows 16 i .. 16 i + 15 and keeps its 16 x M part of the left operand in
// registers as MFMA fragments: V is read once for the six Horner steps, P
// twice.  The right operand U passes through LDS (two buffers, one barrier per
// product) and S = P W, which every Horner step adds, stays in registers.
//
// Bound: latency.  At these sizes a product of the GEMM chain is 10-30 us of
// launch, first loads and a short k loop for under 2 us of MFMA; here a product
// costs its MFMAs, the LDS reads of U and a barrier.  Measured per substep
// (MI355X, eight-product chain -> this kernel, us), walkers at orbitals /
// electrons: FP64 16 at 64 / 16 63 -> 25, 512 at 128 / 64 1404 -> 1289; FP32
// 128 at 192 / 48 667 -> 365; split-BF16 64 at 96 / 24 129 -> 22, 128 at 192 /
// 48 389 -> 197, 512 at 192 / 96 2230 -> 1426.  It won at every size tried up
// to 192 orbitals (128 in FP64), where the fragments stop fitting the
// registers.
//
// The arithmetic is the chain's, in its order: per k-tile (split-BF16: 16
// complex, h*h, h*m, m*h; FP32 and FP64: 4 complex, a_re then a_im), FP32 or
// FP64 accumulation, epilogues in FP64, terms rounded to the format between
// products; the results are the same bit for bit.
#include "prop_small.hpp"

#include <type_traits>

namespace {

template <class Z> struct Fmt;
template <> struct Fmt<zd> {
  using ACC = doublex4;
  using R = double;
  static constexpr int PAD = 1, FMT = 0;
};
template <> struct Fmt<zf> {
  using ACC = floatx4;
  using R = float;
  static constexpr int PAD = 1, FMT = 1;
};
template <> struct Fmt<zb> {
  using ACC = floatx4;
  using R = float;
  static constexpr int PAD = 2, FMT = 2;
};

// the left operand's 16 rows x 16 k of one lane: zb 4 consecutive k (4g ..),
// zf and zd k = 4 q + g
template <class Z> struct Frag {
  Z v[4];
};

// s + i al (re + i im), products and sums rounded one by one as the chain's
// epilogues round them
__device__ __forceinline__ zd horner_term(double sr, double si, double al, double re, double im)
{
#pragma clang fp contract(off)
  const double o_r = al * im, o_i = al * re;
  return zd{sr - o_r, si + o_i};
}

__device__ __forceinline__ zd conv(zd v, zd) { return v; }
__device__ __forceinline__ zf conv(zd v, zf) { return zf{(float)v.re, (float)v.im}; }
__device__ __forceinline__ zb conv(zd v, zb) { return split_z((float)v.re, (float)v.im); }

template <class Z, int MT, int NB> __global__ __launch_bounds__(64 * MT) void prop_small_kernel(PropSmallArgs a)
{
  using F = Fmt<Z>;
  using ACC = typename F::ACC;
  using R = typename F::R;
  constexpr int NT = 64 * MT, MP = 16 * MT, LD = MP + F::PAD, NJ = NB / 16;
  __shared__ __align__(16) Z u0[NB * LD];
  __shared__ __align__(16) Z u1[NB * LD];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 4, r = lane & 15;
  const int M = a.M, N = a.N, nk = (M + 15) / 16;
  // the column blocks of one walker run on one XCD: its V comes into one L2
  long lin = blockIdx.x;
  {
    const long T = gridDim.x, per = T / 8;
    if (per > 0 && lin < per * 8) lin = (lin % 8) * per + lin / 8;
  }
  const int w = (int)(lin / a.ncb), c0 = (int)(lin % a.ncb) * NB;
  zd* Ww = a.W + (long)w * 2 * M * N;
  const Z* Vw = (const Z*)a.V + (long)w * M * M;
  const Z* P = (const Z*)a.P;

  const int row = 16 * wave + r;  // the lane's row of the left operand
  Frag<Z> fa[MT];
  auto load = [&](const Z* A) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < MT; t++) {
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int k = 16 * t + (F::FMT == 2 ? 4 * g + q : 4 * q + g);
        fa[t].v[q] = Z{0, 0};
        if (row < M && k < M) fa[t].v[q] = A[(long)row * M + k];
      }
    }
  };
  // rows of 4 k at a time where they are 16-byte aligned (split-BF16)
  auto load4 = [&](const Z* A) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < MT; t++) {
      const int k = 16 * t + 4 * g;
      uint4 x = make_uint4(0, 0, 0, 0), y = x;
      if (row < M && k < M) {
        const uint4* p4 = (const uint4*)(A + (long)row * M + k);
        x = p4[0];
        y = p4[1];
      }
      if constexpr (F::FMT == 2) {
        fa[t].v[0] = zb{x.x, x.y};
        fa[t].v[1] = zb{x.z, x.w};
        fa[t].v[2] = zb{y.x, y.y};
        fa[t].v[3] = zb{y.z, y.w};
      }
    }
  };
  const bool wide = F::FMT == 2 && (M & 3) == 0 && (((uintptr_t)P | (uintptr_t)Vw) & 15) == 0;
  auto load_left = [&](const Z* A) __attribute__((always_inline)) {
    if (wide) load4(A);
    else load(A);
  };

  ACC cr[NJ], ci[NJ];
  // (cr, ci) = left operand times U
  auto product = [&](const Z* U) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NJ; j++)
#pragma unroll
      for (int q = 0; q < 4; q++) cr[j][q] = ci[j][q] = 0;
#pragma unroll
    for (int t = 0; t < MT; t++) {
      if (t >= nk) continue;
      if constexpr (F::FMT == 2) {
        auto ng = [](uint32_t x) { return x ^ 0x80000000u; };
        auto rt = [](uint32_t x) { return __builtin_amdgcn_alignbit(x, x, 16u); };
        const Frag<Z>& f = fa[t];
        const bf16x8 ah = __builtin_bit_cast(bf16x8, make_uint4(f.v[0].hi, f.v[1].hi, f.v[2].hi, f.v[3].hi));
        const bf16x8 al = __builtin_bit_cast(bf16x8, make_uint4(f.v[0].lo, f.v[1].lo, f.v[2].lo, f.v[3].lo));
#pragma unroll
        for (int j = 0; j < NJ; j++) {
          const uint4* q4 = (const uint4*)&U[(16 * j + r) * LD + 16 * t + 4 * g];
          const uint4 v0 = q4[0], v1 = q4[1];
          const bf16x8 rh = __builtin_bit_cast(bf16x8, make_uint4(ng(v0.x), ng(v0.z), ng(v1.x), ng(v1.z)));
          const bf16x8 rl = __builtin_bit_cast(bf16x8, make_uint4(ng(v0.y), ng(v0.w), ng(v1.y), ng(v1.w)));
          const bf16x8 ih = __builtin_bit_cast(bf16x8, make_uint4(rt(v0.x), rt(v0.z), rt(v1.x), rt(v1.z)));
          const bf16x8 il = __builtin_bit_cast(bf16x8, make_uint4(rt(v0.y), rt(v0.w), rt(v1.y), rt(v1.w)));
          cr[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, rh, cr[j], 0, 0, 0);
          ci[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, ih, ci[j], 0, 0, 0);
          cr[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, rl, cr[j], 0, 0, 0);
          ci[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, il, ci[j], 0, 0, 0);
          cr[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, rh, cr[j], 0, 0, 0);
          ci[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, ih, ci[j], 0, 0, 0);
        }
      } else {
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const Z av = fa[t].v[q];
#pragma unroll
          for (int j = 0; j < NJ; j++) {
            const Z b = U[(16 * j + r) * LD + 16 * t + 4 * q + g];
            if constexpr (F::FMT == 0) {
              cr[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(av.re, b.re, cr[j], 0, 0, 0);
              ci[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(av.re, b.im, ci[j], 0, 0, 0);
              cr[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(av.im, -b.im, cr[j], 0, 0, 0);
              ci[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(av.im, b.re, ci[j], 0, 0, 0);
            } else {
              cr[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(av.re, b.re, cr[j], 0, 0, 0);
              ci[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(av.re, b.im, ci[j], 0, 0, 0);
              cr[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(av.im, -b.im, cr[j], 0, 0, 0);
              ci[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(av.im, b.re, ci[j], 0, 0, 0);
            }
          }
        }
      }
    }
  };
  // the lane's elements of a product: column 16 j + r, rows 4 g + q (4 q + g
  // in FP64) of the wave's 16
  auto orow = [&](int q) { return 16 * wave + (F::FMT == 0 ? 4 * q + g : 4 * g + q); };

  load_left(P);
  // W's columns, spin c / N, orbital c % N; padding rows and columns are zero
  for (int e = tid; e < NB * MP; e += NT) {
    const int cc = e % NB, i = e / NB, c = c0 + cc;
    zd v{0.0, 0.0};
    if (i < M && c < 2 * N) v = Ww[((long)(c / N) * M + i) * N + (c % N)];
    u0[cc * LD + i] = conv(v, Z());
  }
  __syncthreads();
  product(u0);
  load_left(Vw);  // on its way while S is stored
  R sr[NJ][4], si[NJ][4];
#pragma unroll
  for (int j = 0; j < NJ; j++)
#pragma unroll
    for (int q = 0; q < 4; q++) {
      sr[j][q] = cr[j][q];
      si[j][q] = ci[j][q];
      u1[(16 * j + r) * LD + orow(q)] = conv(zd{(double)sr[j][q], (double)si[j][q]}, Z());
    }
  __syncthreads();
  // U_k = S + (i/k) V U_{k+1}
  auto horner = [&](const Z* in, Z* out, int k, bool last) __attribute__((always_inline)) {
    product(in);
    if (last) load_left(P);
    const double al = 1.0 / (double)k;
#pragma unroll
    for (int j = 0; j < NJ; j++)
#pragma unroll
      for (int q = 0; q < 4; q++) {
        out[(16 * j + r) * LD + orow(q)] =
            conv(horner_term((double)sr[j][q], (double)si[j][q], al, (double)cr[j][q], (double)ci[j][q]), Z());
      }
    __syncthreads();
  };
  horner(u1, u0, 6, false);
  horner(u0, u1, 5, false);
  horner(u1, u0, 4, false);
  horner(u0, u1, 3, false);
  horner(u1, u0, 2, false);
  horner(u0, u1, 1, true);
  product(u1);
#pragma unroll
  for (int j = 0; j < NJ; j++) {
    const int c = c0 + 16 * j + r;
    if (c >= 2 * N) continue;
    zd* Wc = Ww + (long)(c / N) * M * N + (c % N);
#pragma unroll
    for (int q = 0; q < 4; q++)
      if (orow(q) < M) Wc[(long)orow(q) * N] = zd{(double)cr[j][q], (double)ci[j][q]};
  }
}

template <class Z, int MT> void go_nb(hipStream_t st, PropSmallArgs a)
{
  // 32 columns per workgroup read V half as often; 16 where that leaves CUs
  // without one, and where the registers would spill (FP64, more than 8 waves)
  const int n2 = 2 * a.N;
  if constexpr (!std::is_same<Z, zd>::value && MT <= 8) {
    if ((long)a.nw * ((n2 + 31) / 32) >= 256) {
      a.ncb = (n2 + 31) / 32;
      hipLaunchKernelGGL((prop_small_kernel<Z, MT, 32>), dim3((unsigned)(a.nw * a.ncb)), dim3(64 * MT), 0, st, a);
      return;
    }
  }
  a.ncb = (n2 + 15) / 16;
  hipLaunchKernelGGL((prop_small_kernel<Z, MT, 16>), dim3((unsigned)(a.nw * a.ncb)), dim3(64 * MT), 0, st, a);
}

template <class Z> void go(hipStream_t st, const PropSmallArgs& a)
{
  if (a.M <= 32) return go_nb<Z, 2>(st, a);
  if (a.M <= 64) return go_nb<Z, 4>(st, a);
  if (a.M <= 96) return go_nb<Z, 6>(st, a);
  if constexpr (std::is_same<Z, zd>::value) {
    go_nb<Z, 8>(st, a);
  } else {
    if (a.M <= 128) return go_nb<Z, 8>(st, a);
    if (a.M <= 160) return go_nb<Z, 10>(st, a);
    go_nb<Z, 12>(st, a);
  }
}

} // namespace

bool prop_small_ok(int fmt, int M) { return M <= (fmt == 0 ? PS_MMAX_F64 : PS_MMAX); }

void prop_small_launch(hipStream_t st, PropSmallArgs a, int fmt)
{
  if (fmt == 0) go<zd>(st, a);
  else if (fmt == 1) go<zf>(st, a);
  else go<zb>(st, a);
}
