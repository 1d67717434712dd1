// Non-GEMM kernels of the walker step (FP64 unless stated).
#pragma once
#include "common.hpp"
#include "fieldrng.hpp"

#include <type_traits>

// ---------------------------------------------------------------------------
// Batched in-place Gauss-Jordan inverse + determinant of N x N complex
// matrices, FP64.  Follows LAPACK's pivoting on the column-major view used by
// ma::invert / ma::determinant (src/Numerics/ma_operations.hpp:244-291,
// ma_lapack.hpp:33-79): the matrix factorised is X = T^T, the pivot of step k
// is the first row i >= k maximising |Re|+|Im| of X(i,k) (izamax), and
// det = prod(pivots) * (-1)^(#swaps).  The Gauss-Jordan eliminations below
// the diagonal are those of the LU factorisation, so pivots and determinant
// match getrf; the inverse equals getri's up to rounding.
//
// The signed pivots also give the log-determinant (store_log_det).
// batch b: input T + b*mstride; det written to det[(b/2)*dq + (b%2)*dr] and
// to dcache[b] when dcache != null.
// log det = sum_k log(pv_k), principal logs, imaginary part wrapped to
// [-pi, pi], from the signed pivots pv[0..N) in LDS; summed by one wave in a
// fixed order (every lane returns the same value).  The overlap ratios of
// the weights are taken from these logs, so that a determinant that
// underflows or overflows as a product of N pivots keeps its ratio.
__device__ inline zd log_det_sum(const zd* pv, int N)
{
  const int lane = threadIdx.x & 63;
  double lr = 0.0, li = 0.0;
  for (int q = lane; q < N; q += 64) {
    const zd v = pv[q];
    lr += log(hypot(v.re, v.im));
    li += atan2(v.im, v.re);
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    lr += __shfl_xor(lr, off);
    li += __shfl_xor(li, off);
  }
  return zd{lr, remainder(li, 6.283185307179586476925286766559)};
}

// log det of matrix b (log_det_sum of its signed pivots, {-inf, 0} when
// singular) to ldet[(b/2)*4 + b%2] and lcache[b] where those are set;
// called by every thread after the elimination.
__device__ inline void store_log_det(const zd* pv, int N, bool singular, long b, zd* ldet, zd* lcache)
{
  if ((!ldet && !lcache) || threadIdx.x >= 64) return;
  const zd L = singular ? zd{-INFINITY, 0.0} : log_det_sum(pv, N);
  if (threadIdx.x == 0) {
    if (ldet) ldet[(b / 2) * 4 + (b % 2)] = L;
    if (lcache) lcache[b] = L;
  }
}

// value of lane j (j the same in every lane) without going through LDS
__device__ __forceinline__ double rdlane(double x, int j)
{
  const long long v = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_readlane((int)(v & 0xffffffffLL), j);
  const int hi = __builtin_amdgcn_readlane((int)(v >> 32), j);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
__device__ __forceinline__ zd rdlane(zd x, int j) { return zd{rdlane(x.re, j), rdlane(x.im, j)}; }

// Maximum of v over the wave, uniform: DPP moves within quads, half-rows and
// rows, then row broadcasts (0 is the identity).
template <int CTRL, int RM> __device__ __forceinline__ uint32_t umax_step(uint32_t v)
{
  return max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, RM, 0xF, false));
}
__device__ __forceinline__ uint32_t wave_umax(uint32_t v)
{
  v = umax_step<0xB1, 0xF>(v);   // quad_perm [1,0,3,2]
  v = umax_step<0x4E, 0xF>(v);   // quad_perm [2,3,0,1]
  v = umax_step<0x141, 0xF>(v);  // row_half_mirror
  v = umax_step<0x140, 0xF>(v);  // row_mirror
  v = umax_step<0x142, 0xA>(v);  // row_bcast15 into rows 1 and 3
  v = umax_step<0x143, 0xC>(v);  // row_bcast31 into rows 2 and 3
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// 1 / b for a finite, nonzero b to about an ulp: b scaled by a power of two to
// a largest component in [1/2, 1), |b|^2 inverted by the hardware's estimate
// and two Newton steps (a third of the latency of two dependent divisions);
// other b as zdiv gives it.
__device__ __forceinline__ zd zrecip(zd b)
{
  const int e = __builtin_amdgcn_frexp_exp(fmax(fabs(b.re), fabs(b.im)));
  const double a = __builtin_amdgcn_ldexp(b.re, -e), c = __builtin_amdgcn_ldexp(b.im, -e);
  const double d = fma(a, a, c * c);
  if (!(d >= 0.25 && d <= 2.0)) return zdiv(zd{1.0, 0.0}, b);
  double y = __builtin_amdgcn_rcp(d);
  y = fma(y, fma(-d, y, 1.0), y);
  y = fma(y, fma(-d, y, 1.0), y);
  return zd{__builtin_amdgcn_ldexp(a * y, -e), __builtin_amdgcn_ldexp(-c * y, -e)};
}

// One workgroup per matrix.  Lane l holds row l (RPL = 2: rows l and l + 64) at
// the CPW columns of its wave, column j = wave * CPW + c in register slot c, so
// a step touches registers statically and a row never leaves its lane.  Rows
// are not swapped: pos is the position LAPACK's interchanges would have
// brought the row to, and a row is a pivot candidate while pos >= k.  A pivot
// row is not scaled when it is chosen but once at the end (it is no candidate
// any more, and the other rows' multipliers hold the reciprocal), so a step is
// x += multiplier * pivot row in every lane, with multiplier 0 in the pivot
// row's, and only column k's slot is set apart.
//
// Step k: the wave that owns column k finds the pivot row p (wave maximum of
// |Re| + |Im|, the lowest position among equals), the pivot's reciprocal and
// the multipliers -X(i,k)/piv of all rows and leaves them in LDS (two buffers
// by step parity); after a barrier every wave takes row p's entries of its own
// columns by readlane and updates its rows.  The owner of column k + 1 updates
// that column first and searches it before its other columns, so one barrier
// and one search chain bound a step.
//
// Bound: that chain (key maximum, reciprocal, LDS round trip, barrier: 0.5 to
// 0.7 us a step with nothing else to do), and from 64 electrons on the
// readlanes and FP64 FMAs of four waves per SIMD (0.9 us a step at 128), which
// the owner's own columns keep from overlapping fully.  Measured (MI355X, us
// per batch; before: the matrix split over the rows' threads, two barriers per
// step, the pivot row read from LDS by all, a serial unscrambling of the
// interchanges): 2048 x N = 128 3070 -> 1930, 512 x 96 541 -> 319, 512 x 64
// 150 -> 90, 192 x 32 48 -> 29, 32 x 16 23 -> 17.  With the search, the
// reciprocal and all updates but the searched column's taken out, 128 x N = 128
// went from 230 to 93 us.
//
// SCALED (the mixed modes): the pivot row is scaled as it is chosen, by its
// one lane after the other rows' updates, with the reciprocal by division.
// That is the elimination's textbook rounding; the mixed modes round T^-1 to
// FP32, where an ulp of FP64 now and then turns an FP32 rounding and with it
// everything the walker does afterwards, so their bits do not follow the
// faster form (2048 x N = 128 2390 us against 2080, 512 x 96 385 against 321,
// 512 x 64 117 against 96, one box).
template <int RPL, int NW, int CPW, bool SCALED>
__global__ __launch_bounds__(64 * NW) void gj_inverse_kernel(const zd* __restrict__ T, zd* __restrict__ Tinv,
                                                             zd* __restrict__ det, long dq, long dr, int N,
                                                             long mstride, int* __restrict__ info,
                                                             zd* __restrict__ dcache, zd* __restrict__ ldet,
                                                             zd* __restrict__ lcache)
{
  constexpr int NMAX = NW * CPW;  // columns
  static_assert(CPW % 2 == 0, "buffers alternate by slot parity");
  __shared__ zd gqs[2][64 * RPL];  // multipliers by row
  __shared__ zd ipvs[2], pv[NMAX];
  __shared__ int ctl[2];   // pivot row, or -1 when the pivot is zero
  __shared__ int prow[NMAX];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const long b = blockIdx.x;
  const zd* Tb = T + b * mstride;
  const int j0 = wave * CPW;
  zd x[RPL][CPW];
  int pos[RPL];
  zd scale[RPL];  // reciprocal of the row's pivot
#pragma unroll
  for (int q = 0; q < RPL; q++) {
    const int i = lane + 64 * q;
    pos[q] = i < N ? i : 0x7fffffff;
    scale[q] = zd{1.0, 0.0};
#pragma unroll
    for (int c = 0; c < CPW; c++)
      x[q][c] = (i < N && j0 + c < N) ? Tb[(long)(j0 + c) * N + i] : zd{0.0, 0.0};  // X = T^T
  }
  // search column k (slot c of this wave) and publish the step
  auto publish = [&](int k, auto cc) __attribute__((always_inline)) {
    constexpr int c = decltype(cc)::value, st = c & 1;
    // keys: the high word of |Re| + |Im| plus 1 (nonnegative doubles order as
    // their bits), 0 for rows that are no candidates and for NaN; the low
    // words decide among equal high words, then the position
    uint32_t hi[RPL], lo[RPL], m = 0;
#pragma unroll
    for (int q = 0; q < RPL; q++) {
      const double v = zcabs1(x[q][c]);
      const unsigned long long u = (unsigned long long)__double_as_longlong(v);
      hi[q] = (pos[q] >= k && pos[q] < N && v == v) ? (uint32_t)(u >> 32) + 1u : 0u;
      lo[q] = (uint32_t)u;
      m = max(m, hi[q]);
    }
    m = wave_umax(m);
    unsigned long long cand[RPL];
    int n = 0;
#pragma unroll
    for (int q = 0; q < RPL; q++) {
      // no candidate compares (all NaN): the row at position k
      cand[q] = m ? __ballot(hi[q] == m) : __ballot(pos[q] == k);
      n += __popcll(cand[q]);
    }
    if (n > 1) {
      uint32_t ml = 0;
#pragma unroll
      for (int q = 0; q < RPL; q++)
        if (hi[q] == m) ml = max(ml, lo[q]);
      ml = wave_umax(ml);
      n = 0;
#pragma unroll
      for (int q = 0; q < RPL; q++) {
        cand[q] = __ballot(hi[q] == m && lo[q] == ml);
        n += __popcll(cand[q]);
      }
    }
    int p = -1;
    if (n == 1) {
#pragma unroll
      for (int q = 0; q < RPL; q++)
        if (cand[q]) p = (__ffsll((long long)cand[q]) - 1) + 64 * q;
    } else {
      int best = 0x7fffffff;
#pragma unroll
      for (int q = 0; q < RPL; q++)
        for (unsigned long long s = cand[q]; s; s &= s - 1) {
          const int l = __ffsll((long long)s) - 1;
          const int ps = __builtin_amdgcn_readlane(pos[q], l);
          if (ps < best) {
            best = ps;
            p = l + 64 * q;
          }
        }
    }
    zd piv = rdlane(x[0][c], p & 63);
    int pp = __builtin_amdgcn_readlane(pos[0], p & 63);
    if constexpr (RPL == 2) {
      if (p >= 64) {
        piv = rdlane(x[1][c], p - 64);
        pp = __builtin_amdgcn_readlane(pos[1], p - 64);
      }
    }
    const bool zero = piv.re == 0.0 && piv.im == 0.0;
    const zd ipv = SCALED ? zdiv(zd{1.0, 0.0}, piv) : zrecip(piv);
#pragma unroll
    for (int q = 0; q < RPL; q++)
      gqs[st][lane + 64 * q] = lane + 64 * q == p ? zd{0.0, 0.0} : zmul(zd{-x[q][c].re, -x[q][c].im}, ipv);
    if (lane == 0) {
      ctl[st] = zero ? -1 : p;
      ipvs[st] = ipv;
      prow[k] = p;
      pv[k] = pp != k ? zd{-piv.re, -piv.im} : piv;  // signed pivot
    }
  };
  if (wave == 0) publish(0, std::integral_constant<int, 0>());
  __syncthreads();
  zd dt{1.0, 0.0};
  bool singular = false;
  const int nblk = (N + CPW - 1) / CPW;
  for (int kb = 0; kb < nblk && !singular; kb++) {
    // wave kb owns the block's columns
    auto step = [&](auto cc) __attribute__((always_inline)) {
      constexpr int c = decltype(cc)::value, st = c & 1, c1 = (c + 1) % CPW;
      const int k = kb * CPW + c;
      if (k >= N || singular) return;
      const int pl = ctl[st];
      const zd ipv = ipvs[st], spv = pv[k];
      zd gq[RPL];
#pragma unroll
      for (int q = 0; q < RPL; q++) gq[q] = gqs[st][lane + 64 * q];
      const int p = __builtin_amdgcn_readfirstlane(pl);
      if (p < 0) {
        singular = true;
        dt = zd{0.0, 0.0};
        return;
      }
      // positions: the pivot row to k, the row there to the pivot's
      int pp = __builtin_amdgcn_readlane(pos[0], p & 63);
      if constexpr (RPL == 2)
        if (p >= 64) pp = __builtin_amdgcn_readlane(pos[1], p - 64);
#pragma unroll
      for (int q = 0; q < RPL; q++) {
        const bool mine = lane + 64 * q == p;
        pos[q] = mine ? k : (pos[q] == k ? pp : pos[q]);
        if (!SCALED && mine) scale[q] = ipv;
      }
      auto update = [&](int s, bool colk) __attribute__((always_inline)) {
        // row p's entry of the slot
        zd pr;
        if constexpr (RPL == 2) pr = p >= 64 ? rdlane(x[1][s], p - 64) : rdlane(x[0][s], p);
        else pr = rdlane(x[0][s], p);
#pragma unroll
        for (int q = 0; q < RPL; q++) {
          const double xr = x[q][s].re, xi = x[q][s].im;
          x[q][s].re = xr + gq[q].re * pr.re - gq[q].im * pr.im;
          x[q][s].im = xi + gq[q].re * pr.im + gq[q].im * pr.re;
          if (colk) x[q][s] = lane + 64 * q == p ? zd{1.0, 0.0} : gq[q];
        }
        __builtin_amdgcn_sched_barrier(0);  // one slot at a time: bounds the live registers
      };
      // the pivot row's entry of one slot, or of all others
      auto rescale = [&](int s0, bool only) __attribute__((always_inline)) {
        if constexpr (SCALED) {
          auto row = [&](auto qc) __attribute__((always_inline)) {
            constexpr int q = decltype(qc)::value;
            if (lane == (p & 63)) {
#pragma unroll
              for (int s = 0; s < CPW; s++)
                if ((s == s0) == only) {
                  x[q][s] = zmul(x[q][s], ipv);
                  __builtin_amdgcn_sched_barrier(0);
                }
            }
          };
          if (RPL == 2 && p >= 64) row(std::integral_constant<int, RPL - 1>());
          else row(std::integral_constant<int, 0>());
        }
      };
      const int k1 = k + 1;
      // the search chain ahead of the other waves' updates
      if (wave == k1 / CPW) __builtin_amdgcn_s_setprio(3);
      update(c1, false);
      rescale(c1, true);
      if (k1 < N && wave == k1 / CPW) publish(k1, std::integral_constant<int, c1>());
      __builtin_amdgcn_s_setprio(0);
#pragma unroll
      for (int s = 0; s < CPW; s++)
        if (s != c1) update(s, s == c && wave == kb);
      rescale(c1, false);
      if (wave == 0) dt = zmul(dt, spv);
      __syncthreads();
    };
    step(std::integral_constant<int, 0>());
    step(std::integral_constant<int, 1>());
    if constexpr (CPW > 2) {
      step(std::integral_constant<int, 2>());
      step(std::integral_constant<int, 3>());
    }
    if constexpr (CPW > 4) {
      step(std::integral_constant<int, 4>());
      step(std::integral_constant<int, 5>());
      step(std::integral_constant<int, 6>());
      step(std::integral_constant<int, 7>());
    }
  }
  if (tid == 0) {
    if (singular && info) atomicAdd(info, 1);
    det[(b / 2) * dq + (b % 2) * dr] = dt;
    if (dcache) dcache[b] = dt;
  }
  if (Tinv) {
    // with the rows in LAPACK's positions the result would be the inverse of
    // the interchanged matrix: its column k belongs to the row p chosen at
    // step k, so T^-1[p_j][pos_i] = X(i, j)
#pragma unroll
    for (int q = 0; q < RPL; q++)
#pragma unroll
      for (int c = 0; c < CPW; c++) {
        const int i = lane + 64 * q, j = j0 + c;
        if (i < N && j < N) {
          if (singular) Tinv[b * mstride + (long)j * N + i] = zd{0, 0};  // a defined value
          else Tinv[b * mstride + (long)prow[j] * N + pos[q]] = SCALED ? x[q][c] : zmul(x[q][c], scale[q]);
        }
      }
  }
  store_log_det(pv, N, singular, b, ldet, lcache);
}

// The same elimination for N too large for the registers of one workgroup
// (N <= GJ_GMAX): the working matrix X = T^T lives in global memory (work +
// b*mstride, X(i, j) at [j*N + i]), one workgroup of 1024 threads per matrix,
// thread (jg, i) with row i and columns jg, jg + G, ... (G = 1024 / N, so
// consecutive threads touch consecutive addresses and nothing is divided).
// As in the register kernel rows are not moved or scaled, so row p is not
// written in its own step and every thread reads its entries (one or two
// addresses a wave) while the others' rows change: one barrier per step.  The
// threads of column k + 1 leave its new values in LDS, where every wave finds
// the next pivot for itself.  SCALED as in the register kernel: the row's own
// threads scale it in the following step (2450 against 2340 us at N = 160).
//
// Bound: the caches behind the L2 (the matrix is read and written once a
// step; 128 matrices of 410 KB move 7 TB/s).  Measured (MI355X): 128 matrices
// of N = 160 2.88 -> 2.30 ms (before: four barriers per step and a 64-bit
// division by N per entry).
constexpr int GJ_GMAX = 256;
template <bool SCALED>
__global__ __launch_bounds__(1024) void gj_inverse_global_kernel(const zd* __restrict__ T, zd* __restrict__ Tinv,
                                                                 zd* __restrict__ work, zd* __restrict__ det, long dq,
                                                                 long dr, int N, long mstride, int* __restrict__ info,
                                                                 zd* __restrict__ dcache, zd* __restrict__ ldet,
                                                                 zd* __restrict__ lcache)
{
  constexpr int Q = GJ_GMAX / 64;
  __shared__ zd colk[2][GJ_GMAX], pv[GJ_GMAX];
  __shared__ int perm[GJ_GMAX];
  const int tid = threadIdx.x, lane = tid & 63;
  const long b = blockIdx.x;
  const zd* Tb = T + b * mstride;
  zd* X = work + b * mstride;
  const int G = 1024 / N, i = tid % N, jg = tid / N;
  const bool active = jg < G;
  // the wave's own bookkeeping of all rows' positions (row lane + 64 q)
  int pos[Q], mypos = i;
#pragma unroll
  for (int q = 0; q < Q; q++) pos[q] = lane + 64 * q < N ? lane + 64 * q : 0x7fffffff;
  // X(i, j) = T[j][i]: X's column j is T's row j, so the copy is contiguous
  if (active)
    for (int j = jg; j < N; j += G) {
      const zd v = Tb[(long)j * N + i];
      X[(long)j * N + i] = v;
      if (j == 0) colk[0][i] = v;
    }
  __syncthreads();
  zd dt{1.0, 0.0}, scale{1.0, 0.0};
  bool singular = false, last = false;  // last: row i was the last step's pivot row
  for (int k = 0; k < N; k++) {
    const zd* ck = colk[k & 1];
    // pivot: |Re| + |Im| largest, the lowest position among equals (keys as
    // in the register kernel)
    uint32_t hi[Q], lo[Q], m = 0;
#pragma unroll
    for (int q = 0; q < Q; q++) {
      hi[q] = lo[q] = 0;
      if (lane + 64 * q < N) {
        const double v = zcabs1(ck[lane + 64 * q]);
        const unsigned long long u = (unsigned long long)__double_as_longlong(v);
        hi[q] = (pos[q] >= k && v == v) ? (uint32_t)(u >> 32) + 1u : 0u;
        lo[q] = (uint32_t)u;
      }
      m = max(m, hi[q]);
    }
    m = wave_umax(m);
    uint32_t ml = 0;
#pragma unroll
    for (int q = 0; q < Q; q++)
      if (hi[q] == m) ml = max(ml, lo[q]);
    ml = wave_umax(ml);
    int p = 0, pp = 0x7fffffff;
#pragma unroll
    for (int q = 0; q < Q; q++) {
      unsigned long long c = m ? __ballot(hi[q] == m && lo[q] == ml) : __ballot(pos[q] == k);
      for (; c; c &= c - 1) {
        const int l = __ffsll((long long)c) - 1;
        const int ps = __builtin_amdgcn_readlane(pos[q], l);
        if (ps < pp) {
          pp = ps;
          p = l + 64 * q;
        }
      }
    }
    const zd piv = ck[p];
    if (piv.re == 0.0 && piv.im == 0.0) {
      singular = true;
      dt = zd{0.0, 0.0};
      break;
    }
    const zd spv = pp != k ? zd{-piv.re, -piv.im} : piv;  // signed pivot
    dt = zmul(dt, spv);
    if (tid == 0) {
      pv[k] = spv;
      perm[k] = p;
    }
    const zd ipv = SCALED ? zdiv(zd{1.0, 0.0}, piv) : zrecip(piv);
#pragma unroll
    for (int q = 0; q < Q; q++) pos[q] = lane + 64 * q == p ? k : (pos[q] == k ? pp : pos[q]);
    mypos = i == p ? k : (mypos == k ? pp : mypos);
    const zd f = ck[i];
    const zd gq = i == p ? zd{0.0, 0.0} : zmul(zd{-f.re, -f.im}, ipv);
    if (active) {
      zd* Xi = X + i;
      const zd* Xp = X + p;
#pragma unroll 4
      for (int j = jg; j < N; j += G) {
        const long o = (long)j * N;
        zd x = Xi[o];
        if (SCALED && last) x = zmul(x, scale);
        const zd pr = Xp[o];
        x.re = x.re + gq.re * pr.re - gq.im * pr.im;
        x.im = x.im + gq.re * pr.im + gq.im * pr.re;
        if (j == k) x = i == p ? zd{1.0, 0.0} : gq;
        if (i != p || j == k) Xi[o] = x;
        if (j == k + 1) colk[(k + 1) & 1][i] = SCALED && i == p ? zmul(x, ipv) : x;
      }
    }
    last = i == p;
    if (last) scale = ipv;
    __syncthreads();
  }
  if (tid == 0) {
    if (singular && info) atomicAdd(info, 1);
    det[(b / 2) * dq + (b % 2) * dr] = dt;
    if (dcache) dcache[b] = dt;
  }
  store_log_det(pv, N, singular, b, ldet, lcache);
  if (!Tinv || !active) return;
  zd* Ob = Tinv + b * mstride;
  // T^-1[p_j][pos_i] = X(i, j) / pivot of row i, zeros when singular
  for (int j = jg; j < N; j += G) {
    if (singular) Ob[(long)j * N + i] = zd{0, 0};
    else Ob[(long)perm[j] * N + mypos] = !SCALED || last ? zmul(X[(long)j * N + i], scale) : X[(long)j * N + i];
  }
}

// n bytes of device memory (16-byte aligned) to mapped host memory: the
// downloads' copy (the runtime's takes a copy engine, whose first use by a
// stream can cost 8 ms).
__global__ __launch_bounds__(256) void copy_out_kernel(const char* __restrict__ in, char* __restrict__ out, size_t n)
{
  const size_t n16 = n / 16, i0 = blockIdx.x * (size_t)256 + threadIdx.x;
  for (size_t i = i0; i < n16; i += gridDim.x * (size_t)256) ((uint4*)out)[i] = ((const uint4*)in)[i];
  if (i0 < n % 16) out[n16 * 16 + i0] = in[n16 * 16 + i0];
}

// Three-piece split-BF16 of n complex values: (h, m) to hm (a zb per
// element; may alias the input when IT is zf, each element being read before
// its slot is written by the same thread) and the third pieces to l.
template <class IT>
__global__ void split3_kernel(const IT* in, zb* hm, uint32_t* __restrict__ l, long n)
{
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    const IT v = in[i];
    zb h;
    uint32_t t;
    split3_z((double)v.re, (double)v.im, h, t);
    hm[i] = h;
    l[i] = t;
  }
}

// Third pieces of a split-BF16 array from its FP64 source: the stored (h, m)
// pieces are taken as they are, l = bf16(x - h - m) per component.  Element o
// of the split array (and of l) comes from src[(o % R) * C + o / R] when
// trans (the split array is the [C][R] transpose of the [R][C] source), else
// from src[o].
__global__ void third_piece_kernel(const zd* __restrict__ src, const zb* __restrict__ hm, uint32_t* __restrict__ l,
                                   long n, long R, long C, int trans)
{
  for (long o = blockIdx.x * (long)blockDim.x + threadIdx.x; o < n; o += (long)gridDim.x * blockDim.x) {
    const zd x = src[trans ? (o % R) * C + o / R : o];
    const zb v = hm[o];
    const double rr = x.re - (double)bf2f((unsigned short)(v.hi & 0xffff)) - (double)bf2f((unsigned short)(v.lo & 0xffff));
    const double ri = x.im - (double)bf2f((unsigned short)(v.hi >> 16)) - (double)bf2f((unsigned short)(v.lo >> 16));
    l[o] = (uint32_t)d2bf(rr) | ((uint32_t)d2bf(ri) << 16);
  }
}

// Batched transpose into split-BF16: in [b][R][C] (row stride C, item stride
// R*C) -> out [b][C][ldo] (zb), with P3 as three pieces (the third ones to
// out3), per 32 x 32 tile through LDS; grid (C/32, R/32, b).
template <class IT, bool P3>
__global__ __launch_bounds__(256) void transpose_split_kernel(const IT* __restrict__ in, zb* __restrict__ out,
                                                               uint32_t* __restrict__ out3, int R, int C, long ldo)
{
  __shared__ zd tile[32][33];
  const long item = (long)blockIdx.z * R * C;
  const int bx = blockIdx.x * 32, by = blockIdx.y * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8
  for (int yy = ty; yy < 32; yy += 8) {
    const int rr = by + yy, cc = bx + tx;
    if (rr < R && cc < C) tile[yy][tx] = to_zd(in[item + (long)rr * C + cc]);
  }
  __syncthreads();
  for (int yy = ty; yy < 32; yy += 8) {
    const int cc = bx + yy, rr = by + tx;
    if (rr < R && cc < C) {
      const zd v = tile[tx][yy];
      const long o = ((long)blockIdx.z * C + cc) * ldo + rr;
      if constexpr (P3) split3_z(v.re, v.im, out[o], out3[o]);
      else out[o] = split_z((float)v.re, (float)v.im);
    }
  }
}

// W_data[w][2+s] = dcache[2w+s] (determinants cached by the last inverse of
// the same walkers)
__global__ void det_restore_kernel(zd* __restrict__ Wd, const zd* __restrict__ dcache, zd* __restrict__ Wl,
                                   const zd* __restrict__ lcache, int nw)
{
  int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b < 2 * nw) {
    Wd[(long)(b / 2) * 8 + 2 + (b % 2)] = dcache[b];
    Wl[(long)(b / 2) * 4 + (b % 2)] = lcache[b];
  }
}

// log-overlaps [nw][4] (current spin 0, 1; saved spin 0, 1) taken from the
// overlaps a caller wrote into W_data (columns 2, 3, 6, 7)
__global__ void wd_logs_kernel(const zd* __restrict__ Wd, zd* __restrict__ Wl, int nw)
{
  const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= 4L * nw) return;
  const long w = e / 4, q = e % 4;
  const zd v = Wd[w * 8 + (q < 2 ? 2 + q : 4 + q)];
  Wl[e] = zd{log(hypot(v.re, v.im)), atan2(v.im, v.re)};
}

// ---------------------------------------------------------------------------
// CSR x dense, mySPBLAS::csrmm 'N' semantics (src/Numerics/sparse.hpp:166-180):
// C(r, w) = alpha * sum_{p in row r, col<K} val[p] * B(col[p], w) + beta*C(r,w)
// B(c, w) at B[c*ldb + w]; C(r, w) at C[r*ldc + w] (row-major, walker last).

// a += v * b in four fused multiply-adds
__device__ __forceinline__ void zfma(zd& a, zd v, zd b)
{
  a.re = fma(v.re, b.re, a.re);
  a.im = fma(v.re, b.im, a.im);
  a.re = fma(-v.im, b.im, a.re);
  a.im = fma(v.im, b.re, a.im);
}
__device__ inline void csr_store(zd* C, zd acc, zd alpha, zd beta)
{
  zd o = zmul(alpha, acc);
  if (beta.re != 0.0 || beta.im != 0.0) o = zadd(o, zmul(beta, *C));
  *C = o;
}

// S waves per row and chunk of WL walkers (64 / WL groups of lanes take
// entries side by side), four entries in flight per group; the partial sums
// are joined in a fixed order (entries of a group, groups, waves).
// Bound: latency when rows x chunks are few, then the L2 (each entry reads
// 16 B of B per walker).  Measured (MI355X, before -> after): 2048 rows of
// 2048 entries, 16 walkers: 285 -> 72 us (16 waves per row, 16-lane groups;
// one 64-lane wave per row left 48 lanes idle); 384 rows of 1382, 64
// walkers: 788 -> 44 us (16 waves; 96 workgroups of 4 rows before); 65536
// rows of 205, 256 walkers: 2360 -> 1757 us (31 TB/s of L2 reads).
template <int S, int WL>
__global__ __launch_bounds__(S == 1 ? 256 : 64 * S) void csrmm_row_kernel(int nrows, int nw, int K,
                                                                       const int* __restrict__ rowptr,
                                                                       const int* __restrict__ col,
                                                                       const zd* __restrict__ val,
                                                                       const zd* __restrict__ B, long ldb,
                                                                       zd* __restrict__ C, long ldc, zd alpha, zd beta)
{
  constexpr int NG = 64 / WL;  // entries taken side by side by the lane groups
  constexpr int U = 4;
  constexpr int RW = S == 1 ? 4 : 1;  // rows per workgroup
  __shared__ zd part[S == 1 ? 1 : S][WL];
  const int nchunk = (nw + WL - 1) / WL;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const long item = (long)blockIdx.x * RW + (S == 1 ? wave : 0);
  const int r = (int)(item / nchunk), ch = (int)(item % nchunk);
  const int sw = S == 1 ? 0 : wave;
  if (r >= nrows) return;  // S == 1 only (whole waves; no barrier follows)
  const int grp = lane / WL;
  const int w = ch * WL + lane % WL;
  const int wc = min(w, nw - 1);
  const int p0 = rowptr[0];
  const int pb = __builtin_amdgcn_readfirstlane(rowptr[r] - p0), pe = __builtin_amdgcn_readfirstlane(rowptr[r + 1] - p0);
  const int len = pe - pb, per = ((len + S - 1) / S + NG - 1) / NG * NG;
  const int qb = pb + min(len, sw * per), qe = pb + min(len, (sw + 1) * per);
  zd acc[U];
#pragma unroll
  for (int u = 0; u < U; u++) acc[u] = zd{0, 0};
  int p = qb;
  for (; p + U * NG <= qe; p += U * NG) {
    int c[U];
    zd v[U], b[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int q = NG == 1 ? p + u : p + u * NG + grp;
      c[u] = col[q];
      v[u] = val[q];
    }
#pragma unroll
    for (int u = 0; u < U; u++) b[u] = c[u] < K ? B[(long)c[u] * ldb + wc] : zd{0, 0};
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (c[u] >= K) v[u] = zd{0, 0};
      zfma(acc[u], v[u], b[u]);
    }
  }
  for (; p < qe; p += NG) {
    const int q = NG == 1 ? p : p + grp;
    if (q < qe) {
      const int c = col[q];
      if (c < K) {
        const zd v = val[q], b = B[(long)c * ldb + wc];
        acc[0].re += v.re * b.re - v.im * b.im;
        acc[0].im += v.re * b.im + v.im * b.re;
      }
    }
  }
  zd a = zadd(zadd(acc[0], acc[1]), zadd(acc[2], acc[3]));
#pragma unroll
  for (int o = WL; o < 64; o <<= 1) {
    a.re += __shfl_xor(a.re, o);
    a.im += __shfl_xor(a.im, o);
  }
  if constexpr (S == 1) {
    if (lane < WL && w < nw) csr_store(&C[(long)r * ldc + w], a, alpha, beta);
  } else {
    if (lane < WL) part[sw][lane] = a;
    __syncthreads();
    if (sw == 0 && lane < WL && w < nw) {
      zd t = part[0][lane];
#pragma unroll
      for (int q = 1; q < S; q++) t = zadd(t, part[q][lane]);
      csr_store(&C[(long)r * ldc + w], t, alpha, beta);
    }
  }
}

// Rows whose columns are sorted, against a B that exceeds the L2: a workgroup
// of 16 waves takes 16 rows and 64 walkers and walks the columns in windows
// of 64, each window of B staged once for the 16 rows by direct loads into
// one of two LDS buffers while the other is read.  An entry's value and
// column come through scalar registers (one row per wave).  Measured: 1024
// rows of 13110 entries over 65536 columns, 256 walkers 3.90 ms (row kernel
// 5.19 ms, single-buffered windows with entries read from lanes 4.83 ms).
// More rows per wave are slower (the per-row overhead of a window).
__global__ __launch_bounds__(1024) void csrmm_win_kernel(int nrows, int nw, int K, const int* __restrict__ rowptr,
                                                         const int* __restrict__ col, const zd* __restrict__ val,
                                                         const zd* __restrict__ B, long ldb, zd* __restrict__ C,
                                                         long ldc, zd alpha, zd beta)
{
  __shared__ __align__(16) zd b0[64 * 64];
  __shared__ __align__(16) zd b1[64 * 64];
  const int nchunk = (nw + 63) / 64;
  const int rb = blockIdx.x / nchunk, ch = blockIdx.x % nchunk;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int w = ch * 64 + lane, wc = min(w, nw - 1);
  const int p0 = rowptr[0];
  const int r = rb * 16 + wave;
  int p = __builtin_amdgcn_readfirstlane(r < nrows ? rowptr[r] - p0 : 0);
  const int pe = __builtin_amdgcn_readfirstlane(r < nrows ? rowptr[r + 1] - p0 : 0);
  // lane i holds the column of the row's i-th entry that is still to come
  int cl = p + lane < pe ? col[p + lane] : 0x7fffffff;
  zd acc{0, 0};
  auto issue = [&](zd* dst, int c0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int cc = i * 16 + wave;
      __builtin_amdgcn_global_load_lds((const void*)(B + (long)min(c0 + cc, K - 1) * ldb + wc),
                                       (__attribute__((address_space(3))) void*)&dst[cc * 64], 16, 0, 0);
    }
  };
  auto window = [&](const zd* bs, int c0) __attribute__((always_inline)) {
    const int cend = min(c0 + 64, K);
    for (;;) {
      // the window's entries are a prefix of those to come; the next lane
      // load is issued before they are summed
      const int m = __popcll(__ballot(cl < cend));
      const int q = p + m + lane;
      cl = q < pe ? col[q] : 0x7fffffff;
      int j = 0;
      for (; j + 4 <= m; j += 4) {
        int c[4];
        zd v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
          c[u] = col[p + j + u] - c0;
          v[u] = val[p + j + u];
        }
#pragma unroll
        for (int u = 0; u < 4; u++) zfma(acc, v[u], bs[c[u] * 64 + lane]);
      }
      for (; j < m; j++) zfma(acc, val[p + j], bs[(col[p + j] - c0) * 64 + lane]);
      p += m;
      if (m < 64) break;  // 64: more may follow (repeated columns)
    }
  };
  const int nwin = (K + 63) / 64;
  issue(b0, 0);
  for (int t = 0; t < nwin; t += 2) {
    __builtin_amdgcn_s_waitcnt(0 | (7 << 4) | (15 << 8));
    __builtin_amdgcn_s_barrier();
    if (t + 1 < nwin) issue(b1, (t + 1) * 64);
    window(b0, t * 64);
    if (t + 1 < nwin) {
      __builtin_amdgcn_s_waitcnt(0 | (7 << 4) | (15 << 8));
      __builtin_amdgcn_s_barrier();
      if (t + 2 < nwin) issue(b0, (t + 2) * 64);
      window(b1, (t + 1) * 64);
    }
  }
  if (r < nrows && w < nw) csr_store(&C[(long)r * ldc + w], acc, alpha, beta);
}

// ---------------------------------------------------------------------------
// Tiled transpose of complex matrices: out[c][r] = in[r][c], in is R x Cc.
// Output precision OT (double or float pairs).  With ci, row c of the output
// goes to row (c / ci) * co + c % ci.
template <class IT, class OT>
__global__ __launch_bounds__(256) void ztranspose_kernel(const IT* __restrict__ in, OT* __restrict__ out, int R,
                                                         int Cc, long ldi, long ldo, int ci = 0, int co = 0)
{
  __shared__ zd tile[32][33];
  const int bx = blockIdx.x * 32, by = blockIdx.y * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8
  for (int yy = ty; yy < 32; yy += 8) {
    int rr = by + yy, cc = bx + tx;
    if (rr < R && cc < Cc) tile[yy][tx] = to_zd(in[(long)rr * ldi + cc]);
  }
  __syncthreads();
  for (int yy = ty; yy < 32; yy += 8) {
    int cc = bx + yy, rr = by + tx;
    if (rr < R && cc < Cc) {
      OT o;
      from_zd(tile[tx][yy], o);
      out[(ci ? (long)(cc / ci) * co + cc % ci : (long)cc) * ldo + rr] = o;
    }
  }
}

// elementwise precision conversion / copy of n complex values, rows of li
// to rows lo apart where these differ
template <class IT, class OT>
__global__ void zconvert_kernel(const IT* __restrict__ in, OT* __restrict__ out, long n, long li = 0, long lo = 0)
{
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  long st = (long)gridDim.x * blockDim.x;
  for (; i < n; i += st) {
    OT o;
    from_zd(to_zd(in[i]), o);
    out[li != lo ? i / li * lo + i % li : i] = o;
  }
}

__global__ void fill_int_kernel(int* __restrict__ p, int n, int v)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}
__global__ void set_long_kernel(long* __restrict__ p, long v)
{
  if (threadIdx.x == 0 && blockIdx.x == 0) *p = v;
}

// out[i] = sum_s in[s*n + i] (FP64 accumulation, fixed order)
template <class PZ>
__global__ void zsum_slices_kernel(const PZ* __restrict__ in, zd* __restrict__ out, long n, int ns)
{
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long st = (long)gridDim.x * blockDim.x;
  for (; i < n; i += st) {
    zd acc{0.0, 0.0};
    for (int q = 0; q < ns; q++) acc = zadd(acc, to_zd(in[(long)q * n + i]));
    out[i] = acc;
  }
}

__device__ inline zd ztwice(zd v) { return zd{2.0 * v.re, 2.0 * v.im}; }
__device__ inline zf ztwice(zf v) { return zf{2.0f * v.re, 2.0f * v.im}; }
__device__ inline uint32_t bf2_twice(uint32_t w)
{
  const unsigned short a = f2bf(2.0f * bf2f((unsigned short)(w & 0xffff)));
  const unsigned short b = f2bf(2.0f * bf2f((unsigned short)(w >> 16)));
  return (uint32_t)a | ((uint32_t)b << 16);
}
__device__ inline zb ztwice(zb v) { return zb{bf2_twice(v.hi), bf2_twice(v.lo)}; }

// nmat symmetric n x n matrices -> their lower triangles with the strictly
// lower part doubled, upper part zero, so that
//   sum_pq g_p V_pq g_q = sum_p g_p sum_{q <= p} V'_pq g_q
// (half the work of the full quadratic form).  Scaling by 2 is exact in
// every storage format.
template <class ZT>
__global__ void sym_lower_kernel(ZT* __restrict__ V, long n, long nmat)
{
  const long tot = nmat * n * n;
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long st = (long)gridDim.x * blockDim.x;
  for (; i < tot; i += st) {
    const long col = i % n, row = (i / n) % n;
    if (col > row) {
      ZT z;
      zero_z(z);
      V[i] = z;
    } else if (col < row) {
      V[i] = ztwice(V[i]);
    }
  }
}

// y += x (complex, FP64)
__global__ void zaxpy1_kernel(const zd* __restrict__ x, zd* __restrict__ y, long n)
{
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  long st = (long)gridDim.x * blockDim.x;
  for (; i < n; i += st) y[i] = zadd(y[i], x[i]);
}

// ---------------------------------------------------------------------------
// X / hybrid weight (src/miniapps/miniafqmc_base.cpp:281-289):
//   X(n, w) = x(n, w) + i vbias(n, w),  hybridW[w] = -sum_n i vb (x + i/2 vb).
// The real draws x come from a staged block (x(n, w) at x[n*nw + w]; with
// xslice != null the block of substep *xslice, an index kept in device memory
// so that a captured graph can be replayed) or, when x is null, are generated
// on the fly from (seed, substep, walker) exactly as afqmc_synth_fields does
// on the host (the reference draws them inside the substep,
// miniafqmc_base.cpp:282).  Non-finite staged draws raise *nonfinite.
struct FieldSrc {
  const double* x;      // staged draws (null: generate)
  const long* xslice;   // device substep index, or null
  long substep;         // substep index when xslice is null
  uint64_t seed;        // generator seed (x == null)
};

__device__ inline void field_term(zd b, double xr, zd& h, zd& Xo)
{
  // t1 = i*vb ; t3 = x + i/2*vb ; hybridW -= t1*t3 ; X = x + i*vb
  const zd t1{-b.im, b.re};
  const zd t3{xr - 0.5 * b.im, 0.5 * b.re};
  const zd t4 = zmul(t1, t3);
  h.re -= t4.re;
  h.im -= t4.im;
  Xo = zd{xr - b.im, b.re};
}

// What a substep leaves to its fields kernel, which has a thread for every
// bias entry and walker anyway: the sum of the bias contraction's ns partial
// products (into vb, in order), and the saved overlaps (save_overlaps_kernel),
// taken from the last inverse's determinants where the density matrix reused
// it (dcache, lcache: det_restore_kernel).  Zero: neither.
struct FieldPre {
  const void* slices;  // [ns][nw*K]
  int ns;
  zd* Wd;              // not null: save the overlaps
  zd* Wl;
  const zd* dcache;    // null: from W_data
  const zd* lcache;
};

__device__ inline void save_overlaps_row(zd* d, zd* l, const zd* dc, const zd* lc)
{
  d[5] = d[4];
  d[6] = dc ? dc[0] : d[2];
  d[7] = dc ? dc[1] : d[3];
  l[2] = lc ? lc[0] : l[0];
  l[3] = lc ? lc[1] : l[1];
}
__device__ inline void field_pre_save(const FieldPre& p, long w)
{
  save_overlaps_row(p.Wd + w * 8, p.Wl + w * 4, p.dcache ? p.dcache + 2 * w : nullptr,
                    p.lcache ? p.lcache + 2 * w : nullptr);
}
// bias entry o (of tot), summed from the slices and stored when there are any
template <class PZ> __device__ inline zd field_bias(const FieldPre& p, zd* vb, long o, long tot)
{
  if (!p.ns) return vb[o];
  const PZ* s = (const PZ*)p.slices + o;
  zd a{0.0, 0.0};
#pragma unroll 4
  for (int q = 0; q < p.ns; q++) a = zadd(a, to_zd(s[(long)q * tot]));
  vb[o] = a;
  return a;
}

// Walker-first layouts (vbias [nw][K], X [nw][ldk]): one workgroup per walker, the
// lanes along n (coalesced), each thread a pair (2j, 2j+1) of draws at a
// time; fixed-order block reduction of hybridW.
template <class XT, class PZ>
__global__ __launch_bounds__(256) void fields_wfirst_kernel(int K, int nw, zd* __restrict__ vb, FieldSrc src,
                                                            XT* __restrict__ X, zd* __restrict__ hybridW,
                                                            int* __restrict__ nonfinite, uint32_t* __restrict__ X3,
                                                            FieldPre pre, int ldk)
{
  __shared__ zd part[4];
  const int w = blockIdx.x;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const long sub = src.xslice ? *src.xslice : src.substep;
  const double* x = src.x ? src.x + (src.xslice ? sub * (long)K * nw : 0L) : nullptr;
  const long tot = (long)nw * K, o0 = (long)w * K;
  XT* Xw = X + (long)w * ldk;
  uint32_t* X3w = X3 ? X3 + (long)w * K : nullptr;
  if (pre.Wd && threadIdx.x == 0) field_pre_save(pre, w);
  // split X with its third pieces (three-piece split-BF16), else as XT
  auto put = [&](int n, zd o) {
    if constexpr (std::is_same<XT, zb>::value) {
      if (X3w) {
        split3_z(o.re, o.im, Xw[n], X3w[n]);
        return;
      }
    }
    from_zd(o, Xw[n]);
  };
  zd h{0, 0};
  bool bad = false;
  for (int n = 2 * threadIdx.x; n < K; n += 512) {
    double xa, xb = 0.0;
    if (x) {
      xa = x[(long)n * nw + w];
      if (n + 1 < K) xb = x[(long)(n + 1) * nw + w];
      bad |= !isfinite(xa) || !isfinite(xb);
    } else {
      afqmc_rng::field_pair(src.seed, sub, w, n, xa, xb);
    }
    zd o;
    field_term(field_bias<PZ>(pre, vb, o0 + n, tot), xa, h, o);
    put(n, o);
    if (n + 1 < K) {
      field_term(field_bias<PZ>(pre, vb, o0 + n + 1, tot), xb, h, o);
      put(n + 1, o);
    }
  }
  if (bad) atomicOr(nonfinite, 1);
  for (int off = 32; off >= 1; off >>= 1) {
    h.re += __shfl_xor(h.re, off);
    h.im += __shfl_xor(h.im, off);
  }
  if (lane == 0) part[wv] = h;
  __syncthreads();
  if (threadIdx.x == 0) hybridW[w] = zadd(zadd(part[0], part[1]), zadd(part[2], part[3]));
}

// Walker-last layout (vbias, X [K][nw], the FP64 CSR mode): one workgroup per
// LW walkers, its 1024 / LW groups of LW lanes taking pairs (2j, 2j+1) of n in
// turn; fixed-order reduction over the groups.
template <class XT, int LW>
__global__ __launch_bounds__(1024) void fields_wlast_kernel(int K, int nw, zd* __restrict__ vb, FieldSrc src,
                                                            XT* __restrict__ X, zd* __restrict__ hybridW,
                                                            int* __restrict__ nonfinite, FieldPre pre)
{
  constexpr int NG = 1024 / LW;
  __shared__ zd part[NG][LW];
  const int lw = threadIdx.x % LW, grp = threadIdx.x / LW;
  const int w = blockIdx.x * LW + lw;
  const long sub = src.xslice ? *src.xslice : src.substep;
  const double* x = src.x ? src.x + (src.xslice ? sub * (long)K * nw : 0L) : nullptr;
  const long tot = (long)nw * K;
  zd h{0, 0};
  bool bad = false;
  if (w < nw) {
    if (pre.Wd && grp == 0) field_pre_save(pre, w);
    for (int n = 2 * grp; n < K; n += 2 * NG) {
      double xa, xb = 0.0;
      if (x) {
        xa = x[(long)n * nw + w];
        if (n + 1 < K) xb = x[(long)(n + 1) * nw + w];
        bad |= !isfinite(xa) || !isfinite(xb);
      } else {
        afqmc_rng::field_pair(src.seed, sub, w, n, xa, xb);
      }
      zd o;
      field_term(field_bias<zd>(pre, vb, (long)n * nw + w, tot), xa, h, o);
      from_zd(o, X[(long)n * nw + w]);
      if (n + 1 < K) {
        field_term(field_bias<zd>(pre, vb, (long)(n + 1) * nw + w, tot), xb, h, o);
        from_zd(o, X[(long)(n + 1) * nw + w]);
      }
    }
  }
  if (bad) atomicOr(nonfinite, 1);
  part[grp][lw] = h;
  __syncthreads();
  for (int s = NG / 2; s >= 1; s >>= 1) {
    if (grp < s) part[grp][lw] = zadd(part[grp][lw], part[grp + s][lw]);
    __syncthreads();
  }
  if (grp == 0 && w < nw) hybridW[w] = part[0][lw];
}

// W_data[:,5] = W_data[:,4]; W_data[:,6..7] = W_data[:,2..3]; the
// log-overlaps likewise
__global__ void save_overlaps_kernel(zd* __restrict__ Wd, zd* __restrict__ Wl, int nw)
{
  int w = blockIdx.x * blockDim.x + threadIdx.x;
  if (w >= nw) return;
  save_overlaps_row(Wd + (long)w * 8, Wl + (long)w * 4, nullptr, nullptr);
}

// weights / hybrid energy / Eshift (src/miniapps/miniafqmc_base.cpp:317-327).
// The overlap ratio W_data[2]W_data[3] / (W_data[6]W_data[7]) enters as its
// log, from the log-overlaps Wl (log |ratio| and its phase, wrapped to
// [-pi, pi]), so that overlaps beyond the FP64 range keep their ratio.
// One block of up to 1024 threads; fixed-order tree reduction for Eshift.
__global__ __launch_bounds__(1024) void weights_kernel(zd* __restrict__ Wd, const zd* __restrict__ Wl,
                                                       const zd* __restrict__ hybridW, int nw, double dt,
                                                       double* __restrict__ eshift)
{
  __shared__ double red[1024];
  const double Es = *eshift;
  double et = 0.0;
  for (int w = threadIdx.x; w < nw; w += blockDim.x) {
    zd* d = Wd + (long)w * 8;
    const zd* l = Wl + (long)w * 4;
    const double lr = (l[0].re + l[1].re) - (l[2].re + l[3].re);
    const double ang = remainder((l[0].im + l[1].im) - (l[2].im + l[3].im), 6.283185307179586476925286766559);
    double scale = fmax(0.0, cos(ang));
    zd h = hybridW[w];
    d[4] = zd{-(h.re + lr) / dt, -(h.im + ang) / dt};
    double f = scale * exp(-dt * (0.5 * (d[4].re + d[5].re) - Es));
    d[1] = zd{d[1].re * f, d[1].im * f};
    et += d[4].re;
  }
  red[threadIdx.x] = et;
  __syncthreads();
  for (int s = blockDim.x / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) *eshift = red[0] / nw;
}

// Comb population control, selection (one workgroup).  Weights are
// w_i = Re W_data[i][1] (the phaseless weights are >= 0; a negative weight
// counts as 0); cum_i = w_0 + ... + w_i is summed in index order by one
// thread so that every caller gets the same rounding; tooth j sits at
// t_j = (u + j) * (cum_{nw-1} / nw) and takes the first walker with
// cum_i > t_j, or the last walker of positive weight when rounding puts t_j
// at or past the total.  flag[0] is set when the total is not positive and
// finite or a weight is not finite.
__global__ __launch_bounds__(1024) void comb_select_kernel(const zd* __restrict__ Wd, int nw, double u,
                                                            double* __restrict__ cum, int* __restrict__ parent,
                                                            double* __restrict__ wnew, int* __restrict__ flag)
{
  __shared__ int last_pos;
  if (threadIdx.x == 0) {
    double sum = 0.0;
    int lp = -1, bad = 0;
    for (int i = 0; i < nw; i++) {
      const double w = Wd[(long)i * 8 + 1].re;
      if (!isfinite(w)) bad = 1;
      if (w > 0.0) {
        sum += w;
        lp = i;
      }
      cum[i] = sum;
    }
    if (bad || !(sum > 0.0) || !isfinite(sum)) flag[0] = 1;
    *wnew = sum / nw;
    last_pos = lp;
  }
  __syncthreads();
  const double total = cum[nw - 1];
  const double step = total / nw;
  for (int j = threadIdx.x; j < nw; j += blockDim.x) {
    const double t = (u + j) * step;
    int lo = 0, hi = nw;  // first i with cum[i] > t, nw if none
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (cum[mid] > t) hi = mid;
      else lo = mid + 1;
    }
    parent[j] = lo < nw ? lo : max(last_pos, 0);
  }
}

// Walkers and W_data rows of the selected parents: Wout[j] = W[parent[j]],
// Wdout[j] = Wd[parent[j]] with the weight replaced by the common weight.
__global__ void comb_gather_kernel(const zd* __restrict__ W, zd* __restrict__ Wout, const zd* __restrict__ Wd,
                                   zd* __restrict__ Wdout, const zd* __restrict__ Wl, zd* __restrict__ Wlout,
                                   const int* __restrict__ parent, const double* __restrict__ wnew, long per, int nw)
{
  const long n = (long)nw * per;
  for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x) {
    const long j = e / per, q = e - j * per;
    Wout[e] = W[(long)parent[j] * per + q];
  }
  for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < (long)nw * 8; e += (long)gridDim.x * blockDim.x) {
    const long j = e / 8, k = e % 8;
    Wdout[e] = (k == 1) ? zd{*wnew, 0.0} : Wd[(long)parent[j] * 8 + k];
  }
  for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < (long)nw * 4; e += (long)gridDim.x * blockDim.x)
    Wlout[e] = Wl[(long)parent[e / 4] * 4 + e % 4];
}

// W = conj(trial) per spin, W_data row = (0, 1, 0, ...), log-overlaps
// log 0 = {-inf, 0}
__global__ void init_walkers_kernel(zd* __restrict__ W, zd* __restrict__ Wd, zd* __restrict__ Wl,
                                    const zd* __restrict__ trial, int nw, long MN)
{
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  long tot = (long)nw * 2 * MN;
  if (i < tot) {
    long rem = i % (2 * MN);
    W[i] = zconj(trial[rem]);
  }
  if (i < (long)nw * 8) Wd[i] = zd{(i % 8 == 1) ? 1.0 : 0.0, 0.0};
  if (i < (long)nw * 4) Wl[i] = zd{-INFINITY, 0.0};
}

// ---------------------------------------------------------------------------
// Householder LQ with LAPACK conventions on the column-major view A = W^T
// (N x M) of each W[w][s] ([M][N] row-major): the blocked zgelqf followed by
// the blocked zunglq (ma::gelqf / ma::glq, src/Numerics/ma_lapack.hpp:134-221;
// called by afqmc_sys::orthogonalize, src/AFQMC/afqmc_sys.hpp:175-207).
// A(i, c) is W[c][i]: row i of A is column i of W.  One block of 256 threads
// per matrix.  Panels of NB rows are factorised in LDS (zgelq2 / zungl2);
// the rows below a panel get the block reflector I - V^H T V (zlarft
// 'Forward','Rowwise' + zlarfb 'Right') in two passes through L2.
__device__ inline zd wave_zsum(zd v)
{
  for (int o = 32; o >= 1; o >>= 1) {
    v.re += __shfl_xor(v.re, o);
    v.im += __shfl_xor(v.im, o);
  }
  return v;
}
__device__ inline double block_dsum(double v, double* sh)
{
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) sh[wv] = v;
  __syncthreads();
  return sh[0] + sh[1] + sh[2] + sh[3];
}

// V(r, c) of a panel held in LDS rows P[r*LP + c]: 1 on the diagonal, the
// stored tail right of it, 0 left of it.
__device__ inline zd vpanel(const zd* P, int LP, int r, int c)
{
  if (c == r) return zd{1.0, 0.0};
  if (c < r) return zd{0.0, 0.0};
  return P[r * LP + c];
}

// zlarfg on panel row r (already conjugated), LAPACK sign rule.
__device__ inline bool householder_row(zd* P, int LP, int r, double* sh, zd& alpha, zd& taui, double& beta)
{
  const int tid = threadIdx.x;
  double ss = 0.0;
  for (int c = r + 1 + tid; c < LP; c += 256) ss += P[r * LP + c].re * P[r * LP + c].re + P[r * LP + c].im * P[r * LP + c].im;
  const double xn2 = block_dsum(ss, sh);
  alpha = P[r * LP + r];
  const bool apply = !(xn2 == 0.0 && alpha.im == 0.0);
  taui = zd{0, 0};
  beta = 0.0;
  if (apply) {
    const double nrm = sqrt(alpha.re * alpha.re + alpha.im * alpha.im + xn2);
    beta = -copysign(nrm, alpha.re);
    taui = zd{(beta - alpha.re) / beta, -alpha.im / beta};
    const zd scal = zdiv(zd{1.0, 0.0}, zd{alpha.re - beta, alpha.im});
    for (int c = r + 1 + tid; c < LP; c += 256) P[r * LP + c] = zmul(scal, P[r * LP + c]);
  }
  __syncthreads();
  return apply;
}

// apply I - t v v^H (v = panel row r with unit diagonal) from the right to
// panel rows r+1..ib-1 over columns r..LP-1
template <int NB>
__device__ inline void panel_apply(zd* P, int LP, int r, int ib, zd t, zd* red)
{
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  zd acc[NB];
#pragma unroll
  for (int q = 0; q < NB; q++) acc[q] = zd{0, 0};
  for (int c = r + tid; c < LP; c += 256) {
    const zd vc = (c == r) ? zd{1.0, 0.0} : P[r * LP + c];
#pragma unroll
    for (int q = 0; q < NB; q++)
      if (q > r && q < ib) acc[q] = zadd(acc[q], zmul(P[q * LP + c], vc));
  }
#pragma unroll
  for (int q = 0; q < NB; q++) {
    zd s = wave_zsum(acc[q]);
    if (lane == 0) red[wv * NB + q] = s;
  }
  __syncthreads();
  zd wq[NB];
#pragma unroll
  for (int q = 0; q < NB; q++) wq[q] = zmul(t, zadd(zadd(red[q], red[NB + q]), zadd(red[2 * NB + q], red[3 * NB + q])));
  for (int c = r + tid; c < LP; c += 256) {
    const zd vcc = zconj((c == r) ? zd{1.0, 0.0} : P[r * LP + c]);
#pragma unroll
    for (int q = 0; q < NB; q++)
      if (q > r && q < ib) P[q * LP + c] = zsub(P[q * LP + c], zmul(wq[q], vcc));
  }
  __syncthreads();
}

// T (ib x ib, upper) of zlarft('Forward','Rowwise') from the panel and taus.
// The ib(ib-1)/2 dot products V(j,:) V(i,:)^H (j < i, columns >= i) are
// reduced block-wide, then one thread runs the triangular recursion.
template <int NB>
__device__ inline void form_T(const zd* P, int LP, int ib, const zd* tau, zd* T, zd* red)
{
  constexpr int NP = NB * (NB - 1) / 2;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  zd acc[NP];
#pragma unroll
  for (int e = 0; e < NP; e++) acc[e] = zd{0, 0};
  for (int c = tid; c < LP; c += 256) {
    zd pj[NB];
#pragma unroll
    for (int j = 0; j < NB; j++) pj[j] = (j < ib) ? P[j * LP + c] : zd{0, 0};
#pragma unroll
    for (int i = 1; i < NB; i++) {
      if (i >= ib || c < i) continue;
      const zd vi = zconj((c == i) ? zd{1.0, 0.0} : pj[i]);
#pragma unroll
      for (int j = 0; j < i; j++) acc[i * (i - 1) / 2 + j] = zadd(acc[i * (i - 1) / 2 + j], zmul(pj[j], vi));
    }
  }
#pragma unroll
  for (int e = 0; e < NP; e++) {
    zd s = wave_zsum(acc[e]);
    if (lane == 0) red[wv * NP + e] = s;
  }
  __syncthreads();
  if (tid == 0) {
    for (int i = 0; i < ib; i++) {
      const zd ti = tau[i];
      if (ti.re == 0.0 && ti.im == 0.0) {
        for (int j = 0; j <= i; j++) T[j * NB + i] = zd{0, 0};
        continue;
      }
      // T(0:i-1, i) = -tau_i V(0:i-1, :) V(i, :)^H, then T(0:i-1,0:i-1) times it (in place, ascending rows)
      for (int j = 0; j < i; j++) {
        const int e = i * (i - 1) / 2 + j;
        zd d = zadd(zadd(red[e], red[NP + e]), zadd(red[2 * NP + e], red[3 * NP + e]));
        T[j * NB + i] = zmul(zd{-ti.re, -ti.im}, d);
      }
      for (int j = 0; j < i; j++) {
        zd s{0, 0};
        for (int l = j; l < i; l++) s = zadd(s, zmul(T[j * NB + l], T[l * NB + i]));
        T[j * NB + i] = s;
      }
      T[i * NB + i] = ti;
    }
  }
  __syncthreads();
}

// C <- C (I - V^H op(T) V) for rows rb..N-1 of A, columns c0..M-1 (panel
// columns are local c = global - c0).  conjT: op(T) = T^H (zunglq), else T.
// Threads: 128 rows x 2 column halves; each thread keeps UNR independent
// loads in flight per iteration.
template <int NB>
__device__ inline void trailing_update(zd* W, int N, int rb, int c0, int LP, const zd* P, int ib, const zd* T,
                                       bool conjT, zd* W1)
{
  constexpr int UNR = 8;
  const int tid = threadIdx.x;
  const int nr = N - rb;
  const int half = tid >> 7;
  const int hl = (LP + 1) / 2;           // columns of half 0
  const int cb = half ? hl : 0, ce = half ? LP : hl;
  for (int q0 = 0; q0 < nr; q0 += 128) {
    const int ql = tid & 127;
    const int q = q0 + ql;
    const bool active = q < nr;
    zd acc[NB];
#pragma unroll
    for (int r = 0; r < NB; r++) acc[r] = zd{0, 0};
    for (int c = cb; c < ce; c += UNR) {
      zd cv[UNR];
#pragma unroll
      for (int u = 0; u < UNR; u++)
        cv[u] = (active && c + u < ce) ? W[(long)(c0 + c + u) * N + rb + q] : zd{0, 0};
#pragma unroll
      for (int u = 0; u < UNR; u++) {
        if (c + u >= ce) break;
#pragma unroll
        for (int r = 0; r < NB; r++)
          if (r < ib) acc[r] = zadd(acc[r], zmul(cv[u], zconj(vpanel(P, LP, r, c + u))));
      }
    }
    if (half == 1) {
#pragma unroll
      for (int r = 0; r < NB; r++) W1[ql * NB + r] = acc[r];
    }
    __syncthreads();
    zd w2[NB];
    if (half == 0) {
#pragma unroll
      for (int r = 0; r < NB; r++) acc[r] = zadd(acc[r], W1[ql * NB + r]);
      // W2 = W1 op(T)
#pragma unroll
      for (int r = 0; r < NB; r++) {
        zd s{0, 0};
#pragma unroll
        for (int j = 0; j < NB; j++) {
          if (j >= ib || r >= ib) continue;
          zd tjr = conjT ? ((r <= j) ? zconj(T[r * NB + j]) : zd{0, 0}) : ((j <= r) ? T[j * NB + r] : zd{0, 0});
          s = zadd(s, zmul(acc[j], tjr));
        }
        w2[r] = s;
      }
    }
    __syncthreads();
    if (half == 0) {
#pragma unroll
      for (int r = 0; r < NB; r++) W1[ql * NB + r] = w2[r];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < NB; r++) w2[r] = W1[ql * NB + r];
    if (active) {
      for (int c = cb; c < ce; c += UNR) {
        zd cv[UNR];
#pragma unroll
        for (int u = 0; u < UNR; u++) cv[u] = (c + u < ce) ? W[(long)(c0 + c + u) * N + rb + q] : zd{0, 0};
#pragma unroll
        for (int u = 0; u < UNR; u++) {
          if (c + u >= ce) break;
          zd s{0, 0};
#pragma unroll
          for (int r = 0; r < NB; r++)
            if (r < ib) s = zadd(s, zmul(w2[r], vpanel(P, LP, r, c + u)));
          W[(long)(c0 + c + u) * N + rb + q] = zsub(cv[u], s);
        }
      }
    }
    __syncthreads();
  }
}

// only != null: matrices b with only[b] == 0 are skipped (the fallback pass
// after the Cholesky route).
template <int NB>
__global__ __launch_bounds__(256) void lq_blocked_kernel(zd* __restrict__ Wall, int M, int N,
                                                         const int* __restrict__ only)
{
  if (only && only[blockIdx.x] == 0) return;
  extern __shared__ zd sm[];
  zd* P = sm;                  // [NB][M]
  zd* W1 = P + NB * M;         // [128][NB] (trailing rows go in chunks of 128)
  zd* T = W1 + 128 * NB;       // [NB][NB]
  zd* tau = T + NB * NB;       // [N]
  zd* red = tau + N;           // [4][NB*NB]
  __shared__ double sh[8];
  zd* W = Wall + (long)blockIdx.x * M * N;
  const int tid = threadIdx.x;
  auto load_panel = [&](int i0, int ib, int LP) {
    for (int e = tid; e < ib * LP; e += 256) {
      const int r = e % ib, c = e / ib;
      P[r * LP + c] = W[(long)(i0 + c) * N + i0 + r];
    }
    __syncthreads();
  };
  auto store_panel = [&](int i0, int ib, int LP) {
    for (int e = tid; e < ib * LP; e += 256) {
      const int r = e % ib, c = e / ib;
      W[(long)(i0 + c) * N + i0 + r] = P[r * LP + c];
    }
    __syncthreads();
  };
  // ---- zgelqf ----
  for (int i0 = 0; i0 < N; i0 += NB) {
    const int ib = min(NB, N - i0), LP = M - i0;
    load_panel(i0, ib, LP);
    for (int r = 0; r < ib; r++) {
      for (int c = r + tid; c < LP; c += 256) P[r * LP + c] = zconj(P[r * LP + c]);
      __syncthreads();
      zd alpha, taui;
      double beta;
      const bool apply = householder_row(P, LP, r, sh, alpha, taui, beta);
      if (tid == 0) tau[i0 + r] = taui;
      if (apply && r < ib - 1) panel_apply<NB>(P, LP, r, ib, taui, red);
      if (tid == 0) P[r * LP + r] = apply ? zd{beta, 0.0} : alpha;
      __syncthreads();
      for (int c = r + tid; c < LP; c += 256) P[r * LP + c] = zconj(P[r * LP + c]);
      __syncthreads();
    }
    store_panel(i0, ib, LP);
    if (i0 + ib < N) {
      form_T<NB>(P, LP, ib, tau + i0, T, red);
      trailing_update<NB>(W, N, i0 + ib, i0, LP, P, ib, T, false, W1);
    }
  }
  // ---- zunglq (k = N reflectors, blocks from last to first) ----
  const int last = ((N - 1) / NB) * NB;
  for (int i0 = last; i0 >= 0; i0 -= NB) {
    const int ib = min(NB, N - i0), LP = M - i0;
    load_panel(i0, ib, LP);
    if (i0 + ib < N) {
      form_T<NB>(P, LP, ib, tau + i0, T, red);
      trailing_update<NB>(W, N, i0 + ib, i0, LP, P, ib, T, true, W1);
    }
    // zungl2 on the panel rows
    for (int r = ib - 1; r >= 0; r--) {
      const zd ti = tau[i0 + r];
      if (r < LP - 1) {
        for (int c = r + 1 + tid; c < LP; c += 256) P[r * LP + c] = zconj(P[r * LP + c]);
        __syncthreads();
        if (r < ib - 1 && !(ti.re == 0.0 && ti.im == 0.0)) panel_apply<NB>(P, LP, r, ib, zconj(ti), red);
        const zd mt{-ti.re, -ti.im};
        for (int c = r + 1 + tid; c < LP; c += 256) P[r * LP + c] = zconj(zmul(mt, P[r * LP + c]));
      }
      __syncthreads();
      if (tid == 0) P[r * LP + r] = zd{1.0 - ti.re, ti.im};
      for (int c = tid; c < r; c += 256) P[r * LP + c] = zd{0, 0};
      __syncthreads();
    }
    store_panel(i0, ib, LP);
    for (int e = tid; e < ib * i0; e += 256) {
      const int r = e % ib, c = e / ib;
      W[(long)c * N + i0 + r] = zd{0, 0};
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Orthogonalisation through Cholesky QR.  For B = conj(W_s) (M x N), the
// reference's zgelqf + zunglq on the column-major view W_s^T equals
// zgeqrf + zungqr on B, so the new walker is conj(Q_h) with B = Q_h R_h and
// R_h's diagonal real with LAPACK's sign rule (beta = -sign(Re alpha) |x|).
// With the positive factorisation B = Q+ R+ (Cholesky of B^H B), Q_h = Q+ D
// for a diagonal D of +-1.  D is recovered without the reflectors: the
// no-pivot LU of the top N x N block X of Q+ in which each pivot is first
// shifted by s_k = -sign(Re X_kk) (the Householder reconstruction of Ballard
// et al., "Reconstructing Householder vectors from tall-skinny QR", 2015)
// yields exactly D_k = s_k, because that shift is the reconstructed
// reflector's choice of beta and the Householder factorisation of B is
// unique once the signs are fixed.

// Cholesky S = R^H R (R upper, positive diagonal) of a batch of Hermitian
// N x N matrices (row-major, upper triangle read) followed by the in-place
// Gauss-Jordan inverse of R: writes U = R^{-1} (upper, row-major).  Thread
// (i, cg) holds row i, columns cg + CG*t in registers.  A pivot below
// tol * max_k S_kk marks the matrix in fail[b] (its U is then undefined).
template <int NMAX, int CG>
__global__ __launch_bounds__(NMAX* CG) void chol_inv_kernel(const zd* __restrict__ S, zd* __restrict__ U, int N,
                                                            double tol, int* __restrict__ fail)
{
  constexpr int NC = NMAX / CG;
  __shared__ zd prow[2][NMAX];
  __shared__ zd colk[2][NMAX];
  __shared__ double dmax;
  const int tid = threadIdx.x;
  const int i = tid / CG, cg = tid % CG;
  const long b = blockIdx.x;
  const zd* Sb = S + b * (long)N * N;
  zd x[NC];
#pragma unroll
  for (int t = 0; t < NC; t++) {
    const int j = cg + CG * t;
    x[t] = (i < N && j < N && j >= i) ? Sb[(long)i * N + j] : zd{(i == j) ? 1.0 : 0.0, 0.0};
  }
  if (tid == 0) {
    double m = 0.0;
    for (int k = 0; k < N; k++) m = fmax(m, Sb[(long)k * N + k].re);
    dmax = m;
  }
  __syncthreads();
  const double thr = tol * dmax;
  bool bad = false;
  // Cholesky, right-looking on the upper triangle
  for (int k = 0; k < N; k++) {
    const int tk = k / CG, ck = k % CG, st = k & 1;
    if (i == k) {
#pragma unroll
      for (int t = 0; t < NC; t++) prow[st][cg + CG * t] = x[t];
    }
    __syncthreads();
    const double d = prow[st][k].re;
    if (!(d > thr)) {
      bad = true;
      break;
    }
    const double r = sqrt(d), rinv = 1.0 / r;
    if (i == k) {
#pragma unroll
      for (int t = 0; t < NC; t++) {
        const int j = cg + CG * t;
        x[t] = (j < k) ? zd{0, 0} : ((j == k) ? zd{r, 0.0} : zd{x[t].re * rinv, x[t].im * rinv});
      }
    } else if (i > k && i < N) {
      // conj(R_ki) R_kj = conj(S_ki) S_kj / d, on every column: the entries
      // left of the diagonal take garbage that is never read and is zeroed
      // before the inverse (padded columns of row k are zero)
      const zd ski = prow[st][i];
      const zd f{ski.re / d, -ski.im / d};
#pragma unroll
      for (int t = 0; t < NC; t++) {
        x[t] = zsub(x[t], zmul(f, prow[st][cg + CG * t]));
        if ((t & 7) == 7) asm volatile("" ::: "memory");  // bound the LDS loads in flight
      }
    }
    (void)tk;
    (void)ck;
  }
  if (bad) {
    if (tid == 0) fail[b] = 1;
    return;
  }
  // the last Cholesky step read prow[(N - 1) & 1], which the inverse's first
  // step (buffer 0) overwrites before its own barrier when N is odd
  __syncthreads();
  // rows i < N now hold R (upper); rows >= N the identity.  In-place
  // Gauss-Jordan inverse, pivots on the diagonal, the columns in blocks of CG
  // as gj_inverse_kernel: slot tk of block tk is held in xc, addressed
  // statically, for the block's CG steps.
#pragma unroll
  for (int t = 0; t < NC; t++) {
    const int j = cg + CG * t;
    if (j < i) x[t] = zd{0, 0};
  }
  const int nblk = (N + CG - 1) / CG;
  for (int tk = 0; tk < nblk; tk++) {
    zd xc{0, 0};
#pragma unroll
    for (int t = 0; t < NC; t++)
      if (t == tk) xc = x[t];
    const int jc = cg + CG * tk;
#pragma unroll
    for (int ck = 0; ck < CG; ck++) {
      const int k = CG * tk + ck, st = k & 1;
      if (k >= N) break;
      const bool own = (cg == ck);
      if (i == k) {
#pragma unroll
        for (int t = 0; t < NC; t++) prow[st][cg + CG * t] = x[t];
        prow[st][jc] = xc;  // after slot tk's stale copy: the later store wins
      }
      if (own) colk[st][i] = xc;
      __syncthreads();
      const double ipv = 1.0 / prow[st][k].re;  // R_kk is real
      if (i == k) {
#pragma unroll
        for (int t = 0; t < NC; t++) x[t] = zd{x[t].re * ipv, x[t].im * ipv};
        xc = own ? zd{ipv, 0.0} : zd{xc.re * ipv, xc.im * ipv};
      } else if (i < k) {
        const zd g = colk[st][i];
        const zd gq{-g.re * ipv, -g.im * ipv};
#pragma unroll
        for (int t = 0; t < NC; t++) {
          x[t] = zadd(x[t], zmul(gq, prow[st][cg + CG * t]));
          if ((t & 7) == 7) asm volatile("" ::: "memory");
        }
        xc = own ? gq : zadd(xc, zmul(gq, prow[st][jc]));
      }
    }
#pragma unroll
    for (int t = 0; t < NC; t++)
      if (t == tk) x[t] = xc;
  }
  zd* Ub = U + b * (long)N * N;
#pragma unroll
  for (int t = 0; t < NC; t++) {
    const int j = cg + CG * t;
    if (i < N && j < N) Ub[(long)i * N + j] = x[t];
  }
}

// Signs D of the LAPACK factor from the shifted no-pivot LU of the top
// N x N block of Q+ (conjugation leaves the real parts of the pivots
// unchanged, so the walker-layout block conj(Q+) is used as is), then
// Wout = Win D for every row.  Matrices with fail[b] set are skipped.
template <int NMAX, int CG>
__global__ __launch_bounds__(NMAX* CG) void ortho_sign_kernel(const zd* __restrict__ Win, zd* __restrict__ Wout,
                                                              int M, int N, const int* __restrict__ fail)
{
  constexpr int NC = NMAX / CG;
  __shared__ zd prow[2][NMAX];
  __shared__ zd colk[2][NMAX];
  __shared__ double sgn[NMAX];
  const long b = blockIdx.x;
  if (fail[b]) return;
  const int tid = threadIdx.x;
  const int i = tid / CG, cg = tid % CG;
  const zd* Wb = Win + b * (long)M * N;
  zd x[NC];
#pragma unroll
  for (int t = 0; t < NC; t++) {
    const int j = cg + CG * t;
    x[t] = (i < N && j < N) ? Wb[(long)i * N + j] : zd{0, 0};
  }
  for (int k = 0; k < N; k++) {
    const int tk = k / CG, ck = k % CG, st = k & 1;
    if (i == k) {
#pragma unroll
      for (int t = 0; t < NC; t++) prow[st][cg + CG * t] = x[t];
    }
    if (cg == ck) {
#pragma unroll
      for (int t = 0; t < NC; t++)
        if (t == tk) colk[st][i] = x[t];
    }
    __syncthreads();
    const zd pk = prow[st][k];
    const double sk = (pk.re >= 0.0) ? -1.0 : 1.0;
    if (tid == 0) sgn[k] = sk;
    if (i > k && i < N) {
      const zd l = zdiv(colk[st][i], zd{pk.re - sk, pk.im});
#pragma unroll
      for (int t = 0; t < NC; t++) {
        const int j = cg + CG * t;
        if (j > k) x[t] = zsub(x[t], zmul(l, prow[st][j]));
      }
    }
  }
  __syncthreads();
  zd* Wo = Wout + b * (long)M * N;
  const long tot = (long)M * N;
  for (long e = tid; e < tot; e += NMAX * CG) {
    const double s = sgn[e % N];
    const zd v = Wb[e];
    Wo[e] = zd{s * v.re, s * v.im};
  }
}

// ---------------------------------------------------------------------------
// Per-walker complex dot products without conjugation, reduction over i:
//   out[w] = scale * sum_i A(i, w) * B(i, w) (+ out[w] if accumulate)
// A(i,w) at A[i*asi + w*asw], same for B.  One block per walker.
template <class AT, class BT>
__global__ __launch_bounds__(256) void coldot_kernel(int n, const AT* __restrict__ A, long asi, long asw,
                                                     const BT* __restrict__ B, long bsi, long bsw, zd* out, long osw,
                                                     double scale, int accumulate)
{
  __shared__ zd sh[256];
  const int w = blockIdx.x;
  zd acc{0, 0};
  for (int i = threadIdx.x; i < n; i += 256) {
    const zd a = to_zd(A[(long)i * asi + (long)w * asw]);
    const zd bb = to_zd(B[(long)i * bsi + (long)w * bsw]);
    acc.re += a.re * bb.re - a.im * bb.im;
    acc.im += a.re * bb.im + a.im * bb.re;
  }
  sh[threadIdx.x] = acc;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) sh[threadIdx.x] = zadd(sh[threadIdx.x], sh[threadIdx.x + s]);
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    zd r{sh[0].re * scale, sh[0].im * scale};
    if (accumulate) r = zadd(r, out[(long)w * osw]);
    out[(long)w * osw] = r;
  }
}

// out[2 w + sp] = sum_t part[sp][t][w] (the exchange energy's partials), 16
// walkers and 16 groups of items per workgroup, summed in a fixed order.
__global__ __launch_bounds__(256) void exch_sum_kernel(const zd* __restrict__ part, int xt, int nw,
                                                       zd* __restrict__ out)
{
  __shared__ zd sh[16][16];
  const int wl = threadIdx.x & 15, grp = threadIdx.x >> 4, sp = blockIdx.y;
  const int w = blockIdx.x * 16 + wl;
  zd a{0, 0};
  if (w < nw)
    for (int t = grp; t < xt; t += 16) a = zadd(a, part[((long)sp * xt + t) * nw + w]);
  sh[grp][wl] = a;
  __syncthreads();
  if (grp == 0 && w < nw) {
    for (int q = 1; q < 16; q++) a = zadd(a, sh[q][wl]);
    out[2 * w + sp] = a;
  }
}

// Exchange reduction: for batch item q (a walker-spin), the sum over its nq
// Cholesky vectors of sum_ab Y_n(a,b) Y_n(b,a), Y stored [nq][N][N] per item.
// Workgroup (q, grp) of ngrp takes vectors grp, grp + ngrp, ... and leaves one
// partial; every entry is read once and coalesced, 32 x 32 blocks against
// their mirror blocks turned through LDS (128 items of 10 x 160 x 160: 637 ->
// 108 us; before, the mirror entries were read by single values and the
// index was divided by N per entry).
template <class YT>
__global__ __launch_bounds__(256) void trace_sq_kernel(const YT* __restrict__ Y, int N, int nq, long ystride,
                                                       zd* __restrict__ part, int ngrp)
{
  __shared__ zd tile[32][33];
  __shared__ zd sh[256];
  const int q = blockIdx.x, grp = blockIdx.y;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8
  const int nb = (N + 31) / 32;
  zd acc{0, 0};
  for (int n = grp; n < nq; n += ngrp) {
    const YT* Yn = Y + (long)q * ystride + (long)n * N * N;
    for (int bi = 0; bi < nb; bi++)
      for (int bj = bi; bj < nb; bj++) {
        zd d{0, 0};
        zd v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const int yy = ty + 8 * u;
          // block (bi, bj) to LDS, its mirror block (bj, bi) to registers
          const int r1 = bi * 32 + yy, c1 = bj * 32 + tx, r2 = bj * 32 + yy, c2 = bi * 32 + tx;
          tile[yy][tx] = r1 < N && c1 < N ? to_zd(Yn[(long)r1 * N + c1]) : zd{0, 0};
          v[u] = r2 < N && c2 < N ? to_zd(Yn[(long)r2 * N + c2]) : zd{0, 0};
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const zd t = tile[tx][ty + 8 * u];
          d.re += t.re * v[u].re - t.im * v[u].im;
          d.im += t.re * v[u].im + t.im * v[u].re;
        }
        __syncthreads();
        const double f = bi == bj ? 1.0 : 2.0;
        acc.re += f * d.re;
        acc.im += f * d.im;
      }
  }
  sh[threadIdx.x] = acc;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) sh[threadIdx.x] = zadd(sh[threadIdx.x], sh[threadIdx.x + s]);
    __syncthreads();
  }
  if (threadIdx.x == 0) part[(long)grp * gridDim.x + q] = sh[0];
}

// out[q] += sum_g part[g][q] in order, q < n
__global__ void add_parts_kernel(const zd* __restrict__ part, int ng, zd* __restrict__ out, int n)
{
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n) return;
  zd a = out[q];
  for (int g = 0; g < ng; g++) a = zadd(a, part[(long)g * n + q]);
  out[q] = a;
}

// The local energy's last step, one workgroup per walker: the Coulomb sum
// direct = inv_dt * sum_n v(w,n)^2, the exchange from its two spins, the
// one-body term sum_i G(w,i) haj(i), and W_data[w][0] = (direct - exch)/2 +
// e1 (energy.hpp:93-100 in the Cholesky form).  G and v walker-first.
template <class GZ>
__global__ __launch_bounds__(256) void energy_finish_kernel(int K, const zd* __restrict__ v, double inv_dt, int n,
                                                            const GZ* __restrict__ G, const zd* __restrict__ haj,
                                                            const zd* __restrict__ exch_part, zd* __restrict__ direct,
                                                            zd* __restrict__ exch, zd* __restrict__ one,
                                                            zd* __restrict__ Wd)
{
  __shared__ zd sh[2][256];
  const int w = blockIdx.x, tid = threadIdx.x;
  zd a{0, 0}, b{0, 0};
  for (int i = tid; i < K; i += 256) {
    const zd x = v[(long)w * K + i];
    a.re += x.re * x.re - x.im * x.im;
    a.im += 2.0 * x.re * x.im;
  }
  for (int i = tid; i < n; i += 256) {
    const zd g = to_zd(G[(long)w * n + i]), h = haj[i];
    b.re += g.re * h.re - g.im * h.im;
    b.im += g.re * h.im + g.im * h.re;
  }
  sh[0][tid] = a;
  sh[1][tid] = b;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (tid < s) {
      sh[0][tid] = zadd(sh[0][tid], sh[0][tid + s]);
      sh[1][tid] = zadd(sh[1][tid], sh[1][tid + s]);
    }
    __syncthreads();
  }
  if (tid == 0) {
    const zd d{inv_dt * sh[0][0].re, inv_dt * sh[0][0].im};
    const zd x = zadd(exch_part[2 * w], exch_part[2 * w + 1]);
    direct[w] = d;
    exch[w] = x;
    one[w] = sh[1][0];
    Wd[(long)w * 8] = zadd(zd{0.5 * (d.re - x.re), 0.5 * (d.im - x.im)}, sh[1][0]);
  }
}

// The same with Vakbl kept dense: Y = Vakbl G as ns partial products
// [ns][nw][n] (summed in order), one workgroup per walker; G(w, i) at
// G[w * gsw + i * gsi].
__global__ __launch_bounds__(512) void energy_vakbl_dense_kernel(int n, int nw, const zd* __restrict__ G, long gsw,
                                                                 long gsi, const zd* __restrict__ Y, int ns,
                                                                 const zd* __restrict__ haj, zd* __restrict__ direct,
                                                                 zd* __restrict__ exch, zd* __restrict__ one,
                                                                 zd* __restrict__ Wd)
{
  __shared__ zd sh[2][512];
  const int w = blockIdx.x, tid = threadIdx.x;
  zd a{0, 0}, b{0, 0};
  for (int i = tid; i < n; i += 512) {
    zd y{0, 0};
#pragma unroll 4
    for (int q = 0; q < ns; q++) y = zadd(y, Y[((long)q * nw + w) * n + i]);
    const zd g = G[w * gsw + i * gsi], h = haj[i];
    a.re += g.re * y.re - g.im * y.im;
    a.im += g.re * y.im + g.im * y.re;
    b.re += g.re * h.re - g.im * h.im;
    b.im += g.re * h.im + g.im * h.re;
  }
  sh[0][tid] = a;
  sh[1][tid] = b;
  __syncthreads();
  for (int s = 256; s > 0; s >>= 1) {
    if (tid < s) {
      sh[0][tid] = zadd(sh[0][tid], sh[0][tid + s]);
      sh[1][tid] = zadd(sh[1][tid], sh[1][tid + s]);
    }
    __syncthreads();
  }
  if (tid == 0) {
    direct[w] = sh[0][0];
    exch[w] = zd{0, 0};
    one[w] = sh[1][0];
    Wd[(long)w * 8] = zadd(zd{0.5 * sh[0][0].re, 0.5 * sh[0][0].im}, sh[1][0]);
  }
}

// The same with Vakbl in CSR (energy.hpp:93-100): direct = sum_i G(i,w) Y(i,w) with
// Y = Vakbl G, no exchange; G and Y walker-last, one workgroup per 16 walkers.
__global__ __launch_bounds__(1024) void energy_vakbl_kernel(int n, int nw, const zd* __restrict__ G,
                                                            const zd* __restrict__ Y, const zd* __restrict__ haj,
                                                            zd* __restrict__ direct, zd* __restrict__ exch,
                                                            zd* __restrict__ one, zd* __restrict__ Wd)
{
  __shared__ zd sh[2][64][16];
  const int lw = threadIdx.x & 15, grp = threadIdx.x >> 4;
  const int w = blockIdx.x * 16 + lw;
  zd a{0, 0}, b{0, 0};
  if (w < nw)
    for (int i = grp; i < n; i += 64) {
      const zd g = G[(long)i * nw + w], y = Y[(long)i * nw + w], h = haj[i];
      a.re += g.re * y.re - g.im * y.im;
      a.im += g.re * y.im + g.im * y.re;
      b.re += g.re * h.re - g.im * h.im;
      b.im += g.re * h.im + g.im * h.re;
    }
  sh[0][grp][lw] = a;
  sh[1][grp][lw] = b;
  __syncthreads();
  for (int s = 32; s >= 1; s >>= 1) {
    if (grp < s) {
      sh[0][grp][lw] = zadd(sh[0][grp][lw], sh[0][grp + s][lw]);
      sh[1][grp][lw] = zadd(sh[1][grp][lw], sh[1][grp + s][lw]);
    }
    __syncthreads();
  }
  if (grp == 0 && w < nw) {
    const zd d = sh[0][0][lw], e1 = sh[1][0][lw];
    direct[w] = d;
    exch[w] = zd{0, 0};
    one[w] = e1;
    Wd[(long)w * 8] = zadd(zd{0.5 * d.re, 0.5 * d.im}, e1);
  }
}

// ---------------------------------------------------------------------------
// Setup kernels.
// Scatter CSR Spvn [M*M][K] into dense Ld[n][ik] (Cholesky-vector major).
__global__ void csr_densify_kernel(int nrows, const int* __restrict__ rowptr, const int* __restrict__ col,
                                   const zd* __restrict__ val, zd* __restrict__ Ld, long ldn)
{
  int r = blockIdx.x * (blockDim.x / 64) + (threadIdx.x >> 6);
  int lane = threadIdx.x & 63;
  if (r >= nrows) return;
  int p0 = rowptr[0];
  for (int p = rowptr[r] - p0 + lane; p < rowptr[r + 1] - p0; p += 64) Ld[(long)col[p] * ldn + r] = val[p];
}

// CSR rows into a dense row-major matrix D[r][col] (zeroed beforehand;
// rowptr starts at 0, no repeated columns within a row)
__global__ void csr_densify_rows_kernel(int nrows, const int* __restrict__ rowptr, const int* __restrict__ col,
                                        const zd* __restrict__ val, zd* __restrict__ D, long ld)
{
  const int r = blockIdx.x * (blockDim.x / 64) + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (r >= nrows) return;
  for (int p = rowptr[r] + lane; p < rowptr[r + 1]; p += 64) D[(long)r * ld + col[p]] = val[p];
}

// per-row count of |Lt(n, j)| > cutoff, Lt spin-major [2][K][NM]: row n of
// SpvnT is (Lt[0][n][:], Lt[1][n][:]).
__global__ void rot_count_kernel(const zd* __restrict__ Lt, int K, long NM, double cutoff, int* __restrict__ cnt)
{
  __shared__ int sh[256];
  const int n = blockIdx.x;
  int c = 0;
  for (long j = threadIdx.x; j < 2 * NM; j += 256) {
    int sp = (int)(j / NM);
    zd v = Lt[(long)sp * K * NM + (long)n * NM + (j % NM)];
    if (hypot(v.re, v.im) > cutoff) c++;
  }
  sh[threadIdx.x] = c;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) cnt[n] = sh[0];
}

// fill of the CSR rows in ascending column order: one block per row, a
// block-wide prefix over chunks of 256 columns.
__global__ void rot_fill_kernel(const zd* __restrict__ Lt, int K, long NM, double cutoff,
                                const int* __restrict__ rowptr, int* __restrict__ colo, zd* __restrict__ valo)
{
  __shared__ int sh[256];
  const int n = blockIdx.x;
  int base = rowptr[n];
  for (long j0 = 0; j0 < 2 * NM; j0 += 256) {
    long j = j0 + threadIdx.x;
    bool keep = false;
    zd v{0, 0};
    if (j < 2 * NM) {
      int sp = (int)(j / NM);
      v = Lt[(long)sp * K * NM + (long)n * NM + (j % NM)];
      keep = hypot(v.re, v.im) > cutoff;
    }
    sh[threadIdx.x] = keep ? 1 : 0;
    __syncthreads();
    // inclusive scan (Hillis-Steele)
    for (int o = 1; o < 256; o <<= 1) {
      int t = (threadIdx.x >= o) ? sh[threadIdx.x - o] : 0;
      __syncthreads();
      sh[threadIdx.x] += t;
      __syncthreads();
    }
    if (keep) {
      int pos = base + sh[threadIdx.x] - 1;
      colo[pos] = (int)j;
      valo[pos] = v;
    }
    int tot = sh[255];
    __syncthreads();
    base += tot;
  }
}
