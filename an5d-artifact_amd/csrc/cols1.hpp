// One step per launch for the radius-1 3D boxes (27 taps): a column of cells per
// lane, streamed by planes with partial sums.
//
// The column kernel of the wide boxes (cols.hpp) with what 27 taps allow: the
// coefficients stay in scalar registers for the whole segment, the three rows
// of a plane are loaded together one plane ahead, and the loop is unrolled by
// the three planes in flight, so no sum moves.  Against the plane-streamed wave
// tiles (rows.hpp): no coefficient is read from LDS into vector registers, no
// DPP and selects for the row ends, and no tile of 64-128 cells by 16-32 rows
// whose last ones are part empty (411 cells are 3.2 of them).
// Bound by vector issue in FP32 (53 operations a cell), by memory in FP64.
// Measured, one step, best wave tile -> here: j3d27pt FP32 128^3 12.5 -> 7.8
// us, 256^3 45.5 -> 34.6, 257x300x411 88.8 -> 63.5, 512^3 321 -> 304; FP64 128^3
// 15.5 -> 11.7, 257x300x411 161 -> 153, 512^3 568 -> 568; 64^3 (direct kernel)
// FP32 4.05 -> 3.2, FP64 4.9 -> 3.9.
#pragma once

#include "cols.hpp"

namespace an5d {

template <int ID, typename T, int CK, bool EXACT>
__global__ __launch_bounds__(256) void cols1_kernel(SweepArgs<T> a) {
#pragma clang fp contract(off)
  using D = Def<ID>;
  static_assert(cols_order<D>() && D::rad == 1, "plane-grouped 27-point boxes");
  constexpr int P = 3, W = CK + 2, NP = 9;  // taps per plane
  // a.ntk: runs per row; a.ntj: workgroups per segment
  const int b = xcd_tile(blockIdx.x, gridDim.x);
  const int seg = b / a.ntj;
  const int nk = a.D2 - 2, nj = a.D1 - 2;
  const int run = (b - seg * a.ntj) * 256 + threadIdx.x;
  const int jn = run / a.ntk;
  const int kn = (run - jn * a.ntk) * CK;
  const bool own = jn < nj;
  const int j = min(jn, nj - 1);
  const int k = min(kn, nk - CK);
  const int i0 = 1 + seg * a.sl;
  const int sle = min(a.sl, a.D0 - 1 - i0);
  if (sle <= 0) return;
  const long long voff = j * a.s1 + k;
  const Uniform<T> tab = (Uniform<T>)(unsigned long long)a.coef;
  T c[D::ntaps + 2];
#pragma unroll
  for (int q = 0; q < D::ntaps + 2; q++) c[q] = tab[q];

  T acc[P][CK];
#pragma unroll
  for (int d = 0; d < P; d++)
#pragma unroll
    for (int kk = 0; kk < CK; kk++) acc[d][kk] = T(0);
  const int nit = sle + 2;
  const T* plane = a.src + (long long)(i0 - 1) * a.s0 + voff;
  T nxt[P][W];
#pragma unroll
  for (int r = 0; r < P; r++) load_run(nxt[r], plane + r * a.s1);
  T* out = a.dst + (long long)i0 * a.s0 + (1 + j) * a.s1 + 1 + k;
  for (int n0 = 0; n0 < nit; n0 += P) {
    static_for<0, P>([&](auto uc) {
      constexpr int U = decltype(uc)::value;
      const int n = n0 + U;
      if (n < nit) {
        T x[P][W];
#pragma unroll
        for (int r = 0; r < P; r++)
#pragma unroll
          for (int e = 0; e < W; e++) x[r][e] = nxt[r][e];
        if (n + 1 < nit) plane += a.s0;
#pragma unroll
        for (int r = 0; r < P; r++) load_run(nxt[r], plane + r * a.s1);
        static_for<0, P>([&](auto dc) {
          constexpr int DI = decltype(dc)::value;
          if (n >= DI && n - DI < sle) {
            static_for<0, NP>([&](auto qc) {
              constexpr int Q = DI * NP + decltype(qc)::value;
              constexpr TapDef t = D::taps[Q];
#pragma unroll
              for (int kk = 0; kk < CK; kk++) {
                T& s = acc[(U - DI + P) % P][kk];
                const T v = x[1 + t.d1][1 + kk + t.d2];
                if constexpr (EXACT) {
                  const T prod = c[Q] * v;
                  if constexpr (Q == 0) s = t.sign > 0 ? prod : -prod;
                  else if constexpr (t.sign > 0) s = s + prod;
                  else s = s - prod;
                } else {
                  if constexpr (Q == 0) s = c[0] * v;
                  else s = fma_t(c[Q], v, s);
                }
              }
            });
          }
        });
        if (n >= 2) {
          T o[CK];
#pragma unroll
          for (int kk = 0; kk < CK; kk++) {
            o[kk] = acc[(U + 1) % P][kk];
            if (EXACT && a.has_div) o[kk] = div_by(o[kk], c[D::ntaps], c[D::ntaps + 1], a.has_div);
          }
          if (own) {
            if (k == kn) {
              if (a.nt_store) gstore_run<true, T, CK>(out, o);
              else gstore_run<false, T, CK>(out, o);
            } else {
#pragma unroll
              for (int kk = 0; kk < CK; kk++)
                if (k + kk >= kn) out[kk] = o[kk];
            }
          }
          out += a.s0;
        }
      }
    });
  }
}

}  // namespace an5d
