// One step per launch for the 2D boxes of radius >= 2 (25 to 81 taps): a run of
// cells per lane, streamed by rows with partial sums.
//
// The sums are the row kernel's (rows.hpp): each input row adds its taps to the
// 2R+1 output rows it belongs to.  What differs is what that kernel spends
// beyond the expression: its coefficients are broadcast reads from LDS into
// vector registers and its row ends come by DPP and selects; here a lane reads
// its own window of CK + 2R cells (the caches serve the overlap) and the
// coefficients are scalar operands.  Lanes take the runs of all segments
// row-major, with no wave tile, so a narrow or ragged grid still fills its
// waves, and warm-up rows add only to the outputs they belong to, so segments
// may be a row long.  The last run of a row and the last segment end at the
// interior's end (they overlap their neighbours and store only their own
// cells): no load needs a clamp.
// Bound by vector issue from about 1024^2 on, by latency below.  Measured, one
// step, row kernel at its best segment -> here: box2d4r FP32 256^2 16.3 -> 6.7
// us, 1024^2 25.0 -> 8.5, 4096^2 76.2 -> 62.9, 8192^2 254 -> 196; FP64 1024^2
// 31.5 -> 12.6, 8192^2 450 -> 390; box2d3r FP32 8192^2 168 -> 136; box2d2r FP32
// 141 -> 111.  Eight cells a lane: equal in FP32, up to 1.6x slower in FP64.
#pragma once

#include "cols.hpp"
#include "rows.hpp"

namespace an5d {

template <int ID, typename T, int CK, bool EXACT>
__global__ __launch_bounds__(256) void cols2_kernel(SweepArgs<T> a) {
#pragma clang fp contract(off)
  using D = Def<ID>;
  constexpr int R = D::rad, P = 2 * R + 1, W = CK + 2 * R;
  static_assert(rows_order<D>(), "row-major box taps only");
  // a.ntk: runs per row
  const int run = xcd_tile(blockIdx.x, gridDim.x) * 256 + threadIdx.x;
  const int sn = run / a.ntk;
  const bool own = sn < a.nseg;  // lanes past the last segment repeat it and store nothing
  const int seg = min(sn, a.nseg - 1);
  const int kn = (run - sn * a.ntk) * CK;
  const int k = min(kn, a.D2 - 2 * R - CK);
  const int in = seg * a.sl;
  const int i = min(in, a.D0 - 2 * R - a.sl);
  const T* row = a.src + (long long)i * a.s0 + k;  // the window of the first input row
  T* out = a.dst + (long long)(i + R) * a.s0 + R + k;
  const Uniform<T> tab = (Uniform<T>)(unsigned long long)a.coef;

  T acc[P][CK];  // slot m mod P: output row m
#pragma unroll
  for (int d = 0; d < P; d++)
#pragma unroll
    for (int kk = 0; kk < CK; kk++) acc[d][kk] = T(0);
  const int nit = a.sl + 2 * R;
  T nxt[W];
  load_run(nxt, row);
  for (int n0 = 0; n0 < nit; n0 += P) {
    static_for<0, P>([&](auto uc) {
      constexpr int U = decltype(uc)::value;
      const int n = n0 + U;
      if (n < nit) {
        T x[W];
#pragma unroll
        for (int e = 0; e < W; e++) x[e] = nxt[e];
        if (n + 1 < nit) row += a.s0;
        load_run(nxt, row);
        static_for<0, P>([&](auto dc) {
          constexpr int DI = decltype(dc)::value;
          // the box row's coefficients through an offset the compiler cannot
          // hoist out of the loop
          int off = DI * P;
          asm volatile("" : "+s"(off));
          T c[P];
#pragma unroll
          for (int e = 0; e < P; e++) c[e] = tab[off + e];
          if (n >= DI && n - DI < a.sl) {
            static_for<0, P>([&](auto ec) {
              constexpr int E = decltype(ec)::value;
              constexpr int sign = D::taps[DI * P + E].sign;
#pragma unroll
              for (int kk = 0; kk < CK; kk++) {
                T& s = acc[(U - DI + P) % P][kk];
                const T v = x[kk + E];
                if constexpr (EXACT) {
                  const T prod = c[E] * v;
                  if constexpr (DI == 0 && E == 0) s = sign > 0 ? prod : -prod;
                  else if constexpr (sign > 0) s = s + prod;
                  else s = s - prod;
                } else {
                  if constexpr (DI == 0 && E == 0) s = c[E] * v;
                  else s = fma_t(c[E], v, s);
                }
              }
            });
          }
        });
        const int m = n - 2 * R;
        if (m >= 0) {
          T o[CK];
#pragma unroll
          for (int kk = 0; kk < CK; kk++) {
            o[kk] = acc[(U + 1) % P][kk];
            if (EXACT && a.has_div) o[kk] = div_by(o[kk], (T)tab[D::ntaps], (T)tab[D::ntaps + 1], a.has_div);
          }
          if (own && i + m >= in) {
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
