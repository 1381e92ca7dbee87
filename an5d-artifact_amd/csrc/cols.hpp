// One step per launch for the 3D boxes of radius >= 2 (125 to 729 taps): a
// column of cells per lane, streamed by planes with partial sums.
//
// A launch is bound by vector issue (249 to 1457 unfused operations a cell
// against 8 or 16 bytes).  The direct kernel gathers every tap of every cell
// from the caches, one load and its address arithmetic per multiply-add: that
// left box3d2r FP64 at 27 GStencil/s on 512^3.  Here a lane owns CK adjacent
// cells of a (row, run) of the plane and walks a segment of planes.  Each input
// plane is read row by row, one window of CK + 2R cells per lane, and every
// row adds its taps to the partial sums of the 2R+1 output planes it belongs
// to, so a loaded value feeds up to (2R+1)^2 multiply-adds from a register.
// The coefficients are wave-uniform and come through the scalar cache as
// scalar operands: no vector register and no LDS holds one.
//   - Lanes take runs row-major over the plane, with no tile: a grid of odd
//     extents wastes only the last run of a row.  That run ends at the
//     interior's end (it overlaps its neighbour and stores only its own
//     cells), so every window lies inside its row.
//   - A segment's warm-up planes add only to the outputs they belong to (a
//     wave-uniform branch per plane offset), so short segments cost loads and
//     no arithmetic, and a small grid can be cut into segments of one plane.
//   - The row loop is not unrolled: its body (648 to 1296 instructions at
//     radius 4) stays within the instruction cache.
// Measured (512^3, one step): box3d2r FP32 1994 -> 716 us, FP64 4964 -> 1386;
// box3d3r FP32 5830 -> 1727, FP64 11688 -> 3418; 256^3: box3d4r FP32 2052 ->
// 488, FP64 3163 -> 886 (27.6 T lane-operations/s, FP32 50 T).  Tried and
// slower: 8 cells a lane in FP32 (equal at 512^3, too few waves below 128^3),
// 2 cells (4-15 % from 128^3 on), two or three rows in flight (3-10 %).
#pragma once

#include "engine.hpp"
#include "sweep.hpp"

namespace an5d {

// Taps grouped by plane in ascending d0 over the full box; in each plane the
// centre tap first, then the others row-major (d1, then d2, ascending), as
// box3d2r.c, box3d3r.c and box3d4r.c list them: the partial sums then keep the
// C expression's order.
template <class D>
constexpr bool cols_order() {
  if (D::dim != 3 || !D::linear) return false;
  constexpr int R = D::rad, P = 2 * R + 1;
  if (D::ntaps != P * P * P) return false;
  int q = 0;
  for (int d0 = -R; d0 <= R; d0++) {
    if (D::taps[q].d0 != d0 || D::taps[q].d1 != 0 || D::taps[q].d2 != 0) return false;
    q++;
    for (int d1 = -R; d1 <= R; d1++)
      for (int d2 = -R; d2 <= R; d2++) {
        if (d1 == 0 && d2 == 0) continue;
        if (D::taps[q].d0 != d0 || D::taps[q].d1 != d1 || D::taps[q].d2 != d2) return false;
        q++;
      }
  }
  return true;
}

// Values of the coefficient table before the divisor (see cols_coefs).
constexpr int cols_table(int r) { return (2 * r + 1) * (1 + (2 * r + 1) * (2 * r + 1)); }

// Wave-uniform reads through the scalar cache (constant address space).
template <typename T>
using Uniform = const T __attribute__((address_space(4)))*;

template <int ID, typename T, int CK, bool EXACT>
__global__ __launch_bounds__(256) void cols_kernel(SweepArgs<T> a) {
#pragma clang fp contract(off)
  using D = Def<ID>;
  constexpr int R = D::rad, P = 2 * R + 1, W = CK + 2 * R;
  static_assert(cols_order<D>(), "plane-grouped box taps, centre first");
  // a.ntk: runs per row; a.ntj: workgroups per segment
  const int b = xcd_tile(blockIdx.x, gridDim.x);
  const int seg = b / a.ntj;
  const int nk = a.D2 - 2 * R, nj = a.D1 - 2 * R;
  const int run = (b - seg * a.ntj) * 256 + threadIdx.x;
  const int jn = run / a.ntk;
  const int kn = (run - jn * a.ntk) * CK;
  const bool own = jn < nj;         // lanes past the last row repeat it and store nothing
  const int j = min(jn, nj - 1);
  const int k = min(kn, nk - CK);   // nk >= CK (plan_launch)
  const int i0 = R + seg * a.sl;
  const int sle = min(a.sl, a.D0 - R - i0);
  if (sle <= 0) return;

  const long long s1 = a.s1;
  // the window's first cell (row j - R, column k - R) in a plane
  const long long voff = j * s1 + k;
  const Uniform<T> tab = (Uniform<T>)(unsigned long long)a.coef;

  T acc[P][CK];  // acc[d]: output plane n - d while input plane n is added
#pragma unroll
  for (int d = 0; d < P; d++)
#pragma unroll
    for (int kk = 0; kk < CK; kk++) acc[d][kk] = T(0);

  auto load = [&](auto& dst, const T* base) { load_run(dst, base + voff); };
  // one row is in flight while its predecessor is summed, the next plane's
  // centres for a whole plane; after the last plane they read it again
  const int nit = sle + 2 * R;
  const T* plane = a.src + (long long)(i0 - R) * a.s0;
  T row[W], cen[CK];
  load(row, plane);
  load(cen, plane + R * s1 + R);
  for (int n = 0; n < nit; n++) {
    // outputs n - d with 0 <= n - d < sle
    const int dlo = max(0, n - sle + 1), dhi = min(P - 1, n);
    // centre taps first
#pragma unroll
    for (int d = 0; d < P; d++) {
      const T c = tab[d];
#pragma unroll
      for (int kk = 0; kk < CK; kk++) {
        const T v = cen[kk];
        if constexpr (EXACT) {
          const T prod = c * v;
          acc[d][kk] = d == 0 ? prod : acc[d][kk] + prod;
        } else {
          acc[d][kk] = d == 0 ? c * v : fma_t(c, v, acc[d][kk]);
        }
      }
    }
    const T* const next = n + 1 < nit ? plane + a.s0 : plane;
    load(cen, next + R * s1 + R);
    auto do_row = [&](const T(&x)[W], Uniform<T> cr, auto center) {
#pragma unroll
      for (int d = 0; d < P; d++) {
        Uniform<T> crd = cr + d * P;
        T c[P];
#pragma unroll
        for (int e = 0; e < P; e++) c[e] = crd[e];
        if (d >= dlo && d <= dhi) {
#pragma unroll
          for (int e = 0; e < P; e++) {
            if (decltype(center)::value && e == R) continue;
#pragma unroll
            for (int kk = 0; kk < CK; kk++) {
              if constexpr (EXACT) acc[d][kk] = acc[d][kk] + c[e] * x[kk + e];
              else acc[d][kk] = fma_t(c[e], x[kk + e], acc[d][kk]);
            }
          }
        }
      }
    };
    Uniform<T> cr = tab + P;
    const T* rp = plane + s1;
#pragma unroll 1
    for (int r = 0; r < P; r++) {
      T x[W];
#pragma unroll
      for (int e = 0; e < W; e++) x[e] = row[e];
      load(row, r + 1 < P ? rp : next);
      rp += s1;
      if (r == R) do_row(x, cr, std::true_type{});
      else do_row(x, cr, std::false_type{});
      cr += P * P;
    }
    plane = next;
    // output plane m = n - 2R received its last input plane
    const int m = n - 2 * R;
    if (m >= 0) {
      T out[CK];
#pragma unroll
      for (int kk = 0; kk < CK; kk++) {
        out[kk] = acc[P - 1][kk];
        if (EXACT && a.has_div) out[kk] = div_by(out[kk], (T)tab[cols_table(R)], (T)tab[cols_table(R) + 1], a.has_div);
      }
      T* o = a.dst + (long long)(i0 + m) * a.s0 + (R + j) * s1 + R + k;
      if (own) {
        if (k == kn) {
          if (a.nt_store) gstore_run<true, T, CK>(o, out);
          else gstore_run<false, T, CK>(o, out);
        } else {
#pragma unroll
          for (int kk = 0; kk < CK; kk++)
            if (k + kk >= kn) o[kk] = out[kk];
        }
      }
    }
#pragma unroll
    for (int d = P - 1; d > 0; d--)
#pragma unroll
      for (int kk = 0; kk < CK; kk++) acc[d][kk] = acc[d - 1][kk];
  }
}

}  // namespace an5d
