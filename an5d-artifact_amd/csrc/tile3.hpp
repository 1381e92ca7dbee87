// A few steps of a radius-1 3D stencil per launch on a tile held in registers.
//
// On grids of up to about 200^3 the streamed sweep has few segments of few
// planes and walks every warm-up plane through all stages behind one barrier
// each (128^3 FP64: 12 us a step).  Here a workgroup holds CI = OP + 2*BT planes
// of 32 rows x 64 cells in registers, every plane at once: the neighbours along
// dim 0 are the lane's own registers, those along the row come by DPP, and one
// exchange of edge rows through LDS per step serves all planes.  Step s only
// computes the planes that still count (OP + 2*(BT-s)), so the overlap along
// dim 0 costs loads but few operations.  Rows and columns give up BT cells on
// every side that is not the grid's edge.
// Bound by launch latency to 64^3, by vector issue above.  One step, sweep ->
// here: star3d1r 128^3 FP32 7.0 -> 5.6 us, FP64 12.7 -> 7.7; in FMA mode the boxes
// where their steps are bound by memory: j3d27pt FP32 512^3 287 -> 205 us, FP64
// 481 -> 412, 257x300x411 134 -> 107.  The exact boxes stay with one step per
// launch (twice the operations).
// Shapes (tile3_inst.hip): eight planes of 32 rows by 64 cells compute fewest
// cells; where they are fewer than the CUs, four planes and 16 rows.  star3d1r
// FP64 100x90x110, one step: 7.6 us on 104 tiles of eight planes, 5.3 on four
// planes, 4.8 on four planes of 16 rows; 64^3 7.2, 4.9, 3.2; FP32 100x90x110 5.4,
// 3.7, 3.5.  Tried: two cells a lane (slower from 128^3 on), four planes of two
// rows on 16 waves (3-20 % slower than on 8).
#pragma once

#include "engine.hpp"
#include "sweep.hpp"

namespace an5d {

// Stage input of cell (JJ, KK) of plane PP: the extended planes for taps off the
// cell's own column, the old planes for the column.
template <class D, typename T, int CI, int CJ, int CK, int PP, int JJ, int KK>
struct Tile3Get {
  const T (&u)[CI][CJ][CK];
  const T (&x)[3][CJ + 2][CK + 2];  // extended copies of planes PP-1 .. PP+1, where the stencil has them
  template <int A0, int A1, int A2>
  __device__ __forceinline__ T at() const {
    if constexpr (A1 == 0 && A2 == 0) return u[PP + A0][JJ][KK];
    else return x[1 + A0][JJ + A1 + 1][KK + A2 + 1];
  }
};

template <typename T, int CI, int CJ, int CK, int NW>
constexpr size_t tile3_buf_bytes() { return (size_t)CI * NW * 2 * 64 * CK * sizeof(T); }
template <typename T, int CI, int CJ, int CK, int NW>
constexpr int tile3_bufs() { return 2 * tile3_buf_bytes<T, CI, CJ, CK, NW>() <= 80 * 1024 ? 2 : 1; }

template <int ID, typename T, int BT, int OP, int CK, int CJ, int NW, bool EXACT, int DM>
__device__ __forceinline__ void tile3_body(const SweepArgs<T>& a) {
  using D = Def<ID>;
  static_assert(D::dim == 3 && D::rad == 1 && CJ >= 2, "radius-1 3D stencils");
  constexpr int NT = D::ntaps;
  constexpr int CI = OP + 2 * BT, W = 64 * CK, TJ = NW * CJ;
  constexpr int NB = tile3_bufs<T, CI, CJ, CK, NW>();
  constexpr size_t BUF = (size_t)CI * NW * 2 * W;
  extern __shared__ __align__(16) unsigned char an5d_lds[];
  T* const lds = reinterpret_cast<T*>(an5d_lds);

  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int b = xcd_tile(blockIdx.x, gridDim.x);
  const int tk = b % a.ntk;
  b /= a.ntk;
  const int tj = b % a.ntj, ti = b / a.ntj;
  // first plane (may lie before the grid), row and column; what the tile owns
  const int i0 = 1 + ti * OP - BT, j0 = tj * a.SJ, c0 = tk * a.SK;
  const int ihi = min(1 + (ti + 1) * OP, a.D0 - 1);
  const int jlo = tj == 0 ? 1 : j0 + BT, jhi = tj == a.ntj - 1 ? a.D1 - 1 : j0 + TJ - BT;
  const int klo = tk == 0 ? 1 : c0 + BT, khi = tk == a.ntk - 1 ? a.D2 - 1 : c0 + W - BT;
  const int jw = j0 + w * CJ, kl = c0 + lane * CK;

  bool kin[CK], kst[CK], cells_in = true, kst_all = true;
#pragma unroll
  for (int kk = 0; kk < CK; kk++) {
    const int k = kl + kk;
    kin[kk] = k >= 1 && k < a.D2 - 1;
    kst[kk] = k >= klo && k < khi;
    cells_in = cells_in && kin[kk];
    kst_all = kst_all && kst[kk];
  }
  const bool wave_in = __builtin_amdgcn_ballot_w64(!cells_in) == 0 && jw >= 1 && jw + CJ <= a.D1 - 1;

  T c[NT + 2];
#pragma unroll
  for (int q = 0; q < NT + 2; q++) c[q] = a.coef[q];
  const T div = c[NT];
  const int has_div = a.has_div;

  // every load reads a real cell: indices are clamped into the grid (the
  // stand-ins never reach a stored cell)
  T u[BT + 1][CI][CJ][CK];
#pragma unroll
  for (int p = 0; p < CI; p++) {
    const T* plane = a.src + (long long)min(max(i0 + p, 0), a.D0 - 1) * a.s0;
#pragma unroll
    for (int jj = 0; jj < CJ; jj++) {
      const T* row = plane + (long long)min(jw + jj, a.D1 - 1) * a.s1;
#pragma unroll
      for (int kk = 0; kk < CK; kk++) u[0][p][jj][kk] = row[min(kl + kk, a.D2 - 1)];
    }
  }
  static_for<1, BT + 1>([&](auto sc) {
    constexpr int S = decltype(sc)::value;
    constexpr int A = S - 1;  // planes [A, CI - A) hold step A
    T* buf = lds + (NB == 2 ? (S & 1) * BUF : 0);
    if constexpr (NB == 1 && S > 1) __syncthreads();
#pragma unroll
    for (int p = A; p < CI - A; p++) {
      T* o = buf + ((size_t)(p * NW + w) * 2) * W + lane * CK;
      store_run<T, CK>(o, u[A][p][0]);
      store_run<T, CK>(o + W, u[A][p][CJ - 1]);
    }
    __syncthreads();
    auto extend = [&](int p, T(&x)[CJ + 2][CK + 2]) {
      const int wu = max(w - 1, 0), wd = min(w + 1, NW - 1);
      T up[CK], dn[CK];
      load_run<T, CK>(up, buf + ((size_t)(p * NW + wu) * 2 + 1) * W + lane * CK);
      load_run<T, CK>(dn, buf + ((size_t)(p * NW + wd) * 2) * W + lane * CK);
#pragma unroll
      for (int r = 0; r < CJ + 2; r++) {
#pragma unroll
        for (int kk = 0; kk < CK; kk++) x[r][kk + 1] = r == 0 ? up[kk] : (r == CJ + 1 ? dn[kk] : u[A][p][r - 1][kk]);
        x[r][0] = from_left(x[r][CK]);
        x[r][CK + 1] = from_right(x[r][1]);
      }
    };
    constexpr bool BOX = needs_corners<D>();
    T x[3][CJ + 2][CK + 2];
    if constexpr (BOX) {
      extend(A, x[0]);
      extend(A + 1, x[1]);
    }
    static_for<S, CI - S>([&](auto pc) {
      constexpr int P = decltype(pc)::value;
      if constexpr (BOX) extend(P + 1, x[2]);
      else extend(P, x[1]);
      constexpr bool BATCHDIV = EXACT && DM == 2;
      T val[CJ][CK];
      static_for<0, CJ>([&](auto jc) {
        constexpr int JJ = decltype(jc)::value;
        static_for<0, CK>([&](auto kc) {
          constexpr int KK = decltype(kc)::value;
          Tile3Get<D, T, CI, CJ, CK, P, JJ, KK> get{u[A], x};
          if constexpr (BATCHDIV) val[JJ][KK] = eval_point<D, T, 0>(get, c, div, has_div, 1.0);
          else if constexpr (EXACT) val[JJ][KK] = eval_point<D, T, DM>(get, c, div, has_div, 1.0);
          else val[JJ][KK] = eval_fast<D, T>(get, c);
        });
      });
      if constexpr (BATCHDIV) {
        bool ok = true;
        T sum[CJ][CK];
#pragma unroll
        for (int jj = 0; jj < CJ; jj++)
#pragma unroll
          for (int kk = 0; kk < CK; kk++) {
            sum[jj][kk] = val[jj][kk];
            val[jj][kk] = div_fast(sum[jj][kk], div, c[NT + 1]);
            ok = ok && zero_or_normal(val[jj][kk]);
          }
        if (__builtin_amdgcn_ballot_w64(!ok) != 0) {
#pragma unroll
          for (int jj = 0; jj < CJ; jj++)
#pragma unroll
            for (int kk = 0; kk < CK; kk++)
              if (!zero_or_normal(val[jj][kk])) val[jj][kk] = sum[jj][kk] / div;
        }
      }
      const bool pin = i0 + P >= 1 && i0 + P < a.D0 - 1;
      if (pin && wave_in) {
#pragma unroll
        for (int jj = 0; jj < CJ; jj++)
#pragma unroll
          for (int kk = 0; kk < CK; kk++) u[S][P][jj][kk] = val[jj][kk];
      } else {
#pragma unroll
        for (int jj = 0; jj < CJ; jj++) {
          const bool rin = pin && jw + jj >= 1 && jw + jj < a.D1 - 1;
#pragma unroll
          for (int kk = 0; kk < CK; kk++) u[S][P][jj][kk] = rin && kin[kk] ? val[jj][kk] : u[A][P][jj][kk];
        }
      }
      if constexpr (BOX) {
#pragma unroll
        for (int r = 0; r < CJ + 2; r++)
#pragma unroll
          for (int kk = 0; kk < CK + 2; kk++) {
            x[0][r][kk] = x[1][r][kk];
            x[1][r][kk] = x[2][r][kk];
          }
      }
    });
  });
  static_for<BT, BT + OP>([&](auto pc) {
    constexpr int P = decltype(pc)::value;
    if (i0 + P < ihi) {
#pragma unroll
      for (int jj = 0; jj < CJ; jj++) {
        const int j = jw + jj;
        if (j < jlo || j >= jhi) continue;
        T* row = a.dst + (long long)(i0 + P) * a.s0 + (long long)j * a.s1 + kl;
        if (kst_all) {
          gstore_run<false, T, CK>(row, u[BT][P][jj]);
        } else {
#pragma unroll
          for (int kk = 0; kk < CK; kk++)
            if (kst[kk]) row[kk] = u[BT][P][jj][kk];
        }
      }
    }
  });
}

template <int ID, typename T, int BT, int OP, int CK, int CJ, int NW, bool EXACT>
__global__ __launch_bounds__(64 * NW) void tile3_kernel(SweepArgs<T> a) {
  if constexpr (!EXACT) {
    tile3_body<ID, T, BT, OP, CK, CJ, NW, EXACT, 0>(a);
  } else if constexpr (Def<ID>::divisor != 0) {
    if (a.has_div == 2) tile3_body<ID, T, BT, OP, CK, CJ, NW, EXACT, 2>(a);
    else tile3_body<ID, T, BT, OP, CK, CJ, NW, EXACT, -1>(a);
  } else {
    if (a.has_div == 0) tile3_body<ID, T, BT, OP, CK, CJ, NW, EXACT, 0>(a);
    else tile3_body<ID, T, BT, OP, CK, CJ, NW, EXACT, -1>(a);
  }
}

}  // namespace an5d
