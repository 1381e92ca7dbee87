// The reverse block of a 2D linear stencil on a tile held in registers.
//
// A streamed block runs its warm-up planes one after the other in every
// segment (18 for bt = 5), each through all stages: a grid of 300 x 500 gave 24
// waves to 1024 SIMDs, and 31 us a block whatever its work.  Here a workgroup
// holds a tile of u_t0 and lambda in registers (CJ rows x CK cells per lane, NW
// waves along the rows), steps the states u_t0 .. u_t0+BT-1 forward, keeps them
// all, and walks back: edge rows through LDS and one barrier per step, DPP for
// the neighbours within a row, no plane order to wait for.  A linear block
// needs no state outside its own cells' neighbours, so a tile gives up only
// BT*R cells per side, none at the grid's own edges.
// Bound by latency and barriers below about 512^2 and by vector issue above;
// where streams fill the chip they do less work per cell (adj_launch_plan has
// the times of both).  Built for FP64 only: see there.
// Precision: a lane sums at most BT*CJ*CK products before the FP64 reduction of
// the wave, fewer than a streamed lane does.
#pragma once

#include "adjoint.hpp"
#include "tile2.hpp"

namespace an5d {

// The rows of `v` and the R rows above and below (from the neighbour waves'
// published edges at `in`), each extended by R cells with DPP.
template <int R, typename T, int CJ, int CK, int NW>
__device__ __forceinline__ void tile_extend(const T (&v)[CJ][CK], const T* in, int w,
                                            T (&x)[CJ + 2 * R][CK + 2 * R]) {
  constexpr int W = 64 * CK, ER = edge_rows<CJ, R>();
  static_for<0, CJ + 2 * R>([&](auto rc) {
    constexpr int RR = decltype(rc)::value, JR = RR - R;
    T r[CK];
    if constexpr (JR >= 0 && JR < CJ) {
#pragma unroll
      for (int kk = 0; kk < CK; kk++) r[kk] = v[JR][kk];
    } else {
      constexpr int WOFF = JR >= 0 ? JR / CJ : -((-JR + CJ - 1) / CJ);
      constexpr int E = edge_index<CJ, R>(JR - WOFF * CJ);
      static_assert(E >= 0, "halo row must be published");
      const int ws = min(max(w + WOFF, 0), NW - 1);
      load_run<T, CK>(r, in + (ws * ER + E) * W);
    }
#pragma unroll
    for (int kk = 0; kk < CK; kk++) x[RR][kk + R] = r[kk];
#pragma unroll
    for (int m = 1; m <= R; m++) {
      x[RR][R - m] = from_left(r[CK - m]);
      x[RR][R + CK - 1 + m] = from_right(r[m - 1]);
    }
  });
}

// LDS: two buffers, each with the published edge rows of the states and of the
// adjoint; reused by the waves' gradient sums at the end.
template <int ID, typename T, int CK, int CJ, int NW>
constexpr size_t adj_tile_lds_bytes() {
  const size_t rows = 4 * tile2_buf_bytes<ID, T, CK, CJ, NW>();
  const size_t sums = (size_t)NW * Def<ID>::ntaps * sizeof(double);
  return rows > sums ? rows : sums;
}

template <int ID, typename T, int BT, int CK, int CJ, int NW>
__global__ __launch_bounds__(64 * NW) void adjoint_tile_kernel(AdjArgs<T> a) {
  using D = Def<ID>;
  static_assert(D::dim == 2 && D::linear, "2D linear stencils");
  constexpr int R = D::rad, NT = D::ntaps, H = BT * R;
  constexpr int W = 64 * CK, TH = NW * CJ, ER = edge_rows<CJ, R>();
  constexpr int BUF = NW * ER * W;  // elements of one set of edge rows
  extern __shared__ __align__(16) unsigned char an5d_lds[];
  T* const lds = reinterpret_cast<T*>(an5d_lds);

  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int b = xcd_tile(blockIdx.x, gridDim.x);
  const int ti = b / a.ntk, tk = b - ti * a.ntk;
  const int r0 = ti * a.sl, c0 = tk * a.SK;
  const int olo = ti == 0 ? R : r0 + H, ohi = ti == a.nseg - 1 ? a.D0 - R : r0 + TH - H;
  const int klo = tk == 0 ? R : c0 + H, khi = tk == a.ntk - 1 ? a.D2 - R : c0 + W - H;
  const int rw = r0 + w * CJ, kl = c0 + lane * CK;

  bool kin[CK], kown[CK], rin[CJ], rown[CJ];
  bool own_all = true;
#pragma unroll
  for (int kk = 0; kk < CK; kk++) {
    kin[kk] = kl + kk >= R && kl + kk < a.D2 - R;
    kown[kk] = kl + kk >= klo && kl + kk < khi;
    own_all = own_all && kown[kk];
  }
#pragma unroll
  for (int jj = 0; jj < CJ; jj++) {
    rin[jj] = rw + jj >= R && rw + jj < a.D0 - R;
    rown[jj] = rw + jj >= olo && rw + jj < ohi;
  }

  // transposed taps and forward taps alike: s_q c_q / div
  const T div = a.coef[NT];
  T ct[NT];
  static_for<0, NT>([&](auto qc) {
    constexpr int Q = decltype(qc)::value;
    const T v = D::taps[Q].sign > 0 ? a.coef[Q] : -a.coef[Q];
    ct[Q] = a.has_div ? v / div : v;
  });

  // cells beyond the grid come from the workspace's zero padding
  T us[BT][CJ][CK], mu[CJ][CK];
#pragma unroll
  for (int jj = 0; jj < CJ; jj++) {
    load_run<T, CK>(us[0][jj], a.U + (long long)(rw + jj) * a.s0 + kl);
    load_run<T, CK>(mu[jj], a.Lin + (long long)(rw + jj) * a.s0 + kl);
  }
  int buf = 0;  // alternates: one barrier separates the writers of a buffer from its readers
  auto publish = [&](const T(&v)[CJ][CK], int set) {
    T* o = lds + (size_t)(2 * buf + set) * BUF + (size_t)w * ER * W + lane * CK;
#pragma unroll
    for (int jj = 0; jj < CJ; jj++) {
      const int e = edge_index<CJ, R>(jj);
      if (e >= 0) store_run<T, CK>(o + e * W, v[jj]);
    }
  };
  auto edges = [&](int set) { return lds + (size_t)(2 * buf + set) * BUF + lane * CK; };

  // states u_{t0+1} .. u_{t0+BT-1}
  static_for<1, BT>([&](auto mc) {
    constexpr int M = decltype(mc)::value;
    publish(us[M - 1], 0);
    __syncthreads();
    T x[CJ + 2 * R][CK + 2 * R];
    tile_extend<R, T, CJ, CK, NW>(us[M - 1], edges(0), w, x);
    buf ^= 1;
#pragma unroll
    for (int jj = 0; jj < CJ; jj++)
#pragma unroll
      for (int kk = 0; kk < CK; kk++) {
        T v = T(0);
        static_for<0, NT>([&](auto qc) {
          constexpr int Q = decltype(qc)::value;
          constexpr TapDef t = D::taps[Q];
          v = fma_t(ct[Q], x[jj + R + t.d0][kk + R + t.d2], v);
        });
        us[M][jj][kk] = rin[jj] && kin[kk] ? v : us[M - 1][jj][kk];
      }
  });
  // adjoint steps t = t0+BT-1 .. t0
  T gp[NT];
#pragma unroll
  for (int q = 0; q < NT; q++) gp[q] = T(0);
  static_for<1, BT + 1>([&](auto ac) {
    constexpr int M = BT - decltype(ac)::value;
    publish(us[M], 0);
    publish(mu, 1);
    __syncthreads();
    {
      T x[CJ + 2 * R][CK + 2 * R];
      tile_extend<R, T, CJ, CK, NW>(us[M], edges(0), w, x);
#pragma unroll
      for (int jj = 0; jj < CJ; jj++)
#pragma unroll
        for (int kk = 0; kk < CK; kk++) {
          const T m = rown[jj] && kown[kk] ? mu[jj][kk] : T(0);
          static_for<0, NT>([&](auto qc) {
            constexpr int Q = decltype(qc)::value;
            constexpr TapDef t = D::taps[Q];
            gp[Q] = fma_t(m, x[jj + R + t.d0][kk + R + t.d2], gp[Q]);
          });
        }
    }
    // formed here: interleaved with the transposed taps both extensions would
    // be live at once (128 registers and spills for the 9-point stencils)
#pragma unroll
    for (int q = 0; q < NT; q++) asm volatile("" : "+v"(gp[q]));
    T x[CJ + 2 * R][CK + 2 * R];
    tile_extend<R, T, CJ, CK, NW>(mu, edges(1), w, x);
    buf ^= 1;
#pragma unroll
    for (int jj = 0; jj < CJ; jj++)
#pragma unroll
      for (int kk = 0; kk < CK; kk++) {
        T v = T(0);
        static_for<0, NT>([&](auto qc) {
          constexpr int Q = decltype(qc)::value;
          constexpr TapDef t = D::taps[Q];
          v = fma_t(ct[Q], x[jj + R - t.d0][kk + R - t.d2], v);
        });
        mu[jj][kk] = rin[jj] && kin[kk] ? v : T(0);
      }
  });
#pragma unroll
  for (int jj = 0; jj < CJ; jj++) {
    if (!rown[jj]) continue;
    T* row = a.Lout + (long long)(rw + jj) * a.s0 + kl;
    if (own_all) {
      gstore_run<false, T, CK>(row, mu[jj]);
    } else {
#pragma unroll
      for (int kk = 0; kk < CK; kk++)
        if (kown[kk]) row[kk] = mu[jj][kk];
    }
  }
  // the tile's gradient sums: lanes, then waves, in a fixed order; FP64
  double* sums = reinterpret_cast<double*>(an5d_lds);
  __syncthreads();  // the last step's edge rows are read
  static_for<0, NT>([&](auto qc) {
    constexpr int Q = decltype(qc)::value;
    const double v = wave_sum<T>((double)gp[Q]);
    if (lane == 0) sums[w * NT + Q] = v;
  });
  __syncthreads();
  if (threadIdx.x < NT) {
    double v = 0.0;
    for (int i = 0; i < NW; i++) v += sums[i * NT + threadIdx.x];
    double s = 1.0;
    static_for<0, NT>([&](auto qc) {
      constexpr int Q = decltype(qc)::value;
      if (threadIdx.x == Q && D::taps[Q].sign < 0) s = -1.0;
    });
    a.gslot[(size_t)b * NT + threadIdx.x] += s * v / (a.has_div ? (double)div : 1.0);
  }
}

}  // namespace an5d
