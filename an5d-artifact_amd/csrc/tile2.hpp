// Several steps of a 2D stencil per launch on a tile held in registers.
//
// The streamed sweep runs a segment's planes one after the other through every
// stage; a grid too small to give each SIMD a few waves of long segments waits
// on that chain (256^2: 16 waves, 40 planes, 44 us for four steps).  Here a
// workgroup holds a tile of NW*CJ rows x 64*CK cells in registers and advances
// all of it step by step: lanes hold CK cells of CJ rows, neighbours in the row
// come by DPP, a wave's R edge rows go through LDS (two buffers and one barrier
// per step where they fit).  The tile gives up R cells per step on every side
// that is not the grid's own edge, so the number of steps is a trade of halo
// against launches; it is a run-time value, one kernel serves every depth.
// Waves whose rows are all given up stop computing and only keep the barriers.
// Bound by launch latency, barriers and a lone wave's LDS round trips up to about
// 512^2 (256^2: the vector units issue a fifth of the time), by vector issue and
// those phases together above (FMA 1000x3001: they issue half of it; a tile of 128 x
// 64 computes 1.3-2 cells per stored one).  Measured, one step,
// best streamed configuration -> tile: j2d5pt FP32 256^2 1.43 -> 0.62 us, 512^2
// 1.73 -> 0.98, 1024^2 2.69 -> 1.80; star2d2r FP32 1024^2 5.97 -> 1.92, 4096^2
// 18.2 -> 14.5; star2d4r FP32 1024^2 10.2 -> 4.9; gradient2d FP64 2048^2 14.7 ->
// 10.6.  The streams win from about 6144^2 (star2d1r, box2d1r FP32) to 8192^2 on
// (j2d5pt FP32), sooner at radius 2 and more.
// Shapes (tile2_inst.hip): 64 x 32 cells (few per lane, most workgroups) for the
// smallest grids, 128 x 64 on 16 or 8 waves above; radius 3-4 needs four cells
// a lane (256 wide).  FP32 also has 128 x 128 on 16 waves, which computes 1.2-1.5
// cells per stored one where 128 x 64 computes 1.4-2, and 256 x 64 on 8, which
// moves half as many cells between lanes: the first is best where one or two of
// its tiles fill each CU (j2d9pt-gol FMA 1000x3001, one step: 2.78 -> 2.16 us,
// 6144^2 20.1 -> 16.4; star2d2r 1000x3001 4.25 -> 4.02), the second from 6144^2
// (j2d5pt FMA 8192^2 20.9 -> 20.2 us).  Tried: 64 x 32 on 8 waves, 64 x 64, 128 x
// 32 (within 5 % of a kept shape or slower everywhere); resident workgroups that
// take tiles in turn and load the next one's cells under this one's steps (8
// waves 13-18 % slower at 4096^2 and 8192^2, 16 waves 5-8 % faster).
#pragma once

#include "engine.hpp"
#include "sweep.hpp"

namespace an5d {

template <class D, typename T, int CJ, int CK, int JJ, int KK>
struct TileGet {
  const T (&x)[CJ + 2 * D::rad][CK + 2 * D::rad];
  template <int A0, int A1, int A2>
  __device__ __forceinline__ T at() const { return x[JJ + A0 + D::rad][KK + A2 + D::rad]; }
};

// LDS buffers of the edge-row exchange: two (one barrier per step) where they
// fit, else one (two barriers).
template <int ID, typename T, int CK, int CJ, int NW>
constexpr size_t tile2_buf_bytes() {
  return (size_t)NW * edge_rows<CJ, Def<ID>::rad>() * 64 * CK * sizeof(T);
}
template <int ID, typename T, int CK, int CJ, int NW>
constexpr int tile2_bufs() { return 2 * tile2_buf_bytes<ID, T, CK, CJ, NW>() <= 160 * 1024 ? 2 : 1; }

// Where a wave's part of a tile lies: its first row, the lane's first column,
// the rows and columns the tile owns, and the wave's last step.
template <int CK, int CJ, int NW>
struct Tile2Pos {
  int rw, kl, olo, ohi, last;
  bool kin[CK], kst[CK], kst_all, wave_in;
  __device__ __forceinline__ Tile2Pos(int R, int D0, int D2, int ntk, int nseg, int SJ, int SK, int tile, int steps,
                                      int lane, int w) {
    constexpr int W = 64 * CK, TH = NW * CJ;
    const int H = steps * R;
    const int ti = tile / ntk, tk = tile - ti * ntk;
    const int r0 = ti * SJ, c0 = tk * SK;
    const bool top = ti == 0, bot = ti == nseg - 1;
    rw = r0 + w * CJ;
    kl = c0 + lane * CK;
    olo = top ? R : r0 + H;
    ohi = bot ? D0 - R : r0 + TH - H;
    // a row that stays exact: R rows are lost per step from every tile edge
    // that is not the grid's
    last = min(top ? steps : (w * CJ + CJ - 1) / R, bot ? steps : (TH - w * CJ - 1) / R);
    const int klo = tk == 0 ? R : c0 + H, khi = tk == ntk - 1 ? D2 - R : c0 + W - H;
    bool cells_in = true;
    kst_all = true;
#pragma unroll
    for (int kk = 0; kk < CK; kk++) {
      const int k = kl + kk;
      kin[kk] = k >= R && k < D2 - R;
      kst[kk] = k >= klo && k < khi;
      cells_in = cells_in && kin[kk];
      kst_all = kst_all && kst[kk];
    }
    wave_in = __builtin_amdgcn_ballot_w64(!cells_in) == 0 && rw >= R && rw + CJ <= D0 - R;
  }
};

// The lane's cells of a tile, rows and columns clamped into the grid.
template <typename T, int CK, int CJ>
__device__ __forceinline__ void tile2_load(T (&d)[CJ][CK], const T* src, long long s0, int D0, int D2, int ntk, int SJ,
                                           int SK, int tile, int lane, int w) {
  const int ti = tile / ntk, c0 = (tile - ti * ntk) * SK;
  const int rw = ti * SJ + w * CJ, kl = c0 + lane * CK;
  if (c0 + 64 * CK <= D2) {
#pragma unroll
    for (int jj = 0; jj < CJ; jj++) load_run<T, CK>(d[jj], src + (long long)min(rw + jj, D0 - 1) * s0 + kl);
  } else {
#pragma unroll
    for (int jj = 0; jj < CJ; jj++) {
      const T* row = src + (long long)min(rw + jj, D0 - 1) * s0;
#pragma unroll
      for (int kk = 0; kk < CK; kk++) d[jj][kk] = row[min(kl + kk, D2 - 1)];
    }
  }
}

template <typename T, int CK, int CJ, class Pos>
__device__ __forceinline__ void tile2_store(const T (&u)[CJ][CK], const Pos& p, T* dst, long long s0) {
#pragma unroll
  for (int jj = 0; jj < CJ; jj++) {
    const int r = p.rw + jj;
    if (r < p.olo || r >= p.ohi) continue;
    T* row = dst + (long long)r * s0 + p.kl;
    if (p.kst_all) {
      gstore_run<false, T, CK>(row, u[jj]);
    } else {
#pragma unroll
      for (int kk = 0; kk < CK; kk++)
        if (p.kst[kk]) row[kk] = u[jj][kk];
    }
  }
}

// All steps of one tile.
template <int ID, typename T, int CK, int CJ, int NW, bool EXACT, int DM, class Pos>
__device__ __forceinline__ void tile2_steps(T (&u)[CJ][CK], T* lds, const Pos& p,
                                            const T (&c)[(Def<ID>::linear ? Def<ID>::ntaps : 1) + 2], int has_div,
                                            double gscale, int D0, int steps, int lane, int w) {
  using D = Def<ID>;
  constexpr int R = D::rad;
  constexpr int NT = D::linear ? D::ntaps : 1;
  constexpr int W = 64 * CK;
  constexpr int ER = edge_rows<CJ, R>();
  constexpr int NB = tile2_bufs<ID, T, CK, CJ, NW>();
  static_assert(CK >= R, "a lane must hold at least R cells");
  const T div = c[NT];
  auto publish = [&](int to) {
    T* o = lds + (size_t)to * (NW * ER * W) + (size_t)w * ER * W + lane * CK;
#pragma unroll
    for (int jj = 0; jj < CJ; jj++) {
      const int e = edge_index<CJ, R>(jj);
      if (e >= 0) store_run<T, CK>(o + e * W, u[jj]);
    }
  };
  publish(0);
#pragma unroll 1
  for (int s = 1; s <= steps; s++) {
    __syncthreads();
    const bool live = s <= p.last;
    T x[CJ + 2 * R][CK + 2 * R];
    if (live) {
      const T* in = lds + (size_t)(NB == 2 ? (s - 1) & 1 : 0) * (NW * ER * W) + lane * CK;
      static_for<0, CJ + 2 * R>([&](auto rc) {
        constexpr int RR = decltype(rc)::value, JR = RR - R;  // row relative to the wave's first
        T v[CK];
        if constexpr (JR >= 0 && JR < CJ) {
#pragma unroll
          for (int kk = 0; kk < CK; kk++) v[kk] = u[JR][kk];
        } else {
          constexpr int WOFF = JR >= 0 ? JR / CJ : -((-JR + CJ - 1) / CJ);
          constexpr int E = edge_index<CJ, R>(JR - WOFF * CJ);
          static_assert(E >= 0, "halo row must be published");
          const int ws = min(max(w + WOFF, 0), NW - 1);
          load_run<T, CK>(v, in + (ws * ER + E) * W);
        }
#pragma unroll
        for (int kk = 0; kk < CK; kk++) x[RR][kk + R] = v[kk];
#pragma unroll
        for (int m = 1; m <= R; m++) {
          x[RR][R - m] = from_left(v[CK - m]);
          x[RR][R + CK - 1 + m] = from_right(v[m - 1]);
        }
      });
    }
    if constexpr (NB == 1) __syncthreads();
    if (live) {
      constexpr bool BATCHDIV = EXACT && D::linear && DM == 2;
      T val[CJ][CK];
      static_for<0, CJ>([&](auto jc) {
        constexpr int JJ = decltype(jc)::value;
        static_for<0, CK>([&](auto kc) {
          constexpr int KK = decltype(kc)::value;
          TileGet<D, T, CJ, CK, JJ, KK> get{x};
          if constexpr (BATCHDIV) val[JJ][KK] = eval_point<D, T, 0>(get, c, div, has_div, gscale);
          else if constexpr (EXACT || !D::linear) val[JJ][KK] = eval_point<D, T, DM>(get, c, div, has_div, gscale);
          else val[JJ][KK] = eval_fast<D, T>(get, c);
        });
      });
      if constexpr (BATCHDIV) {
        const T rc = c[NT + 1];
        T sum[CJ][CK];
        bool ok = true;
#pragma unroll
        for (int jj = 0; jj < CJ; jj++)
#pragma unroll
          for (int kk = 0; kk < CK; kk++) {
            sum[jj][kk] = val[jj][kk];
            val[jj][kk] = div_fast(sum[jj][kk], div, rc);
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
      if (p.wave_in) {
#pragma unroll
        for (int jj = 0; jj < CJ; jj++)
#pragma unroll
          for (int kk = 0; kk < CK; kk++) u[jj][kk] = val[jj][kk];
      } else {
#pragma unroll
        for (int jj = 0; jj < CJ; jj++) {
          const bool rin = p.rw + jj >= R && p.rw + jj < D0 - R;
#pragma unroll
          for (int kk = 0; kk < CK; kk++) u[jj][kk] = rin && p.kin[kk] ? val[jj][kk] : u[jj][kk];
        }
      }
      if (s < steps) publish(NB == 2 ? s & 1 : 0);
    }
  }
}

template <int ID, typename T, int CK, int CJ, int NW, bool EXACT, int DM>
__device__ __forceinline__ void tile2_body(const SweepArgs<T>& a) {
  using D = Def<ID>;
  constexpr int NT = D::linear ? D::ntaps : 1;
  extern __shared__ __align__(16) unsigned char an5d_lds[];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  T c[NT + 2];
#pragma unroll
  for (int q = 0; q < NT + 2; q++) c[q] = a.coef[q];
  const Tile2Pos<CK, CJ, NW> p(D::rad, a.D0, a.D2, a.ntk, a.nseg, a.SJ, a.SK, tile, a.steps, lane, w);
  T u[CJ][CK];
  tile2_load<T, CK, CJ>(u, a.src, a.s0, a.D0, a.D2, a.ntk, a.SJ, a.SK, tile, lane, w);
  tile2_steps<ID, T, CK, CJ, NW, EXACT, DM>(u, reinterpret_cast<T*>(an5d_lds), p, c, a.has_div, a.gscale, a.D0,
                                            a.steps, lane, w);
  tile2_store<T, CK, CJ>(u, p, a.dst, a.s0);
}

template <int ID, typename T, int CK, int CJ, int NW, bool EXACT>
__global__ __launch_bounds__(64 * NW) void tile2_kernel(SweepArgs<T> a) {
  if constexpr (!EXACT || !Def<ID>::linear) {
    tile2_body<ID, T, CK, CJ, NW, EXACT, 0>(a);
  } else if constexpr (Def<ID>::divisor != 0) {
    if (a.has_div == 2) tile2_body<ID, T, CK, CJ, NW, EXACT, 2>(a);
    else if (a.has_div == 0) tile2_body<ID, T, CK, CJ, NW, EXACT, 0>(a);  // no test per cell
    else tile2_body<ID, T, CK, CJ, NW, EXACT, -1>(a);
  } else {
    if (a.has_div == 0) tile2_body<ID, T, CK, CJ, NW, EXACT, 0>(a);
    else tile2_body<ID, T, CK, CJ, NW, EXACT, -1>(a);
  }
}

}  // namespace an5d
