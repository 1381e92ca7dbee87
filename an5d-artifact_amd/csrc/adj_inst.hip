// Instantiates and registers the adjoint kernels of one 2D stencil x dtype
// (-DAN5D_SID=<stencil id> -DAN5D_F64=<0|1>).
#include "adj_tile.hpp"
#include "adjoint.hpp"
#include "engine.hpp"

namespace an5d {
namespace {

using T = std::conditional_t<AN5D_F64, double, float>;
constexpr int SID = AN5D_SID;
using D = Def<SID>;

// cells per lane and deepest block: keeps the kernels within 256 VGPRs (two
// waves per SIMD)
constexpr int adj_ck() {
  if (!D::linear) return 2;
  if (D::rad <= 2 && !AN5D_F64) return 4;
  return D::rad <= 2 ? 2 : 4;  // a lane holds at least R cells
}
constexpr int adj_btmax() {
  if (!D::linear) return 2;
  if (D::rad == 1) return D::ntaps > 5 ? 4 : 5;
  if (D::rad == 2) return AN5D_F64 ? 2 : 3;  // deeper blocks exceed 256 VGPRs
  return 1;
}

AdjArgs<T> to_adj_args(const AdjLaunch& l) {
  AdjArgs<T> a;
  a.U = static_cast<const T*>(l.U);
  a.Lin = static_cast<const T*>(l.Lin);
  a.Lout = static_cast<T*>(l.Lout);
  a.coef = static_cast<const T*>(l.coef);
  a.gscale = l.gscale;
  a.has_div = l.has_div;
  a.gslot = l.gslot;
  a.D0 = l.D0; a.D2 = l.D2; a.s0 = l.s0;
  a.ntk = l.ntk; a.nseg = l.nseg; a.sl = l.sl; a.SK = l.SK;
  return a;
}

template <int BT>
hipError_t launch_adj(const AdjLaunch& l, dim3 grid, dim3 block, hipStream_t st) {
  hipLaunchKernelGGL((adjoint_kernel<SID, T, BT, adj_ck(), 4>), grid, block, 0, st, to_adj_args(l));
  return hipGetLastError();
}

template <int BT>
int occupancy_of() {
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
          &n, reinterpret_cast<const void*>(&adjoint_kernel<SID, T, BT, adj_ck(), 4>), 64 * 4, 0) !=
      hipSuccess)
    return 0;
  return n;
}
int occupancy(int bt) {
  int n = 0;
  static_for<1, adj_btmax() + 1>([&](auto bc) {
    constexpr int BT = decltype(bc)::value;
    if (bt == BT) n = occupancy_of<BT>();
  });
  return n;
}

// Register-tile shapes (adj_tile.hpp), FP64 stencils of up to 25 taps: 16 waves
// of few cells for the smallest grids of radius 1, 8 waves (whose 256 registers
// hold the block's states, and less halo) above.  At radius 2 the 8 waves alone: 16
// of half their cells cover the same tile and are slower (60 steps of 256^2: j2d9pt
// 546 us against 465; the box spills, 3199 against 769); at radius 3-4 the edge
// rows of a larger tile than the first exceed LDS.
template <int I>
constexpr bool adj_tiled() {
  if (!AN5D_F64 || !D::linear || D::ntaps > 25) return false;
  return I == 0 ? D::rad != 2 : D::rad <= 2;
}
template <int I> constexpr int tile_ck() { return D::rad >= 3 ? 4 : (I == 0 && D::rad == 1 ? 1 : 2); }
template <int I> constexpr int tile_cj() { return I == 0 ? 2 : 4; }
template <int I> constexpr int tile_nw() { return I == 1 || D::rad >= 3 ? 8 : 16; }

template <int BT, int I>
hipError_t launch_adj_tile(const AdjLaunch& l, dim3 grid, dim3 block, hipStream_t st) {
  constexpr int CK = tile_ck<I>(), CJ = tile_cj<I>(), NW = tile_nw<I>();
  constexpr size_t lds = adj_tile_lds_bytes<SID, T, CK, CJ, NW>();
  constexpr auto kern = &adjoint_tile_kernel<SID, T, BT, CK, CJ, NW>;
  static_assert(lds <= 160 * 1024, "edge rows exceed LDS");
  if (lds > 65536) {
    static std::atomic<int> done[kMaxDevices];
    const hipError_t e = lds_opt_in(reinterpret_cast<const void*>(kern), lds, done);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(kern, grid, block, lds, st, to_adj_args(l));
  return hipGetLastError();
}

template <int I>
void add_tile(AdjVariant& v) {
  if constexpr (adj_tiled<I>()) {
    v.tile[I].ck = tile_ck<I>();
    v.tile[I].cj = tile_cj<I>();
    v.tile[I].nw = tile_nw<I>();
    static_for<1, adj_btmax() + 1>([&](auto bc) {
      constexpr int BT = decltype(bc)::value;
      v.tile[I].fn[BT] = &launch_adj_tile<BT, I>;
    });
  }
}

hipError_t launch_seed(const void* uT, const void* target, void* lam, double* lslot, int D0, int D2,
                       long long s0, long long stgt, int R, hipStream_t st) {
  hipLaunchKernelGGL((adjoint_seed_kernel<T>), dim3(kSeedBlocks), dim3(256), 0, st, static_cast<const T*>(uT),
                     static_cast<const T*>(target), static_cast<T*>(lam), lslot, D0, D2, s0, stgt, R);
  return hipGetLastError();
}

hipError_t launch_halo(const void* src, void* dst, long long stride, int ndst, int D0, int D2, long long s0, int R,
                       hipStream_t st) {
  const long long cells = (2LL * R * D2 + 2LL * R * (D0 - 2 * R)) * ndst;
  long long blocks = (cells + 255) / 256;
  if (blocks > 1024) blocks = 1024;
  if (blocks < 1) blocks = 1;
  hipLaunchKernelGGL((halo_copy_kernel<T>), dim3((unsigned)blocks), dim3(256), 0, st, static_cast<const T*>(src),
                     static_cast<T*>(dst), stride, ndst, D0, D2, s0, R);
  return hipGetLastError();
}

}  // namespace

#define AN5D_CAT2(a, b, c) a##b##_##c
#define AN5D_CAT(a, b, c) AN5D_CAT2(a, b, c)
void AN5D_CAT(register_adjoint_, AN5D_SID, AN5D_F64)(std::vector<AdjVariant>& out) {
  AdjVariant v{};
  v.stencil = SID;
  v.dtype = AN5D_F64 ? kF64 : kF32;
  v.ck = adj_ck();
  v.nw = 4;
  v.btmax = adj_btmax();
  v.reach = adj_reach<D>();
  v.seed = &launch_seed;
  v.halo = &launch_halo;
  v.occupancy = &occupancy;
  static_for<1, adj_btmax() + 1>([&](auto bc) {
    constexpr int BT = decltype(bc)::value;
    v.fn[BT] = &launch_adj<BT>;
  });
  add_tile<0>(v);
  add_tile<1>(v);
  out.push_back(v);
}

}  // namespace an5d
