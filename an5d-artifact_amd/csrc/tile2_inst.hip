// Instantiates and registers the register-tile kernels of one 2D stencil x
// dtype (-DAN5D_SID=<stencil id> -DAN5D_F64=<0|1>).
#include "launch.hpp"
#include "tile2.hpp"

namespace an5d {
namespace {

using T = std::conditional_t<AN5D_F64, double, float>;
constexpr int SID = AN5D_SID;
constexpr int R = Def<SID>::rad;

template <int CK, int CJ, int NW, bool EXACT>
hipError_t launch_tile2(const LaunchArgs& a, dim3 grid, dim3 block, size_t lds, hipStream_t st) {
  constexpr auto kern = &tile2_kernel<SID, T, CK, CJ, NW, EXACT>;
  if (lds > 65536) {
    static std::atomic<int> done[kMaxDevices];
    const hipError_t e = lds_opt_in(reinterpret_cast<const void*>(kern), lds, done);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(kern, grid, block, lds, st, to_args<T>(a));
  return hipGetLastError();
}

template <int CK, int CJ, int NW>
void add_tile2(std::vector<Variant>& out) {
  Variant v{};
  v.stencil = SID;
  v.dtype = AN5D_F64 ? kF64 : kF32;
  v.kind = kTile;
  v.ck = CK; v.cj = CJ; v.nw = NW;
  // at least a quarter of the tile's rows is its own
  v.btmax = NW * CJ * 3 / 8 / R < kMaxBT ? NW * CJ * 3 / 8 / R : kMaxBT;
  for (int bt = 1; bt <= v.btmax; bt++) {
    v.lds[bt] = tile2_bufs<SID, T, CK, CJ, NW>() * tile2_buf_bytes<SID, T, CK, CJ, NW>();
    v.fn[bt] = &launch_tile2<CK, CJ, NW, true>;
    v.fn_fast[bt] = &launch_tile2<CK, CJ, NW, false>;
  }
  out.push_back(v);
}

}  // namespace

#define AN5D_CAT2(a, b, c) a##b##_##c
#define AN5D_CAT(a, b, c) AN5D_CAT2(a, b, c)
void AN5D_CAT(register_tile2_, AN5D_SID, AN5D_F64)(std::vector<Variant>& out) {
  if constexpr (R == 1) {
    add_tile2<1, 2, 16>(out);
    add_tile2<2, 4, 16>(out);
    add_tile2<2, 8, 8>(out);
    if constexpr (!AN5D_F64) {
      add_tile2<2, 8, 16>(out);
      add_tile2<4, 8, 8>(out);
    }
  } else if constexpr (R == 2) {
    add_tile2<2, 2, 16>(out);
    add_tile2<2, 4, 16>(out);
    add_tile2<2, 8, 8>(out);
    if constexpr (!AN5D_F64) {
      add_tile2<2, 8, 16>(out);
      add_tile2<4, 8, 8>(out);
    }
  } else {
    add_tile2<4, 2, 16>(out);
    if constexpr (!AN5D_F64) {
      add_tile2<4, 4, 8>(out);
      add_tile2<4, 4, 16>(out);
    }
  }
}

}  // namespace an5d
