// Instantiates and registers the 3D register-tile kernels of one radius-1
// stencil x dtype (-DAN5D_SID=<stencil id> -DAN5D_F64=<0|1>).
#include "launch.hpp"
#include "tile3.hpp"

namespace an5d {
namespace {

using T = std::conditional_t<AN5D_F64, double, float>;
constexpr int SID = AN5D_SID;
constexpr bool BOX = needs_corners<Def<SID>>();

template <int BT, int OP, int CK, int CJ, int NW, bool EXACT>
hipError_t launch_tile3(const LaunchArgs& a, dim3 grid, dim3 block, size_t lds, hipStream_t st) {
  constexpr auto kern = &tile3_kernel<SID, T, BT, OP, CK, CJ, NW, EXACT>;
  if (lds > 65536) {
    static std::atomic<int> done[kMaxDevices];
    const hipError_t e = lds_opt_in(reinterpret_cast<const void*>(kern), lds, done);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(kern, grid, block, lds, st, to_args<T>(a));
  return hipGetLastError();
}

template <int OP, int CK, int CJ, int NW, int BTMAX>
void add_tile3(std::vector<Variant>& out) {
  Variant v{};
  v.stencil = SID;
  v.dtype = AN5D_F64 ? kF64 : kF32;
  v.kind = kTile;
  v.ck = CK; v.cj = CJ; v.nw = NW; v.btmax = BTMAX;
  v.planes = OP;
  static_for<1, BTMAX + 1>([&](auto bc) {
    constexpr int BT = decltype(bc)::value, CI = OP + 2 * BT;
    static_assert(tile3_buf_bytes<T, CI, CJ, CK, NW>() <= 160 * 1024, "edge rows exceed LDS");
    v.lds[BT] = tile3_bufs<T, CI, CJ, CK, NW>() * tile3_buf_bytes<T, CI, CJ, CK, NW>();
    v.fn[BT] = &launch_tile3<BT, OP, CK, CJ, NW, true>;
    v.fn_fast[BT] = &launch_tile3<BT, OP, CK, CJ, NW, false>;
  });
  out.push_back(v);
}

}  // namespace

#define AN5D_CAT2(a, b, c) a##b##_##c
#define AN5D_CAT(a, b, c) AN5D_CAT2(a, b, c)
void AN5D_CAT(register_tile3_, AN5D_SID, AN5D_F64)(std::vector<Variant>& out) {
  add_tile3<8, 1, 4, 8, BOX ? 3 : 4>(out);
  if constexpr (!BOX) {
    add_tile3<4, 1, 4, 8, 4>(out);
    add_tile3<4, 1, 2, 8, 4>(out);
  }
}

}  // namespace an5d
