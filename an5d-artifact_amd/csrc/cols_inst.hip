// Instantiates and registers the column kernels of one box x dtype
// (-DAN5D_SID=<stencil id> -DAN5D_F64=<0|1>).
#include "cols.hpp"
#include "cols1.hpp"
#include "cols2.hpp"
#include "launch.hpp"

namespace an5d {
namespace {

using T = std::conditional_t<AN5D_F64, double, float>;
constexpr int SID = AN5D_SID;

template <int CK, bool EXACT>
constexpr auto cols_fn() {
  if constexpr (Def<SID>::dim == 3 && Def<SID>::rad == 1) return &cols1_kernel<SID, T, CK, EXACT>;
  else if constexpr (Def<SID>::dim == 3) return &cols_kernel<SID, T, CK, EXACT>;
  else return &cols2_kernel<SID, T, CK, EXACT>;
}

template <int CK, bool EXACT>
hipError_t launch_cols(const LaunchArgs& a, dim3 grid, dim3 block, size_t, hipStream_t st) {
  constexpr auto kern = cols_fn<CK, EXACT>();
  hipLaunchKernelGGL(kern, grid, block, 0, st, to_args<T>(a));
  return hipGetLastError();
}

template <int CK>
void add_cols(std::vector<Variant>& out) {
  Variant v{};
  v.stencil = SID;
  v.dtype = AN5D_F64 ? kF64 : kF32;
  v.kind = kCols;
  v.ck = CK; v.cj = 1; v.nw = 4; v.btmax = 1;
  v.fn[1] = &launch_cols<CK, true>;
  v.fn_fast[1] = &launch_cols<CK, false>;
  out.push_back(v);
}

}  // namespace

#define AN5D_CAT2(a, b, c) a##b##_##c
#define AN5D_CAT(a, b, c) AN5D_CAT2(a, b, c)
void AN5D_CAT(register_cols_, AN5D_SID, AN5D_F64)(std::vector<Variant>& out) {
  // radius-1 3D: two cells a lane in FP64 (bound by memory: more waves) and for
  // the smaller FP32 grids
  constexpr bool narrow = Def<SID>::dim == 3 && Def<SID>::rad == 1;
  if constexpr (!(narrow && AN5D_F64)) add_cols<4>(out);
  if constexpr (narrow) add_cols<2>(out);
}

}  // namespace an5d
