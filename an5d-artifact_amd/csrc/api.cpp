// C ABI of the engine: registry, launch schedule, device-buffer management
// and the forward entry points.  Host code only; kernels live in the
// per-stencil translation units built from fwd_inst.hip.
#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <time.h>

#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/an5d.h"
#include "engine.hpp"
#include "internal.hpp"
#include "staging.hpp"
#include "stencil_defs.hpp"

namespace an5d {

// ---- errors -----------------------------------------------------------------
static thread_local std::string g_err;

int fail(int code, const std::string& msg) {
  g_err = msg;
  return code;
}

int hip_fail(hipError_t e, const char* what) {
  return fail(AN5D_E_HIP, std::string(what) + ": " + hipGetErrorString(e));
}

// ---- registry -----------------------------------------------------------------
#define AN5D_DECL_REG(id, ident, dim, rad, fpp, n, div, lin) \
  void register_variants_##id##_0(std::vector<Variant>&);     \
  void register_variants_##id##_1(std::vector<Variant>&);
AN5D_STENCILS(AN5D_DECL_REG)
// cols_inst.hip, tile2_inst.hip, tile3_inst.hip: the stencils the Makefile builds them for
#define AN5D_COLS_IDS(X) X(5) X(6) X(7) X(16) X(20) X(17) X(18) X(19)
#define AN5D_TILE_IDS(X) X(0) X(1) X(2) X(3) X(4) X(5) X(8) X(9) X(10) X(11)
#define AN5D_TILE3_IDS(X) X(12) X(16) X(20)
#define AN5D_DECL_TILE3(id)                            \
  void register_tile3_##id##_0(std::vector<Variant>&); \
  void register_tile3_##id##_1(std::vector<Variant>&);
AN5D_TILE3_IDS(AN5D_DECL_TILE3)
#define AN5D_DECL_COLS(id)                            \
  void register_cols_##id##_0(std::vector<Variant>&); \
  void register_cols_##id##_1(std::vector<Variant>&);
#define AN5D_DECL_TILE(id)                             \
  void register_tile2_##id##_0(std::vector<Variant>&); \
  void register_tile2_##id##_1(std::vector<Variant>&);
AN5D_COLS_IDS(AN5D_DECL_COLS)
AN5D_TILE_IDS(AN5D_DECL_TILE)

std::vector<Variant>& registry() {
  static std::vector<Variant> v = [] {
    std::vector<Variant> out;
#define AN5D_CALL_REG(id, ident, dim, rad, fpp, n, div, lin) \
  register_variants_##id##_0(out);                            \
  register_variants_##id##_1(out);
    AN5D_STENCILS(AN5D_CALL_REG)
    // after the others, so the indices of those stay put
#define AN5D_CALL_COLS(id)    \
  register_cols_##id##_0(out); \
  register_cols_##id##_1(out);
#define AN5D_CALL_TILE(id)     \
  register_tile2_##id##_0(out); \
  register_tile2_##id##_1(out);
#define AN5D_CALL_TILE3(id)     \
  register_tile3_##id##_0(out); \
  register_tile3_##id##_1(out);
    AN5D_COLS_IDS(AN5D_CALL_COLS)
    AN5D_TILE_IDS(AN5D_CALL_TILE)
    AN5D_TILE3_IDS(AN5D_CALL_TILE3)
    return out;
  }();
  return v;
}

const std::vector<const Variant*>& variants_of(int stencil, int dtype) {
  // indexed once: a scan of the registry costs more than a kernel launch
  static const std::vector<std::vector<const Variant*>> table = [] {
    std::vector<std::vector<const Variant*>> t(2 * kNumStencils);
    for (const Variant& v : registry()) t[2 * v.stencil + (v.dtype == kF64)].push_back(&v);
    return t;
  }();
  static const std::vector<const Variant*> none;
  if (stencil < 0 || stencil >= kNumStencils || (dtype != kF32 && dtype != kF64)) return none;
  return table[2 * stencil + (dtype == kF64)];
}

const StencilRT& stencil_rt(int id) {
  static const std::vector<StencilRT> table = [] {
    std::vector<StencilRT> t;
#define AN5D_RT(id_, ident, dim_, rad_, fpp_, n_, div_, lin_)                       \
  {                                                                                  \
    StencilRT s;                                                                     \
    s.name = #ident;                                                                 \
    for (char& ch : s.name) if (ch == '_') ch = '-';                                 \
    s.dim = dim_; s.rad = rad_; s.fpp = fpp_; s.ntaps = n_; s.divisor = div_;        \
    s.linear = lin_;                                                                 \
    for (int q = 0; q < n_; q++) s.taps.push_back(Def<id_>::taps[q]);                \
    t.push_back(s);                                                                  \
  }
    AN5D_STENCILS(AN5D_RT)
    return t;
  }();
  return table[id];
}

// ---- geometry ---------------------------------------------------------------
bool make_geom(const an5d_problem* p, Geom& g, std::string& err) {
  if (!p) { err = "null problem"; return false; }
  if (p->stencil < 0 || p->stencil >= kNumStencils) { err = "unknown stencil id"; return false; }
  if (p->dtype != AN5D_FLOAT32 && p->dtype != AN5D_FLOAT64) { err = "bad dtype"; return false; }
  const StencilRT& s = stencil_rt(p->stencil);
  const int nd = s.dim;
  for (int d = 0; d < nd; d++)
    if (p->n[d] < 1) { err = "interior extents must be >= 1"; return false; }
  g.r = s.rad;
  g.dim = nd;
  g.D0 = p->n[0] + 2 * s.rad;
  if (nd == 2) { g.D1 = 1; g.D2 = p->n[1] + 2 * s.rad; }
  else { g.D1 = p->n[1] + 2 * s.rad; g.D2 = p->n[2] + 2 * s.rad; }
  if (g.D0 > (1LL << 30) || g.D1 > (1LL << 30) || g.D2 > (1LL << 30)) {
    err = "extent too large";
    return false;
  }
  g.area = g.D0 * g.D1 * g.D2;
  return true;
}

an5d_layout reference_layout(const Geom& g) {
  an5d_layout L;
  L.s1 = g.D2;
  L.s0 = g.D1 * g.D2;
  L.buf_stride = g.area;
  return L;
}

// ---- launch planning ----------------------------------------------------------
static long long cdiv(long long a, long long b) { return (a + b - 1) / b; }

int device_cus() {
  static std::mutex mu;
  static std::map<int, int> cache;
  int dev = 0, n = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 0;
  std::lock_guard<std::mutex> lk(mu);
  auto it = cache.find(dev);
  if (it != cache.end()) return it->second;
  if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
  cache[dev] = n;
  return n;
}

// Default segment length along dim 0.  The time of a launch is taken as
//   (planes a segment runs) x max(L, waves per SIMD on the busiest CU)
// in units of one wave's time per plane: waves share a SIMD's issue, fewer
// than L of them leave latency exposed, and a segment runs its own planes,
// the 2*bt*R warm-up planes of the sweeps and what fills whole loop bodies.
// L and the warm-up were fitted to the times of every segment length 1 .. 128
// over 256^2 .. 8192^2 and 64^3 .. 384^3 (squares, cubes and ragged
// rectangles, both dtypes).  Against "as many segments as fill the resident
// workgroups in one round, 8*bt*R planes at least": 0.63 of the time in the
// geometric mean over 5280 calls of every 2D sweep, depth and mode at 700^2 ..
// 5000^2 (a 256^2 grid got 16 waves), 6 % of them 3 % or more slower.
int default_sl(const Variant& v, int bt, const Geom& g, long long ntk, long long ntj, int mode) {
  const long long n0 = g.D0 - 2 * g.r;
  const long long cus = device_cus() > 0 ? device_cus() : 256;
  const bool tiles3 = g.dim == 3;     // a segment holds ntk * ntj workgroups, else ntk waves
  const bool cols = v.kind == kCols;  // 3D: ntk workgroups; 2D: ntk runs of a lane
  double lat = 1.5, warm = 2.0 * bt * g.r + 1;
  int body = 1;
  long long longest = n0;
  if (cols) {
    // warm-up planes cost their loads only; longer segments lose the rows that
    // neighbours share in L2 (box3d2r FP64 512^3: 1386 us at 32, 1527 at 128;
    // box2d4r FP32 8192^2: 196 us at 16, 214 at 32)
    lat = 2.4;
    warm = 0.5;
    longest = g.dim == 3 ? 32 : 16;
  } else if (v.kind == kPlane && g.r > 1) {
    lat = 4;  // every plane waits for the tiles of LDS at a barrier
  } else if (v.kind == kSweep && g.r <= 2) {
    body = g.r == 1 && bt * v.cj * v.ck <= 36 ? 6 : 2 * g.r + 1;
  }
  // Grids past the 256 MB last-level cache wait for memory: 2D sweeps want as
  // many waves a SIMD as their registers hold.  Where one round of them has
  // segments of 8*bt*R planes, that round is the choice (the model: 1.02 of its
  // time in the geometric mean over 5600 calls at 4000^2 .. 12000^2, up to 1.43;
  // box2d3r FP64 FMA 12000^2, two steps a launch: 471 us a step in one round,
  // 573 at half its waves), and that length where it has a tenth less (435
  // calls: 0.99 of the model's time; a fifth less, 356 calls: 1.06).  Else the
  // model with L from an estimate of the registers (0.93 of the time of that
  // least length over 1561 calls; the compiler's count in its place, 0.935).
  // And the LDS-staged planes of the 3D stars want no more workgroups than run
  // together, which share their halos in L2 (star3d4r FP32 400x420x390: 193 us
  // with two a CU, 217 with three).
  const bool past_llc = 2 * g.area * (v.dtype == kF64 ? 8 : 4) > (192LL << 20);
  long long most_wgs = 1LL << 60;
  const int occ = v.occ[bt] ? v.occ[bt](mode) : 0;  // workgroups a CU holds (0: not a 2D sweep, or no device)
  if (past_llc && occ > 0) {
    const long long nseg = occ * cus * v.nw / ntk;
    const long long round = cdiv(n0, nseg > 1 ? nseg : 1);
    const long long least = 8LL * bt * g.r < n0 ? 8LL * bt * g.r : n0;
    if (10 * round >= 9 * least) return (int)(round > least ? round : least);
  }
  if (past_llc && !tiles3 && v.kind == kSweep) {
    const int w = v.dtype == kF64 ? 2 : 1;
    const bool box = stencil_rt(v.stencil).ntaps > 4 * g.r + 1;
    int regs = bt * (2 * g.r + 1) * v.ck * w + 28 + 5 * w * g.r + (w == 2 ? 4 : 0) + (box ? 5 * g.r * g.r * w : 0);
    if (v.regcap > 0 && regs > v.regcap) regs = v.regcap;
    lat = 512 / ((regs + 7) / 8 * 8);
    lat = lat < 1 ? 1 : (lat > 5 ? 5 : lat);
  }
  // a kernel that holds one wave a SIMD gains nothing from a second (box2d4r FP32
  // 5000^2, three steps: 187 us a step in one round, 222 in two)
  if (occ > 0 && occ * v.nw <= 4) lat = 1;
  if (past_llc && v.kind == kPlane && g.r > 1) most_wgs = 2 * cus;
  double best_t = 1e300;
  long long best = n0 < longest ? n0 : longest;
  // every count up to 64, then steps of a sixteenth
  for (long long nseg = cdiv(n0, longest); nseg <= n0; nseg += 1 + (nseg >= 64 ? nseg / 16 : 0)) {
    const long long sl = cdiv(n0, nseg);
    const long long waves = cols && !tiles3 ? cdiv(ntk * nseg, 64) : ntk * nseg;
    const long long wgs = tiles3 ? ntk * ntj * nseg : cdiv(waves, v.nw);
    if (wgs > most_wgs && nseg > cdiv(n0, longest)) break;
    const double share = (double)cdiv(wgs, cus) * v.nw / 4;
    const double planes = body > 1 ? (double)cdiv(sl + (long long)warm, body) * body : sl + warm;
    const double t = planes * (share > lat ? share : lat);
    if (t < best_t) {
      best_t = t;
      best = sl;
    }
    if (share > 8 * lat) break;  // more segments only add warm-up
  }
  return (int)(best < 1 ? 1 : best);
}

bool plan_launch(const Variant& v, int bt, const Geom& g, int sl, LaunchPlan& lp,
                 std::string& err, int mode) {
  const int R = g.r;
  const long long n0 = g.D0 - 2 * R, nj = g.D1 - (g.dim == 3 ? 2 * R : 0), nk = g.D2 - 2 * R;
  LaunchArgs& a = lp.args;
  a.D0 = (int)g.D0; a.D1 = (int)g.D1; a.D2 = (int)g.D2;
  lp.fn = nullptr;
  if (bt >= 1 && bt <= v.btmax)
    lp.fn = mode == AN5D_FAST ? v.fn_fast[bt] : (mode == kLaunchShare ? v.fn_share[bt] : v.fn[bt]);
  if (!lp.fn) { err = "no kernel for bt=" + std::to_string(bt) + " in this variant"; return false; }
  lp.lds = (bt >= 1 && bt <= kMaxBT) ? v.lds[bt] : 0;
  a.steps = bt;
  if (v.kind == kDirect) {
    const long long total = cdiv(nk, v.ck) * nj * n0;
    lp.block = dim3(256);
    lp.grid = dim3((unsigned)cdiv(total, 256));
    a.ntk = a.ntj = a.nseg = a.sl = a.SK = a.SJ = 0;
    if (cdiv(total, 256) >= (1LL << 31)) { err = "grid too large"; return false; }
    return true;
  }
  if (v.kind == kCols) {
    if (nk < v.ck) { err = "rows shorter than a lane's run"; return false; }
    if (g.dim == 2) {
      // lanes of ck cells over the segments, row-major
      const long long ntk = cdiv(nk, v.ck);
      if (sl <= 0) sl = default_sl(v, bt, g, ntk, 1, mode);
      if (sl > n0) sl = (int)n0;
      const long long nseg = cdiv(n0, sl);
      if (ntk * nseg >= (1LL << 30)) { err = "grid too large"; return false; }
      a.ntk = (int)ntk; a.ntj = 1; a.nseg = (int)nseg; a.sl = sl;
      a.SK = v.ck; a.SJ = 1;
      lp.block = dim3(256);
      lp.grid = dim3((unsigned)cdiv(ntk * nseg, 256));
      return true;
    }
    // lanes of ck cells over the plane, row-major, in blocks of 256 per segment
    const long long ntk = cdiv(nk, v.ck), nblk = cdiv(ntk * nj, 256);
    if (ntk * nj >= (1LL << 30)) { err = "grid too large"; return false; }
    if (sl <= 0) sl = default_sl(v, bt, g, nblk, 1, mode);
    const long long nseg = cdiv(n0, sl);
    a.ntk = (int)ntk; a.ntj = (int)nblk; a.nseg = (int)nseg; a.sl = sl;
    a.SK = v.ck; a.SJ = 1;
    lp.block = dim3(256);
    if (nblk * nseg >= (1LL << 31)) { err = "grid too large"; return false; }
    lp.grid = dim3((unsigned)(nblk * nseg));
    return true;
  }
  if (v.kind == kTile) {
    // tiles of nw*cj rows x 64*ck cells that give up bt*R cells on every side
    // but the grid's own edges
    const long long TH = (long long)v.nw * v.cj, TW = 64LL * v.ck, H = (long long)bt * R;
    if (TH <= 2 * H || TW <= 2 * H) { err = "bt too deep for this variant's tile"; return false; }
    if (g.dim == 3) {
      const long long nti = cdiv(n0, v.planes);
      const long long ntj = g.D1 > TH ? cdiv(g.D1 - 2 * H, TH - 2 * H) : 1;
      const long long ntk = g.D2 > TW ? cdiv(g.D2 - 2 * H, TW - 2 * H) : 1;
      if (nti * ntj >= (1LL << 31) || nti * ntj * ntk >= (1LL << 31)) { err = "grid too large"; return false; }
      a.ntk = (int)ntk; a.ntj = (int)ntj; a.nseg = (int)nti; a.sl = v.planes;
      a.SK = (int)(TW - 2 * H); a.SJ = (int)(TH - 2 * H);
      lp.block = dim3(64 * v.nw);
      lp.grid = dim3((unsigned)(nti * ntj * ntk));
      return true;
    }
    const long long nti = g.D0 > TH ? cdiv(g.D0 - 2 * H, TH - 2 * H) : 1;
    const long long ntk = g.D2 > TW ? cdiv(g.D2 - 2 * H, TW - 2 * H) : 1;
    if (nti * ntk >= (1LL << 31)) { err = "grid too large"; return false; }
    a.ntk = (int)ntk; a.ntj = 1; a.nseg = (int)nti; a.sl = (int)(TH - 2 * H);
    a.SK = (int)(TW - 2 * H); a.SJ = (int)(TH - 2 * H);
    lp.block = dim3(64 * v.nw);
    lp.grid = dim3((unsigned)(nti * ntk));
    return true;
  }
  if (v.kind == kPlane) {
    // tiles of nw*cj rows x 64*ck cells, halos staged, nothing recomputed
    if (g.dim != 3) { err = "the plane kernel is 3D only"; return false; }
    const long long TK = 64LL * v.ck, TJ = (long long)v.nw * v.cj;
    const long long ntk = cdiv(nk, TK), ntj = cdiv(nj, TJ);
    if (sl <= 0) sl = default_sl(v, bt, g, ntk, ntj, mode);
    const long long nseg = cdiv(n0, sl);
    a.ntk = (int)ntk; a.ntj = (int)ntj; a.nseg = (int)nseg; a.sl = sl;
    a.SK = (int)TK; a.SJ = (int)TJ;
    lp.block = dim3(64 * v.nw);
    const long long blocks = ntk * ntj * nseg;
    if (blocks >= (1LL << 31)) { err = "grid too large"; return false; }
    lp.grid = dim3((unsigned)blocks);
    return true;
  }
  // the sweep kernels address a plane (3D) or a row (2D) with 32-bit byte
  // offsets from a per-plane base
  const long long elem = v.dtype == kF64 ? 8 : 4;
  if ((g.dim == 3 ? g.D1 * g.D2 : g.D2) * elem >= (1LL << 31)) {
    err = "plane of 2 GiB or more: the register-streamed kernels address planes with 32-bit offsets";
    return false;
  }
  // the row partial-sum kernels read their tile edges themselves: no overlap
  const long long SK = v.kind == kRows ? 64LL * v.ck : 64LL * v.ck - 2LL * bt * R;
  if (SK <= 0) { err = "bt too deep for this variant's tile width"; return false; }
  const long long ntk = cdiv(nk, SK);
  long long SJ = 1, ntj = 1;
  if (g.dim == 3) {
    SJ = (long long)v.nw * v.cj - 2LL * bt * R;
    if (SJ <= 0) { err = "bt too deep for this variant's tile height"; return false; }
    ntj = cdiv(nj, SJ);
  }
  if (sl <= 0) sl = default_sl(v, bt, g, ntk, ntj, mode);
  const long long nseg = cdiv(n0, sl);
  a.ntk = (int)ntk; a.ntj = (int)ntj; a.nseg = (int)nseg; a.sl = sl;
  a.SK = (int)SK; a.SJ = (int)SJ;
  lp.block = dim3(64 * v.nw);
  long long blocks = (g.dim == 3) ? ntk * ntj * nseg : cdiv(ntk * nseg, v.nw);
  if (blocks >= (1LL << 31)) { err = "grid too large"; return false; }
  lp.grid = dim3((unsigned)blocks);
  return true;
}

// ---- coefficient buffers -------------------------------------------------------
// Host image of the kernel's coefficient array: ntaps values (T), the
// divisor and RN(1/divisor); for gradient2d {eps, 0, 0}.  has_div: 0 none,
// 1 IEEE division, 2 the corrected reciprocal product (only for the source
// divisors 118 and 159, for which it was checked against IEEE division).
bool build_coefs(const an5d_problem* p, std::vector<unsigned char>& bytes, int& has_div,
                 double& gscale, std::string& err, int mode) {
  const StencilRT& s = stencil_rt(p->stencil);
  const bool f64 = p->dtype == AN5D_FLOAT64;
  const int nt = s.linear ? s.ntaps : 1;
  std::vector<double> vals(nt + 2, 0.0);
  gscale = 1.0;
  has_div = 0;
  if (s.linear) {
    for (int q = 0; q < s.ntaps; q++)
      vals[q] = p->coefs ? p->coefs[q] : (double)s.taps[q].coef;
    double d = 0.0;
    if (p->divisor < 0) d = s.divisor;
    else if (p->divisor > 0) d = p->divisor;
    if (d != 0.0) {
      if (!(d == d) || d == INFINITY) { err = "divisor must be finite"; return false; }
      has_div = (d == 118.0 || d == 159.0) ? 2 : 1;
      vals[nt] = d;
    }
  } else {
    vals[0] = p->coefs ? p->coefs[0] : (double)0.0001f;
    gscale = p->coefs ? p->coefs[1] : 1.0;
    if (!(gscale == gscale)) { err = "scale is NaN"; return false; }
  }
  if (mode == AN5D_FAST && s.linear) {
    // fold signs and the divisor into the coefficients: sum_q fma(c'_q, v_q, .)
    const double d = has_div ? vals[nt] : 1.0;
    for (int q = 0; q < s.ntaps; q++) vals[q] = (s.taps[q].sign > 0 ? vals[q] : -vals[q]) / d;
    has_div = 0;
    vals[nt] = 0.0;
  }
  const size_t esz = f64 ? 8 : 4;
  bytes.resize((nt + 2) * esz);
  for (int q = 0; q <= nt; q++) {
    if (f64) {
      double v = vals[q];
      memcpy(&bytes[q * 8], &v, 8);
    } else {
      float v = (float)vals[q];
      memcpy(&bytes[q * 4], &v, 4);
    }
  }
  if (f64) {
    double rc = has_div ? 1.0 / vals[nt] : 0.0;
    memcpy(&bytes[(nt + 1) * 8], &rc, 8);
  } else {
    float rc = has_div ? 1.0f / (float)vals[nt] : 0.0f;
    memcpy(&bytes[(nt + 1) * 4], &rc, 4);
  }
  return true;
}

// The column kernel's order of the table build_coefs made: the centre taps by
// plane, then for every row d1 the (2r+1) x (2r+1) block [plane d0][d2] (the
// centre's place is there and not read), then the divisor and its reciprocal
// as before.  The taps' signs go into the values (a - c*v == a + (-c)*v); the
// fast mode's table has them already.
void cols_coefs(const an5d_problem* p, std::vector<unsigned char>& bytes, int mode) {
  const StencilRT& s = stencil_rt(p->stencil);
  const size_t esz = p->dtype == AN5D_FLOAT64 ? 8 : 4;
  const int r = s.rad, w = 2 * r + 1;
  std::vector<unsigned char> out((size_t)(w + w * w * w + 2) * esz, 0);
  for (int q = 0; q < s.ntaps; q++) {
    const TapDef& t = s.taps[q];
    const int slot = t.d1 == 0 && t.d2 == 0 ? t.d0 + r : w + ((t.d1 + r) * w + t.d0 + r) * w + t.d2 + r;
    memcpy(&out[slot * esz], &bytes[q * esz], esz);
    if (t.sign < 0 && mode != AN5D_FAST) out[slot * esz + esz - 1] ^= 0x80;  // little-endian sign bit
  }
  memcpy(&out[out.size() - 2 * esz], &bytes[s.ntaps * esz], 2 * esz);
  bytes.swap(out);
}

// The shared-product form applies when the stencil is a radius-1 star (a
// centre and its 2*dim face taps) and the coefficient table gives every face
// tap the same value in the working precision (bit for bit: each product
// c * u is then one rounded value, whichever sum it enters).
bool coefs_shareable(const an5d_problem* p, const std::vector<unsigned char>& bytes) {
  const StencilRT& s = stencil_rt(p->stencil);
  if (!s.linear || s.rad != 1 || s.ntaps != 2 * s.dim + 1) return false;
  int centre = -1;
  for (int q = 0; q < s.ntaps; q++) {
    const TapDef& t = s.taps[q];
    if (t.d1 != 0 && t.d2 != 0) return false;
    if (t.d0 == 0 && t.d1 == 0 && t.d2 == 0) centre = q;
  }
  if (centre < 0) return false;
  const size_t esz = p->dtype == AN5D_FLOAT64 ? 8 : 4;
  const int ref = centre == 0 ? 1 : 0;
  for (int q = 0; q < s.ntaps; q++)
    if (q != centre && memcmp(&bytes[q * esz], &bytes[ref * esz], esz) != 0) return false;
  return true;
}

struct DeviceCache {
  std::mutex mu;
  std::map<std::pair<int, std::string>, void*> coefs;  // (device, bytes) -> device copy
  std::map<int, std::pair<void*, size_t>> grids;       // device -> staging grid buffer
  std::map<int, Staging> stagings;                     // device -> pinned ring of its transfers
  std::map<int, std::mutex> grid_users;                // device -> holder of its staging grid and ring
};
static DeviceCache& cache() {
  static DeviceCache* c = new DeviceCache();
  return *c;
}

int device_coefs(const std::vector<unsigned char>& bytes, const void** out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return hip_fail(e, "hipGetDevice");
  DeviceCache& c = cache();
  std::lock_guard<std::mutex> lk(c.mu);
  std::string key(bytes.begin(), bytes.end());
  auto it = c.coefs.find({dev, key});
  if (it != c.coefs.end()) {
    *out = it->second;
    return AN5D_OK;
  }
  void* d = nullptr;
  e = hipMalloc(&d, bytes.size());
  if (e != hipSuccess) return hip_fail(e, "hipMalloc(coefficients)");
  e = hipMemcpy(d, bytes.data(), bytes.size(), hipMemcpyHostToDevice);
  if (e != hipSuccess) { (void)hipFree(d); return hip_fail(e, "hipMemcpy(coefficients)"); }
  c.coefs[{dev, key}] = d;
  *out = d;
  return AN5D_OK;
}

int device_grid(size_t bytes, void** out, Staging** ring, std::unique_lock<std::mutex>& hold) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return hip_fail(e, "hipGetDevice");
  DeviceCache& c = cache();
  std::mutex* user;
  {
    std::lock_guard<std::mutex> lk(c.mu);
    user = &c.grid_users[dev];  // map nodes stay put
  }
  // one host call at a time uses (and may regrow) a device's staging grid
  hold = std::unique_lock<std::mutex>(*user);
  std::lock_guard<std::mutex> lk(c.mu);
  auto& slot = c.grids[dev];
  if (slot.second < bytes) {
    if (slot.first) (void)hipFree(slot.first);
    slot = {nullptr, 0};
    void* d = nullptr;
    e = hipMalloc(&d, bytes);
    if (e != hipSuccess) return fail(AN5D_E_ALLOC, std::string("hipMalloc(grid): ") + hipGetErrorString(e));
    slot = {d, bytes};
  }
  *out = slot.first;
  *ring = &c.stagings[dev];  // map nodes stay put
  return staging_init(**ring);
}

// ---- variant / bt resolution ---------------------------------------------------
int default_bt(const StencilRT& s, int dtype) {
  if (s.dim == 2) return s.rad == 1 ? 4 : 2;
  return s.rad == 1 ? 2 : 1;
}

// Time per step of a 2D register-tile launch, in microseconds: a launch's own
// time, and per step and for the loads and stores (3 steps) the tiles of the
// busiest CU one after the other at the rate of the vector units.
static double tile_step_us(const StencilRT& s, const Variant& v, int bt, const Geom& g, int mode, int cus) {
  const long long TH = (long long)v.nw * v.cj, TW = 64LL * v.ck, H = (long long)bt * g.r;
  if (TH <= 2 * H || TW <= 2 * H) return 1e300;
  const long long nti = g.D0 > TH ? cdiv(g.D0 - 2 * H, TH - 2 * H) : 1;
  const long long ntk = g.D2 > TW ? cdiv(g.D2 - 2 * H, TW - 2 * H) : 1;
  const double ops = s.linear ? (mode == AN5D_FAST ? s.ntaps : s.fpp) : 2 * s.fpp;
  const double tile_us = 4e-6 * (ops + 4) * (v.dtype == kF64 ? 2 : 1) * TH * TW;
  return (2 + (bt + 3) * tile_us * cdiv(nti * ntk, cus)) / bt;
}

// A 2D register tile chosen by a table row of another size: which shape and
// depth fit depends on how many tiles of them the busiest CU gets, so the row
// stands only if no other is 10 % faster by the estimate above.  Its constants
// were fitted to every shape and depth on 14 grids (245x315 .. 2273x2923, six of
// them 4:1) of five stencils in both dtypes and FMA mode: the rows alone are 8.7
// % off the best in the geometric mean (74 % at 1000x3001), with the rule 2.5 %;
// without the 10 % 2.2 %, but more grids get slower.
static void fit_tile(const an5d_problem* p, int mode, const std::vector<const Variant*>& vs, const Variant** v,
                     int* bt) {
  Geom g;
  std::string err;
  if (!make_geom(p, g, err) || g.dim != 2) return;
  // larger grids are bound by memory, which the estimate leaves out (j2d5pt FP32
  // 2600x10400: 23.5 us at its choice, 20.0 on streams)
  if (2 * g.area * (p->dtype == AN5D_FLOAT64 ? 8 : 4) > (128LL << 20)) return;
  const StencilRT& s = stencil_rt(p->stencil);
  const int cus = device_cus() > 0 ? device_cus() : 256;
  double best = 0.9 * tile_step_us(s, **v, *bt, g, mode, cus);
  for (const Variant* x : vs) {
    if (x->kind != kTile) continue;
    for (int k = 1; k <= x->btmax; k++) {
      const double t = tile_step_us(s, *x, k, g, mode, cus);
      if (t < best) {
        best = t;
        *v = x;
        *bt = k;
      }
    }
  }
}

// A caller's depth beyond the one that a table row was measured at.  A kernel
// held to fewer registers spills there: its uncapped twin (star2d3r FP64
// 3500x3500, six steps: 9.8 times faster, star2d4r FP64 FMA, four: 5.4 times).  A
// 2D register tile that gives up too much of itself: the stencil's sweep.  Of
// the tiles that keep less than 0.3 more than half are slower than it, up to 1.8
// times; between 0.3 and 0.5 so are those past 128 MB (1.07 of its time in the
// geometric mean of 20 calls; star2d2r FP64 5000^2, eight steps, 1.23), those
// below take 0.71 of it.
static const Variant* deeper_variant(const an5d_problem* p, const std::vector<const Variant*>& vs, const Variant* v,
                                     int bt) {
  Geom g;
  std::string err;
  if (!make_geom(p, g, err)) return v;
  if (v->kind == kSweep && v->regcap > 0) {
    for (const Variant* x : vs)
      if (x->kind == kSweep && x->regcap == 0 && x->ck == v->ck && x->cj == v->cj && x->nw == v->nw) return x;
  }
  if (v->kind == kTile && g.dim == 2 && vs[0]->kind == kSweep && vs[0]->btmax >= bt) {
    const double TH = (double)v->nw * v->cj, TW = 64.0 * v->ck, H = (double)bt * g.r;
    const double kept = TH > 2 * H && TW > 2 * H ? (1 - 2 * H / TH) * (1 - 2 * H / TW) : 0;
    const bool large = 2 * g.area * (p->dtype == AN5D_FLOAT64 ? 8 : 4) > (128LL << 20);
    if (kept < (large ? 0.5 : 0.3)) return vs[0];
  }
  return v;
}

int resolve(const an5d_problem* p, const an5d_config* cfg, const Variant** vout, int* btout,
            int* slout, bool row_shape) {
  const auto& vs = variants_of(p->stencil, p->dtype);
  if (vs.empty()) return fail(AN5D_E_UNSUPPORTED, "no kernels compiled for this stencil/dtype");
  const StencilRT& s = stencil_rt(p->stencil);
  int want_bt = cfg ? cfg->bt : 0;
  int want_v = cfg ? cfg->variant : -1;
  int sl = cfg ? cfg->sl : 0;
  const int mode = cfg ? cfg->mode : AN5D_EXACT;
  if (want_v >= (int)vs.size()) return fail(AN5D_E_INVALID, "variant index out of range");
  if (want_bt < 0 || want_bt > kMaxBT) return fail(AN5D_E_INVALID, "bt out of range");
  const Variant* v = nullptr;
  if (want_v >= 0) {
    v = vs[want_v];
  } else {
    TunedChoice tc;
    if (tuned_lookup(p, mode, &tc) && tc.variant < (int)vs.size() &&
        (want_bt == 0 || want_bt <= vs[tc.variant]->btmax)) {
      v = vs[tc.variant];
      if (want_bt == 0) {
        want_bt = tc.bt;
        if (!tc.same_size && !row_shape && v->kind == kTile) fit_tile(p, mode, vs, &v, &want_bt);
      } else if (want_bt > tc.bt) {
        v = deeper_variant(p, vs, v, want_bt);
      }
      if (sl == 0 && v == vs[tc.variant]) sl = tc.sl;
    } else {
      v = vs[0];  // first sweep shape, or the direct kernel when none exists
    }
  }
  // a table row of a like size may not fit this grid's extents
  if (want_v < 0 && v->kind == kCols) {
    Geom g;
    LaunchPlan lp;
    std::string err;
    if (!make_geom(p, g, err) || !plan_launch(*v, 1, g, sl, lp, err, mode)) {
      v = vs[0];
      sl = cfg ? cfg->sl : 0;
    }
  }
  int bt = want_bt ? want_bt : default_bt(s, p->dtype);
  if (bt > v->btmax) {
    if (want_bt && cfg && cfg->bt) return fail(AN5D_E_UNSUPPORTED, "bt=" + std::to_string(bt) + " exceeds the variant's btmax=" + std::to_string(v->btmax));
    bt = v->btmax;
  }
  *vout = v;
  *btout = bt;
  *slout = sl;
  return AN5D_OK;
}

}  // namespace an5d

using namespace an5d;

extern "C" int an5d_resolve_config(const an5d_problem* p, const an5d_config* cfg,
                                   an5d_config* out) {
  if (!p || !out) return fail(AN5D_E_INVALID, "null argument");
  Geom g;
  std::string err;
  if (!make_geom(p, g, err)) return fail(AN5D_E_INVALID, err);
  const Variant* v = nullptr;
  int bt = 0, sl = 0;
  const int mode = cfg ? cfg->mode : AN5D_EXACT;
  an5d_config rcfg = cfg ? *cfg : an5d_config{0, -1, 0, AN5D_EXACT};
  if (mode == AN5D_EXACT_GENERAL) rcfg.mode = AN5D_EXACT;  // tiled like exact mode
  int rc = resolve(p, &rcfg, &v, &bt, &sl);
  if (rc) return rc;
  LaunchPlan lp;
  if (!plan_launch(*v, bt, g, sl, lp, err, rcfg.mode)) return fail(AN5D_E_UNSUPPORTED, err);
  const auto& vs = variants_of(p->stencil, p->dtype);
  int vi = 0;
  while (vi < (int)vs.size() && vs[vi] != v) vi++;
  *out = an5d_config{bt, vi, v->kind == kDirect ? 0 : lp.args.sl, mode};
  return AN5D_OK;
}

// ---- schedule -------------------------------------------------------------------
extern "C" int an5d_schedule(int T, int bt, int* steps, int max_launches) {
  if (T < 0 || bt < 1) return fail(AN5D_E_INVALID, "schedule needs T >= 0 and bt >= 1");
  std::vector<int> out;
  const int full = T / bt, r = T % bt;
  const int nat = (T + bt - 1) / bt;  // launches of the plain split
  const bool mismatch = (T % 2) != (nat % 2);
  int main_count = full;
  if (mismatch && r < 2) main_count -= 1;  // __c0Padr (host.cu:72)
  for (int c = 0; c < main_count; c++) out.push_back(bt);
  if (mismatch) {
    if (r == 0) {
      out.push_back((bt + 1) / 2);
      out.push_back(bt / 2);
    } else if (r == 1) {
      const int b = (bt + 1) / 3;
      out.push_back(bt + 1 - 2 * b);
      out.push_back(b);
      out.push_back(b);
    } else {
      out.push_back((r + 1) / 2);
      out.push_back(r / 2);
    }
  } else if (r) {
    out.push_back(r);
  }
  if (steps) {
    if ((int)out.size() > max_launches) return fail(AN5D_E_INVALID, "steps[] too small");
    for (size_t c = 0; c < out.size(); c++) steps[c] = out[c];
  }
  return (int)out.size();
}

// ---- registry queries ---------------------------------------------------------
extern "C" int an5d_stencil_count(void) { return kNumStencils; }

extern "C" int an5d_stencil_id(const char* name) {
  if (!name) return fail(AN5D_E_INVALID, "null name");
  for (int i = 0; i < kNumStencils; i++)
    if (stencil_rt(i).name == name) return i;
  return fail(AN5D_E_INVALID, std::string("unknown stencil: ") + name);
}

extern "C" int an5d_stencil_get_info(int id, an5d_stencil_info* out) {
  if (id < 0 || id >= kNumStencils || !out) return fail(AN5D_E_INVALID, "bad stencil id");
  const StencilRT& s = stencil_rt(id);
  memset(out, 0, sizeof(*out));
  snprintf(out->name, sizeof(out->name), "%s", s.name.c_str());
  out->dim = s.dim; out->rad = s.rad; out->fpp = s.fpp; out->ntaps = s.ntaps;
  out->divisor = s.divisor; out->linear = s.linear;
  return AN5D_OK;
}

extern "C" int an5d_stencil_taps(int id, int* offsets, double* coefs, int max_taps) {
  if (id < 0 || id >= kNumStencils) return fail(AN5D_E_INVALID, "bad stencil id");
  const StencilRT& s = stencil_rt(id);
  if (max_taps < s.ntaps) return fail(AN5D_E_INVALID, "buffer too small");
  for (int q = 0; q < s.ntaps; q++) {
    if (offsets) {
      offsets[4 * q] = s.taps[q].sign;
      offsets[4 * q + 1] = s.taps[q].d0;
      offsets[4 * q + 2] = s.taps[q].d1;
      offsets[4 * q + 3] = s.taps[q].d2;
    }
    if (coefs) coefs[q] = s.taps[q].coef;
  }
  return s.ntaps;
}

extern "C" int an5d_variant_count(int stencil, int dtype) {
  if (stencil < 0 || stencil >= kNumStencils) return fail(AN5D_E_INVALID, "bad stencil id");
  return (int)variants_of(stencil, dtype).size();
}

extern "C" int an5d_variant_get_info(int stencil, int dtype, int variant, an5d_variant_info* out) {
  const auto& vs = variants_of(stencil, dtype);
  if (variant < 0 || variant >= (int)vs.size() || !out) return fail(AN5D_E_INVALID, "bad variant");
  const Variant* v = vs[variant];
  out->kind = v->kind; out->ck = v->ck; out->cj = v->cj; out->nw = v->nw;
  out->btmax = v->btmax; out->lds_bytes = (long long)v->lds[v->btmax];
  out->regcap = v->regcap;
  return AN5D_OK;
}

// ---- forward ------------------------------------------------------------------------
namespace an5d {

int run_schedule(const an5d_problem* p, void* dA, const an5d_layout* layout,
                 const an5d_config* cfg, int steps_only, int c0_first, hipStream_t st, int* launches) {
  Geom g;
  std::string err;
  if (!make_geom(p, g, err)) return fail(AN5D_E_INVALID, err);
  if (!dA) return fail(AN5D_E_INVALID, "null device pointer");
  an5d_layout L = layout ? *layout : reference_layout(g);
  if (L.s1 < g.D2 || (g.dim == 3 && L.s0 < g.D1 * L.s1) || (g.dim == 2 && L.s0 < g.D2) ||
      L.buf_stride < g.D0 * L.s0)
    return fail(AN5D_E_INVALID, "layout strides smaller than the grid");
  const int mode = cfg ? cfg->mode : AN5D_EXACT;
  if (mode != AN5D_EXACT && mode != AN5D_FAST && mode != AN5D_EXACT_GENERAL)
    return fail(AN5D_E_INVALID, "bad mode");
  // AN5D_EXACT_GENERAL tiles like AN5D_EXACT (same table entries)
  an5d_config rcfg = cfg ? *cfg : an5d_config{0, -1, 0, AN5D_EXACT};
  if (mode == AN5D_EXACT_GENERAL) rcfg.mode = AN5D_EXACT;
  const Variant* v = nullptr;
  int bt = 0, sl = 0;
  int rc = resolve(p, &rcfg, &v, &bt, &sl);
  if (rc) return rc;
  std::vector<unsigned char> cbytes;
  int has_div = 0;
  double gscale = 1.0;
  if (!build_coefs(p, cbytes, has_div, gscale, err, rcfg.mode)) return fail(AN5D_E_INVALID, err);
  // launch mode per step count: the shared-product form where it applies
  // (bitwise the same) and its kernel does not spill
  const bool share = mode == AN5D_EXACT && v->kind == kSweep && coefs_shareable(p, cbytes);
  auto launch_mode = [&](int k) {
    if (share && v->fn_share[k] && v->share_scratch[k] && v->share_scratch[k]() == 0) return kLaunchShare;
    return rcfg.mode;
  };
  if (v->kind == kCols && g.dim == 3 && g.r > 1) cols_coefs(p, cbytes, rcfg.mode);
  const void* dcoef = nullptr;
  rc = device_coefs(cbytes, &dcoef);
  if (rc) return rc;
  const size_t esz = p->dtype == AN5D_FLOAT64 ? 8 : 4;
  std::vector<int> steps;
  if (steps_only > 0) {
    steps.push_back(steps_only);
  } else {
    int n = an5d_schedule(p->timesteps, v->kind == kDirect ? 1 : bt, nullptr, 0);
    if (n < 0) return n;
    steps.resize(n);
    an5d_schedule(p->timesteps, v->kind == kDirect ? 1 : bt, steps.data(), n);
  }
  if (launches) *launches = (int)steps.size();
  int c0 = c0_first;
  // one plan per distinct step count (a schedule has at most three)
  LaunchPlan plans[kMaxBT + 1];
  bool planned[kMaxBT + 1] = {};
  for (int k : steps) {
    if (k < 1 || k > kMaxBT) return fail(AN5D_E_INVALID, "bad step count");
    if (!planned[k]) {
      if (!plan_launch(*v, k, g, sl, plans[k], err, launch_mode(k))) return fail(AN5D_E_UNSUPPORTED, err);
      planned[k] = true;
    }
    LaunchPlan lp = plans[k];
    char* base = static_cast<char*>(dA);
    lp.args.src = base + (size_t)(c0 % 2) * L.buf_stride * esz;
    lp.args.dst = base + (size_t)((c0 + 1) % 2) * L.buf_stride * esz;
    lp.args.coef = dcoef;
    lp.args.gscale = gscale;
    lp.args.has_div = has_div;
    lp.args.s0 = L.s0;
    lp.args.s1 = L.s1;
    lp.args.nt_store = (size_t)2 * L.buf_stride * esz > kStreamBytes;
    hipError_t e = lp.fn(lp.args, lp.grid, lp.block, lp.lds, st);
    if (e != hipSuccess) return hip_fail(e, "kernel launch");
    c0++;
  }
  return AN5D_OK;
}

double sb_time_ms() {
  struct timespec tp;
  clock_gettime(CLOCK_MONOTONIC_RAW, &tp);
  return (tp.tv_sec + tp.tv_nsec * 1.0e-9) * 1.0e3;
}

}  // namespace an5d

extern "C" int an5d_forward_device(const an5d_problem* p, void* dA, const an5d_layout* layout,
                                   const an5d_config* cfg, void* stream) {
  if (!p) return fail(AN5D_E_INVALID, "null problem");
  if (p->timesteps < 0) return fail(AN5D_E_INVALID, "timesteps must be >= 0");
  if (p->timesteps == 0) return AN5D_OK;
  return run_schedule(p, dA, layout, cfg, 0, 0, static_cast<hipStream_t>(stream));
}

extern "C" int an5d_launch(const an5d_problem* p, void* dA, const an5d_layout* layout,
                           const an5d_config* cfg, int steps, int c0, void* stream) {
  if (steps < 1 || c0 < 0) return fail(AN5D_E_INVALID, "steps must be >= 1 and c0 >= 0");
  return run_schedule(p, dA, layout, cfg, steps, c0, static_cast<hipStream_t>(stream));
}

extern "C" int an5d_forward_host(const an5d_problem* p, void* A, const an5d_config* cfg,
                                 double* ms) {
  Geom g;
  std::string err;
  if (!make_geom(p, g, err)) return fail(AN5D_E_INVALID, err);
  if (!A) return fail(AN5D_E_INVALID, "null host array");
  if (ms) *ms = 0.0;
  if (p->timesteps < 0) return fail(AN5D_E_INVALID, "timesteps must be >= 0");
  if (p->timesteps == 0) return AN5D_OK;
  const size_t esz = p->dtype == AN5D_FLOAT64 ? 8 : 4;
  const size_t gb = (size_t)g.area * esz;
  void* dA = nullptr;
  Staging* ring = nullptr;
  std::unique_lock<std::mutex> hold;  // the staging grid and ring are ours until we return
  int rc = device_grid(2 * gb, &dA, &ring, hold);
  if (rc) return rc;
  char* h0 = static_cast<char*>(A);
  char* h1 = h0 + gb;
  char* d0 = static_cast<char*>(dA);
  char* d1 = d0 + gb;
  // The array may be pinned memory that work already enqueued on the device still
  // writes or reads (a copy on the null stream, say): the threads that copy it
  // below are ordered after no stream, so wait for all of them.
  hipError_t e = hipDeviceSynchronize();
  if (e != hipSuccess) return hip_fail(e, "hipDeviceSynchronize");
  // The first launch writes the whole interior of buffer 1: of that buffer only
  // the halo is read, so only the halo goes up.
  rc = staging_upload(*ring, d0, h0, gb);
  if (rc == AN5D_OK) rc = staging_upload_halo(*ring, d1, h1, g, esz);
  e = hipStreamSynchronize(ring->st);
  if (rc) return rc;
  if (e != hipSuccess) return hip_fail(e, "H2D copies");
  int launches = 0;
  const double t0 = sb_time_ms();
  rc = run_schedule(p, dA, nullptr, cfg, 0, 0, ring->st, &launches);
  e = hipStreamSynchronize(ring->st);
  const double t1 = sb_time_ms();
  if (rc) return rc;
  if (e != hipSuccess) return hip_fail(e, "kernel execution");
  // a single launch leaves buffer 0 as it came
  if (launches > 1) rc = staging_download(*ring, h0, d0, gb);
  if (rc == AN5D_OK) rc = staging_download(*ring, h1, d1, gb);
  if (rc) {
    (void)hipStreamSynchronize(ring->st);
    return rc;
  }
  if (ms) *ms = t1 - t0;
  return AN5D_OK;
}

extern "C" int an5d_kernel_stencil(int stencil, int dtype, void* A1, int compsize, int timestep,
                                   int scop, double* ms) {
  if (stencil < 0 || stencil >= kNumStencils) return fail(AN5D_E_INVALID, "bad stencil id");
  const StencilRT& s = stencil_rt(stencil);
  an5d_problem p;
  memset(&p, 0, sizeof(p));
  p.stencil = stencil;
  p.dtype = dtype;
  for (int d = 0; d < s.dim; d++) p.n[d] = compsize;
  p.timesteps = timestep;
  p.coefs = nullptr;
  p.divisor = -1.0;
  if (ms) *ms = 0.0;
  // host.cu:17: nothing to do unless dimsize >= 2r+1 and timestep >= 1
  if ((long long)compsize + 2 * s.rad < 2 * s.rad + 1 || timestep < 1) return AN5D_OK;
  if (scop) {
    // tiling overrides for run drivers: AN5D_BT, AN5D_VARIANT, AN5D_SL
    an5d_config cfg{0, -1, 0, AN5D_EXACT};
    if (const char* e = getenv("AN5D_BT")) cfg.bt = atoi(e);
    if (const char* e = getenv("AN5D_VARIANT")) cfg.variant = atoi(e);
    if (const char* e = getenv("AN5D_SL")) cfg.sl = atoi(e);
    if (const char* e = getenv("AN5D_MODE")) cfg.mode = atoi(e);
    return an5d_forward_host(&p, A1, &cfg, ms);
  }
  return an5d_cpu_forward(&p, A1, 0, ms);
}

extern "C" int an5d_release(void) {
  DeviceCache& c = cache();
  // host calls under way keep their grid and ring until they return
  std::vector<std::unique_lock<std::mutex>> users;
  {
    std::vector<std::mutex*> all;
    {
      std::lock_guard<std::mutex> lk(c.mu);
      for (auto& kv : c.grid_users) all.push_back(&kv.second);
    }
    for (std::mutex* m : all) users.emplace_back(*m);
  }
  std::lock_guard<std::mutex> lk(c.mu);
  for (auto& kv : c.coefs) (void)hipFree(kv.second);
  c.coefs.clear();
  for (auto& kv : c.grids)
    if (kv.second.first) (void)hipFree(kv.second.first);
  c.grids.clear();
  for (auto& kv : c.stagings) staging_free(kv.second);
  return AN5D_OK;
}

extern "C" const char* an5d_last_error(void) { return g_err.c_str(); }
