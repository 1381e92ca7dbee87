// Kernel arguments from the dtype-erased host form.
#pragma once

#include "engine.hpp"
#include "sweep.hpp"

namespace an5d {

template <typename U>
SweepArgs<U> to_args(const LaunchArgs& a) {
  SweepArgs<U> s;
  s.src = static_cast<const U*>(a.src);
  s.dst = static_cast<U*>(a.dst);
  s.coef = static_cast<const U*>(a.coef);
  s.gscale = a.gscale;
  s.has_div = a.has_div;
  s.D0 = a.D0; s.D1 = a.D1; s.D2 = a.D2;
  s.s0 = a.s0; s.s1 = a.s1;
  s.ntk = a.ntk; s.ntj = a.ntj; s.nseg = a.nseg; s.sl = a.sl;
  s.SK = a.SK; s.SJ = a.SJ;
  s.mid = static_cast<U*>(a.mid);
  s.mid_stride = a.mid_stride;
  s.mid_mask = a.mid_mask;
  s.nt_store = a.nt_store;
  s.steps = a.steps;
  return s;
}

}  // namespace an5d
