"""Build the autotuner table for a set of workloads on the current GPU.

    python -m pyan5d.tune [--set bench|ladder|all] [--stencils A,B] [--out FILE] [--max-measured K]

"ladder": every stencil, dtype and mode at sides of powers of two and, up to
the sizes where launches fill the chip many times over, one size between, so
that a grid of any size has a row of about its own cell count (the library
takes the nearest one within 8x; kernel and depth carry over, the segment
length is chosen for the grid at hand).  "all" is both sets.

For every (stencil, dtype, size, mode, run length) of the set, an5d_autotune
ranks all (kernel shape, register cap, bt, sl) candidates with the analytic
model, times the best K on the GPU (on the field halfway through the run,
with the benchmark's coefficients: pyan5d.presets "baseline") and keeps the
fastest; the table is then written to FILE (default:
the file the library loads, an5d-artifact_amd/tuned.tsv).  This replaces the
reference's Excel model + top-5 compile/run scripts
(compiled/nvcc_compile_top5.sh, compiled/run.sh), which pick one
configuration per stencil by compiling and timing separate binaries.
"""
from __future__ import annotations

import argparse
import os
import sys
import time

import numpy as np

from . import EXACT, FAST, autotune, info, presets, tune_clear, tune_load, tune_save

STENCILS_2D = ["star2d1r", "star2d2r", "star2d3r", "star2d4r", "box2d1r", "box2d2r", "box2d3r",
               "box2d4r", "j2d5pt", "j2d9pt", "j2d9pt-gol", "gradient2d"]
STENCILS_3D = ["star3d1r", "star3d2r", "star3d3r", "star3d4r", "box3d1r", "box3d2r", "box3d3r",
               "box3d4r", "j3d27pt"]

# (stencil, dtype, interior size, modes, timesteps of the run)
BENCH = [
    ("star3d1r", np.float32, [512, 512, 512], (EXACT, FAST), 1000),
    ("star3d1r", np.float64, [512, 512, 512], (EXACT, FAST), 1000),
    ("j2d5pt", np.float32, [16384, 16384], (EXACT, FAST), 1000),
    ("j2d5pt", np.float32, [4096, 4096], (EXACT, FAST), 100),
    ("box2d4r", np.float32, [16384, 16384], (EXACT,), 1000),
    ("box2d4r", np.float64, [16384, 16384], (EXACT,), 1000),
    ("star3d4r", np.float32, [512, 512, 512], (EXACT,), 1000),
    ("star3d4r", np.float64, [512, 512, 512], (EXACT,), 1000),
    ("j3d27pt", np.float32, [512, 512, 512], (EXACT,), 1000),
    ("j3d27pt", np.float64, [512, 512, 512], (EXACT,), 1000),
    ("gradient2d", np.float32, [8192, 8192], (EXACT,), 256),
    ("j2d9pt", np.float32, [8192, 8192], (EXACT,), 256),
    ("j2d9pt-gol", np.float32, [8192, 8192], (EXACT,), 256),
]


LADDER_2D = [256, 384, 512, 768, 1024, 1536, 2048, 3072, 4096, 6144, 8192, 16384]
LADDER_3D = [64, 96, 128, 192, 256, 512]
# the radius-1 boxes change kernel between 256^3 and 512^3; the stars do not
LADDER_BOX3D1 = {np.float32: [320, 400], np.float64: [320]}


def workloads(which):
    out = [] if which == "ladder" else list(BENCH)
    if which in ("ladder", "all"):
        seen = {(s, np.dtype(d).name, tuple(n), m) for s, d, n, ms, _ in out for m in ms}
        for s in STENCILS_2D + STENCILS_3D:
            for dt in (np.float32, np.float64):
                sides = LADDER_3D + (LADDER_BOX3D1[dt] if s in ("box3d1r", "j3d27pt") else [])
                for n in [[x] * 2 for x in LADDER_2D] if s in STENCILS_2D else [[x] * 3 for x in sides]:
                    modes = tuple(m for m in (EXACT, FAST) if (s, np.dtype(dt).name, tuple(n), m) not in seen)
                    if modes:
                        out.append((s, dt, n, modes, 100))
    return out


def main(argv=None):
    ap = argparse.ArgumentParser(description=__doc__.splitlines()[0])
    ap.add_argument("--set", choices=("bench", "ladder", "all"), default="all")
    ap.add_argument("--stencils", default="", help="only these, comma-separated (default: every one of the set)")
    ap.add_argument("--out", default=None, help="table file (default: the library's tuned.tsv)")
    ap.add_argument("--max-measured", type=int, default=1000)
    ap.add_argument("--fresh", action="store_true", help="start from an empty table")
    args = ap.parse_args(argv)
    if args.fresh:
        tune_clear()
    elif args.out and os.path.exists(args.out):
        tune_load(args.out)
    only = [s for s in args.stencils.split(",") if s]
    for name, dt, n, modes, steps in workloads(args.set):
        if only and name not in only:
            continue
        info(name)  # validates the name
        for mode in modes:
            t0 = time.perf_counter()
            coefs, div = presets.coefficients(name, "baseline")
            cfg, gs = autotune(name, n, dt, mode=mode, max_measured=args.max_measured, timesteps=steps,
                               coefs=coefs, divisor=div)
            print(f"[tune] {name} {np.dtype(dt).name} {'x'.join(map(str, n))} "
                  f"{'fast' if mode == FAST else 'exact'}: variant {cfg['variant']} bt {cfg['bt']} "
                  f"sl {cfg['sl']} -> {gs:.1f} GStencil/s ({time.perf_counter() - t0:.1f} s)", flush=True)
    tune_save(args.out)
    print(f"[tune] table written to {args.out or 'the default tuned.tsv'}", flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
