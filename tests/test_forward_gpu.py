"""GPU parity of the forward sweep: the HIP kernels against the CPU oracle,
bit for bit (every stencil x dtype x kernel shape x several bt), tiling
invariance, the kernel_stencil drop-in, device-resident layouts and the
golden fixtures made from the reference's own programs."""
import os

import numpy as np
import pytest

import oracle_lib as O
import pyan5d

pytestmark = pytest.mark.gpu
GOLD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")


def small_n(name):
    d = O.info(name)
    if d["dim"] == 2:
        return [37, 300]  # two column tiles, ragged edges
    if d["ntaps"] > 100:
        return [6, 7, 9]
    return [11, 45, 150]


def rand_grid(name, n, dt, seed):
    d = O.info(name)
    rng = np.random.default_rng(seed)
    shape = tuple(x + 2 * d["rad"] for x in n)
    u = rng.random(shape).astype(dt)
    return np.stack([u, u])


def same(a, b):
    return np.array_equal(a.view(np.uint8), b.view(np.uint8))


def cases():
    out = []
    for name in O.NAMES:
        for dt in (np.float32, np.float64):
            for v in pyan5d.variants(name, 0 if dt == np.float32 else 1):
                bts = sorted({1, v["btmax"], max(1, v["btmax"] // 2)})
                for bt in bts:
                    out.append((name, dt, v["index"], bt))
    return out


@pytest.mark.parametrize("name,dt,variant,bt", cases())
def test_forward_bitwise_vs_oracle(name, dt, variant, bt):
    n = small_n(name)
    T = 2 * bt + 1 if O.info(name)["ntaps"] <= 100 else 2
    print(f"case {name} {np.dtype(dt).name} variant={variant} bt={bt} n={n} T={T}", flush=True)
    A = rand_grid(name, n, dt, seed=bt * 7 + variant)
    B = A.copy()
    pyan5d.forward_host(name, A, n, T, bt=bt, variant=variant)
    O.run(name, B, n, T)
    assert same(A[T % 2], B[T % 2])


@pytest.mark.parametrize("name,dt", [("j2d5pt", np.float32), ("star3d1r", np.float32),
                                     ("box3d1r", np.float64), ("gradient2d", np.float32)])
def test_tiling_invariance(name, dt):
    d = O.info(name)
    n = [300, 1030] if d["dim"] == 2 else [40, 130, 200]
    T = 13
    base = rand_grid(name, n, dt, seed=3)
    results = []
    for v in pyan5d.variants(name, 0 if dt == np.float32 else 1):
        for bt in range(1, v["btmax"] + 1):
            for sl in (0, 7, 64):
                A = base.copy()
                print(f"case {name} variant={v['index']} bt={bt} sl={sl}", flush=True)
                pyan5d.forward_host(name, A, n, T, bt=bt, variant=v["index"], sl=sl)
                results.append(A[T % 2].copy())
    B = base.copy()
    pyan5d.cpu_forward(name, B, n, T)
    for r in results:
        assert same(r, B[T % 2])


def test_kernel_stencil_dropin_config0_size():
    """j2d5pt FP32 4096^2, 100 steps, reference init; GPU path vs
    the CPU path (OpenMP loop), whole grid, both buffers' halo untouched."""
    print("case j2d5pt 4096^2 T=100 drop-in", flush=True)
    A = O.init_grid("j2d5pt", 4096, np.float32)
    B = A.copy()
    halo = A[:, 0, :].copy()
    pyan5d.kernel_stencil("j2d5pt", A, 4096, 100, scop=True)
    pyan5d.kernel_stencil("j2d5pt", B, 4096, 100, scop=False)
    assert same(A[0], B[0])
    assert np.array_equal(A[:, 0, :], halo)


@pytest.mark.parametrize("name", O.NAMES)
@pytest.mark.parametrize("dt,tname", [(np.float32, "float"), (np.float64, "double")])
def test_golden_fixture_on_gpu(name, dt, tname):
    g = np.load(os.path.join(GOLD, f"stencil_{name}_{tname}.npz"))
    n, T = int(g["n"]), int(g["T"])
    print(f"case golden {name} {tname} n={n} T={T}", flush=True)
    d = O.info(name)
    A = O.init_grid(name, n, dt)
    pyan5d.kernel_stencil(name, A, n, T, scop=True)
    assert same(A[T % 2], g["out"][T % 2])


def test_forward_device_layouts(torch_cuda):
    torch = torch_cuda
    name, n, T = "star3d1r", [20, 33, 70], 9
    d = O.info(name)
    base = rand_grid(name, n, np.float32, seed=11)
    B = base.copy()
    O.run(name, B, n, T)
    # reference layout
    t = torch.from_numpy(base.copy()).cuda()
    print("case forward_device reference layout", flush=True)
    pyan5d.forward_device(name, t, n, T, bt=3)
    torch.cuda.synchronize()
    assert same(t.cpu().numpy()[T % 2], B[T % 2])
    # padded rows and planes (strided view)
    D = [x + 2 * d["rad"] for x in n]
    big = torch.zeros((2, D[0], D[1] + 3, D[2] + 29), dtype=torch.float32, device="cuda")
    view = big[:, :, :D[1], :D[2]]
    view.copy_(torch.from_numpy(base))
    print("case forward_device strided layout", flush=True)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        pyan5d.forward_device(name, view, n, T, bt=2, stream=s)
    s.synchronize()
    assert same(view.cpu().numpy()[T % 2], B[T % 2])


def test_single_launch_entry(torch_cuda):
    torch = torch_cuda
    name, n = "j2d9pt", [50, 400]
    base = rand_grid(name, n, np.float32, seed=2)
    B = base.copy()
    O.run(name, B, n, 5)
    t = torch.from_numpy(base.copy()).cuda()
    print("case single launches 3+2", flush=True)
    pyan5d.launch(name, t, n, 3, c0=0)
    pyan5d.launch(name, t, n, 2, c0=1)
    torch.cuda.synchronize()
    assert same(t.cpu().numpy()[0], B[1])


@pytest.mark.parametrize("name", ["j2d5pt", "star3d1r", "box2d4r", "j3d27pt", "gradient2d"])
def test_other_coefficients_and_divisor(name):
    d = O.info(name)
    n = [30, 270] if d["dim"] == 2 else [10, 40, 140]
    rng = np.random.default_rng(1)
    if d["linear"]:
        c = rng.random(d["ntaps"]) + 0.01
        c = c / c.sum()
        div = 0.0
    else:
        c = [1e-4, 0.01]
        div = -1.0
    for dt in (np.float32, np.float64):
        A = rand_grid(name, n, dt, seed=4)
        B = A.copy()
        print(f"case coefs {name} {np.dtype(dt).name}", flush=True)
        pyan5d.forward_host(name, A, n, 6, coefs=c, divisor=div)
        O.run(name, B, n, 6, coefs=c, divisor=div)
        assert same(A[0], B[0])


def test_rectangular_and_tiny_grids():
    for name, n in [("star2d1r", [1, 1]), ("star2d2r", [3, 700]), ("j2d5pt", [900, 5]),
                    ("star3d1r", [1, 2, 3]), ("star3d1r", [70, 3, 9]), ("box3d1r", [5, 60, 2])]:
        A = rand_grid(name, n, np.float32, seed=9)
        B = A.copy()
        print(f"case rect {name} {n}", flush=True)
        pyan5d.forward_host(name, A, n, 7)
        O.run(name, B, n, 7)
        assert same(A[1], B[1])


@pytest.mark.parametrize("name", ["star3d2r", "star3d3r", "star3d4r"])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_plane_kernel_ragged_grids(name, dt):
    """The LDS-staged one-step kernel (kind 2) on grids smaller than one tile,
    ragged tile edges in both in-plane dims and segments shorter than 2R+1."""
    vs = [v for v in pyan5d.variants(name, 0 if dt == np.float32 else 1) if v["kind"] == 2]
    assert len(vs) == 1
    v = vs[0]
    for n, sl in [([1, 1, 1], 0), ([3, 17, 130], 1), ([9, 5, 300], 2), ([20, 33, 257], 7), ([13, 16, 128], 0)]:
        A = rand_grid(name, n, dt, seed=sum(n))
        B = A.copy()
        T = 3
        print(f"case plane {name} {np.dtype(dt).name} n={n} sl={sl}", flush=True)
        pyan5d.forward_host(name, A, n, T, variant=v["index"], sl=sl)
        O.run(name, B, n, T)
        assert same(A[T % 2], B[T % 2])
        C = rand_grid(name, n, dt, seed=sum(n))
        D = C.copy()
        pyan5d.forward_host(name, C, n, T, variant=v["index"], sl=sl, mode=pyan5d.FAST)
        O.run(name, D, n, T)
        got, ref = C[T % 2].astype(np.float64), D[T % 2].astype(np.float64)
        rel = np.max(np.abs(got - ref) / np.maximum(np.abs(ref), np.finfo(dt).tiny))
        assert rel <= (1e-5 if dt == np.float32 else 1e-12), rel


@pytest.mark.parametrize("name", ["j3d27pt", "box3d1r"])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_box3d_plane_partial_sums_ragged_grids(name, dt):
    """The plane-streamed partial-sum kernels of the radius-1 3D boxes (kind 2
    for a box): bit for bit the oracle on grids smaller than one tile, ragged
    tiles in both in-plane dims, segments of 1-7 planes and the default, in
    exact mode; within 1e-5 / 1e-12 relative in FMA mode; j3d27pt also with
    its /159 divisor and other coefficients."""
    vs = [v for v in pyan5d.variants(name, 0 if dt == np.float32 else 1) if v["kind"] == 2]
    assert len(vs) == 2
    for v in vs:
        for n, sl in [([1, 1, 1], 0), ([3, 17, 130], 1), ([9, 5, 300], 2), ([20, 33, 257], 7),
                      ([13, 16, 128], 0), ([40, 70, 260], 0)]:
            T = 4
            print(f"case box3d partial sums {name} {np.dtype(dt).name} variant {v['index']} n={n} sl={sl}",
                  flush=True)
            A = rand_grid(name, n, dt, seed=sum(n) + v["index"])
            B = A.copy()
            pyan5d.forward_host(name, A, n, T, variant=v["index"], sl=sl)
            O.run(name, B, n, T)
            assert same(A[T % 2], B[T % 2])
            C = rand_grid(name, n, dt, seed=sum(n) + 1)
            D = C.copy()
            pyan5d.forward_host(name, C, n, T, variant=v["index"], sl=sl, mode=pyan5d.FAST)
            O.run(name, D, n, T)
            got, ref = C[T % 2].astype(np.float64), D[T % 2].astype(np.float64)
            rel = np.max(np.abs(got - ref) / np.maximum(np.abs(ref), np.finfo(dt).tiny))
            assert rel <= (1e-5 if dt == np.float32 else 1e-12), rel
        if name == "j3d27pt":
            n, T = [30, 40, 200], 5
            rng = np.random.default_rng(3)
            coefs = rng.random(27).astype(np.float64)
            for div in (159.0, 0.0):
                print(f"case box3d partial sums {name} {np.dtype(dt).name} variant {v['index']} "
                      f"divisor {div}", flush=True)
                A = rand_grid(name, n, dt, seed=9)
                B = A.copy()
                pyan5d.forward_host(name, A, n, T, coefs=coefs, divisor=div, variant=v["index"])
                O.run(name, B, n, T, coefs=coefs, divisor=div)
                assert same(A[T % 2], B[T % 2])


@pytest.mark.parametrize("name", ["j2d5pt", "j2d9pt", "star2d3r", "box2d2r", "gradient2d",
                                  "star3d1r", "box3d1r", "j3d27pt", "star3d4r"])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_fast_mode_within_tolerance(name, dt):
    """FMA mode (divisor folded into the coefficients): within 1e-5 (FP32) /
    1e-12 (FP64) relative of the oracle, relative to max(|ref|, smallest normal)."""
    d = O.info(name)
    n = [200, 700] if d["dim"] == 2 else [30, 60, 140]
    T = 40 if d["dim"] == 2 else 12
    A = rand_grid(name, n, dt, seed=21)
    B = A.copy()
    vs = pyan5d.variants(name, 0 if dt == np.float32 else 1)
    bt = min(3, vs[0]["btmax"])
    print(f"case fast {name} {np.dtype(dt).name} bt={bt}", flush=True)
    pyan5d.forward_host(name, A, n, T, bt=bt, mode=pyan5d.FAST)
    O.run(name, B, n, T)
    got, ref = A[T % 2].astype(np.float64), B[T % 2].astype(np.float64)
    floor = np.finfo(dt).tiny
    rel = np.max(np.abs(got - ref) / np.maximum(np.abs(ref), floor))
    assert rel <= (1e-5 if dt == np.float32 else 1e-12), rel


SHARE_CASES = [("star3d1r", np.float32), ("star3d1r", np.float64), ("star2d1r", np.float32),
               ("star2d1r", np.float64), ("j2d5pt", np.float32), ("j2d5pt", np.float64)]


@pytest.mark.parametrize("name,dt", SHARE_CASES)
def test_shared_product_form_bitwise(name, dt):
    """Radius-1 stars whose face taps carry one coefficient run the
    shared-product kernels (each c * u formed once per cell): bit for bit
    the oracle and the general kernels, for every shape and depth."""
    d = O.info(name)
    n = [37, 70, 300] if d["dim"] == 3 else [57, 700]
    T = 11
    ctr = [i for i, t in enumerate(O.taps(name)[0]) if not t[1:].any()][0]
    coefs = np.full(d["ntaps"], 0.1)
    coefs[ctr] = 0.4
    div = 118.0 if d["divisor"] else 0.0
    rng = np.random.default_rng(3)
    u = rng.random([x + 2 * d["rad"] for x in n]).astype(dt)
    A0 = np.stack([u, u])  # both buffers alike: the halo is one fixed boundary
    ref = A0.copy()
    O.run(name, ref, n, T, coefs=coefs, divisor=div)
    dcode = 0 if dt == np.float32 else 1
    for v in pyan5d.variants(name, dcode):
        if v["kind"] != 0:
            continue
        for bt in sorted({1, 2, min(3, v["btmax"]), v["btmax"]}):
            print(f"case shared-product {name} {np.dtype(dt).name} variant {v['index']} bt {bt}", flush=True)
            A = A0.copy()
            pyan5d.forward_host(name, A, n, T, coefs=coefs, divisor=div, bt=bt, variant=v["index"])
            B = A0.copy()
            pyan5d.forward_host(name, B, n, T, coefs=coefs, divisor=div, bt=bt, variant=v["index"],
                                mode=pyan5d.EXACT_GENERAL)
            assert np.array_equal(A[T % 2].view(np.uint8), ref[T % 2].view(np.uint8)), (v, bt)
            assert np.array_equal(B[T % 2].view(np.uint8), ref[T % 2].view(np.uint8)), (v, bt)


def test_forward_host_from_several_threads():
    """Host calls from several threads on one device, with grids of
    different sizes (the staging grid grows while others are running): every
    result equals the oracle's."""
    import threading
    cases = [([300, 700], 9), ([900, 1200], 7), ([150, 2000], 5), ([1100, 900], 8)]
    print("case threads forward_host j2d5pt x4", flush=True)
    # both buffers hold the same field (the halo is read from either one)
    inputs = []
    for i, (n, _) in enumerate(cases):
        u = np.random.default_rng(i).random((n[0] + 2, n[1] + 2)).astype(np.float32)
        inputs.append(np.stack([u, u]))
    outs = [a.copy() for a in inputs]
    errors = []

    def work(i):
        try:
            n, T = cases[i]
            pyan5d.forward_host("j2d5pt", outs[i], n, T)
        except Exception as e:  # reported below
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(cases))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    for (n, T), a, o in zip(cases, inputs, outs):
        ref = a.copy()
        O.run("j2d5pt", ref, n, T)
        assert np.array_equal(o[T % 2], ref[T % 2])


def test_forward_host_waits_for_copies_under_way(torch_cuda):
    """A pinned host array that a copy enqueued on the null stream is still to
    fill (behind a few milliseconds of work): the call waits for it; and a copy
    out of the array enqueued before the call takes the state before it."""
    torch = torch_cuda
    name, n, T = "j2d5pt", [500, 700], 6
    print("case host array with copies under way", name, flush=True)
    A = rand_grid(name, n, np.float32, seed=3)
    ref = A.copy()
    O.run(name, ref, n, T)
    dev = torch.from_numpy(A).cuda()
    pinned = torch.zeros(A.shape, pin_memory=True)
    back = torch.zeros_like(dev)
    m = torch.rand(4096, 4096, device="cuda")
    torch.mm(m, m)
    torch.cuda.synchronize()
    for _ in range(40):
        torch.mm(m, m)
    pinned.copy_(dev, non_blocking=True)
    pyan5d.forward_host(name, pinned.numpy(), n, T)
    assert same(pinned.numpy()[T % 2], ref[T % 2])
    pinned.copy_(torch.from_numpy(A))
    for _ in range(40):
        torch.mm(m, m)
    back.copy_(pinned, non_blocking=True)
    pyan5d.forward_host(name, pinned.numpy(), n, T)
    torch.cuda.synchronize()
    assert same(back.cpu().numpy(), A)


@pytest.mark.parametrize("name", ["box3d2r", "box3d3r", "box3d4r"])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_box3d_column_kernel_ragged_grids(name, dt):
    """The column kernel of the wide 3D boxes (kind 4): rows that end inside a
    lane's run, rows of one run only, a last workgroup that is nearly empty,
    segments of one plane, of fewer planes than the stencil's and the default;
    bit for bit the oracle in exact mode (also over a divisor), within 1e-5 /
    1e-12 of the field's largest value in FMA mode."""
    v, = [v for v in pyan5d.variants(name, 0 if dt == np.float32 else 1) if v["kind"] == 4]
    for n, sl, div in [([1, 1, 4], 0, -1.0), ([3, 5, 7], 1, 7.0), ([9, 17, 66], 3, -1.0), ([12, 33, 31], 0, 118.0)]:
        T = 3
        print(f"case columns {name} {np.dtype(dt).name} n={n} sl={sl} divisor={div}", flush=True)
        A = rand_grid(name, n, dt, seed=sum(n))
        B, C = A.copy(), A.copy()
        pyan5d.forward_host(name, A, n, T, variant=v["index"], sl=sl, divisor=div)
        O.run(name, B, n, T, divisor=div)
        assert same(A[T % 2], B[T % 2])
        pyan5d.forward_host(name, C, n, T, variant=v["index"], sl=sl, divisor=div, mode=pyan5d.FAST)
        got, ref = C[T % 2].astype(np.float64), B[T % 2].astype(np.float64)
        assert np.max(np.abs(got - ref)) <= (1e-5 if dt == np.float32 else 1e-12) * np.max(np.abs(ref))


def test_box3d_rows_shorter_than_a_run():
    """Below one run per row the tuned choice does not fit: the default path
    takes the direct kernel as before."""
    n, T = [40, 60, 3], 2
    print("case columns fallback box3d2r", n, flush=True)
    assert pyan5d.resolve_config("box3d2r", n, np.float64)["variant"] == 0
    A = rand_grid("box3d2r", n, np.float64, seed=5)
    B = A.copy()
    pyan5d.forward_host("box3d2r", A, n, T)
    O.run("box3d2r", B, n, T)
    assert same(A[T % 2], B[T % 2])


@pytest.mark.parametrize("name", ["star2d4r", "box3d2r", "box3d3r"])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_direct_kernel_fast_mode_with_subtracted_taps(name, dt):
    """The FMA table carries the taps' signs, so the direct kernel must not
    apply them again."""
    v, = [v for v in pyan5d.variants(name, 0 if dt == np.float32 else 1) if v["kind"] == 1]
    n, T = ([9, 40] if O.info(name)["dim"] == 2 else [6, 7, 9]), 2
    print(f"case direct fast {name} {np.dtype(dt).name}", flush=True)
    A = rand_grid(name, n, dt, seed=8)
    B = A.copy()
    pyan5d.forward_host(name, A, n, T, variant=v["index"], mode=pyan5d.FAST)
    O.run(name, B, n, T)
    got, ref = A[T % 2].astype(np.float64), B[T % 2].astype(np.float64)
    assert np.max(np.abs(got - ref)) <= (1e-5 if dt == np.float32 else 1e-12) * np.max(np.abs(ref))


@pytest.mark.parametrize("name", ["box2d2r", "box2d3r", "box2d4r"])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_box2d_run_kernel_ragged_grids(name, dt):
    """The run kernel of the wide 2D boxes (kind 4): one row, one run per row,
    rows that end inside a run, a last segment that overlaps its neighbour,
    more lanes than runs; bit for bit the oracle, also over a divisor, and
    within 1e-5 / 1e-12 of the field's largest value in FMA mode."""
    v, = [v for v in pyan5d.variants(name, 0 if dt == np.float32 else 1) if v["kind"] == 4]
    for n, sl, div in [([1, 4], 0, -1.0), ([7, 5], 3, 7.0), ([23, 131], 5, -1.0), ([64, 258], 0, 118.0),
                       ([50, 70], 16, -1.0)]:
        T = 3
        print(f"case runs {name} {np.dtype(dt).name} n={n} sl={sl} divisor={div}", flush=True)
        A = rand_grid(name, n, dt, seed=sum(n))
        B, C = A.copy(), A.copy()
        pyan5d.forward_host(name, A, n, T, variant=v["index"], sl=sl, divisor=div)
        O.run(name, B, n, T, divisor=div)
        assert same(A[T % 2], B[T % 2])
        pyan5d.forward_host(name, C, n, T, variant=v["index"], sl=sl, divisor=div, mode=pyan5d.FAST)
        got, ref = C[T % 2].astype(np.float64), B[T % 2].astype(np.float64)
        assert np.max(np.abs(got - ref)) <= (1e-5 if dt == np.float32 else 1e-12) * np.max(np.abs(ref))


TILE_NAMES = ["star2d1r", "star2d2r", "star2d3r", "star2d4r", "box2d1r", "box2d2r", "j2d5pt", "j2d9pt",
              "j2d9pt-gol", "gradient2d"]


@pytest.mark.parametrize("name", TILE_NAMES)
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_register_tiles_at_their_edges(name, dt):
    """The register-tile kernels (kind 5): a grid of one cell, of exactly one
    tile, one cell more in either direction (two tiles, the second owning
    little), several tiles; the deepest block and one that is not; bit for bit
    the oracle."""
    r = O.info(name)["rad"]
    for v in pyan5d.variants(name, 0 if dt == np.float32 else 1):
        if v["kind"] != 5:
            continue
        th, tw = v["nw"] * v["cj"] - 2 * r, 64 * v["ck"] - 2 * r  # interior of a grid that is one tile
        for bt in sorted({1, max(1, v["btmax"] // 2), v["btmax"]}):
            for n in ([1, 1], [th, tw], [th + 1, tw], [th, tw + 1], [2 * th + 5, tw + 70]):
                T = bt + max(1, bt // 2)
                print(f"case tiles {name} {np.dtype(dt).name} variant {v['index']} bt={bt} n={n}", flush=True)
                A = rand_grid(name, n, dt, seed=sum(n) + bt)
                B = A.copy()
                pyan5d.forward_host(name, A, n, T, variant=v["index"], bt=bt)
                O.run(name, B, n, T)
                assert same(A[T % 2], B[T % 2])


@pytest.mark.parametrize("name,n", [("star2d2r", [1500, 3000]), ("star2d1r", [3, 5]), ("star3d2r", [30, 41, 53]),
                                    ("box3d1r", [1, 2, 3])])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_host_arrays_with_two_halos(name, n, dt):
    """Host arrays whose buffers hold different halos: every step reads the
    halo of its own input buffer and writes none (bt = 1, so the C loop does
    the same); both buffers come back, also after a single launch; arrays
    beyond the pinned ring and of a few cells."""
    r = O.info(name)["rad"]
    rng = np.random.default_rng(6)
    A0 = rng.random([2] + [x + 2 * r for x in n]).astype(dt)
    for T in (1, 2, 3):
        print(f"case host halos {name} {np.dtype(dt).name} {n} T={T}", flush=True)
        A, B = A0.copy(), A0.copy()
        pyan5d.forward_host(name, A, n, T, bt=1)
        O.run(name, B, n, T)
        # the schedule may end with fewer launches than steps only for bt > 1
        assert same(A, B)


@pytest.mark.parametrize("name", ["box3d1r", "j3d27pt"])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_box3d1_column_kernel_ragged_grids(name, dt):
    """The column kernel of the 27-point boxes (kind 4): one run per row, rows
    that end inside a run, a nearly empty last workgroup, segments of one plane,
    fewer than three and the default; with and without the division, and in FMA
    mode within 1e-5 / 1e-12 of the field's largest value."""
    for v in pyan5d.variants(name, 0 if dt == np.float32 else 1):
        if v["kind"] != 4:
            continue
        for n, sl, div in [([1, 1, 4], 0, -1.0), ([5, 6, 7], 1, 7.0), ([9, 17, 66], 2, 159.0), ([12, 33, 31], 0, 0.0)]:
            T = 4
            print(f"case columns {name} {np.dtype(dt).name} variant {v['index']} n={n} sl={sl} divisor={div}",
                  flush=True)
            A = rand_grid(name, n, dt, seed=sum(n))
            B, C = A.copy(), A.copy()
            pyan5d.forward_host(name, A, n, T, variant=v["index"], sl=sl, divisor=div)
            O.run(name, B, n, T, divisor=div)
            assert same(A[T % 2], B[T % 2])
            pyan5d.forward_host(name, C, n, T, variant=v["index"], sl=sl, divisor=div, mode=pyan5d.FAST)
            got, ref = C[T % 2].astype(np.float64), B[T % 2].astype(np.float64)
            assert np.max(np.abs(got - ref)) <= (1e-5 if dt == np.float32 else 1e-12) * np.max(np.abs(ref))


@pytest.mark.parametrize("name", ["star3d1r", "box3d1r", "j3d27pt"])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_3d_register_tiles_at_their_edges(name, dt):
    """The 3D register tiles (kind 5: 8 planes of 32 rows x 64 cells): a grid of
    one cell, of exactly one tile, a plane, row or cell more, several tiles, at
    every depth; bit for bit the oracle."""
    for v in pyan5d.variants(name, 0 if dt == np.float32 else 1):
        if v["kind"] != 5:
            continue
        for bt in range(1, v["btmax"] + 1):
            for n in ([1, 1, 1], [8, 30, 62], [9, 30, 62], [8, 31, 62], [8, 30, 63], [19, 61, 130]):
                T = bt + 1
                print(f"case tiles {name} {np.dtype(dt).name} variant {v['index']} bt={bt} n={n}", flush=True)
                A = rand_grid(name, n, dt, seed=sum(n) + bt)
                B = A.copy()
                pyan5d.forward_host(name, A, n, T, variant=v["index"], bt=bt)
                O.run(name, B, n, T)
                assert same(A[T % 2], B[T % 2])


@pytest.mark.parametrize("name", ["j2d5pt", "j2d9pt", "j2d9pt-gol", "gradient2d"])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_register_tiles_division_modes(name, dt):
    """The register tiles' three division forms (none, the source's divisor, any
    other) on a grid of a few tiles with remainders; bit for bit the oracle."""
    for v in pyan5d.variants(name, 0 if dt == np.float32 else 1):
        if v["kind"] != 5:
            continue
        for div in (0.0, 118.0, 7.0) if name != "gradient2d" else (-1.0,):
            n, T = [v["nw"] * v["cj"] + 9, 64 * v["ck"] + 21], 5
            print(f"case tile divisions {name} {np.dtype(dt).name} variant {v['index']} divisor={div}", flush=True)
            A = rand_grid(name, n, dt, seed=3)
            B = A.copy()
            pyan5d.forward_host(name, A, n, T, variant=v["index"], bt=3, divisor=div)
            O.run(name, B, n, T, divisor=div)
            assert same(A[T % 2], B[T % 2])


@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_3d_register_tiles_of_four_planes(dt):
    """The tiles of four planes by 16 or 32 rows: exactly one tile, a plane, a
    row or a cell more, at every depth; bit for bit the oracle."""
    name = "star3d1r"
    for v in pyan5d.variants(name, 0 if dt == np.float32 else 1):
        if v["kind"] != 5:
            continue
        for bt in range(1, v["btmax"] + 1):
            for n in ([4, 14, 62], [5, 14, 62], [4, 15, 62], [4, 30, 63], [13, 45, 127]):
                T = bt + 1
                print(f"case tiles {name} {np.dtype(dt).name} variant {v['index']} bt={bt} n={n}", flush=True)
                A = rand_grid(name, n, dt, seed=sum(n) + bt)
                B = A.copy()
                pyan5d.forward_host(name, A, n, T, variant=v["index"], bt=bt)
                O.run(name, B, n, T)
                assert same(A[T % 2], B[T % 2])


@pytest.mark.parametrize("name", ["j2d5pt", "j2d9pt-gol", "star2d2r", "star2d4r", "box2d2r", "gradient2d"])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_default_choice_on_ragged_grids(name, dt):
    """The kernel and depth that a call without a configuration takes, at sizes
    between the table's rows: long, tall and odd grids; bit for bit the oracle."""
    for n in ([3, 9001], [9001, 3], [311, 517], [256, 1025], [700, 901]):
        T = 18
        print(f"case default {name} {np.dtype(dt).name} n={n}", flush=True)
        A = rand_grid(name, n, dt, seed=sum(n))
        B = A.copy()
        pyan5d.forward_host(name, A, n, T)
        O.run(name, B, n, T)
        assert same(A[T % 2], B[T % 2])


def test_star3d_neighbour_waits():
    """FP32 exact star3d1r at three steps a launch and more, where the waves wait
    for their two neighbours: ragged grids of several workgroups and segments, the
    general and the shared-product form; bit for bit the oracle, twice."""
    name = "star3d1r"
    for v in pyan5d.variants(name, 0):
        if v["kind"] != 0:
            continue
        for bt in range(3, v["btmax"] + 1):
            for n, sl in (([1, 1, 1], 0), ([29, 70, 131], 7), ([61, 33, 200], 0)):
                print(f"case neighbour waits variant {v['index']} bt={bt} n={n} sl={sl}", flush=True)
                A = rand_grid(name, n, np.float32, seed=sum(n) + bt)
                ref = A.copy()
                O.run(name, ref, n, bt + 1)
                for mode in (pyan5d.EXACT, pyan5d.EXACT_GENERAL):
                    for _ in range(2):
                        B = A.copy()
                        pyan5d.forward_host(name, B, n, bt + 1, variant=v["index"], bt=bt, sl=sl, mode=mode)
                        assert same(B[(bt + 1) % 2], ref[(bt + 1) % 2])


@pytest.mark.parametrize("name,dt,mode,bt,n,ck,waves", [
    ("box2d3r", np.float64, pyan5d.FAST, 2, [12000, 12000], 4, 2),
    ("box2d3r", np.float64, pyan5d.FAST, 2, [14000, 3500], 4, 2),
    ("box2d4r", np.float32, pyan5d.EXACT, 3, [5000, 5000], 4, 1)])
def test_segments_of_large_grids_fill_one_round(name, dt, mode, bt, n, ck, waves):
    """The default segment length of a 2D sweep on a grid that fills the chip: as
    many waves as the kernel's registers hold (the last argument, per SIMD), no
    second round and not half of one."""
    r = O.info(name)["rad"]
    print(f"case segments {name} {np.dtype(dt).name} n={n}", flush=True)
    v = pyan5d.variants(name, 0 if dt == np.float32 else 1)[0]
    assert v["kind"] == 0 and v["ck"] == ck
    sl = pyan5d.resolve_config(name, n, dt, mode=mode, bt=bt, variant=0)["sl"]
    runs = -(-n[0] // sl) * -(-n[1] // (64 * ck - 2 * bt * r))
    assert 0.9 * waves * 1024 <= runs <= waves * 1024


def fma_bound(name, dt, A, n, T, div):
    """How far FMA mode may lie from the C loop after T steps (linear stencils),
    from the unit roundoff u: a step's products, sums and division round ntaps + 1
    times, and so do the folded coefficients and the chained FMAs, each time by u
    times sum |c v| at most, and a step passes on the difference that it finds
    times sum |c| / divisor.  The field's bound is the oracle's largest value."""
    taps, c = O.taps(name)
    d = O.info(name)["divisor"] if div < 0 else div
    S = float(np.sum(np.abs(np.asarray(c, dtype=np.float64)))) / (d or 1.0)
    u = 2.0 ** -24 if dt == np.float32 else 2.0 ** -53
    err, M = 0.0, float(np.max(np.abs(A)))
    for _ in range(T):
        err = S * err + 1.01 * 2 * (len(taps) + 1) * u * S * (M + err)
        M *= max(1.0, S)
    return err


@pytest.mark.parametrize("name", TILE_NAMES + ["star3d1r", "box3d1r", "j3d27pt"])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_register_tiles_in_fma_mode(name, dt):
    """Every register-tile kernel (kind 5) in FMA mode: several tiles with
    remainders, a shallow and the deepest block, the source's divisor and another;
    within the rounding bound of the C loop, gradient2d (which has no FMA form) bit
    for bit."""
    r = O.info(name)["rad"]
    dim = O.info(name)["dim"]
    for v in pyan5d.variants(name, 0 if dt == np.float32 else 1):
        if v["kind"] != 5:
            continue
        th, tw = v["nw"] * v["cj"] - 2 * r, 64 * v["ck"] - 2 * r
        for bt in sorted({min(2, v["btmax"]), v["btmax"]}):
            for div in (-1.0, 7.0) if name != "gradient2d" else (-1.0,):
                n = [2 * th + 5, tw + 70] if dim == 2 else [19, 2 * th + 1, 130]
                T = bt + 2
                print(f"case tiles FMA {name} {np.dtype(dt).name} variant {v['index']} bt={bt} n={n} divisor={div}",
                      flush=True)
                A = rand_grid(name, n, dt, seed=sum(n) + bt)
                B = A.copy()
                pyan5d.forward_host(name, A, n, T, variant=v["index"], bt=bt, divisor=div, mode=pyan5d.FAST)
                tol = 0.0 if name == "gradient2d" else fma_bound(name, dt, B, n, T, div)
                O.run(name, B, n, T, divisor=div)
                got, ref = A[T % 2].astype(np.float64), B[T % 2].astype(np.float64)
                assert np.max(np.abs(got - ref)) <= tol


def test_box3d_rows_shorter_than_a_run_beside_a_row_of_columns(tmp_path):
    """A grid whose nearest table row names the column kernel, but whose rows are
    shorter than a lane's run: the default path takes the direct kernel, one cell
    more the columns."""
    name, T = "box3d2r", 2
    vs = pyan5d.variants(name, 1)
    cols, = [v["index"] for v in vs if v["kind"] == 4]
    path = tmp_path / "t.tsv"
    path.write_text(f"{name} 1 0 96 96 96 {cols} 1 4 1.0\n")
    pyan5d.tune_clear()
    pyan5d.tune_load(str(path))
    try:
        for n, kind in (([500, 600, 3], 1), ([500, 600, 4], 4)):
            c = pyan5d.resolve_config(name, n, np.float64)
            print("case columns beside a row", name, n, c, flush=True)
            assert vs[c["variant"]]["kind"] == kind
            A = rand_grid(name, n, np.float64, seed=5)
            B = A.copy()
            pyan5d.forward_host(name, A, n, T)
            O.run(name, B, n, T)
            assert same(A[T % 2], B[T % 2])
    finally:
        pyan5d.tune_clear()
        pyan5d.tune_load()
