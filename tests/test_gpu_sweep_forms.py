"""The default sweep shapes and the persistent FP64 solve against launches of
one stage and one check each: every form evaluates the same expressions per
cell and takes the same stopping decisions, so the results are the same
bits, at tile edges, odd widths, single tiles, and where the sweeps run out
inside a chunk.  Fields come back through the packed rectangles; a field
that is set reads back as it was set."""
import numpy as np
import pytest

import immerseflow_amd as iff

pytestmark = pytest.mark.gpu

FIELDS = ("u", "v", "p", "uf", "vf")


def _faces(n, length, stretch):
    x = np.linspace(0.0, 1.0, n + 1)
    return length * (x + stretch * np.sin(2.0 * np.pi * x) / (2.0 * np.pi))


def _cases(nx, ny, stretch, moving):
    body = iff.heaving_circle(3.0, 2.0, 0.5, 0.3, 0.5) if moving else iff.circle(3.0, 2.0, 0.5)
    return dict(xf=_faces(nx, 8.0, stretch), yf=_faces(ny, 4.0, 0.0), bodies=[body] if min(nx, ny) > 12 else [])


def _run(g, precision, check, itermax, tol, shape, steps=3):
    with iff.Case(g["xf"], g["yf"], precision=precision, dt=0.002, re=100.0, bodies=g["bodies"], ppe_itermax=itermax,
                  ppe_tol=tol, check_every=check) as c:
        if shape:
            c.tune(shape[0], shape[1], shape[2], check)
        sweeps = [c.step(1)["ppe_sweeps"] for _ in range(steps)]
        st = c.step(1)
        assert st["persistent_timeouts"] == 0 and st["failed"] == 0
        return sweeps + [st["ppe_sweeps"]], st["ppe_res"], {f: c.get(f) for f in FIELDS}


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("nx,ny,check,itermax,stretch,moving", [
    (9, 7, 1, 400, 0.0, False),        # one tile, smaller than its halo
    (64, 48, 10, 4000, 0.0, False),    # one tile
    (80, 64, 12, 4000, 0.0, False),    # exact tiles; a chunk is one whole stage
    (81, 65, 24, 4000, 0.3, False),    # a last tile of one column and row
    (161, 33, 13, 4000, 0.0, True),    # odd width, moving body
    (243, 151, 7, 95, 0.3, False),     # the sweeps run out inside a chunk
    (401, 260, 160, 3000, 0.0, False),
])
def test_default_form_equals_stages(precision, nx, ny, check, itermax, stretch, moving):
    prec = {"fp64": iff.IF_FP64, "mixed": iff.IF_MIXED}[precision]
    g = _cases(nx, ny, stretch, moving)
    a = _run(g, prec, check, itermax, 1e-7, None)
    b = _run(g, prec, check, itermax, 1e-7, (3, 32, 4))  # 8-wave tiles: a launch per stage
    assert a[0] == b[0] and a[1] == b[1]
    for f in FIELDS:
        assert np.array_equal(a[2][f], b[2][f]), f


def test_fp64_batch_solves_end_apart():
    """Cases of one persistent FP64 solve stop at their own checks."""
    grids = [_cases(64, 48, 0.0, False), _cases(243, 90, 0.0, True), _cases(130, 131, 0.3, False)]
    b = iff.Batch(iff.IF_FP64)
    try:
        slots = [b.add(g["xf"], g["yf"], 4, dt=0.002, re=100.0, bodies=g["bodies"], ppe_tol=1e-6, ppe_itermax=3000,
                       check_every=10) for g in grids]
        b.step(4)
        for s, g in zip(slots, grids):
            alone = _run(g, iff.IF_FP64, 10, 3000, 1e-6, (3, 32, 4))
            assert b.state(s)[2]["ppe_sweeps"] == alone[0][-1]
            for f in FIELDS:
                assert np.array_equal(b.get(s, f), alone[2][f]), f
    finally:
        b.close()


@pytest.mark.parametrize("precision", ["fp64", "mixed", "mixed_v32"])
@pytest.mark.parametrize("nx,ny", [(4, 4), (7, 300), (257, 5), (130, 131)])
def test_fields_round_trip(precision, nx, ny):
    prec = {"fp64": iff.IF_FP64, "mixed": iff.IF_MIXED, "mixed_v32": iff.IF_MIXED_V32}[precision]
    rng = np.random.default_rng(3)
    with iff.Case(_faces(nx, 8.0, 0.0), _faces(ny, 4.0, 0.0), precision=prec, dt=0.002, re=100.0) as c:
        want = {}
        for f in FIELDS:
            want[f] = rng.standard_normal(c.get(f).size).astype(np.float32).astype(np.float64)
            c.set(f, want[f])
        for f in FIELDS:
            assert np.array_equal(c.get(f), want[f]), f
        assert np.all(c.get("iblank") == (c.get("flags").astype(np.uint8) & 1))


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("nx,ny,check", [
    (5, 4, 1),        # fewer cells than lanes
    (128, 33, 2),     # 2 cells a lane; a chunk is one stage, split for its parity
    (129, 60, 7),     # 3, and a last segment of one cell
    (256, 24, 40),    # 4
    (300, 41, 9),     # 5
    (384, 100, 3),    # 6
    (430, 9, 5),      # 7
    (512, 50, 12),    # 8, the most
    (520, 20, 6),     # 9: one launch per colour in both
])
def test_persistent_line_equals_launches(precision, nx, ny, check):
    prec = {"fp64": iff.IF_FP64, "mixed": iff.IF_MIXED}[precision]
    g = _cases(nx, ny, 0.2, nx == 256)
    out = []
    for persistent in (True, False):
        with iff.Case(g["xf"], g["yf"], precision=prec, dt=0.002, re=100.0, bodies=g["bodies"], ppe_tol=1e-8,
                      ppe_solver=iff.IF_PPE_LINE, ppe_omega=1.5, ppe_itermax=235, check_every=check) as c:
            c.persistent(persistent)
            st = [c.step(1) for _ in range(3)]
            assert all(s["persistent_timeouts"] == 0 for s in st)
            out.append(([s["ppe_sweeps"] for s in st], [s["ppe_res"] for s in st], {f: c.get(f) for f in FIELDS}))
    assert out[0][:2] == out[1][:2]
    for f in FIELDS:
        assert np.array_equal(out[0][2][f], out[1][2][f]), f


def test_autotune_times_open_cases():
    """The autotuner times sweeps that run.  One is two dependent half-sweeps
    with a block barrier each, which take over 100 ns between them; launches over
    a closed case take a few us for 256 sweeps, 10 to 20 ns each."""
    n = 256
    xf = _faces(n, 8.0, 0.0)
    with iff.Case(xf, xf.copy(), precision=iff.IF_MIXED, dt=0.002, re=100.0, ppe_itermax=320, check_every=160) as c:
        c.step(1)
        assert c.autotune()["sweep_ns"] * n * n > 50.0
        st = c.step(1)
        assert st["persistent_timeouts"] == 0 and st["failed"] == 0
