"""Every default shape against launches of one stage and one check each, bit for
bit, on grids just large enough to get it: the shape rule goes by tile counts
(reg_auto_shape), so each shape's own tile edges, strip reach and form of
exchange are run.  Beside them the persistent forms that only mixed sets of
cases take, and the line solver's give-up path."""
import numpy as np
import pytest

import immerseflow_amd as iff

pytestmark = pytest.mark.gpu

FIELDS = ("u", "v", "p", "uf", "vf")
MIXED, FP64 = iff.IF_MIXED, iff.IF_FP64


def _faces(n, length, stretch):
    x = np.linspace(0.0, 1.0, n + 1)
    return length * (x + stretch * np.sin(2.0 * np.pi * x) / (2.0 * np.pi))


def _grid(nx, ny, stretch):
    return dict(xf=_faces(nx, 16.0, stretch), yf=_faces(ny, 16.0 * ny / nx, 0.0),
                bodies=[iff.circle(5.0, 8.0 * ny / nx, 0.12 * 16.0 * min(nx, ny) / nx)])


def _alone(g, precision, check, itermax, persistent, shape=None, steps=2, **kw):
    with iff.Case(g["xf"], g["yf"], precision=precision, dt=0.001, re=100.0, bodies=g["bodies"], ppe_itermax=itermax,
                  ppe_tol=1e-9, check_every=check, **kw) as c:
        if shape:
            c.tune(*shape, check)
        c.persistent(persistent)
        st = [c.step(1) for _ in range(steps)]
        assert all(s["persistent_timeouts"] == 0 and s["failed"] == 0 for s in st)
        return [s["ppe_sweeps"] for s in st], st[-1]["ppe_res"], {f: c.get(f) for f in FIELDS}


@pytest.mark.parametrize("precision,nx,ny,stretch", [
    (MIXED, 611, 600, 0.0),     # 32 x 16
    (MIXED, 601, 610, 0.3),
    (MIXED, 801, 790, 0.0),     # 48 x 12
    (MIXED, 799, 801, 0.3),
    (MIXED, 1101, 1000, 0.0),   # 64 x 8, a tile a CU
    (MIXED, 1301, 1350, 0.0),   # 96 x 8, a tile a CU
    (MIXED, 1949, 1001, 0.3),
    (MIXED, 1601, 1500, 0.0),   # 64 x 8, two tiles a CU
    (MIXED, 1601, 1500, 0.3),
    (MIXED, 1949, 1800, 0.0),   # 96 x 8, two tiles a CU
    (FP64, 701, 690, 0.0),      # 32 x 8
    (FP64, 651, 701, 0.3),
    (FP64, 1001, 990, 0.0),     # 48 x 8
    (FP64, 999, 1001, 0.3),
    (FP64, 1101, 1110, 0.0),    # 64 x 8
    (FP64, 1401, 1390, 0.0),    # 80 x 4
    (FP64, 2041, 1001, 0.3),
])
def test_default_shape_equals_stages(require_gpu, precision, nx, ny, stretch):
    print("[gpu-test] default shape", precision, nx, ny, stretch, flush=True)
    g = _grid(nx, ny, stretch)
    a = _alone(g, precision, 37, 163, True)
    b = _alone(g, precision, 37, 163, False, (3, 32, 4))
    assert a[:2] == b[:2] and a[0] == [163, 163]
    for f in FIELDS:
        assert np.array_equal(a[2][f], b[2][f]), f


def test_mixed_weights_on_polled_strips(require_gpu):
    """A uniform and a stretched grid side by side (each case its own form of
    the update), in one persistent launch."""
    print("[gpu-test] mixed weights, default shape", flush=True)
    grids = [_grid(300, 200, 0.0), _grid(243, 151, 0.3)]
    b = iff.Batch(MIXED)
    try:
        slots = [b.add(g["xf"], g["yf"], 2, dt=0.001, re=100.0, bodies=g["bodies"], ppe_itermax=210, ppe_tol=1e-9)
                 for g in grids]
        b.step(2)   # (a batch checks every 10 sweeps)
        for s, g in zip(slots, grids):
            ref = _alone(g, MIXED, 10, 210, False, (3, 32, 4))
            assert b.state(s)[2]["ppe_sweeps"] == ref[0][-1]
            for f in FIELDS:
                assert np.array_equal(b.get(s, f), ref[2][f]), f
    finally:
        b.close()


@pytest.mark.parametrize("precision", [FP64, MIXED])
def test_chunks_beside_other_solvers(require_gpu, precision):
    """Red-black cases beside a line and a Jacobi case: plain persistent chunks
    with a check each, not one launch a solve."""
    print("[gpu-test] persistent chunks beside other solvers", precision, flush=True)
    # (point Jacobi diverges beyond omega = 1)
    grids = [(_grid(300, 200, 0.0), iff.IF_PPE_RBSOR, 1.5), (_grid(201, 190, 0.0), iff.IF_PPE_RBSOR, 1.5),
             (_grid(129, 100, 0.2), iff.IF_PPE_LINE, 1.5), (_grid(64, 50, 0.0), iff.IF_PPE_JACOBI, 1.0)]
    b = iff.Batch(precision)
    try:
        slots = [b.add(g["xf"], g["yf"], 2, dt=0.001, re=100.0, bodies=g["bodies"], ppe_itermax=205, ppe_tol=1e-9,
                       ppe_solver=solver, ppe_omega=omega) for g, solver, omega in grids]
        b.step(2)
        for s, (g, solver, omega) in zip(slots, grids):
            ref = _alone(g, precision, 10, 205, False, (3, 32, 4), ppe_solver=solver, ppe_omega=omega)
            assert b.state(s)[2]["ppe_sweeps"] == ref[0][-1]
            for f in FIELDS:
                assert np.array_equal(b.get(s, f), ref[2][f]), f
    finally:
        b.close()


@pytest.mark.parametrize("precision", [FP64, MIXED])
def test_line_timeout_resolves_per_colour(require_gpu, monkeypatch, precision):
    """The line solver's chunks with a wait limit of one tick: the kernel ends,
    the step solves again with a launch per colour and reports it."""
    print("[gpu-test] line solver time-out path", precision, flush=True)
    monkeypatch.setenv("IFF_PERSISTENT_TIMEOUT_TICKS", "1")
    g = _grid(256, 200, 0.0)
    with iff.Case(g["xf"], g["yf"], precision=precision, dt=0.001, re=100.0, bodies=g["bodies"], ppe_solver=iff.IF_PPE_LINE,
                  ppe_omega=1.7, ppe_itermax=20000, ppe_tol=1e-6, check_every=40) as c:
        st = c.step(1)
        assert st["persistent_timeouts"] == 1 and st["failed"] == 0
        assert st["ppe_res"] <= 1e-6 and st["div_max"] <= 1e-6
        st = c.step(1)
        assert st["persistent_timeouts"] == 0 and st["ppe_res"] <= 1e-6 and st["div_max"] <= 1e-6
