"""The step loop's bookkeeping: a step that returns has ended for every case,
however many viscous iterations and sweeps its cases take or are allowed."""
import numpy as np
import pytest

import immerseflow_amd as iff
import oracle_lib as O

pytestmark = pytest.mark.gpu

FIELDS = ("u", "v", "p", "uf", "vf")
# a creeping flow: dt / (re dx^2) = 10, so that a viscous loop takes hundreds
# of iterations
SLOW = dict(dt=0.05, re=0.05, ad_tol=1e-6)


def _faces(n):
    return np.linspace(0.0, 20.0, n + 1)


@pytest.mark.parametrize("precision", [iff.IF_FP64, iff.IF_MIXED])
def test_step_without_sweeps_ends(require_gpu, precision):
    """No Poisson sweep allowed, and more viscous iterations than a step
    enqueues at first: the step still projects, as with one launch per stage."""
    print("[gpu-test] no sweeps, long viscous loop", precision, flush=True)
    out = []
    for persistent in (True, False):
        with iff.Case(_faces(64), _faces(48), precision=precision, bodies=[iff.circle(6.0, 10.0, 2.0)], ad_itermax=120,
                      ppe_itermax=0, check_every=10, **SLOW) as c:
            c.persistent(persistent)
            st = [c.step(1) for _ in range(2)]
            assert [s["ad_iters"] for s in st] == [120, 120]
            out.append(([s["div_max"] for s in st], {f: c.get(f) for f in FIELDS}))
    assert out[0][0] == out[1][0] and min(out[0][0]) > 0.0
    for f in FIELDS:
        assert np.array_equal(out[0][1][f], out[1][1][f]), f


def test_timeout_leaves_open_viscous_loops(require_gpu, monkeypatch):
    """A neighbour wait of one case gives up (a limit of one tick, as in
    test_gpu_timeout) while another case is still in its viscous loop and takes
    more sweeps afterwards: both end their step, and the second one, a single
    tile that waits for nobody, with the bits of per-stage launches."""
    print("[gpu-test] time-out beside an open viscous loop", flush=True)
    out = []
    for persistent in (True, False):
        if persistent:
            monkeypatch.setenv("IFF_PERSISTENT_TIMEOUT_TICKS", "1")
        else:
            monkeypatch.delenv("IFF_PERSISTENT_TIMEOUT_TICKS")
        b = iff.Batch(iff.IF_MIXED)
        try:
            b.tune(4, 64, 8, 40)
            b.persistent(persistent)
            wide = b.add(_faces(400), _faces(400), 3, dt=0.01, re=100.0, bodies=[iff.circle(6.0, 10.0, 0.5)],
                         ppe_tol=1e-6, ppe_itermax=80)
            slow = b.add(_faces(64), _faces(64), 3, bodies=[iff.circle(6.0, 10.0, 2.0)], ad_itermax=300, ppe_tol=1e-9,
                         ppe_itermax=4000, **SLOW)
            for k in range(2):
                b.step(1)
                assert [b.state(s)[:2] for s in (wide, slow)] == [(0, k + 1), (0, k + 1)]
                assert b.state(slow)[2]["ad_iters"] == 300 and b.state(slow)[2]["ppe_sweeps"] > 80
            assert b.state(wide)[2]["div_max"] < 1e300
            out.append((b.state(slow)[2]["ppe_sweeps"], {f: b.get(slow, f) for f in FIELDS}))
        finally:
            b.close()
    assert out[0][0] == out[1][0]
    for f in FIELDS:
        assert np.array_equal(out[0][1][f], out[1][1][f]), f


@pytest.mark.parametrize("precision", [iff.IF_FP64, iff.IF_MIXED])
def test_stage_counters_start_again(require_gpu, precision):
    """With nearly 2^31 sweeps allowed a step, the stage counters of the
    persistent sweep are zeroed before every third: the bits of per-stage
    launches still."""
    print("[gpu-test] stage counters zeroed between steps", precision, flush=True)
    out = []
    for persistent in (True, False):
        with iff.Case(_faces(300), _faces(210), precision=precision, dt=0.01, re=100.0,
                      bodies=[iff.circle(6.0, 10.0, 0.5)], ppe_tol=1e-5, ppe_itermax=2**31 - 5000, check_every=30) as c:
            c.persistent(persistent)
            st = [c.step(1) for _ in range(4)] + [c.step(5)]
            assert all(s["persistent_timeouts"] == 0 and s["failed"] == 0 for s in st)
            out.append(([s["total_ppe_sweeps"] for s in st], {f: c.get(f) for f in FIELDS}))
    assert out[0][0] == out[1][0]
    for f in FIELDS:
        assert np.array_equal(out[0][1][f], out[1][1][f]), f


@pytest.mark.parametrize("nbody,apart", [(4, False), (9, True)])
def test_ghost_cells_of_the_iterate(require_gpu, nbody, apart):
    """The ghost cells of a viscous iterate, set beside the stopping rule or,
    where a case has more than 512, in a launch of their own: the oracle's
    fields (same expressions in FP64, other reduction orders: 1e-10 relative)."""
    print("[gpu-test] ghost cells of the viscous iterate", nbody, flush=True)
    xf, yf = np.linspace(0.0, 16.0, 161), np.linspace(0.0, 13.0, 131)
    bodies = [iff.circle(3.0 + 4.5 * (k % 3), 2.5 + 4.0 * (k // 3), 1.4 + 0.01 * k) for k in range(nbody)]
    prm = dict(dt=0.01, re=100.0, conv_factor=0.5, ubc=1.0, vbc=0.0, ad_itermax=25, ad_tol=1e-6, ppe_solver=1,
               ppe_omega=1.8, ppe_itermax=200, ppe_tol=1e-9, check_every=10)
    oc = O.PhysCase(xf, yf, [dict(b, c=b.get("cth", 1.0), s=b.get("sth", 0.0)) for b in bodies], prm)
    with iff.Case(xf, yf, precision=iff.IF_FP64, bodies=bodies, **prm) as c:
        assert c.ghosts()[2] == oc.ng and (oc.ng > 512) == apart
        g, o = c.step(3), oc.step(3)[-1]
        assert g["ad_iters"] == o[0] and g["ppe_sweeps"] == o[2]
        for name in FIELDS:
            ref = getattr(oc, name)
            err = np.max(np.abs(c.get(name) - ref)) / max(1.0, np.max(np.abs(ref)))
            assert err <= 1e-10, (name, err)


def test_timeout_captures_its_chunk_again(require_gpu, monkeypatch):
    """Beside a Jacobi case a chunk is several launches, replayed from a graph
    that holds the persistent one.  A forced time-out captures it anew within the
    step: the Jacobi case, which waits for nobody, is solved again from its start
    and ends like the others at its stop level, and later steps replay the new
    graph."""
    print("[gpu-test] time-out with a captured chunk", flush=True)
    monkeypatch.setenv("IFF_PERSISTENT_TIMEOUT_TICKS", "1")
    b = iff.Batch(iff.IF_MIXED)
    try:
        b.tune(4, 64, 8, 40)
        wide = b.add(_faces(400), _faces(400), 9, dt=0.01, re=100.0, bodies=[iff.circle(6.0, 10.0, 0.5)],
                     ppe_tol=1e-5, ppe_itermax=20000)
        jac = b.add(_faces(64), _faces(64), 9, dt=0.01, re=100.0, bodies=[iff.circle(6.0, 10.0, 2.0)],
                    ppe_solver=iff.IF_PPE_JACOBI, ppe_omega=1.0, ppe_tol=1e-4, ppe_itermax=40000)
        for k in range(6):
            b.step(1)
            for s, tol in ((wide, 1e-5), (jac, 1e-4)):
                state, steps, st = b.state(s)
                assert (state, steps) == (0, k + 1) and st["failed"] == 0
                assert st["ppe_res"] <= tol and st["ppe_sweeps"] > 0 and st["div_max"] <= 1.01 * tol
    finally:
        b.close()
