"""The autotuner against the default shapes: they are candidates, timed in the
form they run in, and what it returns can be set by hand."""
import time

import numpy as np
import pytest

import immerseflow_amd as iff

pytestmark = pytest.mark.gpu

FIELDS = ("u", "v", "p", "uf", "vf")


def _case(n, precision, itermax, ny=None, **kw):
    xf = np.linspace(0.0, 20.0, n + 1)
    yf = xf.copy() if ny is None else np.linspace(0.0, 20.0 * ny / n, ny + 1)
    return iff.Case(xf, yf, precision=precision, dt=0.2 * 20.0 / n, re=300.0, bodies=[iff.circle(6.0, 4.0, 0.5)],
                    ppe_itermax=itermax, ppe_tol=1e-30, check_every=160, **kw)


def _in_turn(both, steps):
    """The fastest of eight calls of steps steps of each, in turn."""
    took = [1e9, 1e9]
    for _ in range(8):
        for k, c in enumerate(both):
            t0 = time.perf_counter()
            c.step(steps)
            took[k] = min(took[k], time.perf_counter() - t0)
    return took


@pytest.mark.parametrize("precision,n", [
    (iff.IF_MIXED, 256),   # default 16 x 12
    (iff.IF_MIXED, 611),   # 32 x 16
    (iff.IF_MIXED, 800),   # 48 x 12
    (iff.IF_FP64, 256),    # 16 x 12
    (iff.IF_FP64, 1400),   # 80 x 4
])
def test_tuned_step_is_no_slower(require_gpu, precision, n):
    """Steps of 3,200 sweeps, checked every 160, of an untuned and a tuned case
    in turn: the shapes of the list alone were 8 % (mixed 800^2) to 60 % (FP64
    1400^2) slower than these defaults.  Steps repeat within 1 %; the bound leaves
    5 %."""
    print("[gpu-test] tuned against default", precision, n, flush=True)
    with _case(n, precision, 3200) as a, _case(n, precision, 3200) as b:
        a.step(2)
        b.step(2)
        r = b.autotune()
        b.tune(r["kernel"], r["tile_y"], r["sweeps_per_launch"], 160)
        took = _in_turn((a, b), 2)
        assert took[1] <= 1.05 * took[0], r


@pytest.mark.parametrize("precision", [iff.IF_MIXED, iff.IF_FP64])
def test_default_shapes_can_be_set(require_gpu, precision):
    """The default's low tiles are accepted where the precision has them and
    refused where not, and give the bits of other shapes, persistent or one
    launch a stage."""
    print("[gpu-test] default shapes set by hand", precision, flush=True)
    own = [(4, 16, 12)] + ([(4, 48, 8)] if precision == iff.IF_FP64 else [(4, 32, 16), (4, 48, 12)])
    other = [(4, 32, 16), (4, 48, 12)] if precision == iff.IF_FP64 else [(4, 48, 8)]
    out = []
    for shape in [(3, 32, 4)] + own:
        for persistent in (True, False):
            with _case(401, precision, 333, 170) as c:
                for bad in other:
                    with pytest.raises(iff.ImmerseFlowError):
                        c.tune(*bad, 160)
                c.tune(*shape, 40)
                c.persistent(persistent)
                st = [c.step(1) for _ in range(2)]
                assert all(s["persistent_timeouts"] == 0 for s in st)
                out.append(([s["ppe_sweeps"] for s in st], {f: c.get(f) for f in FIELDS}))
    for sweeps, fields in out[1:]:
        assert sweeps == out[0][0]
        for f in FIELDS:
            assert np.array_equal(fields[f], out[0][1][f]), f


def test_batch_keeps_following_its_cases(require_gpu):
    """A batch whose default shape is not beaten keeps choosing it by its
    cases: after one small case was tuned, a step with a large one beside it
    takes no longer than in a batch that was never tuned."""
    print("[gpu-test] a tuned batch follows its resident set", flush=True)

    def add(b, n):
        xf = np.linspace(0.0, 20.0, n + 1)
        return b.add(xf, xf.copy(), 1000, dt=0.2 * 20.0 / n, re=300.0, bodies=[iff.circle(6.0, 10.0, 0.5)],
                     ppe_itermax=1600, ppe_tol=1e-30)

    plain, tuned = iff.Batch(iff.IF_MIXED), iff.Batch(iff.IF_MIXED)
    try:
        for b in (plain, tuned):
            add(b, 256)
            b.step(1)
        r = tuned.autotune()
        assert (r["kernel"], r["tile_y"], r["sweeps_per_launch"]) == (4, 16, 12)  # 0.56 us a sweep, others 0.65 up
        for b in (plain, tuned):
            add(b, 1600)
            b.step(2)
        # (check intervals differ: 10 sweeps before, about 300 after)
        took = _in_turn((plain, tuned), 1)
        assert took[1] <= 1.05 * took[0]
    finally:
        plain.close()
        tuned.close()
