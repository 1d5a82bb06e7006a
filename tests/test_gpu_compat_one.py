"""The one-workgroup forms of compat mode's ADsolver and PPESolver against the
oracle, bit for bit (the same operations in the same order): one wave, the
register and the LDS coefficient forms, ragged sizes around their limits, the
launch-by-launch form just above, and a solve longer than one launch."""
import ctypes as C

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


def _fields(nx, ny, lx, ly, stretch):
    def faces(n, length):
        t = np.linspace(0.0, 1.0, n + 1)
        return length * (t + stretch * t * (1.0 - t))
    xf, yf = faces(nx - 2, lx), faces(ny - 2, ly)
    rng = np.random.RandomState(nx * 1000 + ny)
    x, y = np.meshgrid(np.linspace(0, 1, nx), np.linspace(0, 1, ny))
    u = 1.0 + 0.3 * np.sin(5 * x + 2 * y) + 0.01 * rng.standard_normal((ny, nx))
    v = 0.2 * np.cos(3 * x - 4 * y) + 0.01 * rng.standard_normal((ny, nx))
    return xf, yf, u.ravel(), v.ravel()


SIZES = [(4, 4), (10, 7), (32, 16), (33, 16), (52, 52), (64, 64), (65, 64), (63, 90), (90, 63), (300, 27), (8, 900),
         (90, 91), (92, 92)]


@pytest.mark.parametrize("nx,ny", SIZES)
@pytest.mark.parametrize("w", [1.0, 0.8])
def test_compat_ad_one_equals_oracle(require_gpu, nx, ny, w):
    import immerseflow_amd as iff
    xf, yf, u, v = _fields(nx, ny, 1.0, 0.7, 0.2)
    c = iff.Case(xf, yf, mode=iff.IF_MODE_COMPAT, dt=0.002, re=120.0, ad_itermax=7, ad_omega=w)
    c.set("u", u)
    c.set("v", v)
    ou, ov = u.copy(), v.copy()
    uf, vf = np.zeros((nx - 1) * (ny - 2)), np.zeros((nx - 2) * (ny - 1))
    L, ib, r = O.lib(), np.ones(nx * ny), C.c_double()
    for _ in range(3):
        st = c.ad_step()
        it = L.of_compat_ad_step_w(nx, ny, O.dptr(c.dx), O.dptr(c.dy), 0.002, 120.0, 7, w, O.dptr(ib), O.dptr(ou),
                                   O.dptr(ov), O.dptr(uf), O.dptr(vf), C.byref(r))
        assert st["ad_iters"] == it and st["ad_res"] == r.value
    for name, ref in (("u", ou), ("v", ov), ("uf", uf), ("vf", vf)):
        assert np.array_equal(c.get(name), ref), name


@pytest.mark.parametrize("nx,ny,most", [(nx, ny, 150) for nx, ny in SIZES] + [(52, 52, 0), (52, 52, 1), (66, 60, 40000)])
def test_compat_ppe_one_equals_oracle(require_gpu, nx, ny, most):
    import immerseflow_amd as iff
    xf, yf, u, v = _fields(nx, ny, 1.0, 1.0 if most > 1000 else 0.7, 0.0 if most > 1000 else 0.3)
    c = iff.Case(xf, yf, mode=iff.IF_MODE_COMPAT, dt=0.002, re=120.0, ppe_itermax=most)
    p = np.zeros(nx * ny) if most > 1000 else 20.0 * u
    c.set("p", p)
    st = c.ppe_solve()
    r = C.c_double()
    it = O.lib().of_compat_ppe(nx, ny, O.dptr(c.dx), O.dptr(c.dy), most, O.dptr(p), C.byref(r))
    assert st["ppe_sweeps"] == it and st["ppe_res"] == r.value
    assert most <= 1000 or it > 16384  # longer than one launch
    assert np.array_equal(c.get("p"), p)
