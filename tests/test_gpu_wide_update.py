"""The update kernel's wide form (more waves than elements, small boxes) against
the oracle bit for bit in the strict build: viscous boxes and Euler ones, whose
volume part it forms beside the faces, at the smallest boxes, odd rows, walls and
every combination of state and compute type; and its edge against the narrow form
and the fast build's tiles through repetition (a flow repeated along z fills a
larger box, which the narrow form takes, with the same element sizes)."""
import numpy as np
import pytest

import opendynamo_amd as od
from helpers import smooth_state
from oracle import oracle as O

pytestmark = pytest.mark.gpu

TYPES = {"f32": dict(u_real=4), "f64": dict(u_real=8),
         "f64_state": dict(u_real=8, compute_real=4, q_real=4, rhs_real=4, rk_accum=1),
         "f32_state": dict(u_real=4, compute_real=8, q_real=4, rhs_real=4)}


def dtype_of(kw):
    return np.float32 if kw["u_real"] == 4 else np.float64


@pytest.mark.parametrize("n", [(1, 1, 1), (2, 1, 1), (1, 2, 3), (3, 2, 2), (5, 4, 3)],
                         ids=lambda d: "x".join(map(str, d)))
@pytest.mark.parametrize("types", list(TYPES))
def test_wide_form_equals_the_oracle(n, types):
    box = (*n, 3.0, 2.0, 2.5)
    for flux, viscous, wall in (("slau2", False, False), ("ausm+", False, True), ("rusanov", False, False),
                                ("slau2", True, True)):
        print(f"CASE test=wide n={n} types={types} flux={flux} viscous={viscous} wall={wall}", flush=True)
        kw = dict(TYPES[types], flux=flux, y_wall=wall, viscous=viscous, viscosity_model=1, mu_ref=2e-3)
        u = smooth_state(*box, seed=sum(n), amp=0.05, dtype=dtype_of(kw))
        po = O.params(*box, **kw)
        with od.Solver(od.params(*box, **kw)) as s:
            s.set_state(u)
            assert s.rhs().tobytes() == np.ascontiguousarray(O.rhs_total(po, u)).tobytes()
            s.step(0.002, 2)
            want = O.step(po, u, float(np.float32(0.002)), 2)
            assert s.get_state().tobytes() == np.ascontiguousarray(want).tobytes()


# tiles per layer (x in pairs) times nz: just below and above both limits (512, 1024)
@pytest.mark.parametrize("n, times", [((5, 3, 2), 28), ((5, 3, 2), 29), ((7, 8, 2), 16), ((7, 8, 2), 17), ((1, 9, 2), 40)],
                         ids=lambda d: "x".join(map(str, d)) if isinstance(d, tuple) else str(d))
@pytest.mark.parametrize("types", ["f32", "f64", "fast_f64_state", "fast"])
def test_wide_and_narrow_form_agree(n, times, types):
    base = {"fast": dict(u_real=4, fast_math=1), "fast_f64_state": dict(TYPES["f64_state"], fast_math=1)}
    for viscous in (True, False):
        print(f"CASE test=wide_edge n={n} times={times} types={types} viscous={viscous}", flush=True)
        kw = dict(base.get(types, TYPES.get(types)), flux="slau2", y_wall=True, viscous=viscous,
                  mu_ref=2e-3 if viscous else 0.0)
        length = [0.5 * d for d in n]  # powers of two times n: the same Jacobians in both boxes
        u = smooth_state(*n, *length, seed=sum(n), amp=0.05, dtype=dtype_of(kw))
        a = u.reshape(5, n[2], -1)
        out = []
        for t in (1, times):
            p = od.params(n[0], n[1], n[2] * t, length[0], length[1], length[2] * t, **kw)
            with od.Solver(p) as s:
                s.set_state(np.ascontiguousarray(np.tile(a, (1, t, 1))).ravel())
                s.step(0.003, 3)
                out.append(s.get_state().reshape(5, t, -1))
        assert np.isfinite(out[0]).all()
        for t in range(times):
            assert out[1][:, t].tobytes() == out[0][:, 0].tobytes()


# blocks of the fast build's visc kernel below and above its wide form's limit (256)
@pytest.mark.parametrize("n, times", [((2, 2, 2), 257), ((8, 8, 8), 5), ((4, 16, 16), 2)],
                         ids=lambda d: "x".join(map(str, d)) if isinstance(d, tuple) else str(d))
def test_wide_and_narrow_blocks_agree(n, times):
    for wall, eddy in ((False, False), (True, True)):
        print(f"CASE test=wide_blocks n={n} times={times} wall={wall}", flush=True)
        kw = dict(u_real=4, fast_math=1, flux="slau2", y_wall=wall, mu_ref=2e-3, viscosity_model=1)
        length = [0.5 * d for d in n]  # powers of two times n: the same Jacobians in both boxes
        u = smooth_state(*n, *length, seed=sum(n), amp=0.05, dtype=np.float32)
        a, mu = u.reshape(5, n[2], -1), np.random.default_rng(2).uniform(0.0, 3e-3, (n[2], n[1] * n[0]))
        out = []
        for t in (1, times):
            with od.Solver(od.params(n[0], n[1], n[2] * t, length[0], length[1], length[2] * t, **kw)) as s:
                s.set_state(np.ascontiguousarray(np.tile(a, (1, t, 1))).ravel())
                if eddy:
                    s.set_eddy_viscosity(np.tile(mu, (t, 1)).ravel())
                s.step(0.003, 3)
                out.append(s.get_state().reshape(5, t, -1))
        assert np.isfinite(out[0]).all()
        for t in range(times):
            assert out[1][:, t].tobytes() == out[0][:, 0].tobytes()
