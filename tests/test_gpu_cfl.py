"""The CFL time step, whose maximum is taken on the device, and the step size,
which the captured step graphs read from device memory."""
import numpy as np
import pytest

import opendynamo_amd as od
from helpers import smooth_state

pytestmark = pytest.mark.gpu


def cfl_dt(state, box, cfl):
    """The definition, in f64: cfl / (7 max sum_d (|u_d| + c) / dx_d), rounded
    to f32; points without a finite speed do not count."""
    nx, ny, nz, lx, ly, lz = box
    r, ru, rv, rw, e = np.asarray(state, dtype=np.float64).reshape(5, -1)
    with np.errstate(all="ignore"):
        ke = 0.5 * (ru * ru + rv * rv + rw * rw) / r
        c = np.sqrt(1.4 * np.fmax(1e-7, 0.4 * (e - ke)) / r)
        lam = sum((np.abs(m / r) + c) / (float(np.float32(ext)) / n) for m, ext, n in
                  ((ru, lx, nx), (rv, ly, ny), (rw, lz, nz)))
    return float(np.float32(cfl / (7.0 * np.fmax.reduce(lam, initial=0.0))))


# fewer elements than a work-group takes, one more, and more than 1024
# work-groups of four (the groups then go round)
@pytest.mark.parametrize("dims", [(1, 1, 1), (3, 1, 1), (5, 1, 1), (16, 16, 16), (17, 16, 16)],
                         ids=lambda d: "x".join(map(str, d)))
@pytest.mark.parametrize("real", [od.OD_F32, od.OD_F64])
def test_cfl_dt_equals_its_definition(dims, real):
    print(f"CASE test=cfl dims={dims} real={real}", flush=True)
    box = (*dims, 3.0, 2.0, 2.5)
    u = smooth_state(*box, seed=sum(dims), dtype=np.float32 if real == 4 else np.float64).reshape(5, -1)
    with od.Solver(od.params(*box, u_real=real)) as s:
        for at in (0, u.shape[1] // 2, u.shape[1] - 1):  # the fastest point, wherever it lies
            v = u.copy()
            v[1, at] = 3.0 + at % 7
            v[4, at] = 20.0
            s.set_state(v.ravel())
            assert s.cfl_dt(0.3) == cfl_dt(v, box, 0.3)
        v[:, 0] = np.nan  # a point without a speed is passed over
        s.set_state(v.ravel())
        assert s.cfl_dt(0.3) == cfl_dt(v, box, 0.3)


@pytest.mark.parametrize("kw", [dict(u_real=od.OD_F32, fast_math=1), dict(u_real=od.OD_F32, fast_math=0),
                                dict(u_real=od.OD_F64), dict(u_real=od.OD_F32, compute_real=od.OD_F64),
                                dict(u_real=od.OD_F64, compute_real=od.OD_F32, q_real=od.OD_F32,
                                     rhs_real=od.OD_F32, rk_accum=1)],
                         ids=["fast", "strict", "f64", "f32_state", "mixed"])
@pytest.mark.parametrize("viscous", [True, False])
def test_changing_the_step_size_keeps_every_step_its_own(kw, viscous):
    """Steps of changing dt enqueued back to back, through the one-step and the
    eight-step graph, equal the same steps each on a solver of its own."""
    print(f"CASE test=dt_sequence kw={kw} viscous={viscous}", flush=True)
    box = (3, 2, 4, 3.0, 2.0, 4.0)
    p = od.params(*box, y_wall=True, viscous=viscous, mu_ref=2e-3 if viscous else 0.0, **kw)
    u = smooth_state(*box, seed=5, dtype=np.float32 if kw["u_real"] == 4 else np.float64)
    plan = [(2e-3, 1), (1e-3, 8), (2e-3, 9), (1.5e-3, 2), (1e-3, 3)]
    with od.Solver(p) as s:
        s.set_state(u)
        for dt, n in plan:
            s.step(dt, n)
        got = s.get_state()
    for dt, n in plan:
        with od.Solver(p) as s:
            s.set_state(u)
            for _ in range(n):
                s.step(dt, 1)
            u = s.get_state()
    assert got.tobytes() == u.tobytes()
