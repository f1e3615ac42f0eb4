"""The timing calls at dt = 0, which they take: each stage then blends the state
with itself, so the state stays what it was, up to the blend's own rounding.
Neither the step size of earlier steps nor what earlier contexts left in device
memory may come in."""
import numpy as np
import pytest

import opendynamo_amd as od
from helpers import smooth_state
from oracle import oracle as O

pytestmark = pytest.mark.gpu

BOX = (3, 2, 4, 3.0, 2.0, 4.0)
N = 9  # steps: one eight-step graph and one more


def same(a, b):
    return bool(a.tobytes() == b.tobytes())


def advance(s, call):
    if call == "steps":
        s.time_steps(0.0, N)
    else:
        s.time_kernels(0.0, N)
    return s.get_state()


@pytest.mark.parametrize("call", ["steps", "kernels"])
@pytest.mark.parametrize("kw", [dict(u_real=od.OD_F32), dict(u_real=od.OD_F64),
                                dict(u_real=od.OD_F64, compute_real=od.OD_F32, q_real=od.OD_F32,
                                     rhs_real=od.OD_F32, rk_accum=1), dict(u_real=od.OD_F32, fast_math=1)],
                         ids=["f32", "f64", "mixed", "fast"])
@pytest.mark.parametrize("viscous", [True, False])
def test_timing_at_dt_zero(call, kw, viscous):
    print(f"CASE test=dt_zero call={call} kw={kw} viscous={viscous}", flush=True)
    flags = dict(kw, y_wall=True, viscous=viscous, mu_ref=2e-3 if viscous else 0.0)
    p = od.params(*BOX, **flags)
    u = smooth_state(*BOX, seed=6, dtype=np.float32 if kw["u_real"] == od.OD_F32 else np.float64)
    with od.Solver(p) as s:  # leaves its step size in device memory that the next context may get
        s.set_state(u)
        s.step(1e-3, N)
        s.synchronize()
    got = []
    with od.Solver(p) as s:  # no step yet
        s.set_state(u)
        got.append(advance(s, call))
    with od.Solver(p) as s:  # after steps of another size
        s.set_state(u)
        s.step(1e-3, 1)
        s.set_state(u)
        got.append(advance(s, call))
        s.set_state(u)
        s.step(1e-3, 3)
        after = s.get_state()
    with od.Solver(p) as s:
        s.set_state(u)
        s.step(1e-3, 3)
        assert same(s.get_state(), after)  # and the next steps have their own again
    assert same(got[0], got[1])
    if kw.get("fast_math"):
        # three stages, each a sum of two products with coefficients rounded once: at
        # most four roundings of the state's own size a stage
        assert np.all(np.abs(got[0] - u) <= 12 * N * 2.0 ** -24 * np.abs(u))
    else:
        flags.pop("fast_math", None)
        want = O.step(O.params(*BOX, **flags), u, 0.0, N)
        assert same(got[0], np.ascontiguousarray(want))
