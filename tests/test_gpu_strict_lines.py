"""The strict visc kernel by lines (four consecutive elements per work-group)
against the oracle, bit for bit: element counts with every remainder by four,
boxes one element wide (an element its own neighbour), rows that end inside a
work-group, walls, and all four combinations of state and compute type."""
import numpy as np
import pytest

import opendynamo_amd as od
from helpers import smooth_state
from oracle import oracle as O

pytestmark = pytest.mark.gpu

TYPES = {"f32": dict(u_real=4), "f64": dict(u_real=8),
         "f64_state": dict(u_real=8, compute_real=4, q_real=4, rhs_real=4, rk_accum=1),
         "f32_state": dict(u_real=4, compute_real=8, q_real=4, rhs_real=4)}


@pytest.mark.parametrize("n", [(1, 1, 1), (2, 1, 1), (1, 3, 1), (1, 1, 5), (3, 2, 1), (3, 3, 1), (5, 2, 3), (4, 3, 2),
                               (7, 3, 5), (3, 5, 7)], ids=lambda d: "x".join(map(str, d)))
@pytest.mark.parametrize("types", list(TYPES))
def test_strict_boxes_equal_the_oracle(n, types):
    box = (*n, 3.0, 2.0, 2.5)
    for wall in (False, True):
        for suth in (0, 1):
            print(f"CASE test=strict_lines n={n} types={types} wall={wall} suth={suth}", flush=True)
            kw = dict(TYPES[types], flux="slau2", y_wall=wall, viscous=True, viscosity_model=suth, mu_ref=2e-3)
            u = smooth_state(*box, seed=sum(n), amp=0.05, dtype=np.float32 if kw["u_real"] == 4 else np.float64)
            po = O.params(*box, **kw)
            with od.Solver(od.params(*box, **kw)) as s:
                s.set_state(u)
                assert s.rhs().tobytes() == np.ascontiguousarray(O.rhs_total(po, u)).tobytes()
                s.step(0.002, 2)
                want = O.step(po, u, float(np.float32(0.002)), 2)
                assert s.get_state().tobytes() == np.ascontiguousarray(want).tobytes()
