"""The fast update kernel with an f64 state, which it loads twice in boxes of up to 4096
tiles and holds in registers in larger ones: both give the same bits, that is, a flow
repeated along z follows the small box it fills.  Tiles of two elements along x: 64 and
18 in the small boxes."""
import numpy as np
import pytest

import opendynamo_amd as od
from helpers import smooth_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, times", [((4, 8, 4), 64), ((4, 8, 4), 65), ((5, 3, 2), 228)],
                         ids=lambda d: "x".join(map(str, d)) if isinstance(d, tuple) else str(d))
@pytest.mark.parametrize("rk_accum", [0, 1])
def test_held_and_reloaded_state_agree(n, times, rk_accum):
    for viscous in (True, False):
        for wall in (True, False):
            print(f"CASE test=held n={n} times={times} rk_accum={rk_accum} viscous={viscous} wall={wall}", flush=True)
            kw = dict(u_real=od.OD_F64, compute_real=od.OD_F32, q_real=od.OD_F32, rhs_real=od.OD_F32, fast_math=1,
                      rk_accum=rk_accum, y_wall=wall, viscous=viscous, mu_ref=2e-3 if viscous else 0.0)
            length = [0.5 * d for d in n]  # elements of side 1/2 in both boxes: the same Jacobians
            u = smooth_state(*n, *length, seed=sum(n), amp=0.05, dtype=np.float64)
            a = u.reshape(5, n[2], -1)
            out = []
            for t in (1, times):
                with od.Solver(od.params(n[0], n[1], n[2] * t, length[0], length[1], length[2] * t, **kw)) as s:
                    s.set_state(np.ascontiguousarray(np.tile(a, (1, t, 1))).ravel())
                    s.step(0.003, 3)
                    out.append(s.get_state().reshape(5, t, -1))
            assert np.isfinite(out[0]).all()
            assert np.array_equal(out[1], np.repeat(out[0], times, axis=1))
