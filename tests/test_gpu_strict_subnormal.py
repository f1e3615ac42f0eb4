"""The strict f32 build's quotients where they are subnormal, bit for bit against
the oracle's divisions: there a quotient can lie exactly in the middle between two
f32 numbers, which a product with a reciprocal must still round to even.

Density (234) and energy are uniform, so that the mass and energy equations hold
nothing but the y momentum, a random multiple of 2^-149 up to 2^-125: one velocity
in 234 is such a middle."""
import numpy as np
import pytest

import opendynamo_amd as od
from oracle import oracle as O

pytestmark = pytest.mark.gpu

RHO = 234.0


def tiny_state(n, seed, dtype):
    rng = np.random.default_rng(seed)
    u = np.zeros((5, n[0] * n[1] * n[2] * 64), np.float32)
    u[0], u[4] = RHO, 37.5
    u[2] = np.ldexp(rng.integers(-2 ** 24 + 1, 2 ** 24, u.shape[1]).astype(np.float64), -149)
    return u.ravel().astype(dtype)


def test_the_state_has_middles_a_product_misses():
    """Without a correction (a y in f64, y the nearest f64 number to 1 / b) some of
    the velocities round the wrong way."""
    v = tiny_state((4, 4, 4), 0, np.float32).reshape(5, -1)[2]
    product = (v.astype(np.float64) * (1.0 / RHO)).astype(np.float32)
    assert np.count_nonzero(product != v / np.float32(RHO)) > 2


@pytest.mark.parametrize("n", [(5, 4, 3), (16, 18, 18)], ids=["tiles", "blocks"])
@pytest.mark.parametrize("flux", ["slau2", "ausm+", "rusanov"])
@pytest.mark.parametrize("u_real", [od.OD_F32, od.OD_F64])
def test_subnormal_quotients_match_the_oracle(n, flux, u_real):
    kw = dict(u_real=u_real, compute_real=od.OD_F32, q_real=od.OD_F32, rhs_real=od.OD_F32, flux=flux, y_wall=False)
    for viscous in (False, True):
        print(f"CASE test=strict_subnormal n={n} flux={flux} u_real={u_real} viscous={viscous}", flush=True)
        flags = dict(kw, viscous=viscous, mu_ref=1e-3 if viscous else 0.0)
        u = tiny_state(n, sum(n), np.float32 if u_real == od.OD_F32 else np.float64)
        with od.Solver(od.params(*n, 2.0, 2.0, 2.0, **flags)) as s:
            s.set_state(u)
            got = s.rhs().reshape(5, -1)
        want = O.rhs_total(O.params(*n, 2.0, 2.0, 2.0, **flags), u).reshape(5, -1)
        assert 0.0 < np.max(np.abs(want[0])) < 1e-30  # the momentum's own size
        wrong = [int(np.count_nonzero(g.view(np.uint32) != w.view(np.uint32))) for g, w in zip(got, want)]
        assert wrong == [0] * 5, wrong
