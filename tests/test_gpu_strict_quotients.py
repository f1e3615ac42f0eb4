"""The strict build's quotients, which share one reciprocal per denominator,
against the oracle's plain divisions, bit for bit: states whose densities,
velocities and energies span many orders of magnitude, with zero and negative
zero momenta, so that the quotients meet every kind of operand."""
import numpy as np
import pytest

import opendynamo_amd as od
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def rough_state(n, seed, dtype):
    """Random points, element by element in one of several units: densities
    1e-4 .. 1e4, Mach numbers 1e-8 .. 2, a quarter of the momenta +0 or -0."""
    rng = np.random.default_rng(seed)
    E, N = n[0] * n[1] * n[2], n[0] * n[1] * n[2] * 64
    rho = np.repeat(10.0 ** rng.uniform(-4.0, 4.0, E), 64) * rng.uniform(0.9, 1.1, N)
    c = np.repeat(10.0 ** rng.uniform(-3.0, 3.0, E), 64)
    mach = np.repeat(10.0 ** rng.uniform(-8.0, 0.3, E), 64)
    m = [rho * c * mach * rng.uniform(-1.0, 1.0, N) for _ in range(3)]
    for q in range(3):
        pick = rng.random(N)
        m[q][pick < 0.125] = 0.0
        m[q][pick > 0.875] = -0.0
    p = rho * c * c / 1.4 * rng.uniform(0.9, 1.1, N)
    e = p / 0.4 + 0.5 * sum(x * x for x in m) / rho
    return np.concatenate([rho, *m, e]).astype(dtype)


@pytest.mark.parametrize("real", [od.OD_F32, od.OD_F64])
@pytest.mark.parametrize("flux", ["slau2", "ausm+", "rusanov"])
@pytest.mark.parametrize("viscous", [True, False])
def test_strict_rhs_of_rough_states_matches_oracle(real, flux, viscous):
    n = (10, 8, 9)
    kw = dict(u_real=real, flux=flux, y_wall=True, viscous=viscous, viscosity_model=1,
              mu_ref=1e-3 if viscous else 0.0)
    dtype = np.float32 if real == od.OD_F32 else np.float64
    with od.Solver(od.params(*n, 6.0, 2.0, 3.0, **kw)) as s:
        for seed in range(3):
            print(f"CASE test=strict_quotients real={real} flux={flux} viscous={viscous} seed={seed}", flush=True)
            u = rough_state(n, seed, dtype)
            s.set_state(u)
            got = s.rhs()
            want = O.rhs_total(O.params(*n, 6.0, 2.0, 3.0, **kw), u)
            assert got.tobytes() == np.asarray(want, dtype=dtype).tobytes()
