"""The CFL time steps of a batch, whose boxes' maxima are taken in one go: each equals
that of its box alone, bit for bit, in boxes of one work-group, of several and of the
most (1024), next to each other in any order."""
import numpy as np
import pytest

import opendynamo_amd as od
from helpers import smooth_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("real", [od.OD_F32, od.OD_F64])
def test_every_box_has_its_own_time_step(real):
    print(f"CASE test=batch_cfl real={real}", flush=True)
    boxes = [(*n, 3.0, 2.0, 2.5) for n in ((1, 1, 1), (17, 16, 16), (3, 2, 1), (5, 4, 3), (16, 16, 16), (1, 1, 1), (9, 1, 1))]
    rng = np.random.default_rng(3)
    with od.Batch(od.params(1, 1, 1, 1.0, 1.0, 1.0, u_real=real), boxes) as b:
        want = []
        for q, x in enumerate(boxes):
            u = smooth_state(*x, seed=q, dtype=np.float32 if real == od.OD_F32 else np.float64).reshape(5, -1)
            u[1:4, rng.integers(u.shape[1])] = 1.0 + q % 3  # the box's fastest point
            b.set_state(q, u.ravel())
            with od.Solver(od.params(*x, u_real=real)) as s:
                s.set_state(u.ravel())
                want.append(s.cfl_dt(0.3))
        assert len(set(want)) > 4
        assert list(b.cfl_dt(0.3)) == want
