"""The static line's step against the oracle, to the bit, at the lengths where its wavefronts (60 slots each, two more at each
end) begin and end, with every wall, order and limiter, the fused step and the plain one.
"""
import numpy as np
import pytest

import oracle
from luna_hydro import hydro, problems

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [3, 4, 59, 60, 61, 62, 63, 119, 120, 121, 182])
@pytest.mark.parametrize("kw", [
    {"periodic": True, "limiter": "vanleer"},
    {"walls": ("reflective", "outflow"), "limiter": "face"},
    {"walls": ("outflow", "reflective"), "limiter": "minmod", "riemann": "hll"},
    {"walls": ("reflective", "reflective"), "order": 0},
], ids=["periodic", "reflective-outflow", "outflow-reflective-hll", "reflective-order0"])
def test_steps_match_oracle(n, kw):
    keys, step, period = problems.line_keys(problems.line_points(n, 1.0, 0.6, seed=n), 1.0)
    rng = np.random.Generator(np.random.MT19937(n))
    gpu, orc = hydro.Line(keys, period, step, 1.4, **kw), oracle.Line(keys, period, step, 1.4, **kw)
    vol = np.array([orc.volume(s) for s in range(n)])
    W = np.column_stack([1 + 0.5 * rng.uniform(-1, 1, n), rng.uniform(-1, 1, n), 1 + 0.9 * rng.uniform(-1, 1, n)])
    q = problems.conserved_rows(W, 1.4) * vol[:, None]
    gpu.set_state(q)
    orc.set_state(q)
    try:
        dt = orc.time_step(0.4, "luna")
        assert gpu.time_step(0.4, "luna") == dt
        for k in range(6):
            if k % 3 == 2:
                gpu.step(dt)
                orc.step(dt)
            else:
                after = orc.step_and_time_step(dt, 0.4)
                assert gpu.step_and_time_step(dt, 0.4) == after
                dt = after
            assert np.array_equal(gpu.state(), orc.state), k
    finally:
        gpu.close()
