"""The static line's step against the oracle, to the bit, at the lengths where its wavefronts (60 slots each, two more at each
end) begin and end, with every wall, order and limiter, the fused step and the plain one.
"""
import time

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


def seeded_line(n, **kw):
    keys, step, period = problems.line_keys(problems.line_points(n, 1.0, 0.6, seed=n), 1.0)
    rng = np.random.Generator(np.random.MT19937(n))
    W = np.column_stack([1 + 0.5 * rng.uniform(-1, 1, n), rng.uniform(-1, 1, n), 1 + 0.9 * rng.uniform(-1, 1, n)])
    gpu = hydro.Line(keys, period, step, 1.4, **kw)
    return gpu, (keys, period, step), problems.conserved_rows(W, 1.4) / n


@pytest.mark.parametrize("n", [16383, 16384, 16385, 16440, 16441, 16561, 40000])
@pytest.mark.parametrize("kw", [
    {"periodic": True, "limiter": "vanleer"},
    {"walls": ("reflective", "outflow"), "limiter": "face", "riemann": "hll"},
], ids=["periodic", "reflective-outflow-hll"])
def test_long_lines_match_oracle(n, kw):
    """Around 16384 cells, where the step's minimum goes from one word to one per work-group of 240 slots, with time_step
    between the fused steps (it writes one word of the same set)."""
    gpu, line, q = seeded_line(n, **kw)
    orc = oracle.Line(*line, 1.4, **kw)
    gpu.set_state(q)
    orc.set_state(q)
    try:
        for k in range(5):
            dt = orc.time_step(0.4, "luna")
            assert gpu.time_step(0.4, "luna") == dt
            for _ in range(k % 3):
                after = orc.step_and_time_step(dt, 0.4)
                assert gpu.step_and_time_step(dt, 0.4) == after
                dt = after
            gpu.step(dt)
            orc.step(dt)
            assert np.array_equal(gpu.state(), orc.state), k
    finally:
        gpu.close()


def test_fused_step_of_a_long_line_takes_no_atomic_per_wavefront():
    """A million cells: the fused step within 3 plain steps and 60 us for the time step's way to the host (30 and 47 us on
    MI355X; with two atomics on one line from each of its 16,667 wavefronts it took 519)."""
    gpu, _, q = seeded_line(1000000, periodic=True, limiter="minmod")
    gpu.set_state(q)
    try:
        dt = gpu.time_step(0.3, "luna")
        plain = fused = np.inf
        for _ in range(5):
            start = time.perf_counter()
            for _ in range(20):
                dt = gpu.step_and_time_step(dt, 0.3)
            fused = min(fused, (time.perf_counter() - start) / 20)
            start = time.perf_counter()
            for _ in range(20):
                gpu.step(dt)
            hydro.lib().luna_synchronize()
            plain = min(plain, (time.perf_counter() - start) / 20)
        print("plain %.1f us, fused %.1f us" % (plain * 1e6, fused * 1e6), flush=True)
        assert fused < 3 * plain + 60e-6
    finally:
        gpu.close()
