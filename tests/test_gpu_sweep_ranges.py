"""The sweep at the ends of its ranges against the oracle, to the bit: cell counts around a wavefront's 64, meshes with many
tiny faces (left out of the limiter's range), and operands outside the exponents that its fast divisions and square roots
take (boxes of 2^-255 and velocities of 2^-950 take the general operators; boxes of 2^-130 and 2^60 are still inside).
"""
import numpy as np
import pytest

import cases
import oracle
from luna_hydro import hydro, problems

pytestmark = pytest.mark.gpu


def scaled(m, s):
    """The mesh in a box s times as large (s a power of two: exact)."""
    D = m["dim"]
    out = dict(m)
    for k, p in (("positions", 1), ("centroid", 1), ("face_centroid", 1), ("area", D - 1), ("volume", D)):
        out[k] = m[k] * s ** p
    out["side"] = [x * s for x in m["side"]]
    out["step"] = m["step"] * s
    return out


def compare(m, q, steps=2, **kw):
    gpu, orc = hydro.FiniteVolume(m, 5.0 / 3.0, **kw), oracle.FiniteVolume(m, 5.0 / 3.0, **kw)
    gpu.set_state(q)
    orc.set_state(q)
    try:
        for _ in range(steps):
            dt = orc.time_step(0.3)
            assert gpu.time_step(0.3) == dt
            assert np.array_equal(gpu.gradients(), orc.grad)
            gpu.step(dt)
            orc.step(dt)
            assert np.array_equal(gpu.state(), orc.q)
    finally:
        gpu.close()


@pytest.mark.parametrize("dim,n,jitter", [(3, 4, 0.25), (3, 5, 0.45), (3, 9, 0.49), (2, 8, 0.25), (2, 9, 0.45), (2, 33, 0.49)])
def test_cell_counts_and_tiny_faces(dim, n, jitter):
    m = cases.voronoi(n, dim, jitter, seed=3)
    compare(m, cases.rough_state(m, blast=1.0))


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("power", [-255, -130, 60])
def test_box_scales(dim, power):
    m = scaled(cases.voronoi(10 if dim == 3 else 24, dim), 2.0 ** power)
    base = cases.voronoi(10 if dim == 3 else 24, dim)
    q = cases.rough_state(base) / base["volume"][:, None] * m["volume"][:, None]
    compare(m, q)


@pytest.mark.parametrize("dim", [2, 3])
def test_velocities_below_the_fast_range(dim):
    m = cases.voronoi(10 if dim == 3 else 24, dim)
    rng = np.random.Generator(np.random.MT19937(4))
    W = np.ones((m["cells"], dim + 2))
    W[:, 0] += 0.1 * rng.uniform(-1, 1, m["cells"])
    W[:, 1:-1] = 2.0 ** -950 * rng.uniform(-1, 1, (m["cells"], dim))
    compare(m, problems.conserved_rows(W, 5.0 / 3.0) * m["volume"][:, None], steps=1)
