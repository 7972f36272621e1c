"""The sweep at the ends of its ranges against the oracle, to the bit: cell counts around a wavefront's 64, meshes with many
tiny faces (left out of the limiter's range) or faces of area zero, and operands outside the exponents that its fast
divisions and square roots take (boxes of 2^-255 take the general operators, velocities of 2^-950 do for their own systems and
clips; boxes of 2^-130 and 2^60 are still inside), with the derivatives' fit beside it; and that the latter cost little.
"""
import numpy as np
import pytest

import cases
import oracle
from luna_hydro import hydro, mesh, problems

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


def faint(m, power, seed=4):
    """Q of a gas with velocities of 2^power, density and pressure about 1."""
    rng = np.random.Generator(np.random.MT19937(seed))
    W = np.ones((m["cells"], m["dim"] + 2))
    W[:, 0] += 0.1 * rng.uniform(-1, 1, m["cells"])
    W[:, 1:-1] = 2.0 ** power * rng.uniform(-1, 1, (m["cells"], m["dim"]))
    return problems.conserved_rows(W, 5.0 / 3.0) * m["volume"][:, None]


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("limiter", ["face", "none"])
@pytest.mark.parametrize("power", [-780, -950, -1005])
def test_right_hand_sides_below_the_fast_range(dim, limiter, power):
    """The fit's right-hand sides are about 2^-10 of the velocities: at 2^-1015 the fast quotients' residual is below the
    subnormal numbers. Without the limiter nothing else looks at the velocities' size."""
    m = cases.voronoi(11 if dim == 3 else 40, dim)
    compare(m, faint(m, power), steps=1, limiter=limiter)


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("power", [-780, -950, -1005])
def test_tangents_below_the_fast_range(dim, power):
    """The same for the tangent of the fit: dq of 2^power (its tangents of W are 2^-10 of that by the cells' volumes and back),
    and velocities of 2^power under a tangent of order 1."""
    m = cases.voronoi(11 if dim == 3 else 40, dim)
    rng = np.random.Generator(np.random.MT19937(6))
    dq = rng.uniform(-1, 1, (m["cells"], dim + 2)) * m["volume"][:, None]
    for q, scale in ((cases.rough_state(m), 2.0 ** power), (faint(m, power), 1.0)):
        gpu, orc = hydro.FiniteVolume(m, 5.0 / 3.0, limiter="none"), oracle.FiniteVolume(m, 5.0 / 3.0, limiter="none")
        try:
            gpu.set_state(q)
            orc.set_state(q)
            dt = orc.time_step(0.3)
            got, want = gpu.step_tangent(dt, dq * scale), orc.step_tangent(dt, dq * scale)
            assert np.array_equal(got, want)
            assert np.array_equal(gpu.state(), orc.q)
        finally:
            gpu.close()


def without_extent(m, every):
    """The mesh with each `every`-th face of area 0 (its neighbours stay in each other's lists)."""
    out = dict(m)
    out["area"] = m["area"].copy()
    out["area"][::every] = 0.0
    return out


@pytest.mark.parametrize("dim", [2, 3])
def test_faces_of_area_zero(dim):
    """Static and moving steps on meshes with a face of |A| = 0 in every wavefront's lists."""
    n = 9 if dim == 3 else 30
    m = without_extent(cases.voronoi(n, dim), 37)
    compare(m, cases.rough_state(m))
    gpu = hydro.FiniteVolume(m, 5.0 / 3.0, motion="moving")
    orc = oracle.FiniteVolume(m, 5.0 / 3.0, moving=True)
    try:
        for fv in (gpu, orc):
            fv.set_state(cases.rough_state(m))
        for s in range(2):
            dt = orc.time_step(0.3)
            assert gpu.time_step(0.3) == dt
            assert np.array_equal(gpu.gradients(), orc.grad)
            x = orc.moving_begin(dt)
            assert np.array_equal(gpu.moving_begin(dt), x)
            nm = without_extent(mesh.build(x, 1.0), 37)
            gpu.moving_finish(nm, dt)
            orc.moving_finish(nm, dt)
            assert np.array_equal(gpu.state(), orc.q), s
    finally:
        gpu.close()


def sweep_ms(m, q, **kw):
    """The least time of a sweep, by the kernel events."""
    fv = hydro.FiniteVolume(m, 5.0 / 3.0, **kw)
    try:
        fv.set_state(q)
        fv.time_step(0.3)
        best = np.inf
        for _ in range(8):
            fv.set_state(q)
            fv.profile(True)
            fv.time_step(0.3)
            best = min(best, fv.kernel_times()["sweep"][1])
        return best
    finally:
        fv.close()


def test_velocities_out_of_range_do_not_cost_a_second_walk():
    """Velocities below the fast operators' range take the general ones for the systems and the clips alone: 1.1 times the time
    of ordinary ones on MI355X (64,000 cells), 1.8 with the whole slice walked again."""
    m = cases.voronoi(40, 3)
    ratio = sweep_ms(m, faint(m, -950)) / sweep_ms(m, faint(m, -1))
    print("velocities of 2^-950: %.2f of the time" % ratio, flush=True)
    assert ratio < 1.45


def test_faces_of_area_zero_do_not_cost_a_second_walk():
    """A face of |A| = 0 stays with the fast operators: 1.0 times the time on MI355X (64,000 cells, every 150th face), 1.8 with
    the whole slice walked again."""
    m = cases.voronoi(40, 3)
    q = cases.rough_state(m)
    ratio = sweep_ms(without_extent(m, 150), q, motion="moving") / sweep_ms(m, q, motion="moving")
    print("|A| = 0: %.2f of the time" % ratio, flush=True)
    assert ratio < 1.45


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("limiter", ["face", "none"])
@pytest.mark.parametrize("power", [-249, -240, -225, 110, 130, 240])
def test_box_scales_between_the_ranges(dim, limiter, power):
    """Boxes in which one part only is out of the fast operators' range: the Cholesky factor's diagonal (2^-225 and below, 2^130
    and above), the right-hand sides, the face offsets (2^110 and above), while the separations are still inside."""
    base = cases.voronoi(10 if dim == 3 else 24, dim)
    m = scaled(base, 2.0 ** power)
    q = cases.rough_state(base) / base["volume"][:, None] * m["volume"][:, None]
    compare(m, q, limiter=limiter)
