"""Cells with far more faces than their neighbours (a generator alone in a shell of others): lists past the geometry pass's 32
staged entries, whose slots and padding go to memory directly. Steps, the moving step's second mesh and the derivatives
against the oracle, to the bit."""
import numpy as np
import pytest

import cases
import oracle
from luna_hydro import hydro, mesh, problems

pytestmark = pytest.mark.gpu
GAMMA = 5.0 / 3.0


def rosette(dim, around, n):
    """A jittered lattice, one generator in the middle of a hole in it and `around` others on a sphere (circle) around that."""
    x = problems.jittered_lattice(n, dim, 0.25, 1)
    x = x[np.linalg.norm(x - 0.5, axis=1) > 0.27]
    k = np.arange(around) + 0.5
    if dim == 3:
        z, a = 1 - 2 * k / around, np.pi * (1 + 5 ** 0.5) * k
        unit = np.column_stack([np.sqrt(1 - z * z) * np.cos(a), np.sqrt(1 - z * z) * np.sin(a), z])
    else:
        unit = np.column_stack([np.cos(2 * np.pi * k / around), np.sin(2 * np.pi * k / around)])
    rng = np.random.default_rng(3)
    shell = 0.5 + 0.18 * (1 + 0.01 * rng.uniform(-1, 1, (around, 1))) * unit
    return mesh.build(np.concatenate([[np.full(dim, 0.5)], x, shell]), 1.0)


@pytest.mark.parametrize("dim,around,n,longest", [(3, 45, 10, 45), (3, 70, 10, 70), (2, 34, 14, 34), (2, 50, 14, 41)])
@pytest.mark.parametrize("device", [False, True], ids=["host", "device"])
def test_long_lists_match_oracle(dim, around, n, longest, device):
    m = rosette(dim, around, n)
    assert np.diff(m["start"]).max() == longest
    given = (lambda mesh_: hydro.DeviceMesh(mesh_)) if device else (lambda mesh_: mesh_)
    q = cases.rough_state(m, blast=2.0)
    gpu, orc = hydro.FiniteVolume(given(m), GAMMA), oracle.FiniteVolume(m, GAMMA)
    try:
        for fv in (gpu, orc):
            fv.set_state(q)
        for _ in range(2):
            dt = orc.time_step(0.3)
            assert gpu.time_step(0.3) == dt
            assert np.array_equal(gpu.gradients(), orc.grad)
            gpu.step(dt)
            orc.step(dt)
            assert np.array_equal(gpu.state(), orc.q)
        rng = np.random.default_rng(5)
        dq = rng.standard_normal(np.shape(q))
        for fv in (gpu, orc):
            fv.set_state(q)
        got, want = gpu.step_adjoint(dt, dq), orc.step_adjoint(dt, dq)
        assert cases.max_relative(got, want) <= 1e-12
        got, want = gpu.step_tangent(dt, dq), orc.step_tangent(dt, dq)
        assert np.array_equal(got, want)
    finally:
        gpu.close()


@pytest.mark.parametrize("dim,around,n", [(3, 45, 10), (3, 70, 10), (2, 50, 14)])
def test_moving_steps_with_long_lists_match_oracle(dim, around, n):
    m = rosette(dim, around, n)
    gpu, orc = hydro.FiniteVolume(m, GAMMA, motion="moving"), oracle.FiniteVolume(m, GAMMA, moving=True)
    try:
        for fv in (gpu, orc):
            fv.set_state(cases.rough_state(m, blast=2.0))
        for s in range(2):
            dt = orc.time_step(0.3)
            assert gpu.time_step(0.3) == dt
            x = orc.moving_begin(dt)
            assert np.array_equal(gpu.moving_begin(dt), x)
            nm = mesh.build(x, 1.0)
            for fv in (gpu, orc):
                fv.moving_finish(nm, dt)
            assert np.array_equal(gpu.state(), orc.q), s
    finally:
        gpu.close()
