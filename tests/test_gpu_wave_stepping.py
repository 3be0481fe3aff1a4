"""Velocity stepping with one instance per wave (few instances) against the
one-instance-per-lane kernel (GP_KERNEL_PLAIN), on the GPU: the same bits, as
both form every value by the same operations in the same order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _model(gp, kind):
    from gorilla_physics_amd import builders
    plane = gp.HalfSpace.new([0.0, 0.0, 1.0], 0.0)
    st = builders.build_quadruped() if kind == "quadruped" else builders.build_cube(1.0, 1.0)
    st.add_halfspace(plane)
    if kind == "cube":  # more candidates than the single-body kernel takes
        st.add_halfspace(gp.HalfSpace.new([np.sin(0.3), 0.0, np.cos(0.3)], 0.0))
    return st.model_desc()


@pytest.mark.parametrize("integrator", [3, 4])
@pytest.mark.parametrize("kind", ["quadruped", "cube"])
@pytest.mark.parametrize("n", [1, 65, 1024, 1025])  # the last one is past the wave kernel's range
def test_wave_stepping_gives_the_lane_kernels_bits(gp, kind, n, integrator):
    from gorilla_physics_amd import batch
    rng = np.random.default_rng(n)
    d = _model(gp, kind)
    q = rng.normal(0.0, 0.1, (n, d.nq))
    q[:, :7] = [0.0, 0.0, 0.0, 1.0, 0.0, 0.0, 1.0]
    q[:, 6] = rng.uniform(0.9, 1.2, n) if kind == "quadruped" else rng.uniform(0.45, 0.7, n)
    v, tau = rng.normal(0.0, 0.5, (n, d.nv)), rng.normal(0.0, 0.1, (n, d.nv))
    got = []
    for kernel in (0, 1):
        b = batch.Batch([batch.Model(d)], [n], kernel=kernel)
        b.set_state(q.ravel(), v.ravel())
        b.set_tau(tau.ravel())
        b.step(1e-2, integrator, 3)
        b.step(1e-2, integrator, 1)
        b.sync()
        got.append(b.get_state() + (b.get_vdot(), b.collision_rounds(), b.faults()))
    assert np.isfinite(got[0][0]).all()
    for x, y in zip(*got):
        assert np.array_equal(x, y)
