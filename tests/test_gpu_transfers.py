"""The device-array transfers (gp_batch_set_state_dev and its kin) against the
host calls: one launch moves every bucket, so the batches mix topologies, with
instances of one bucket apart in the flattened arrays, at lane counts around
a workgroup's 64 and row counts around its four waves. Values are copied, so
they are equal bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 64, 65, 257])
def test_device_arrays_match_the_host_calls(gp, n):
    import ctypes as C
    from test_gpu_rollouts import _hip
    from gorilla_physics_amd import abi, batch, builders, workloads
    from gorilla_physics_amd.mechanism import Isometry3, ModelDesc, SpatialInertia, body_desc
    box = SpatialInertia.cuboid_at([0, 0, 0], 1.0, 0.1, 0.1, 0.1, "b")
    welded = ModelDesc([body_desc(-1, abi.GP_JOINT_FIXED, [0, 0, 1], Isometry3.identity(), box)], [], [])  # no rows
    descs = [workloads.acrobot_desc(), builders.build_cube(1.0, 1.0).model_desc(), welded,
             workloads.arms(1, dof=5)["models"][0], builders.build_quadruped().model_desc(),
             workloads.hexapod_desc(dict(bw=0.5, bd=0.3, bh=0.1, bm=3.0, lt=[0.2] * 6, ls=[0.2] * 6, mt=[0.2] * 6,
                                         ms=[0.2] * 6))]
    models = [batch.Model(d) for d in descs]
    # n rounds over the models: a bucket's instances lie apart in the flat arrays
    b = batch.Batch([m for _ in range(n) for m in models], [1] * (n * len(models)))
    rng = np.random.default_rng(n)
    q, v, tau = rng.normal(size=b.nq_total), rng.normal(size=b.nv_total), rng.normal(size=b.nv_total)
    print(f"case transfers: {b.n_instances} instances, {b.n_buckets} buckets", flush=True)

    hip, bufs = _hip(), []

    def dev(x):  # a device copy of x
        p = C.c_void_p()
        assert hip.hipMalloc(C.byref(p), x.nbytes) == 0
        bufs.append(p)
        assert hip.hipMemcpy(p, x.ctypes.data, x.nbytes, 1) == 0
        return p.value

    def host(p, like):
        out = np.empty_like(like)
        assert hip.hipMemcpy(out.ctypes.data, p, out.nbytes, 2) == 0
        return out
    try:
        _check(b, descs, q, v, tau, dev, host, abi)
    finally:
        for p in bufs:
            hip.hipFree(p)


def _check(b, descs, q, v, tau, dev, host, abi):
    dt = dev(tau)
    b.set_state_dev(dev(q), dev(v))
    b.sync()
    hq, hv = b.get_state()
    assert np.array_equal(hq, q) and np.array_equal(hv, v)
    oq, ov, oa = dev(np.zeros_like(q)), dev(np.zeros_like(v)), dev(np.zeros_like(v))
    b.get_state_dev(oq, ov)
    b.sync()
    assert np.array_equal(host(oq, q), q) and np.array_equal(host(ov, v), v)
    # torques set either way give the same step
    q[:], v[:] = 0.0, 0.1 * v
    at = 0
    for i in range(b.n_instances):
        if descs[i % len(descs)]._bodies[0].jtype == abi.GP_JOINT_FLOATING:
            q[at + 3] = 1.0
        at += descs[i % len(descs)].nq
    out = []
    for set_tau in (lambda: b.set_tau(tau), lambda: b.set_tau_dev(dt)):
        b.set_tau(None)
        b.set_state(q, v)
        set_tau()
        b.step(1e-4)
        b.get_vdot_dev(oa)
        b.sync()
        assert np.array_equal(host(oa, v), b.get_vdot())
        out.append(host(oa, v))
    assert np.array_equal(out[0], out[1]) and np.isfinite(out[0]).all()


@pytest.mark.parametrize("n", [63, 64, 65, 16384, 16385, 40000])
def test_host_arrays_of_one_bucket(gp, n):
    """Host calls on a batch of one bucket, around the sizes at which rows are
    copied straight in (256 state values, 32,768 torques) or staged, and a
    read-back that crosses in one copy or in two (1 MiB): values come back bit
    for bit, also when only q or v changes, and torques act as set."""
    from gorilla_physics_amd import batch, workloads
    b = batch.Batch([batch.Model(workloads.acrobot_desc())], [n])
    rng = np.random.default_rng(n)
    q, v = rng.normal(size=2 * n), rng.normal(size=2 * n)
    for _ in range(2):
        b.set_state(q, v)
        hq, hv = b.get_state()
        assert np.array_equal(hq, q) and np.array_equal(hv, v)
        v = rng.normal(size=2 * n)
    b.set_state(q, 0 * v)
    free, tau = b.dynamics(), rng.normal(size=2 * n)
    b.set_tau(tau)
    held = b.dynamics()
    assert np.array_equal(held, b.dynamics(tau)) and (held != free).any()
    b.set_tau(None)
    assert np.array_equal(b.dynamics(), free)
