"""Trees of 1-64 bodies on the one-body-per-lane kernel, packed several to a
wave: body counts around where an instance more or less fits in 64 lanes,
instance counts that leave a wave part empty, trees below 13 bodies (with the
automatic choice of kernel) with contacts, fixed-base and floating, a second
floating joint, every step against the oracle from the same state, FP64
within the 1e-10 per-step bound. What the kernel does not take stays as it
was: GP_KERNEL_FAST refuses a topology without a compiled kernel."""
import numpy as np
import pytest

from gpu_helpers import step_errors

pytestmark = pytest.mark.gpu

TOL = 1e-10


def _tree(rng, nb, root):
    """A random tree on a floating or revolute root; for root "two" the second
    body hangs on a floating joint as well."""
    from gorilla_physics_amd import abi, workloads
    parents, jtypes = workloads.random_tree_shape(rng, nb)
    for i in range(1, nb):  # at most 8 children a body
        while parents[:i].count(parents[i]) >= 8:
            parents[i] = int(rng.integers(0, i))
    if root == "revolute":
        jtypes[0] = abi.GP_JOINT_REVOLUTE
    if root == "two" and nb > 1:
        jtypes[1] = abi.GP_JOINT_FLOATING
    return workloads.random_tree_desc(rng, nb, (parents, jtypes))


def _state(d, rng):
    from gorilla_physics_amd import abi
    q = []
    for i in range(d.n_bodies):
        jt = d._bodies[i].jtype
        if jt == abi.GP_JOINT_FLOATING:
            q += [0.0, 0.0, 0.0, 1.0, 0.0, 0.0, rng.uniform(0.0, 0.3)]
        elif jt != abi.GP_JOINT_FIXED:
            q.append(rng.normal(0.0, 0.2))
    return np.array(q), rng.normal(0.0, 0.3, d.nv), rng.normal(0.0, 0.05, d.nv)


@pytest.mark.parametrize("nb", [1, 2, 5, 9, 12, 13, 16, 21, 22, 32, 33, 64])
@pytest.mark.parametrize("root", ["floating", "revolute", "two"])
@pytest.mark.parametrize("precision", [0, 1])
def test_trees_packed_in_waves_match_the_oracle(gp, oracle, nb, root, precision):
    from gorilla_physics_amd import batch
    if precision == 1 and not 5 <= nb < 13:
        pytest.skip("compiled topologies compute in FP32 there: test_gpu_trees, test_gpu_parity")
    rng = np.random.default_rng(100 * nb + len(root))
    d = _tree(rng, nb, root)
    n = 2 * (64 // nb) + 1  # two full waves' instances and one more
    parts = [_state(d, rng) for _ in range(n)]
    q, v, tau = (np.concatenate([p[k] for p in parts]) for k in range(3))
    b = batch.Batch([batch.Model(d)], [n], precision=precision)
    print(f"case small tree: {nb} bodies, root {root}, precision {precision}, {n} instances", flush=True)
    b.set_state(q, v)
    b.set_tau(tau)
    worst = 0.0
    for _ in range(3):
        q0, v0 = b.get_state()
        b.step(1e-4)
        q1, v1 = b.get_state()
        eq, ev, ea = step_errors(oracle, [d] * n, q0, v0, tau, q1, v1, b.get_vdot(), 1e-4)
        worst = max(worst, eq.max(), ev.max(), ea.max())
    assert worst <= TOL and not b.faults().any()
    if 5 <= nb < 13:  # with a contact point: no compiled topology
        assert b.get_opts().kernel == 0
        b.set_opts(kernel=2)
        with pytest.raises(gp.abi.GPError) as e:
            b.step(1e-4)
        assert e.value.code == gp.abi.GP_ERR_UNSUPPORTED


def test_small_trees_in_one_launch_give_the_same_bits(gp):
    """Several small tree topologies of a batch share a launch; steps per
    launch, workgroup size and separate launches change no bit."""
    from gorilla_physics_amd import batch
    rng = np.random.default_rng(5)
    descs = [_tree(rng, nb, "floating") for nb in (3, 7, 9, 12, 19, 40)]
    counts = [5, 11, 30, 6, 4, 3]
    inst = [d for d, c in zip(descs, counts) for _ in range(c)]
    parts = [_state(d, rng) for d in inst]
    q, v, tau = (np.concatenate([p[k] for p in parts]) for k in range(3))
    ref = None
    for kw in ({}, {"separate_launches": 1}, {"steps_per_launch": 3}, {"block_size": 256}, {"use_graph": 1}):
        b = batch.Batch([batch.Model(d) for d in descs], counts, **kw)
        b.set_state(q, v)
        b.set_tau(tau)
        b.step(1e-4, n_steps=12)
        got = b.get_state() + (b.get_vdot(),)
        launches = b.last_timing()[1]
        assert launches == (6 if kw.get("separate_launches") else 4 if kw.get("steps_per_launch") else 1)
        if ref is None:
            ref = got
        assert all(np.array_equal(x, y) for x, y in zip(ref, got)), kw
    b.step(1e-4, n_steps=0)


@pytest.mark.parametrize("nb", [1, 2, 9, 21, 22, 33, 64])
@pytest.mark.parametrize("root", ["floating", "revolute", "two"])
def test_joint_space_terms_of_packed_trees(gp, oracle, nb, root):
    """M, c and vdot of every instance by the one-body-per-lane kernels and by
    the one-instance-per-lane ones (GP_KERNEL_PLAIN), each against the
    oracle's CRBA, RNEA and LU, e <= 1e-10 (the FP64 bound)."""
    from gorilla_physics_amd import batch
    from gpu_helpers import rel_err
    rng = np.random.default_rng(300 * nb + len(root))
    d = _tree(rng, nb, root)
    n = 64 // nb + 1
    parts = [_state(d, rng) for _ in range(n)]
    q, v, tau = (np.concatenate([p[k] for p in parts]) for k in range(3))
    print(f"case terms of small tree: {nb} bodies, root {root}, {n} instances", flush=True)
    for kernel in (0, 1):
        b = batch.Batch([batch.Model(d)], [n], kernel=kernel)
        b.set_state(q, v)
        b.set_tau(tau)
        Ms, c, held, given = b.mass_matrices(), b.dynamics_bias(), b.dynamics(), b.dynamics(2.0 * tau)
        assert len(Ms) == n and not b.faults().any()
        for i, (qi, vi, ti) in enumerate(parts):
            Mr, cr = oracle.mass_matrix(d, qi, vi)
            s = slice(i * d.nv, (i + 1) * d.nv)
            assert rel_err(Ms[i], Mr) <= TOL and rel_err(c[s], cr) <= TOL and np.array_equal(Ms[i], Ms[i].T)
            assert rel_err(held[s], oracle.dynamics(d, qi, vi, ti)) <= TOL
            assert rel_err(given[s], oracle.dynamics(d, qi, vi, 2.0 * ti)) <= TOL
