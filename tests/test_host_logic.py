"""Host-side logic of the reference-interface mirror and the workload
generators (CPU only)."""
import math

import numpy as np
import pytest


def test_mechanism_state_validation_like_the_reference(gp):
    """MechanismState::new panics when joint i's child is not body i or a
    parent frame is unknown (mechanism.rs:91-115)."""
    b1 = gp.RigidBody.new_sphere(1.0, 1.0, "a")
    with pytest.raises(ValueError, match="child body"):
        gp.MechanismState([gp.RevoluteJoint(gp.Transform3D.identity("b", gp.WORLD_FRAME), [0, 1, 0])], [b1])
    with pytest.raises(ValueError, match="no parent body"):
        gp.MechanismState([gp.RevoluteJoint(gp.Transform3D.identity("a", "nowhere"), [0, 1, 0])], [b1])


def test_parents_found_by_frame_name(gp):
    """test_supports tree of mechanism.rs:793 (bodies 1..5)."""
    joints = [gp.FloatingJoint(gp.Transform3D.identity("1", gp.WORLD_FRAME)),
              gp.RevoluteJoint(gp.Transform3D.move_x("2", "1", -1.0), [0, 1, 0]),
              gp.RevoluteJoint(gp.Transform3D.move_z("3", "2", 1.0), [0, 1, 0]),
              gp.RevoluteJoint(gp.Transform3D.move_x("4", "1", 1.0), [0, 1, 0]),
              gp.RevoluteJoint(gp.Transform3D.move_z("5", "4", 1.0), [0, 1, 0])]
    bodies = [gp.RigidBody.new_sphere(1.0, 1.0, str(i)) for i in range(1, 6)]
    st = gp.MechanismState(joints, bodies)
    assert st.parents == [0, 1, 2, 1, 4]
    d = st.model_desc()
    assert [d._bodies[i].parent for i in range(5)] == [-1, 0, 1, 0, 3]
    assert (d.nq, d.nv) == (7 + 4, 6 + 4)


def test_flattening_round_trip(gp):
    """joint/mod.rs:208-303: Pose -> [x,y,z,w,tx,ty,tz]; spatial -> [w; v]."""
    from gorilla_physics_amd import mechanism as m
    joints = [gp.FloatingJoint(gp.Transform3D.identity("a", gp.WORLD_FRAME)),
              gp.FixedJoint(gp.Transform3D.identity("b", "a")),
              gp.RevoluteJoint(gp.Transform3D.identity("c", "b"), [0, 0, 1])]
    q = [gp.Pose(gp.UnitQuaternion.from_axis_angle([0, 0, 1], 0.3), [1, 2, 3]), None, 0.7]
    v = [gp.SpatialVector([1, 2, 3], [4, 5, 6]), None, -2.0]
    fq, fv = m.flatten_q(q), m.flatten_v(v)
    assert len(fq) == 8 and len(fv) == 7
    assert fq[3] == pytest.approx(math.cos(0.15)) and fq[4:7] == [1, 2, 3]
    q2, v2 = m.unflatten_q(fq, joints), m.unflatten_v(fv, joints)
    assert q2[1] is None and v2[1] is None and q2[2] == 0.7 and list(v2[0].linear) == [4, 5, 6]


def test_tau_length_assertion(gp):
    """simulate.rs:39-45 asserts len(tau) == len(v); empty tau means zeros."""
    from gorilla_physics_amd import builders, mechanism
    st = builders.build_cube(1.0, 1.0)
    assert np.all(mechanism._tau_flat(st, []) == 0) and len(mechanism._tau_flat(st, [])) == 6
    with pytest.raises(AssertionError):
        mechanism._tau_flat(st, [0.0, 0.0])


def test_euler_angles_match_rotation_composition(gp):
    """from_euler_angles(r, p, y) = Rz(y) Ry(p) Rx(r)."""
    def rot(axis, a):
        return gp.UnitQuaternion.from_axis_angle(axis, a).to_matrix()
    q = gp.UnitQuaternion.from_euler_angles(0.1, 0.2, 0.3).to_matrix()
    assert np.allclose(q, rot([0, 0, 1], 0.3) @ rot([0, 1, 0], 0.2) @ rot([1, 0, 0], 0.1), atol=1e-15)


def test_workload_prefix_property(gp):
    """Instance i gets the same parameters and state whatever the batch size."""
    from gorilla_physics_amd import workloads
    a, b = workloads.arms(n=5), workloads.arms(n=9)
    assert np.array_equal(a["q"], b["q"][:35]) and np.array_equal(a["tau"], b["tau"][:35])
    for i in range(5):
        assert bytes(a["models"][i]._bodies) == bytes(b["models"][i]._bodies)


def test_cube_workload_starts_above_plane(gp, oracle):
    from gorilla_physics_amd import workloads
    w = workloads.cubes(n=32)
    for i in range(32):
        d = oracle.contact_distances(w["models"][0], w["q"][7 * i:7 * i + 7])
        assert 0.5 - 1e-12 <= d.min() <= 2.0 + 1e-12
        assert abs(np.linalg.norm(w["q"][7 * i:7 * i + 4]) - 1) < 1e-12


def test_mixed_workload_shape(gp):
    from gorilla_physics_amd import workloads
    w = workloads.mixed(n=400)
    nb = [d.n_bodies for d in w["models"]]
    trees = sum(1 for d in w["models"] if d.n_bodies == 13 and d._bodies[0].jtype == 3)
    assert 0.15 < trees / 400 < 0.35
    assert set(nb) - {13} <= set(range(1, 13))
    assert sum(d.nq for d in w["models"]) == len(w["q"])
    assert sum(d.nv for d in w["models"]) == len(w["v"]) == len(w["tau"])


def test_interface_poses_and_contact_positions(gp):
    """The browser-client calls (interface/mod.rs:172-220): poses as
    [qx, qy, qz, qw, tx, ty, tz] per body, contact positions in the world."""
    from gorilla_physics_amd import builders, interface
    st = builders.build_cube(1.0, 2.0)
    rot = gp.UnitQuaternion.from_axis_angle([0, 0, 1.0], math.pi / 2)
    st.update([gp.Pose(rot, [1.0, 2.0, 3.0])], [gp.SpatialVector()])
    sim = interface.InterfaceSimulator(st)
    p = sim.poses()
    assert p.shape == (7,) and np.allclose(p[:4], rot.coords()) and np.allclose(p[4:], [1, 2, 3])
    c = sim.contact_positions().reshape(-1, 3)
    assert c.shape == (8, 3)
    # corners at (+-1, +-1, +-1) rotated 90 degrees about z, then moved
    assert np.allclose(sorted(map(tuple, np.round(c - [1, 2, 3], 12))),
                       sorted((x, y, z) for x in (-1.0, 1.0) for y in (-1.0, 1.0) for z in (-1.0, 1.0)))
    sim.addHalfSpace([0, 0, 2.0], 0.5)
    assert np.allclose(st.halfspaces[0].normal, [0, 0, 1]) and np.allclose(st.halfspaces[0].point, [0, 0, 0.5])


def test_interface_biped_and_leg_poses(gp):
    """createBiped lowers the biped until the right foot's frame origin is
    at z = 0 and createLeg moves the foot's origin to the world origin
    (interface/biped.rs:16-95); with the legs bent (thigh -pi/4, calf pi/2)
    the base stands pelvis (0.2) + ankle-to-foot (0.05) + thigh and calf at
    45 degrees (2 x 0.2 cos(pi/4)) above the feet."""
    from gorilla_physics_amd import interface
    st = interface.create_biped()
    p = st.poses()
    names = [b.inertia.frame for b in st.bodies]
    assert abs(p[-1].translation[2]) < 1e-15
    base = p[names.index("base")].translation
    assert abs(base[2] - (0.2 + 0.05 + 2 * 0.2 * math.cos(math.pi / 4))) < 1e-12
    assert np.allclose(p[names.index("foot_left")].translation[2], p[names.index("foot_right")].translation[2])
    st = interface.create_leg()
    assert np.abs(st.poses()[-1].translation).max() < 1e-15
    st = interface.create_leg_from_foot()
    assert np.abs(st.poses()[0].translation).max() == 0.0 and st.q[1] == math.pi / 4 - 0.4


def test_bodies_to_root_of_a_branched_tree(gp, oracle):  # spatial/transform.rs:242
    """Bodies 2 and 4 at x = -1 and +1 beside body 1, bodies 3 and 5 one
    above each: at zero angles body 2 sits at (-1, 0, 0) and body 5 at
    (1, 0, 1) in the world; the oracle's gravitational energy (m g z of each
    frame origin) sees the two raised bodies."""
    T = gp.Transform3D
    joints = [gp.FloatingJoint(T.identity("1", gp.WORLD_FRAME)),
              gp.RevoluteJoint(T.move_x("2", "1", -1.0), [0, 1.0, 0]),
              gp.RevoluteJoint(T.move_z("3", "2", 1.0), [0, 1.0, 0]),
              gp.RevoluteJoint(T.move_x("4", "1", 1.0), [0, 1.0, 0]),
              gp.RevoluteJoint(T.move_z("5", "4", 1.0), [0, 1.0, 0])]
    st = gp.MechanismState(joints, [gp.RigidBody.new_sphere(1.0, 1.0, f) for f in "12345"])
    p = st.poses()
    assert np.array_equal(p[0].translation, [0, 0, 0]) and p[0].rotation.coords() == [0, 0, 0, 1.0]
    assert np.array_equal(p[1].translation, [-1.0, 0, 0]) and np.array_equal(p[4].translation, [1.0, 0, 1.0])
    assert abs(oracle.gravitational_energy(st.model_desc(), st.flat_q()) - 2 * 9.81) < 1e-12


def test_so101_workload_shape_and_prefix(gp):
    """One model, six coordinates per arm, and instance i's state and
    torques do not depend on the batch size."""
    from gorilla_physics_amd import workloads
    a, b = workloads.so101(n=5), workloads.so101(n=9)
    assert a["counts"] == [5] and a["models"][0].nq == 6 and a["q"].size == 30 and a["integrator"] == 2
    for key in ("q", "v", "tau"):
        assert np.array_equal(a[key], b[key][:30])


def test_a_kept_mass_matrix_keeps_little_else(gp):
    """Batch.mass_matrices over runs of instances of 7, 0, 3 and 100 values a
    side: every matrix its own values, square and writable, and what one of them
    keeps alive is itself or at most 64 KiB, not the whole batch's."""
    import ctypes
    from gorilla_physics_amd import batch
    sizes = np.array([7] * 5000 + [0] * 3 + [3] * 2000 + [100] * 2 + [7])
    values = np.random.default_rng(0).normal(size=int((sizes ** 2).sum()))

    class Lib:
        def gp_mass_matrix(self, handle, out):
            ctypes.memmove(out, values.ctypes.data, values.nbytes)
            return 0
    b = batch.Batch.__new__(batch.Batch)
    b.handle, b.lib = None, Lib()
    b.offsets = lambda: (None, np.concatenate([[0], np.cumsum(sizes)]))
    got = b.mass_matrices()
    assert [m.shape for m in got] == [(n, n) for n in sizes]
    assert np.array_equal(np.concatenate([m.reshape(-1) for m in got]), values)
    for m in got:
        kept = m
        while kept.base is not None:
            kept = kept.base
        assert m.flags.writeable and kept.nbytes <= max(64 << 10, m.nbytes)
    got[0][:] = 0.0
    assert np.array_equal(got[1].reshape(-1), values[49:98])
