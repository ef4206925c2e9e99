"""GPU parity: libvbd_hip (through SolverVBD / CollisionPipeline) against the FP32 CPU oracle.

The HIP kernels evaluate every FP32 expression in the reference's CPU order
(no FMA contraction, serial CSR-order sums), so positions and velocities are
required to be bit-identical to the oracle (tolerance 0) on the short runs; the
600-frame run checks the stated bar of 1e-5 m max-abs per frame and reports the
drift and both implementations' error against the FP64 oracle.
"""

import numpy as np
import pytest

import oracle
from _sim import gpu_run, initial, oracle_run

pytestmark = pytest.mark.gpu


def _scene(name, dev):
    from newton_amd import scenes

    return {
        "hanging": lambda: scenes.cloth_hanging(dev),
        "strip": lambda: scenes.cloth_strip_pinned(dev),
        "cube": lambda: scenes.soft_cube(dev),
    }[name]()


def _fan_scene(dev, segments=160):
    """A triangle fan: the centre vertex has `segments` triangles and ~2x that many hinges (> 256 items)."""
    import math

    from newton_amd import ModelBuilder

    b = ModelBuilder(up_axis="Y", gravity=-9.81)
    b.add_ground_plane(cfg=ModelBuilder.ShapeConfig(ke=1.0e4, kd=0.0, mu=0.5))
    verts = [(0.0, 0.0, 0.0)] + [(0.5 * math.cos(2 * math.pi * i / segments), 0.5 * math.sin(2 * math.pi * i / segments),
                                  0.0) for i in range(segments)]
    tris = []
    for i in range(segments):
        tris += [0, 1 + i, 1 + (i + 1) % segments]
    b.add_cloth_mesh(pos=(0.0, 0.3, 0.0), rot=(0.7071068, 0.0, 0.0, 0.7071068), scale=1.0, vel=(0.0, 0.0, 0.0),
                     vertices=verts, indices=tris, density=0.1, tri_ke=1.0e3, tri_ka=1.0e3, tri_kd=1.0e-3,
                     edge_ke=0.1, edge_kd=1.0e-4, particle_radius=0.02)
    b.color(include_bending=True)
    model = b.finalize(dev)
    model.soft_contact_ke, model.soft_contact_kd, model.soft_contact_mu = 1.0e4, 0.0, 0.5
    state = model.state()
    info = {"dt": 1.0 / 600.0, "substeps": 10, "iterations": 4}
    return model, state, info


def _many_planes_scene(dev, planes=24):
    """A 16x16 cloth resting within the margin of `planes` coincident ground planes: > 512 rows per batch."""
    import math

    from newton_amd import ModelBuilder
    from newton_amd.sim.builder import cloth_grid_mesh, quat_from_axis_angle

    b = ModelBuilder(up_axis="Y", gravity=-9.81)
    for k in range(planes):
        b.add_ground_plane(cfg=ModelBuilder.ShapeConfig(ke=1.0e3 + 10.0 * k, kd=0.5, mu=0.3 + 0.01 * k))
    verts, tris = cloth_grid_mesh(15, 15, 0.02, 0.02)
    b.add_cloth_mesh(pos=(0.0, 0.05, 0.0), rot=quat_from_axis_angle((1.0, 0.0, 0.0), math.pi / 2), scale=1.0,
                     vel=(0.0, -0.2, 0.0), vertices=verts, indices=tris, density=0.1, tri_ke=1.0e3, tri_ka=1.0e3,
                     tri_kd=1.0e-4, edge_ke=0.1, edge_kd=0.0, particle_radius=0.06)
    b.color(include_bending=True)
    model = b.finalize(dev)
    model.soft_contact_ke, model.soft_contact_kd, model.soft_contact_mu = 1.0e3, 0.5, 0.5
    state = model.state()
    info = {"dt": 1.0 / 600.0, "substeps": 10, "iterations": 3}
    return model, state, info


def test_generic_path_for_high_valence_vertex_bitexact(cuda_device):
    from newton_amd.solvers import SolverVBD

    model, state, info = _fan_scene(cuda_device)
    stats = SolverVBD(model, iterations=1).layout_stats()
    assert stats["generic_vertices"] == 1, stats
    q0, qd0 = initial(state)
    q_gpu, qd_gpu, _ = gpu_run(model, state, info, 8)
    q_ref, qd_ref, _ = oracle_run(model, q0, qd0, info, 8)
    np.testing.assert_array_equal(q_gpu, q_ref)
    np.testing.assert_array_equal(qd_gpu, qd_ref)


@pytest.mark.parametrize("planes", [24, 40])
def test_serial_contact_mode_bitexact(cuda_device, planes):
    """Contacts that overflow the batch's LDS rows are summed serially; with 40 planes every particle
    carries 40 entries (past the 32 its position's key sort keeps in LDS)."""
    model, state, info = _many_planes_scene(cuda_device, planes)
    q0, qd0 = initial(state)
    q_gpu, qd_gpu, _ = gpu_run(model, state, info, 4)
    q_ref, qd_ref, _ = oracle_run(model, q0, qd0, info, 4)
    np.testing.assert_array_equal(q_gpu, q_ref)
    np.testing.assert_array_equal(qd_gpu, qd_ref)


def test_notify_model_changed_rebuilds_layout(cuda_device):
    """Editing element materials after construction takes effect after notify_model_changed(), also when
    the edit switches elements to zero stiffness (the layout then changes shape and is re-allocated)."""
    import torch

    from newton_amd.solvers import SolverVBD

    model, state, info = _scene("strip", cuda_device)
    q0, qd0 = initial(state)
    solver = SolverVBD(model, iterations=info["iterations"])
    stats0 = solver.layout_stats()
    model.tri_materials[:, 0] *= 3.0
    model.tri_materials[:4, :2] = 0.0  # these triangles now contribute nothing and leave the layout
    model.edge_bending_properties[:, 0] *= 0.5
    solver.notify_model_changed()
    assert solver.layout_stats()["items"] < stats0["items"]
    s1 = model.state()
    solver.step(state, s1, None, None, info["dt"])
    torch.cuda.synchronize()
    om = oracle.OracleModel(model)
    _, q_ref, qd_ref = oracle.step(om, oracle.params(info["iterations"]), q0, qd0, None, None, info["dt"])
    np.testing.assert_array_equal(s1.particle_q.cpu().numpy(), q_ref)


def test_library_is_native(cuda_device):
    from newton_amd import _native

    lib = _native.hip_lib()
    assert lib.vbd_version() >= 1


def test_soft_contacts_bitexact(cuda_device):
    import torch

    from newton_amd import CollisionPipeline

    model, state, info = _scene("strip", cuda_device)
    pipe = CollisionPipeline(model, soft_contact_margin=0.05)
    contacts = pipe.contacts()
    pipe.collide(state, contacts)
    torch.cuda.synchronize()
    om = oracle.OracleModel(model)
    oc = oracle.Contacts(pipe.soft_contact_max)
    n = oracle.create_soft_contacts(om, state.particle_q.cpu().numpy(), 0.05, oc)
    assert n > 0
    assert int(contacts.soft_contact_count.item()) == n
    for name, ref in (("soft_contact_indices", oc.indices), ("soft_contact_shape", oc.shape),
                      ("soft_contact_particle", oc.particle)):
        np.testing.assert_array_equal(getattr(contacts, name).cpu().numpy()[:n], ref[:n])
    for name, ref in (("soft_contact_body_pos", oc.body_pos), ("soft_contact_body_vel", oc.body_vel),
                      ("soft_contact_normal", oc.normal)):
        np.testing.assert_array_equal(getattr(contacts, name).cpu().numpy()[:n], ref[:n])


def test_soft_contact_overflow_keeps_count(cuda_device):
    """More contacts than soft_contact_max: count reports all, records stop at max (geometry/kernels.py:1165-1167)."""
    import torch

    from newton_amd import CollisionPipeline

    model, state, info = _scene("hanging", cuda_device)
    state.particle_q[:, 1] = 0.05  # every particle within the ground margin
    pipe = CollisionPipeline(model, soft_contact_margin=0.01, soft_contact_max=100)
    contacts = pipe.contacts()
    pipe.collide(state, contacts)
    torch.cuda.synchronize()
    active = int((model.particle_flags.cpu().numpy() & 1).sum())
    assert int(contacts.soft_contact_count.item()) == active
    assert np.all(contacts.soft_contact_particle.cpu().numpy()[:100] >= 0)


@pytest.mark.parametrize("scene", ["hanging", "strip", "cube"])
@pytest.mark.parametrize("substeps", [1, 12])
def test_substeps_bitexact(cuda_device, scene, substeps):
    model, state, info = _scene(scene, cuda_device)
    q0, qd0 = initial(state)
    q_gpu, qd_gpu, _ = gpu_run(model, state, info, substeps)
    q_ref, qd_ref, _ = oracle_run(model, q0, qd0, info, substeps)
    print(f"{scene} x{substeps}: max|dq| {np.abs(q_gpu - q_ref).max():.3e} max|dv| {np.abs(qd_gpu - qd_ref).max():.3e}")
    np.testing.assert_array_equal(q_gpu, q_ref)
    np.testing.assert_array_equal(qd_gpu, qd_ref)


def test_contact_overflow_step_bitexact(cuda_device):
    """A contact buffer smaller than the pair count: the solver consumes min(count, max) records."""
    model, state, info = _scene("strip", cuda_device)
    q0, qd0 = initial(state)
    q_gpu, qd_gpu, _ = gpu_run(model, state, info, 6, margin=0.05, contact_max=7)
    q_ref, qd_ref, _ = oracle_run(model, q0, qd0, info, 6, margin=0.05, contact_max=7)
    np.testing.assert_array_equal(q_gpu, q_ref)
    np.testing.assert_array_equal(qd_gpu, qd_ref)


def test_fp64_ill_conditioned_mode_bitexact(cuda_device):
    """Nearly massless beads on stiff springs (block condition numbers >> 1e6): the FP64 block solve is
    taken, changes the result, and the GPU equals the oracle bit for bit with it on and off."""
    from newton_amd import scenes

    out = {}
    for fp64 in (True, False):
        model, state, info = scenes.bead_rope_light(cuda_device)
        q0, qd0 = initial(state)
        q_gpu, qd_gpu, _ = gpu_run(model, state, info, 10, solver_kwargs={"fp64_ill_conditioned": fp64})
        q_ref, qd_ref, _ = oracle_run(model, q0, qd0, info, 10, fp64_ill_conditioned=fp64)
        np.testing.assert_array_equal(q_gpu, q_ref)
        np.testing.assert_array_equal(qd_gpu, qd_ref)
        out[fp64] = q_gpu
    assert np.abs(out[True] - out[False]).max() > 1e-4


@pytest.mark.parametrize("mass", [1.0e-2, 1.0e-3, 1.0e-4, 1.0e-5, 1.0e-6])
def test_condition_screen_bitexact(cuda_device, mass):
    """Block conditions from about 1 to 1e4, most of which the single-precision screen clears: with the estimate skipped
    or evaluated the solve is the single-precision one of the oracle, which always evaluates it.  That the screen never
    clears a block beyond 1e6 is test_scalar_formulas.py's; conditions around and beyond it follow below."""
    from newton_amd import scenes

    model, state, info = scenes.bead_rope_light(cuda_device, mass=mass)
    q0, qd0 = initial(state)
    q_gpu, qd_gpu, _ = gpu_run(model, state, info, 10, solver_kwargs={"fp64_ill_conditioned": True})
    q_ref, qd_ref, _ = oracle_run(model, q0, qd0, info, 10, fp64_ill_conditioned=True)
    assert np.array_equal(q_gpu, q_ref) and np.array_equal(qd_gpu, qd_ref)


@pytest.mark.parametrize("shape", [(256, 1, 0), (256, 7, 1), (192, 1, 1), (128, 1, 0)])
def test_cloth_springs_and_tets_in_one_model_bitexact(cuda_device, shape):
    """Every element kind in one pass: cloth with springs over a tet cube with a stiff skin on the ground, damped."""
    from newton_amd import ModelBuilder
    from newton_amd.solvers import SolverVBD

    b = ModelBuilder(up_axis="Y", gravity=-9.81)
    b.add_ground_plane(cfg=ModelBuilder.ShapeConfig(ke=1.0e4, kd=1.0, mu=0.5))
    b.add_soft_grid(pos=(0.0, 0.005, 0.0), rot=(0.0, 0.0, 0.0, 1.0), vel=(0.0, -0.3, 0.0), dim_x=4, dim_y=3, dim_z=3,
                    cell_x=0.05, cell_y=0.05, cell_z=0.05, density=300.0, k_mu=1.0e4, k_lambda=1.0e4, k_damp=1.0e-3,
                    tri_ke=1.0e2, tri_ka=1.0e2, tri_kd=1.0e-3, edge_ke=0.05, edge_kd=1.0e-4, particle_radius=0.01)
    tets = b.particle_count
    b.add_cloth_grid(pos=(-0.05, 0.162, 0.25), rot=(-np.sqrt(0.5), 0.0, 0.0, np.sqrt(0.5)), vel=(0.0, -0.4, 0.0),
                     dim_x=9, dim_y=9, cell_x=0.03, cell_y=0.03, mass=0.01, tri_ke=1.0e3, tri_ka=1.0e3, tri_kd=1.0e-3,
                     edge_ke=0.1, edge_kd=1.0e-3, particle_radius=0.01)
    for i in range(tets, tets + 60):
        b.add_spring(i, i + 1, 30.0, 0.01)
    b.color(include_bending=True)
    model = b.finalize(cuda_device)
    model.soft_contact_ke, model.soft_contact_kd, model.soft_contact_mu = 1.0e4, 1.0, 0.5
    state, info = model.state(), {"dt": 1.0 / 600.0, "iterations": 4}
    q0, qd0 = initial(state)
    solver = SolverVBD(model, iterations=4)
    solver.set_pass_shape(*shape)
    q_gpu, qd_gpu, _ = gpu_run(model, state, info, 6, solver=solver)
    q_ref, qd_ref, _ = oracle_run(model, q0, qd0, info, 6)
    np.testing.assert_array_equal(q_gpu, q_ref)
    np.testing.assert_array_equal(qd_gpu, qd_ref)


def _held_by_three_springs(dev, stiff, soft):
    """A particle at the origin on springs along x and y (stiff) and z (soft, stretched) to pinned particles: a block
    of diagonal about (stiff, stiff, soft)."""
    from newton_amd import ModelBuilder, ParticleFlags

    b = ModelBuilder(up_axis="Y", gravity=0.0)
    b.add_particle((0.0, 0.0, 0.0), (0.0, 0.0, 0.0), 1.0, radius=0.01, flags=int(ParticleFlags.ACTIVE))
    for k in range(3):
        at = [0.0, 0.0, 0.0]
        at[k] = 1.0
        b.add_particle(tuple(at), (0.0, 0.0, 0.0), 0.0, radius=0.01, flags=0)
        b.add_spring(0, k + 1, soft if k == 2 else stiff, 0.0)
    b.set_coloring([np.array([0]), np.array([1, 2, 3])])
    model = b.finalize(dev)
    model.spring_rest_length[2] = 0.9
    return model, model.state(), {"dt": 1.0 / 600.0, "iterations": 1}


@pytest.mark.parametrize("stiff,soft", [(1.0e16, 1.0e7), (3.0e15, 1.0e9), (1.0e13, 1.0e13), (1.0e18, 1.0e3)])
def test_determinant_beyond_single_precision_bitexact(cuda_device, stiff, soft):
    """Blocks whose single-precision determinant overflows while the squared norm does not: ill-conditioned ones are
    solved in double precision, as the oracle does, which moves the particle."""
    model, state, info = _held_by_three_springs(cuda_device, stiff, soft)
    q0, qd0 = initial(state)
    q_gpu, qd_gpu, _ = gpu_run(model, state, info, 1, solver_kwargs={"fp64_ill_conditioned": True})
    q_ref, qd_ref, _ = oracle_run(model, q0, qd0, info, 1, fp64_ill_conditioned=True)
    np.testing.assert_array_equal(q_gpu, q_ref)
    np.testing.assert_array_equal(qd_gpu, qd_ref)
    if stiff >= 1.0e6 * soft:
        assert np.abs(q_ref[0]).max() > 1.0e-4


def test_both_block_solves_are_taken_bitexact(cuda_device):
    """Bead masses whose block conditions lie on both sides of the 1e6 at which the solve turns to double precision
    (the oracle's result depends on it from 6e-8 down), around and beyond the screen's 1.6e5."""
    from newton_amd import scenes

    differ = []
    for mass in (3.0e-7, 1.0e-7, 6.0e-8, 3.0e-8, 1.0e-8, 5.0e-9):
        model, state, info = scenes.bead_rope_light(cuda_device, mass=mass)
        q0, qd0 = initial(state)
        q_gpu, qd_gpu, _ = gpu_run(model, state, info, 10, solver_kwargs={"fp64_ill_conditioned": True})
        q_ref, qd_ref, _ = oracle_run(model, q0, qd0, info, 10, fp64_ill_conditioned=True)
        np.testing.assert_array_equal(q_gpu, q_ref)
        np.testing.assert_array_equal(qd_gpu, qd_ref)
        differ.append(bool(np.any(oracle_run(model, q0, qd0, info, 10, fp64_ill_conditioned=False)[0] != q_ref)))
    assert differ == [False, False, True, True, True, True]


@pytest.mark.parametrize("scene", ["strip", "springs"])
@pytest.mark.parametrize("case", ["flat", "tiny_parts", "shrunk", "stretched", "far_out"])
def test_shared_quotient_ranges_bitexact(cuda_device, scene, case):
    """Square roots and quotients that share a reciprocal, at the edges of their ranges: exact zeros (an axis-aligned
    flat sheet), components below 2^-60 beside ordinary ones, and lengths under and over the ranges, where the IEEE
    operations take over."""
    import torch

    from newton_amd import scenes

    if scene == "strip":
        model, state, info = scenes.cloth_strip_pinned(cuda_device)
    else:
        model, state, info = scenes.cloth_drop_on_sphere(cuda_device, verts_per_side=9, springs=True)
    q = model.particle_q.clone()
    rng = np.random.default_rng(5)
    q[:, 1] = q[0, 1]
    if case == "tiny_parts":
        q[:, 1] = torch.as_tensor(rng.choice([0.0, -0.0, 1.0e-22, -3.0e-20, 2.0e-19, 1.0e-9], q.shape[0]))
    elif case != "flat":
        q *= {"shrunk": 1.0e-7, "stretched": 3.0e3, "far_out": 1.0e7}[case]
        q += torch.as_tensor(rng.normal(0.0, 0.01, q.shape), device=q.device) * q.abs().max()
    state.particle_q.copy_(q)
    q0, qd0 = initial(state)
    q_gpu, qd_gpu, _ = gpu_run(model, state, info, 1)
    q_ref, qd_ref, _ = oracle_run(model, q0, qd0, info, 1)
    np.testing.assert_array_equal(q_gpu.view(np.uint32), q_ref.view(np.uint32))
    np.testing.assert_array_equal(qd_gpu, qd_ref)


def test_penalty_ramp_bitexact(cuda_device):
    """rigid_avbd_beta > 0 exercises the per-iteration penalty update (rigid_vbd_kernels.py:4861-4926)."""
    model, state, info = _scene("strip", cuda_device)
    q0, qd0 = initial(state)
    kw = {"rigid_avbd_beta": 1.0e5, "rigid_contact_k_start": 1.0e2}
    q_gpu, qd_gpu, _ = gpu_run(model, state, info, 4, solver_kwargs=kw)
    q_ref, qd_ref, _ = oracle_run(model, q0, qd0, info, 4, avbd_beta=1.0e5, k_start=1.0e2)
    np.testing.assert_array_equal(q_gpu, q_ref)
    np.testing.assert_array_equal(qd_gpu, qd_ref)


def test_no_contacts_step(cuda_device):
    """contacts=None: pure elastic step, still bit-exact."""
    import torch

    from newton_amd.solvers import SolverVBD

    model, state, info = _scene("strip", cuda_device)
    q0, qd0 = initial(state)
    solver = SolverVBD(model, iterations=info["iterations"])
    s1 = model.state()
    solver.step(state, s1, None, None, info["dt"])
    torch.cuda.synchronize()
    om = oracle.OracleModel(model)
    _, q_ref, qd_ref = oracle.step(om, oracle.params(info["iterations"]), q0, qd0, None, None, info["dt"])
    np.testing.assert_array_equal(s1.particle_q.cpu().numpy(), q_ref)
    np.testing.assert_array_equal(s1.particle_qd.cpu().numpy(), qd_ref)


@pytest.mark.parametrize("scene", ["strip", "cube", "fan"])
def test_residual_matches_oracle(cuda_device, scene):
    """The force residual (the force-only color-pass kernels and the generic kernel) equals the oracle's
    per-vertex assembly bit for bit: the damped strip with contacts, a damped tet cube on the ground,
    and a fan whose centre has > 256 items."""
    import torch

    from newton_amd import CollisionPipeline
    from newton_amd.solvers import SolverVBD

    model, state, info = _fan_scene(cuda_device) if scene == "fan" else _scene(scene, cuda_device)
    solver = SolverVBD(model, iterations=info["iterations"])
    pipe = CollisionPipeline(model, soft_contact_margin=0.05)
    contacts = pipe.contacts()
    pipe.collide(state, contacts)
    solver.begin_step(state, contacts, info["dt"])
    solver.iterate(state, info["dt"], 1)
    g = torch.zeros_like(state.particle_q)
    r2 = solver.residual(state, info["dt"], g)
    torch.cuda.synchronize()
    om = oracle.OracleModel(model)
    oc = oracle.Contacts.from_device(contacts)
    g_ref, n_ref = oracle.residual(om, oracle.params(info["iterations"]), oc, state.particle_q.cpu().numpy(),
                                   solver.scratch("q_prev").cpu().numpy(), solver.scratch("inertia").cpu().numpy(),
                                   info["dt"], precision="f32")
    np.testing.assert_array_equal(g.cpu().numpy(), g_ref)
    assert abs(float(r2.item()) ** 0.5 - n_ref) <= 1e-6 * max(n_ref, 1.0)


def test_graph_capture_replay_matches_eager(cuda_device):
    """A captured substep (collide + step) replayed several times equals the eager run, every replay."""
    import torch

    from newton_amd import CollisionPipeline
    from newton_amd.solvers import SolverVBD

    model, state, info = _scene("hanging", cuda_device)
    q0, qd0 = initial(state)
    solver = SolverVBD(model, iterations=info["iterations"])
    pipe = CollisionPipeline(model, soft_contact_margin=0.01)
    contacts = pipe.contacts()
    s0, s1 = state, model.state()

    def substep():
        s0.clear_forces()
        pipe.collide(s0, contacts)
        solver.step(s0, s1, None, contacts, info["dt"])
        s0.particle_q.copy_(s1.particle_q)
        s0.particle_qd.copy_(s1.particle_qd)

    substep()  # warm-up (eager) step
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        snap_q, snap_qd = s0.particle_q.clone(), s0.particle_qd.clone()
        with torch.cuda.graph(graph, stream=stream):
            substep()
    torch.cuda.synchronize()
    s0.particle_q.copy_(snap_q)
    s0.particle_qd.copy_(snap_qd)
    torch.cuda.synchronize()
    replays = []
    for _ in range(4):
        graph.replay()
        torch.cuda.synchronize()
        replays.append(s0.particle_q.cpu().numpy().copy())
    q_ref, _, rec = oracle_run(model, q0, qd0, info, 5, record_every=1)
    for k in range(4):
        np.testing.assert_array_equal(replays[k], rec[k + 1])


def test_drift_600_frames(cuda_device):
    """32x32 hanging cloth, 600 frames (6000 substeps): per-frame max-abs <= 1e-5 m against the FP32 oracle.

    Also reports each implementation's error against the FP64 oracle of the same iteration.
    """
    model, state, info = _scene("hanging", cuda_device)
    q0, qd0 = initial(state)
    frames = 600
    sub = info["substeps"]
    _, _, rec_gpu = gpu_run(model, state, info, frames * sub, record_every=sub)
    _, _, rec_f32 = oracle_run(model, q0, qd0, info, frames * sub, record_every=sub)
    _, _, rec_f64 = oracle_run(model, q0, qd0, info, frames * sub, record_every=sub, precision="f64")
    per_frame = np.abs(rec_gpu - rec_f32).reshape(frames, -1).max(axis=1)
    gpu_vs_f64 = np.abs(rec_gpu.astype(np.float64) - rec_f64).reshape(frames, -1).max(axis=1)
    f32_vs_f64 = np.abs(rec_f32.astype(np.float64) - rec_f64).reshape(frames, -1).max(axis=1)
    print(f"drift GPU vs FP32 oracle: max {per_frame.max():.3e} (frame {int(per_frame.argmax())}), "
          f"final {per_frame[-1]:.3e}")
    print(f"error vs FP64 oracle: GPU max {gpu_vs_f64.max():.3e}, FP32 oracle max {f32_vs_f64.max():.3e}")
    assert np.all(np.isfinite(rec_gpu))
    assert per_frame.max() <= 1e-5


@pytest.mark.parametrize("scene", ["strip", "cube", "hanging"])
def test_128_lane_block_shape_bitexact(cuda_device, scene):
    """The 128-lane work-group shape (batches of <= 10 vertices) gives the oracle's bits too."""
    model, state, info = _scene(scene, cuda_device)
    q0, qd0 = initial(state)
    q_gpu, qd_gpu, _ = gpu_run(model, state, info, 6, block_shape=128)
    q_ref, qd_ref, _ = oracle_run(model, q0, qd0, info, 6)
    np.testing.assert_array_equal(q_gpu, q_ref)
    np.testing.assert_array_equal(qd_gpu, qd_ref)


@pytest.mark.parametrize("scene", ["strip", "cube", "hanging"])
def test_seven_wave_pass_bitexact(cuda_device, scene):
    """The 256-lane pass built for seven waves per SIMD (a smaller register budget) gives the oracle's bits."""
    model, state, info = _scene(scene, cuda_device)
    q0, qd0 = initial(state)
    q_gpu, qd_gpu, _ = gpu_run(model, state, info, 6, waves=7)
    q_ref, qd_ref, _ = oracle_run(model, q0, qd0, info, 6)
    np.testing.assert_array_equal(q_gpu, q_ref)
    np.testing.assert_array_equal(qd_gpu, qd_ref)


@pytest.mark.parametrize("scene", ["strip", "cube", "hanging"])
def test_wave_aligned_items_bitexact(cuda_device, scene):
    """Item ranges starting on wave boundaries (fewer vertices per batch, contact rows after the static
    rows) give the oracle's bits too, at both register budgets."""
    for lanes, waves in ((256, 1), (256, 7), (192, 1), (192, 7)):
        model, state, info = _scene(scene, cuda_device)
        q0, qd0 = initial(state)
        q_gpu, qd_gpu, _ = gpu_run(model, state, info, 6, aligned=True, waves=waves, block_shape=lanes)
        q_ref, qd_ref, _ = oracle_run(model, q0, qd0, info, 6)
        np.testing.assert_array_equal(q_gpu, q_ref)
        np.testing.assert_array_equal(qd_gpu, qd_ref)


def test_autotune_keeps_results(cuda_device):
    """autotune() picks a shape and leaves the state alone; the trajectory stays bit-exact."""
    import torch

    from newton_amd import CollisionPipeline
    from newton_amd.solvers import SolverVBD

    model, state, info = _scene("hanging", cuda_device)
    q0, qd0 = initial(state)
    solver = SolverVBD(model, iterations=info["iterations"])
    pipe = CollisionPipeline(model, soft_contact_margin=0.01)
    contacts = pipe.contacts()
    state.clear_forces()
    pipe.collide(state, contacts)
    before = state.particle_q.clone()
    choice = solver.autotune(state, contacts, info["dt"])
    torch.cuda.synchronize()
    assert choice["block"] in (128, 192, 256) and choice["waves"] in (1, 7) and choice["aligned"] in (0, 1)
    assert choice["ms_256"] > 0 and choice["ms_256_w7"] > 0 and choice["ms_128"] > 0
    assert torch.equal(state.particle_q, before)
    q_gpu, qd_gpu, _ = gpu_run(model, state, info, 4, solver=solver)
    q_ref, qd_ref, _ = oracle_run(model, q0, qd0, info, 4)
    np.testing.assert_array_equal(q_gpu, q_ref)
