"""The color-pass layout (newton_amd/csrc/vbd_layout.h) on the CPU: every vertex in one batch or on the generic
path, every item's vertices found through the batch's vertex list, rows in canonical order, slots in range."""

import ctypes
import subprocess
from pathlib import Path

import numpy as np
import pytest

from newton_amd import ModelBuilder, scenes
from newton_amd.solvers.solver_vbd import color_layout

HERE = Path(__file__).resolve().parent


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    so = tmp_path_factory.mktemp("layout") / "layout_check.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-o", str(so), str(HERE / "layout_check.cpp")],
                   check=True)
    return ctypes.CDLL(str(so))


def _fan(segments):
    """A fan whose centre has `segments` triangles and twice as many hinges and neighbours."""
    b = ModelBuilder(up_axis="Y")
    a = 2.0 * np.pi * np.arange(segments) / segments
    verts = [(0.0, 0.0, 0.0)] + [(r * np.cos(x), 0.0, r * np.sin(x)) for r in (0.5, 1.0) for x in a]
    tris = []
    for i in range(segments):
        j = (i + 1) % segments
        tris += [0, 1 + i, 1 + j, 1 + i, 1 + segments + i, 1 + j]
    b.add_cloth_mesh(pos=(0.0, 0.0, 0.0), rot=(0.0, 0.0, 0.0, 1.0), scale=1.0, vel=(0.0, 0.0, 0.0), vertices=verts,
                     indices=tris, density=0.1, tri_ke=1.0e3, tri_ka=1.0e3, tri_kd=1.0e-3, edge_ke=0.1, edge_kd=0.0)
    b.color(include_bending=True)
    return b.finalize("cpu")


def _spring_tet_cloth():
    """A cloth whose corner carries a spring and a tet cube: five kinds at one vertex, more than 256 aligned lanes."""
    b = ModelBuilder(up_axis="Y")
    b.add_soft_grid(pos=(0.0, 0.0, 0.0), rot=(0.0, 0.0, 0.0, 1.0), vel=(0.0, 0.0, 0.0), dim_x=2, dim_y=2, dim_z=2,
                    cell_x=0.1, cell_y=0.1, cell_z=0.1, density=100.0, k_mu=1.0e3, k_lambda=1.0e3, k_damp=0.0,
                    tri_ke=1.0e3, tri_ka=1.0e3, tri_kd=0.0, edge_ke=0.1, edge_kd=0.0)
    b.add_spring(0, b.particle_count - 1, 10.0, 0.0)
    b.color(include_bending=True)
    return b.finalize("cpu")


MODELS = {
    "strip": lambda: scenes.cloth_strip_pinned("cpu")[0],
    "cloth_17": lambda: scenes.cloth_hanging("cpu", verts_per_side=17)[0],
    "springs": lambda: scenes.cloth_drop_on_sphere("cpu", verts_per_side=13, springs=True)[0],
    "rope": lambda: scenes.bead_rope_light("cpu")[0],
    "cube": lambda: scenes.soft_cube("cpu", cells=4)[0],
    "worlds": lambda: scenes.cloth_batched("cpu", worlds=3, side_min=5, side_max=12)[0],
    "fan_40": lambda: _fan(40),    # 120 items, 81 vertices: every packed shape holds it
    "fan_80": lambda: _fan(80),    # 240 items, 161 vertices: only the widest shape holds it
    "fan_120": lambda: _fan(120),  # generic path
    "five_kinds": _spring_tet_cloth,
}


def _model_args(m):
    """The leading arguments of layout_check.cpp's functions, and the arrays they point to."""
    adj = m.soft_mesh_adjacency
    co, cp = color_layout(m)

    def arr(x, dtype):
        x = x.cpu().numpy() if hasattr(x, "cpu") else x
        return np.ascontiguousarray(np.zeros(1) if x is None else x, dtype=dtype).reshape(-1)

    f, i = np.float32, np.int32
    keep = [arr(m.particle_mass, f), arr(m.particle_flags, i), arr(m.tri_indices, i), arr(m.tri_materials, f),
            arr(m.edge_indices, i), arr(m.edge_bending_properties, f), arr(m.tet_indices, i), arr(m.tet_materials, f),
            arr(adj.v_adj_tris_offsets, i), arr(adj.v_adj_tris, i), arr(adj.v_adj_edges_offsets, i),
            arr(adj.v_adj_edges, i), arr(adj.v_adj_tets_offsets, i), arr(adj.v_adj_tets, i),
            arr(m.spring_indices if m.spring_count else None, i), co, cp]
    return [m.particle_count, m.tri_count, m.edge_count, m.tet_count, int(m.spring_count), len(co) - 1,
            *[a.ctypes.data_as(ctypes.c_void_p) for a in keep]], keep


@pytest.mark.parametrize("name", sorted(MODELS))
@pytest.mark.parametrize("block,aligned", [(256, 0), (256, 1), (192, 0), (192, 1), (128, 0), (128, 1)])
def test_layout(check, name, block, aligned):
    m = MODELS[name]()
    args, keep = _model_args(m)
    stats = (ctypes.c_longlong * 4)()
    rc = check.check_layout(*args, block, block // 12, aligned, stats)
    assert rc == 0, f"layout_check.cpp:{rc}"
    assert stats[0] + stats[1] > 0
    if name == "fan_120":
        assert stats[1] >= 1


@pytest.mark.parametrize("name", ["cloth_17", "springs", "cube", "fan_80", "five_kinds"])
@pytest.mark.parametrize("block,aligned", [(256, 0), (192, 1)])
def test_damping_edit_keeps_the_layout(check, name, block, aligned):
    """Damping switched from or to zero changes no array size, batch range or launch argument, so a rebuild writes in
    place under captured graphs."""
    args, keep = _model_args(MODELS[name]())
    rc = check.check_damping_edit(*args, block, block // 12, aligned)
    assert rc == 0, f"layout_check.cpp:{rc}"


def _spring_cloth(tri_ke, tri_ka):
    b = ModelBuilder(up_axis="Y")
    b.add_cloth_grid(pos=(0.0, 0.0, 0.0), rot=(0.0, 0.0, 0.0, 1.0), vel=(0.0, 0.0, 0.0), dim_x=5, dim_y=4, cell_x=0.1,
                     cell_y=0.1, mass=0.1, tri_ke=tri_ke, tri_ka=tri_ka, tri_kd=0.0, edge_ke=0.0, edge_kd=0.0)
    for i in range(29):
        if i % 6 != 5:
            b.add_spring(i, i + 1, 10.0, 0.0)
    b.color()
    return b.finalize("cpu")


@pytest.mark.parametrize("name,shared", [("cloth_17", 0), ("springs", 0), ("cube", 0), ("fan_80", 0), ("rope", 0),
                                         ("springs_only", 1), ("no_area_term", 1)])
def test_corners_of_one_color_are_found(check, name, shared):
    """Triangles without stiffness are not part of the coloring graph: their corners, and those of their edges, may
    share a color, and a color pass then moves what an edge or face contact of the same pass reads."""
    build = {"springs_only": lambda: _spring_cloth(0.0, 0.0), "no_area_term": lambda: _spring_cloth(1.0e3, 0.0)}
    args, keep = _model_args(build.get(name, MODELS.get(name))())
    assert check.shares_corners(*args, 256, 21, 0) == shared


@pytest.mark.parametrize("name,block", [("cloth_17", 128), ("strip", 128), ("worlds", 128), ("cloth_17", 192),
                                        ("springs", 192), ("springs", 256), ("cube", 128), ("five_kinds", 256)])
def test_wave_aligned_ranges_hold_what_fits(check, name, block):
    """Wave-aligned layouts send no vertex to the generic path whose kinds fit with both forms of its hinges in one
    range."""
    m = MODELS[name]()
    args, keep = _model_args(m)
    stats = (ctypes.c_longlong * 4)()
    rc = check.check_layout(*args, block, block // 12, 1, stats)
    assert rc == 0, f"layout_check.cpp:{rc}"
    assert stats[1] == 0


def test_every_combination_of_kinds_has_a_pass(check):
    rc = check.check_kinds()
    assert rc == 0, f"layout_check.cpp:{rc}"
