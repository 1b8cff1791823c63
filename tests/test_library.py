"""CPU checks of the product library: it loads, exports every symbol include/sbs_gpu.h declares,
its host mesh utilities match the oracle bit for bit, and argument errors come back as status
codes. No device work is done here."""
import ctypes

import numpy as np
import pytest

import oracle as O
import sbs_amd as S
from sbs_amd import scenes


def test_library_exports_every_header_symbol():
    L = S.lib()
    names = S.header_functions()
    assert len(names) >= 25
    for n in names:
        assert hasattr(L, n), n


@pytest.mark.parametrize("dims", [(12, 4, 4), (5, 2, 2), (2, 2, 2), (7, 3, 5), (1, 3, 3)])
def test_bar5_matches_oracle(dims):
    a, b = S.bar5(*dims), O.bar5(*dims)
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])


@pytest.mark.parametrize("dims", [(10, 3, 3), (4, 5, 6), (1, 1, 1)])
def test_box6_and_boundary_match_oracle(dims):
    a = S.box6(*dims, 0.1, (0.3, -0.2, 0.1))
    b = O.box6(*dims, 0.1, (0.3, -0.2, 0.1))
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
    s1, t1 = S.boundary(len(a[0]), a[1])
    s2, t2, _ = O.boundary(len(a[0]), a[1])
    assert np.array_equal(s1, s2) and np.array_equal(t1, t2)


def test_boundary_of_reference_bar_matches_oracle():
    p, t = S.bar5(12, 4, 4)
    s1, t1 = S.boundary(len(p), t)
    s2, t2, _ = O.boundary(len(p), t)
    assert np.array_equal(s1, s2) and np.array_equal(t1, t2)


def test_lumped_mass_totals_density_times_volume():
    p, t = S.box6(5, 4, 3, 0.2)
    m = S.lumped_mass(p, t, 750.0)
    assert np.isclose(m.sum(), 750.0 * 1.0 * 0.8 * 0.6, rtol=1e-12)
    # a corner vertex of the lattice belongs to 1 or 2 tets of its cell (the diagonal corners to 6)
    assert m.min() > 0


def test_mesh_errors_are_status_codes():
    L = S.lib()
    tets = np.array([0, 1, 2, 9], dtype=np.uint32)
    ns, nt = ctypes.c_uint32(), ctypes.c_uint32()
    code = L.sbs_mesh_boundary(4, tets.ctypes.data_as(ctypes.POINTER(ctypes.c_uint32)), 1, None, None,
                               ctypes.byref(ns), ctypes.byref(nt))
    assert code == 1
    assert b"out of range" in L.sbs_gpu_last_error()


def test_benchmark_scene_sizes():
    sc = scenes.beam_540()
    assert (sc.num_vertices, sc.num_tets, len(sc.bodies[0].surface)) == (176, 540, 140)
    pinned = sc.bodies[0].mass == 0
    assert pinned.sum() == 4 * 4 and np.all(sc.bodies[0].x0[pinned, 0] == 0.0)
    assert np.isclose(sc.bodies[0].mass.sum() + 0, 1000.0 * 1.0 * 0.3 * 0.3 - 0, rtol=0.2)
    demo = scenes.reference_demo()
    assert (demo.num_vertices, demo.num_tets) == (192, 495)


def test_cpp_mirror_example_builds_against_the_c_abi():
    # the C++ mirror of simulation_t / timestep_t compiles and links against the library
    import os
    import subprocess
    import tempfile
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    pkg = os.path.join(root, "soft-body-simulator_amd")
    with tempfile.TemporaryDirectory() as d:
        out = os.path.join(d, "demo")
        subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", f"-I{root}/include", f"-I{pkg}/host",
                        f"{pkg}/host/examples/reference_demo.cpp", "-o", out, f"-L{pkg}/_build", "-lsbs_gpu",
                        f"-Wl,-rpath,{pkg}/_build"], check=True)
        assert os.path.exists(out)


def test_ellipsoid6_cells_volume_and_conformity():
    import itertools
    rx, ry, rz, h = 0.33, 0.21, 0.27, 0.05
    pos, tets = S.ellipsoid6(rx, ry, rz, h)
    # brute force: cells of the centred lattice whose centres are inside
    n = [int(np.ceil(2 * r / h)) for r in (rx, ry, rz)]
    o = [-0.5 * k * h for k in n]
    inside = 0
    for i, j, k in itertools.product(*(range(a) for a in n)):
        c = np.array([o[0] + (i + 0.5) * h, o[1] + (j + 0.5) * h, o[2] + (k + 0.5) * h])
        inside += np.sum((c / np.array([rx, ry, rz])) ** 2) <= 1.0
    assert len(tets) == 6 * inside
    e = pos[tets[:, :3]] - pos[tets[:, 3:4]]
    V = np.linalg.det(np.transpose(e, (0, 2, 1))) / 6.0
    assert np.all(V < 0) and np.isclose(-V.sum(), inside * h ** 3)
    faces = {}
    for t in tets:
        for f in itertools.combinations(sorted(t), 3):
            faces[f] = faces.get(f, 0) + 1
    assert max(faces.values()) == 2
    assert len(np.unique(tets)) == len(pos)  # every vertex is used


def test_batch_scene_shape():
    sc = scenes.batch(6, tet_range=(2e3, 1e4))
    g = sc.groups[0]
    assert len(sc.bodies) == 6 and len(g.conn) == sum(len(b.tets) for b in sc.bodies)
    assert np.all(np.diff(g.body.astype(np.int64)) >= 0)
    for b in sc.bodies:
        assert b.x0[:, 1].min() >= 0.5 - 1e-9


def test_batch_scene_clusters_take_eight_balanced_colors():
    # ellipsoid cells come grouped by lattice parity, so the index-order greedy coloring of the
    # hex clusters needs one color per parity class, for every body of the batch
    from helpers import build_oracle
    sc = scenes.batch(8, tet_range=(2e3, 8e3))
    orc = build_oracle(sc)
    orc.step(sc.dt, 1, 1)
    col, nc = orc.group_colors(0, sc.num_tets)
    assert nc == 8
    per_color = np.bincount(col, minlength=8)
    assert per_color.min() > 0.5 * per_color.max()  # odd box dimensions make parity classes uneven


def test_null_handles_are_status_codes():
    # every sbs_gpu_* entry point taking the handle first rejects a null one with a status code and a
    # message (no device work: the check comes before any)
    from sbs_amd import _lib
    L = S.lib()
    skip = {"sbs_gpu_destroy", "sbs_gpu_last_error", "sbs_gpu_create", "sbs_gpu_extract_boundary"}
    checked = 0
    for name, argtypes in _lib._SIGS.items():
        if not name.startswith("sbs_gpu_") or name in skip or not argtypes or argtypes[0] is not _lib._p:
            continue
        args = []
        for t in argtypes:
            if t in (_lib._d, _lib._f):
                args.append(t(0.0))
            elif t in (_lib._i, _lib._u32, _lib._u64):
                args.append(t(0))
            else:
                args.append(None)
        rc = getattr(L, name)(*args)
        assert rc != 0, name
        assert L.sbs_gpu_last_error().decode(), name
        checked += 1
    assert checked >= 30


def test_diverged_capture_episodes_are_named():
    # episodes (first row, end row, largest frame residual): a blow-up (non-finite, or 20x the
    # median of the episodes' largest residuals) is named; the others are kept
    from sbs_amd.autotune import diverged_episodes
    rec = [(0, 10, 2.0), (10, 20, 2.5), (20, 30, float("inf")), (30, 40, 1.8), (40, 50, 60.0), (50, 60, 3.0)]
    assert diverged_episodes(rec) == [(20, 30), (40, 50)]
    assert diverged_episodes(rec[:2]) == []
    assert diverged_episodes([(0, 5, float("nan"))]) == [(0, 5)]


def test_body_contact_workloads_are_the_batches_with_contacts():
    # the contact workloads are the batch configurations themselves (same bodies, places and
    # materials) with contacts between bodies and of each body with its own surface
    a, b = scenes.batch(8), scenes.batch_512_contacts(8)
    assert a.body_contacts is None and b.body_contacts == (0.0, 0.0, 0.0)
    assert all(np.array_equal(x.x0, y.x0) and np.array_equal(x.tets, y.tets) for x, y in zip(a.bodies, b.bodies))
    assert np.array_equal(a.groups[0].young, b.groups[0].young)
    big = scenes.batch_512_large_contacts(4, large=(1, 2e3))
    assert big.body_contacts == (0.0, 0.0, 0.0) and big.name.endswith("_with_body_contacts")
    assert len(big.bodies) == 5


def test_bench_refuses_more_than_one_gpu():
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, os.path.join(root, "bench.py"), "--gpus", "2"], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 2 and "--gpus must be 1" in r.stderr


@pytest.mark.parametrize("device", [0, 63])
def test_refused_boundary_extraction_leaves_its_outputs_alone(device):
    """A bad index is the caller's error with a device, without one, and on a device that does not exist."""
    L = S.lib()
    tets = np.array([0, 1, 2, 3, 1, 2, 3, 9], dtype=np.uint32)
    ns, nt = ctypes.c_uint32(77), ctypes.c_uint32(78)
    code = L.sbs_gpu_extract_boundary(device, 9, tets.ctypes.data_as(ctypes.POINTER(ctypes.c_uint32)), 2, None, None,
                                      ctypes.byref(ns), ctypes.byref(nt))
    assert code == 1 and b"out of range" in L.sbs_gpu_last_error()
    assert (ns.value, nt.value) == (77, 78)
