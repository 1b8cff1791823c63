"""GPU checks of the launches that run several colors in tiles: positions, velocities, contacts and
multipliers are the bits of the launch-per-stage path, which frames with timing on take."""
import numpy as np
import pytest

import sbs_amd as S
from sbs_amd import scenes

pytestmark = pytest.mark.gpu


def say(msg):
    print(f"[gpu-case] {msg}", flush=True)


def _single(tets_of, kind, clusters, beta=0.0, spheres=0, self_contacts=False):
    x0, tets = tets_of
    sc = scenes.Scene("tile", gravity_is_force=False, coloring="index" if clusters else "hash")
    s2t, tris = S.boundary(len(x0), tets)
    sc.bodies.append(scenes.Body(x0=x0, tets=tets, mass=S.lumped_mass(x0, tets, 1000.0), surface=s2t, triangles=tris))
    sc.groups.append(scenes.Group(kind, 0, tets, alpha=1e-4, beta=beta, young=2e5, poisson=0.3,
                                  clusters=scenes.hex_clusters(len(tets)) if clusters else None))
    sc.planes.append(((0.0, 1.0, 0.0), (0.0, x0[:, 1].min() + 0.01, 0.0), (-1e30,) * 3, (1e30,) * 3))
    rng = np.random.default_rng(3)
    for _ in range(spheres):
        sc.spheres.append((tuple(rng.uniform(x0.min(0), x0.max(0))), 0.05))
    if self_contacts:
        sc.body_contacts = (0.0, 0.0, 0.0)
    return sc


def _loose_point(sc):
    """A second body with particles and no constraints."""
    sc.bodies.append(scenes.Body(x0=np.array([[9.0, 1.0, 0.0], [9.5, 1.0, 0.0]]), tets=np.zeros((0, 4), np.uint32)))
    return sc


def _with_tiny_bodies(n, tets_of, kind, clusters, beta):
    """One large body and n bodies of one cell, all in one group: a tiny body's tile has elements of one color
    (clusters) or of six, and none in the launches of the other colors."""
    parts = [tets_of] + [S.box6(1, 1, 1, 0.1, (0.0, 0.05, 3.0 + k)) for k in range(n)]
    sc = scenes.Scene("tile", gravity_is_force=False, coloring="index" if clusters else "hash")
    for x0, tets in parts:
        s2t, tris = S.boundary(len(x0), tets)
        sc.bodies.append(scenes.Body(x0=x0, tets=tets, mass=S.lumped_mass(x0, tets, 1000.0), surface=s2t,
                                     triangles=tris))
    tets = np.concatenate([t for _, t in parts])
    sc.groups.append(scenes.Group(kind, np.repeat(np.arange(n + 1, dtype=np.uint32), [len(t) for _, t in parts]), tets,
                                  alpha=1e-4, beta=beta, young=np.full(len(tets), 2e5),
                                  poisson=np.full(len(tets), 0.3),
                                  clusters=scenes.hex_clusters(len(tets)) if clusters else None))
    sc.planes.append(((0.0, 1.0, 0.0), (0.0, 0.01, 0.0), (-1e30,) * 3, (1e30,) * 3))
    return sc


def _batch(n, sizes, seed):
    sc = scenes.batch(n, sizes, seed=seed, young_range=(1e4, 1e5), drop_range=(-0.01, 0.0))
    sc.body_contacts = (0.0, 0.0, 0.0)
    return sc


# contacts between bodies keep a scene of small bodies from the one-workgroup-per-body launch
CASES = {
    "hex_one_cell": lambda: _single(S.box6(1, 1, 1, 0.1), "neohookean", True, self_contacts=True),
    "hex_thin": lambda: _single(S.box6(40, 2, 1, 0.1), "neohookean", True, spheres=3, self_contacts=True),
    "hex_wide": lambda: _single(S.box6(41, 17, 15, 0.1), "neohookean", True, spheres=3),
    "hex_damped": lambda: _single(S.box6(31, 18, 17, 0.1), "neohookean", True, beta=1e-3),
    "hex_green": lambda: _single(S.box6(33, 13, 12, 0.1), "green", True, spheres=2),
    "hex_green_damped": lambda: _single(S.box6(23, 21, 15, 0.1), "green", True, beta=1e-3),
    "tets_green": lambda: _loose_point(_single(S.bar5(17, 18, 41), "green", False, spheres=2)),
    "tets_green_damped": lambda: _single(S.bar5(18, 18, 31), "green", False, beta=1e-3),
    "tets_neohookean": lambda: _single(S.ellipsoid6(0.9, 1.1, 1.4, 0.1), "neohookean", False, spheres=2),
    "tets_damped": lambda: _single(S.box6(23, 19, 17, 0.1), "neohookean", False, beta=1e-3),
    # tiles without an element of a launch's colors: nothing of theirs reaches the damping term
    "hex_damped_tiny": lambda: _with_tiny_bodies(5, S.box6(130, 22, 22, 0.1), "neohookean", True, 1e-3),
    "hex_green_damped_tiny": lambda: _loose_point(_with_tiny_bodies(5, S.box6(23, 21, 15, 0.1), "green", True, 1e-3)),
    "tets_damped_tiny": lambda: _loose_point(_with_tiny_bodies(5, S.box6(23, 19, 17, 0.1), "neohookean", False, 1e-3)),
    "tets_green_damped_tiny": lambda: _loose_point(_with_tiny_bodies(5, S.bar5(18, 18, 31), "green", False, 1e-3)),
    "hex_damped_loose": lambda: _loose_point(_single(S.box6(31, 18, 17, 0.1), "neohookean", True, beta=1e-3)),
    # tiles with more than 256 elements of a color, run in two parts
    "hex_two_chunks": lambda: _single(S.box6(280, 34, 35, 0.1), "neohookean", True, spheres=3),
    "tets_two_chunks": lambda: _single(S.box6(110, 14, 14, 0.1), "neohookean", False, spheres=3),
    "tets_green_wide": lambda: _single(S.box6(12, 12, 10, 0.1), "green", False, spheres=4),
    "batch_contacts": lambda: _batch(9, (6.0, 9000.0), 4),
    "batch_wide": lambda: _batch(5, (20000.0, 90000.0), 6),
}

# colors a launch, where not all of a cluster group's or 7 of a tet group's
COLORS = {"hex_one_cell": 1, "hex_thin": 4, "hex_two_chunks": 4, "batch_wide": 4, "hex_damped_tiny": 4}


@pytest.mark.parametrize("name", sorted(CASES))
@pytest.mark.parametrize("graphs", [False, True])
def test_tiles_are_the_staged_frames(name, graphs):
    sc = CASES[name]()
    say(f"tile {name}: {sc.num_tets} tets, {sc.num_vertices} vertices, graphs {graphs}")
    a, b = scenes.build_device(sc), scenes.build_device(sc)
    assert a.frame_path() == ("tiles", COLORS.get(name, 8 if sc.groups[0].clusters is not None else 7))
    b.set_timing(True)
    a.use_graphs(graphs)
    rng = np.random.default_rng(8)
    for k, body in enumerate(sc.bodies):
        x = body.x0 * (1.0 + 0.02 * rng.uniform(-1, 1, 3))
        v = rng.uniform(-0.3, 0.3, body.x0.shape)
        for sim in (a, b):
            sim.write_body(k, x, v)
    for frame, (iterations, substeps) in enumerate([(4, 2), (4, 2), (1, 1), (0, 2), (7, 3)]):
        for sim in (a, b):
            sim.step(1.0 / 60.0, iterations, substeps)
        for k in range(len(sc.bodies)):
            for got, want in zip(a.read_body(k), b.read_body(k)):
                assert np.all(np.isfinite(got)) and np.array_equal(got, want), (name, frame, k)
        assert np.array_equal(a.residual(0, 1.0 / 60.0 / substeps), b.residual(0, 1.0 / 60.0 / substeps)), (name, frame)


@pytest.mark.parametrize("mode", ["previous", "learned", "explicit"])
@pytest.mark.parametrize("iterations", [1, 4, 5])
def test_tiles_after_a_warm_start(mode, iterations):
    sc = _single(S.box6(24, 17, 18, 0.1), "neohookean", True, spheres=4)
    say(f"tile warm start {mode}, {iterations} iterations")
    a, b = scenes.build_device(sc), scenes.build_device(sc)
    assert a.frame_path()[0] == "tiles"
    b.set_timing(True)
    nets = []
    for sim in (a, b):
        net = S.Mlp(39, 12, 2) if mode == "learned" else None
        if net:
            net.set_normalization(np.zeros(39), np.full(39, 0.1), np.full(12, 1e-3))
        nets.append(net)
        sim.set_warm_start(mode, net)
        sim.set_warm_start_scale(0.5 if mode != "explicit" else 0.2)
        for _ in range(2):
            sim.step(1.0 / 60.0, iterations, 4)
    for got, want in zip(a.read_body(0), b.read_body(0)):
        assert np.all(np.isfinite(got)) and np.array_equal(got, want)
    a.close(), b.close()


@pytest.mark.parametrize("mode", ["previous", "explicit"])
@pytest.mark.parametrize("iterations", [1, 4, 5])
def test_tiles_of_single_tets_after_a_warm_start(mode, iterations):
    sc = CASES["tets_neohookean"]()
    say(f"tile warm start {mode} of single tets, {iterations} iterations")
    a, b = scenes.build_device(sc), scenes.build_device(sc)
    assert a.frame_path() == ("tiles", 7)
    b.set_timing(True)
    for sim in (a, b):
        sim.set_warm_start(mode)
        sim.set_warm_start_scale(0.5 if mode != "explicit" else 0.2)
        for _ in range(2):
            sim.step(1.0 / 60.0, iterations, 4)
    for got, want in zip(a.read_body(0), b.read_body(0)):
        assert np.all(np.isfinite(got)) and np.array_equal(got, want)
    assert np.array_equal(a.residual(0, 1.0 / 240.0), b.residual(0, 1.0 / 240.0))
    a.close(), b.close()
