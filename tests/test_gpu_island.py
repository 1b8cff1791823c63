"""GPU checks of the whole-frame launch of small bodies (one workgroup per body): positions, velocities
and multipliers are the bits of the launch-per-stage path, which frames with timing on take."""
import numpy as np
import pytest

import sbs_amd as S
from sbs_amd import scenes

pytestmark = pytest.mark.gpu


def say(msg):
    print(f"[gpu-case] {msg}", flush=True)


def _single(tets_of, kind, clusters, beta=0.0, spheres=0, poisson=0.3):
    x0, tets = tets_of
    sc = scenes.Scene("island", gravity_is_force=False, coloring="index" if clusters else "hash")
    s2t, tris = S.boundary(len(x0), tets)
    sc.bodies.append(scenes.Body(x0=x0, tets=tets, mass=S.lumped_mass(x0, tets, 1000.0), surface=s2t, triangles=tris))
    sc.groups.append(scenes.Group(kind, 0, tets, alpha=1e-4, beta=beta, young=2e5, poisson=poisson,
                                  clusters=scenes.hex_clusters(len(tets)) if clusters else None))
    sc.planes.append(((0.0, 1.0, 0.0), (0.0, 0.01, 0.0), (-1e30,) * 3, (1e30,) * 3))
    rng = np.random.default_rng(3)
    for _ in range(spheres):
        sc.spheres.append((tuple(rng.uniform(x0.min(0), x0.max(0))), 0.05))
    return sc


def _loose_point(sc):
    """A second body with particles and no constraints."""
    sc.bodies.append(scenes.Body(x0=np.array([[9.0, 1.0, 0.0], [9.5, 1.0, 0.0]]), tets=np.zeros((0, 4), np.uint32)))
    return sc


def _many(n, tets_of, kind, clusters=False, beta=0.0):
    """n bodies of one mesh side by side."""
    x0, tets = tets_of
    sc = scenes.Scene("islands", gravity_is_force=False, coloring="index" if clusters else "hash")
    s2t, tris = S.boundary(len(x0), tets)
    step = np.array([float(np.ptp(x0[:, 0])) + 1.0, 0.0, 0.0])
    for k in range(n):
        sc.bodies.append(scenes.Body(x0=x0 + k * step, tets=tets, mass=S.lumped_mass(x0, tets, 1000.0), surface=s2t,
                                     triangles=tris))
    sc.groups.append(scenes.Group(kind, np.repeat(np.arange(n, dtype=np.uint32), len(tets)), np.tile(tets, (n, 1)),
                                  alpha=1e-4, beta=beta, young=np.full(n * len(tets), 2e5),
                                  poisson=np.full(n * len(tets), 0.3),
                                  clusters=scenes.hex_clusters(n * len(tets)) if clusters else None))
    sc.planes.append(((0.0, 1.0, 0.0), (0.0, 0.01, 0.0), (-1e30,) * 3, (1e30,) * 3))
    return sc


CASES = {
    # elements of a stage: under one wave, one to four waves, colors that some bodies have no element of
    "hex_small": lambda: _single(S.box6(5, 3, 4, 0.1), "neohookean", True, spheres=3),
    "hex_one_cell": lambda: _single(S.box6(1, 1, 1, 0.1), "neohookean", True),
    "hex_256": lambda: _single(S.box6(16, 16, 8, 0.1), "neohookean", True),
    "hex_damped": lambda: _single(S.box6(6, 5, 4, 0.1), "neohookean", True, beta=1e-3),
    "hex_green": lambda: _single(S.box6(6, 5, 4, 0.1), "green", True, spheres=2),
    "hex_green_damped": lambda: _single(S.box6(6, 5, 4, 0.1), "green", True, beta=1e-3),
    "tets_green": lambda: _loose_point(_single(S.bar5(4, 4, 12), "green", False, spheres=2)),
    "tets_green_damped": lambda: _single(S.bar5(3, 3, 5), "green", False, beta=1e-3),
    "tets_neohookean": lambda: _single(S.ellipsoid6(0.4, 0.3, 0.5, 0.1), "neohookean", False, beta=1e-3),
    # more elements in a stage than 256 lanes
    "tets_wide": lambda: _single(S.box6(13, 13, 11, 0.1), "neohookean", False, spheres=4),
    # the same of Green tets, with enough bodies that one workgroup each is the faster way
    "tets_green_wide_many": lambda: _many(45, S.box6(12, 12, 10, 0.1), "green"),
    "tets_wide_damped": lambda: _single(S.box6(13, 13, 11, 0.1), "neohookean", False, beta=1e-3),
    "tets_green_wide_many_damped": lambda: _many(45, S.box6(12, 12, 10, 0.1), "green", beta=1e-3),
    # the same of hex cells (workgroups of 512 threads)
    "hex_wide_damped": lambda: _many(60, S.box6(15, 15, 14, 0.1), "neohookean", True, beta=1e-3),
    "hex_green_wide": lambda: _many(60, S.box6(15, 15, 14, 0.1), "green", True),
    "hex_green_wide_damped": lambda: _many(60, S.box6(15, 15, 14, 0.1), "green", True, beta=1e-3),
    # 5,650 particles, the most that an island holds
    "hex_largest": lambda: _many(60, S.box6(112, 9, 4, 0.1), "neohookean", True),
    # bodies from one cell up, boxes and ellipsoids
    "batch": lambda: scenes.batch(9, (6.0, 9000.0), seed=4, young_range=(1e4, 1e5), drop_range=(-0.01, 0.0)),
    # up to 4,862 particles and 540 cells of a color in a body, enough bodies that it is worth it
    "batch_wide": lambda: scenes.batch(70, (9000.0, 24000.0), seed=7, young_range=(1e4, 1e5), drop_range=(-0.01, 0.0)),
}

# threads of the workgroup where a stage of a body has more than 256 elements
WIDE = {"tets_wide": 1024, "tets_wide_damped": 1024, "tets_green_wide_many": 1024,
        "tets_green_wide_many_damped": 1024, "batch_wide": 512, "hex_wide_damped": 512, "hex_green_wide": 512,
        "hex_green_wide_damped": 512, "hex_largest": 512}


@pytest.mark.parametrize("name", sorted(CASES))
@pytest.mark.parametrize("graphs", [False, True])
def test_island_frames_are_the_staged_frames(name, graphs):
    sc = CASES[name]()
    say(f"island {name}: {sc.num_tets} tets, {sc.num_vertices} vertices, graphs {graphs}")
    a, b = scenes.build_device(sc), scenes.build_device(sc)
    assert a.frame_path() == ("islands", WIDE.get(name, 256))
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
def test_island_iterations_after_a_warm_start(mode):
    sc = CASES["hex_256"]()
    say(f"island warm start {mode}")
    a, b = scenes.build_device(sc), scenes.build_device(sc)
    assert a.frame_path()[0] == "islands"
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
            sim.step(1.0 / 60.0, 5, 4)
    for got, want in zip(a.read_body(0), b.read_body(0)):
        assert np.all(np.isfinite(got)) and np.array_equal(got, want)
    a.close(), b.close()


@pytest.mark.parametrize("mode", ["previous", "explicit"])
@pytest.mark.parametrize("name", ["tets_neohookean", "tets_wide"])
def test_island_iterations_of_single_tets_after_a_warm_start(name, mode):
    sc = CASES[name]()
    say(f"island warm start {mode} of {name}")
    a, b = scenes.build_device(sc), scenes.build_device(sc)
    assert a.frame_path() == ("islands", WIDE.get(name, 256))
    b.set_timing(True)
    for sim in (a, b):
        sim.set_warm_start(mode)
        sim.set_warm_start_scale(0.5 if mode != "explicit" else 0.2)
        for iterations in (5, 1, 4):
            sim.step(1.0 / 60.0, iterations, 4)
    for got, want in zip(a.read_body(0), b.read_body(0)):
        assert np.all(np.isfinite(got)) and np.array_equal(got, want)
    assert np.array_equal(a.residual(0, 1.0 / 240.0), b.residual(0, 1.0 / 240.0))
    a.close(), b.close()


def test_bodies_of_more_particles_than_an_island_holds():
    sc = _many(60, S.box6(28, 14, 12, 0.1), "neohookean", True)
    assert len(sc.bodies[0].x0) == 5655
    dev = scenes.build_device(sc)
    assert dev.frame_path()[0] != "islands"
    dev.close()
