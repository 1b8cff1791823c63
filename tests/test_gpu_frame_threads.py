"""GPU checks of two simulations stepped by two host threads at the same time, whose whole-frame or tile launches
use the same kernels with different amounts of LDS (more than the 64 KiB that need no asking for): both end in the
states they reach alone."""
import threading

import numpy as np
import pytest

import sbs_amd as S
from sbs_amd import scenes

pytestmark = pytest.mark.gpu


def _beam(nx, ny, nz):
    return scenes.cantilever(nx, ny, nz, 0.1, "neohookean", 5e5, 0.45, 1000.0, num_spheres=4, iterations=4, substeps=2,
                             cluster=True, coloring="index")


PAIRS = {
    # 3,175 and 2,601 particles, 28 B each
    "islands": lambda: [_beam(126, 4, 4), _beam(16, 16, 8)],
    # 256 tiles of a larger and of a smaller part of the particles
    "tiles": lambda: [_beam(160, 20, 20), _beam(60, 14, 14)],
}


def _run(sim, sc, frames):
    for _ in range(frames):
        sim.step(sc.dt, sc.iterations, sc.substeps)
    return sim.read_body(0)


@pytest.mark.parametrize("path", sorted(PAIRS))
def test_two_threads_reach_the_states_of_one(path):
    pair, frames = PAIRS[path](), 150
    alone = []
    for sc in pair:
        sim = scenes.build_device(sc)
        print(f"[gpu-case] {path}: {len(sc.bodies[0].x0)} particles, {sim.frame_path()}", flush=True)
        assert sim.frame_path()[0] == path
        alone.append(_run(sim, sc, frames))
        sim.close()
    sims, got, failed = [scenes.build_device(sc) for sc in pair], [None, None], []

    def work(k):
        try:
            got[k] = _run(sims[k], pair[k], frames)
        except S.SbsError as e:
            failed.append(e)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed
    for g, want in zip(got, alone):
        assert np.all(np.isfinite(g[0])) and np.array_equal(g[0], want[0]) and np.array_equal(g[1], want[1])
    for sim in sims:
        sim.close()
