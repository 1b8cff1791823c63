"""CPU checks of the launch tuner: it tries the settings that the scene's frames use, and no others."""
import pytest

from sbs_amd import autotune


class _Sim:
    """Records what the tuner asks of a simulation."""

    def __init__(self, path):
        self.path, self.tried = path, []

    def frame_path(self):
        return self.path, 0

    def set_launch_config(self, block, cluster_block):
        self.tried.append((block, cluster_block))

    def step(self, dt, iterations, substeps):
        pass

    def snapshot(self):
        pass

    restore = synchronize = snapshot


class _Scene:
    dt, iterations, substeps = 1.0 / 60.0, 8, 4


@pytest.mark.parametrize("path,want", [
    ("colors", [(b, c) for b in (128, 256) for c in (64, 128, 65)]),
    ("tiles", [(128, 64), (256, 64)]),
    ("islands", [(256, 64)]),
])
def test_the_tuner_tries_what_frames_use(path, want):
    sim = _Sim(path)
    best = autotune.tune_launch(sim, _Scene())
    assert sim.tried[:-1] == want and sim.tried[-1] == (best["block"], best["cluster_block"]) and sim.tried[-1] in want


def test_the_callers_candidates_are_kept_to():
    sim = _Sim("islands")
    assert autotune.tune_launch(sim, _Scene(), blocks=(64, 128), cluster_blocks=(128,))["block"] == 64
    assert sim.tried == [(64, 128), (64, 128)]
