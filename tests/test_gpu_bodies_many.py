"""GPU checks of the contacts of many surface vertices, where fewer lanes share a vertex than in the scenes
of test_gpu_bodies.py: bodies side by side, and folded onto themselves, against the oracle."""
import numpy as np
import pytest

from helpers import build_oracle
from sbs_amd import scenes
from test_gpu_bodies import _sorted

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("frames", [1, 10])
def test_contacts_of_many_vertices_match_the_oracle(frames):
    sc = scenes.batch(64, tet_range=(2e3, 2e4), name="batch_64", drop_range=(-0.004, 0.02))
    sc.body_contacts = (0.0, 0.0, 0.0)
    vertices = sum(len(b.surface) for b in sc.bodies)
    print(f"[gpu-case] contacts of {vertices} surface vertices after {frames} frames", flush=True)
    assert vertices > 32768
    dev = scenes.build_device(sc)
    for _ in range(frames):
        dev.step(sc.dt, sc.iterations, sc.substeps)
    orc = build_oracle(sc)
    for b in range(len(sc.bodies)):
        x, v = dev.read_body(b)
        assert np.all(np.isfinite(x))
        dev.write_body(b, x, v)
        orc.set_body_state(b, x, v)
    ids_d, qn_d = _sorted(*dev.read_contacts())
    ids_o, qn_o = _sorted(*orc.detect_contacts())
    assert np.sum(ids_d[:, 3] >= len(sc.planes)) > 100
    assert dev.contact_overflow() == 0
    assert np.array_equal(ids_d, ids_o)
    assert np.array_equal(qn_d[:, :3], qn_o[:, :3])
    assert np.allclose(qn_d[:, 3:], qn_o[:, 3:], rtol=0, atol=1e-7)
