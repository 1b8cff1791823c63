"""GPU checks of the packed reads of a body's state: particle counts around the read chunk (16,384) and its
two buffers, either output left out, a larger body after a smaller one."""
import ctypes

import numpy as np
import pytest

import sbs_amd as S
from sbs_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [(1, 7), (16383, 16384, 16385), (32768, 32769), (100001, 3)])
def test_read_returns_what_was_written(sizes):
    print(f"[gpu-case] read bodies of {sizes} particles", flush=True)
    rng = np.random.default_rng(sum(sizes))
    sim = S.Simulation()
    for n in sizes:
        sim.add_body(rng.normal(size=(n, 3)))
    sim.commit()
    state = [(rng.normal(size=(n, 3)), rng.normal(size=(n, 3)).astype(np.float32).astype(np.float64)) for n in sizes]
    for b, (x, v) in enumerate(state):
        sim.write_body(b, x, v)
    for b, (x, v) in enumerate(state):
        got = sim.read_body(b)
        assert np.array_equal(got[0], x) and np.array_equal(got[1], v)
        only = np.full((sizes[b], 3), np.nan)
        p = only.ctypes.data_as(ctypes.POINTER(ctypes.c_double))
        _lib.check(_lib.lib().sbs_gpu_read_body(sim.h, b, p, None))
        assert np.array_equal(only, x)
        _lib.check(_lib.lib().sbs_gpu_read_body(sim.h, b, None, p))
        assert np.array_equal(only, v)
        _lib.check(_lib.lib().sbs_gpu_read_body(sim.h, b, None, None))
