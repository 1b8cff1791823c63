"""GPU checks of the boundary extraction on meshes where faces meet in other numbers than two: the same
surface as the host extraction, index by index."""
import ctypes

import numpy as np
import pytest

import sbs_amd as S

pytestmark = pytest.mark.gpu


def _random(nv, nt, seed, repeats=False):
    rng = np.random.default_rng(seed)
    if repeats:  # degenerate tets too
        return nv, rng.integers(0, nv, (nt, 4))
    return nv, np.argsort(rng.random((nt, nv)), axis=1)[:, :4] if nv <= 64 else rng.permuted(
        np.tile(np.arange(nv), (nt, 1)), axis=1)[:, :4]


CASES = {
    "one_tet": lambda: (4, np.array([[3, 1, 0, 2]])),
    # 8 tets have 32 faces, one word of bits; 9 one tet more
    "eight_apart": lambda: (32, np.arange(32).reshape(8, 4)),
    "nine_apart": lambda: (36, np.arange(36).reshape(9, 4)),
    "same_tet_twice": lambda: (5, np.array([[0, 1, 2, 3], [0, 1, 2, 3]])),
    "same_tet_1000_times": lambda: (4, np.tile([[2, 0, 3, 1]], (1000, 1))),
    "fan_around_an_edge": lambda: (302, np.stack([np.zeros(300), np.ones(300), 2 + np.arange(300),
                                                  2 + (np.arange(300) + 1) % 300], 1)),
    "star_around_a_vertex": lambda: (3001, np.concatenate([np.zeros((1000, 1)), 1 + np.arange(3000).reshape(1000, 3)], 1)),
    # every face many times
    "few_vertices": lambda: _random(7, 5000, 1),
    "some_vertices": lambda: _random(40, 9001, 2),
    "degenerate": lambda: _random(30, 4000, 3, repeats=True),
    "unused_vertices": lambda: (2 ** 21, 2 ** 21 - 1 - np.arange(40).reshape(10, 4)),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_faces_that_meet_in_any_number(name):
    nv, tets = CASES[name]()
    tets = np.ascontiguousarray(tets, dtype=np.uint32)
    print(f"[gpu-case] boundary {name}: {len(tets)} tets", flush=True)
    for got, want in zip(S.extract_boundary(nv, tets), S.boundary(nv, tets)):
        assert got.shape == want.shape and np.array_equal(got, want)


def test_an_index_out_of_range_is_refused():
    tets = np.arange(400, dtype=np.uint32).reshape(100, 4)
    with pytest.raises(S.SbsError, match="out of range"):
        S.extract_boundary(399, tets)


def test_a_refused_call_leaves_its_outputs_alone():
    tets = np.array([0, 1, 2, 3, 1, 2, 3, 9], dtype=np.uint32)
    ns, nt = ctypes.c_uint32(77), ctypes.c_uint32(78)
    code = S.lib().sbs_gpu_extract_boundary(0, 9, tets.ctypes.data_as(ctypes.POINTER(ctypes.c_uint32)), 2, None, None,
                                            ctypes.byref(ns), ctypes.byref(nt))
    assert code == 1 and (ns.value, nt.value) == (77, 78)
