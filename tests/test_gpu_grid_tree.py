"""GPU checks of the mesh-distance scan and tree walk at their edges: triangle counts around the tree's arity and one
level more, nodes equally far from many triangles (the ball's center), ties between equally near triangles,
repeated and degenerate triangles, coordinates whose squares leave the FP32 range of the walk's tests; node
values equal the oracle's."""
import numpy as np
import pytest

import oracle as O
import sbs_amd as S
from test_oracle_grid import icosphere

pytestmark = pytest.mark.gpu


def _strip(n):
    """n triangles of a flat strip: nodes above its edges are equally near to two of them."""
    v = np.array([[i // 2, i % 2, 0.0] for i in range(n + 2)], dtype=np.float64)
    return v, np.array([[i, i + 1, i + 2] if i % 2 == 0 else [i + 1, i, i + 2] for i in range(n)], dtype=np.uint32)


def _ball():
    return icosphere(0.5, 4)


def _messy():
    V, F = icosphere(0.5, 2)
    return V, np.concatenate([F, F[:7], F[:3][:, [1, 2, 0]], [[0, 0, 1], [5, 5, 5]]]).astype(np.uint32)


@pytest.mark.parametrize("mesh", [f"strip_{n}" for n in (1, 3, 4, 5, 16, 17, 65)] + ["ball", "messy"])
def test_node_values_at_the_trees_edges(mesh):
    V, F = _strip(int(mesh[6:])) if mesh.startswith("strip") else (_ball() if mesh == "ball" else _messy())
    # the ball's box is symmetric: the middle node is its center
    lo, hi = V.min(0) - 0.25, V.max(0) + 0.25
    res = [4, 4, 4] if mesh == "ball" else [5, 3, 2]
    print(f"[gpu-case] grid tree {mesh}: {len(F)} triangles", flush=True)
    assert np.array_equal(S.grid_from_mesh(V, F, lo, hi, res), O.grid_from_mesh(V, F, lo, hi, res))


@pytest.mark.parametrize("triangles", [511, 512, 513, 1024, 1025, 4096, 4097])
def test_node_values_where_the_tree_begins(triangles):
    """Up to 512 triangles are scanned, more walked; trees of one node more and fewer on a level."""
    V, F = _strip(triangles)
    lo, hi = V.min(0) - 0.25, V.max(0) + 0.25
    print(f"[gpu-case] grid of {triangles} triangles", flush=True)
    assert np.array_equal(S.grid_from_mesh(V, F, lo, hi, [31, 3, 2]), O.grid_from_mesh(V, F, lo, hi, [31, 3, 2]))


@pytest.mark.parametrize("mesh", ["strip_1", "strip_7", "strip_9", "messy", "fan"])
@pytest.mark.parametrize("res", [(1, 1, 1), (25, 25, 25), (26, 26, 26)])
def test_scanned_meshes_with_eight_lanes_a_node_and_one(mesh, res):
    """Grids of up to 131,072 nodes (25^3 cells have 118,976, 26^3 133,407) take eight lanes a node."""
    if mesh == "fan":
        a = 2 * np.pi * np.arange(150) / 150
        V = np.concatenate([[[0.0, 0.0, 1.0], [0.0, 0.0, -1.0]], np.stack([np.cos(a), np.sin(a), 0 * a], 1)])
        i, j = 2 + np.arange(150), 2 + (np.arange(150) + 1) % 150
        F = np.concatenate([np.stack([0 * i, i, j], 1), np.stack([0 * i + 1, j, i], 1)]).astype(np.uint32)
    else:
        V, F = _messy() if mesh == "messy" else _strip(int(mesh[6:]))
    lo, hi = V.min(0) - 0.25, V.max(0) + 0.25
    print(f"[gpu-case] scanned grid {mesh} {res}", flush=True)
    assert np.array_equal(S.grid_from_mesh(V, F, lo, hi, list(res)), O.grid_from_mesh(V, F, lo, hi, list(res)))


@pytest.mark.parametrize("exponent", [-45, -40, -30, *range(-23, -15), 15, 18, 19, 20, 37, 38, 39, 60])
@pytest.mark.parametrize("shift", [0.0, 0.25])
@pytest.mark.parametrize("levels", [2, 3])
def test_node_values_at_any_scale(exponent, shift, levels):
    V, F = icosphere(0.5, levels)
    scale = 10.0 ** exponent
    V, lo, hi = (V + shift) * scale, (V.min(0) - 0.25) * scale, (V.max(0) + 0.25) * scale
    print(f"[gpu-case] grid tree at scale 1e{exponent}", flush=True)
    got, want = S.grid_from_mesh(V, F, lo, hi, [5, 4, 3]), O.grid_from_mesh(V, F, lo, hi, [5, 4, 3])
    assert np.array_equal(got, want), (int(np.sum(got != want)), float(np.abs(got - want).max() / scale))


@pytest.mark.parametrize("height", [0.0, 1e-19, 1e-20])
def test_nodes_just_above_a_plate(height):
    """Nodes above a plate at its center's height: the nearest triangle's centroid is that near to some of them."""
    n = 24
    i, j = np.meshgrid(np.arange(n + 1), np.arange(n + 1), indexing="ij")
    V = np.stack([i.ravel() - n / 2, j.ravel() - n / 2, np.zeros((n + 1) ** 2)], 1).astype(np.float64)
    a = (np.arange(n)[:, None] * (n + 1) + np.arange(n)[None, :]).ravel()
    F = np.concatenate([np.stack([a, a + n + 1, a + 1], 1), np.stack([a + n + 1, a + n + 2, a + 1], 1)]).astype(np.uint32)
    # the grid's nodes at thirds of the cells of the plate are its triangles' centroids
    lo, hi = np.array([-n / 2, -n / 2, height]), np.array([n / 2, n / 2, 1.0])
    res = [n // 2, n // 2, 2]
    print(f"[gpu-case] grid tree {height} above a plate", flush=True)
    assert np.array_equal(S.grid_from_mesh(V, F, lo, hi, res), O.grid_from_mesh(V, F, lo, hi, res))


def test_more_tree_nodes_than_waves():
    """A plate of 16.8M triangles, whose lowest tree level has more nodes than the launch that makes it has waves."""
    n = 2900
    assert 2 * n * n / 4 > 4 << 20
    i, j = np.meshgrid(np.arange(n + 1), np.arange(n + 1), indexing="ij")
    V = np.stack([i.ravel(), j.ravel(), np.zeros((n + 1) ** 2)], 1).astype(np.float64)
    a = (np.arange(n)[:, None] * (n + 1) + np.arange(n)[None, :]).ravel()
    F = np.concatenate([np.stack([a, a + n + 1, a + 1], 1), np.stack([a + n + 1, a + n + 2, a + 1], 1)]).astype(np.uint32)
    lo, hi, res = np.array([1.3, 2.1, -40.0]), np.array([n - 2.7, n - 1.9, 50.0]), [17, 19, 2]
    print(f"[gpu-case] grid tree of {len(F)} triangles", flush=True)
    got = S.grid_from_mesh(V, F, lo, hi, res)
    z = S.grid_node_positions(lo, hi, res)[:, 2]
    # the nearest point lies straight below or above: coordinates of up to 2,900 round to 5e-13
    assert np.allclose(got, z, rtol=0.0, atol=1e-10)
