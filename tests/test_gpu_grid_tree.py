"""GPU checks of the mesh-distance tree walk at its edges: triangle counts around the tree's arity and one
level more, nodes equally far from many triangles (the ball's center, finished by a workgroup each), ties
between equally near triangles, repeated and degenerate triangles; node values equal the oracle's."""
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
