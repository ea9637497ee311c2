"""The device postprocess where its forms meet, against the oracle: components around the size whose
state fits LDS (loops about 2 700 vertices, trees about 5 300), repeated rows, join cells that fit
one 64-bit key and cells that do not (a millionth wide, where a label's radii are 0), waves of few and of many."""
import numpy as np
import pytest

import oracle

from .test_post import as_packed, gpu_same, packed


@pytest.fixture(scope="module")
def post():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import brook_amd
    return brook_amd.device_post


def _tree(rng, n, branch):
    """n vertices: mostly a chain, each new vertex off a random earlier one with probability branch."""
    parent = np.arange(n) - 1
    jump = np.flatnonzero(rng.random(n) < branch)
    jump = jump[jump > 1]
    parent[jump] = (rng.random(len(jump)) * jump).astype(int)
    verts = np.zeros((n, 3), np.float32)
    step = rng.integers(-1, 2, (n, 3))
    step[(step == 0).all(1), 0] = 1
    for i in range(1, n):
        verts[i] = verts[parent[i]] + step[i]
    edges = [(int(parent[i]), i) for i in range(1, n)]
    return verts + rng.uniform(0, 0.01, (n, 3)).astype(np.float32), edges


def _cyclic(seed, n, chords, repeats=0):
    rng = np.random.default_rng(seed)
    verts, edges = _tree(rng, n, 0.01)
    for _ in range(chords):
        a, b = sorted(rng.choice(n, 2, replace=False).tolist())
        if (a, b) not in edges:
            edges.append((a, b))
    for _ in range(repeats):
        edges.append(edges[int(rng.integers(0, len(edges)))])
    return packed((3, verts, edges, rng.uniform(0.5, 4, n).astype(np.float32)))


@pytest.mark.gpu
@pytest.mark.parametrize("n,chords,repeats", [(63, 2, 0), (65, 3, 2), (900, 4, 3), (2600, 3, 0), (2790, 3, 2), (3100, 3, 1)])
def test_loops_of_components_by_size(post, n, chords, repeats):
    p = _cyclic(n, n, chords, repeats)
    gpu_same(post.remove_loops(as_packed(p)), oracle.post("remove_loops", p, 0, 0), n)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [40, 1000, 5000, 5500, 7000])
def test_ticks_of_trees_by_size(post, n):
    verts, edges = _tree(np.random.default_rng(n), n, 0.02)
    p = packed((2, verts, edges, 1.0))
    gpu_same(post.remove_ticks(as_packed(p), 9.0), oracle.post("remove_ticks", p, 9.0, 0), n)


@pytest.mark.gpu
@pytest.mark.parametrize("radius,spread", [(2.0, 40.0), (8.0, 40.0), (30.0, 40.0), (0.0, 40.0), (1.5, 3e7), (0.0, 3e7)])
def test_joins_in_packed_and_wide_cells(post, radius, spread):
    """Short chains of two labels; some ends meet a chain of the other end of the volume exactly. Their
    vertices lie in a few cells (radius 30) up to one each."""
    rng = np.random.default_rng(int(spread) + int(radius * 10))
    parts = []
    for label in (1, 2):
        verts, edges = [], []
        for c in range(30):
            at = rng.uniform(-spread, spread, 3)
            if c % 5 == 4:
                at = verts[int(rng.integers(0, len(verts)))]  # coincident with an earlier chain's vertex
            base = len(verts)
            for k in range(4):
                verts.append(np.asarray(at, np.float32) + np.float32([k, 0, 0]))
            edges += [(base + k, base + k + 1) for k in range(3)]
        parts.append((label, np.asarray(verts, np.float32), edges, radius))
    p = packed(*parts)
    gpu_same(post.join_close_components(as_packed(p)), oracle.post("join_components", p, 0, 0), (radius, spread))
