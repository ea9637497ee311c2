"""The target order's pairs at the edges of their tiles: volumes of 64, 1024 and 4096 voxels, one less and
one more, and foreground that starts or ends a stretch of 64; skeletons equal the oracle's."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(7, 9, 1), (8, 8, 1), (13, 5, 1), (31, 33, 1), (16, 8, 8), (41, 5, 5), (21, 65, 3), (16, 16, 16), (17, 241, 1),
                                   (64, 65, 2)])
@pytest.mark.parametrize("empty", [0.0, 0.2])
def test_order_at_tile_edges(shape, empty):
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import brook_amd
    rng = np.random.default_rng(sum(shape))
    vol = np.asfortranarray((rng.random(shape) >= empty).astype(np.uint8))
    vol[shape[0] // 2:] *= 2  # two labels
    options = dict(teasar_params=dict(scale=1.0, const=2, pdrf_scale=100000, pdrf_exponent=4), anisotropy=(1, 2, 3), dust_threshold=2)
    got = brook_amd.skeletonize(vol, output="packed", progress=False, **options).as_dict()
    want = oracle.skeletonize(vol, **options)
    for name in ("labels", "vertices", "edges", "radii"):
        assert np.array_equal(np.asarray(got[name]).ravel(), np.asarray(want[name]).ravel()), name
