"""The component unions' left-out contacts against the oracle on random volumes (every density, rows
and planes of one voxel, the remainders of a wave, more than one stretch per wave), and hole filling
over more than one group of boxes against the volume filled beforehand."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


@pytest.mark.parametrize("shape", [(1, 1, 1), (1, 9, 7), (9, 1, 7), (9, 7, 1), (63, 5, 6), (64, 4, 9), (65, 7, 5), (33, 31, 29),
                                   (130, 20, 17), (101, 103, 107)])
@pytest.mark.parametrize("labels,density", [(1, 0.08), (1, 0.3), (2, 0.55), (3, 0.9), (2, 1.0)])
def test_components_of_random_volumes(torch, shape, labels, density):
    from brook_amd import device
    rng = np.random.default_rng(shape[0] * 100 + shape[1] * 10 + shape[2] + labels)
    vol = np.asfortranarray((rng.integers(1, labels + 1, shape) * (rng.random(shape) < density)).astype(np.uint16))
    vol[0, 0, 0] = 1
    ids, mapping, roots = device.connected_components(vol)
    cc, m, r = oracle.ccl(vol)
    assert np.array_equal(ids.cpu().numpy().astype(np.uint32), cc)
    assert np.array_equal(mapping, m) and np.array_equal(roots, r)


def test_holes_of_more_boxes_than_a_group(torch):
    """Four labels whose boxes are about the whole volume, so that each is a group of its own: a line
    each, with a hollow 3 x 3 x 3 cube on it. The result is that of the volume with the hollows painted."""
    import brook_amd
    n = 150
    i = np.arange(n)
    vol = np.zeros((n, n, n), np.uint8, order="F")
    filled = []
    for k in range(4):
        vol[i, np.clip(i + 6 * k, 0, n - 1), i] = k + 1
        vol[i, 6 * k, 0] = np.where(vol[i, 6 * k, 0], vol[i, 6 * k, 0], k + 1)  # to the far x at z = 0
        c = 30 + 22 * k
        at = (c, min(c + 6 * k, n - 1), c)
        vol[at[0] - 1:at[0] + 2, at[1] - 1:at[1] + 2, at[2] - 1:at[2] + 2] = k + 1
        vol[at] = 0
        filled.append((at, k + 1))
    whole = vol.copy(order="F")
    for at, label in filled:
        whole[at] = label
    options = dict(teasar_params=dict(scale=1.5, const=4, pdrf_scale=100000, pdrf_exponent=4), anisotropy=(1, 1, 1),
                   dust_threshold=50, output="packed", progress=False)
    got = brook_amd.skeletonize(vol, fill_holes=True, **options).as_dict()
    want = brook_amd.skeletonize(whole, **options).as_dict()
    plain = brook_amd.skeletonize(vol, **options).as_dict()
    assert len(want["labels"]) == 4 and not np.array_equal(plain["radii"], want["radii"])  # the hollows matter
    for name in want:
        assert np.array_equal(got[name], want[name]), name
