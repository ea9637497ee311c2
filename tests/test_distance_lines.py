"""The distance transform's line kernel against the oracle, bit for bit: line lengths at the edges of
its words, seeds and groups, each number of lines per block (256 up to 27 positions) and the run lists beyond them, few and
many runs per line, lines without walls, and the per-label maxima through the skeleton's radii."""
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


def _volume(shape, kind, rng):
    if kind == "solid":
        return np.ones(shape, np.uint8)
    if kind == "noise":
        return (rng.random(shape) < 0.7).astype(np.uint16) * rng.integers(1, 4, shape).astype(np.uint16)
    vol = np.zeros(shape, np.uint32)  # long and short boxes
    for label in range(1, 30):
        lo = [rng.integers(0, s) for s in shape]
        hi = [min(s, a + 1 + rng.integers(0, max(1, s // 2 if label % 3 else 7))) for s, a in zip(shape, lo)]
        vol[lo[0]:hi[0], lo[1]:hi[1], lo[2]:hi[2]] = label
    return vol


@pytest.mark.parametrize("shape", [(5, 1, 1), (3, 2, 5), (31, 33, 3), (300, 27, 1), (257, 28, 2), (19, 27, 28), (17, 16, 15), (40, 63, 64), (33, 65, 66), (20, 96, 31), (7, 128, 129),
                                   (9, 534, 5), (6, 5, 545), (4, 1067, 3), (3, 4, 1100), (2, 3300, 2), (2, 2, 4300)])
@pytest.mark.parametrize("kind,aniso,border", [("solid", (1, 1, 1), True), ("solid", (3, 0.3, 7), False), ("noise", (4, 4, 40), False),
                                               ("boxes", (0.37, 1.1, 0.9), True), ("boxes", (16, 16, 40), False)])
def test_lines_equal_the_oracle(torch, shape, kind, aniso, border):
    from brook_amd import device
    vol = np.asfortranarray(_volume(shape, kind, np.random.default_rng(sum(shape))))
    got = device.edt(vol, aniso, border).cpu().numpy()
    want = oracle.edt(oracle.ccl(vol)[0], aniso, border)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("step", [1e18, 1e-18, 2e-20, 3e-21, 1e-22, 1e-23])
@pytest.mark.parametrize("border", [True, False])
def test_steps_at_the_ends_of_their_range(torch, step, border):
    """Steps whose squares are huge, subnormal or 0 in 32 bits: the same bits as the oracle's."""
    from brook_amd import device
    vol = np.asfortranarray((np.random.default_rng(3).random((9, 80, 70)) < 0.8).astype(np.uint8))
    aniso = (step, step, 1.5 * step)
    got = device.edt(vol, aniso, border).cpu().numpy()
    assert np.array_equal(got, oracle.edt(oracle.ccl(vol)[0], aniso, border))


@pytest.mark.parametrize("shape", [(40, 37, 70), (64, 65, 5)])
def test_label_maxima(torch, shape):
    """The transform's per-label maxima decide roots and scales: skeletons of blobs equal the oracle's."""
    import brook_amd
    rng = np.random.default_rng(7)
    vol = np.asfortranarray(_volume(shape, "boxes", rng).astype(np.uint16))
    options = dict(teasar_params=dict(scale=1.5, const=3, pdrf_scale=100000, pdrf_exponent=4), anisotropy=(1, 1, 1), dust_threshold=5)
    got = brook_amd.skeletonize(vol, output="packed", progress=False, **options).as_dict()
    want = oracle.skeletonize(vol, **options)
    for name in ("labels", "vertices", "edges", "radii"):
        assert np.array_equal(np.asarray(got[name]).ravel(), np.asarray(want[name]).ravel()), name
