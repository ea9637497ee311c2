"""The frontier kernels' words and index arithmetic (CPU, compiled from their headers), and their
wide form, which volumes beyond 32-bit byte offsets take, against the narrow one (GPU)."""
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc (host compile only)")
def test_words_slots_and_divisions(tmp_path):
    exe = tmp_path / "word_check"
    src = os.path.join(HERE, "indexing", "word_check.cpp")
    subprocess.run(["hipcc", "-x", "hip", "--offload-arch=gfx950", "-O1", "-std=c++17", src, "-o", str(exe)],
                   check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr


@pytest.mark.gpu
@pytest.mark.parametrize("fix_branching", [True, False])
def test_wide_volume_equals_its_content_alone(fix_branching):
    """Content in the far corner of a 9000 x 9000 x 5 volume (its words lie beyond 4 GiB) gives the
    skeletons it gives alone, moved: the flat order of its voxels is the same, and without border
    targets nothing else depends on the place (tube coordinates below 2^24: exact as floats)."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import brook_amd
    from brook_amd import synth
    small = synth.volume("tubes", (90, 70, 5), 4, 17).astype(np.uint8)
    small[0], small[-1], small[:, 0], small[:, -1] = 0, 0, 0, 0
    shape, at = (9000, 9000, 5), (9000 - 90, 9000 - 70, 0)
    big = torch.zeros(shape[::-1], dtype=torch.uint8, device="cuda")
    big[at[2]:, at[1]:, at[0]:] = torch.from_numpy(np.ascontiguousarray(small.transpose(2, 1, 0))).cuda()
    options = dict(teasar_params=dict(scale=1.5, const=20, pdrf_scale=100000, pdrf_exponent=4), anisotropy=(1, 1, 1),
                   dust_threshold=50, fix_borders=False, fix_branching=fix_branching, output="packed", progress=False)
    want = brook_amd.skeletonize(small, **options).as_dict()
    got = brook_amd.skeletonize(big.permute(2, 1, 0), **options).as_dict()
    assert len(want["labels"]) > 0
    assert np.array_equal(got["vertices"] - np.asarray(at, np.float32), want["vertices"])
    for name in ("labels", "v_off", "e_off", "edges", "radii"):
        assert np.array_equal(got[name], want[name]), name
