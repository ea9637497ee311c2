"""The label workgroups' kernels run on the CPU (tests/emulation) under schedules that let one wave run
ahead of the others between two barriers: all waves have to meet at the same barriers, and the
fields, paths and claims have to be those of a workgroup of one wave, for several workgroup sizes and numbers
of words in flight, and where lists overflow LDS, far lists are compacted and stale notes overflow."""
import os
import platform
import shutil
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "brook_amd", "csrc")
EMULATION = os.path.join(HERE, "emulation")


# Limits that labels of this size never reach, set so that they do: the lists' room in LDS, the length at which
# far lists are compacted, the notes of stale offers.
TIGHT = {"fields.hip": {"kFloodFront = 4096, kFloodFar = 2048": "kFloodFront = 9, kFloodFar = 5", "end > count)": "end > 4)"},
         "trace.hip": {"kLdsFront = 3072, kLdsFar = 2048": "kLdsFront = 11, kLdsFar = 7", "end > to.count)": "end > 4)",
                       "l.stale, 2 * count, 0u": "l.stale, 2, 0u"}}


def device_part(source, end, path, changes):
    """The kernels of `source` (its host part begins at `end`), in a namespace of their own."""
    with open(os.path.join(CSRC, source)) as f:
        text = f.read()
    begin = "namespace brook {\nnamespace {"
    body = text[text.index(begin) + len("namespace brook {\n"):text.index(end)]
    for old, new in changes.items():
        assert body.count(old) == 1, old
        body = body.replace(old, new)
    with open(path, "w") as f:
        f.write("namespace brook {\nusing namespace ::brook;\n" + body + "}\n}\n")


@pytest.mark.skipif(shutil.which("g++") is None or platform.machine() != "x86_64", reason="needs g++ on x86-64")
def test_every_schedule_gives_the_same(tmp_path):
    def run(shape):
        block, batch, tight = shape
        parts = tmp_path / f"{block}_{batch}_{tight}"
        parts.mkdir()
        for source, end, part in [("fields.hip", "unsigned grid_for(", "flood_device.inc"),
                                  ("trace.hip", "}  // namespace\n\nvoid trace_all", "trace_device.inc")]:
            device_part(source, end, parts / part, TIGHT[source] if tight else {})
        exe = parts / "check"
        subprocess.run(["g++", "-std=c++17", "-O1", "-w", f"-DBROOK_TRACE_BLOCK={block}", f"-DBROOK_FLOOD_BLOCK={block}",
                        f"-DBROOK_NB_BATCH={batch}", f"-DBROOK_FLOOD_NB_BATCH={batch}", "-I" + EMULATION, "-I" + CSRC,
                        "-I" + str(parts), os.path.join(EMULATION, "frontier_check.cpp"), "-o", str(exe)], check=True)
        r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, (shape, r.stdout)
        return r.stdout

    with ThreadPoolExecutor() as pool:
        alone, *others = pool.map(run, [(64, 9, False), (256, 9, False), (128, 13, False), (256, 26, False),
                                            (128, 9, True)])
    assert alone.count("\n") == 9
    for out in others:
        assert out == alone
