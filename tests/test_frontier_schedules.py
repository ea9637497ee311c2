"""The label workgroups' kernels run on the CPU (tests/emulation) under schedules that let one wave run
ahead of the others between two barriers: all waves have to meet at the same barriers, and the
fields, paths and claims have to be those of a workgroup of one wave, for several workgroup sizes and numbers
of words in flight."""
import os
import platform
import shutil
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "brook_amd", "csrc")
EMULATION = os.path.join(HERE, "emulation")


def device_part(source, end, path):
    """The kernels of `source` (its host part begins at `end`), in a namespace of their own."""
    with open(os.path.join(CSRC, source)) as f:
        text = f.read()
    begin = "namespace brook {\nnamespace {"
    body = text[text.index(begin) + len("namespace brook {\n"):text.index(end)]
    with open(path, "w") as f:
        f.write("namespace brook {\nusing namespace ::brook;\n" + body + "}\n}\n")


@pytest.mark.skipif(shutil.which("g++") is None or platform.machine() != "x86_64", reason="needs g++ on x86-64")
def test_every_schedule_gives_the_same(tmp_path):
    device_part("fields.hip", "unsigned grid_for(", tmp_path / "flood_device.inc")
    device_part("trace.hip", "}  // namespace\n\nvoid trace_all", tmp_path / "trace_device.inc")

    def run(shape):
        block, batch = shape
        exe = tmp_path / f"check_{block}_{batch}"
        subprocess.run(["g++", "-std=c++17", "-O1", "-w", f"-DBROOK_TRACE_BLOCK={block}", f"-DBROOK_FLOOD_BLOCK={block}",
                        f"-DBROOK_NB_BATCH={batch}", f"-DBROOK_FLOOD_NB_BATCH={batch}", "-I" + EMULATION, "-I" + CSRC,
                        "-I" + str(tmp_path), os.path.join(EMULATION, "frontier_check.cpp"), "-o", str(exe)], check=True)
        r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, (shape, r.stdout)
        return r.stdout

    with ThreadPoolExecutor() as pool:
        alone, *others = pool.map(run, [(64, 9), (256, 9), (128, 13), (256, 26)])
    assert alone.count("\n") == 9
    for out in others:
        assert out == alone
