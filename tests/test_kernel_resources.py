"""The crossing kernels keep their values in registers: a kernel that spills many of them takes
scratch memory for every lane of the device on its first launch, and time for each access.
(Compiles lvn_kernels.hip for gfx950 with the library's flags; runs without a GPU.)"""
import os
import re
import subprocess

from leven_amd import build


def test_crossing_kernels_do_not_spill(tmp_path):
    src = os.path.join(build.CSRC, "lvn_kernels.hip")
    out = subprocess.run([build.HIPCC] + build.FLAGS + ["--cuda-device-only", "-Rpass-analysis=kernel-resource-usage", "-c",
                                                        src, "-o", str(tmp_path / "k.o")], capture_output=True, text=True)
    assert out.returncode == 0, out.stderr[-2000:]
    scratch, name = {}, None
    for line in out.stderr.splitlines():
        m = re.search(r"Function Name: (\S+)", line)
        if m:
            name = m.group(1)
        m = re.search(r"ScratchSize \[bytes/lane\]: (\d+)", line)
        if m:
            scratch[name] = int(m.group(1))
    crossing = {k: v for k, v in scratch.items() if "k_edge_cross" in k}
    assert len(crossing) >= 12
    # a few bytes (one or two values of the work-counting and 16-lane forms) are the compiler's
    assert all(v <= 64 for v in crossing.values()), {k: v for k, v in crossing.items() if v > 64}
