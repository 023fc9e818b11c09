"""The barriers and waits that the passes write themselves (fft_dev.hpp), as the compiler is told of them: each inline
asm must stand between two fences in the forward passes' code. Without them the asm is marked noalias for the LDS
arrays that the z forward pass takes through __restrict__ pointers, and their reads and writes, which other
work-items' accesses depend on, could be moved across it."""
import os
import re
import subprocess

import pytest

from laps_amd import build

pytestmark = pytest.mark.skipif(not os.path.exists(build._hipcc()), reason="needs hipcc")


def test_hand_written_barriers_are_fenced(tmp_path):
    out = tmp_path / "fwd.ll"
    flags = [f for f in build.FLAGS if f != "-Wall"]
    subprocess.run([build._hipcc(), *flags, "-w", "--cuda-device-only", "-S", "-emit-llvm", "-o", str(out),
                    os.path.join(build.SRC, "fwd_fused.hip")], check=True, timeout=300)
    lines = [s.strip() for s in out.read_text().splitlines()]
    at = [i for i, s in enumerate(lines) if re.search(r'asm sideeffect "s_waitcnt', s)]
    assert len(at) > 100
    for i in at:
        assert lines[i - 1].startswith("fence ") and lines[i + 1].startswith("fence "), lines[i - 1:i + 2]
