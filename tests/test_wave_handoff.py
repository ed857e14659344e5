"""Values that lanes of one wave pass through LDS go through wave_handoff()
(nexus_amd/csrc/nx_device.hpp): the wave barrier with a memory fence on each side.
The barrier builtin alone lets the compiler move an LDS load above another
lane's store that it proves apart within one lane (CPU only: reads the sources).
"""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nexus_amd", "csrc")


def test_no_bare_wave_barrier():
    seen = 0
    for path in sorted(glob.glob(os.path.join(CSRC, "*.h*"))):
        lines = [line.strip() for line in open(path)]
        for i, line in enumerate(lines):
            if "__builtin_amdgcn_wave_barrier" not in line:
                continue
            seen += 1
            for near in (lines[i - 1], lines[i + 1]):
                assert re.match(r'__builtin_amdgcn_fence\(__ATOMIC_\w+, "wavefront"\);', near), f"{path}:{i + 1}"
    assert seen > 0
