"""Tuning builds outside what the kernels' loops assume do not compile."""
import os
import subprocess

import pytest

from bitsparse_amd.build import CSRC, INCLUDE, hipcc


# the rounds of a store pass are ranked in pairs, and whole passes make up a tile's eight rounds
@pytest.mark.parametrize("rounds", [1, 2, 3, 4, 6])
def test_stream_rounds(rounds):
    r = subprocess.run([hipcc(), "--offload-arch=gfx950", "--cuda-host-only", "-fsyntax-only", "-std=c++17", "-I", INCLUDE,
                        "-I", CSRC, f"-DBS_STREAM_ROUNDS={rounds}", os.path.join(CSRC, "codec.hip")],
                       capture_output=True, text=True)
    assert (r.returncode == 0) == (rounds in (2, 4)), r.stderr
