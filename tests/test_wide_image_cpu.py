"""Images past the reach of the forward projector's 32-bit gathers (wide_image,
internal.h), for every side and slice batch: where it says an image is within
reach, the byte offset of every index a segment can have, up to N^2 + N for a
segment on the far grid lines, is its true value (no wrap at 2^32), and those
past the image lie outside the buffer resource, which reads 0 there."""
import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = """
#include <hip/hip_runtime.h>
#include "internal.h"
extern "C" int wide(int N, int sb) { return trace_hip::wide_image(N, sb) ? 1 : 0; }
"""


@pytest.fixture(scope="module")
def wide(tmp_path_factory):
    from trace_amd import build
    d = tmp_path_factory.mktemp("wide")
    src, lib = d / "wide.hip", d / "libwide.so"
    src.write_text(SOURCE)
    subprocess.run([build.hipcc(), *build.flags(), "-O1", "--offload-host-only", "-shared",
                    "-I", build.CSRC, str(src), "-o", str(lib)], check=True,
                   stderr=subprocess.DEVNULL)
    return ctypes.CDLL(str(lib)).wide


@pytest.mark.parametrize("sb", [1, 2, 4, 8, 16, 32])
def test_offsets_within_reach(wide, sb):
    narrow = 0
    for N in range(2, 32769):
        if wide(N, sb):
            continue
        narrow = N
        resource = N * N * sb * 4  # bytes
        assert resource < 2 ** 32, N
        for ix in (0, 1, N - 1, N):  # iy = N
            off = (N * N + ix) * sb * 4
            for byte in (off, off + sb * 4 - 1):
                assert resource <= byte % 2 ** 32 == byte, (N, ix)
    # the sides within reach are the small ones, and nearly all that fit 2^32
    assert wide(narrow + 1, sb) or narrow == 32768
    assert (narrow + 2) ** 2 * sb * 4 >= 2 ** 32 or narrow == 32768
