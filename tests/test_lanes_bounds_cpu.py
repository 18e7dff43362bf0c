"""What the lane kernels ask for ahead of need stays inside their buffers: the ranges of ``csrc/ixh_lanes_bounds.h`` walked
on the host (the header is plain C++)."""
import ctypes as C
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ixrun_amd", "csrc")
SOURCE = """
#include "ixh_lanes_bounds.h"
extern "C" void groups(uint32_t first, uint32_t end, uint32_t n, uint32_t *out) {
    const ixh::LnGroups g = ixh::ln_groups(first, end, n);
    out[0] = g.first; out[1] = g.last; out[2] = g.n;
}
"""


@pytest.fixture(scope="module")
def bounds(tmp_path_factory):
    d = tmp_path_factory.mktemp("bounds")
    (d / "bounds.cpp").write_text(SOURCE)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-I", CSRC, str(d / "bounds.cpp"),
                           "-o", str(d / "bounds.so")])
    return C.CDLL(str(d / "bounds.so"))


@pytest.mark.parametrize("total", [0, 1, 63, 64, 65, 127, 128, 129, 192])
def test_requests_of_the_list_stay_in_it(bounds, total):
    """Every share of a list of `total` quads (also an empty one at its end): no request goes to a group that the list does
    not have, and the groups that count are those of the share's quads."""
    groups, out = max(-(-total // 64), 1), (C.c_uint32 * 3)()
    for first in range(total + 1):
        for end in range(first, total + 1):
            bounds.groups(first, end, groups, out)
            g_first, last, n = out
            assert last < groups  # a request is for group min(first + i, last)
            if end > first:
                assert list(range(g_first, g_first + n)) == sorted({q // 64 for q in range(first, end)})
                assert last == g_first + n - 1
            else:
                assert n == 0
