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
extern "C" int whole(uint64_t x, uint32_t in_f, int m, int64_t ldx) { return ixh::ln_whole_pieces(x, in_f, m, ldx); }
extern "C" uint32_t column(uint32_t col, uint32_t in_f) { return ixh::ln_piece_column(col, in_f); }
"""


@pytest.fixture(scope="module")
def bounds(tmp_path_factory):
    d = tmp_path_factory.mktemp("bounds")
    (d / "bounds.cpp").write_text(SOURCE)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-I", CSRC, str(d / "bounds.cpp"),
                           "-o", str(d / "bounds.so")])
    lib = C.CDLL(str(d / "bounds.so"))
    lib.whole.argtypes = [C.c_uint64, C.c_uint32, C.c_int, C.c_int64]
    return lib


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


@pytest.mark.parametrize("in_f", list(range(1, 34)) + [511, 512, 513, 1024, 1031])
def test_requests_of_the_activations_stay_in_their_row(bounds, in_f):
    """Rows shorter than a piece are read element by element; of others each request is a whole piece of the row, its own
    one where the row has that."""
    assert bool(bounds.whole(0x1000, in_f, 1, in_f)) == (in_f >= 8)
    assert not bounds.whole(0x1002, in_f, 1, in_f)
    assert bool(bounds.whole(0x1000, in_f, 2, in_f)) == (in_f >= 8 and in_f % 8 == 0)
    if in_f >= 8:
        for col in range(0, -(-in_f // 512) * 512, 8):
            at = bounds.column(col, in_f)
            assert at % 8 == 0 and at + 8 <= in_f and (at == col or col + 8 > in_f)
