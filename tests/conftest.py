import ctypes as C
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)
CSRC = os.path.join(ROOT, "ixrun_amd", "csrc")
BOUNDS = """
#include "ixh_lanes_bounds.h"
#include <vector>
extern "C" void groups(uint32_t first, uint32_t end, uint32_t n, uint32_t *out) {
    const ixh::LnGroups g = ixh::ln_groups(first, end, n);
    out[0] = g.first; out[1] = g.last; out[2] = g.n;
}
extern "C" uint32_t four_quads(uint32_t from, uint32_t lane, uint32_t end) { return ixh::ln_four_quads(from, lane, end); }
extern "C" int whole(uint64_t x, uint32_t in_f, int m, int64_t ldx) { return ixh::ln_whole_pieces(x, in_f, m, ldx); }
extern "C" uint32_t column(uint32_t col, uint32_t in_f) { return ixh::ln_piece_column(col, in_f); }
extern "C" uint32_t share(uint32_t n, uint32_t wave, uint32_t log_waves) { return ixh::ln_share(n, wave, log_waves); }
extern "C" uint32_t listed_at(uint32_t pos, uint32_t value, int in_range, uint32_t seg, uint32_t cells) {
    return ixh::ln_listed_at(pos, value, in_range, seg, cells);
}
extern "C" uint32_t begin(uint32_t g, uint32_t groups, uint32_t tiles, uint32_t cells) { return ixh::lp_begin(g, groups, tiles, cells); }
extern "C" uint32_t group_of(uint32_t c, uint32_t groups, uint32_t tiles, uint32_t cells) { return ixh::lp_group_of(c, groups, tiles, cells); }
extern "C" uint32_t part(uint32_t g, uint32_t tile, int begins, uint32_t groups, uint32_t tiles) { return ixh::lp_part(g, tile, begins, groups, tiles); }
extern "C" uint32_t parts(uint32_t groups, uint32_t tiles) { return ixh::lp_parts(groups, tiles); }

extern "C" uint32_t first(uint32_t i, uint32_t n, uint32_t k) {
    const ixh::LgSplit p(n, k);
    return ixh::lg_first(i, p.share, p.more);
}
// blocks of k_lanes_gemm that are not in work exactly once
extern "C" uint32_t uncovered(uint32_t blocks, uint32_t groups) {
    const ixh::LgSplit split(blocks, groups);
    const uint32_t most_at_once = ixh::lg_most_at_once(blocks, groups);
    std::vector<int> times(blocks);
    for (uint32_t g = 0; g < groups; ++g) {
        const uint32_t b0 = ixh::lg_first(g, split.share, split.more), b1 = ixh::lg_first(g + 1, split.share, split.more);
        const uint32_t at_once = ixh::lg_at_once(b1 - b0, most_at_once);
        if (at_once > ixh::kLgBlocks) return blocks;
        for (uint32_t round = 0; round < ixh::lg_rounds(b1 - b0); ++round)
            for (uint32_t wave = 0; wave < at_once; ++wave)
                if (const uint32_t b = b0 + round * at_once + wave; b < b1) ++times[b];
    }
    return blocks - (uint32_t)std::count(times.begin(), times.end(), 1);
}
extern "C" void plan(uint32_t out_f, uint32_t cells, int m, uint32_t cus, uint32_t *out) {
    const ixh::LgPlan p = ixh::lg_plan((out_f + 3) / 4, cells, m, cus);
    out[0] = p.m_groups; out[1] = p.mb; out[2] = p.slices; out[3] = p.groups;
}
"""


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (run with -m gpu on the GPU box)")


@pytest.fixture(scope="session")
def oracle():
    from oracle import ix_oracle

    ix_oracle.build()
    return ix_oracle


@pytest.fixture
def force_decoder():
    """Force one of the library's decoders for the duration of a test (``ixh_set_option``), then give the choice
    back to the library."""
    from ixrun_amd import _lib

    def force(name: str) -> None:
        _lib.set_option("decode_kernel", name)

    yield force
    _lib.set_option("decode_kernel", "auto")


@pytest.fixture
def gemv_option():
    """Set a kernel-selection switch of ixh_gemv or ixh_gemm for the duration of a test (``ixh_set_option``)."""
    from ixrun_amd import _lib

    defaults = {"gemv_strips": 0, "gemv_shared_x": 8, "gemv_tiles": 0, "gemv_tile_rows": 0, "gemv_tile_cus": 0, "gemv_tile_split": 0, "gemv_dense_tiles": 0, "gemv_slots": 0, "gemv_slot_waves": 0, "gemm_tiles": 0}
    touched = []

    def set_(name: str, value: int) -> None:
        touched.append(name)
        _lib.set_option(name, value)

    yield set_
    for name in touched:
        _lib.set_option(name, defaults[name])


@pytest.fixture(scope="session")
def bounds(tmp_path_factory):
    """``csrc/ixh_lanes_bounds.h``, which is plain C++, compiled for the host."""
    d = tmp_path_factory.mktemp("bounds")
    (d / "bounds.cpp").write_text(BOUNDS)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-I", CSRC, str(d / "bounds.cpp"),
                           "-o", str(d / "bounds.so")])
    lib = C.CDLL(str(d / "bounds.so"))
    lib.whole.argtypes = [C.c_uint64, C.c_uint32, C.c_int, C.c_int64]
    return lib
