"""What the lane kernels ask for ahead of need stays inside their buffers, and what the prompts' workgroups leave in memory has
places of its own: the ranges of ``csrc/ixh_lanes_bounds.h`` walked on the host (the header is plain C++)."""
import ctypes as C

import pytest


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


@pytest.mark.parametrize("total", [0, 1, 3, 4, 63, 64, 65, 130, 192])
def test_requests_of_a_cells_list_stay_in_the_list(bounds, total):
    """Any part of a list of `total` quads as one cell's (also an empty one at its end), 64 quads at a time: no request goes behind the
    list's last group, and each of the cell's quads is asked for by its own lanes."""
    fours = 16 * max(-(-total // 64), 1)
    for first in range(total + 1):
        for end in range(first, total + 1):
            asked, start = set(), first & ~3
            while start == first & ~3 or start < end:
                for lane in range(0, 64, 4):
                    at = bounds.four_quads(start, lane, end)
                    assert at < fours
                    quad = start + lane
                    asked |= {q for q in range(max(quad, first), min(quad + 4, end)) if q >> 2 == at}
                start += 64
            assert asked == set(range(first, end))


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


@pytest.mark.parametrize("cells", [64, 65, 67, 70, 127, 128, 129, 150])
def test_listed_elements_of_long_rows_are_gathered_from_their_row(bounds, cells):
    """A group of the list holds quads of several segments of a row, whose positions start over in each: those of the segment in
    work have their own activation, all others the zeros behind the row."""
    segments = -(-cells // 64)
    for seg in range(segments):
        for of in range(segments):
            end = min(65536, cells * 1024 - of * 65536)
            for pos in [*range(0, min(end, 64), 2), *range(1024, end, 1024), end - 2]:
                at = bounds.listed_at(pos, 90, of == seg, seg, cells)
                assert at == (seg * 65536 + pos if of == seg else cells * 1024) and at + 2 <= cells * 1024 + 64
        assert bounds.listed_at(0, 0, True, seg, cells) == cells * 1024


@pytest.mark.parametrize("log_waves", [0, 1, 2, 3, 4])
def test_shares_of_the_cells_follow_one_another(bounds, log_waves):
    """Each cell in one wave's run, in order, and no wave without one where all others have several."""
    waves = 1 << log_waves
    for n in list(range(1, 400)) + [5440, 65535, 5 << 20]:
        ends = [bounds.share(n, w, log_waves) for w in range(waves + 1)]
        assert ends[0] == 0 and ends[-1] == n and ends == sorted(ends)
        assert n < 32 * waves or 0.5 * n <= waves * min(b - a for a, b in zip(ends, ends[1:]))
        assert all(abs(b - a - n / waves) < 9 for a, b in zip(ends, ends[1:]))  # (a lead of some cells, however many there are)


@pytest.mark.parametrize("cells", [1, 2, 3, 5, 34])
def test_parts_of_shared_tiles_each_have_a_place(bounds, cells):
    """Every part of a tile that a workgroup leaves in memory has a place of its own, all places that are asked for are taken but
    those of runs that happen to begin or end with a tile, and the reader of a tile finds its parts in the order of the columns."""
    for tiles in (1, 2, 3, 7, 8, 40, 136):
        for groups in sorted({1, 2, 3, tiles, tiles + 1, 2 * tiles, 2 * tiles - 1, 3 * tiles - 2, 6 * tiles, tiles // 2, tiles // 3 + 1, 61} - {0}):
            if groups > tiles * cells:
                continue
            parts, written, at_an_edge = bounds.parts(groups, tiles), {}, 0
            of_tile = [[] for _ in range(tiles)]
            assert bounds.begin(0, groups, tiles, cells) == 0 and bounds.begin(groups, groups, tiles, cells) == tiles * cells
            for g in range(groups):
                u0, end = (bounds.begin(k, groups, tiles, cells) for k in (g, g + 1))
                assert end > u0
                at_an_edge += u0 % cells == 0
                u = u0
                while u < end:
                    tile, c0 = divmod(u, cells)
                    c1 = min(cells, c0 + end - u)
                    if c1 - c0 < cells:
                        part = bounds.part(g, tile, u == u0, groups, tiles)
                        assert part < parts and part not in written
                        written[part] = g
                        of_tile[tile].append(part)
                    u += c1 - c0
            assert parts <= 2 * groups and parts - len(written) <= 2 * at_an_edge
            for tile, own in enumerate(of_tile):
                g0, g1 = (bounds.group_of(tile * cells + c, groups, tiles, cells) for c in (0, cells - 1))
                begins = bounds.begin(g0, groups, tiles, cells) == tile * cells
                assert own == ([] if g0 == g1 else [bounds.part(g0, tile, begins, groups, tiles)] + list(range(g0 + 1, g1 + 1)))


@pytest.mark.parametrize("groups", [1, 2, 3, 7, 8, 19, 32, 51, 64, 85, 128, 256])
def test_blocks_of_a_workgroups_rounds_follow_one_another(bounds, groups):
    """Every block of weight rows in work once, whatever a workgroup has more or less than the others: shares of all sizes up to five rounds."""
    for blocks in [*range(groups, 5 * 16 * groups + groups, max(1, groups // 5)), *(k * groups + d for k in (16, 17, 32, 33, 48, 64) for d in (-1, 0, 1))]:
        if blocks >= groups:
            assert bounds.uncovered(blocks, groups) == 0, (blocks, groups)


def test_parts_of_a_whole_are_those_of_a_division(bounds):
    for n in [*range(1, 70), 136, 1088, 1089, 65535, 8388608]:
        for k in [k for k in (*range(1, 40), 61, 85, 127, 128, 253, 256, 1021, 65521, 65536) if k <= n]:
            for i in {0, 1, 2, k // 3, k // 2, k - 1, k}:
                assert bounds.first(i, n, k) == i * n // k, (i, n, k)


@pytest.mark.parametrize("cus", [256, 304, 64, 1])
def test_cuts_of_prompts_take_everything(bounds, cus):
    """Over the shapes and row counts that the kernel is given: slices and groups of at least a cell and a block, all activation rows in
    groups of at most 128, every block in work once."""
    out, seen = (C.c_uint32 * 4)(), set()
    for out_f in (1, 16, 17, 260, 512, 1536, 2752, 4100, 5120, 8208, 8256, 9808, 10240, 13120, 13616, 16400, 16512, 16640, 17408, 40000, 70000):
        for cells in (1, 2, 3, 5, 8, 10, 13, 16, 22, 34, 130):
            if out_f * cells * 512 > 9e7 and out_f <= 17408 and cells <= 34:
                continue
            for m in (1, 9, 16, 17, 25, 33, 64, 65, 100, 128, 129, 160, 512, 1024, 4096):
                bounds.plan(out_f, cells, m, cus, out)
                m_groups, mb, slices, groups = out
                blocks = -(-out_f // 16)
                assert 1 <= slices <= cells and 1 <= groups <= blocks and 1 <= mb <= 8 and m_groups * mb * 16 >= m
                if (blocks, groups) not in seen:
                    seen.add((blocks, groups))
                    assert bounds.uncovered(blocks, groups) == 0, (out_f, cells, m)


def described(out_f, in_f, bits=3):
    """A layout to ask sizes of (no memory is read for that)."""
    from ixrun_amd import _lib

    some = 1 << 12
    return _lib.IxhLanes(bits, out_f, in_f, some, int(_lib.lib().ixh_lanes_plane_words(out_f, in_f, bits)), some, some, some, 64, some)


def prompt_bytes(out_f, in_f, rows):
    from ixrun_amd import _lib

    return int(_lib.lib().ixh_lanes_gemm_workspace_bytes(C.byref(described(out_f, in_f)), rows))


@pytest.mark.parametrize("bits", [3, 4, 5, 8])
def test_few_rows_ask_for_no_scratch(bits):
    """One to four rows whose activations fit into LDS whole are summed there; longer rows go in slices, which need scratch as 5 to
    16 rows do."""
    from ixrun_amd import _lib

    def need(out_f, in_f, m):
        return int(_lib.lib().ixh_lanes_gemv_workspace_bytes(C.byref(described(out_f, in_f, bits)), m))

    for out_f, in_f in ((1536, 1536), (256, 17408), (5120, 17408), (17408, 5120)):
        assert [need(out_f, in_f, m) for m in (1, 2)] == [0, 0]
        assert need(out_f, in_f, 16) > 0
    assert need(17408, 5120, 4) == need(1536, 1536, 3) == 0
    assert all(need(64, 100000, m) > 0 for m in (1, 2, 3, 4))


@pytest.mark.parametrize("rows,need", [(1, 0), (4, 0), (8, 1), (16, 1), (100, 1), (512, 1)])
def test_too_little_scratch_is_refused(rows, need):
    """With the bytes that the size call names less one, and with none: before anything is launched."""
    from ixrun_amd import _lib

    L, s, some = _lib.lib(), described(5120, 17408), 1 << 12
    call, size = (L.ixh_lanes_gemv, L.ixh_lanes_gemv_workspace_bytes) if rows <= 4 else (L.ixh_lanes_gemm, L.ixh_lanes_gemm_workspace_bytes)
    if 4 < rows <= 16:  # (the size call answers for any count up to sixteen: what this count takes is in the refusal)
        call = L.ixh_lanes_gemv
        assert call(C.byref(s), some, 17408, None, rows, some, 5120, None, 0, None) == -4
        n = int(L.ixh_last_error().split(b" bytes needed")[0].split()[-1])
        assert 0 < n <= int(L.ixh_lanes_gemv_workspace_bytes(C.byref(s), rows))
    else:
        n = int(size(C.byref(s), rows))
    assert (n > 0) == bool(need)
    if n:
        for at, given in ((some, n - 1), (None, n), (None, 0)):
            assert call(C.byref(s), some, 17408, None, rows, some, 5120, at, given, None) == -4
            assert b"%d bytes needed, %d given" % (n, given if at else 0) in L.ixh_last_error()


@pytest.mark.parametrize("out_f,in_f,rows,parts", [
    (32768, 4096, 512, 0),  # as many tiles as workgroups
    (131072, 5120, 512, 0), (131072, 5120, 1024, 0),  # whole tiles for each
    (5120, 17408, 512, 240),  # six workgroups to a tile
    (17408, 5120, 512, 256 + 135),  # 256 workgroups share 136 tiles
    (40000, 5120, 512, 256 + 255),  # and 313
])
def test_scratch_of_prompts_is_what_is_written(out_f, in_f, rows, parts):
    """The activations in the kernel's order and 256 KB for each part of a tile, nothing for tiles that one workgroup finishes
    (256 CUs: without a GPU the library plans for as many)."""
    import torch

    if torch.cuda.is_available() and torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("figures of 256 CUs")
    x = -(-in_f // 512) * 512 * rows * 2
    assert prompt_bytes(out_f, in_f, rows) == 15 + x + parts * 512 * 128 * 4
