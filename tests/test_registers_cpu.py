"""Registers that the lane kernels of the built library spill to memory, from the code objects' metadata (no GPU needed)."""
import os
import re
import shutil
import struct
import subprocess

import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ixrun_amd", "csrc", "libixhip.so")
READELF = shutil.which("llvm-readelf", path="/opt/rocm/llvm/bin") or shutil.which("llvm-readelf")
# 512 rows a tile: 128 sums a lane and the operands beside them; eight blocks of 16 rows on a plane of 8 bits
KNOWN = {**{f"k_lanes_prompt<{bits},4,1>": 18 for bits in (3, 4, 5, 8)}, "k_lanes_gemm<8,8,2>": 3}


def spilled(tmp_path):
    data, at, found = open(LIB, "rb").read(), -1, {}
    while (at := data.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 1)) >= 0:
        entry = at + 32
        for _ in range(struct.unpack_from("<Q", data, at + 24)[0]):
            offset, size, length = struct.unpack_from("<QQQ", data, entry)
            target, entry = data[entry + 24 : entry + 24 + length], entry + 24 + length
            if b"gfx950" not in target or not size:
                continue
            (tmp_path / "code").write_bytes(data[at + offset : at + offset + size])
            notes = subprocess.run([READELF, "--notes", str(tmp_path / "code")], capture_output=True, text=True, check=True).stdout
            for kernel in re.split(r"\n  - ", notes)[1:]:
                name = re.search(r"\.name: +\S*?(k_lanes_[a-z]+)I((?:L\w\d+E)+)", kernel)
                count = re.search(r"\.vgpr_spill_count: +(\d+)", kernel)
                if name and count:
                    found["%s<%s>" % (name.group(1), ",".join(re.findall(r"L\w(\d+)E", name.group(2))))] = int(count.group(1))
    return found


@pytest.mark.skipif(READELF is None or not os.path.exists(LIB), reason="needs the built library and llvm-readelf")
def test_lane_kernels_spill_no_more_than_is_known(tmp_path):
    found = spilled(tmp_path)
    assert {"k_lanes_gemm<3,6,2>", "k_lanes_rows<5,16,0>", "k_lanes_gemv<5,1,1>", "k_lanes_prompt<5,4,1>"} <= set(found)
    assert {name: n for name, n in found.items() if n > KNOWN.get(name, 0)} == {}
