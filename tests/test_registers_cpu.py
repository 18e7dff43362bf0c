"""What the built library's code objects say of its kernels (no GPU needed): registers that the lane kernels spill to memory, and the
mode for denormals."""
import os
import re
import shutil
import struct
import subprocess

import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ixrun_amd", "csrc", "libixhip.so")
HIPCC = "/opt/rocm/bin/hipcc"
READELF = shutil.which("llvm-readelf", path="/opt/rocm/llvm/bin") or shutil.which("llvm-readelf")
# 512 rows a tile: 128 sums a lane and the operands beside them; eight blocks of 16 rows on a plane of 8 bits
KNOWN = {**{f"k_lanes_prompt<{bits},4,1>": 18 for bits in (3, 4, 5, 8)}, "k_lanes_gemm<8,8,2>": 3}


def code_objects(data):
    at = -1
    while (at := data.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 1)) >= 0:
        entry = at + 32
        for _ in range(struct.unpack_from("<Q", data, at + 24)[0]):
            offset, size, length = struct.unpack_from("<QQQ", data, entry)
            target, entry = data[entry + 24 : entry + 24 + length], entry + 24 + length
            if b"gfx950" in target and size:
                yield data[at + offset : at + offset + size]


def spilled(tmp_path):
    found = {}
    for code in code_objects(open(LIB, "rb").read()):
        (tmp_path / "code").write_bytes(code)
        notes = subprocess.run([READELF, "--notes", str(tmp_path / "code")], capture_output=True, text=True, check=True).stdout
        for kernel in re.split(r"\n  - ", notes)[1:]:
            name = re.search(r"\.name: +\S*?(k_lanes_[a-z]+)I((?:L\w\d+E)+)", kernel)
            count = re.search(r"\.vgpr_spill_count: +(\d+)", kernel)
            if name and count:
                found["%s<%s>" % (name.group(1), ",".join(re.findall(r"L\w(\d+)E", name.group(2))))] = int(count.group(1))
    return found


def symbols(code):
    """(name, its bytes' place in the code object, their number) of all symbols that have a place."""
    sections, section_size, n_sections = struct.unpack_from("<Q10xHH", code, 0x28)[0], *struct.unpack_from("<HH", code, 0x3A)
    headers = [struct.unpack_from("<IIQQQQIIQQ", code, sections + i * section_size) for i in range(n_sections)]
    for _, kind, _, _, offset, size, link, _, _, _ in headers:
        if kind != 2:  # the symbol table
            continue
        names = headers[link][4]
        for at in range(offset, offset + size, 24):
            name_at, _, _, section, value, length = struct.unpack_from("<IBBHQQ", code, at)
            if section and section < n_sections:
                name = code[names + name_at : code.index(b"\0", names + name_at)].decode()
                yield name, value - headers[section][3] + headers[section][4], length


def denormal_modes(code):
    """{kernel: its descriptor's mode for fp32 denormals}: 3 where they are kept, 0 where they are flushed."""
    return {name[:-3]: (struct.unpack_from("<I", code, at + 48)[0] >> 16) & 3 for name, at, length in symbols(code)
            if name.endswith(".kd") and length == 64}


@pytest.mark.skipif(READELF is None or not os.path.exists(LIB), reason="needs the built library and llvm-readelf")
def test_lane_kernels_spill_no_more_than_is_known(tmp_path):
    found = spilled(tmp_path)
    assert {"k_lanes_gemm<3,6,2>", "k_lanes_rows<5,16,0>", "k_lanes_gemv<5,1,1>", "k_lanes_prompt<5,4,1>"} <= set(found)
    assert {name: n for name, n in found.items() if n > KNOWN.get(name, 0)} == {}


@pytest.mark.skipif(not os.path.exists(LIB), reason="needs the built library")
def test_kernels_keep_denormals():
    """Addresses are worked out in them."""
    found = {}
    for code in code_objects(open(LIB, "rb").read()):
        found.update(denormal_modes(code))
    assert sum("k_lanes_" in name or "dense" in name for name in found) > 50
    assert [name for name, mode in found.items() if mode != 3] == []


@pytest.mark.skipif(not os.path.exists(LIB), reason="needs the built library")
def test_kernels_of_small_layers_are_short():
    """A launch fetches its instructions anew, and a small layer of a graph waits for little else: its kernel has at most half of
    k_lanes_gemv's."""
    size = {name: length for code in code_objects(open(LIB, "rb").read()) for name, _, length in symbols(code) if "k_lanes_gemv" in name and not name.endswith(".kd")}
    of = lambda *parts: next(length for name, length in size.items() if all(p in name for p in parts))
    for bits in (3, 4, 5, 8):
        for rows in (1, 2, 4):
            assert of("k_lanes_gemv_fewI", f"ILi{bits}ELi{rows}ELi1E") <= 0.5 * of("k_lanes_gemvI", f"ILi{bits}ELi{rows}ELb1E")


@pytest.mark.skipif(shutil.which(HIPCC) is None, reason="needs hipcc")
@pytest.mark.parametrize("given", [[], ["-ffast-math", "-fgpu-flush-denormals-to-zero"], ["-fdenormal-fp-math=preserve-sign"]])
def test_build_keeps_denormals_whatever_flags_it_is_given(tmp_path, given):
    """build.sh with stand-ins for the compilers, which write down what they are given; a kernel compiled that way."""
    csrc, tools = tmp_path / "ixrun_amd" / "csrc", tmp_path / "tools"
    csrc.mkdir(parents=True)
    tools.mkdir()
    shutil.copy(os.path.join(os.path.dirname(LIB), "build.sh"), csrc)
    (tools / "hipcc").write_text('#!/bin/sh\nout=; for a in "$@"; do case "$out" in next) out="$a";; esac; case "$a" in -o) out=next;; esac; done\n'
                                 'case " $* " in *" -c "*) echo "$@" > "$out.flags"; touch "$out";; esac\n')
    (tools / "g++").write_text("#!/bin/sh\n")
    for tool in ("hipcc", "g++"):
        (tools / tool).chmod(0o755)
    env = dict(os.environ, PATH=f"{tools}:{os.environ['PATH']}", HIPCC=str(tools / "hipcc"))
    subprocess.run(["sh", str(csrc / "build.sh"), *given], env=env, check=True, capture_output=True)
    commands = sorted((csrc / "build").glob("*.flags"))
    assert len(commands) > 10
    (tmp_path / "k.hip").write_text("__attribute__((global)) void k(float *p) { p[0] = p[1] * p[2]; }\n")
    lines = {" ".join(c.read_text().split(" -c ")[0].split()) for c in commands}
    for flags in lines:
        asm = subprocess.run([HIPCC, *flags.split(), "--cuda-device-only", "-S", str(tmp_path / "k.hip"), "-o", "-"], capture_output=True, text=True,
                             check=True).stdout
        assert ".amdhsa_float_denorm_mode_32 3" in asm, flags
