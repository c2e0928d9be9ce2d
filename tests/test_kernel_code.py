"""What the compiler made of the kernels in the library that is built, where a kernel's speed hangs on it and its results
do not show it. Reads the code of this project's own build; needs no GPU."""

import os
import re
import shutil
import struct
import subprocess

import msgpack
import pytest

from llama_lite_npu_amd import _lib
from llama_lite_npu_amd.build import LIB_PATH

EM_AMDGPU = 224


@pytest.fixture(scope="module")
def code_objects():
    _lib.load()                                         # (builds the library if there is none)
    data = LIB_PATH.read_bytes()
    found = [m.start() for m in re.finditer(b"\x7fELF", data)]
    found = [data[at:] for at in found if struct.unpack_from("<H", data, at + 18)[0] == EM_AMDGPU]
    assert found
    return found


@pytest.fixture(scope="module")
def listings(code_objects, tmp_path_factory):
    """Instructions per kernel."""
    tool = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"
    if not os.path.exists(tool):
        pytest.skip("no llvm-objdump")
    out = {}
    for i, code in enumerate(code_objects):
        path = tmp_path_factory.mktemp("code") / f"{i}.co"
        path.write_bytes(code)
        text = subprocess.run([tool, "-d", "--no-show-raw-insn", "--no-leading-addr", str(path)], capture_output=True,
                              text=True, check=True).stdout
        for body in re.split(r"\n(?=<\S+>:)", text):
            name = re.match(r"<(\S+)>:", body)
            if name:
                out[name[1]] = [line.split("//")[0].strip() for line in body.splitlines()[1:]]
    return out


@pytest.fixture(scope="module")
def metadata(code_objects):
    """The compiler's notes per kernel (section type 7, AMDGPU metadata: note type 32)."""
    out = {}
    for code in code_objects:
        sections, = struct.unpack_from("<Q", code, 40)
        size, count = struct.unpack_from("<HH", code, 58)
        for at in range(sections, sections + size * count, size):
            if struct.unpack_from("<I", code, at + 4)[0] != 7:
                continue
            note, = struct.unpack_from("<Q", code, at + 24)
            name_bytes, bytes_, kind = struct.unpack_from("<III", code, note)
            if kind == 32:
                first = note + 12 + (name_bytes + 3) // 4 * 4
                notes = msgpack.unpackb(code[first:first + bytes_], strict_map_key=False)
                out.update({k[".name"]: k for k in notes["amdhsa.kernels"]})
    return out


def test_a_prefix_step_of_narrow_heads_leaves_room_beside_a_workgroup(metadata):
    """Head dim 64: three wavefronts per SIMD, which 168 registers (of 512, in steps of 8) allow, and LDS for two workgroups:
    the four wavefronts of a prefix workgroup over codes and eight of the other role. Nothing spilled for it."""
    kernels = {name: k for name, k in metadata.items() if "hd6418prefix_step_kernel" in name}
    assert len(kernels) == 4
    for name, k in kernels.items():
        assert k[".vgpr_count"] <= 168 and k[".vgpr_spill_count"] == 0, (name, k[".vgpr_count"], k[".vgpr_spill_count"])
        assert 2 * k[".group_segment_fixed_size"] <= 160 * 1024, name


def test_page_ids_are_requested_behind_the_barrier(listings):
    """A wavefront waits for all of its requests in front of a tile's barrier. Page ids (the only single dwords a tile
    loop loads from memory) that are requested between a tile's last MFMA and that wait are a round trip in the open: once
    where the loop is entered, never inside it."""
    forms = ("prefix_step_kernelILi2ELi0E", "prefill_tiled_kernelILi0E", "prefill_tiled_kernelILi7E", "two_group_kernelILi0E")
    kernels = {name: code for name, code in listings.items() if any(form in name for form in forms)}
    assert len(kernels) >= 12
    load = re.compile(r"global_load_dword v\d+, v(\d+, s)?\[")
    for name, code in kernels.items():
        assert any(load.match(ins) for ins in code), name
        exposed = 0
        for i, ins in enumerate(code):
            if not ins.startswith("s_barrier"):
                continue
            before = []
            for prev in reversed(code[:i]):
                if "mfma" in prev or prev.startswith("s_barrier"):
                    break
                before.append(prev)
            exposed += len(before) < 60 and any(load.match(x) for x in before)
        assert exposed <= 1, f"{name}: {exposed} waits for page ids"
