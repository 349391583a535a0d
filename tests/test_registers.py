"""What the compiler made of the decode products' kernels, as the built library itself says: nothing spilled to memory."""
import os
import re
import struct
import subprocess

import pytest


def _device_code(path):
    """The gfx950 code object that a built library carries (`__CLANG_OFFLOAD_BUNDLE__`: a count, then offset, size and target of each)."""
    with open(path, "rb") as f:
        data = f.read()
    start = data.index(b"__CLANG_OFFLOAD_BUNDLE__")
    at = start + 24
    count, = struct.unpack_from("<Q", data, at)
    at += 8
    for _ in range(count):
        offset, size, length = struct.unpack_from("<QQQ", data, at)
        target = data[at + 24:at + 24 + length]
        at += 24 + length
        if target.endswith(b"gfx950"):
            return data[start + offset:start + offset + size]
    raise AssertionError(f"{path}: no gfx950 code")


def _scratch_bytes(path, folder):
    from minfer_amd.kernels import build
    readelf = os.path.join(os.path.dirname(os.path.realpath(build._hipcc())), "..", "lib", "llvm", "bin", "llvm-readelf")
    if not os.path.exists(readelf):
        pytest.skip("no llvm-readelf beside hipcc")
    code = os.path.join(folder, "code.o")
    with open(code, "wb") as f:
        f.write(_device_code(path))
    notes = subprocess.run([readelf, "--notes", code], capture_output=True, text=True, check=True).stdout
    return {name: int(size) for size, name in
            re.findall(r"\.private_segment_fixed_size:\s*(\d+)(?:(?!\.private_segment)[\s\S])*?\.symbol:\s*(\S+?)\.kd", notes)}


def test_products_of_few_rows_spill_nothing(tmp_path):
    """A reload from scratch is counted with the weights in flight and waits for them: the kernels that stream weights keep to
    their registers at every width they are built for."""
    from minfer_amd.kernels import build
    if not build.is_current("gemm_bf16"):
        build.compile_library("gemm_bf16")
    scratch = _scratch_bytes(build.lib_path("gemm_bf16"), str(tmp_path))
    kinds = ("stationary16_kernel", "rolling16_kernel", "whole_kernel", "skinny_ring_kernel", "panel_kernel", "panel_dma_kernel",
             "tile_stream_kernel", "tile_step_kernel")
    few = {n: b for n, b in scratch.items() if any(k + "I" in n for k in kinds)}
    assert all(any(k + "I" in n for n in few) for k in kinds)
    assert not {n: b for n, b in few.items() if b}


def _loads_marked_as_read_once(path, folder, names):
    """Of the named kernels: how many loads of 16 bytes they have, how many of those are marked, and how many exchanges of values between the
    lanes l and l ^ 8 of 16."""
    from minfer_amd.kernels import build
    objdump = os.path.join(os.path.dirname(os.path.realpath(build._hipcc())), "..", "lib", "llvm", "bin", "llvm-objdump")
    if not os.path.exists(objdump):
        pytest.skip("no llvm-objdump beside hipcc")
    code = os.path.join(folder, "code.o")
    with open(code, "wb") as f:
        f.write(_device_code(path))
    text = subprocess.run([objdump, "-d", "--no-show-raw-insn", "--disassemble-symbols=" + ",".join(names), code], capture_output=True,
                          text=True, check=True).stdout
    found, name = {n: [0, 0, 0] for n in names}, None
    for line in text.splitlines():
        head = re.match(r"[0-9a-f]+ <(\S+)>:", line)
        if head:
            name = head.group(1)
        elif name in found and re.search(r"\b(global|flat)_load_dwordx4\b", line):
            found[name][0] += 1
            found[name][1] += bool(re.search(r"\bnt\b", line))
        elif name in found:
            found[name][2] += "row_ror:8" in line
    return found


def test_which_weights_are_marked_as_read_once(tmp_path):
    """The kernels of few rows mark the weights that they read from the tiled copy, whose loads take whole lines.  From the matrix a
    load takes half a line of each row: marked, the line would be fetched again for the other half, and so none is but with a K of up to 2,048
    in `stationary16_kernel`, where both halves are asked for close together."""
    from minfer_amd.kernels import build
    if not build.is_current("gemm_bf16"):
        build.compile_library("gemm_bf16")
    path = build.lib_path("gemm_bf16")
    once, tiled = {}, 0                           # (the last yes-or-no parameters: the copy; of one kernel the mark behind it)
    for n in _scratch_bytes(path, str(tmp_path)):
        kind = re.search(r"\d(rolling16|skinny_ring|panel)_kernelI(?:L[ib]\d+E)*?Lb([01])EEE", n)
        if kind:
            once[n] = kind.group(2) == "1"
            tiled += once[n]
        kind = re.search(r"\d+stationary16_kernelILi(\d+)ELi\d+ELi\d+ELb([01])ELb[01]ELb([01])ELi(\d)ELb([01])EEE", n)
        if kind:
            steps, pair, copy, waves, mark = (int(x) for x in kind.groups())
            once[n] = mark == 1
            tiled += copy
            assert mark >= copy and (mark == copy or (not pair and steps * waves * 32 <= 2048)), n
    assert len(once) > 2 * tiled > 0
    for n, (loads, marked, _) in _loads_marked_as_read_once(path, str(tmp_path), sorted(once)).items():
        assert loads > 0 and (marked > 0) == once[n], (n, loads, marked)


def test_experts_marked_loads_take_whole_lines(tmp_path):
    """The chosen experts' matrices are rows, marked as read once: a load takes 128 bytes of eight of them, and lanes exchange
    four values of every two such loads to have the rows as MFMA operands."""
    from minfer_amd.kernels import build
    if not build.is_current("moe"):
        build.compile_library("moe")
    path = build.lib_path("moe")
    names = sorted(n for n in _scratch_bytes(path, str(tmp_path)) if "moe_sparse_mfma_kernel" in n)
    assert len(names) == 4
    for n, (loads, marked, exchanges) in _loads_marked_as_read_once(path, str(tmp_path), names).items():
        assert loads > marked > 0 and exchanges >= 2 * marked, (n, loads, marked, exchanges)
