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
