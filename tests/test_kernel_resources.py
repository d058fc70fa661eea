"""What the built library says of its kernels: registers that a kernel puts into memory because it has too many ("spilled") come back in its hot
loops, where a wait for them is a wait for every load that was to stay on its way."""
import os
import re
import struct
import subprocess

import pytest

from kutacc_amd import build

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"
# kernels with spilled registers that were measured with them: two and three outside of the loop, and the accumulators of the 256-wide products
MEASURED = ("persistent_pair_kernel", "pair_gemm_big_kernel", "pair_gemm_direct_kernel")


def code_objects(data):
    """The gfx950 code objects of a library's bundles: magic, number of entries, then (offset, size, length of the target's name, name) each."""
    start = data.find(BUNDLE)
    while start >= 0:
        at = start + len(BUNDLE)
        (entries,) = struct.unpack_from("<Q", data, at)
        at += 8
        for _ in range(entries):
            offset, size, length = struct.unpack_from("<QQQ", data, at)
            target = data[at + 24:at + 24 + length].decode()
            at += 24 + length
            if "gfx950" in target and size:
                yield data[start + offset:start + offset + size]
        start = data.find(BUNDLE, at)


def test_attention_kernels_keep_their_registers(tmp_path):
    if not os.path.exists(READELF) or not os.path.exists(build.LIB_PATH):
        pytest.skip("needs the built library and ROCm's llvm-readelf")
    kernels = {}
    with open(build.LIB_PATH, "rb") as f:
        data = f.read()
    for i, code in enumerate(code_objects(data)):
        path = tmp_path / f"{i}.elf"
        path.write_bytes(code)
        notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        for name, spilled in re.findall(r"\.symbol:\s+(\S+)\.kd.*?\.vgpr_spill_count:\s+(\d+)", notes, re.S):
            kernels[name] = int(spilled)
    assert len(kernels) > 100 and any("fused_head_kernel" in k for k in kernels), len(kernels)
    spilled = {k: n for k, n in kernels.items() if n and not any(m in k for m in MEASURED)}
    assert not spilled, spilled
