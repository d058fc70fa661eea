"""What the built library says of its kernels: registers that a kernel puts into memory because it has too many ("spilled") come back in its hot
loops, where a wait for them is a wait for every load that was to stay on its way."""
import os
import re
import shutil
import struct
import subprocess
import sys

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


# Launches that print what they ask for instead of starting anything, on a device of 256 CUs
LAUNCHES = r"""
#include <stddef.h>
#include <stdint.h>
#include <stdio.h>
typedef struct { uint32_t x, y, z; } dim3;
int hipGetDevice(int *d) { *d = 0; return 0; }
int hipDeviceGetAttribute(int *v, int which, int d) { *v = 256; return 0; }
int hipFuncSetAttribute(const void *f, int which, int v) { return 0; }
int hipGetLastError(void) { return 0; }
unsigned __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, void *stream)
{
    printf("launch %u %u %zu\n", grid.x, block.x, lds);
    fflush(stdout);
    return 1; // not 0: what <<<>>> expands to goes no further
}
"""
CALL = """
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)  # in front of the runtime that the library brings
L = ctypes.CDLL(sys.argv[2])
v, i = ctypes.c_void_p, ctypes.c_int64
L.kutacc_hip_transition_block.argtypes = [v, v, v, ctypes.c_float, v, v, v, v, v, i, i, i, i, ctypes.c_int32, v]
at = 1 << 32  # an address that nothing reads
rows, c_o, c_i, dtype = map(int, sys.argv[3:])
print("rc", L.kutacc_hip_transition_block(at, at, at, 1e-5, at, at, at, at, at, 1 << 40, rows, c_o, c_i, dtype, None), flush=True)
"""


# The largest hidden layers that a CU's workgroups have room for, and the model's own.  The LDS comes in pieces of 1280 bytes.
@pytest.mark.parametrize("c_o,c_i,per_cu", [(64, 256, 4), (64, 2048, 4), (128, 64, 3), (128, 512, 3), (128, 1088, 3), (128, 1152, 3), (256, 64, 2),
                                            (256, 1024, 2), (256, 2048, 2)])
def test_transition_fits_its_workgroups_into_the_lds(tmp_path, c_o, c_i, per_cu):
    cc = shutil.which("gcc") or shutil.which("cc")
    if cc is None or not os.path.exists(build.LIB_PATH):
        pytest.skip("needs the built library and a C compiler")
    from kutacc_amd import capi
    source, shim = tmp_path / "launches.c", tmp_path / "launches.so"
    source.write_text(LAUNCHES)
    subprocess.run([cc, "-shared", "-fPIC", "-O1", str(source), "-o", str(shim)], check=True)
    out = subprocess.run([sys.executable, "-c", CALL, str(shim), build.LIB_PATH, "600000", str(c_o), str(c_i), str(capi.K_BF16)], capture_output=True,
                         text=True, check=True).stdout
    assert "rc 0" in out, out
    launches = re.findall(r"launch (\d+) (\d+) (\d+)", out)
    assert len(launches) == 1 and launches[0][1] == "256", out
    pieces = -(-int(launches[0][2]) // 1280)
    assert per_cu * pieces <= 160 * 1024 // 1280, f"{launches[0][2]} bytes: {160 * 1024 // 1280 // pieces} workgroups a CU"


# (on 256 CUs) one workgroup of eight waves a CU where that pays: not for few rows with few hidden units, which it slowed down by up to 8 %
@pytest.mark.parametrize("rows,c_o,c_i,threads", [(9000, 128, 64, 256), (32768, 128, 64, 256), (32769, 128, 64, 512), (9000, 128, 128, 256), (32768, 128, 128, 256),
                                                  (33000, 128, 128, 512), (9000, 128, 192, 512), (65536, 128, 512, 512), (65537, 128, 512, 256),
                                                  (50000, 256, 64, 256), (32768, 256, 1024, 256), (32769, 256, 128, 512), (65537, 256, 1024, 256)])
def test_transition_takes_one_workgroup_a_cu_where_that_pays(tmp_path, rows, c_o, c_i, threads):
    cc = shutil.which("gcc") or shutil.which("cc")
    if cc is None or not os.path.exists(build.LIB_PATH):
        pytest.skip("needs the built library and a C compiler")
    from kutacc_amd import capi
    source, shim = tmp_path / "launches.c", tmp_path / "launches.so"
    source.write_text(LAUNCHES)
    subprocess.run([cc, "-shared", "-fPIC", "-O1", str(source), "-o", str(shim)], check=True)
    out = subprocess.run([sys.executable, "-c", CALL, str(shim), build.LIB_PATH, str(rows), str(c_o), str(c_i), str(capi.K_BF16)], capture_output=True,
                         text=True, check=True).stdout
    launches = re.findall(r"launch (\d+) (\d+) (\d+)", out)
    assert "rc 0" in out and [int(n) for _, n, _ in launches] == [threads], out
