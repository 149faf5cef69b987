"""The built gfx950 code objects' metadata: no kernel that a call can reach by
its own schedule keeps registers in scratch memory."""

import os
import shutil
import struct
import subprocess

import pytest
import yaml

from flaggems_sglang import _capi

LLVM = "/opt/rocm/llvm/bin"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"

# fp8 on the 160-row configuration (forced by flag only) and GEMM1 streaming 64
# rows on eight waves (instantiated, never launched: GEMM1 takes eight for one
# token only)
SPILLING = ("moe_gemm_tiled_kernelILi1ENS_7TileCfgILi160E",
            "moe_gemm_stream_kernelILi0ELi4ELi8ELb1ELb0ELb0E",
            "moe_gemm_stream_kernelILi2ELi4ELi8ELb1ELb0ELb0E")


def _kernels(lib, tmp):
    """[(name, metadata)] of every kernel for gfx950 in the library."""
    fat = os.path.join(tmp, "fat")
    subprocess.run([f"{LLVM}/llvm-objcopy", "--dump-section", f".hip_fatbin={fat}", lib,
                    os.path.join(tmp, "copy.so")], check=True, capture_output=True)
    with open(fat, "rb") as f:
        data = f.read()
    out, at = [], data.find(MAGIC)
    while at >= 0:  # one bundle per object file
        count, = struct.unpack_from("<Q", data, at + 24)
        p = at + 32
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, p)
            triple = data[p + 24:p + 24 + length].decode()
            p += 24 + length
            if "gfx950" not in triple or size == 0:
                continue
            obj = os.path.join(tmp, "obj")
            with open(obj, "wb") as f:
                f.write(data[at + offset:at + offset + size])
            notes = subprocess.run([f"{LLVM}/llvm-readelf", "--notes", obj], check=True,
                                   capture_output=True, text=True).stdout
            meta = notes[notes.index("---"):notes.index("...\n")]
            kernels = yaml.safe_load(meta).get("amdhsa.kernels") or []
            out += [(k[".name"], k) for k in kernels]
        at = data.find(MAGIC, at + 1)
    return out


@pytest.mark.skipif(not all(shutil.which(f"{LLVM}/{t}") for t in ("llvm-objcopy", "llvm-readelf")),
                    reason="no LLVM object tools under /opt/rocm")
def test_no_scratch_memory(tmp_path):
    lib = os.path.join(os.path.dirname(_capi.__file__), _capi.LIB_NAME)
    kernels = _kernels(lib, str(tmp_path))
    assert len(kernels) > 150
    spilled = {n: (k[".private_segment_fixed_size"], k[".vgpr_spill_count"]) for n, k in kernels
               if (k[".private_segment_fixed_size"] or k[".vgpr_spill_count"])
               and not any(s in n for s in SPILLING)}
    assert not spilled, spilled
