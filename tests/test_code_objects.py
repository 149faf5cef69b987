"""The built gfx950 code objects: no kernel that a call can reach by its own
schedule keeps registers in scratch memory, and the quantisers' divisions."""

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


LIB = os.path.join(os.path.dirname(_capi.__file__), _capi.LIB_NAME)
pytestmark = pytest.mark.skipif(
    not all(shutil.which(f"{LLVM}/{t}") for t in ("llvm-objcopy", "llvm-readelf", "llvm-objdump")),
    reason="no LLVM object tools under /opt/rocm")


def _objects(lib, tmp):
    """The paths of the library's gfx950 code objects."""
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
            out.append(os.path.join(tmp, f"obj{len(out)}"))
            with open(out[-1], "wb") as f:
                f.write(data[at + offset:at + offset + size])
        at = data.find(MAGIC, at + 1)
    return out


def _tool(name, *args):
    return subprocess.run([f"{LLVM}/{name}", *args], check=True, capture_output=True,
                          text=True).stdout


def _kernels(obj):
    """[(name, metadata)] of an object's kernels."""
    notes = _tool("llvm-readelf", "--notes", obj)
    meta = notes[notes.index("---"):notes.index("...\n")]
    return [(k[".name"], k) for k in yaml.safe_load(meta).get("amdhsa.kernels") or []]


def test_no_scratch_memory(tmp_path):
    kernels = [k for obj in _objects(LIB, str(tmp_path)) for k in _kernels(obj)]
    assert len(kernels) > 150
    spilled = {n: (k[".private_segment_fixed_size"], k[".vgpr_spill_count"]) for n, k in kernels
               if (k[".private_segment_fixed_size"] or k[".vgpr_spill_count"])
               and not any(s in n for s in SPILLING)}
    assert not spilled, spilled


def test_plain_sum_carries_no_output_scale(tmp_path):
    """The unscaled sum of eight (or two) slots rounds its eight values once:
    no second rounding behind a test of the output's scale."""
    packs = {}
    for obj in _objects(LIB, str(tmp_path)):
        for n in (n for n, _ in _kernels(obj) if "moe_sum_tk_kernel" in n):
            code = _tool("llvm-objdump", "-d", f"--disassemble-symbols={n}", obj)
            packs[n] = code.count("v_cvt_pk_bf16_f32")
    plain = [c for n, c in packs.items() if "Lb0E" in n]
    assert len(plain) == 2 and all(c <= 4 for c in plain), packs


def test_quantisers_divide_per_row_only(tmp_path):
    """The quantisers divide twice a row or group (its scale and the scale's
    reciprocal) and not per value, infinities included."""
    seen = set()
    for obj in _objects(LIB, str(tmp_path)):
        names = [n for n, _ in _kernels(obj) if "quant_int8_token" in n or "quant_fp8_group" in n]
        for n in names:
            code = _tool("llvm-objdump", "-d", f"--disassemble-symbols={n}", obj)
            seen.add(n)
            assert code.count("v_div_fixup_f32") <= 2, n
    assert len(seen) > 10
