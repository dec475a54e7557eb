"""What the kernels of the built library keep in registers: none puts values in scratch memory but the one that is known to (read from the code
objects' own notes; no GPU needed)."""
import os
import re
import shutil
import struct
import subprocess

import pytest

from modular_amd import _lib

LLVM = "/opt/rocm/llvm/bin"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def scratch_bytes(tmp_path):
    """kernel's mangled name -> scratch bytes per lane"""
    fat = tmp_path / "fat.bin"
    subprocess.run([f"{LLVM}/llvm-objcopy", "--dump-section", f".hip_fatbin={fat}", _lib.LIB_PATH, os.devnull], check=True)
    data, out, at = fat.read_bytes(), {}, 0
    while (at := data.find(MAGIC, at)) >= 0:
        (entries,), p = struct.unpack_from("<Q", data, at + 24), at + 32
        for _ in range(entries):
            offset, size, name_len = struct.unpack_from("<QQQ", data, p)
            target, p = data[p + 24:p + 24 + name_len], p + 24 + name_len
            if b"gfx950" not in target:
                continue
            code = tmp_path / "code.elf"
            code.write_bytes(data[at + offset:at + offset + size])
            notes = subprocess.run([f"{LLVM}/llvm-readelf", "--notes", str(code)], check=True, capture_output=True, text=True).stdout
            names = re.findall(r"^ +\.symbol: +(\S+?)\.kd$", notes, re.M)
            sizes = re.findall(r"^ +\.private_segment_fixed_size: +(\d+)$", notes, re.M)
            assert len(names) == len(sizes)
            out.update(zip(names, map(int, sizes)))
        at += len(MAGIC)
    return out


@pytest.mark.skipif(not shutil.which(f"{LLVM}/llvm-readelf"), reason="needs ROCm's LLVM tools")
def test_matmul_kernels_of_few_tokens_keep_out_of_scratch_memory(tmp_path):
    kernels = {n: s for n, s in scratch_bytes(tmp_path).items() if "gemm_skinny_kernel" in n or "gemm_mid_kernel" in n}
    assert sum("gemm_skinny_kernel" in n for n in kernels) > 50 and sum("gemm_mid_kernel" in n for n in kernels) > 50
    # 64 rows of weights against four groups of 16 tokens with block scales: 33 registers more than there are, with either epilogue
    known = "gemm_skinny_kernelILi4ELi4ELb1ELi32ELi4E"
    assert {n for n, s in kernels.items() if s > 0 and known not in n} == set()
    assert all(s <= 120 for s in kernels.values())
