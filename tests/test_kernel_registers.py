"""Vector registers that the compiled kernels keep in scratch memory.

Each is a store and a load in memory that the kernel's own traffic pushes out: the 20 that
decode_splitk<float, 128, 4> once had cost 18 % of a launch. The kernels listed here keep a few
outside their innermost products; all others keep none.
"""

import pathlib
import re
import shutil
import subprocess

import pytest

LIB = pathlib.Path(__file__).resolve().parents[1] / "flat-attention_amd/flat_attention_amd/libflat_hip.so"
LLVM = pathlib.Path("/opt/rocm/llvm/bin")
ALLOWED = {"decode_splitkIfLi32ELi16E": 8, "decode_splitkIfLi64ELi16E": 8, "decode_splitkIfLi128ELi16E": 8,
           "decode_splitkIfLi128ELi4E": 2, "bwd_f32_dkdvILi128E": 12}


@pytest.mark.skipif(not LIB.exists() or not (LLVM / "llvm-readelf").exists(),
                    reason="no built library or no ELF reader")
def test_no_kernel_spills_more_than_listed(tmp_path):
    shutil.copy(LIB, tmp_path / "l.so")
    subprocess.run([LLVM / "llvm-objdump", "--offloading", "l.so"], cwd=tmp_path, check=True,
                   capture_output=True)
    spills = {}
    for obj in sorted(p for p in tmp_path.glob("l.so*gfx950*") if p.stat().st_size):
        notes = subprocess.run([LLVM / "llvm-readelf", "--notes", obj], check=True,
                               capture_output=True, text=True).stdout
        spills.update((name, int(n)) for name, n in re.findall(
            r"\.name:\s+(_Z\S+).*?\.vgpr_spill_count:\s+(\d+)", notes, re.S))
    assert any("decode_splitk" in name for name in spills)
    over = {name: n for name, n in spills.items()
            if n > max((most for key, most in ALLOWED.items() if key in name), default=0)}
    assert not over, over
