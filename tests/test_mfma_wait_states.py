"""Wait states after matrix instructions, in the code the compiler made of the HIP kernels.

The hardware does not hold a vector instruction back until an MFMA's result is there: the compiler
puts enough instructions between. It counts them along one way to the reader only, so where a
branch lies between, a shorter way can arrive too soon and the reader gets some of the results
without the last product. The kernels wait by themselves there (wait_mfma); this test walks every
way from each MFMA of the built library.

Wait states needed by a vector or memory instruction that reads or writes the result: two more than
the passes of an f32 MFMA, three more than those of a 16-bit one.
"""

import pathlib
import re
import shutil
import subprocess

import pytest

LIB = pathlib.Path(__file__).resolve().parents[1] / "flat-attention_amd/flat_attention_amd/libflat_hip.so"
OBJDUMP = pathlib.Path("/opt/rocm/llvm/bin/llvm-objdump")
PASSES = {"f32_32x32x2_f32": 16, "f32_16x16x4_f32": 8,
          "f32_32x32x16_bf16": 8, "f32_32x32x16_f16": 8, "f32_32x32x8_bf16": 8, "f32_32x32x8_f16": 8,
          "f32_16x16x32_bf16": 4, "f32_16x16x32_f16": 4, "f32_16x16x16_bf16": 4, "f32_16x16x16_f16": 4}
REG = re.compile(r"\b([va])(?:\[(\d+):(\d+)\]|(\d+)\b)")


def registers(text):
    out = set()
    for kind, lo, hi, one in REG.findall(text):
        out.update((kind, r) for r in range(int(lo or one), int(hi or one) + 1))
    return out


def parse(listing):
    """{kernel: [(op, operands, index of the branch's target or None)]}"""
    kernels, code, at = {}, None, {}
    for line in listing.splitlines():
        head = re.match(r"[0-9a-f]+ <(\w+)>:", line)
        if head:
            code, at = [], {}
            kernels[head[1]] = (code, at)
            continue
        m = re.match(r"\t(\w+)\s*(.*?)\s*// ([0-9A-F]{12}):.*?(?:<\w+\+0x([0-9a-f]+)>)?$", line)
        if m and code is not None:
            addr = int(m[3], 16)
            at[addr] = len(code)
            code.append((m[1], m[2], addr, m[4]))
    out = {}
    for name, (code, at) in kernels.items():
        base = code[0][2] if code else 0
        out[name] = [(op, args, at.get(base + int(to, 16)) if to and "branch" in op else None)
                     for op, args, _, to in code]
    return out


def too_soon(code):
    """[(MFMA, reader, wait states, needed)] over every way from each MFMA of one kernel."""
    found = []
    for n, (op, args, _) in enumerate(code):
        if not op.startswith("v_mfma_"):
            continue
        kind = re.match(r"v_mfma_(f32_\d+x\d+x\d+_(?:f32|bf16|f16))", op)[1]
        passes = PASSES[kind]
        need = passes + (2 if kind.endswith("x2_f32") or kind.endswith("x4_f32") else 3)
        dst = registers(args.split(", ")[0])
        seen, ways = {}, [(n + 1, 0)]
        while ways:
            i, states = ways.pop()
            while i < len(code) and states < need and seen.get(i, need) > states:
                seen[i] = states
                o, a, to = code[i]
                if o.startswith("s_cbranch"):
                    ways.append((to, states + 1))
                elif o == "s_branch":
                    i, states = to, states + 1
                    continue
                elif o == "s_endpgm":
                    break
                elif o.startswith("v_mfma"):
                    parts = a.split(", ")
                    if dst & registers(" ".join(parts[1:3])):
                        found.append((op + " " + args, o + " " + a, states, need))
                    if dst & registers(parts[0]):
                        break  # from here on it is that product's result
                    states = max(states, passes)  # the matrix core takes it after the first one's passes
                elif o.startswith(("v_", "ds_", "global_", "buffer_", "flat_", "scratch_")):
                    if dst & registers(a):
                        found.append((op + " " + args, o + " " + a, states, need))
                        break
                states += int(a, 0) + 1 if o == "s_nop" else 1
                i += 1
    return found


def test_walk_takes_the_shortest_way():
    nop = [("s_nop", "9", None)]
    mfma = ("v_mfma_f32_16x16x4_f32", "v[0:3], v8, v9, v[0:3]", None)
    read = ("v_max_f32_e32", "v4, v3, v3", None)
    branch = ("s_cbranch_scc0", "3", 3)
    assert not too_soon([mfma, *nop, read])
    assert [f[2] for f in too_soon([mfma, branch, *nop, read])] == [1]
    assert not too_soon([mfma, ("v_max_f32_e32", "v4, v5, v5", None), *nop, read])


@pytest.mark.skipif(not LIB.exists() or not OBJDUMP.exists(), reason="no built library or no disassembler")
def test_no_result_is_read_before_it_is_there(tmp_path):
    shutil.copy(LIB, tmp_path / "l.so")
    subprocess.run([OBJDUMP, "--offloading", "l.so"], cwd=tmp_path, check=True, capture_output=True)
    objects = sorted(p for p in tmp_path.glob("l.so*gfx950*") if p.stat().st_size)
    assert objects
    products, bad = 0, []
    for obj in objects:
        text = subprocess.run([OBJDUMP, "-d", obj], check=True, capture_output=True, text=True).stdout
        for name, code in parse(text).items():
            products += sum(op.startswith("v_mfma_") for op, _, _ in code)
            bad += [(name, *f) for f in too_soon(code)]
    assert products > 10000
    assert not bad, "\n".join(map(str, bad[:20]))
