"""CPU check of the rule that splits a backward's dK/dV over workgroups (fa::backward_split,
BackwardSplit in csrc/kernels.hpp): the partials' workspace stays under its limit, whatever the
shape, and the index arithmetic of the kernels (chunk and slot of a workgroup, slots of a key block)
agrees with plain loops. A small host program, built here, calls the library's own functions."""
import heapq
import os
import shutil
import subprocess

import numpy as np
import pytest

import flat_attention_amd as fa

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "flat-attention_amd")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
MIB = 1 << 20
LIMIT = 256 * MIB  # kBackwardPartialBytes


@pytest.fixture(scope="module")
def split(tmp_path_factory):
    if not shutil.which(HIPCC):
        pytest.skip("needs hipcc")
    exe = str(tmp_path_factory.mktemp("split") / "check")
    lib = os.path.join(PKG, "flat_attention_amd")
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-std=c++17", "-O1", "-x", "hip",
                    os.path.join(ROOT, "tests", "backward_split_check.cpp"),
                    "-I", os.path.join(PKG, "csrc"), "-o", exe, "-L", lib, "-lflat_hip",
                    "-Wl,-rpath," + lib], check=True, capture_output=True)

    def run(cases):
        text = "".join(" ".join(str(int(x)) for x in c) + "\n" for c in cases)
        out = subprocess.run([exe], input=text, capture_output=True, text=True, check=True)
        lines = out.stdout.splitlines()
        assert len(lines) == len(cases)
        for c, line in zip(cases, lines):
            assert not line.startswith("fault"), (c, line)
        return [tuple(int(x) for x in line.split()) for line in lines]
    return run


LONG = [(1, 64, 1, 131071, 128), (1, 64, 1, 8000, 128), (1, 64, 4, 65537, 128),
        (1, 64, 8, 131073, 128), (1, 8, 1, 16383, 128), (1, 32, 8, 32767, 128), (1, 6, 1, 131071, 64),
        (2, 32, 8, 3000, 128), (4, 12, 4, 70001, 32)]


@pytest.mark.parametrize("dtype", [fa.DTYPE_F32, fa.DTYPE_F16, fa.DTYPE_BF16])
def test_partials_stay_under_the_limit(split, dtype):
    """Long sequences of few kv heads took up to 7 GiB for a few per cent."""
    cases = [(dtype, *dims, causal, LIMIT) for dims in LONG for causal in (0, 1)]
    for case, (chunk, parts, slots, nbytes, _) in zip(cases, split(cases)):
        assert nbytes <= LIMIT, case
        if parts:  # (an f32 call may leave the split kernels)
            assert chunk > 0 and (parts == 1) == (slots == 0), case


def test_index_arithmetic_over_drawn_shapes(split):
    """Every chunk has one workgroup and one slot, under any limit; a limit of zero leaves one
    chunk to each key block, and a larger limit never a split that takes more than it."""
    rng = np.random.default_rng(5)
    cases = []
    for _ in range(400):
        hkv = int(rng.integers(1, 9))
        shape = (int(rng.integers(1, 5)), hkv * int(rng.integers(1, 17)), hkv,
                 int(np.exp(rng.uniform(0, np.log(9000)))), int(rng.choice([32, 64, 80, 128])))
        cases.append((int(rng.integers(0, 3)), *shape, int(rng.integers(0, 2)),
                      int(rng.choice([0, MIB, 8 * MIB, LIMIT]))))
    got = split(cases)
    for case, (chunk, parts, slots, nbytes, _) in zip(cases, got):
        assert nbytes <= case[-1], case
        if case[-1] == 0 and parts:
            assert parts == 1 and slots == 0, case
    assert sum(parts > 1 for _, parts, _, _, _ in got) > 50


def test_short_sequences_keep_their_split(split):
    """The limit leaves the shapes alone that the split was made for (one round of workgroups)."""
    cases = [(fa.DTYPE_BF16, 1, 6, 1, 1500, 128, 1, LIMIT), (fa.DTYPE_BF16, 1, 32, 8, 2000, 128, 1, LIMIT),
             (fa.DTYPE_BF16, 1, 8, 2, 512, 64, 1, LIMIT), (fa.DTYPE_F32, 1, 8, 2, 512, 64, 1, LIMIT)]
    assert [r[:2] for r in split(cases)] == [(2, 36), (22, 3), (1, 16), (4, 16)]


def _makespan(dims, causal, chunk, cus=256):
    """Tiles of time of a dK/dV launch in chunks of `chunk` tiles: its workgroups in dispatch order,
    each on the first CU that is free; two tiles for a workgroup, four for one with partials."""
    b, hq, hkv, s, _ = dims
    group, nkb = hq // hkv, -(-s // 128)
    all_tiles = [group * (nkb - kb if causal else nkb) for kb in range(nkb)]
    free = [0] * cus
    for p in range(-(-group * nkb // chunk) - 1, -1, -1):
        for t in all_tiles:
            if t <= p * chunk:
                break
            cost = min(chunk, t - p * chunk) + (4 if t > chunk else 2)
            for _ in range(b * hkv):
                heapq.heapreplace(free, free[0] + cost)
    return max(free)


def test_split_has_the_least_time_of_all_splits(split):
    """The chosen split's time is within 3 % (the candidates are few, time is counted in steps) of
    the best of every number of chunks that gives up to four rounds of workgroups."""
    rng = np.random.default_rng(8)
    cases = []
    while len(cases) < 40:
        hq, hkv = [(8, 2), (16, 4), (32, 8), (8, 8), (12, 4), (6, 1)][int(rng.integers(6))]
        cases.append((fa.DTYPE_BF16, int(rng.integers(1, 3)), hq, hkv,
                      int(np.exp(rng.uniform(np.log(64), np.log(4096)))), 128,
                      int(rng.integers(0, 2)), 1 << 40))
    cases += [(fa.DTYPE_BF16, 2, 32, 8, 1000, 128, 1, LIMIT), (fa.DTYPE_BF16, 1, 16, 4, 4000, 128, 1, LIMIT)]
    for case, (chunk, parts, slots, _, several) in zip(cases, split(cases)):
        dims, causal = case[1:6], case[6]
        longest = dims[1] // dims[2] * -(-dims[3] // 128)
        best = min(_makespan(dims, causal, -(-longest // p)) for p in range(1, min(longest, 40) + 1)
                   if p < 3 or dims[0] * dims[2] * p * -(-dims[3] // 128) < 8 * 256)
        assert _makespan(dims, causal, chunk) <= 1.03 * best + 1, case
