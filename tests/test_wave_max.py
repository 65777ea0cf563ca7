"""The wavefront maximum's lane moves, replayed on the CPU against its butterfly.

wave_max (osqp_amd/csrc/hip/hip_internal.h) is a butterfly of xor distances 32,
16, 8, 4, 2, 1 whose step keeps a lane's own NaN and passes over the other
lane's.  With NaNs the two lanes of a pair may then hold different values, so
each step has to read the xor's own lane.  This test reads the steps and the
DPP moves from the source, models each move as __builtin_amdgcn_update_dpp does
(lanes outside the bank mask or without a source keep `old`), and compares all
64 lanes with the butterfly, NaNs in every number of lanes.
"""
import math
import os
import random
import re

from .conftest import ROOT

SRC = os.path.join(ROOT, "osqp_amd", "csrc", "hip", "hip_internal.h")


def _moves():
    """{D: [(ctrl, bank mask)]} of lane_xor_row, in order."""
    src = open(SRC).read()
    body = src[src.index("T lane_xor_row(T v)"):]
    body = body[:body.index("\n}\n")]
    out = {}
    for line in body.splitlines():
        d = re.search(r"D == (\d+)\)? ?(?:return|,)", line)
        if d:
            cur = int(d.group(1))
        m = re.search(r"update_dpp\(\w+, w, (0x[0-9A-Fa-f]+), 0xf, (0x[0-9a-f]+), false\)", line)
        if m:
            out.setdefault(cur, []).append((int(m.group(1), 16), int(m.group(2), 16)))
    return out


def _steps():
    src = open(SRC).read()
    body = src[src.index("T wave_max(T v)"):]
    body = body[:body.index("\n}\n")]
    return [(k, int(d)) for k, d in re.findall(r"step\((lane_\w+)<(\d+)>\(v\)\);", body)]


def _dpp(old, v, ctrl, banks):
    out = []
    for lane in range(64):
        row, i = lane // 16 * 16, lane % 16
        src = None
        if (banks >> (i // 4)) & 1:
            if ctrl <= 0xFF:                  # quad_perm
                src = lane // 4 * 4 + ((ctrl >> (2 * (i % 4))) & 3)
            elif 0x101 <= ctrl <= 0x10F:      # row_shl:n
                src = lane + ctrl - 0x100 if i + ctrl - 0x100 < 16 else None
            elif 0x111 <= ctrl <= 0x11F:      # row_shr:n
                src = lane - (ctrl - 0x110) if i >= ctrl - 0x110 else None
            elif 0x121 <= ctrl <= 0x12F:      # row_ror:n
                src = row + (i - (ctrl - 0x120)) % 16
            else:
                raise AssertionError(f"DPP control {ctrl:#x} not modelled")
        out.append(v[src] if src is not None else old[lane])
    return out


def _read(kind, d, v, moves):
    if kind == "lane_xor_wide":
        return [v[i ^ d] for i in range(64)]
    if kind == "lane_ror":
        return _dpp(v, v, 0x120 + d, 0xF)
    assert kind == "lane_xor_row", kind
    out = [None] * 64
    for ctrl, banks in moves[d]:
        out = _dpp(out, v, ctrl, banks)
    return out


def _run(v, steps, moves):
    for kind, d in steps:
        o = _read(kind, d, v, moves)
        v = [b if b > a else a for a, b in zip(v, o)]
    return v


def _same(a, b):
    return all((math.isnan(x) and math.isnan(y)) or x == y for x, y in zip(a, b))


def test_wave_max_reads_the_butterflys_lanes():
    steps, moves = _steps(), _moves()
    assert [d for _, d in steps] == [32, 16, 8, 4, 2, 1] and sorted(moves) == [1, 2, 4, 8]
    rng = random.Random(7)
    rotated = [("lane_ror", d) if d < 16 else (k, d) for k, d in steps]
    caught = 0
    for k in range(2000):
        v = [rng.uniform(0, 1) for _ in range(64)]
        for i in rng.sample(range(64), k % 65):
            v[i] = math.nan
        want = list(v)
        for d in (32, 16, 8, 4, 2, 1):
            want = [b if b > a else a for a, b in zip(want, [want[i ^ d] for i in range(64)])]
        assert _same(_run(v, steps, moves), want)
        caught += not _same(_run(v, rotated, moves), want)
    assert caught > 100  # rotations read other lanes of the pair
