"""The GEMM kernels' LDS reads in flight, checked in the compiled gfx950 code.

csrc/mlp_gemm.hip reads its fragments with inline assembly and waits for them
later (a builtin makes the compiler drain every LDS DMA before each read).  The
compiler takes such a read's destination as written at once, so nothing in the
language keeps it from copying, spilling or reusing those registers before the
data lands.  This test follows every path of every kernel in the assembly this
tree's compiler makes of the source and asserts that no instruction touches a
register that an LDS read may still write.
"""
from __future__ import annotations

import re
import subprocess

import pytest

from reversability_amd import _build


def registers(text: str) -> frozenset:
    """The vector and accumulator registers an operand list names."""
    out = set()
    for kind, first, last in re.findall(r"\b([va])\[(\d+):(\d+)\]", text):
        out |= {(kind, r) for r in range(int(first), int(last) + 1)}
    out |= {(kind, int(r)) for kind, r in re.findall(r"\b([va])(\d+)\b", text)}
    return frozenset(out)


def parse(text: str) -> dict:
    """{kernel: [(label, op, operands)]} of a gfx950 assembly file."""
    kernels, body = {}, None
    for line in text.splitlines():
        line = line.split(";")[0].strip()
        label = re.match(r"([.\w$]+):", line)
        if label:
            if not label[1].startswith("."):
                body = kernels.setdefault(label[1], [])
            elif body is not None:
                body.append((label[1], None, ""))
        elif body is not None and line and not line.startswith("."):
            op, _, rest = line.partition(" ")
            body.append((None, op, rest.strip()))
    return {name: body for name, body in kernels.items() if body}


def lgkmcnt(operands: str):
    """The LDS counter an s_waitcnt waits for, None if it leaves it alone."""
    named = re.search(r"lgkmcnt\((\d+)\)", operands)
    if named:
        return int(named[1])
    if re.fullmatch(r"0x[0-9a-fA-F]+|\d+", operands):  # the encoded form: bits 8 .. 11
        count = int(operands, 0) >> 8 & 15
        return count if count < 15 else None
    return None


def hazards(body: list) -> tuple[int, list]:
    """(LDS reads, instructions that touch a destination still in flight).  LDS
    instructions complete in order among themselves; scalar loads, which share
    their counter out of order, are taken to be done first."""
    at = {label: i for i, (label, _, _) in enumerate(body) if label}
    seen, todo, found, reads = set(), [(0, ())], set(), set()
    while todo:
        i, queue = todo.pop()
        while i < len(body):
            if (i, queue) in seen:
                break
            label, op, operands = body[i]
            if label or op.startswith("s_cbranch") or op == "s_branch":
                seen.add((i, queue))  # states meet at labels and branches only
            if label:
                i += 1
                continue
            if op == "s_endpgm":
                break
            if op == "s_branch":
                i = at[operands]
                continue
            if op.startswith("s_cbranch"):
                todo.append((at[operands], queue))
            elif op == "s_waitcnt":
                count = lgkmcnt(operands)
                if count is not None:
                    queue = queue[len(queue) - count:] if count < len(queue) else queue
            else:
                if queue and registers(operands) & frozenset().union(*queue):
                    found.add((i, op + " " + operands))
                if op.startswith("ds_"):
                    is_read = op.startswith("ds_read")
                    reads.update({i} if is_read else ())
                    queue += (registers(operands.split(",")[0]) if is_read else frozenset(),)
            i += 1
    return len(reads), sorted(found)


LOOP = """
_Zkernel:
  ds_read_b128 v[0:3], v9
  ds_read_b128 v[12:15], v9
.LBB0_1:
  {first}
  s_waitcnt lgkmcnt({wait})
  v_mfma_f32_32x32x16_f16 a[0:15], v[0:3], v[4:7], a[0:15]
  s_waitcnt 0xc07f
  ds_read_b128 v[0:3], v9
  ds_read_b128 v[12:15], v9
  {after}
  s_cbranch_scc1 .LBB0_1
  s_endpgm
"""


@pytest.mark.parametrize("first,wait,after,count", [
    ("s_nop 0", 1, "v_add_u32_e32 v8, v9, v8", 0),
    ("s_load_dword s0, s[2:3], 0x0", 1, "s_nop 0", 0),
    ("s_nop 0", 2, "s_nop 0", 1),                          # one read short
    ("ds_write_b32 v9, v8", 2, "s_nop 0", 0),
    ("s_nop 0", 1, "v_add_u32_e32 v8, v2, v8", 1),         # a value not there yet
    ("v_mov_b32_e32 v3, 0", 1, "s_nop 0", 1),              # overwritten by the landing read
    ("s_nop 0", 1, "scratch_store_dword off, v14, s0", 1),  # spilled too early
    ("v_accvgpr_write_b32 a0, v13", 1, "s_nop 0", 1),      # copied too early, round the loop
])
def test_scan_finds_planted_mistakes(first, wait, after, count):
    reads, found = hazards(parse(LOOP.format(first=first, wait=wait, after=after))["_Zkernel"])
    assert reads == 4 and len(found) == count, found


def test_no_lds_read_destination_is_touched_in_flight(tmp_path):
    out = tmp_path / "mlp_gemm.s"
    subprocess.run([_build.hipcc(), *_build.HIPCC_FLAGS, "--cuda-device-only", "-S",
                    str(_build.CSRC / "mlp_gemm.hip"), "-o", str(out)], check=True,
                   capture_output=True)
    total = 0
    for name, body in parse(out.read_text()).items():
        reads, found = hazards(body)
        total += reads
        assert not found, (name, found[:5])
    assert total > 1000  # the fragment reads of every kernel were seen
