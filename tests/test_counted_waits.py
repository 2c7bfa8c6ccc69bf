"""The tile kernels of the grouped GEMMs (gemm.hip, gemm_fp4.hip) wait for the rows in their
LDS ring by counting: "all but the newest n loads have landed".  That holds only while n loads
lie behind the awaited ones, and the compiler drops a register load that nothing reads.  So the
counts are checked against the loads that are in the built library, along every path through
the disassembled kernels, without a GPU."""
import glob
import os
import re
import shutil
import struct
import subprocess

import pytest

from gpt_oss_amd import build

OBJDUMP = shutil.which("llvm-objdump", path="/opt/rocm/llvm/bin:" + os.environ.get("PATH", ""))
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
RING = 4  # LDS stages of steps (down) or double steps (gate_up): a wait reads what RING - 1 barriers ago was asked for
CAP = 64  # vmcnt counts to 63


def gfx950_code_objects(data):
    at = data.find(MAGIC)
    while at >= 0:
        p = at + 32
        for _ in range(struct.unpack_from("<Q", data, at + 24)[0]):
            off, size, n = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + n]
            p += 24 + n
            if size and b"gfx950" in name:
                yield data[at + off:at + off + size]
        at = data.find(MAGIC, at + 24)


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """name -> [(mnemonic, operands, index of a branch's target or None)]"""
    if OBJDUMP is None:
        pytest.skip("no llvm-objdump")
    out = {}
    path = str(tmp_path_factory.mktemp("co") / "co.o")
    for code in gfx950_code_objects(open(build.LIB, "rb").read()):
        if b"gemm_kernel" not in code:
            continue
        with open(path, "wb") as f:
            f.write(code)
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", path], capture_output=True, text=True,
                              check=True).stdout
        for m in re.finditer(r"^([0-9a-f]+) <(\S+)>:\n(.*?)(?=^[0-9a-f]+ <|\Z)", text, re.S | re.M):
            if "grouped_gemm_kernel" not in m[2] and "fp4_gemm_kernel" not in m[2]:
                continue
            rows, addr = [], {}
            for line in m[3].splitlines():
                i = re.match(r"\s+(\S+)(.*?)\s*// ([0-9A-F]+):.*?(?:<\S+?(?:\+0x([0-9a-f]+))?>)?$", line)
                if i:
                    addr[int(i[3], 16)] = len(rows)
                    rows.append((i[1], i[2], int(m[1], 16) + int(i[4] or "0", 16)))
            out[m[2]] = [(op, args, addr.get(to) if "branch" in op else None) for op, args, to in rows]
    assert out, "no tile kernels in the library"
    return out


LOADS = ("global_load", "global_store", "buffer_", "flat_", "scratch_")


def wait_in_front(code, pc):
    """The count of the last s_waitcnt on vector memory in front of instruction pc, with no other load between."""
    while pc > 0 and not code[pc - 1][0].startswith(LOADS) and code[pc - 1][2] is None:
        pc -= 1
        n = re.search(r"vmcnt\((\d+)\)", code[pc][1]) if code[pc][0] == "s_waitcnt" else None
        if n:
            return int(n[1])
    return None


def slack_of_waits(code):
    """{barrier with a ring behind it: (loads behind the rows that have to have landed there, the
    fewest over all paths) - (loads that the wait in front of it leaves in flight)}"""
    # state at an instruction: for 0 .. RING - 1 barriers ago, the loads issued since the last DMA
    # between that barrier and the next, CAP where there is none.  There the DMAs come in front of
    # the register loads; a DMA behind one begins a tile, whose first filling, of several
    # stages at once, is not looked at.
    state, todo, found = {}, [(0, (CAP,) * RING, False, True)], {}
    while todo:
        pc, s, loaded, fill = todo.pop()
        while pc < len(code):
            old = state.get((pc, loaded, fill))
            new = s if old is None else tuple(map(min, s, old))
            if new == old:
                break
            state[pc, loaded, fill] = s = new
            op, args, to = code[pc]
            if op.startswith("global_load_lds"):
                fill = fill or loaded
                s = (CAP,) * RING if fill else (0,) + tuple(min(n + 1, CAP) for n in s[1:])
            elif op.startswith(LOADS):
                s, loaded = tuple(min(n + 1, CAP) for n in s), True
            elif op == "s_barrier":
                if s[RING - 2] < CAP:
                    n = wait_in_front(code, pc)
                    assert n is not None, f"instruction {pc}: a barrier without a wait in front"
                    found[pc] = s[RING - 2] - n
                s, loaded, fill = (CAP,) + s[:-1], False, False
            elif op == "s_endpgm":
                break
            if to is not None:
                todo.append((to, s, loaded, fill))
                if op == "s_branch":
                    break
            pc += 1
    return found


def test_waits_leave_no_awaited_row_in_flight(kernels):
    checked = 0
    for name, code in kernels.items():
        found = slack_of_waits(code)
        assert found, f"{name}: no ring found"
        lax = {pc: s for pc, s in found.items() if s < 0}
        assert not lax, f"{name}: waits that leave awaited rows in flight (instruction: loads too many): {lax}"
        checked += len(found)
    assert checked >= 100


def test_assembly_names_m0_where_it_writes_it():
    """A DMA's LDS address goes into m0: assembly that writes it has to tell the compiler, which may
    hold something of its own there."""
    writes = 0
    for path in sorted(glob.glob(os.path.join(build.CSRC, "*.hip")) + glob.glob(os.path.join(build.CSRC, "*.h"))):
        for m in re.finditer(r"\basm\s+volatile\s*\((.*?)\);", open(path).read(), re.S):
            if re.search(r"s_mov_b32 m0", m[1]):
                writes += 1
                assert '"m0"' in m[1].rsplit(":", 1)[1], f"{os.path.basename(path)}: {m[1]}"
    assert writes
