"""The built library's kernels keep the wait states that the compiler does not
check inside inline assembly (`gemm_tile.h`'s LDS copies): on gfx950 a
vector-memory instruction may read a scalar register only five wait states
after a vector instruction wrote it. Every kernel's assembly is read from the
library as built here; no GPU is needed."""

import collections
import os
import re
import subprocess

import pytest

OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")
WAIT = 5  # between a vector write of a scalar register and a vector-memory read


def _sregs(arg):
    """Numbers of the scalar registers that an operand names (vcc: -1)."""
    m = re.fullmatch(r"s\[(\d+):(\d+)\]", arg)
    if m:
        return set(range(int(m[1]), int(m[2]) + 1))
    m = re.fullmatch(r"s(\d+)", arg)
    return {int(m[1])} if m else ({-1} if arg.startswith("vcc") else set())


def _violations(lines):
    """(kernel, instruction, earlier write, wait states) of every vector-memory
    read of a scalar register too soon after its vector write. Instructions
    are taken in the order of the text."""
    kernel, found, recent = None, [], collections.deque(maxlen=WAIT)
    for line in lines:
        m = re.match(r"[0-9a-f]+ <(.+)>:", line)
        if m:
            kernel = m[1]
            recent.clear()
            continue
        text = line.split("//")[0].strip()
        if not line.startswith("\t") or not text:
            continue
        op, _, rest = text.partition(" ")
        args = [a for a in re.split(r"[ ,]+", rest) if a]
        if op.startswith(("global_", "buffer_", "flat_", "scratch_")):
            use, waits = set().union(*map(_sregs, args)) if args else set(), 0
            for earlier, written, states in reversed(recent):
                if waits >= WAIT:
                    break
                if written & use:
                    found.append((kernel, text, earlier, waits))
                waits += states
        written = set().union(*map(_sregs, args[:2] if "_co_" in op or "div_scale" in op else args[:1])) \
            if op.startswith("v_") and args else set()
        recent.append((text, written, int(args[0], 0) + 1 if op == "s_nop" else 1))
    return found


def test_assembly_that_writes_m0_says_so():
    """The compiler keeps its own values in M0 (LDS copies, indexed moves) and
    reads nothing in an assembly text: the clobber list has to name it."""
    from qmoe import build

    checked = 0
    for name in sorted(os.listdir(build.CSRC)):
        with open(os.path.join(build.CSRC, name)) as f:
            for stmt in re.findall(r"\basm\b[^;]*;", f.read()):
                if re.search(r"s_mov_b32 m0", stmt):
                    checked += 1
                    assert re.search(r':[^:]*"m0"[^:]*\)\s*;$', stmt), f"{name}: {stmt}"
    assert checked >= 3


def test_scan_finds_a_short_wait():
    """The scan itself, on text with and without the wait states."""
    k = ["0000 <k>:", "\tv_readfirstlane_b32 s2, v1 // 00: 00"]
    copy = ["\ts_mov_b32 m0, s9", "\ts_nop 0", "\tglobal_load_lds_dwordx4 v0, s[2:3] // 10: 00"]
    assert [v[3] for v in _violations(k + copy)] == [2]
    assert not _violations(k + ["\ts_nop 2"] + copy)
    assert not _violations([k[0], "\ts_mov_b32 s2, s5"] + copy)
    assert not _violations(["0000 <k>:", "\tv_readfirstlane_b32 s4, v1"] + copy)


@pytest.fixture(scope="module")
def disassembly(tmp_path_factory):
    from qmoe import build

    d = tmp_path_factory.mktemp("code")
    lib = d / "libqmoe.so"
    lib.symlink_to(build.LIB)
    subprocess.run([OBJDUMP, "--offloading", str(lib)], check=True, capture_output=True)
    objs = sorted(d.glob("*gfx950"))
    assert len(objs) >= 8
    return [subprocess.Popen([OBJDUMP, "-d", "--no-show-raw-insn", str(o)], stdout=subprocess.PIPE, text=True)
            for o in objs]


def test_scalar_operands_of_memory_instructions(disassembly):
    found, kernels = [], 0
    for proc in disassembly:
        def lines():
            nonlocal kernels
            for line in proc.stdout:
                kernels += bool(re.match(r"[0-9a-f]+ <.*kernel", line))
                yield line
        found += _violations(lines())
        assert proc.wait() == 0
    assert kernels > 100
    assert not found, f"{len(found)} in {sorted({f[0] for f in found})}, first {found[:2]}"
