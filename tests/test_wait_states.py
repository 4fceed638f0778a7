"""Wait states that gfx950 wants and the compiler does not add inside inline assembly, read from the
built library's own disassembly (no GPU): one between a scalar write of M0 and the LDS-DMA load that
takes its LDS address from it, and five between a vector instruction's write of a scalar register
and a vector-memory instruction that reads it."""

import os
import re
import subprocess

import pytest

from decentrik_prime_amd import _lib

OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")
VMEM = re.compile(r"(global|buffer|flat|scratch)_")
LDS_DMA = re.compile(r"(global|buffer)_load_lds_|(global|buffer)_load\w* .*\blds\b")


def _scalars(token):
    """The scalar registers a token of the disassembly names."""
    m = re.fullmatch(r"s\[(\d+):(\d+)\]", token)
    if m:
        return {f"s{i}" for i in range(int(m[1]), int(m[2]) + 1)}
    return {token} if re.fullmatch(r"s\d+|vcc", token) else set()


def _split(text):
    op, _, rest = text.partition(" ")
    return op, [t for t in re.split(r",(?![^\[]*\])| ", rest) if t]


def _valu_writes(op, args):
    """Scalar registers a vector instruction writes."""
    if op.startswith(("v_readfirstlane", "v_readlane", "v_cmp")):
        return _scalars(args[0])
    if "_co_" in op or "div_scale" in op:
        return _scalars(args[1])
    return set()


def findings(listing):
    """(function, rule, instruction) per violation in an llvm-objdump listing, and the LDS-DMA loads
    seen.  Straight-line order: the wait states between two instructions are those listed between
    them (s_nop n counts n + 1)."""
    out, dma, name, before = [], 0, None, []
    for line in listing.splitlines():
        m = re.match(r"[0-9a-f]+ <(.*)>:", line)
        if m:
            name, before = m[1], []
            continue
        text = line.split("//")[0].strip()
        if not text:
            continue
        op, args = _split(text)
        if VMEM.match(op):
            is_dma = bool(LDS_DMA.match(text))
            dma += is_dma
            used = set().union(*(_scalars(a) for a in args)) if args else set()
            states = 0
            for o, a in reversed(before):
                if is_dma and states < 1 and o.startswith("s_") and a[:1] == ["m0"]:
                    out.append((name, "M0", text))
                if states < 5 and o.startswith("v_") and _valu_writes(o, a) & used:
                    out.append((name, "SGPR", text))
                states += int(a[0]) + 1 if o == "s_nop" else 1
                if states >= 5:
                    break
        before = (before + [(op, args)])[-8:]
    return out, dma


def test_the_reader_finds_both():
    head = "0000 <k>:\n"
    load = "\tglobal_load_lds_dwordx4 v1, s[4:5] // 0\n"
    mov = "\ts_mov_b32 m0, s2 // 0\n"
    assert findings(head + mov + load) == ([("k", "M0", load.split(" //")[0].strip())], 1)
    assert findings(head + mov + "\ts_nop 0\n" + load) == ([], 1)
    lane = "\tv_readfirstlane_b32 s5, v3\n"
    assert [f[1] for f in findings(head + lane + "\ts_nop 3\n" + load)[0]] == ["SGPR"]
    assert findings(head + lane + "\ts_nop 4\n" + load) == ([], 1)


def test_library_keeps_the_wait_states(tmp_path):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    lib = tmp_path / "lib.so"
    lib.symlink_to(_lib.LIB_PATH)
    subprocess.run([OBJDUMP, "--offloading", str(lib)], check=True, capture_output=True, cwd=tmp_path)
    objects = sorted(tmp_path.glob("*gfx950"))
    assert objects, "no gfx950 code objects in the library"
    bad, loads = [], 0
    for obj in objects:
        res = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(obj)], check=True,
                             capture_output=True, text=True)
        found, dma = findings(res.stdout)
        bad += found
        loads += dma
    assert loads > 0, "no LDS-DMA load found"
    assert not bad, f"{len(bad)} of {loads} loads, e.g. {bad[:3]}"
