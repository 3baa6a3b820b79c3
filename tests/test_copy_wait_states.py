"""The copies from memory into LDS that the cooperative kernels write by hand
(lds_copy16, csrc/kv_decode_mfma.h) keep the wait states that gfx950 asks of
software and that the compiler cannot add inside an asm statement: one between
a scalar write of m0 and the copy reading it, five between a VALU write of an
SGPR and the vector memory instruction whose base it is.  Read from the
disassembly of the library as built here."""
import os
import re
import shutil
import subprocess

import pytest

from knlp_amd import build

OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")
SGPR = re.compile(r"s\[(\d+):(\d+)\]|s(\d+)|(vcc)(?:_lo|_hi)?")


def _sgprs(operand):
    m = SGPR.fullmatch(operand)
    if m is None:
        return set()
    if m[4]:
        return {"vcc"}
    return set(range(int(m[1]), int(m[2]) + 1)) if m[1] else {int(m[3])}


def _written(op, args):
    """SGPRs that an instruction writes: a scalar one's or v_readlane's first
    operand, a compare's, a carry's second operand."""
    if op.startswith(("s_cmp", "s_bitcmp", "s_waitcnt", "s_nop", "s_barrier", "s_store")):
        return set()
    return _sgprs(args[0]) | (_sgprs(args[1]) if op.startswith("v_") and "_co_" in op else set())


def violations(lines):
    """(number of copies, the copies too close to a write of their operands)."""
    copies, bad, recent = 0, [], []
    for line in lines:
        text = line.split("//")[0].strip()
        if line[:1] != "\t":
            recent = []                                  # a label: another function
            continue
        op, _, rest = text.partition(" ")
        args = [a.strip() for a in rest.split(",")]
        if "_load_lds_" in op or (op.startswith("buffer_load") and " lds" in rest):
            copies += 1
            base = set().union(*(_sgprs(a.split(" ")[0]) for a in args))
            states = 0
            for prev, prev_args in reversed(recent):
                if states < 1 and prev.startswith("s_") and prev_args[0] == "m0":
                    bad.append(f"m0 written before {text}")
                written = _written(prev, prev_args)
                if states < 5 and prev.startswith("v_") and written & base:
                    bad.append(f"{prev} {', '.join(prev_args)} before {text}")
                base -= written                          # (only its last writer counts)
                states += 1 + (int(prev_args[0], 0) if prev == "s_nop" else 0)
        recent = recent[-5:] + [(op, args)]
    return copies, bad


def test_checker_sees_both_hazards():
    m0 = ["\ts_mov_b32 m0, s5", "\tglobal_load_lds_dwordx4 v4, s[8:9] nt"]
    assert violations(m0)[1] and not violations([m0[0], "\ts_nop 0", m0[1]])[1]
    base = ["\tv_readfirstlane_b32 s9, v2", "\ts_mov_b32 m0, s5", "\ts_nop 2", m0[1]]
    assert len(violations(base)[1]) == 1
    assert not violations([*base[:2], "\ts_nop 3", m0[1]])[1]


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="llvm-objdump not installed")
def test_hand_written_copies_keep_their_wait_states(tmp_path):
    if not os.path.exists(build.LIB):
        pytest.skip("library not built")
    lib = shutil.copy(build.LIB, tmp_path / "lib.so")        # (extracts beside its input)
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, capture_output=True)
    objects = sorted(p for p in os.listdir(tmp_path) if p.endswith(build.ARCH))
    assert objects
    copies = 0
    for name in objects:
        with subprocess.Popen([OBJDUMP, "-d", "--no-show-raw-insn", tmp_path / name], text=True,
                              stdout=subprocess.PIPE) as p:
            n, bad = violations(p.stdout)
        assert p.returncode == 0
        copies += n
        assert not bad, (len(bad), bad[:4])
    assert copies > 0
