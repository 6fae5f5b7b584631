"""The built library's gfx950 code keeps the wait states that inline assembly
has to keep by itself: the compiler inserts them between its own instructions
only."""
import glob
import os
import re
import shutil
import subprocess

import pytest

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


def kernels(tmp_path):
    """(symbol, [instruction, ...]) of every straight run of the library's device code."""
    from gopherllm_amd import _lib
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    assert os.path.exists(_lib.LIB_PATH), "libgllm_hip.so is not built (run __graft_entry__.build())"
    shutil.copy(_lib.LIB_PATH, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=tmp_path, check=True, capture_output=True)
    objects = sorted(glob.glob(str(tmp_path / "*gfx950")))
    assert objects
    for obj in objects:
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", obj], check=True, capture_output=True,
                              text=True).stdout
        name, code = "", []
        for line in text.splitlines():
            m = re.match(r"[0-9a-f]+ <(\S+)>:", line)
            if m:
                yield name, code
                name, code = m.group(1), []
            elif line.startswith("\t"):
                code.append(line.split("//")[0].strip())
        yield name, code


def wait_states(ins):
    return int(ins.split()[1], 0) + 1 if ins.startswith("s_nop") else 1


def sgprs(operand):
    m = re.fullmatch(r"s(\d+)|s\[(\d+):(\d+)\]", operand)
    if not m:
        return set()
    lo = int(m.group(1) or m.group(2))
    return set(range(lo, int(m.group(3) or lo) + 1))


def test_loads_to_lds_keep_their_wait_states(tmp_path):
    """One between a scalar write of M0 and the load to LDS that reads it, five
    between a vector instruction's SGPR result and the load that takes it as
    its base address."""
    seen, wrong = 0, []
    for name, code in kernels(tmp_path):
        for i, ins in enumerate(code):
            if not ins.startswith("global_load_lds"):
                continue
            seen += 1
            base = set().union(*(sgprs(o) for o in re.split(r"[ ,]+", ins)[1:]))
            states = 0
            for before in reversed(code[max(0, i - 5):i]):
                ops = re.split(r"[ ,]+", before)
                if ops[0].startswith("s_") and ops[1:2] == ["m0"] and states < 1:
                    wrong.append((name, before, ins))
                if ops[0].startswith("v_") and states < 5 and any(sgprs(o) & base for o in ops[1:3]):
                    # the second operand counts for the carry-outs alone
                    if sgprs(ops[1]) & base or "_co_" in ops[0]:
                        wrong.append((name, before, ins))
                states += wait_states(before)
    assert seen, "no load to LDS in the library"
    assert not wrong, wrong[:5]
