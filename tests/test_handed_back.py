"""CPU: the three-pass code that other kernels hand rows back to, looked up in the built gfx950 code. Nothing of its caller is wanted behind it, so it must not
begin by putting the caller's registers away: a scalar register that finds no room in a vector register goes to memory by way of one that has to be put
away and fetched again for it, a round trip each."""
import os
import re
import subprocess

import pytest

from test_meeting_order import LIB, OBJDUMP, code_objects


@pytest.fixture(scope="module")
def functions(tmp_path_factory):
    """Instructions of every instance, by (mangled) name and translation unit."""
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    out = {}
    for i, blob in enumerate(code_objects(LIB)):
        path = tmp_path_factory.mktemp("co") / f"{i}.elf"
        path.write_bytes(blob)
        names = re.findall(r"\.text\s+\S+\s+(\S*three_pass_row\S*)$", subprocess.run([OBJDUMP, "-t", str(path)], capture_output=True, text=True, check=True).stdout, re.M)
        for name in names:
            text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", f"--disassemble-symbols={name}", str(path)], capture_output=True, text=True, check=True).stdout
            out[i, name] = [line.split("//")[0].strip() for line in text.splitlines() if line.startswith("\t")]
    return out


def test_no_callers_registers_are_put_away(functions):
    # the lean, the bf16, the short-list (two) and the few-row (two) kernels' own
    assert len(functions) == 6, sorted(functions)
    for name, code in functions.items():
        first = next(i for i, op in enumerate(code) if op.startswith(("s_cbranch", "s_branch", "s_swappc", "s_barrier")))
        round_trips = [op for op in code[:first] if op.startswith("scratch_load")]
        assert len(round_trips) <= 4, (name, len(round_trips))


def test_arguments_are_scalar(functions):
    """What it reads of the kernel's arguments comes by scalar loads: with the argument segment's address in vector registers every one of them, and all that follows
    from it, would be a value of its own in every lane."""
    for name, code in functions.items():
        first = next(i for i, op in enumerate(code) if op.startswith("s_barrier"))
        assert sum(op.startswith("s_load") for op in code[:first]) >= 10, name
        assert sum(op.startswith("scratch_store") for op in code[:first]) <= 24, name
