"""CPU: the kernels whose workgroups meet by a ticket - whoever draws the last one reads what all the others have left in the
workspace, clears it and goes on - draw it only when every store before it has arrived. Otherwise a key could come after its place
had been cleared and would stand there for the next launch. Looked up in the built gfx950 code: from the ticket's atomic
addition backwards there has to be the workgroup's barrier, and a wait for all of the wave's stores between that barrier and
the last store to global memory before it."""
import os
import re
import shutil
import struct
import subprocess

import pytest

import wo

LIB = os.path.join(wo.ROOT, "whirl-llm_amd", "libwhirl_sampling_hip.so")
OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"


def code_objects(path):
    """The gfx950 code objects bundled in the library, one a translation unit."""
    with open(path, "rb") as f:
        data = f.read()
    at = data.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        n, p = struct.unpack_from("<Q", data, at + 24)[0], at + 32
        for _ in range(n):
            off, size, length = struct.unpack_from("<QQQ", data, p)
            if b"gfx950" in data[p + 24:p + 24 + length]:
                yield data[at + off:at + off + size]
            p += 24 + length
        at = data.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 24)


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """Instructions of every kernel that draws a ticket, by (mangled) name."""
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    out = {}
    for i, blob in enumerate(code_objects(LIB)):
        path = tmp_path_factory.mktemp("co") / f"{i}.elf"
        path.write_bytes(blob)
        names = re.findall(r"\.text\s+\S+\s+\S*\s*(\S+)$", subprocess.run([OBJDUMP, "-t", str(path)], capture_output=True, text=True, check=True).stdout, re.M)
        names = [n for n in names if re.search(r"few_batch_kernel|few_own_kernel|topk_rows_shared|dflash_topk_shared|draft_sample_rows_shared|spec_verify_kernel|short_batch_kernelILi[01]ELb[01]ELb1E", n) and not n.endswith(".kd")]
        if not names:
            continue
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", f"--disassemble-symbols={','.join(names)}", str(path)], capture_output=True, text=True, check=True).stdout
        for name, body in re.findall(r"^[0-9a-f]+ <(\w+)>:\n(.*?)(?=^[0-9a-f]+ <|\Z)", text, re.M | re.S):
            out[name] = [line.split("//")[0].strip() for line in body.splitlines() if line.strip()]
    return out


def before_the_ticket(code):
    """What stands between the ticket and the last store to global memory before it, nearest first."""
    tickets = [i for i, op in enumerate(code) if op.startswith("global_atomic_add ") and " sc0" in op]
    assert tickets, "no ticket"
    back = []
    for op in reversed(code[:tickets[0]]):
        if re.match(r"(global|flat|buffer)_store", op):
            return back
        back.append(op)
    raise AssertionError("no store before the ticket")


def test_stores_have_arrived_before_the_ticket_is_drawn(kernels):
    # dtype x mask x size of the few-row sampler, and its two for a row that comes with the launch; three kernels of three sizes; the classic verification; the short-list kernel's shared rows
    assert len(kernels) == 16 + 2 + 9 + 1 + 4, sorted(kernels)
    for name, code in kernels.items():
        back = before_the_ticket(code)
        assert "s_barrier" in back, name
        waits = [op for op in back[back.index("s_barrier"):] if op.startswith("s_waitcnt") and "vmcnt(0)" in op]
        assert waits, f"{name}: its stores may still be on their way"


def test_the_kernels_that_may_leave_a_row_wait_as_well(tmp_path):
    """The builds of the lone row's kernel without the three-pass code (few_try_kernel), looked at the same way."""
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    found = 0
    for i, blob in enumerate(code_objects(LIB)):
        path = tmp_path / f"{i}.elf"
        path.write_bytes(blob)
        names = re.findall(r"\.text\s+\S+\s+\S*\s*(\S*few_try_kernel\S*)$", subprocess.run([OBJDUMP, "-t", str(path)], capture_output=True, text=True, check=True).stdout, re.M)
        for name in (n for n in names if not n.endswith(".kd")):
            text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", f"--disassemble-symbols={name}", str(path)], capture_output=True, text=True, check=True).stdout
            back = before_the_ticket([line.split("//")[0].strip() for line in text.splitlines() if line.startswith("\t")])
            assert "s_barrier" in back, name
            assert any(op.startswith("s_waitcnt") and "vmcnt(0)" in op for op in back[back.index("s_barrier"):]), name
            found += 1
    assert found == 2
