"""CPU: the LDS that every batch kernel declares, as the built gfx950 code says it, against what plan_batch sets aside for it (kStatic* in ws_abi.hip). A plan may
fill the compute unit to the last byte, so a kernel that outgrows its share would be refused at the launch, and at the largest shapes only."""
import os
import re
import shutil
import subprocess

import pytest

import wo
from test_meeting_order import LIB, code_objects

READELF = shutil.which("llvm-readelf") or "/opt/rocm/llvm/bin/llvm-readelf"
BUDGETS = {"sample_batch_kernel": "kStaticLds", "lean_batch_kernel": "kStaticLean", "code_batch_kernel": "kStaticCode", "short_batch_kernel": "kStaticShort",
           "short_rest_kernel": "kStaticShort", "twin_batch_kernel": "kStaticTwin", "few_batch_kernel": "kStaticFew", "few_own_kernel": "kStaticFew"}


def test_kernels_fit_what_is_set_aside_for_them(tmp_path):
    if not os.path.exists(READELF):
        pytest.skip("no llvm-readelf")
    with open(os.path.join(wo.ROOT, "whirl-llm_amd", "csrc", "ws_abi.hip")) as f:
        text = re.sub(r"#ifdef WS_PHASE_TIMERS\n.*?#else\n", "", f.read(), flags=re.S)  # (the builds that are timed inside have room of their own)
    room = {name: int(value) for name, value in re.findall(r"constexpr uint32_t (kStatic\w+) = (\d+)u;", text)}
    seen = dict.fromkeys(BUDGETS, 0)
    for i, blob in enumerate(code_objects(LIB)):
        path = tmp_path / f"{i}.elf"
        path.write_bytes(blob)
        notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        for lds, name in re.findall(r"\.group_segment_fixed_size: (\d+).*?\.name: +(\S+)", notes, re.S):
            for kernel, budget in BUDGETS.items():
                if kernel in name:
                    seen[kernel] += 1
                    assert int(lds) <= room[budget], (name, lds, budget, room[budget])
    assert all(seen.values()), seen
