"""The instructions of the built kernels, where correctness rests on something the compiler
does not check: the load-to-LDS copies are inline assembly, which its hazard handling does
not look into.  Runs on the CPU, on the gfx950 code of lib/libqxg.so."""
import os
import re
import shutil
import subprocess

import pytest

import qxg

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


@pytest.fixture(scope="module")
def listing(tmp_path_factory):
    """{kernel: [instruction, ...]} of every kernel of the library."""
    d = tmp_path_factory.mktemp("listing")
    shutil.copy(os.path.join(qxg.LIB_DIR, "libqxg.so"), d)
    subprocess.run([OBJDUMP, "--offloading", "libqxg.so"], cwd=d, check=True, stdout=subprocess.DEVNULL)
    kernels, name = {}, None
    for f in sorted(d.glob("*gfx950")):
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(f)], check=True, capture_output=True, text=True).stdout
        for line in text.splitlines():
            head = re.match(r"[0-9a-f]+ <(.*)>:", line)
            if head:
                name = head.group(1)
                kernels[name] = []
            elif name and line.startswith("\t"):
                kernels[name].append(line.split("//")[0].strip())
    assert len(kernels) > 40
    return kernels


def _wait_states(ins):
    nop = re.match(r"s_nop (\d+)", ins)
    return 1 + int(nop.group(1)) if nop else 1


def test_load_to_lds_hazards(listing):
    """A load-to-LDS instruction comes at least one wait state after the write of M0 it uses, and
    at least five after a vector instruction that wrote a scalar register of its address."""
    copies = 0
    for name, code in listing.items():
        for i, ins in enumerate(code):
            if not ins.startswith("global_load_lds"):
                continue
            copies += 1
            base = re.search(r"s\[(\d+):(\d+)\]", ins)
            regs = {f"s{r}" for r in range(int(base.group(1)), int(base.group(2)) + 1)} if base else set()
            states = 0
            for before in reversed(code[max(0, i - 6):i]):
                op, _, rest = before.partition(" ")
                dest = rest.split(",")[0]
                assert dest != "m0" or states >= 1, (name, i, before, ins)
                pair = re.match(r"s\[(\d+):(\d+)\]", dest)
                wrote = {f"s{r}" for r in range(int(pair.group(1)), int(pair.group(2)) + 1)} if pair else {dest}
                assert not (op.startswith("v_") and wrote & regs) or states >= 5, (name, i, before, ins)
                states += _wait_states(before)
    assert copies > 100
