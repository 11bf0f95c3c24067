"""The instructions of the built kernels, where correctness rests on something the compiler
does not check: it handles neither the hazards nor the outstanding loads of inline assembly.
Runs on the CPU, on the gfx950 code of lib/libqxg.so."""
import os
import re
import shutil
import subprocess
from collections import namedtuple

import pytest

import qxg

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
Ins = namedtuple("Ins", "at op args text")   # address, mnemonic, operands


@pytest.fixture(scope="module")
def listing(tmp_path_factory):
    """{kernel: [Ins, ...]} of every kernel of the library."""
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
            elif name and line.startswith("\t") and "//" in line:   # (not the "..." of a run of zeros)
                code, at = line.split("//")
                op, _, rest = code.strip().partition(" ")
                kernels[name].append(Ins(int(at.split(":")[0], 16), op, [a.strip() for a in rest.split(",")] if rest else [], code.strip()))
    assert len(kernels) > 40
    return kernels


def _regs(kind, arg):
    """Numbers of the registers of a kind ("v" or "s") that an operand names."""
    m = re.search(rf"\b{kind}\[(\d+):(\d+)\]", arg)
    if m:
        return set(range(int(m.group(1)), int(m.group(2)) + 1))
    m = re.search(rf"\b{kind}(\d+)\b", arg)
    return {int(m.group(1))} if m else set()


def _wait_states(ins):
    return 1 + int(ins.args[0]) if ins.op == "s_nop" else 1


def _recent(code, i, states):
    """(instruction, wait states between it and instruction i) of those fewer than `states` before i."""
    seen = 0
    for before in reversed(code[max(0, i - states):i]):
        if seen >= states:
            return
        yield before, seen
        seen += _wait_states(before)


def test_load_to_lds_hazards(listing):
    """A load-to-LDS instruction comes at least one wait state after the write of M0 it uses, and
    at least five after a vector instruction that wrote a scalar register of its address."""
    copies = 0
    for name, code in listing.items():
        for i, ins in enumerate(code):
            if not ins.op.startswith("global_load_lds"):
                continue
            copies += 1
            base = _regs("s", ins.text)
            for before, states in _recent(code, i, 5):
                dest = before.args[0] if before.args else ""
                assert dest != "m0" or states >= 1, (name, before, ins)
                assert not (before.op.startswith("v_") and _regs("s", dest) & base), (name, before, ins)
    assert copies > 100


def test_dot_hazards(listing):
    """A dot product's result is read or overwritten by another vector opcode, or read as a factor by
    the same, at least three wait states later (v_dot4 and v_dot4c are different opcodes)."""
    dots = 0
    for name, code in listing.items():
        for i, ins in enumerate(code):
            if not ins.op.startswith("v_") or not ins.args:
                continue
            dots += ins.op.startswith("v_dot")
            for before, _ in _recent(code, i, 3):
                if not before.op.startswith("v_dot"):
                    continue
                used = ins.args[1:3] if before.op == ins.op else ins.args
                assert not _regs("v", before.args[0]) & set().union(*(_regs("v", a) for a in used)), (name, before, ins)
    assert dots > 1000


def _flow(code):
    """Indexes of the instructions that may follow each instruction."""
    index = {ins.at: i for i, ins in enumerate(code)}
    follow = []
    for i, ins in enumerate(code):
        after = [] if ins.op in ("s_branch", "s_endpgm") or i + 1 == len(code) else [i + 1]
        if ins.op.startswith(("s_branch", "s_cbranch")):
            off = int(ins.args[0])
            after.append(index[ins.at + 4 + 4 * (off - 0x10000 if off >= 0x8000 else off)])
        follow.append(after)
    return follow


def test_assembly_loads_in_flight(listing):
    """The exchange words' loads (inline assembly; their wait comes later, behind the loads of
    the other words) land in registers that nothing reads or writes before a wait for them."""
    loads = 0
    for name, code in listing.items():
        starts = [i for i, ins in enumerate(code) if ins.op == "global_load_dwordx4" and ins.text.endswith("off sc1")]
        loads += len(starts)
        if not starts:
            continue
        follow = _flow(code)
        flying = [frozenset()] * len(code)   # registers with a load in flight before each instruction
        first, queued, work = set(starts), set(starts), list(starts)
        while work:
            i = work.pop()
            queued.discard(i)
            ins, now = code[i], flying[i]
            if ins.op == "s_waitcnt" and "vmcnt(0)" in ins.text:
                now = frozenset()
            else:
                used = set().union(set(), *(_regs("v", a) for a in ins.args))
                assert not used & now, (name, ins)
                if i in first:
                    now = now | _regs("v", ins.args[0])
            for j in follow[i]:
                if not now <= flying[j]:
                    flying[j] = flying[j] | now
                    if j not in queued:
                        queued.add(j)
                        work.append(j)
    assert loads > 50


def test_gate_up_counted_wait(listing):
    """Gate/up waits for its staged rows by leaving the weights' loads, the youngest, in flight: the
    counted wait in the middle of a block leaves no more than were issued behind the last copy."""
    waits = 0
    for name, code in listing.items():
        if "qxp_gate_up" not in name:
            continue
        for i in (i for i, ins in enumerate(code) if ins.op == "s_barrier"):
            left = since = None   # loads that the barrier's wait leaves in flight; loads since the last copy
            for before in reversed(code[:i]):
                if before.op.startswith(("s_branch", "s_cbranch", "global_load_lds")):
                    break
                m = re.search(r"vmcnt\((\d+)\)", before.text) if before.op == "s_waitcnt" else None
                if m and left is None:
                    left, since = int(m.group(1)), 0
                elif since is not None:
                    since += before.op.startswith(("global_load", "global_store", "buffer_", "flat_"))
            if left:
                waits += 1
                assert before.op.startswith("global_load_lds") and since >= left, (name, left, since, code[i])
    assert waits == 4   # two formats, passes of 16 and of 32 rows
