"""The gfx950 code of the built library (no GPU call): what the kernels' cooperating wavefronts
need of the compiler, read from the disassembly of libf16hip.so.

  * The step kernels' state and output pointers are global ones: a flat access counts as an LDS
    access too, so every workgroup barrier and LDS read after a flat store waits for that store.
  * No barrier in a loop that lanes leave one by one.  Every wavefront of a workgroup has to meet
    each barrier the same number of times; a loop that the compiler has split by a per-lane
    condition (for instance "this lane stores") would send part of a wavefront through it again.
"""
import os
import re
import shutil
import subprocess

import pytest

from conftest import import_pkg

OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")
_INSN = re.compile(r"^\t(\S+)\s*(.*?)\s*// ([0-9A-F]+):")
_TARGET = re.compile(r"<[^>+]+(?:\+0x([0-9a-f]+))?>\s*$")


def disassemble(lib, folder):
    """{kernel symbol: [(offset, mnemonic, operands, branch target offset or None)]}."""
    shutil.copy(lib, os.path.join(folder, "lib.so"))
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=folder, check=True,
                   stdout=subprocess.DEVNULL)
    kernels = {}
    for name in sorted(os.listdir(folder)):
        if not name.endswith("gfx950"):
            continue
        text = subprocess.run([OBJDUMP, "-d", name], cwd=folder, check=True, capture_output=True,
                              text=True).stdout
        code = None
        for line in text.split("\n"):
            head = re.match(r"^([0-9a-f]+) <(\S+)>:", line)
            if head:
                base, code = int(head.group(1), 16), kernels.setdefault(head.group(2), [])
                continue
            insn = _INSN.match(line)
            if insn and code is not None:
                op, args, addr = insn.groups()
                target = None
                if op.startswith(("s_cbranch", "s_branch")):
                    target = int(_TARGET.search(line).group(1) or "0", 16)
                code.append((int(addr, 16) - base, op, args, target))
    return kernels


def masked_barrier_loops(code):
    """Offsets of the latches (exec &= ~left, then a branch on exec) of loops that hold a barrier."""
    at = {c[0]: i for i, c in enumerate(code)}
    starts = {0} | {at[c[3]] for c in code if c[3] is not None}
    starts |= {i + 1 for i, c in enumerate(code[:-1])
               if c[1].startswith(("s_cbranch", "s_branch", "s_endpgm"))}
    starts = sorted(starts)
    number = {s: b for b, s in enumerate(starts)}
    blocks = list(zip(starts, starts[1:] + [len(code)]))
    succ = []
    for b, (lo, hi) in enumerate(blocks):
        _, op, _, target = code[hi - 1]
        out = [] if target is None else [number[at[target]]]
        if not op.startswith(("s_branch", "s_endpgm")) and b + 1 < len(blocks):
            out.append(b + 1)
        succ.append(out)
    pred = [[] for _ in blocks]
    for b, out in enumerate(succ):
        for s in out:
            pred[s].append(b)
    holds = [any(c[1] == "s_barrier" for c in code[lo:hi]) for lo, hi in blocks]
    found = []
    for b, (lo, hi) in enumerate(blocks):
        tail = code[max(lo, hi - 4):hi]
        if not (tail[-1][1].startswith("s_cbranch_exec") and
                any(c[1] == "s_andn2_b64" and c[2].startswith("exec, exec") for c in tail)):
            continue
        for header in succ[b]:
            # the natural loop of the edge b -> header, if the header dominates b
            loop, work = {header, b}, [b] if b != header else []
            while work:
                for p in pred[work.pop()]:
                    if p not in loop:
                        loop.add(p)
                        work.append(p)
            if (0 not in loop or header == 0) and any(holds[x] for x in loop):
                found.append(hex(code[lo][0]))
    return found


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    if not os.path.exists(OBJDUMP):
        pytest.skip("llvm-objdump not available")
    return disassemble(import_pkg("_lib").LIB_PATH, str(tmp_path_factory.mktemp("device_code")))


def test_step_kernels_have_no_flat_accesses(kernels):
    steps = {k: code for k, code in kernels.items()
             if "fdm_step_quad_kernel" in k or "env_step_quad_kernel" in k}
    assert len(steps) == 24              # fp64 and fp32 steps, and the one-launch env steps
    flat = {k: n for k, code in steps.items()
            if (n := sum(c[1].startswith("flat_") for c in code))}
    assert flat == {}


def test_no_barrier_in_a_lane_masked_loop(kernels):
    barriers = [k for k, code in kernels.items() if any(c[1] == "s_barrier" for c in code)]
    assert len(barriers) > 20
    bad = {k: f for k in barriers if (f := masked_barrier_loops(kernels[k]))}
    assert bad == {}
