"""Every LDS stage a wave reads was waited for by the waves that filled it.

The LDS-DMA tile kernels hand a stage to the other waves of the workgroup with
a counted wait (vmcnt) and a barrier.  The count is right only if the loads it
counts are really issued, which is a matter of the compiled code: a load whose
value is never used is deleted.  So the built code is replayed here, on the
CPU: along every path through a kernel, the vector memory operations in issue
order, the waits (they complete in order) and the barriers.  A wave's DMAs fill
one K step's stage after the other, `per_stage` of them each, and barrier k
stands in front of the reads of step k's stage.  gemm_pipe_kernel promises more:
barrier k hands over the stage of step k + 1 (`lead` = 1).
"""

from __future__ import annotations

import re
import shutil
import subprocess
from pathlib import Path

import pytest

from pageserve_amd import _native

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
VMEM = re.compile(r"(buffer|global|flat)_(load|store|atomic)")
ENDS = ("s_endpgm", "s_branch", "s_setpc_b64")


def kernels(lib: Path, tmp: Path) -> dict[str, list[tuple[str, str]]]:
    """Demangled kernel name -> its instructions and labels of the tile GEMMs."""
    so = tmp / "lib.so"
    shutil.copyfile(lib, so)
    subprocess.run([OBJDUMP, "--offloading", str(so)], cwd=tmp, check=True, capture_output=True)
    found: dict[str, list[tuple[str, str]]] = {}
    for obj in sorted(tmp.glob("lib.so.*gfx950*")):
        out = subprocess.run([OBJDUMP, "-d", "--symbolize-operands", "--demangle", "--no-show-raw-insn", str(obj)],
                             check=True, capture_output=True, text=True).stdout
        body = None
        for line in out.splitlines():
            label = re.match(r"(?:[0-9a-f]+ )?<(.*)>:$", line.strip())
            if label and re.fullmatch(r"L\d+", label[1]):
                if body is not None:
                    body.append(("label", label[1]))
            elif label:
                name = re.search(r"(gemm_(?:dma|pipe|once)_kernel<[^>]*>)", label[1])
                body = found.setdefault(name[1], []) if name else None
            elif body is not None and line.startswith("\t"):
                op, _, args = line.split("//")[0].strip().partition(" ")
                body.append((op, args.strip()))
    return found


def events(code):
    """The instructions that matter, and where each jump goes.  Of the waits
    only those written in front of a barrier: the ones the compiler adds for a
    wave's own operands are not what a stage's hand-over may rest on."""
    ev, labels = [], {}
    for at, (op, args) in enumerate(code):
        if op == "label":
            labels[args] = len(ev)
        elif VMEM.match(op):
            ev.append(("dma" if re.search(r"\blds\b", args) else "vmem", None))
        elif op == "s_waitcnt" and (n := re.search(r"vmcnt\((\d+)\)", args)):
            if next(o for o, _ in code[at + 1:] if o != "s_waitcnt") == "s_barrier":
                ev.append(("wait", int(n[1])))
        elif op == "s_barrier":
            ev.append(("barrier", None))
        elif op.startswith("s_cbranch") or op in ENDS:
            ev.append((op, args or None))
    return ev, labels


def uncovered(code, per_stage: int, closing: int, lead: int = 0) -> set[tuple[int, int]]:
    """(event, missing DMAs) of barriers that hand over a stage some of whose
    DMAs may be in flight.  The state of a path: the operations in flight in
    issue order, the DMAs landed beyond those of the stages handed over, and
    the barriers that left some missing, each with how many more barriers show
    that the step it should have served followed (the path ends with `closing`
    barriers that hand over no stage)."""
    ev, labels = events(code)
    bad, seen, todo = set(), set(), [(0, (), -lead * per_stage, ())]
    while todo:
        state = todo.pop()
        if state in seen:
            continue
        seen.add(state)
        at, flight, ahead, short = state
        kind, arg = ev[at]
        if kind in ("dma", "vmem"):
            flight += (kind,)
        elif kind == "wait":
            landed = flight[:max(0, len(flight) - arg)]
            ahead += landed.count("dma")
            flight = flight[len(landed):]
        elif kind == "barrier":
            bad.update(s[:2] for s in short if s[2] == 1)
            ahead -= per_stage
            short = tuple((a, n, left - 1) for a, n, left in short if left > 1)
            if ahead < 0:
                short += ((at, -ahead, closing + lead + 1),)
        if kind == "s_endpgm":
            continue
        if arg in labels:
            todo.append((labels[arg], flight, ahead, short))
        if kind not in ENDS:
            todo.append((at + 1, flight, ahead, short))
    return bad


@pytest.fixture(scope="module")
def tile_kernels(native_lib, tmp_path_factory):
    if not Path(OBJDUMP).exists():
        pytest.skip("no disassembler")
    return kernels(Path(_native.LIB_PATH), tmp_path_factory.mktemp("isa"))


def test_stages_are_waited_for(tile_kernels):
    """Every remainder length of the unrolled K loop, the loop entered or not."""
    faults, count = {}, {"dma": 0, "pipe": 0}
    for name, code in tile_kernels.items():
        kind, args = re.match(r"gemm_(\w+)_kernel<(.*)>", name).groups()
        if kind not in count:
            continue
        count[kind] += 1
        p = [int(v) for v in re.findall(r"\d+", args)]
        bm, kg = p[0], p[-1] if kind == "dma" else p[3]
        waves = 4 if kind == "dma" else p[4]
        # (two K groups exchange their sums in two halves, two barriers each)
        bad = uncovered(code, bm * 8 // (64 * waves), 4 if kg == 2 else 0, lead=kind == "pipe")
        if bad:
            faults[name] = sorted(bad)
    assert count == {"dma": 8, "pipe": 7}, count
    assert not faults, faults


def test_one_shot_tile_is_waited_for(tile_kernels):
    """gemm_once_kernel: none of a wave's DMAs is in flight at the first barrier."""
    names = [n for n in tile_kernels if "once" in n]
    assert len(names) == 12, names
    for name in names:
        ev, labels = events(tile_kernels[name])
        seen, todo, reached = set(), [(0, ())], 0
        while todo:
            state = todo.pop()
            if state in seen:
                continue
            seen.add(state)
            at, flight = state
            kind, arg = ev[at]
            if kind in ("dma", "vmem"):
                flight += (kind,)
            elif kind == "wait":
                flight = flight[max(0, len(flight) - arg):]
            elif kind == "barrier":
                assert "dma" not in flight, (name, flight)
                reached += 1
                continue
            if arg in labels:
                todo.append((labels[arg], flight))
            if kind not in ENDS:
                todo.append((at + 1, flight))
        assert reached, name
