"""The built code of the register-staged small encode tiles (csrc/encode_slim.h): each K-step waits for
its x' by count (s_waitcnt vmcnt), which is right only while the step's x' DMAs are issued before its W
loads and no W load slips behind the next step's wait. No test on a GPU shows a wrong order reliably, so
the order is read from the objects that the library was linked from."""

import re
import subprocess
from pathlib import Path

import pytest

from saeflow_amd import build

LLVM = Path("/opt/rocm/llvm/bin")
OBJECTS = {dt: build.BUILD / f"encode_slim_reg_{dt}.o" for dt in ("f32", "bf16", "f16")}


def instructions(obj, tmp):
    """{kernel: [(address, mnemonic and operands, branch target or None)]} of an object's gfx950 code."""
    fat, code = tmp / "fat", tmp / "code"
    run = lambda *cmd: subprocess.run([str(c) for c in cmd], check=True, capture_output=True, text=True).stdout  # noqa: E731
    run(LLVM / "llvm-objcopy", f"--dump-section=.hip_fatbin={fat}", obj, tmp / "unused.o")
    run(LLVM / "clang-offload-bundler", "--type=o", "--unbundle", f"--input={fat}", f"--output={code}",
        f"--targets=hipv4-amdgcn-amd-amdhsa--{build.ARCH}")
    kernels, cur = {}, None
    for line in run(LLVM / "llvm-objdump", "-d", "--no-show-raw-insn", code).splitlines():
        if m := re.match(r"([0-9a-f]+) <(\w+)>:", line):
            base, cur = int(m[1], 16), kernels.setdefault(m[2], [])
        elif cur is not None and (m := re.match(r"\t(.*?)\s*// ([0-9A-F]{12}):", line)):
            to = re.search(r"\+0x([0-9a-f]+)>", line) if "branch" in m[1] else None
            cur.append((int(m[2], 16), m[1], base + int(to[1], 16) if to else None))
    return kernels


def misplaced(code):
    """W loads that, on some way through the code, come ahead of a DMA of their step (the stretch between
    two barriers) or ahead of the step's wait. The prologue before the first barrier waits for all."""
    at = {a: i for i, (a, _, _) in enumerate(code)}
    bad, seen, todo = set(), set(), [(0, "prologue")]
    while todo:
        i, state = todo.pop()
        if i >= len(code) or (i, state) in seen:
            continue
        seen.add((i, state))
        addr, ins, to = code[i]
        if ins.startswith("s_barrier"):
            state = "entered"
        elif "vmcnt" in ins:
            state = "waited" if state == "entered" else state
        elif re.match(r"buffer_load_dword\S* .*\blds\b", ins):
            bad |= {(hex(addr), ins)} if state == "loaded" else set()
        elif ins.startswith("global_load"):
            bad |= {(hex(addr), ins)} if state == "entered" else set()
            state = "loaded" if state == "waited" else state
        if to is not None:
            todo.append((at[to], state))
        if not ins.startswith(("s_branch", "s_endpgm")):
            todo.append((i + 1, state))
    return sorted(bad)


@pytest.mark.skipif(not (LLVM / "llvm-objdump").exists(), reason="no llvm-objdump")
@pytest.mark.parametrize("dt", list(OBJECTS))
def test_dma_before_w_loads(dt, tmp_path):
    if not OBJECTS[dt].exists():
        pytest.skip("no objects beside the built library")
    kernels = {k: v for k, v in instructions(OBJECTS[dt], tmp_path).items() if "gemm_slim_kernel" in k}
    assert len(kernels) >= 8
    for name, code in kernels.items():
        assert sum(ins.startswith("s_barrier") for _, ins, _ in code) >= 6, name
        assert any(re.match(r"buffer_load_dword\S* .*\blds\b", ins) for _, ins, _ in code), name
        assert misplaced(code) == [], name


def test_a_wrong_order_is_found():
    wait, bar = "s_waitcnt vmcnt(4)", "s_barrier"
    dma, load = "buffer_load_dwordx4 v1, s[0:3], 0 offen lds", "global_load_dwordx4 v[0:3], v[4:5], off"
    code = lambda *ins: [(4 * i, s, None) for i, s in enumerate(ins)]  # noqa: E731
    assert misplaced(code(bar, wait, dma, dma, load, bar, wait, dma, load)) == []
    assert len(misplaced(code(bar, wait, dma, load, dma))) == 1
    assert len(misplaced(code(bar, wait, dma, bar, load, wait))) == 1
