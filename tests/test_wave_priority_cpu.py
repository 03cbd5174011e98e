"""The gradient wave of the role-split dk/dv form polls for what the score wave on the same SIMD publishes: it must not do so
at the raised issue priority of the matrix phases.  Read from the built code object: the priorities that can reach an
s_sleep (the polls are the only ones) along any path of a kernel."""
import re
import subprocess
from collections import deque
from pathlib import Path

import pytest

from flash_mi355 import build

LLVM = Path("/opt/rocm/llvm/bin")
OBJ = build.OBJ_DIR / "fa_bwd_dkdv.o"
LINE = re.compile(r"^\t(\S+)\s*([^/]*?)\s*// ([0-9A-F]+):")


def _kernels(tmp_path):
    fat, co = tmp_path / "fat.bin", tmp_path / "k.co"
    subprocess.run([LLVM / "llvm-objcopy", "--dump-section", f".hip_fatbin={fat}", OBJ, "/dev/null"], check=True)
    subprocess.run([LLVM / "clang-offload-bundler", "--unbundle", "--type=o", "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", f"--input={fat}",
                    f"--output={co}"], check=True)
    text = subprocess.run([LLVM / "llvm-objdump", "-d", "--no-show-raw-insn", co], check=True, capture_output=True, text=True).stdout
    code = None
    for line in text.splitlines():
        if line.endswith(">:"):
            if code:
                yield name, code
            name, code = line.split("<")[1][:-2], []
        elif code is not None and (m := LINE.match(line)):
            code.append((int(m[3], 16), m[1], m[2]))
    if code:
        yield name, code


def _priorities_at_sleep(code):
    """For every s_sleep the issue priorities it can be reached with (a kernel starts at 0)."""
    at = {a: i for i, (a, _, _) in enumerate(code)}
    seen, todo, found = set(), deque([(0, 0)]), {}
    while todo:
        i, prio = todo.popleft()
        while i < len(code) and (i, prio) not in seen:
            seen.add((i, prio))
            addr, op, arg = code[i]
            assert op not in ("s_setpc_b64", "s_swappc_b64")   # no calls: all paths are in the listing
            if op == "s_setprio":
                prio = int(arg, 0)
            elif op == "s_sleep":
                found.setdefault(addr, set()).add(prio)
            if op == "s_endpgm":
                break
            if op == "s_branch" or op.startswith("s_cbranch"):
                off = int(arg, 0)
                to = at[addr + 4 + 4 * (off - 65536 if off > 32767 else off)]
                if op == "s_branch":
                    i = to
                    continue
                todo.append((to, prio))
            i += 1
    return found


def test_the_pair_is_polled_at_the_lowest_priority(tmp_path):
    if not OBJ.exists() or not (LLVM / "llvm-objdump").exists():
        pytest.skip("needs the objects of a build and the LLVM tools")
    kernels = polled = 0
    for name, code in _kernels(tmp_path):
        found = _priorities_at_sleep(code)
        assert all(p == {0} for p in found.values()), (name, found)
        assert len(found) == sum(op == "s_sleep" for _, op, _ in code), name   # (every poll was reached)
        kernels += any(op == "s_setprio" and arg == "1" for _, op, arg in code)
        polled += bool(found)
    assert kernels > polled > 0
