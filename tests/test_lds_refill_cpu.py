"""Kernels in which a wave streams tiles through LDS of its own have no barrier between the reads of a buffer and the loads that fill
it again: the wave waits for its reads instead.  Read from the built code objects: along no path of such a kernel is a load to
LDS issued while a read or write of LDS is outstanding."""
import re
from collections import deque

import pytest

from flash_mi355 import build
from tests import test_wave_priority_cpu as listing

OBJECTS = {"fa_bwd_small.o": "dkdv_small_kernel", "fa_decode.o": "decode_kernel"}


def _to_lds(op, arg):
    return op.startswith("global_load_lds") or (op.startswith("buffer_load") and arg.split()[-1] == "lds")


def refills_behind_open_reads(code):
    """Addresses of the loads to LDS that can be reached with an LDS access in flight (they complete in order)."""
    at = {a: i for i, (a, _, _) in enumerate(code)}
    seen, todo, found = set(), deque([(0, ())]), set()
    while todo:
        i, open_ = todo.popleft()   # one entry per operation in flight: whether it accesses memory (lane permutations do not)
        while i < len(code) and (i, open_) not in seen:
            seen.add((i, open_))
            addr, op, arg = code[i]
            if op.startswith("ds_"):
                open_ = (open_ + (not re.search("permute|swizzle", op),))[-16:]
            elif op == "s_waitcnt" and (m := re.search(r"lgkmcnt\((\d+)\)", arg)):
                open_ = open_[max(0, len(open_) - int(m[1])):]
            elif _to_lds(op, arg) and any(open_):
                found.add(addr)
            if op == "s_endpgm":
                break
            if op == "s_branch" or op.startswith("s_cbranch"):
                off = int(arg, 0)
                to = at[addr + 4 + 4 * (off - 65536 if off > 32767 else off)]
                if op == "s_branch":
                    i = to
                    continue
                todo.append((to, open_))
            i += 1
    return found


def test_the_reader_sees_an_open_read():
    code = [(0, "ds_read_b128", "v[0:3], v4"), (8, "ds_bpermute_b32", "v5, v6, v7"), (16, "s_waitcnt", "lgkmcnt(1)"), (20, "buffer_load_dwordx4", "v1, s[0:3], s4 offen lds"),
            (28, "s_endpgm", "")]
    assert refills_behind_open_reads(code) == set()
    assert refills_behind_open_reads([c if c[1] != "s_waitcnt" else (16, "s_waitcnt", "vmcnt(0)") for c in code]) == {20}


@pytest.mark.parametrize("obj", OBJECTS)
def test_no_buffer_is_filled_while_it_is_read(obj, tmp_path, monkeypatch):
    monkeypatch.setattr(listing, "OBJ", build.OBJ_DIR / obj)
    if not listing.OBJ.exists() or not (listing.LLVM / "llvm-objdump").exists():
        pytest.skip("needs the objects of a build and the LLVM tools")
    kernels = 0
    for name, code in listing._kernels(tmp_path):
        if OBJECTS[obj] not in name:
            continue
        kernels += 1
        assert any(_to_lds(op, arg) for _, op, arg in code), name
        assert not refills_behind_open_reads(code), name
    assert kernels
