"""The order of memory operations in the built staged kernels (k_plan5, k_hlt5).  Their waits count
operations: at the wait for a field's box only the stores of the field before may be outstanding,
which holds only if every load into LDS of a step is issued before the step's stores.  Read from
the gfx950 code of gem_amd/libadz_hip.so as llvm-objdump prints it: between two barriers no load
into LDS follows a buffer store."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "gem_amd", "libadz_hip.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


def events(code):
    """B barrier, L load into LDS, S buffer store, in the order of the code."""
    out = ""
    for line in code.splitlines():
        if "s_barrier" in line:
            out += "B"
        elif "buffer_load" in line and " lds" in line:
            out += "L"
        elif "buffer_store" in line:
            out += "S"
    return out


def in_order(ev):
    return all(not re.search("S.*L", step) for step in ev.split("B"))


def test_rule_tells_a_store_before_a_load():
    assert in_order("BBLLLSBLLLSBLLLSB") and in_order("BBLLSSSSSBLLSSSSBLLB")
    assert not in_order("BBLLLSBLLSLSB") and not in_order("BBSLLLSB")


@pytest.mark.skipif(not (os.path.exists(LIB) and os.path.exists(OBJDUMP)), reason="needs the built library and llvm-objdump")
def test_loads_into_lds_before_the_stores_of_a_step(tmp_path):
    os.symlink(LIB, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=tmp_path, check=True, capture_output=True)
    seen = 0
    for f in sorted(tmp_path.glob("*gfx950")):
        syms = subprocess.run([OBJDUMP, "--syms", f], check=True, capture_output=True, text=True).stdout
        names = {n for n in re.findall(r"_ZN3adz\d+k_(?:hlt5|plan5)\S+", syms) if not n.endswith(".kd")}
        if not names:
            continue
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--disassemble-symbols=" + ",".join(sorted(names)), f],
                              check=True, capture_output=True, text=True).stdout
        for block in text.split("\n\n"):
            m = re.search(r"<(_ZN3adz\S+)>:", block)
            if not m:
                continue
            ev = events(block)
            assert ev.count("L") >= 3 and "S" in ev, m.group(1)
            assert in_order(ev), (m.group(1), ev)
            seen += 1
    assert seen > 100
