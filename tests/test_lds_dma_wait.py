"""The direct global-memory-to-LDS loads of the built kernels: each takes its
LDS address from M0 and its base from scalar registers, through inline
assembly, where the compiler inserts no wait states.  gfx9 needs one between
a scalar write of M0 and the load that reads it, and five between a vector
instruction's write of a scalar register and a vector memory instruction that
reads it.  Checked in the assembly of the library that is built here."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "blasx_amd", "lib", "libblasx.so")
OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"
# vector instructions whose first operand is a scalar register
VALU_TO_SGPR = re.compile(r"v_(readfirstlane|readlane|cmp)")


def sgprs(op):
    """the scalar registers that an operand names: s7, s[4:5]"""
    m = re.fullmatch(r"s(\d+)|s\[(\d+):(\d+)\]", op.strip())
    if not m:
        return set()
    if m.group(1):
        return {int(m.group(1))}
    return set(range(int(m.group(2)), int(m.group(3)) + 1))


def scan(lines):
    """(loads, faults) of one code object's assembly: wait states are counted
    along the text, one an instruction, s_nop N counting N + 1"""
    loads, faults = 0, []
    fn, m0, valu = "", 99, {}  # wait states since M0 / a register's vector write
    for line in lines:
        if line.endswith(">:"):
            fn, m0, valu = line.split("<")[-1][:-2], 99, {}
            continue
        text = line.split("//")[0].strip()
        if not text or text.startswith(";") or not re.match(r"[a-z]+_", text):
            continue
        name, _, rest = text.partition(" ")
        ops = [o.strip() for o in rest.split(",")]
        if "_load_lds_" in name or (name.startswith("buffer_load") and rest.endswith(" lds")):
            loads += 1
            if m0 < 1:
                faults.append((fn, "M0", text))
            # "s[4:5] offset:16": the last operand may carry modifiers
            for o in ops:
                for r in sgprs(o.split(" ")[0]):
                    if valu.get(r, 99) < 5:
                        faults.append((fn, f"s{r}", text))
        passed = int(ops[0], 0) + 1 if name == "s_nop" else 1
        m0 = 0 if name.startswith("s_") and ops and ops[0] == "m0" else m0 + passed
        valu = {r: w + passed for r, w in valu.items() if w + passed < 5}
        if VALU_TO_SGPR.match(name):
            valu.update({r: 0 for r in sgprs(ops[0])})
    return loads, faults


def test_scan_sees_missing_waits():
    load = "\tglobal_load_lds_dwordx4 v1, s[4:5]   // 0: 0"
    mov, nop = "\ts_mov_b32 m0, s3", "\ts_nop 0"
    assert scan([mov, load])[1] and not scan([mov, nop, load])[1]
    assert not scan([mov, "\ts_add_u32 s6, s6, s7", load])[1]
    rfl = "\tv_readfirstlane_b32 s5, v0"
    assert scan([rfl, mov, nop, load])[1]
    assert not scan([rfl, mov, "\ts_nop 3", load])[1]
    assert scan(["\tglobal_load_lds_dwordx4 v[0:1], off"])[0] == 1


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="needs llvm-objdump")
def test_built_kernels_wait_before_lds_loads(bx, tmp_path):
    lib = shutil.copy(LIB, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", str(lib)], cwd=tmp_path, check=True,
                   stdout=subprocess.DEVNULL)
    objs = [f for f in sorted(os.listdir(tmp_path)) if f.endswith("gfx950")]
    assert objs
    loads, faults = 0, []
    for f in objs:
        out = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", f], cwd=tmp_path, check=True,
                             capture_output=True, text=True).stdout
        n, bad = scan(out.splitlines())
        loads += n
        faults += bad
    assert loads > 1000  # the GEMM and split-product kernels
    assert not faults, (len(faults), faults[:3])
