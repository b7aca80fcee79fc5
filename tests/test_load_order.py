"""The pipelined GEMMs wait for their first activations by counting the loads issued behind them, so the
loads of their prologue have to be issued in the source's order. This reads the compiled kernels (the
objects the library was linked from) and checks, for every instantiation, that the direct loads of
the first sub-step come before the loads that the first barrier's wait leaves in flight: the compiler
had once moved register loads ahead of them (q4_gemm_wide, 16 rows, two weight terms).
CPU only: it needs the build's objects and binutils."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BUILD = os.path.join(ROOT, "bybylang_amd", "_build")
LLVM = "/opt/rocm/llvm/bin"

# kernel -> (object, direct loads per wave of the first sub-step, from its integer template arguments)
KERNELS = {
    "q4_gemm_wide": ("byhip_gemm.hip.o", lambda t: t[0] * (2 if t[3] == 2 else 1)),
    "q4_gemm_tall": ("byhip_gemm.hip.o", lambda t: 2),
    "gemm_planes": ("byhip_planes.hip.o", lambda t: t[1]),
    "gemm_planes_half": ("byhip_planes.hip.o", lambda t: (4 * t[0] * t[1] + 16) // (t[0] * t[2])),
    "mxfp4_gemm_mid": ("byhip_mxfp4.hip.o", lambda t: 4),
    "gemm_f32_q4": ("byhip_exact.hip.o", lambda t: t[0]),
    "gemm_fp4_mx": ("byhip_fp4mx.hip.o", lambda t: 2 * t[0]),
}


def listing(obj, tmp):
    """The disassembly of an object's gfx950 code, line by line."""
    fb, co = str(tmp / "fatbin"), str(tmp / "code")
    subprocess.run(["objcopy", "--dump-section", ".hip_fatbin=" + fb, obj, os.devnull], check=True, capture_output=True)
    subprocess.run([LLVM + "/clang-offload-bundler", "--unbundle", "--type=o", "--targets=hipv4-amdgcn-amd-amdhsa--gfx950",
                    "--input=" + fb, "--output=" + co], check=True, capture_output=True)
    text = subprocess.run([LLVM + "/llvm-objdump", "-d", "--no-show-raw-insn", co], check=True, capture_output=True, text=True).stdout
    return text.splitlines()


def prologues(obj, tmp):
    """{mangled name: (string of 'D' for direct loads and 'r' for register loads before the first barrier,
    the vmcnt of the last wait before it)}"""
    out, name, seq, wait = {}, None, "", None
    for line in listing(obj, tmp):
        m = re.match(r"[0-9a-f]+ <(.*)>:", line)
        if m:
            name, seq, wait = m.group(1), "", None
        elif name and line.startswith("\t"):
            if re.search(r"\b(buffer|global)_load", line):
                seq += "D" if " lds" in line else "r"
            m = re.search(r"s_waitcnt.*vmcnt\((\d+)\)", line)
            if m:
                wait = int(m.group(1))
            if "s_barrier" in line:
                out[name] = (seq, wait)
                name = None
    return out


@pytest.mark.parametrize("kernel", sorted(KERNELS))
def test_first_loads_precede_the_ones_left_in_flight(kernel, tmp_path):
    obj, direct = KERNELS[kernel]
    path = os.path.join(BUILD, obj)
    if not (os.path.exists(path) and shutil.which("objcopy") and os.path.exists(LLVM + "/llvm-objdump")):
        pytest.skip("the build's objects or binutils are not there")
    seen = 0
    for name, (seq, wait) in prologues(path, tmp_path).items():
        m = re.search(r"%d%sI(.*)EEv" % (len(kernel), kernel), name)
        if not m:
            continue
        args = [int(v) for v in re.findall(r"L[a-zN](?:\w*?BFormatE)?(\d+)E", m.group(1))]
        seen += 1
        assert wait is not None, name
        landed = seq[:max(0, len(seq) - wait)]
        assert landed.count("D") >= direct(args), f"{name}: {seq} with {wait} left in flight"
    assert seen >= 3


def test_column_kernel_leaves_one_step_in_flight(tmp_path):
    """gemm_f32_q4_cols has no barrier in its loop: each wave waits for step t by leaving the loads of step
    t + 1 in flight, so those must be the newest at every such wait, all of them issued since the branch
    before it, and the first step's must stand before the first branch."""
    path = os.path.join(BUILD, "byhip_exact.hip.o")
    if not (os.path.exists(path) and shutil.which("objcopy") and os.path.exists(LLVM + "/llvm-objdump")):
        pytest.skip("the build's objects or binutils are not there")
    seen, name = 0, None
    for line in listing(path, tmp_path):
        m = re.match(r"[0-9a-f]+ <(.*)>:", line)
        if m:
            m = re.search(r"16gemm_f32_q4_colsILb([01])EEEv", m.group(1))
            name, seq, first, waits = m, "", True, 0
            loads = 8 + 2 + (m.group(1) == "0") if m else 0  # activations, weights and scales, zeros per group
        if not name:
            continue
        if re.search(r"\b(buffer|global)_load", line):
            seq += "D" if " lds" in line else "r"
        elif re.search(r"\bs_c?branch", line):
            if first:
                assert seq.count("D") == 8 and len(seq) == loads, seq
            first, seq = False, ""
        elif re.search(r"s_waitcnt vmcnt\(%d\)" % loads, line):
            assert seq.count("D") == 8 and len(seq) == loads, f"{seq} before a wait that leaves {loads} in flight"
            waits += 1
        elif "s_endpgm" in line:
            assert waits == 2, waits
            seen, name = seen + 1, None
    assert seen == 2
