"""Builds ``libhbsattn_amd.so`` in-tree with hipcc for gfx950.

``python -m hbsattn_amd.build`` or ``hbsattn_amd.build.build()``.  hipcc
cross-compiles, so no GPU is needed to build.
"""
from __future__ import annotations

import concurrent.futures
import os
import re
import shutil
import subprocess
import sysconfig
import tempfile

_HERE = os.path.dirname(os.path.abspath(__file__))
_ROOT = os.path.dirname(_HERE)
CSRC = os.path.join(_HERE, "csrc")
API_SOURCE = os.path.join(CSRC, "hbsa_fwd.hip")     # the C ABI and the kernels that are no templates over the head dim
INST_SOURCE = os.path.join(CSRC, "hbsa_inst.hip")   # the attention kernels of one head dim and element type
OUTPUT = os.path.join(_HERE, "libhbsattn_amd.so")
# substrings of the mangled names of the kernels with hand-issued LDS reads ...
HAND_ISSUED_READS = ("hbsa_fwd_kernel", "hbsa_bwd_dq_kernel", "hbsa_bwd_dkv")
COMPILER_ISSUED = "hbsa_fwd_kernelILi256E"   # ... except the head dim 256 instantiations, whose reads the compiler issues (it may move such a register to the other half at any time)

# -packed-fp32-ops: keep the compiler from forming v_pk_*_f32 out of scalar float code.
HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-fvisibility-inlines-hidden",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-I" + os.path.join(_ROOT, "include"), "-I" + CSRC,
]

# At head dim 256 a wavefront has the 512 registers of a SIMD, half of them accumulation registers, which the vector ALU cannot
# read.  Left to itself the compiler writes every matrix product there, the scores among them, moves them over one by one (1133
# moves in the plain kernel, 313 with the flag) and spills 37 to 135 registers beside that (none with it); told to write products
# to vector registers it keeps the output and Q operand in the other half.  8 x 2050 tokens, 16 heads, 260 -> 209 us;
# 8 x 8192 975 -> 826; head dim 208, 307 -> 225; fp32 tensors 261 -> 220; the bits are the same.  At the other head dims all
# products stand in vector registers anyway.
MFMA_IN_VGPRS = ["-mllvm", "-amdgpu-mfma-vgpr-form"]

# The one-launch kernels of eight wavefronts with packed slots: what is only jumped to begins on a line of 64 bytes.  Their tile loop is instruction for
# instruction the plain slots' one, which got 2 % faster when the next tile's look-up moved before the barrier, but where it came to lie it got slower.
# us, before that, since then, aligned (4 x 6000 tokens, 64-key blocks, 15 % kept, slots of eight in use): 32 / 16 heads, 80 rows, 5 of 8, 552, 566, 560; 32 / 8,
# 48 rows, 6, 479, 490, 483; 32 / 16, 112 rows, 7, 446, 451, 449; 32 / 2, 16 rows, 8, 409, 416, 411; 48-key blocks, 5, 616, 604, 601.  Not for all kernels: 16 x 40 .. 500
# tokens, 32 / 8 heads of 128, whose code is mostly fetched for the first time, 35.0 -> 35.7.  (Lines of 32 or 128 bytes, aligned loops, the look-up
# behind the barrier in these kernels alone: 558 to 570 for the first of them.)
ALIGNED = ["-mllvm", "-align-all-nofallthru-blocks=6"]


def units() -> list:
    """``(name, source, extra flags)`` of every translation unit of the library, the ones that take longest first."""
    def inst(d, elem, part):
        flags = [f"-DHBSA_D={d}", f"-DHBSA_E={elem}", f"-DHBSA_PART={part}"]
        return (f"{elem}_{d}_{part}", INST_SOURCE, flags + (MFMA_IN_VGPRS if d == 256 else []))

    out = [inst(d, e, 1) for d in (128, 64, 256, 32) for e in ("ElemBF16", "ElemF16")]
    out += [(n, f, flags + ALIGNED) for n, f, flags in (inst(128, e, 13) for e in ("ElemBF16", "ElemF16"))]
    out += [inst(d, e, 3) for d in (128, 64, 32) for e in ("ElemBF16", "ElemF16")]
    out += [inst(d, e, 5) for d in (192, 160, 256, 128, 96, 64, 32) for e in ("ElemBF16", "ElemF16")]
    out += [inst(d, e, 7) for d in (128, 64, 32) for e in ("ElemBF16", "ElemF16")]
    out += [inst(d, e, 8) for d in (128, 64, 256, 32) for e in ("ElemBF16", "ElemF16")]
    out += [inst(d, e, 12) for d in (128, 64, 256, 32) for e in ("ElemBF16", "ElemF16")]
    out += [inst(d, e, 9) for d in (192, 160, 256, 128, 96, 64, 32) for e in ("ElemBF16", "ElemF16")]
    out += [inst(d, e, 10) for d in (128, 64, 32) for e in ("ElemBF16", "ElemF16")]
    out += [inst(d, e, 11) for d in (128, 96, 64, 32) for e in ("ElemBF16", "ElemF16")]
    out += [inst(d, e, 6) for d in (256, 128, 64, 32) for e in ("ElemBF16", "ElemF16")]
    out += [inst(d, "ElemF16", 2) for d in (128, 64, 256, 32)]
    out += [inst(d, "ElemF16", 4) for d in (256, 128, 64, 32)]
    return out + [("api", API_SOURCE, [])]


def _kernels_with(what: str, remarks: str) -> dict:
    """Kernels whose count of ``what`` is not zero, from the compiler's resource-usage remarks."""
    counts, name = {}, None
    for line in remarks.splitlines():
        m = re.search(r"remark:\s+Function Name: (\S+)", line)
        if m:
            name = m.group(1)
        m = re.search(r"remark:\s+" + what + r": (\d+)", line)
        if m and name is not None and int(m.group(1)) > 0:
            counts[name] = int(m.group(1))
    return counts


def compile_unit(unit, objdir: str):
    """Compiles one unit into ``objdir``; returns (object file, compiler remarks)."""
    name, source, flags = unit
    obj = os.path.join(objdir, name + ".o")
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    cmd = [hipcc] + HIPCC_FLAGS + flags + ["-Rpass-analysis=kernel-resource-usage", "-c", source, "-o", obj]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError("hipcc failed: " + " ".join(cmd) + "\n" + res.stdout + res.stderr)
    return obj, res.stderr


def link(objects, output: str) -> None:
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    cmd = [hipcc, "--offload-arch=gfx950", "-shared", "-fPIC"] + list(objects) + ["-o", output]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError("hipcc failed: " + " ".join(cmd) + "\n" + res.stdout + res.stderr)


def build(verbose: bool = False) -> str:
    jobs = max(1, min(8, os.cpu_count() or 1))
    with tempfile.TemporaryDirectory() as objdir, concurrent.futures.ThreadPoolExecutor(jobs) as pool:
        host = pool.submit(compile_host, objdir)
        done = list(pool.map(lambda u: compile_unit(u, objdir), units()))
        check_registers("".join(remarks for _, remarks in done), verbose)
        link([obj for obj, _ in done], OUTPUT)
        link_host(host.result())
    if verbose:
        print(f"{OUTPUT}: {len(done)} units")
    return OUTPUT


HOST_SOURCE = os.path.join(CSRC, "torch_host.cpp")
HOST_OUTPUT = os.path.join(_HERE, "_torch_host.so")


def compile_host(objdir: str) -> str:
    """Compiles the host path (plain C++ on torch's headers, no device code)."""
    import torch
    from torch.utils import cpp_extension

    obj = os.path.join(objdir, "torch_host.o")
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-I" + os.path.join(_ROOT, "include"),
           "-I" + sysconfig.get_paths()["include"]]
    for path in cpp_extension.include_paths("cuda"):
        cmd += ["-isystem", path]
    res = subprocess.run(cmd + ["-c", HOST_SOURCE, "-o", obj], capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError("g++ failed: " + " ".join(cmd) + "\n" + res.stdout + res.stderr)
    return obj


def link_host(obj: str) -> None:
    """Links the host path against torch and the library built beside it."""
    import torch

    lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    cmd = ["g++", "-shared", obj, "-o", HOST_OUTPUT, "-L" + lib, "-L" + _HERE, "-lhbsattn_amd", "-ltorch_python", "-ltorch_cpu",
           "-ltorch_hip", "-lc10", "-lc10_hip", "-L/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath,$ORIGIN"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError("g++ failed: " + " ".join(cmd) + "\n" + res.stdout + res.stderr)


def check_registers(remarks: str, verbose: bool = False) -> None:
    # The attention kernels named above issue their LDS reads by hand and wait for them by count.  The
    # compiler does not know that such a register has a read in flight; if it spills one, or moves it to an
    # accumulation register, it saves the register before the data has arrived and the result is wrong now
    # and then.  So a build in which such a kernel spills vector registers or has accumulation registers
    # (which it needs for nothing else: its products stand in vector registers) is refused.  (The other
    # kernels leave every wait to the compiler; a spill there only costs time and is reported.)
    for what in ("VGPRs Spill", "AGPRs"):
        found = _kernels_with(what, remarks)
        fatal = {k: v for k, v in found.items() if any(n in k for n in HAND_ISSUED_READS) and COMPILER_ISSUED not in k}
        if fatal:
            raise RuntimeError(f"{what} of {fatal}: reduce register pressure (see the comment here)")
        if found and verbose and what == "VGPRs Spill":
            print(f"note: vector-register spills in {found}")


EXAMPLE_SOURCE = os.path.join(_HERE, "csrc", "cabi_example.cpp")
EXAMPLE_OUTPUT = os.path.join(_HERE, "cabi_example")


def build_example(verbose: bool = False) -> str:
    """The torch-free C++ caller of the library (``csrc/cabi_example.cpp``); run it on a GPU box as
    ``./hbsattn_amd/cabi_example``."""
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    cmd = [hipcc, "--offload-arch=gfx950", "-O2", "-std=c++17", "-I" + os.path.join(_ROOT, "include"), EXAMPLE_SOURCE,
           "-L" + _HERE, "-lhbsattn_amd", "-Wl,-rpath,$ORIGIN", "-o", EXAMPLE_OUTPUT]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError("hipcc failed: " + " ".join(cmd) + "\n" + res.stdout + res.stderr)
    if verbose:
        print(" ".join(cmd))
    return EXAMPLE_OUTPUT


if __name__ == "__main__":
    print(build(verbose=True))
    print(build_example(verbose=True))
