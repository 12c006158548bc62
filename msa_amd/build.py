"""Builds the C-ABI libraries from ``csrc/*.hip`` for gfx950 with hipcc: ``libmsa_amd.so`` (routing / sparse attention)
and ``libmsa_seq.so`` (the layers of the decoders of mixed layers), and the extension module ``_host.so`` (``csrc/host.cpp``).

``python -m msa_amd.build`` compiles all in-tree; the libraries then travel with the source tree.
"""
from __future__ import annotations

import fcntl
import os
import re
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libmsa_amd.so")
SEQ_LIB = os.path.join(HERE, "libmsa_seq.so")
HOST_LIB = os.path.join(HERE, "_host.so")    # the extension module of csrc/host.cpp
SHARED = ("status.hip", "glue.hip")          # linked into both libraries
ARCH = "gfx950"
# packed fp32 VALU ops are switched off for all device code of this library
FLAGS = ["-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}", "-Xclang", "-target-feature", "-Xclang",
         "-packed-fp32-ops", "-Wall", "-Wno-unused-function", "-Wno-inline-asm"]


def sources():
    return sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hip"))


def seq_sources():
    """What ``libmsa_seq.so`` is made of: the ``seq_*`` sources and the shared ones."""
    return [s for s in sources() if os.path.basename(s).startswith("seq_") or os.path.basename(s) in SHARED]


def main_sources():
    return [s for s in sources() if not os.path.basename(s).startswith("seq_")]


def _compile(src: str) -> str:
    obj = src[:-4] + ".o"
    cmd = ["hipcc", *FLAGS, "-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    noise = "is not a recognized feature for this target"
    err = "\n".join(l for l in r.stderr.splitlines() if noise not in l)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{err}")
    if err.strip():
        sys.stderr.write(err + "\n")
    return obj


# ---------------------------------------------------------------------------------------------------------------
# Contracts between hand-written asm statements and the compiler-allocated code around them, checked on the device
# assembly of every build:
#  * score_scan4_kernel (route_score.hip): its asm statements own v128-v255 and all accumulation registers across
#    statements.  The code the compiler generates for that kernel must therefore stay below v128, touch no
#    accumulation register (the compiler would only do so to spill), and use no scratch memory.
#    score_scan4_units_kernel: likewise below v96.
#  * tile_gemm_kernel (gemm.hip): the registers of score_scan4_kernel; tile_flow_kernel: v24-v255 and all accumulation registers.
#  * flash_wide_kernel (flash_attn.hip): likewise, its statements own v56-v255 and all accumulation registers.
#  * flash_attn_kernel (flash_attn.hip): its direct-to-LDS loads are asm statements the compiler does not order
#    against LDS reads; a spill would add vector-memory waits in the middle of that ring.  No scratch, no spills.
#  * score_parts_kernel (route_score.hip), rows_ring_kernel (rows_ring.h), attn_ring_kernel and attn_decode_fused_kernel (attn.hip): likewise, they count what
#    their rings have in flight.  What the first requests into LDS in front of its loop is read by asm statements, for
#    which the compiler does not wait: the first request has to be waited for in front of the first LDS read.
#  * flow_gemm_kernel (flow_gemm.hip): its products are asm statements whose latency the compiler does not know: between the first
#    and the last of them nothing else may touch an accumulation register.  It counts what its ring has in flight.
#  * delta_step_kernel (seq_delta.hip): loads past the end of what it reads rely on the range check of the buffer, which compares
#    the vector offset alone.  No scalar offsets.
# ---------------------------------------------------------------------------------------------------------------
CONTRACTS = {
    "route_score.hip": [("score_scan4_kernel", {"max_compiler_vgpr": 127, "no_agpr": True}),
                        ("score_scan4_units_kernel", {"max_compiler_vgpr": 95, "no_agpr": True}), ("score_parts_kernel", {})],
    "gemm.hip": [("tile_gemm_kernel", {"max_compiler_vgpr": 127, "no_agpr": True}), ("tile_flow_kernel", {"max_compiler_vgpr": 23, "no_agpr": True})],
    "flash_attn.hip": [("flash_attn_kernel", {}), ("flash_wide_kernel", {"max_compiler_vgpr": 55, "no_agpr": True})],
    "linear.hip": [("rows_ring_kernel", {})],
    "flow_gemm.hip": [("flow_gemm_kernel", {"fixed_products": True})],
    "seq_rows.hip": [("rows_ring_kernel", {})],
    "attn.hip": [("attn_ring_kernel", {}), ("attn_decode_fused_kernel", {})],
    "seq_delta.hip": [("delta_step_kernel", {"no_scalar_offset": True})],
}
LDS_WAITS = {"flow_gemm.hip": "flow_gemm_kernel", "linear.hip": "rows_ring_kernel", "seq_rows.hip": "rows_ring_kernel"}


def _device_asm(src: str, extra=()) -> str:
    r = subprocess.run(["hipcc", *FLAGS, *extra, "--cuda-device-only", "-S", src, "-o", "-"], capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc -S failed for {src}:\n{r.stderr}")
    return r.stdout


def check_kernel_contracts(asm: str, kernel_substring: str, max_compiler_vgpr=None, no_agpr=False, no_scalar_offset=False, fixed_products=False):
    """Returns the list of violations found in the device assembly `asm` for every kernel whose symbol contains
    `kernel_substring`: scratch use or spills (always), and, outside inline-asm regions, vector registers above
    `max_compiler_vgpr` / any accumulation register (with `fixed_products` between the products) / any buffer access with a scalar offset."""
    problems = []
    lines = asm.split("\n")
    # function bodies: from "<symbol>:" to s_endpgm
    i, found = 0, 0
    while i < len(lines):
        m = re.match(r"^(\S*%s\S*):" % re.escape(kernel_substring), lines[i])
        if not m or m.group(1).endswith(".kd"):
            i += 1
            continue
        name, found = m.group(1), found + 1
        in_asm, multiplied, between = False, False, []
        i += 1
        while i < len(lines) and "s_endpgm" not in lines[i]:
            line = lines[i]
            i += 1
            if "#ASMSTART" in line:
                in_asm = True
                continue
            if "#ASMEND" in line:
                in_asm = False
                continue
            code = line.split(";")[0].strip()
            if not code or code.endswith(":") or code.startswith("."):
                continue
            if in_asm:
                if code.startswith("v_mfma"):
                    problems += between
                    multiplied, between = True, []
                continue
            if fixed_products and multiplied and re.search(r"\ba\d+\b|\ba\[\d+|accvgpr", code):
                between.append(f"{name}: an accumulation register is touched between the products: {code}")
            if code.startswith("scratch_"):
                problems.append(f"{name}: scratch access: {code}")
            if no_agpr and re.search(r"\ba\d+\b|\ba\[\d+|accvgpr", code):
                problems.append(f"{name}: compiler-generated code touches an accumulation register: {code}")
            if no_scalar_offset and re.match(r"buffer_(load|store)\w* .*\bs\[\d+:\d+\], (?!0\b)", code):
                problems.append(f"{name}: buffer access with a scalar offset: {code}")
            if max_compiler_vgpr is not None:
                for mm in re.finditer(r"\bv(\d+)\b|\bv\[(\d+):(\d+)\]", code):
                    hi = int(mm.group(1) or mm.group(3))
                    if hi > max_compiler_vgpr:
                        problems.append(f"{name}: compiler-generated code uses v{hi}: {code}")
    if found == 0:
        problems.append(f"no kernel matching {kernel_substring!r} in the assembly")
    # resource summary of the code object (YAML metadata at the end of the assembly)
    for m in re.finditer(r"\.name:\s+(\S*%s\S*)\n(.*?)\.wavefront_size" % re.escape(kernel_substring), asm, flags=re.S):
        meta = m.group(2)
        for key in ("private_segment_fixed_size", "vgpr_spill_count"):
            mm = re.search(r"\.%s:\s+(\d+)" % key, meta)
            if mm and int(mm.group(1)) != 0:
                problems.append(f"{m.group(1)}: {key} = {mm.group(1)}")
    return problems


def check_lds_waits(asm: str, kernel_substring: str):
    """Violations in the kernels whose symbol contains `kernel_substring`: an LDS read that no wait covering the kernel's first
    direct-to-LDS load precedes.  Loads return in order, so a wait for all but n operations covers it once n buffer loads are
    younger (other operations may stand in branches and count for nothing)."""
    problems, found = [], 0
    for m in re.finditer(r"^(\S*%s\S*):(.*?)s_endpgm" % re.escape(kernel_substring), asm, flags=re.S | re.M):
        found += 1
        younger, covered = None, False
        for line in m.group(2).split("\n"):
            code = line.split(";")[0].strip()
            wait = re.search(r"vmcnt\((\d+)\)", code)
            if wait and younger is not None:
                covered |= int(wait.group(1)) <= younger
            elif code.startswith("buffer_load"):
                younger = younger + 1 if younger is not None else 0 if code.endswith(" lds") else None
            elif code.startswith("ds_read"):
                if not covered:
                    problems.append(f"{m.group(1)}: LDS is read before the first load into it has been waited for: {code}")
                break
    return problems if found else [f"no kernel matching {kernel_substring!r} in the assembly"]


def _check_contracts(src: str) -> None:
    name = os.path.basename(src)
    asm = _device_asm(src)
    problems = []
    for kernel, kw in CONTRACTS.get(name, ()):
        problems += check_kernel_contracts(asm, kernel, **kw)
    if name in LDS_WAITS:
        problems += check_lds_waits(asm, LDS_WAITS[name])
    if problems:
        raise RuntimeError("inline-asm contract broken in %s:\n  %s" % (src, "\n  ".join(problems[:20])))


def _link(objs, lib: str) -> str:
    tmp = lib + ".tmp"
    r = subprocess.run(["hipcc", "-shared", "-fPIC", f"--offload-arch={ARCH}", *objs, "-o", tmp],
                       capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    os.replace(tmp, lib)
    return lib


def build_host() -> str:
    """Compiles the extension module of the host's side (C++ against PyTorch's headers, no device code)."""
    import sysconfig
    from torch.utils import cpp_extension
    torch_lib = os.path.join(os.path.dirname(cpp_extension.__file__), "..", "lib")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    include = [sysconfig.get_paths()["include"], *cpp_extension.include_paths(), os.path.join(rocm, "include")]
    tmp = HOST_LIB + ".tmp"
    r = subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", *("-I" + i for i in include),
                        os.path.join(CSRC, "host.cpp"), "-o", tmp, "-L" + torch_lib, "-ltorch_python", "-ltorch_cpu", "-lc10_hip", "-lc10",
                        "-L" + os.path.join(rocm, "lib"), "-lamdhip64", "-ldl"], capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"g++ failed for host.cpp:\n{r.stderr}")
    os.replace(tmp, HOST_LIB)
    return HOST_LIB


def build_seq(jobs: int = 8) -> str:
    """Compiles and links ``libmsa_seq.so`` alone."""
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        return _link(list(ex.map(_compile, seq_sources())), SEQ_LIB)


def ensure_seq() -> str:
    """``libmsa_seq.so`` and the extension module, compiled if they are missing (a fresh checkout); concurrent callers wait for the first."""
    if not (os.path.exists(SEQ_LIB) and os.path.exists(HOST_LIB)):
        with open(SEQ_LIB + ".lock", "w") as lock:
            fcntl.flock(lock, fcntl.LOCK_EX)
            if not os.path.exists(SEQ_LIB):
                build_seq()
            if not os.path.exists(HOST_LIB):
                build_host()
    return SEQ_LIB


def build(jobs: int = 8) -> str:
    """Compiles every source (always, even if the libraries exist), checks the inline-asm contracts on the device
    assembly and links both shared libraries."""
    srcs = sources()
    for gen, inc in (("gen_scan_asm.py", "scan_asm.inc"), ("gen_flash_asm.py", "flash_asm.inc")):
        if subprocess.run([sys.executable, os.path.join(CSRC, gen), "--check"]).returncode != 0:
            raise RuntimeError(f"csrc/{inc} is not what csrc/{gen} generates: run the generator")
    checked = [s for s in srcs if os.path.basename(s) in {**CONTRACTS, **LDS_WAITS}]
    with ThreadPoolExecutor(max_workers=min(jobs, len(srcs) + len(checked))) as ex:
        checks = [ex.submit(_check_contracts, s) for s in checked] + [ex.submit(build_host)]
        objs = dict(zip(srcs, ex.map(_compile, srcs)))
        for c in checks:
            c.result()
    _link([objs[s] for s in seq_sources()], SEQ_LIB)
    return _link([objs[s] for s in main_sources()], LIB)


if __name__ == "__main__":
    print(build())
