"""
Ahead-of-time build of ``librtn_native_lstm2.so`` for gfx950 with hipcc.

Takes the place of the reference's run-time compile-and-cache step for native ops
(returnn/util/native_code_compiler.py:216-354, returnn/torch/util/native_op_code_compiler.py:94-131):
there is one fixed target (MI355X), so the library is built once, in-tree, and loaded with ctypes.
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sys
from typing import List, Optional

_dir = os.path.dirname(os.path.abspath(__file__))
CSRC_DIR = os.path.join(_dir, "csrc")
LIB_NAME = "librtn_native_lstm2.so"
LIB_PATH = os.path.join(CSRC_DIR, LIB_NAME)
HOST_SOURCE = "rtn_native_lstm2.hip"
TABLES_SOURCE = "lstm2_kernel_tables.hip"  # compiled once per part: the instantiations of the persistent kernels
TABLE_PARTS = 17
# Matrix instructions that leave their results where vector instructions read them: the bf16 forward kernels add two accumulators per
# tile, and out of accumulation registers every one of them is copied first (B=256 T=200 n=1024: 717 us, 690 without the copies).
# (Not part 17, layers beyond n = 1024, whose tiles have one accumulator: with it T=100 n=2048, 16 and 32 rows, 250 and 273 us, 247 and 271
# without; n=1536, 17 rows 249 / 245; n=1280, 48 rows 255 / 251.)
VGPR_FORM = ["-mllvm", "-amdgpu-mfma-vgpr-form=1"]
VGPR_FORM_PARTS = (1, 2, 14)
SOURCES = [HOST_SOURCE, TABLES_SOURCE]
HEADERS = ["lstm2_kernels.h", "lstm2_step_kernel.h", "lstm2_wide_kernel.h", "lstm2_solo_kernel.h", "lstm2_dual_kernel.h", "lstm2_sparse_kernel.h", "lstm2_bwd_kernels.h", "lstm2_bwd_local_kernel.h", "lstm2_bwd_wide_kernel.h", "weight_grad_kernel.h", "lstm2_params.h", "lstm2_kernel_tables.h",
           os.path.join("..", "..", "include", "rtn_native_lstm2.h")]  # fmt: skip
# the torch side of the calls (host code only)
BINDING_SOURCE = "rtn_torch_binding.cpp"
BINDING_PATH = os.path.join(_dir, "_rtn_torch.so")
OBJ_DIR = os.path.join(CSRC_DIR, "_obj")
OFFLOAD_ARCH = "gfx950"
ROCM_LIB_DIR = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "lib")  # rocBLAS (weight-gradient GEMM of the backward op)


def hipcc_path() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (set HIPCC or install ROCm under /opt/rocm)")


def _flags() -> List[str]:
    """Packed fp32 VALU instructions are disabled on purpose.  Floating-point contraction is off so that every kernel
    variant and decomposition rounds the gate and cell arithmetic identically (results do not depend on the execution
    mode) and like the CPU reference code."""
    return [
        "--offload-arch=%s" % OFFLOAD_ARCH,
        "-O3",
        "-ffp-contract=off",
        "-std=c++17",
        "-fPIC",
        "-Xclang",
        "-target-feature",
        "-Xclang",
        "-packed-fp32-ops",
        "-Wall",
        "-Wno-unused-command-line-argument",
    ]


def compile_commands(obj_dir: Optional[str] = None) -> List[List[str]]:
    """The exact hipcc lines that make the objects: the host code, and the kernel tables once per part."""
    obj_dir = obj_dir or OBJ_DIR
    cmds = [[hipcc_path()] + _flags() + ["-c", os.path.join(CSRC_DIR, HOST_SOURCE), "-o", os.path.join(obj_dir, "host.o")]]
    for part in range(1, TABLE_PARTS + 1):
        cmds.append(
            [hipcc_path()] + _flags() + (VGPR_FORM if part in VGPR_FORM_PARTS else [])
            + ["-DRTN_TABLE_PART=%i" % part, "-Wno-unused-function", "-c", os.path.join(CSRC_DIR, TABLES_SOURCE), "-o", os.path.join(obj_dir, "tables_%i.o" % part)]
        )  # fmt: skip
    return cmds


def link_command(output: Optional[str] = None, obj_dir: Optional[str] = None) -> List[str]:
    obj_dir = obj_dir or OBJ_DIR
    objs = [os.path.join(obj_dir, "host.o")] + [os.path.join(obj_dir, "tables_%i.o" % part) for part in range(1, TABLE_PARTS + 1)]
    return [hipcc_path(), "--offload-arch=%s" % OFFLOAD_ARCH, "-shared", "-fPIC", "-o", output or LIB_PATH] + objs + [
        "-L%s" % ROCM_LIB_DIR, "-lrocblas", "-Wl,-rpath,%s" % ROCM_LIB_DIR,
    ]  # fmt: skip


def binding_command(output: Optional[str] = None) -> List[str]:
    """The g++ line of the torch binding: against the torch and HIP headers, no device code.  The HIP runtime is the one
    torch has loaded by then."""
    import sysconfig

    import torch
    from torch.utils import cpp_extension

    torch_lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    cmd = [os.environ.get("CXX") or "g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-Wall", "-Wno-unknown-pragmas", "-Wno-attributes"]
    cmd += ["-D_GLIBCXX_USE_CXX11_ABI=%i" % int(torch._C._GLIBCXX_USE_CXX11_ABI), "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", "-DTORCH_EXTENSION_NAME=_rtn_torch"]
    cmd += ["-isystem" + d for d in cpp_extension.include_paths("cuda") + [sysconfig.get_paths()["include"]] if os.path.isdir(d)]
    cmd += [os.path.join(CSRC_DIR, BINDING_SOURCE), "-o", output or BINDING_PATH, "-L" + torch_lib, "-L" + ROCM_LIB_DIR]
    return cmd + ["-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_hip", "-ltorch", "-ltorch_python", "-lamdhip64"]


def needs_build() -> bool:
    if not os.path.exists(LIB_PATH) or not os.path.exists(BINDING_PATH):
        return True
    t = min(os.path.getmtime(LIB_PATH), os.path.getmtime(BINDING_PATH))
    deps = [os.path.join(CSRC_DIR, f) for f in SOURCES + HEADERS + [BINDING_SOURCE]] + [os.path.abspath(__file__)]
    return any(os.path.getmtime(d) > t for d in deps if os.path.exists(d))


def _jobs() -> int:
    try:
        limit = int(os.environ.get("MAX_JOBS", "0"))
    except ValueError:
        limit = 0
    return max(1, min(TABLE_PARTS + 1, limit or (os.cpu_count() or 1)))


def build_library(force: bool = True, verbose: bool = False) -> str:
    """
    Compile the HIP library in-tree: the objects side by side (as many at once as the machine has cores, or MAX_JOBS),
    then one link.

    :param force: rebuild even if the library is newer than its sources
    :return: path of the built library
    """
    if not force and not needs_build():
        return LIB_PATH
    from concurrent.futures import ThreadPoolExecutor

    obj_dir = OBJ_DIR + ".tmp.%i" % os.getpid()
    os.makedirs(obj_dir, exist_ok=True)
    tmp = LIB_PATH + ".tmp.%i" % os.getpid()
    tmp_binding = BINDING_PATH + ".tmp.%i" % os.getpid()

    def run(cmd):
        if verbose:
            print("$", " ".join(cmd), file=sys.stderr)
        proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
        return cmd, proc.returncode, proc.stdout

    try:
        with ThreadPoolExecutor(max_workers=_jobs()) as pool:
            results = list(pool.map(run, [binding_command(tmp_binding)] + compile_commands(obj_dir)))
        results.append(run(link_command(tmp, obj_dir)) if all(rc == 0 for _, rc, _ in results) else (["(link skipped)"], 0, ""))
        for cmd, rc, out in results:
            if rc != 0:
                raise RuntimeError("the compiler failed (%i):\n$ %s\n%s" % (rc, " ".join(cmd), out))
            if verbose and out.strip():
                print(out, file=sys.stderr)
        os.replace(tmp, LIB_PATH)
        os.replace(tmp_binding, BINDING_PATH)
    finally:
        shutil.rmtree(obj_dir, ignore_errors=True)
        for left in (tmp, tmp_binding):
            if os.path.exists(left):
                os.remove(left)
    return LIB_PATH


if __name__ == "__main__":
    print(build_library(force=True, verbose=True))
