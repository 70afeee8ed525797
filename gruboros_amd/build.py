"""Build libmingru_hip.so (all HIP kernels + the C ABI) for gfx950 with hipcc, and
_native.so (the host side of the training path on torch tensors) with g++.

The library is written next to this file so that it travels with the source
tree; it links the HIP runtime by SONAME only, so inside a process that has
imported torch it binds to the runtime torch already loaded.
"""
import glob
import os
import shutil
import subprocess
import sys
import tempfile
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
LIB_NAME = "libmingru_hip.so"
LIB_PATH = os.path.join(HERE, LIB_NAME)
NATIVE_PATH = os.path.join(HERE, "_native.so")

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    # Packed-fp32 VALU ops are kept out of every kernel.
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall",
]


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (set HIPCC or install ROCm)")


def sources():
    return sorted(glob.glob(os.path.join(HERE, "csrc", "*.hip")))


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in proc.stdout.splitlines() if "packed-fp32-ops" not in l)
    return proc.returncode, out


# Kernels whose MFMAs are inline assembly on AGPR accumulators (the four-wave
# 16x16x32 loop): the compiler's hazard checks do not see into that assembly,
# whose instruction order keeps the hazards away only as written, so a spill the
# compiler inserts between those instructions can change results. Their
# register use is checked at every build.
NO_SPILL_KERNELS = ("gemm_persist_w4m_kernel", "gemm_kernelILi256ELi256ELi2ELi2E", "gemm_pair_kernel", "gemm_group_kernel", "gemm_t128_")


def _spilled_kernels(remarks):
    """(kernel, VGPR spills) of every guarded kernel that spills, from hipcc's
    -Rpass-analysis=kernel-resource-usage remarks."""
    bad, name = [], None
    for line in remarks.splitlines():
        if "Function Name: " in line:
            name = line.split("Function Name: ", 1)[1].split()[0]
        elif "VGPRs Spill: " in line and name and any(k in name for k in NO_SPILL_KERNELS):
            n = int(line.split("VGPRs Spill: ", 1)[1].split()[0])
            if n:
                bad.append((name, n))
    return bad


def _native_cmds(objdir):
    """(compile, link) commands of _native.so: torch's C++ API and the C ABI only, no GPU code."""
    import sysconfig

    import torch
    from torch.utils import cpp_extension

    obj = os.path.join(objdir, "native.o")
    inc = [a for d in [*cpp_extension.include_paths(), sysconfig.get_paths()["include"]] for a in ("-isystem", d)]
    lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        raise RuntimeError("g++ not found")
    compile_cmd = [cxx, "-O2", "-std=c++17", "-fPIC", "-Wall", "-DTORCH_EXTENSION_NAME=_native",
                   f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-I", os.path.join(ROOT, "include"),
                   *inc, "-c", os.path.join(HERE, "csrc", "host", "native.cpp"), "-o", obj]
    link_cmd = [cxx, "-shared", obj, "-L", HERE, "-lmingru_hip", "-L", lib, "-ltorch", "-ltorch_cpu", "-lc10",
                "-ltorch_python", "-Wl,-rpath,$ORIGIN"]
    return compile_cmd, link_cmd


def _link(cmd, path, verbose):
    """Runs the link command into a directory of its own beside `path` and moves the result there:
    the linker creates the file, so its mode is the umask's (a mkstemp file is 0600, and a linker
    that writes into it leaves a library only its builder can read)."""
    name = os.path.basename(path)
    with tempfile.TemporaryDirectory(prefix=name + ".tmp", dir=os.path.dirname(path)) as tmp:
        rc, out = _run([*cmd, "-o", os.path.join(tmp, name)], verbose)
        if rc != 0:
            raise RuntimeError(f"linking {name} failed ({rc}):\n{out}")
        os.replace(os.path.join(tmp, name), path)


def build(verbose: bool = False) -> str:
    """Compile every csrc/*.hip (one hipcc process per file, in parallel) and link them into one
    shared library, then link _native.so against it; returns the library's path."""
    srcs = sources()
    inc = ["-I", os.path.join(ROOT, "include"), "-I", os.path.join(HERE, "csrc")]
    with tempfile.TemporaryDirectory(prefix="mg_build_") as objdir:
        objs = [os.path.join(objdir, os.path.basename(s) + ".o") for s in srcs]
        jobs = max(1, min(len(srcs) + 1, os.cpu_count() or 1, 16))
        native_compile, native_link = _native_cmds(objdir)
        with ThreadPoolExecutor(jobs) as pool:
            native_done = pool.submit(_run, native_compile, verbose)
            def compile_one(so):
                extra = ["-Rpass-analysis=kernel-resource-usage"] if os.path.basename(so[0]) == "gemm.hip" else []
                return _run([hipcc(), *HIPCC_FLAGS, *extra, *inc, "-c", so[0], "-o", so[1]], verbose and not extra)

            results = list(pool.map(compile_one, zip(srcs, objs)))
        for src, (rc, out) in zip(srcs, results):
            if rc != 0:
                raise RuntimeError(f"hipcc failed on {os.path.basename(src)} ({rc}):\n{out}")
            if os.path.basename(src) == "gemm.hip":
                bad = _spilled_kernels(out)
                if bad:
                    raise RuntimeError("kernels with inline-assembly MFMAs spill registers (their results would not "
                                       "be trustworthy): " + ", ".join(f"{k} ({n})" for k, n in bad))
            elif verbose and out.strip():
                print(out, flush=True)
        rc, out = native_done.result()
        if rc != 0:
            raise RuntimeError(f"g++ failed on native.cpp ({rc}):\n{out}")
        _link([hipcc(), "--offload-arch=gfx950", "-fPIC", "-shared", *objs], LIB_PATH, verbose)
        _link(native_link, NATIVE_PATH, verbose)
    return LIB_PATH


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
