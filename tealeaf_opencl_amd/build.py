"""Build libtealeaf_mi355x.so (gfx950) in-tree with hipcc.

Usage: python -m tealeaf_opencl_amd.build   (or build() from Python)
"""
import os
import re
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIBDIR = os.path.join(HERE, "lib")
LIBNAME = "libtealeaf_mi355x.so"
ARCH = os.environ.get("TL_OFFLOAD_ARCH", "gfx950")

SOURCES = ["tl_kernels.hip", "tl_resident.hip", "tl_refine.hip", "tl_adjoint.hip", "tl_chunk.hip", "tl_driver.hip", "tl_deck.cpp",
           "tl_eigen.cpp"]
HEADERS = ["tl_common.h", "tl_device.h", "tl_state.h", "tl_resident.h", "tl_kernels.h", "tl_chunk.h", "tl_deck.h", "tl_eigen.h"]

# packed FP32 instructions are disabled on every device compile
DEVICE_FLAGS = ["-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]
# an ignored hipError_t (a nodiscard value) fails the build
COMMON = ["-O3", "-std=c++17", "-fPIC", "-Wall", "-Wno-unused-function", "-Werror=shadow", "-Werror=unused-value",
          "-I", os.path.join(HERE, "..", "include")]
# Kernels that must not spill vector registers: the resident solver's hold them to
# the last one, and a spill placed where only some lanes of a wavefront are active,
# reloaded by all of them, has made one fault. The compiler is asked what it used.
NO_SPILL = ("tl_resident.hip", "tl_refine.hip")
USAGE = ["-Rpass-analysis=kernel-resource-usage"]


def lib_path():
    return os.path.join(LIBDIR, LIBNAME)


def _messages(out):
    """The compiler's output without its expected warnings and the usage remarks."""
    keep = []
    remark = False
    for l in out.splitlines():
        # a remark's line is followed by its source line and a caret
        remark = "kernel-resource-usage]" in l or (remark and re.match(r" *\d* \|", l) is not None)
        if not remark and "packed-fp32-ops" not in l and "not a recognized feature" not in l:
            keep.append(l)
    return "\n".join(keep)


def spilling_kernels(out):
    """(number of kernels, those that spill vector registers) by the compiler's
    usage remarks."""
    kernels, name = {}, None
    for l in out.splitlines():
        m = re.search(r"remark: .*?(Function Name|VGPRs Spill): (\S+) \[-Rpass-analysis=kernel-resource-usage\]", l)
        if m and m.group(1) == "Function Name":
            name = m.group(2)
        elif m:
            kernels[name] = int(m.group(2))
    return len(kernels), sorted(k for k, n in kernels.items() if n)


def _run(cmd):
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = _messages(proc.stdout)
    if proc.returncode != 0:
        raise RuntimeError("build failed:\n" + " ".join(cmd) + "\n" + out)
    return out


def build(verbose=False, jobs=4):
    """Compile every source for gfx950 and link the shared library."""
    os.makedirs(LIBDIR, exist_ok=True)
    objdir = os.path.join(LIBDIR, "obj")
    os.makedirs(objdir, exist_ok=True)
    cmds = []
    objs = []
    for src in SOURCES:
        obj = os.path.join(objdir, os.path.splitext(src)[0] + ".o")
        objs.append(obj)
        path = os.path.join(CSRC, src)
        if src.endswith(".hip"):
            cmd = ["hipcc", "--offload-arch=" + ARCH, "-x", "hip"] + COMMON + DEVICE_FLAGS + ["-c", path, "-o", obj]
            if src in NO_SPILL:
                cmd += USAGE
        else:
            cmd = ["g++"] + COMMON + ["-c", path, "-o", obj]
        cmds.append(cmd)
    procs = []
    for cmd in cmds:
        if verbose:
            print(" ".join(cmd), flush=True)
        procs.append((cmd, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)))
    errors = []
    for cmd, p in procs:
        full, _ = p.communicate()
        out = _messages(full)
        if p.returncode != 0:
            errors.append(" ".join(cmd) + "\n" + out)
        elif USAGE[0] in cmd and (not spilling_kernels(full)[0] or spilling_kernels(full)[1]):
            errors.append(" ".join(cmd) + "\nkernels that spill vector registers: %s of %d"
                          % (spilling_kernels(full)[1], spilling_kernels(full)[0]))
        elif verbose and out.strip():
            print(out)
    if errors:
        raise RuntimeError("build failed:\n" + "\n\n".join(errors))
    tmp = lib_path() + ".tmp"
    link = ["hipcc", "--offload-arch=" + ARCH, "-shared", "-fPIC", "-o", tmp] + objs + ["-ldl"]
    if verbose:
        print(" ".join(link), flush=True)
    _run(link)
    os.replace(tmp, lib_path())
    return lib_path()


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
