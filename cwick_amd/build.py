"""Build libcwick_hip.so for gfx950 with hipcc (cross-compiles without a GPU), and the extension
that hip.py makes its step calls through.

    python -m cwick_amd.build            # compile what changed, link
    python -m cwick_amd.build --force    # recompile everything

The library lands in cwick_amd/lib/ so that it travels with the source tree.
"""
import concurrent.futures as cf
import os
import shutil
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIBDIR = os.path.join(HERE, "lib")
OBJDIR = os.path.join(LIBDIR, "obj")
LIB = os.path.join(LIBDIR, "libcwick_hip.so")
# the step calls of hip.py as a CPython extension (host code only)
CALLS = os.path.join(LIBDIR, "_cwick_calls" + sysconfig.get_config_var("EXT_SUFFIX"))

SOURCES = ["runtime.hip", "misc.hip", "gqa_decode.hip", "gqa_prefill.hip", "mla_roles.hip",
           "indexer.hip", "indexer_band.hip", "topk.hip", "probe.hip", "prep.hip", "mla_prefill64.hip", "mm_select.hip"]

COMMON = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
          "-Wall", "-Wno-unused-function",
          # packed-fp32 VALU forms are kept out of every kernel in this library
          "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
          # the first sixteen dwords of a kernel's arguments arrive in registers with its waves, not
          # through a load that every kernel's first address waits for: 0.3 us of each launch (one
          # decode launch 5.3 -> 5.0 us, split and merge 10.4 -> 9.9)
          "-mllvm", "-amdgpu-kernarg-preload-count=16"]
# the indexer's summation order is a contract: nothing may be fused behind its back
PER_FILE = {"indexer.hip": ["-ffp-contract=off"], "indexer_band.hip": ["-ffp-contract=off"]}


def _hipcc():
    for c in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", "hipcc"):
        if c and (os.path.isabs(c) and os.path.exists(c) or not os.path.isabs(c)):
            return c
    return "hipcc"


def _compile(src, force):
    obj = os.path.join(OBJDIR, src.replace(".hip", ".o"))
    path = os.path.join(CSRC, src)
    deps = [path, os.path.join(HERE, "..", "include", "cwick_hip.h"), os.path.abspath(__file__)]
    deps += [os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hpp")]
    if not force and os.path.exists(obj) and all(
            os.path.getmtime(obj) >= os.path.getmtime(d) for d in deps):
        return obj, ""
    cmd = [_hipcc()] + COMMON + PER_FILE.get(src, []) + ["-c", path, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    log = "\n".join(l for l in (r.stdout + r.stderr).splitlines()
                    if "packed-fp32-ops" not in l)
    if r.returncode != 0:
        raise RuntimeError("hipcc failed for %s:\n%s" % (src, log))
    return obj, log


def _build_calls(force):
    """Needs this interpreter's headers and a host compiler; without them hip.py makes its calls through ctypes."""
    src = os.path.join(CSRC, "binding.cpp")
    deps = [src, os.path.join(HERE, "..", "include", "cwick_hip.h"), os.path.abspath(__file__)]
    if not force and os.path.exists(CALLS) and all(os.path.getmtime(CALLS) >= os.path.getmtime(d) for d in deps):
        return
    cxx = os.environ.get("CXX", "g++").split()
    missing = [what for what, there in (("Python.h", os.path.exists(os.path.join(sysconfig.get_path("include"), "Python.h"))),
                                        (cxx[0], shutil.which(cxx[0]))) if not there]
    if missing:
        print("no %s: the step calls of hip.py go through ctypes" % " and no ".join(missing))
        if os.path.exists(CALLS):
            os.remove(CALLS)                    # (of other sources)
        return
    cmd = cxx + ["-O2", "-std=c++17", "-Wall", "-fPIC", "-shared", "-fvisibility=hidden",
           "-I" + sysconfig.get_path("include"), src, "-o", CALLS]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("compiling %s failed:\n%s" % (src, r.stdout + r.stderr))


def build(force=False, verbose=True):
    os.makedirs(OBJDIR, exist_ok=True)
    with cf.ThreadPoolExecutor(max_workers=min(8, len(SOURCES))) as ex:
        results = list(ex.map(lambda s: _compile(s, force), SOURCES))
    objs = [o for o, _ in results]
    for (_, log), src in zip(results, SOURCES):
        if verbose and log.strip():
            print("[%s]\n%s" % (src, log))
    need_link = force or not os.path.exists(LIB) or any(
        os.path.getmtime(o) > os.path.getmtime(LIB) for o in objs)
    if need_link:
        # only the C ABI of include/cwick_hip.h leaves the library
        cmd = [_hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC",
               "-Wl,--version-script=" + os.path.join(CSRC, "exports.map"), "-o", LIB] + objs
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError("link failed:\n" + r.stdout + r.stderr)
    _build_calls(force)
    if verbose:
        print("built", LIB)
    return LIB


if __name__ == "__main__":
    build(force="--force" in sys.argv)
