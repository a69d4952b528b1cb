"""Builds libnntile_hip_sdpa.so (hand-written HIP for gfx950) and the native
front-end of the Python binding (_front.so) in-tree.

    python -m nntile_amd.build [--force]
"""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libnntile_hip_sdpa.so")
SOURCES = ["sdpa_prefill_16bit.hip", "sdpa_prefill_fp32.hip", "sdpa_prefill_f16x2.hip",
           "sdpa_decode_16bit.hip", "sdpa_decode_fp32.hip", "sdpa_bwd_16bit.hip", "rope.hip", "transpose.hip", "kv_cache.hip", "mask_classify.hip",
           "accumulate_attn_output.hip", "sdpa_parts_merge.hip", "capi.hip"]
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
         "-Wall", "-Wno-unused-function"]
FRONT = os.path.join(HERE, "_front.so")
ROCM = os.path.dirname(os.path.dirname(HIPCC)) if os.path.isabs(HIPCC) else "/opt/rocm"


def _stale(obj, src):
    if not os.path.exists(obj):
        return True
    t = os.path.getmtime(obj)
    deps = [src] + [os.path.join(CSRC, f) for f in os.listdir(CSRC)
                    if f.endswith(".hpp")]
    deps.append(os.path.join(HERE, "..", "include", "nntile_hip_sdpa.h"))
    return any(os.path.getmtime(d) > t for d in deps)


def front_tag():
    """What the front-end is compiled against: it reads torch's C++ objects and
    the interpreter's, so it fits one build of each."""
    import platform
    import torch
    return "torch %s, Python %s" % (torch.__version__, platform.python_version())


def _front_stale():
    if _stale(FRONT, os.path.join(CSRC, "front.cpp")):
        return True
    with open(FRONT, "rb") as f:
        return ("nntile_front for %s;" % front_tag()).encode() not in f.read()


def _front_command():
    """g++ on the binding's front-end: host code on torch's headers, linked
    against the kernel library beside it."""
    import sysconfig
    import torch
    from torch.utils.cpp_extension import include_paths, library_paths
    inc = include_paths() + [os.path.join(ROCM, "include"), sysconfig.get_paths()["include"]]
    lib = library_paths()
    return (["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden",
             "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
             '-DNNTILE_FRONT_TAG="%s"' % front_tag(),
             "-D_GLIBCXX_USE_CXX11_ABI=%d" % torch._C._GLIBCXX_USE_CXX11_ABI]
            + [x for d in inc for x in ("-isystem", d)]
            + [os.path.join(CSRC, "front.cpp"), "-o", FRONT]
            + ["-L" + d for d in lib] + ["-L" + HERE, "-lnntile_hip_sdpa", "-ltorch_python",
                                         "-ltorch_cpu", "-lc10", "-lc10_hip",
                                         "-Wl,-rpath,$ORIGIN"])


def build(force=False, verbose=True):
    objs = []
    procs = []
    for name in SOURCES:
        src = os.path.join(CSRC, name)
        obj = os.path.join(CSRC, name.replace(".hip", ".o"))
        objs.append(obj)
        if force or _stale(obj, src):
            cmd = [HIPCC] + FLAGS + ["-c", src, "-o", obj]
            if verbose:
                print(" ".join(cmd), flush=True)
            procs.append((name, subprocess.Popen(
                cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)))
    failed = False
    for name, proc in procs:
        out = proc.communicate()[0].decode()
        out = "\n".join(l for l in out.splitlines()
                        if "packed-fp32-ops" not in l and l.strip())
        if out and verbose:
            print(out)
        if proc.returncode != 0:
            failed = True
            print("FAILED: " + name, file=sys.stderr)
    if failed:
        raise RuntimeError("hipcc failed")
    if force or procs or not os.path.exists(LIB):
        cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-o", LIB] + objs
        if verbose:
            print(" ".join(cmd), flush=True)
        subprocess.check_call(cmd)
    if force or _front_stale():
        cmd = _front_command()
        if verbose:
            print(" ".join(cmd), flush=True)
        subprocess.check_call(cmd)
    return LIB


if __name__ == "__main__":
    build(force="--force" in sys.argv)
