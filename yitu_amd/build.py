"""Builds libyitu_hip.so (gfx950, hipcc), libyitu_host.so and the extension module _ops.so
(g++) in-tree.

Usage: ``python -m yitu_amd.build [-j N] [--force]``. Objects are cached under
``yitu_amd/csrc/build/`` and rebuilt when a source or header is newer.
"""
import argparse
import concurrent.futures
import glob
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(CSRC, "build")
LIB = os.path.join(HERE, "libyitu_hip.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-fvisibility=hidden",
    # packed fp32 instructions are kept out of generated code on purpose
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", "-Wno-unknown-warning-option",
]


def _newest_header():
    hs = glob.glob(os.path.join(CSRC, "*.hpp")) + glob.glob(os.path.join(HERE, "..", "include", "*.h"))
    return max(os.path.getmtime(h) for h in hs)


def _compile(src, force):
    obj = os.path.join(OBJ, os.path.basename(src) + ".o")
    if (not force and os.path.exists(obj) and os.path.getmtime(obj) > os.path.getmtime(src)
            and os.path.getmtime(obj) > _newest_header()):
        return obj
    cmd = [HIPCC] + FLAGS + ["-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    out = "\n".join(l for l in (r.stdout + r.stderr).splitlines()
                    if "packed-fp32-ops" not in l and "is not a recognized feature" not in l)
    if r.returncode != 0:
        raise RuntimeError("hipcc failed for %s:\n%s" % (src, out))
    if out.strip():
        sys.stderr.write(out + "\n")
    return obj


HOST_LIB = os.path.join(HERE, "libyitu_host.so")
# x86-64-v3: built in one container, loaded on another host
HOST_FLAGS = ["-O3", "-mavx2", "-mfma", "-std=c++17", "-fopenmp", "-fPIC", "-fvisibility=hidden",
              "-Wall", "-Wextra", "-shared"]


def build_host(force=False):
    """libyitu_host.so: the CPU graph-preparation code (g++, OpenMP)."""
    srcs = sorted(glob.glob(os.path.join(CSRC, "host", "*.cpp")))
    newest = max([os.path.getmtime(s) for s in srcs] +
                 [os.path.getmtime(os.path.join(HERE, "..", "include", "yitu_host.h"))])
    if not force and os.path.exists(HOST_LIB) and os.path.getmtime(HOST_LIB) > newest:
        return HOST_LIB
    cmd = [os.environ.get("CXX", "g++")] + HOST_FLAGS + srcs + ["-o", HOST_LIB]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("g++ failed:\n" + r.stdout + r.stderr)
    if r.stderr.strip():
        sys.stderr.write(r.stderr)
    return HOST_LIB


OPS_LIB = os.path.join(HERE, "_ops.so")


def _compile_bind(src, force):
    """One source of _ops.so (csrc/bind: the Python-facing side, compiled against torch)."""
    import sysconfig

    from torch.utils import cpp_extension
    obj = os.path.join(OBJ, os.path.basename(src) + ".o")
    deps = glob.glob(os.path.join(CSRC, "bind", "*.hpp")) + \
        glob.glob(os.path.join(HERE, "..", "include", "*.h")) + [src]
    if not force and os.path.exists(obj) and \
            os.path.getmtime(obj) > max(os.path.getmtime(d) for d in deps):
        return obj
    include = cpp_extension.include_paths("cuda") + [sysconfig.get_paths()["include"]]
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-Wall",
           "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", "-DTORCH_API_INCLUDE_EXTENSION_H",
           "-DTORCH_EXTENSION_NAME=_ops"]
    for path in include:
        cmd += ["-isystem", path]
    r = subprocess.run(cmd + ["-c", src, "-o", obj], capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("g++ failed for %s:\n%s" % (src, r.stdout + r.stderr))
    if r.stderr.strip():
        sys.stderr.write(r.stderr)
    return obj


def _link_bind(objs):
    from torch.utils import cpp_extension
    dirs = cpp_extension.library_paths("cuda")
    cmd = [os.environ.get("CXX", "g++"), "-shared", "-o", OPS_LIB] + objs + \
        ["-L" + HERE, "-l:libyitu_hip.so", "-Wl,-rpath,$ORIGIN"]
    for path in dirs:
        cmd += ["-L" + path, "-Wl,-rpath," + path]
    cmd += ["-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_hip", "-ltorch", "-ltorch_python"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link of _ops.so failed:\n" + r.stdout + r.stderr)


def build(force=False, jobs=8):
    build_host(force)
    os.makedirs(OBJ, exist_ok=True)
    srcs = sorted(glob.glob(os.path.join(CSRC, "*.hip")))
    with concurrent.futures.ThreadPoolExecutor(max_workers=jobs) as ex:
        binds = [ex.submit(_compile_bind, s, force)
                 for s in sorted(glob.glob(os.path.join(CSRC, "bind", "*.cpp")))]
        objs = list(ex.map(lambda s: _compile(s, force), srcs))
        binds = [b.result() for b in binds]
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB] + objs
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n" + r.stdout + r.stderr)
    _link_bind(binds)
    return LIB


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("-j", type=int, default=8)
    ap.add_argument("--force", action="store_true")
    a = ap.parse_args()
    print(build(force=a.force, jobs=a.j))
