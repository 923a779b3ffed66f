"""Builds libash_hip.so (gfx950) in-tree with hipcc.

    python torch-ash_amd/build.py            # rebuild when sources are newer
    python torch-ash_amd/build.py --force    # always rebuild

and beside it _ash_host.so, the host side of its calls on torch tensors (plain
C++ against the installed torch).  The libraries land in torch-ash_amd/ash/lib/ so that they travel with the source
tree; nothing is installed into site-packages.
"""
import argparse
import os
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OUT_DIR = os.path.join(HERE, "ash", "lib")
OUT = os.path.join(OUT_DIR, "libash_hip.so")
HOST_SOURCE = os.path.join(CSRC, "ash_host.cpp")
HOST_OUT = os.path.join(OUT_DIR, "_ash_host.so")
SOURCES = ["ash_map.hip", "ash_bulk.hip", "ash_query.hip", "ash_fusion.hip", "ash_mesh.hip",
           "ash_rays.hip", "ash_conv.hip", "ash_surface.hip"]
# compiled once for every width of rows (channels): device code of its own, which the
# runtime loads where it is used
ROWS_SOURCE, ROW_WIDTHS = "ash_rows.hip", (1, 2, 3, 4, 5, 6, 7, 8, 12, 16)
HEADERS = [
    os.path.join(CSRC, "ash_probe.h"),
    os.path.join(CSRC, "ash_dev.h"),
    os.path.join(CSRC, "ash_query.h"),
    os.path.join(CSRC, "ash_table.h"),
    os.path.join(CSRC, "ash_walk.h"),
    os.path.join(CSRC, "ash_mc_table.h"),
    os.path.join(HERE, os.pardir, "include", "ash_hip.h"),
]
ARCH = "gfx950"


def hipcc_path() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (set HIPCC or add /opt/rocm/bin to PATH)")


def compile_flags():
    return [
        "-O3",
        "-std=c++17",
        "-fPIC",
        f"--offload-arch={ARCH}",
        "-Xclang",
        "-target-feature",
        "-Xclang",
        "-packed-fp32-ops",
        "-Wall",
        "-Wno-unused-function",
    ]


def units():
    """(source, object, flags of its own) of everything that is compiled."""
    return [(s, s.replace(".hip", ".o"), []) for s in SOURCES] + [
        (ROWS_SOURCE, f"ash_rows_{width}.o", [f"-DASH_ROW_WIDTH={width}"]) for width in ROW_WIDTHS]


def source_fingerprint() -> str:
    """SHA-256 over the kernel sources (names and contents of csrc/*.hip and
    csrc/*.h).  It is compiled into the library (ash_source_fingerprint), so
    that a benchmark or a test can tell a library that was not built from the
    sources beside it."""
    import hashlib

    h = hashlib.sha256()
    for name in sorted(os.listdir(CSRC)):
        if name.endswith((".hip", ".h")):
            h.update(name.encode())
            with open(os.path.join(CSRC, name), "rb") as f:
                h.update(f.read())
    return h.hexdigest()


def host_fingerprint() -> str:
    """The same for the host module (its source and the header of the C ABI),
    compiled in as _ash_host.source_fingerprint."""
    import hashlib

    h = hashlib.sha256()
    for path in (HOST_SOURCE, HEADERS[-1]):
        h.update(os.path.basename(path).encode())
        with open(path, "rb") as f:
            h.update(f.read())
    return h.hexdigest()


def _older(out, deps) -> bool:
    if not os.path.exists(out):
        return True
    built = os.path.getmtime(out)
    return any(os.path.getmtime(d) > built for d in [*deps, os.path.abspath(__file__)])


def is_stale() -> bool:
    return _older(OUT, [os.path.join(CSRC, s) for s in [*SOURCES, ROWS_SOURCE]] + HEADERS)


def host_is_stale() -> bool:
    return _older(HOST_OUT, [HOST_SOURCE, HEADERS[-1]])


def host_command(out: str):
    import sysconfig

    import torch
    from torch.utils import cpp_extension

    libs = os.path.join(os.path.dirname(torch.__file__), "lib")
    includes = [*cpp_extension.include_paths(), os.environ.get("ROCM_PATH", "/opt/rocm") + "/include",
                sysconfig.get_paths()["include"]]
    return [
        os.environ.get("CXX") or shutil.which("g++") or "c++",
        "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall",
        "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", "-DTORCH_API_INCLUDE_EXTENSION_H",
        f'-DASH_HOST_FINGERPRINT="{host_fingerprint()}"',
        f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
        *[arg for path in dict.fromkeys(includes) for arg in ("-isystem", path)],
        HOST_SOURCE, "-o", out, f"-L{libs}", "-ltorch", "-ltorch_cpu", "-ltorch_python", "-lc10",
        "-lc10_hip", f"-Wl,-rpath,{libs}",
    ]


def build_host(verbose: bool = True):
    """Starts the compiler; returns what finishes the job."""
    os.makedirs(OUT_DIR, exist_ok=True)
    tmp = HOST_OUT + ".tmp"
    cmd = host_command(tmp)
    if verbose:
        print(" ".join(cmd), flush=True)
    process = subprocess.Popen(cmd)

    def finish():
        if process.wait() != 0:
            raise RuntimeError("compile failed: " + " ".join(cmd))
        os.replace(tmp, HOST_OUT)

    return finish


def build(force: bool = False, verbose: bool = True) -> str:
    finish_host = build_host(verbose) if force or host_is_stale() else lambda: None
    try:
        return build_kernels(force, verbose)
    finally:
        finish_host()


def build_kernels(force: bool, verbose: bool) -> str:
    if not force and not is_stale():
        return OUT
    os.makedirs(OUT_DIR, exist_ok=True)
    hipcc = hipcc_path()
    stamp = f'-DASH_SOURCE_FINGERPRINT="{source_fingerprint()}"'
    objs = []
    procs = []
    for src, name, flags in units():
        obj = os.path.join(OUT_DIR, name)
        cmd = [hipcc, *compile_flags(), *flags, "-c", os.path.join(CSRC, src), "-o", obj]
        if src == "ash_map.hip":
            cmd.insert(1, stamp)
        if verbose:
            print(" ".join(cmd), flush=True)
        procs.append((cmd, subprocess.Popen(cmd)))
        objs.append(obj)
    for cmd, p in procs:
        if p.wait() != 0:
            raise RuntimeError("compile failed: " + " ".join(cmd))
    tmp = OUT + ".tmp"
    link = [hipcc, "-shared", "-fPIC", f"--offload-arch={ARCH}", *objs, "-o", tmp]
    if verbose:
        print(" ".join(link), flush=True)
    subprocess.check_call(link)
    os.replace(tmp, OUT)
    for o in objs:
        os.remove(o)
    return OUT


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--force", action="store_true")
    args = ap.parse_args()
    print(build(force=args.force))
    sys.exit(0)
