"""Builds libluisa_compute_backend_hip.so (gfx950) in-tree with hipcc.

Usage: python -m luisacompute_amd.build [--force]
Objects go to luisacompute_amd/_build/, the library to luisacompute_amd/libluisa_compute_backend_hip.so.
"""
import argparse
import concurrent.futures
import os
import subprocess
import sys

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
CSRC = os.path.join(PKG, "csrc")
OUT_DIR = os.path.join(PKG, "_build")
LIB = os.path.join(PKG, "libluisa_compute_backend_hip.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = os.environ.get("LC_HIP_ARCH", "gfx950")

# -ffp-contract=off: the watertight test must round exactly like the CPU oracle (no FMA
# contraction); box tests call __builtin_fmaf explicitly where fusion is wanted.
# -fgpu-flush-denormals-to-zero: f32 denormals flushed, like the reference CPU backend's
# FTZ/DAZ worker threads (src/rust/luisa_compute_backend_impl/src/cpu/mod.rs:503-516).
# -target-feature -packed-fp32-ops: no v_pk_*_f32 generation.
COMMON = ["-O3", "-std=c++17", "-fPIC", "-ffp-contract=off", "-Wall", "-Wno-unused-function", "-Wno-unused-value", "-Wno-unused-result",
          "-I", os.path.join(ROOT, "include"), "-I", CSRC]
HIP_FLAGS = [f"--offload-arch={ARCH}", "-fgpu-flush-denormals-to-zero",
             "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-munsafe-fp-atomics"]

SOURCES = ["bvh_build.hip", "trace.hip", "radix.hip", "raysort.hip", "pathtracer.hip", "instances.hip", "query.hip", "serve.cpp", "runtime.cpp",
           "workload.cpp", "shader.cpp", "lc_api.cpp"]
HEADERS = ["lc_hip_bvh.h", "lc_hip_internal.h", "box_overlap.h", "traverse.h", "wave_walker.h", "oct_walker.h", "ray_query.h", "lc_hip_rtx.h", "lc_hip_device.h"]
# The device library of run-time shaders: embedded into the library as in-memory headers for hiprtc.
DEVICE_HEADERS = ["lc_hip_device.h", "lc_hip_bvh.h", "lc_hip_rtx.h", "ray_query.h", "traverse.h"]


def _newer(src, dst):
    return not os.path.exists(dst) or os.path.getmtime(src) > os.path.getmtime(dst)


def _compile(src, force):
    path = os.path.join(CSRC, src)
    obj = os.path.join(OUT_DIR, src + ".o")
    deps = [path] + [os.path.join(CSRC, h) for h in HEADERS] + [os.path.join(ROOT, "include", h) for h in ("lc_hip.h", "lc_api.h")]
    if not force and not any(_newer(d, obj) for d in deps):
        return obj
    cmd = [HIPCC] + COMMON + ["-c", path, "-o", obj]
    if src.endswith(".hip"):
        cmd[1:1] = HIP_FLAGS
    subprocess.run(cmd, check=True)
    return obj


def _embed_device_headers():
    """Writes _build/device_headers.cpp: the device library headers as string constants."""
    path = os.path.join(OUT_DIR, "device_headers.cpp")
    delim = "LCHIPDEVHDR"
    parts = ["// generated by luisacompute_amd/build.py from csrc/: the device library for hiprtc",
             "namespace lchip {"]
    names, bodies = [], []
    for h in DEVICE_HEADERS:
        text = open(os.path.join(CSRC, h)).read()
        assert delim not in text
        names.append(f'"{h}"')
        bodies.append(f'R"{delim}({text}){delim}"')
    parts.append("extern const char *const kDeviceHeaderNames[] = {" + ", ".join(names) + "};")
    parts.append("extern const char *const kDeviceHeaderSources[] = {\n" + ",\n".join(bodies) + "};")
    parts.append(f"extern const int kDeviceHeaderCount = {len(DEVICE_HEADERS)};")
    parts.append("} // namespace lchip")
    text = "\n".join(parts) + "\n"
    if not os.path.exists(path) or open(path).read() != text:
        with open(path, "w") as f:
            f.write(text)
    obj = path + ".o"
    if _newer(path, obj):
        subprocess.run([HIPCC] + COMMON + ["-c", path, "-o", obj], check=True)
    return obj


def build(force=True):
    os.makedirs(OUT_DIR, exist_ok=True)
    with concurrent.futures.ThreadPoolExecutor(max_workers=4) as ex:
        objs = list(ex.map(lambda s: _compile(s, force), SOURCES))
    objs.append(_embed_device_headers())
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", LIB + ".tmp"] + objs + ["-lpthread", "-lhiprtc", "-lrocprofiler-sdk-roctx"]
    subprocess.run(cmd, check=True)
    os.replace(LIB + ".tmp", LIB)
    return LIB


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--force", action="store_true")
    a = ap.parse_args()
    print(build(force=a.force))
    sys.exit(0)
