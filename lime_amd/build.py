"""Build liblime_hip.so (HIP, gfx950) in-tree with hipcc.

    python -m lime_amd.build            # compiles lime_amd/csrc/*.hip -> lime_amd/liblime_hip.so

Cross-compiles without a GPU.  Packed-FP32 instructions are disabled on every HIP
translation unit (``-Xclang -target-feature -Xclang -packed-fp32-ops``).
"""
import hashlib
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
CSRC = os.path.join(PKG, "csrc")
INCLUDE = os.path.join(ROOT, "include")
LIB = os.path.join(PKG, "liblime_hip.so")
OBJDIR = os.path.join(PKG, "_build")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"
FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-I", CSRC, "-I", INCLUDE,
    "-Wno-unused-result",
]


def sources():
    return sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hip"))


def build_id(extra=()):
    """What the library is built from: a hash of the sources, headers and flags.  Part of
    ``lime_version``, so that launch choices tuned on one build are not taken over by another."""
    h = hashlib.sha256(" ".join([ARCH, *FLAGS[:FLAGS.index("-I")], *extra]).encode())
    for folder in (CSRC, INCLUDE):
        for name in sorted(f for f in os.listdir(folder) if f.endswith((".hip", ".hpp", ".h"))):
            with open(os.path.join(folder, name), "rb") as f:
                h.update(name.encode() + b"\0" + f.read() + b"\0")
    return h.hexdigest()[:12]


def _compile(src, extra):
    obj = os.path.join(OBJDIR, os.path.basename(src)[:-4] + ".o")
    extra = [*extra, f'-DLIME_BUILD_ID="{build_id(extra)}"'] if os.path.basename(src) == "abi.hip" else extra
    cmd = [HIPCC, *FLAGS, *extra, "-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    return obj, r.stderr


def build(verbose=False, extra=()):
    os.makedirs(OBJDIR, exist_ok=True)
    srcs = sources()
    with ThreadPoolExecutor(max_workers=min(8, len(srcs))) as ex:
        results = list(ex.map(lambda s: _compile(s, list(extra)), srcs))
    objs = [o for o, _ in results]
    if verbose:
        for _, err in results:
            if err.strip():
                print(err, file=sys.stderr)
    tmp = LIB + ".tmp"
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    extra = sys.argv[1:]
    print(build(verbose=True, extra=extra))
