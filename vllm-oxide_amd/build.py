"""Builds liboxide_paged_kv.so (gfx950 HIP kernels + C ABI + C++ host layer).

The library is built in-tree, next to this file, with plain hipcc calls (no
cmake, no JIT cache), so the .so travels with the source tree.  Every call
recompiles.  Counterpart of the reference's crates/vllm-oxide/build.rs:1-30
(nvcc via cudaforge -> static lib); here hipcc --offload-arch=gfx950 -> the
shared library Python loads with ctypes, plus the same objects archived as
liboxide_paged_kv.a, and the Python ops' native module against torch's headers (where
torch and g++ are there).  rust/oxide-paged-kv-sys/build.rs and vllm-oxide_amd/Makefile
compile the same library sources with the same flags.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG = Path(__file__).resolve().parent
REPO = PKG.parent
CSRC = PKG / "csrc"
HOST = PKG / "host"
INCLUDE = REPO / "include"
BUILD = PKG / "_build"
LIB = PKG / "liboxide_paged_kv.so"
STATIC_LIB = PKG / "liboxide_paged_kv.a"
# The Python ops' native front end: a CPython module against torch's C++ headers, named
# for the interpreter it is built for.
NATIVE_SRC = PKG / "pyext" / "native_ops.cpp"
NATIVE_LIB = PKG / "oxide_paged_kv" / f"_native{sysconfig.get_config_var('EXT_SUFFIX') or '.so'}"
HOST_TEST_SRC = REPO / "tests" / "cpp" / "test_host.cpp"
HOST_TEST_BIN = REPO / "tests" / "cpp" / "build" / "test_host"
HOST_TEST_STAMP = HOST_TEST_BIN.with_suffix(".sources.sha256")
# Per-kernel register, scratch and LDS use reported by the compiler for the last build.
RESOURCES = BUILD / "kernel_resources.json"

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"

# -packed-fp32-ops off: no v_pk_{add,mul,fma}_f32 in any kernel.
HIP_FLAGS = [
    "-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function",
]


def _sources() -> list[Path]:
    return sorted(CSRC.glob("*.hip")) + sorted(CSRC.glob("*.cpp")) + sorted(HOST.glob("*.cpp"))


def _parse_resources(text: str) -> dict:
    """Kernel resource remarks (-Rpass-analysis=kernel-resource-usage) -> {kernel: {field: value}}."""
    import re

    out, cur = {}, None
    for line in text.splitlines():
        m = re.search(r"remark: Function Name: (\S+)", line)
        if m:
            cur = out.setdefault(m.group(1), {})
            continue
        m = re.search(r"remark:\s+([A-Za-z][A-Za-z /\[\]]*?):\s+(\S+) \[-Rpass-analysis", line)
        if m and cur is not None:
            v = m.group(2)
            cur[m.group(1).strip()] = int(v) if v.lstrip("-").isdigit() else v
    return out


def _compile(src: Path):
    obj = BUILD / (src.parent.name + "_" + src.stem + ".o")
    cmd = [HIPCC, *HIP_FLAGS, "-I", str(INCLUDE), "-I", str(CSRC), "-I", str(HOST)]
    if src.suffix == ".cpp":
        cmd += ["-x", "hip"]
    else:
        cmd += ["-Rpass-analysis=kernel-resource-usage"]
    cmd += ["-c", str(src), "-o", str(obj)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src.name}:\n{r.stdout}\n{r.stderr}")
    return obj, _parse_resources(r.stderr)


def build_native() -> Path | None:
    """The ops' native module with the host compiler; it links torch's libraries, which
    `import torch` has loaded by then.  None without torch or g++: the ops then call the
    library through ctypes only."""
    for old in NATIVE_LIB.parent.glob("_native*.so"):  # never a module of earlier sources
        old.unlink()
    try:
        import torch
    except ImportError as e:
        print(f"native front end not built: {e}", file=sys.stderr)
        return None
    if shutil.which("g++") is None:
        print("native front end not built: no g++", file=sys.stderr)
        return None
    t = Path(torch.__file__).resolve().parent
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}",
           f'-DOXIDE_TORCH_VERSION="{torch.__version__}"', "-I", str(INCLUDE),
           "-isystem", str(t / "include"), "-isystem", str(t / "include" / "torch" / "csrc" / "api" / "include"),
           "-isystem", "/opt/rocm/include", "-isystem", sysconfig.get_paths()["include"], str(NATIVE_SRC),
           "-o", str(NATIVE_LIB), "-L", str(t / "lib"), "-ltorch_python", "-ltorch_cpu", "-lc10", "-lc10_hip"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"g++ failed for {NATIVE_SRC.name}:\n{r.stdout}\n{r.stderr}")
    return NATIVE_LIB


def build(verbose: bool = False) -> Path:
    BUILD.mkdir(exist_ok=True)
    srcs = _sources()
    with ThreadPoolExecutor(max_workers=min(9, len(srcs) + 1)) as ex:
        native = ex.submit(build_native)
        results = list(ex.map(_compile, srcs))
    objs = [o for o, _ in results]
    import json

    resources = {}
    for _, res in results:
        resources.update(res)
    RESOURCES.write_text(json.dumps(resources, indent=1, sort_keys=True))
    cmd = [HIPCC, "-shared", "-fPIC", f"--offload-arch={ARCH}", "-o", str(LIB), *map(str, objs)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    # The same objects as a static archive (what the Rust crate's build.rs and the
    # Makefile produce) for hosts that link the kernels statically.
    STATIC_LIB.unlink(missing_ok=True)
    r = subprocess.run(["ar", "rcs", str(STATIC_LIB), *map(str, objs)], capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"ar failed:\n{r.stdout}\n{r.stderr}")
    build_host_test()
    native.result()  # last: the C libraries do not need it
    if verbose:
        print(f"built {LIB}")
    return LIB


def host_test_digest() -> str:
    """Digest of what the host test binary is built from: its source, the host layer,
    the header and the library it links (content, not mtimes, which a copied tree may
    not keep)."""
    import hashlib

    files = [HOST_TEST_SRC, INCLUDE / "oxide_paged_kv.h", LIB, *sorted(HOST.glob("*"))]
    h = hashlib.sha256()
    for f in files:
        h.update(f.name.encode())
        h.update(f.read_bytes() if f.exists() else b"<missing>")
    return h.hexdigest()


def host_test_current() -> bool:
    return HOST_TEST_BIN.exists() and HOST_TEST_STAMP.exists() and \
        HOST_TEST_STAMP.read_text().strip() == host_test_digest()


def build_host_test() -> Path:
    """C++ test binary of the host layer (tests/cpp/test_host.cpp), linked to the library;
    records the digest of its sources next to it."""
    HOST_TEST_BIN.parent.mkdir(parents=True, exist_ok=True)
    cmd = [HIPCC, *HIP_FLAGS, "-I", str(INCLUDE), "-I", str(HOST), "-I", str(PKG / "csrc"), str(HOST_TEST_SRC), "-o",
           str(HOST_TEST_BIN), "-L", str(PKG), "-loxide_paged_kv", f"-Wl,-rpath,{PKG}",
           "-Wl,-rpath,$ORIGIN/../../../vllm-oxide_amd"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {HOST_TEST_SRC.name}:\n{r.stdout}\n{r.stderr}")
    HOST_TEST_STAMP.write_text(host_test_digest())
    return HOST_TEST_BIN


if __name__ == "__main__":
    if sys.argv[1:] == ["native"]:
        sys.exit(0 if build_native() else 1)
    build(verbose=True)
    sys.exit(0)
