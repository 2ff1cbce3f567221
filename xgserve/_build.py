"""In-tree native build: C++ runtime core (g++) and HIP/CDNA4 kernels (hipcc, gfx950).

Both libraries are pybind11 modules written next to the package so that the
built ``.so`` travels with the repository snapshot to the GPU box:

  xgserve/_runtime*.so   <- csrc/runtime/*.cpp   (host C++17, no GPU deps)
  xgserve/_kernels*.so   <- csrc/kernels/*.hip + csrc/comm/*.hip  (hipcc --offload-arch=gfx950)
  xgserve/_mixers*.so    <- csrc/mixers/*  (the sequence-mixer kernels of the stateful /
                            latent-cache layers; a library of its own, so a model made
                            only of those builds in seconds)

The kernel library is linked against the HIP runtime that PyTorch itself loads
(``torch/lib/libamdhip64.so``, same SONAME as /opt/rocm's), so one HIP runtime
instance serves torch and our kernels. Kernels take raw device pointers and the
current hipStream_t from Python -- no torch C++ headers, no hipify.

Usage:  python -m xgserve._build [--force] [--jobs N] [--only runtime|kernels|mixers]
"""
from __future__ import annotations

import argparse
import concurrent.futures as cf
import hashlib
import os
import re
import shutil
import struct
import subprocess
import sys
import sysconfig
import tempfile
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent
PKG = ROOT / "xgserve"
CSRC = ROOT / "csrc"
BUILD = ROOT / "build" / "obj"
EXT = sysconfig.get_config_var("EXT_SUFFIX") or ".so"
ARCH = os.environ.get("XGS_OFFLOAD_ARCH", "gfx950")


def _pybind_includes() -> list:
    import pybind11
    return [f"-I{pybind11.get_include()}", f"-I{sysconfig.get_paths()['include']}"]


def _torch_lib() -> str:
    import importlib.util
    spec = importlib.util.find_spec("torch")
    return str(Path(spec.origin).parent / "lib")


def _digest(paths, flags) -> str:
    h = hashlib.sha256()
    for p in sorted(paths):
        h.update(str(p).encode())
        h.update(Path(p).read_bytes())
    h.update(" ".join(flags).encode())
    return h.hexdigest()[:16]


def _run(cmd):
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if r.returncode != 0:
        sys.stderr.write(" ".join(cmd) + "\n" + r.stdout)
        raise RuntimeError(f"build step failed: {cmd[0]} ... {cmd[-1]}")
    return r.stdout


def _needs(out: Path, stamp: str, force: bool) -> bool:
    st = out.with_suffix(out.suffix + ".stamp")
    return force or not out.exists() or not st.exists() or st.read_text() != stamp


def _write_stamp(out: Path, stamp: str):
    out.with_suffix(out.suffix + ".stamp").write_text(stamp)


# hipcc -O3 forms packed-fp32 instructions from plain float code by itself; they stay off
NO_PK_F32 = ["-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]


# tile_linear.h's kernels keep their accumulators in registers that their statements name, and nothing tells the compiler that these
# hold something between two statements. What it made is looked at instead: a register of that file may only be written by a product
# onto itself (or onto zero), and only be read into a vector register; and nothing may be spilled.
NAMED_ACCUMULATORS = "tile_linear_kernel"
_PRODUCT = re.compile(r"v_mfma_\w+ (a\[\d+:\d+\]), v\[\d+:\d+\], v\[\d+:\d+\], (a\[\d+:\d+\]|0)$")
_TAKE = re.compile(r"v_accvgpr_read_b32 v\d+, a\d+$")
_ACCUMULATOR = re.compile(r"\ba(\[|\d)")


def check_accumulators(listing: str) -> int:
    """The kernels with named accumulators in a disassembly (llvm-objdump -d); raises where one lets the compiler at them."""
    kernel, count = None, 0
    for line in listing.splitlines():
        if line.endswith(">:"):
            name = line[line.index("<") + 1:-2]
            kernel = name if NAMED_ACCUMULATORS in name else None
            count += kernel is not None
            continue
        if kernel is None:
            continue
        op = line.split("//")[0].strip()
        if op.startswith("scratch_"):
            raise RuntimeError(f"{kernel}: spilled registers ({op})")
        if _ACCUMULATOR.search(op):
            m = _PRODUCT.match(op)
            if not (m and m[2] in (m[1], "0")) and not _TAKE.match(op):
                raise RuntimeError(f"{kernel}: an accumulator that is not the compiler's to use ({op})")
    return count


def _device_code(library: Path):
    """The library's code objects for ARCH."""
    data = library.read_bytes()
    at = data.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        entry = at + 32
        for _ in range(struct.unpack_from("<Q", data, at + 24)[0]):
            offset, size, length = struct.unpack_from("<QQQ", data, entry)
            if ARCH.encode() in data[entry + 24:entry + 24 + length]:
                yield data[at + offset:at + offset + size]
            entry += 24 + length
        at = data.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 24)


def check_library_accumulators(library: Path) -> int:
    """check_accumulators of all kernels of a built library."""
    objdump = shutil.which("llvm-objdump") or os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm/bin/llvm-objdump")
    count = 0
    for code in _device_code(library):
        if NAMED_ACCUMULATORS.encode() in code:
            with tempfile.NamedTemporaryFile(suffix=".elf") as f:
                f.write(code)
                f.flush()
                count += check_accumulators(_run([objdump, "-d", f.name]))
    return count


def build_runtime(force: bool = False, jobs: int = 8, extra=()) -> Path:
    srcs = sorted((CSRC / "runtime").glob("*.cpp"))
    hdrs = sorted((CSRC / "runtime").glob("*.h"))
    out = PKG / f"_runtime{EXT}"
    flags = ["-O3", "-std=c++17", "-fPIC", "-Wall", "-Wno-sign-compare", "-fvisibility=hidden", *extra]
    stamp = _digest(srcs + hdrs, flags)
    if not _needs(out, stamp, force):
        return out
    obj_dir = BUILD / "runtime"
    obj_dir.mkdir(parents=True, exist_ok=True)
    inc = _pybind_includes() + [f"-I{CSRC / 'runtime'}"]

    def cc(src):
        o = obj_dir / (src.stem + ".o")
        _run(["g++", *flags, *inc, "-c", str(src), "-o", str(o)])
        return o

    with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
        objs = list(ex.map(cc, srcs))
    _run(["g++", "-shared", *flags, *map(str, objs), "-o", str(out)])
    _write_stamp(out, stamp)
    return out


def build_kernels(force: bool = False, jobs: int = 8, probes: bool = False) -> Path:
    """probes: also compile the anatomy-probe kernels (gemm_pf without DMA / MFMA,
    decode attention without prologue / key loop). They are measurement builds
    (bench/pf_gemm_bench.py --probe, bench/decode_cold.py --probe), never selected
    by a plan, so the default library leaves them out."""
    srcs = sorted((CSRC / "kernels").glob("*.hip")) + sorted((CSRC / "comm").glob("*.hip"))
    hdrs = sorted((CSRC / "kernels").glob("*.h")) + sorted((CSRC / "comm").glob("*.h"))
    cpp = sorted((CSRC / "kernels").glob("*.cpp"))
    out = PKG / f"_kernels{EXT}"
    flags = ["-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}", "-fvisibility=hidden",
             "-munsafe-fp-atomics", "-Wno-unused-result", *NO_PK_F32] + (["-DXGK_PROBES=1"] if probes else [])
    stamp = _digest(srcs + hdrs + cpp, flags)
    if not _needs(out, stamp, force):
        return out
    obj_dir = BUILD / "kernels"
    obj_dir.mkdir(parents=True, exist_ok=True)
    inc = _pybind_includes() + [f"-I{CSRC / 'kernels'}", f"-I{CSRC / 'comm'}"]

    def cc(src):
        o = obj_dir / (src.stem + ".o")
        _run(["hipcc", *flags, *inc, "-c", str(src), "-o", str(o)])
        return o

    with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
        objs = list(ex.map(cc, srcs + cpp))
    tl = _torch_lib()
    _run(["hipcc", "-shared", f"--offload-arch={ARCH}", "-fPIC", *map(str, objs),
          f"-L{tl}", f"-Wl,-rpath,{tl}", "-lamdhip64", "-o", str(out)])
    _write_stamp(out, stamp)
    return out


def build_mixers(force: bool = False, jobs: int = 8) -> Path:
    # (gemm_pf: the prompt-sized expert products, the same source as in the kernel library)
    srcs = sorted((CSRC / "mixers").glob("*.hip")) + [CSRC / "kernels" / "gemm_pf.hip"]
    cpp = sorted((CSRC / "mixers").glob("*.cpp"))
    hdrs = [CSRC / "kernels" / h for h in ("common.h", "glds.h", "glu.h")] + sorted((CSRC / "mixers").glob("*.h"))
    out = PKG / f"_mixers{EXT}"
    flags = ["-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}", "-fvisibility=hidden", "-Wno-unused-result",
             *NO_PK_F32]
    stamp = _digest(srcs + hdrs + cpp, flags)
    if not _needs(out, stamp, force):
        return out
    obj_dir = BUILD / "mixers"
    obj_dir.mkdir(parents=True, exist_ok=True)
    inc = _pybind_includes() + [f"-I{CSRC / 'kernels'}", f"-I{CSRC / 'mixers'}"]

    def cc(src):
        o = obj_dir / (src.stem + ".o")
        _run(["hipcc", *flags, *inc, "-c", str(src), "-o", str(o)])
        return o

    with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
        objs = list(ex.map(cc, srcs + cpp))
    tl = _torch_lib()
    _run(["hipcc", "-shared", f"--offload-arch={ARCH}", "-fPIC", *map(str, objs),
          f"-L{tl}", f"-Wl,-rpath,{tl}", "-lamdhip64", "-o", str(out)])
    try:
        if check_library_accumulators(out) == 0:
            raise RuntimeError(f"no {NAMED_ACCUMULATORS} found in {out.name}")
    except Exception:
        out.unlink()
        raise
    _write_stamp(out, stamp)
    return out


def build_all(force: bool = False, jobs: int = 8):
    return build_runtime(force, jobs), build_kernels(force, jobs), build_mixers(force, jobs)


def main(argv=None):
    ap = argparse.ArgumentParser()
    ap.add_argument("--force", action="store_true")
    ap.add_argument("--jobs", type=int, default=min(8, os.cpu_count() or 4))
    ap.add_argument("--only", choices=["runtime", "kernels", "mixers"], default=None)
    ap.add_argument("--probes", action="store_true", help="include the anatomy-probe kernels (measurement builds)")
    a = ap.parse_args(argv)
    if a.only in (None, "runtime"):
        print("runtime:", build_runtime(a.force, a.jobs))
    if a.only in (None, "kernels"):
        print("kernels:", build_kernels(a.force, a.jobs, a.probes))
    if a.only in (None, "mixers"):
        print("mixers:", build_mixers(a.force, a.jobs))


if __name__ == "__main__":
    main()
