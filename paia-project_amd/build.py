"""Build libpaia_gemv.so (HIP, gfx950) and the torch.library extension, in-tree.

    python paia-project_amd/build.py            # both
    python paia-project_amd/build.py --lib      # only the HIP library

Outputs (git-ignored, shipped with the tree):
    paia-project_amd/build/libpaia_gemv.so          C ABI declared in include/paia_gemv.h
    paia-project_amd/build/libpaia_gemv_torch.so    torch.ops.paia_gemv.* (links libpaia_gemv.so via $ORIGIN)
    paia-project_amd/build/libpaia_probe.so         measurement kernels of the benchmark harness

Replaces src/paia_gemv/build.sh (nvcc, static cudart). Every HIP source is compiled for gfx950 only, with packed
fp32 VALU instructions disabled (-Xclang -target-feature -Xclang -packed-fp32-ops); translation units build in
parallel and are linked with hipcc.
"""
from __future__ import annotations

import argparse
import concurrent.futures as cf
import os
import shutil
import subprocess
import sys
from pathlib import Path

PKG = Path(__file__).resolve().parent
ROOT = PKG.parent
CSRC = PKG / "csrc"
INCLUDE = ROOT / "include"
BUILD = PKG / "build"
OBJ = BUILD / "obj"
LIB = BUILD / "libpaia_gemv.so"
TORCH_LIB = BUILD / "libpaia_gemv_torch.so"
PROBE_LIB = BUILD / "libpaia_probe.so"

ROCM = Path(os.environ.get("ROCM_PATH", "/opt/rocm"))
HIPCC = str(ROCM / "bin" / "hipcc")
ARCH = "gfx950"
HIP_FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC", "-fvisibility=hidden",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function",
    f"-I{INCLUDE}", f"-I{CSRC}",
]
HIP_SOURCES = ["gemv_runtime.hip", "gemv_bf16.hip", "gemv_fp8.hip", "gemv_int4.hip", "gemv_dequant.hip",
               "gemv_select.hip", "quantize.hip", "gemv_batch.hip",
               "gemv_tile.hip"]


def _run(cmd, quiet_warn=True):
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = r.stdout
    if quiet_warn:   # the host pass does not know the device-only feature flag: harmless, drop the noise
        out = "\n".join(l for l in out.splitlines() if "packed-fp32-ops" not in l)
    if r.returncode != 0:
        raise RuntimeError(f"command failed ({r.returncode}): {' '.join(cmd)}\n{out}")
    return out


TUNED = PKG / "tuned" / "mi355x.json"
GEN = BUILD / "gen"
TUNED_KINDS = {"shapes": 0, "fp8_shapes": 1, "int4_shapes": 2, "int4zp_shapes": 3}
# small-batch sections (no reference counterpart): "MxNxK" -> {"variant": {P,U,W,S,X}}
TUNED_BATCH_KINDS = {"batch_shapes": 0, "fp8_batch_shapes": 1, "int4_batch_shapes": 2, "int4zp_batch_shapes": 3}


def gen_tuned(src: Path = TUNED, out_dir: Path = GEN) -> Path:
    """tuned/mi355x.json (reference tuned-file schema: section -> "NxK" -> {"variant": {R,U,W,S,H}}) -> the C rows
    of the library's per-shape table (gemv_tuned.inc)."""
    import json
    rows = []
    if src.exists():
        data = json.loads(src.read_text())
        for sec, kind in TUNED_KINDS.items():
            for key, e in sorted(data.get(sec, {}).items()):
                N, K = map(int, key.split("x"))
                v = e["variant"]
                rows.append(f"    {{{kind}, {N}, {K}, {v['R']}, {v['U']}, {v['W']}, {v.get('S', 0)}, {v['H']}}},")
    out_dir.mkdir(parents=True, exist_ok=True)
    out = out_dir / "gemv_tuned.inc"
    text = "// generated by build.py from tuned/mi355x.json: {kind, N, K, R, U, W, S, H}\n" + "\n".join(rows) + "\n"
    if not out.exists() or out.read_text() != text:
        out.write_text(text)
    brows = []
    if src.exists():
        for sec, kind in TUNED_BATCH_KINDS.items():
            for key, e in sorted(data.get(sec, {}).items()):
                M, N, K = map(int, key.split("x"))
                v = e["variant"]
                brows.append(f"    {{{kind}, {M}, {N}, {K}, {v['P']}, {v['U']}, {v['W']}, {v['S']}, {v['X']}}},")
    bout = out_dir / "gemv_batch_tuned.inc"
    btext = ("// generated by build.py from tuned/mi355x.json: {kind, M, N, K, P, U, W, S, X}\n" + "\n".join(brows)
             + "\n")
    if not bout.exists() or bout.read_text() != btext:
        bout.write_text(btext)
    return out


def build_lib(jobs: int | None = None, out: Path = LIB, defines=()) -> Path:
    """Compile every HIP translation unit for gfx950 and link libpaia_gemv.so (always rebuilds). `defines` (e.g.
    ["PAIA_GEMV_MAX_WAVES_PER_CU=16"]) and `out` build a differently tuned copy elsewhere for experiments."""
    obj_dir = OBJ if out == LIB else out.parent / "obj"
    obj_dir.mkdir(parents=True, exist_ok=True)
    srcs = [CSRC / s for s in HIP_SOURCES]
    extra = [f"-D{d}" for d in defines] + [f"-I{gen_tuned().parent}"]
    jobs = jobs or min(len(srcs), max(1, min(16, os.cpu_count() or 1)))

    def comp(src: Path) -> Path:
        obj = obj_dir / (src.stem + ".o")
        _run([HIPCC, *HIP_FLAGS, *extra, "-c", str(src), "-o", str(obj)])
        return obj

    with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
        objs = list(ex.map(comp, srcs))
    tmp = out.with_suffix(".so.tmp")
    _run([HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs)])
    os.replace(tmp, out)
    return out


def build_probe() -> Path:
    """The benchmark harness's measurement kernels (streaming-read probe, empty kernel): libpaia_probe.so."""
    tmp = PROBE_LIB.with_suffix(".so.tmp")
    _run([HIPCC, *HIP_FLAGS, "-shared", "-o", str(tmp), str(CSRC / "bench_probe.hip")])
    os.replace(tmp, PROBE_LIB)
    return PROBE_LIB


def build_torch_ext() -> Path:
    """Compile the torch.library ops (host C++ only) against torch's headers, linking libpaia_gemv.so."""
    import torch
    from torch.utils import cpp_extension as ce

    tdir = Path(torch.__file__).resolve().parent
    abi = int(torch._C._GLIBCXX_USE_CXX11_ABI)
    cxx = shutil.which("g++") or "g++"
    cmd = [cxx, "-O2", "-std=c++17", "-fPIC", "-shared", f"-D_GLIBCXX_USE_CXX11_ABI={abi}",
           "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", "-DTORCH_EXTENSION_NAME=paia_gemv_torch",
           *[f"-I{p}" for p in ce.include_paths()], f"-I{ROCM / 'include'}", f"-I{INCLUDE}",
           str(CSRC / "torch_ops.cpp"),
           f"-L{tdir / 'lib'}", "-lc10", "-ltorch", "-ltorch_cpu", "-lc10_hip", "-ltorch_hip",
           f"-L{BUILD}", "-lpaia_gemv", f"-L{ROCM / 'lib'}", "-lamdhip64",
           "-Wl,-rpath,$ORIGIN", f"-Wl,-rpath,{tdir / 'lib'}",
           "-o", str(TORCH_LIB.with_suffix(".so.tmp"))]
    _run(cmd, quiet_warn=False)
    os.replace(TORCH_LIB.with_suffix(".so.tmp"), TORCH_LIB)
    return TORCH_LIB


def build_all() -> None:
    BUILD.mkdir(parents=True, exist_ok=True)
    with cf.ThreadPoolExecutor(max_workers=2) as ex:
        probe_f = ex.submit(build_probe)
        build_lib()
        build_torch_ext()
        probe_f.result()


def main(argv=None):
    ap = argparse.ArgumentParser(description=__doc__.splitlines()[0])
    ap.add_argument("--lib", action="store_true", help="build only libpaia_gemv.so")
    a = ap.parse_args(argv)
    if a.lib:
        print(build_lib())
    else:
        build_all()
        print(LIB, TORCH_LIB)


if __name__ == "__main__":
    sys.exit(main())
