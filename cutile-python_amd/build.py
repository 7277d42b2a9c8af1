"""Builds libmxgemm.so (HIP kernels + C ABI) for gfx950 with hipcc, in-tree.

    python cutile-python_amd/build.py [--force]

Each translation unit is compiled to an object file in parallel and the objects are linked into
cutile-python_amd/cutile_amd/libmxgemm.so.  hipcc cross-compiles: no GPU is needed to build.
"""
from __future__ import annotations

import argparse
import importlib.util
import os
import pathlib
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

ROOT = pathlib.Path(__file__).resolve().parent
CSRC = ROOT / "csrc"
INCLUDE = ROOT.parent / "include"
OUT = ROOT / "cutile_amd" / "libmxgemm.so"
HOST_OUT = ROOT / "cutile_amd" / "_mxhost.so"   # csrc/mx_host.cpp: the operators' native host path
OBJ = ROOT / "build"
SOURCES = ["mx_api.hip", "mx_gemm_mfma.hip", "mx_gemm_pp32.hip", "mx_gemm_w4.hip", "mx_gemm_generic.hip", "mx_gemm_decode.hip", "mx_gemm_stream.hip", "mx_moe.hip", "mx_moe_tile.hip", "mx_aux.hip", "mx_probe.hip"]
# sources compiled once per value of a macro, so that their instances build in parallel: (file, macro, count)
SPLIT = [("mx_gemm_pp.hip", "MX_PP_PAIR", 4), ("mx_gemm_t128.hip", "T128_PAIR", 4)]
UNITS = [(s, None) for s in SOURCES] + [(f, f"-D{m}={i}") for f, m, n in SPLIT for i in range(n)]
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-fvisibility=hidden",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
         f"-I{INCLUDE}", f"-I{CSRC}", "-Wno-unused-command-line-argument"]
# Extra compiler flags for experiments (for example "-DSOMETHING=1"); objects built with a different flag set
# are never reused: the flag list is part of the up-to-date check (stamp file next to the objects).
FLAGS += os.environ.get("MXGEMM_EXTRA_FLAGS", "").split()


def _newer(src: pathlib.Path, obj: pathlib.Path) -> bool:
    if not obj.exists():
        return True
    deps = [src, *CSRC.glob("*.h"), INCLUDE / "mxgemm.h"]
    listed = obj.with_suffix(".d")   # what the compiler read of this tree the last time
    if listed.exists():
        names = [pathlib.Path(w) for w in listed.read_text().replace("\\\n", " ").split()[1:]]
        deps = [d for d in names if ROOT.parent in d.resolve().parents]
        if not all(d.exists() for d in deps):
            return True
    return any(d.stat().st_mtime > obj.stat().st_mtime for d in deps)


def _flags_changed() -> bool:
    """True when the objects on disk were built with other flags (the stamp is removed until the next build has
    compiled every object, so a failed build never leaves old objects looking current)."""
    stamp = OBJ / "flags.txt"
    if stamp.exists() and stamp.read_text() == " ".join(FLAGS):
        return False
    stamp.unlink(missing_ok=True)
    return True


def _compile(unit, force: bool) -> pathlib.Path:
    src, define = unit
    s = CSRC / src
    o = OBJ / (s.stem + (define.replace("=", "_").replace("-D", "_") if define else "") + ".o")
    if force or _newer(s, o):
        cmd = ["hipcc", *FLAGS, *([define] if define else []), "-MD", "-MF", str(o.with_suffix(".d")), "-c", str(s), "-o", str(o)]
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError(f"hipcc failed for {src}:\n{r.stdout}\n{r.stderr}")
    return o


def _build_host(force: bool) -> None:
    """The native host path of the Python operators: host code only, against the torch that will load it."""
    import sysconfig
    spec = importlib.util.find_spec("torch")   # torch's place, without importing it
    torch_dir = pathlib.Path(spec.submodule_search_locations[0])
    src, rocm = CSRC / "mx_host.cpp", pathlib.Path(os.environ.get("ROCM_PATH", "/opt/rocm"))
    if not force and not _newer(src, HOST_OUT):
        return
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM",
           f"-I{INCLUDE}", f"-I{rocm / 'include'}", f"-I{torch_dir / 'include'}",
           f"-I{torch_dir / 'include/torch/csrc/api/include'}", f"-I{sysconfig.get_paths()['include']}", "-o", str(HOST_OUT),
           str(src), f"-L{torch_dir / 'lib'}", "-ltorch_python", "-ltorch_hip", "-ltorch_cpu", "-lc10_hip", "-lc10"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"g++ failed for {src.name}:\n{r.stdout}\n{r.stderr}")


def build(force: bool = False, jobs: int | None = None) -> pathlib.Path:
    OBJ.mkdir(exist_ok=True)
    force = _flags_changed() or force
    jobs = jobs or min(len(UNITS), os.cpu_count() or 4, 8)
    with ThreadPoolExecutor(jobs) as ex:
        host = ex.submit(_build_host, force)
        objs = list(ex.map(lambda u: _compile(u, force), sorted(UNITS, key=lambda u: u[1] is None)))
        host.result()
    (OBJ / "flags.txt").write_text(" ".join(FLAGS))
    cmd = ["hipcc", "--offload-arch=gfx950", "-shared", "-fPIC", "-o", str(OUT), *map(str, objs)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    return OUT


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--force", action="store_true", help="recompile every translation unit")
    a = ap.parse_args()
    print(build(force=a.force))
    sys.exit(0)
