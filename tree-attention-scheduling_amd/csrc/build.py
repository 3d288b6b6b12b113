"""Build ``libtree_attn.so`` (gfx950), ``libtree_plan.so`` (host planner) and
``_fastcall.so`` (Python entry of the per-layer calls) next to the
``tree_attention`` package.

    python tree-attention-scheduling_amd/csrc/build.py

Uses hipcc directly; no CMake, no JIT cache.  The library is placed in-tree so
it travels with the source snapshot to the GPU machine.  Each translation unit
has its own code-generation flags (see ``SOURCES``); the objects are linked
into one shared library.
"""
import os
import shutil
import subprocess
import sys
import tempfile
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

HERE = Path(__file__).resolve().parent
PKG = HERE.parent / "tree_attention"
INCLUDE = HERE.parent.parent / "include"
LIB = PKG / "libtree_attn.so"
PLAN_LIB = PKG / "libtree_plan.so"
FASTCALL = PKG / "_fastcall.so"
# The planner's costs must round exactly like the Python planner's: no FMA
# contraction, no fast-math reassociation.
PLAN_FLAGS = ["-O2", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", "-fno-fast-math", "-Wall"]

COMMON = [
    "-O3", "-std=c++20", "--offload-arch=gfx950", "-fPIC",
    "-mcode-object-version=5",
    # packed-FP32 VALU forms are kept out of every kernel
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # the leading pointer arguments (the work items', the merge's buffers) arrive in scalar
    # registers with the launch instead of by a first load: decode layers 2 % shorter
    # (19.2 -> 18.8 us and 16.3 -> 16.0 us with their append and update launches), the nested
    # tree 33.9 -> 33.3 us
    "-mllvm", "-amdgpu-kernarg-preload-count=16",
    "-Wall", "-Wno-unused-function",
]
# (source, extra flags).  MFMA accumulators in VGPRs: every kernel fits in 256
# VGPRs, and with accumulators in AGPRs the allocator copied O between the two
# register files every step (the rescale multiplies O on the VALU).
# segment_tile.hip also builds with -fno-honor-nans: its row maxima then
# compile to v_max3_f32 chains without a canonicalising v_max per input; the
# kernel never produces NaN scores (masked tokens are selected to -inf).
VGPR_FORM = ["-mllvm", "-amdgpu-mfma-vgpr-form"]
# segment_tile.hip is compiled once per K/V layout (enum Layout, ta_common.h); the
# flag stays off for the layouts of token counts that are no multiple of 8, whose row maxima pass over a NaN
# score wherever it stands (at most 0.4 % of a layer's time either way, 2 % in 256-row items).
SOURCES = [
    (HERE / "tree_attn.hip", VGPR_FORM),
    *[(HERE / "segment_tile.hip", VGPR_FORM + ["-fno-honor-nans", f"-DTA_LAYOUT={layout}"])
      for layout in ("KV_POOL", "KV_TOKEN")],
    *[(HERE / "segment_tile.hip", VGPR_FORM + [f"-DTA_LAYOUT={layout}"]) for layout in ("KV_ODD", "KV_TOKEN_ODD")],
    (HERE / "decode_append.hip", ["-ffp-contract=off"]),  # each RoPE product rounded, as the eager ops
]


def hipcc() -> str:
    found = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(found).exists():
        raise RuntimeError("hipcc not found; ROCm is required to build the tree_attn library")
    return found


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"{Path(cmd[0]).name} failed ({res.returncode}):\n{res.stdout}\n{res.stderr}")
    if verbose and res.stderr.strip():
        print(res.stderr, file=sys.stderr)


def build(verbose: bool = False, out: Path | None = None, defines=()) -> Path:
    """Compile every source and link ``out`` (default: the in-tree library)."""
    target = Path(out) if out is not None else LIB
    tmp = target.with_name(target.name + f".tmp{os.getpid()}")
    with tempfile.TemporaryDirectory() as work:
        def compile_one(i):
            src, extra = SOURCES[i]
            obj = Path(work) / f"{src.stem}_{i}.o"
            _run([hipcc(), *COMMON, *extra, *[f"-D{d}" for d in defines], f"-I{INCLUDE}", f"-I{HERE}",
                  "-c", str(src), "-o", str(obj)], verbose)
            return str(obj)

        with ThreadPoolExecutor(5) as pool:  # each unit takes up to a minute
            objs = list(pool.map(compile_one, range(len(SOURCES))))
        _run([hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", *objs, "-o", str(tmp)], verbose)
    os.replace(tmp, target)
    return target


def build_fastcall(verbose: bool = False, out: Path | None = None) -> Path:
    """Compile the Python entry of the per-layer calls (fastcall.cpp) into ``out`` (default:
    in-tree) with g++ against the installed torch."""
    import sysconfig
    import torch
    from torch.utils.cpp_extension import include_paths
    target = Path(out) if out is not None else FASTCALL
    tmp = target.with_name(target.name + f".tmp{os.getpid()}")
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        raise RuntimeError("g++ not found; it is required to build the host module")
    lib = Path(torch.__file__).parent / "lib"
    _run([cxx, "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
          f'-DTA_BUILT_FOR="{sys.implementation.cache_tag} torch {torch.__version__}"',
          *[f"-isystem{p}" for p in include_paths()], f"-I{sysconfig.get_paths()['include']}", f"-I{INCLUDE}",
          str(HERE / "fastcall.cpp"), f"-L{lib}", "-ltorch_python", "-ltorch_cpu", "-ltorch", "-lc10", "-o", str(tmp)],
         verbose)
    os.replace(tmp, target)
    return target


def build_planner(verbose: bool = False, out: Path | None = None) -> Path:
    """Compile the host planner (planner.cpp) into ``out`` (default: in-tree) with g++."""
    target = Path(out) if out is not None else PLAN_LIB
    tmp = target.with_name(target.name + f".tmp{os.getpid()}")
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        raise RuntimeError("g++ not found; it is required to build the planner library")
    _run([cxx, *PLAN_FLAGS, f"-I{INCLUDE}", str(HERE / "planner.cpp"), "-o", str(tmp)], verbose)
    os.replace(tmp, target)
    return target


if __name__ == "__main__":
    args = sys.argv[1:]
    out = None
    defines = []
    while args:
        a = args.pop(0)
        if a == "-o":
            out = Path(args.pop(0))
        elif a.startswith("-D"):
            defines.append(a[2:])
    print(build(verbose=True, out=out, defines=defines))
    if out is None:
        print(build_planner(verbose=True))
        print(build_fastcall(verbose=True))
