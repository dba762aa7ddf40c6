"""Build libfxpr_hip.so (the gfx950 kernels + C ABI) and libfxpr_torch.so (the
torch.ops.fxpr launchers) in-tree.

    python build.py [--jobs N] [--verbose]

Each csrc/*.hip file is compiled to an object under _build/ and the objects
are linked into fxpr_vllm/libfxpr_hip.so, which fxpr_vllm/_hip.py loads with
ctypes; csrc/torch_ops.cpp is compiled by the host compiler against torch's
headers and linked to it. hipcc cross-compiles for gfx950, so this works
without a GPU.
"""

from __future__ import annotations

import argparse
import concurrent.futures as cf
import os
import shutil
import subprocess
import sys
from pathlib import Path

HERE = Path(__file__).resolve().parent
REPO = HERE.parent
CSRC = HERE / "csrc"
BUILD = HERE / "_build"
OUT = HERE / "fxpr_vllm" / "libfxpr_hip.so"
TORCH_OUT = HERE / "fxpr_vllm" / "libfxpr_torch.so"
ARCH = os.environ.get("FXPR_OFFLOAD_ARCH", "gfx950")

# -packed-fp32-ops: never emit v_pk_{add,mul,fma}_f32.
# -ffp-contract=off: no fused multiply-add, so every fp32 operation rounds on
# its own exactly like the CPU restatement.
COMMON_FLAGS = [
    "-O3",
    "-std=c++17",
    f"--offload-arch={ARCH}",
    "-fPIC",
    "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
    f"-I{REPO / 'include'}",
    f"-I{CSRC}",
]


# Per-source additions. rows.hip: no atomic optimizer. The split log-softmax
# counts each workgroup with one returning atomic from one lane, whose return
# is meant to arrive with the loads issued right after it; the optimizer's
# lane broadcast would wait for it at once, on every workgroup's critical
# path.
# gemm_bf16.hip / gemm_f16.hip: the machine scheduler's memory-clause
# strategy (the kernels' own sched_barrier stages stay as written; inside
# them it orders the fragment reads and DMAs differently): the large-M GEMM
# 1-1.5 % faster at M = 256 .. 8192 in crossed A/B runs, same bits.
_GEMM_SCHED = ["-mllvm", "-amdgpu-sched-strategy=max-memory-clause"]
FILE_FLAGS = {
    "rows.hip": ["-mllvm", "-amdgpu-atomic-optimizer-strategy=None"],
    "gemm_bf16.hip": _GEMM_SCHED,
    "gemm_f16.hip": _GEMM_SCHED,
}


def hipcc() -> str:
    path = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(path).exists():
        raise RuntimeError("hipcc not found; install ROCm or put hipcc on PATH")
    return path


def _run(cmd: list[str], verbose: bool) -> None:
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        sys.stderr.write(res.stdout + res.stderr)
        raise RuntimeError(f"command failed ({res.returncode}): {' '.join(cmd[:4])} ...")
    # the host pass warns that it does not know the packed-fp32 feature
    noise = "packed-fp32-ops"
    for line in (res.stderr or "").splitlines():
        if verbose and noise not in line:
            print(line)


def _check_defined(lib: Path) -> None:
    """Fail if the library references a symbol of its own namespace that no
    object defines (a kernel whose host launch stub was not emitted links
    fine and fails only at load time)."""
    nm = shutil.which("nm")
    if nm is None:
        return
    res = subprocess.run([nm, "-D", "--undefined-only", str(lib)], capture_output=True, text=True)
    missing = [ln.split()[-1] for ln in res.stdout.splitlines() if "4fxpr" in ln]
    if missing:
        raise RuntimeError(f"{lib.name}: undefined symbols of the library's own code: {missing[:4]}")


def torch_commands(obj: Path, hip_lib: Path, out: Path) -> tuple[list[str], list[str]]:
    """Compile and link commands of the torch launchers. (torch's own headers
    for ROCm are plain C++: no device code here, so any host compiler.)"""
    import torch

    root = Path(torch.__file__).resolve().parent
    cxx = shutil.which("g++") or shutil.which("c++") or hipcc()
    compile_ = [cxx, "-O2", "-std=c++17", "-fPIC", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
                f"-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}", f"-I{REPO / 'include'}",
                f"-I{root / 'include'}", f"-I{root / 'include' / 'torch' / 'csrc' / 'api' / 'include'}",
                f"-I{Path(os.environ.get('ROCM_PATH', '/opt/rocm')) / 'include'}",
                "-c", str(CSRC / "torch_ops.cpp"), "-o", str(obj)]
    link = [cxx, "-shared", "-fPIC", str(obj), str(hip_lib), f"-L{root / 'lib'}", "-lc10", "-lc10_hip", "-ltorch_cpu",
            "-ltorch_hip", "-ltorch", "-Wl,-rpath,$ORIGIN", "-o", str(out)]
    return compile_, link


def build(jobs: int | None = None, verbose: bool = False) -> Path:
    sources = sorted(CSRC.glob("*.hip"))
    if not sources:
        raise RuntimeError(f"no HIP sources under {CSRC}")
    BUILD.mkdir(exist_ok=True)
    cc = hipcc()
    objs = [BUILD / (s.stem + ".o") for s in sources]
    jobs = jobs or min(8, len(sources) + 1)
    torch_obj, torch_tmp = BUILD / "torch_ops.o", TORCH_OUT.with_suffix(".so.tmp")
    tmp = OUT.with_suffix(".so.tmp")
    torch_cc, torch_ld = torch_commands(torch_obj, tmp, torch_tmp)
    with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
        futs = [
            ex.submit(_run, [cc, *COMMON_FLAGS, *FILE_FLAGS.get(s.name, []), "-c", str(s), "-o", str(o)], verbose)
            for s, o in zip(sources, objs)
        ]
        futs.append(ex.submit(_run, torch_cc, verbose))
        for f in futs:
            f.result()
    # (the soname is how libfxpr_torch.so finds it, beside itself)
    _run([cc, "-shared", f"--offload-arch={ARCH}", "-fPIC", f"-Wl,-soname,{OUT.name}", *map(str, objs), "-o", str(tmp)],
         verbose)
    _check_defined(tmp)
    _run(torch_ld, verbose)
    # both linked: a failure leaves the old pair, not launchers beside a
    # kernel library that they were not built for
    os.replace(tmp, OUT)
    os.replace(torch_tmp, TORCH_OUT)
    return OUT


def main() -> None:
    ap = argparse.ArgumentParser(description=__doc__)
    ap.add_argument("--jobs", type=int, default=None)
    ap.add_argument("--verbose", action="store_true")
    args = ap.parse_args()
    out = build(args.jobs, args.verbose)
    print(f"built {out}")


if __name__ == "__main__":
    main()
