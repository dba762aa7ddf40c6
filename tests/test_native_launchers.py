"""Which launchers serve torch.ops.fxpr.*: the native ones (libfxpr_torch.so)
where they load, the Python ones otherwise. Each case imports a copy of the
package, with other library files beside it, in a process of its own."""

from __future__ import annotations

import importlib.util
import os
import pathlib
import re
import shutil
import subprocess
import sys
import textwrap

import pytest
import torch

from fxpr_vllm import _hip

PKG = pathlib.Path(_hip.__file__).resolve().parent
OPS = ("float_to_fixed", "fixed_to_float", "rms_norm_fxp", "rms_norm_fxp_residual", "gemm_fxp",
       "unified_attention_fxp", "fixed_row_sum", "log_softmax_fxp", "reshape_and_cache", "sample_greedy_fxp")


@pytest.fixture()
def package(tmp_path):
    """A copy of the package without its libraries."""
    shutil.copytree(PKG, tmp_path / "fxpr_vllm", ignore=shutil.ignore_patterns("*.so", "*.so.*", "__pycache__"))
    return tmp_path / "fxpr_vllm"


def run(package, code, *args):
    code = f"import sys\nsys.path.insert(0, {str(package.parent)!r})\n" + textwrap.dedent(code)
    res = subprocess.run([sys.executable, "-c", code, *map(str, args)], capture_output=True, text=True, timeout=240,
                         cwd=package.parent)
    assert res.returncode == 0, res.stdout + res.stderr[-2000:]
    return res


REPORT = f"""
    import fxpr_vllm
    from fxpr_vllm import _hip, _lib
    import torch
    assert _lib.__file__.startswith(sys.path[0])
    has = torch._C._dispatch_has_kernel_for_dispatch_key
    assert all(has("fxpr::" + op, "CUDA") for op in {OPS!r})
    m = torch.empty(2, 8, dtype=torch.float16, device="meta")
    assert torch.ops.fxpr.gemm_fxp(m, m.t(), None, 32, 16).shape == (2, 2)
    print("native", _lib._NATIVE)
    try:
        _hip.load()
        print("kernels loaded")
    except RuntimeError as e:
        print("kernels:", e)
"""


def test_import_without_the_kernel_library(package):
    shutil.copy(PKG / "libfxpr_torch.so", package)
    res = run(package, REPORT)
    assert "native False" in res.stdout and "not built" in res.stdout


def test_import_without_the_native_launchers(package):
    os.symlink(PKG / "libfxpr_hip.so", package / "libfxpr_hip.so")
    res = run(package, REPORT)
    assert "native False" in res.stdout and "kernels loaded" in res.stdout


def test_native_launchers_that_do_not_load_are_reported(package):
    os.symlink(PKG / "libfxpr_hip.so", package / "libfxpr_hip.so")
    (package / "libfxpr_torch.so").write_text("not a library\n")
    res = run(package, REPORT)
    assert "native False" in res.stdout and "kernels loaded" in res.stdout
    assert "native launchers" in res.stderr and "libfxpr_torch.so" in res.stderr


def test_native_launchers_refuse_another_kernel_library(package):
    # a kernel library of another ABI revision (stubs of what the launchers
    # link to): nothing is registered, and the bindings refuse it per call
    cc = shutil.which("gcc") or shutil.which("cc")
    if cc is None:
        pytest.skip("no C compiler")
    shutil.copy(PKG / "libfxpr_torch.so", package)
    source = (PKG.parent / "csrc" / "torch_ops.cpp").read_text()
    stubs = sorted(set(re.findall(r"\b(fxpr_[a-z0-9_]+)\(", source)) - {"fxpr_abi_version", "fxpr_torch_registered"})
    assert "fxpr_gemm" in stubs
    text = "int fxpr_abi_version(void) { return 999; }\n" + "".join(f"int {n}(void) {{ return 0; }}\n" for n in stubs)
    (package / "stub.c").write_text(text)
    subprocess.run([cc, "-shared", "-fPIC", "-Wl,-soname,libfxpr_hip.so", str(package / "stub.c"), "-o",
                    str(package / "libfxpr_hip.so")], check=True)
    res = run(package, REPORT)
    assert "native False" in res.stdout and "ABI revision 999" in res.stdout
    assert "another revision" in res.stderr


def test_build_links_both_libraries_before_replacing_either(tmp_path, monkeypatch):
    # a launcher library that does not link leaves the old pair in place
    spec = importlib.util.spec_from_file_location("fxpr_build_test", PKG.parent / "build.py")
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    monkeypatch.setattr(build, "BUILD", tmp_path / "_build")
    monkeypatch.setattr(build, "OUT", tmp_path / "libfxpr_hip.so")
    monkeypatch.setattr(build, "TORCH_OUT", tmp_path / "libfxpr_torch.so")
    monkeypatch.setattr(build, "_check_defined", lambda lib: None)
    build.OUT.write_text("old kernels")
    build.TORCH_OUT.write_text("old launchers")

    def fake(cmd, verbose):
        out = pathlib.Path(cmd[cmd.index("-o") + 1])
        if "-shared" in cmd and "torch" in out.name:
            raise RuntimeError("does not link")
        out.write_text("new")

    monkeypatch.setattr(build, "_run", fake)
    with pytest.raises(RuntimeError, match="does not link"):
        build.build(jobs=1)
    assert build.OUT.read_text() == "old kernels" and build.TORCH_OUT.read_text() == "old launchers"


@pytest.mark.gpu
def test_python_launchers_give_the_native_results(package, tmp_path):
    # torch.ops.fxpr.* in a process without the native launchers: the same
    # tensors as here, for every op that has one
    os.symlink(PKG / "libfxpr_hip.so", package / "libfxpr_hip.so")
    calls = """
        def results(ops):
            r = lambda *s, t=torch.float32, seed=0: torch.randn(
                s, generator=torch.Generator().manual_seed(seed)).to(t).cuda()
            x, w = r(5, 264), r(264, seed=1)
            q = ops.float_to_fixed(x, 32, 16)
            res = x * 2
            out = [q, ops.fixed_to_float(q, 32, 16), ops.fixed_row_sum(q, 64), ops.rms_norm_fxp(x, w, 1e-6),
                   ops.rms_norm_fxp_residual(x, res, w, 1e-6), res, ops.log_softmax_fxp(x, 32, 16),
                   *ops.sample_greedy_fxp(x, 3, 32, 16)]
            a, b = r(17, 256, t=torch.bfloat16), r(256, 64, t=torch.bfloat16, seed=2)
            out += [ops.gemm_fxp(a, b, None, 32, 16), ops.gemm_fxp(a[:1], b, b[0], 32, 16)]
            kv = torch.zeros(8, 2, 16, 2, 64, dtype=torch.bfloat16, device="cuda")
            ops.reshape_and_cache(r(90, 2, 64, t=torch.bfloat16), r(90, 2, 64, t=torch.bfloat16, seed=3), kv,
                                  torch.arange(90, device="cuda"))
            i = lambda *v: torch.tensor(v, dtype=torch.int32, device="cuda")
            o = torch.zeros(31, 4, 64, dtype=torch.bfloat16, device="cuda")
            ops.unified_attention_fxp(r(31, 4, 64, t=torch.bfloat16), kv, o, i(0, 30, 31), i(70, 20),
                                      i(0, 1, 2, 3, 4, 5, 1, 2, 3, 4).view(2, 5), 30, None, True, None, 32, 16, 0.0, 0, 0)
            return [t.cpu() for t in out + [kv, o]]
    """
    run(package, textwrap.dedent("""
        import torch, fxpr_vllm
        from fxpr_vllm import _lib
        assert not _lib._NATIVE
    """) + textwrap.dedent(calls) + "torch.save(results(torch.ops.fxpr), sys.argv[1])\n", tmp_path / "out.pt")
    scope = {"torch": torch}
    exec(textwrap.dedent(calls), scope)
    got, want = torch.load(tmp_path / "out.pt", weights_only=True), scope["results"](torch.ops.fxpr)
    assert len(got) == len(want) and all(torch.equal(a, b) for a, b in zip(got, want))
