"""The native launchers behind torch.ops.fxpr.* (csrc/torch_ops.cpp) against
the Python launchers in fxpr_vllm/_kernels: the same bits, shapes and dtypes
over layouts that take a copy or an early return, and the same refusals."""

from __future__ import annotations

import pytest
import torch

import fxpr_vllm  # noqa: F401
from fxpr_vllm import _lib
from fxpr_vllm._kernels import attention as KA
from fxpr_vllm._kernels import cache as KC
from fxpr_vllm._kernels import casts as KX
from fxpr_vllm._kernels import gemm as KG
from fxpr_vllm._kernels import rows as KR
from fxpr_vllm._kernels import sampling as KS

pytestmark = pytest.mark.gpu
ops = torch.ops.fxpr


def _rand(*shape, dtype=torch.float32, seed=0):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)).to(dtype).cuda()


def _same(a, b):
    a, b = (a, b) if isinstance(a, tuple) else ((a,), (b,))
    assert len(a) == len(b)
    for x, y in zip(a, b):
        assert x.shape == y.shape and x.dtype == y.dtype and x.is_contiguous() and torch.equal(x, y)


def test_native_launchers_are_registered():
    assert _lib._NATIVE
    assert "torch_ops.cpp" in torch._C._dispatch_dump("fxpr::gemm_fxp")


@pytest.mark.parametrize("shape", [(7,), (3, 5), (0, 4), (2, 3, 40), ()])
def test_casts_and_row_sum(shape):
    x = _rand(*shape, dtype=torch.float64) * 50
    for bits, frac in ((16, 8), (32, 16), (64, 32)):
        for v in (x, x.float(), x.half(), x.float().t() if x.dim() == 2 else x.float()):
            q = ops.float_to_fixed(v, bits, frac)
            _same(q, KX.float_to_fixed_run(v, bits, frac))
            for fb in (16, 32, 64):
                _same(ops.fixed_to_float(q, fb, frac), KX.fixed_to_float_run(q, fb, frac))
            _same(ops.fixed_row_sum(q, bits), KR.fixed_row_sum_run(q, bits))
    _same(ops.fixed_row_sum(torch.zeros(3, 0, dtype=torch.int32, device="cuda"), 64),
          KR.fixed_row_sum_run(torch.zeros(3, 0, dtype=torch.int32, device="cuda"), 64))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_norms_log_softmax_and_sampler(dtype):
    x, w = _rand(2, 6, 264, dtype=dtype), _rand(264, dtype=dtype, seed=1)
    for v in (x, x[:, ::2], x[0].t().contiguous().t(), x[:0]):
        _same(ops.rms_norm_fxp(v, w, 1e-6), KR.rms_norm_fxp_run(v, w, 1e-6))
        r0 = torch.empty_strided(v.shape, v.stride(), dtype=dtype, device="cuda").copy_(v * 2)
        r1 = torch.empty_strided(v.shape, v.stride(), dtype=dtype, device="cuda").copy_(v * 2)
        _same(ops.rms_norm_fxp_residual(v, r0, w, 1e-6), KR.rms_norm_fxp_residual_run(v, r1, w, 1e-6))
        assert torch.equal(r0, r1)
        for out in (None, torch.float32):
            _same(ops.log_softmax_fxp(v, 32, 16, out), KR.log_softmax_fxp_run(v, 32, 16, out))
        for k in (0, 5):
            _same(ops.sample_greedy_fxp(v, k, 32, 16), KS.sample_greedy_fxp_run(v, k, 32, 16))


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_gemm(dtype):
    a, w = _rand(40, 256, dtype=dtype), _rand(264, 256, dtype=dtype, seed=1) * 0.1
    kn = w.t().contiguous()
    for m in (1, 17, 40):
        for b in (w.t(), kn, kn[:, ::2], kn[:, :5]):
            for av in (a[:m], a[:, ::2].repeat(1, 2)[:m], a.t().contiguous().t()[:m]):
                for bias in (None, _rand(b.shape[1], dtype=dtype, seed=2)):
                    _same(ops.gemm_fxp(av, b, bias, 32, 16), KG.gemm_fxp_run(av, b, bias, 32, 16))
    _same(ops.gemm_fxp(a[:0], kn, None, 64, 16), KG.gemm_fxp_run(a[:0], kn, None, 64, 16))


def test_cache_and_attention():
    k, v = _rand(70, 2, 64, dtype=torch.bfloat16), _rand(70, 2, 64, dtype=torch.bfloat16, seed=1)
    slots = torch.randperm(96, generator=torch.Generator().manual_seed(3))[:70].cuda()
    c0, c1 = (torch.zeros(6, 2, 16, 2, 64, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    ops.reshape_and_cache(k, v, c0, slots.int())
    KC.reshape_and_cache_run(k, v, c1, slots)
    assert torch.equal(c0, c1)
    ops.reshape_and_cache(k.view(70, 128), v.view(70, 128), c0.zero_(), slots)
    assert torch.equal(c0, c1)
    q = _rand(5, 4, 128, dtype=torch.bfloat16, seed=4)
    qsl = torch.tensor([0, 1, 5], dtype=torch.int32, device="cuda")
    sl = torch.tensor([33, 60], dtype=torch.int32, device="cuda")
    bt = torch.tensor([[0, 1, 2, 3], [4, 5, 1, 0]], dtype=torch.int32, device="cuda")
    slopes = torch.tensor([0.1, 0.2, 0.3, 0.4], device="cuda")
    for qv in (q[..., :64], q[..., ::2]):
        for bias, scale, cap, window, splits in ((None, None, 0.0, 0, 0), (slopes, 0.3, 20.0, 7, 2)):
            o0 = torch.zeros(5, 4, 64, dtype=torch.bfloat16, device="cuda")
            o1 = torch.zeros(5, 4, 128, dtype=torch.bfloat16, device="cuda")[..., ::2]
            ops.unified_attention_fxp(qv, c0, o0, qsl, sl, bt, 4, bias, True, scale, 32, 16, cap, window, splits)
            KA.unified_attention_fxp_run(qv, c0, o1, qsl, sl, bt.flatten(), 4, bias, True, scale, 32, 16, cap, window,
                                         splits)
            assert torch.equal(o0, o1)
            o1.zero_()
            ops.unified_attention_fxp(qv, c0, o1, qsl, sl, bt.flatten(), 4, bias, True, scale, 32, 16, cap, window, splits)
            assert torch.equal(o0, o1)


def test_refusals():
    f, h = _rand(4, 8), _rand(4, 8, dtype=torch.float16)
    i = torch.ones(4, 8, dtype=torch.int32, device="cuda")
    kv = torch.zeros(2, 2, 16, 2, 64, device="cuda")
    q, o = _rand(1, 2, 64), torch.zeros(1, 2, 64, device="cuda")
    n1 = torch.ones(1, dtype=torch.int32, device="cuda")
    qsl = torch.tensor([0, 1], dtype=torch.int32, device="cuda")
    att = lambda **k: ops.unified_attention_fxp(*{**dict(  # noqa: E731
        q=q, kv=kv, o=o, qsl=qsl, sl=n1, bt=n1.view(1, 1), m=1, al=None, c=True, s=None, b=32, f=16, cap=0.0, w=0,
        n=0), **k}.values())
    att()
    for err, call in [
        (ValueError, lambda: ops.float_to_fixed(f, 8, 16)),
        (ValueError, lambda: ops.float_to_fixed(f, 32, 12)),
        (TypeError, lambda: ops.float_to_fixed(f.bfloat16(), 32, 16)),
        (ValueError, lambda: ops.fixed_to_float(i, 8, 16)),
        (TypeError, lambda: ops.fixed_to_float(f, 32, 16)),
        (TypeError, lambda: ops.fixed_row_sum(f, 32)),
        (TypeError, lambda: ops.rms_norm_fxp(f, h[0], 1e-6)),
        (ValueError, lambda: ops.rms_norm_fxp(f, f[0, :3], 1e-6)),
        (ValueError, lambda: ops.rms_norm_fxp_residual(f, f[:2], f[0], 1e-6)),
        (RuntimeError, lambda: ops.rms_norm_fxp(f, f[0].cpu(), 1e-6)),
        (TypeError, lambda: ops.log_softmax_fxp(f, 32, 16, torch.float16)),
        (ValueError, lambda: ops.sample_greedy_fxp(f, 9, 32, 16)),
        (TypeError, lambda: ops.sample_greedy_fxp(i, 1, 32, 16)),
        (TypeError, lambda: ops.gemm_fxp(f, h.t(), None, 32, 16)),
        (ValueError, lambda: ops.gemm_fxp(f, f, None, 32, 16)),
        (ValueError, lambda: ops.gemm_fxp(f, f.t(), f[0], 32, 16)),
        (RuntimeError, lambda: ops.gemm_fxp(f, f.t().cpu(), None, 32, 16)),
        (ValueError, lambda: att(kv=kv[0])),
        (TypeError, lambda: att(sl=n1.long())),
        (TypeError, lambda: att(kv=kv.half())),
        (ValueError, lambda: att(n=-1)),
        (ValueError, lambda: att(o=o[:, :1])),
        (ValueError, lambda: ops.reshape_and_cache(q, q[:, :1], kv, n1.long())),
        (TypeError, lambda: ops.reshape_and_cache(q.half(), q.half(), kv, n1.long())),
    ]:
        with pytest.raises(err):
            call()
