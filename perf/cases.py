"""The work that programs give these operators, as cases that can be timed.

A case is one call (or the few calls of one step) of `torch.ops.fxpr.*` at sizes that serving and scoring a
language model reach: single-row decode linears up to the whole lm_head over a scoring batch, paged attention
for decode, prefill and both in one batch, norms, the step from logits to tokens, and the fixed-point encode /
sum / decode chain. `listed()` holds one case for each of these; `draw()` gives others of the same ranges.

Kinds and what `run` returns:

  linear   gemm_fxp of activations with a weight; the output rows.
  attn     unified_attention_fxp over a paged cache; the output rows.
  norm     rms_norm_fxp_residual (or rms_norm_fxp); the normalised rows and the updated residual stream.
  head     sample_greedy_fxp and log_softmax_fxp on a batch of logits; tokens, their log-probabilities, the
           top five and the whole log-probability rows.
  chain    float_to_fixed, fixed_row_sum, fixed_to_float; the integers, the sums, the decoded values and sums.
"""

import math
import pathlib
import random
import sys

import torch

sys.path.insert(0, str(pathlib.Path(__file__).resolve().parents[1] / "vllm-triton-fixed-point-reductions_amd"))

import fxpr_vllm  # noqa: E402,F401  (registers torch.ops.fxpr.*)

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32, "f64": torch.float64}
SIZE = {"bf16": 2, "f16": 2, "f32": 4, "f64": 8}
EPS = 1e-6
TOP = 5


def _linear(m, k, n, dtype="bf16", layout="nk", bias=False, int_bits=32, frac_bits=16, **kw):
    return dict(kw, kind="linear", m=m, k=k, n=n, dtype=dtype, layout=layout, bias=bias, int_bits=int_bits,
                frac_bits=frac_bits)


def _attn(decodes, ctx_lo, ctx_hi, prefills=0, new=0, past=0, heads=32, kv_heads=8, head_dim=128, page=16,
          dtype="bf16", window=0, softcap=0.0, int_bits=32, frac_bits=16, lens=0, **kw):
    """`decodes` one-token requests with contexts in [ctx_lo, ctx_hi]; `prefills` requests of up to `new` new
    tokens each after up to `past` cached ones (the first has exactly these)."""
    return dict(kw, kind="attn", decodes=decodes, ctx_lo=ctx_lo, ctx_hi=ctx_hi, prefills=prefills, new=new,
                past=past, heads=heads, kv_heads=kv_heads, head_dim=head_dim, page=page, dtype=dtype,
                window=window, softcap=softcap, int_bits=int_bits, frac_bits=frac_bits, lens=lens)


def listed():
    return [
        # one user's token: the attention output projection at batch 1, the smallest linear of a decode step
        _linear(1, 4096, 4096, name="linear_one_row"),
        # a decode batch of 32 through the merged gate / up projection
        _linear(32, 4096, 28672, name="linear_decode_batch"),
        # a ragged chunk of prompt tokens through the down projection
        _linear(509, 14336, 4096, name="linear_prompt_chunk"),
        # float16 with a bias and the weight kept [K, N] row-major, as a plain matmul call has it
        _linear(1000, 4096, 6144, dtype="f16", layout="kn", bias=True, name="linear_kn_f16"),
        # full-precision evaluation: float32 activations and weights
        _linear(777, 4096, 14336, dtype="f32", name="linear_f32"),
        # scoring: every position's logits over the whole vocabulary
        _linear(8192, 4096, 128256, name="lm_head_scoring"),
        # a serving batch in decode: 64 requests, contexts from 512 to 8192
        _attn(64, 512, 8192, name="attn_decode"),
        # four fresh prompts of up to 2048 tokens
        _attn(0, 1, 1, prefills=4, new=2048, lens=1, name="attn_prefill"),
        # continuous batching: a 512-token chunk of one long prompt beside 31 decoding requests
        _attn(31, 512, 8192, prefills=1, new=512, past=3500, dtype="f16", lens=2, name="attn_mixed"),
        # the residual norm over a large prefill batch
        dict(kind="norm", rows=16384, cols=4096, dtype="bf16", residual=True, name="norm_residual"),
        # from the logits of a decode batch to tokens and log-probabilities
        dict(kind="head", rows=32, cols=128256, dtype="bf16", int_bits=32, frac_bits=16, name="head_step"),
        # encode, sum and decode a float32 tensor in the wide format
        dict(kind="chain", rows=4096, cols=4096, dtype="f32", int_bits=64, frac_bits=16, name="fixed_chain"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "attn", "attn", "attn", "norm", "head", "chain"])
    if kind == "linear":
        dtype = rng.choice(["bf16", "bf16", "bf16", "f16", "f16", "f32"])
        int_bits, frac_bits = rng.choice([(32, 16), (32, 16), (32, 16), (64, 16), (16, 8)])
        layout = rng.choice(["nk", "nk", "kn"])
        # hidden and FFN widths: multiples of 128, and ones that are not a whole number of K-tiles
        k = rng.choice([128 * _log_int(rng, 4, 112), 16 * _log_int(rng, 32, 896)])
        if rng.random() < 0.15:
            m, n = _log_int(rng, 1, 1024), _log_int(rng, 32000, 128256)  # a vocabulary, odd ones among them
        else:
            m, n = _log_int(rng, 1, 4096), 64 * _log_int(rng, 16, 448) + rng.choice([0, 0, 8, 1])
        if layout == "kn":
            n = -(-n // 8) * 8
        if dtype == "f32":
            m = min(m, 1024)
            n = min(n, 28672)
        return _linear(m, k, n, dtype, layout, rng.random() < 0.3, int_bits, frac_bits)
    if kind == "attn":
        heads, kv_heads, head_dim = rng.choice([(32, 8, 128), (32, 8, 128), (28, 4, 128), (16, 16, 64), (24, 8, 64)])
        what = rng.choice(["decode", "prefill", "mixed"])
        hi = _log_int(rng, 256, 12288)
        decodes = 0 if what == "prefill" else _log_int(rng, 1, 96)
        prefills = 0 if what == "decode" else rng.randint(1, 4)
        new = 0 if what == "decode" else _log_int(rng, 16, 2048)
        past = 0 if rng.random() < 0.5 else rng.randint(0, 6000)
        window, softcap = rng.choice([(0, 0.0), (0, 0.0), (0, 0.0), (1024, 0.0), (0, 50.0)])
        return _attn(decodes, max(1, hi // 16), hi, prefills, new, past if prefills else 0, heads, kv_heads, head_dim,
                     rng.choice([16, 16, 32, 64]), rng.choice(["bf16", "f16"]), window, softcap,
                     lens=rng.randrange(1 << 20))
    if kind == "norm":
        return dict(kind="norm", rows=_log_int(rng, 1, 16384), cols=8 * _log_int(rng, 64, 1024) + rng.choice([0, 0, 1]),
                    dtype=rng.choice(["bf16", "bf16", "f16", "f32"]), residual=rng.random() < 0.7)
    if kind == "head":
        int_bits, frac_bits = rng.choice([(32, 16), (32, 16), (64, 32)])
        return dict(kind="head", rows=_log_int(rng, 1, 256), cols=_log_int(rng, 16000, 160000),
                    dtype=rng.choice(["bf16", "bf16", "f16", "f32"]), int_bits=int_bits, frac_bits=frac_bits)
    int_bits, frac_bits = rng.choice([(16, 8), (32, 16), (64, 16)])
    return dict(kind="chain", rows=_log_int(rng, 1, 8192), cols=_log_int(rng, 64, 8192),
                dtype=rng.choice(["f32", "f32", "f16", "f64"]), int_bits=int_bits, frac_bits=frac_bits)


def _requests(case):
    """[(new tokens, context length after them)] of an attention case: prefills first, then decodes."""
    r = random.Random(case["lens"])
    reqs = []
    for i in range(case["prefills"]):
        new = case["new"] if i == 0 else r.randint(max(1, case["new"] // 2), case["new"])
        past = case["past"] if i == 0 else r.randint(0, case["past"])
        reqs.append((new, past + new))
    for _ in range(case["decodes"]):
        reqs.append((1, r.randint(case["ctx_lo"], case["ctx_hi"])))
    return reqs


def _gen(seed):
    return torch.Generator("cuda").manual_seed(int(seed))


def _randn(g, shape, dtype, std=1.0, mean=0.0):
    """Normal values drawn on the GPU (in slices: the draw itself is float32)."""
    out = torch.empty(shape, device="cuda", dtype=dtype)
    flat = out.view(-1)
    step = 1 << 27
    for i in range(0, flat.numel(), step):
        part = flat[i:i + step]
        x = torch.randn(part.numel(), generator=g, device="cuda")
        part.copy_(x.mul_(std).add_(mean))
    return out


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    dtype = DTYPES[case["dtype"]]
    if kind == "linear":
        # normalised activations, weights at initialisation's scale
        a = _randn(g, (case["m"], case["k"]), dtype)
        w = _randn(g, (case["n"], case["k"]) if case["layout"] == "nk" else (case["k"], case["n"]), dtype, 0.02)
        bias = _randn(g, (case["n"],), dtype, 0.1) if case["bias"] else None
        return {"case": case, "a": a, "b": w.t() if case["layout"] == "nk" else w, "bias": bias}
    if kind == "attn":
        reqs = _requests(case)
        page, hk, d = case["page"], case["kv_heads"], case["head_dim"]
        pages = [-(-ctx // page) for _, ctx in reqs]
        table = torch.zeros(len(reqs), max(pages), dtype=torch.int32)
        order = torch.randperm(sum(pages), generator=torch.Generator().manual_seed(int(seed))).to(torch.int32)
        at = 0
        for i, n in enumerate(pages):
            table[i, :n] = order[at:at + n]
            at += n
        starts = [0]
        for new, _ in reqs:
            starts.append(starts[-1] + new)
        q = _randn(g, (starts[-1], case["heads"], d), dtype)
        kv = _randn(g, (sum(pages), 2, page, hk, d), dtype)
        return {"case": case, "q": q, "kv": kv, "o": torch.empty_like(q),
                "starts": torch.tensor(starts, dtype=torch.int32, device="cuda"),
                "lens": torch.tensor([ctx for _, ctx in reqs], dtype=torch.int32, device="cuda"),
                "table": table.to("cuda"), "max_new": max(new for new, _ in reqs), "scale": d ** -0.5}
    rows, cols = case["rows"], case["cols"]
    if kind == "norm":
        x = _randn(g, (rows, cols), dtype)
        w = _randn(g, (cols,), dtype, 0.1, 1.0)
        res = _randn(g, (rows, cols), dtype, 3.0) if case["residual"] else None  # the stream grows over the layers
        return {"case": case, "x": x, "w": w, "res": res}
    if kind == "head":
        x = torch.randn(rows, cols, generator=g, device="cuda").mul_(4.0)
        far = torch.rand(rows, cols, generator=g, device="cuda")
        x = torch.where(far < 0.005, 30.0, torch.where(far > 0.995, -30.0, x))  # a few confident entries
        return {"case": case, "x": (x + torch.rand(rows, cols, generator=g, device="cuda")).to(dtype)}
    return {"case": case, "x": _randn(g, (rows, cols), dtype)}


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    ops = torch.ops.fxpr
    if kind == "linear":
        return ops.gemm_fxp(state["a"], state["b"], state["bias"], case["int_bits"], case["frac_bits"])
    if kind == "attn":
        ops.unified_attention_fxp(state["q"], state["kv"], state["o"], state["starts"], state["lens"], state["table"],
                                  state["max_new"], None, True, state["scale"], case["int_bits"], case["frac_bits"],
                                  case["softcap"], case["window"], 0)
        return state["o"]
    if kind == "norm":
        if state["res"] is None:
            return ops.rms_norm_fxp(state["x"], state["w"], EPS)
        y = ops.rms_norm_fxp_residual(state["x"], state["res"], state["w"], EPS)
        return {"y": y, "residual": state["res"]}
    if kind == "head":
        ids, lp, top, top_lp = ops.sample_greedy_fxp(state["x"], TOP, case["int_bits"], case["frac_bits"])
        full = ops.log_softmax_fxp(state["x"], case["int_bits"], case["frac_bits"], torch.float32)
        return {"ids": ids, "logprob": lp, "top": top, "top_logprobs": top_lp, "logprobs": full}
    q = ops.float_to_fixed(state["x"], case["int_bits"], case["frac_bits"])
    s = ops.fixed_row_sum(q, case["int_bits"])
    return {"q": q, "sums": s, "decoded": ops.fixed_to_float(q, 32, case["frac_bits"]),
            "decoded_sums": ops.fixed_to_float(s, 32, case["frac_bits"])}


def _visible(case):
    """(query, key) pairs that an attention case attends, over all requests, and the cache rows it has to read."""
    pairs = rows = 0
    w = case["window"]
    for new, ctx in _requests(case):
        first = ctx - new  # position of the first new token
        if not w:
            pairs += new * first + new * (new + 1) // 2
            rows += ctx
        else:
            for p in range(first, ctx):
                pairs += min(p + 1, w)
            rows += min(ctx, new + w - 1)
    return pairs, rows


def work(case):
    kind, es = case["kind"], SIZE[case["dtype"]]
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": es * (m * k + k * n + m * n + (n if case["bias"] else 0)), "flops": 2 * m * k * n}
    if kind == "attn":
        pairs, rows = _visible(case)
        tokens = sum(new for new, _ in _requests(case))
        d = case["head_dim"]
        return {"bytes": es * d * (2 * rows * case["kv_heads"] + 2 * tokens * case["heads"]),
                "flops": 4 * case["heads"] * d * pairs}
    n = case["rows"] * case["cols"]
    if kind == "norm":
        return {"bytes": es * (n * (4 if case["residual"] else 2) + case["cols"]), "flops": 4 * n}
    if kind == "head":
        return {"bytes": n * (es + 4), "flops": 4 * n}
    return {"bytes": n * (es + case["int_bits"] // 8 + 4), "flops": 3 * n}


def tolerance(case):
    """About four times the error against exact() that the operators show (16-bit outputs: their own rounding)."""
    kind = case["kind"]
    sixteen = case["dtype"] in ("bf16", "f16")
    if kind == "chain":
        return "exact"
    if kind == "linear":
        if case["int_bits"] == 16:
            return {"rel": 2e-2, "max": 0.1}  # each K-tile's partial is rounded to 2^-8
        return {"rel": 8e-3 if case["dtype"] == "bf16" else 1e-3 if sixteen else 1.2e-4, "max": 0.05 if sixteen else 2e-3}
    if kind == "attn":
        return {"rel": 1e-2 if case["dtype"] == "bf16" else 1.5e-3, "max": 0.1}
    if kind == "norm":
        return {"rel": 8e-3 if case["dtype"] == "bf16" else 1e-3 if sixteen else 1e-6, "max": 0.05 if sixteen else 1e-5}
    return {"rel": 5e-6, "max": 1e-4, "differ": 1e-4}


def _exact_attn(s):
    case = s["case"]
    group = case["heads"] // case["kv_heads"]
    out = torch.empty(s["q"].shape, dtype=torch.float64, device="cuda")
    starts, lens = s["starts"].tolist(), s["lens"].tolist()
    for i, ctx in enumerate(lens):
        rows = s["table"][i, :-(-ctx // case["page"])].long()
        k, v = (s["kv"][rows, j].flatten(0, 1)[:ctx].double() for j in (0, 1))  # [ctx, kv heads, d]
        lo, hi = starts[i], starts[i + 1]
        pos = torch.arange(ctx - (hi - lo), ctx, device="cuda")[:, None]
        key = torch.arange(ctx, device="cuda")[None, :]
        hide = key > pos
        if case["window"]:
            hide = hide | (key <= pos - case["window"])
        for h in range(case["heads"]):
            x = s["q"][lo:hi, h].double() @ k[:, h // group].t().contiguous() * s["scale"]
            if case["softcap"]:
                x = case["softcap"] * torch.tanh(x / case["softcap"])
            out[lo:hi, h] = torch.softmax(x.masked_fill_(hide, -math.inf), 1) @ v[:, h // group].contiguous()
    return out


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind == "linear":
        a, n, step = s["a"].double(), case["n"], 16384
        y = torch.empty(case["m"], n, dtype=torch.float64, device="cuda")
        for i in range(0, n, step):
            y[:, i:i + step] = a @ s["b"][:, i:i + step].double()
        return y if s["bias"] is None else y + s["bias"].double()
    if kind == "attn":
        return _exact_attn(s)
    x = s["x"].double()
    if kind == "norm":
        # the stream is stored, and normalised, in the activations' type
        v = x if s["res"] is None else x + s["res"].double()
        y = v * torch.rsqrt(v.square().mean(1, keepdim=True) + EPS) * s["w"].double()
        return y if s["res"] is None else {"y": y, "residual": v}
    if kind == "head":
        full = torch.log_softmax(x, 1)
        top = full.topk(TOP, 1).values
        return {"ids": None, "logprob": top[:, 0].contiguous(), "top": None, "top_logprobs": top, "logprobs": full}
    one, top = 2.0 ** case["frac_bits"], 2.0 ** (case["int_bits"] - 1)
    q = torch.round(x * one).clamp(-top, top - 1)
    return {"q": None, "sums": None, "decoded": q / one, "decoded_sums": q.sum(1).clamp(-top, top - 1) / one}
