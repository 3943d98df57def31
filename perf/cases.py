"""The work that the performance of this library is measured on, through its public Python entry points.

Each case is one call, or one short chain of calls, that a serving or loading program makes.  ``listed()`` holds the
fixed ones, ``draw(rng)`` gives more of the same ranges.  ``prepare`` makes what such a program has in hand (inputs,
weights in the layout that it keeps, a captured graph), ``run`` is one pass, ``exact`` the same pass in plain torch
with 64-bit products and sums.

Kinds
  gemm     one block-FP8 linear layer on bf16 activations: ops.block_fp8_gemm
  layer    the block-FP8 part of one decoder layer at a decode batch, captured once in a HIP graph and replayed, as a
           serving loop runs it: add + RMSNorm + quantizer, QKV, output projection, add + RMSNorm + quantizer,
           gate_up, SiLU-and-mul + quantizer, down (attention itself is not part of this library: the query columns of
           the QKV output stand in for its result)
  channel  one per-token / per-channel W8A8 linear layer on bf16 activations: ops.token_channel_gemm
  moe      one block-FP8 mixture-of-experts layer: ops.moe_block_fp8
  rows     the row-wise operations between the linear layers of a prefill: ops.rms_norm_quant with its residual and
           ops.silu_mul_quant
  shard    one rank's part of a row-parallel linear layer: its K range as an fp32 partial, then the ordered sum of the
           gathered partials and the bf16 finish
  load     what loading does to one weight on the GPU: the finite check, both directions of the codec, the packing
"""

import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "gaudi-kernels_amd", "python"))

from gaudi_kernels import ops  # noqa: E402

DEV = "cuda"


def listed():
    return [
        # one token through a QKV projection: the smallest call, where the launch and the host path count
        dict(name="decode_m1", kind="gemm", m=1, n=6144, k=4096, packed=True, half=False, bias=False),
        # a batch of 40 sequences through a down projection in the half-range mode, on checkpoint-order weights
        dict(name="decode_m40_half", kind="gemm", m=40, n=4096, k=14336, packed=False, half=True, bias=True),
        # a decoder layer at batch 16
        dict(name="layer_m16", kind="layer", m=16, hidden=4096, kv=1024, inter=14336),
        # a short prompt, or a chunk of one, of an odd length
        dict(name="prefill_m300", kind="gemm", m=300, n=6144, k=4096, packed=True, half=False, bias=False),
        # a long prefill: the largest dense product
        dict(name="prefill_m4096", kind="gemm", m=4096, n=7168, k=7168, packed=True, half=False, bias=False),
        # a hidden size that is no multiple of the 128-column scale block, in both dimensions
        dict(name="ragged_k", kind="gemm", m=200, n=2880, k=2880, packed=False, half=False, bias=True),
        # a prefill through the per-token / per-channel path
        dict(name="channel_m2048", kind="channel", m=2048, n=7168, k=4096, bias=True),
        # a mixture-of-experts layer on a prefill chunk, and on a decode batch
        dict(name="moe_t512", kind="moe", t=512, hidden=4096, inter=14336, experts=8, top_k=2, packed=True, half=False),
        dict(name="moe_t16", kind="moe", t=16, hidden=4096, inter=14336, experts=8, top_k=2, packed=True, half=False),
        # the row operations of a long prefill of an odd length
        dict(name="rows_4093", kind="rows", m=4093, hidden=4096, inter=14336, half=False),
        # one of four ranks of a row-parallel down projection
        dict(name="shard_m256", kind="shard", m=256, n=4096, k=14336, ranks=4, packed=True, half=False),
        # loading one gate_up weight
        dict(name="load_gate_up", kind="load", n=28672, k=4096),
    ]


def _log(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def _of128(rng, lo, hi):
    return 128 * _log(rng, lo // 128, hi // 128)


def draw(rng):
    kind = rng.choice(["gemm", "gemm", "gemm", "gemm", "layer", "channel", "moe", "rows", "shard", "load"])
    flag = lambda: rng.random() < 0.5  # noqa: E731
    if kind == "gemm":
        if rng.random() < 0.15:  # a K that is no multiple of 128
            m, n, k = _log(rng, 1, 256), _log(rng, 200, 2880), _log(rng, 200, 2880)
            return dict(kind=kind, m=m, n=n, k=k + (k % 128 == 0), packed=False, half=flag(), bias=flag())
        m, k = _log(rng, 1, 4096), _of128(rng, 512, 14336)
        top = max(512, min(28672, 4096 * 7168 * 7168 // (m * k)))
        n = _of128(rng, 512, top) if flag() else _log(rng, 500, top)
        return dict(kind=kind, m=m, n=n, k=k, packed=flag(), half=rng.random() < 0.25, bias=rng.random() < 0.25)
    if kind == "layer":
        hidden = 128 * rng.randint(16, 32)
        return dict(kind=kind, m=_log(rng, 1, 64), hidden=hidden, kv=128 * rng.randint(2, 8),
                    inter=128 * rng.randint(32, 112))
    if kind == "channel":
        return dict(kind=kind, m=_log(rng, 1, 2048), n=_log(rng, 500, 7168), k=_of128(rng, 512, 4096), bias=flag())
    if kind == "moe":
        experts = rng.choice([4, 8, 16, 32])
        hidden = 128 * rng.randint(8, 32)
        inter = 128 * rng.randint(4, max(4, 112 * 8 // max(8, experts)))
        return dict(kind=kind, t=_log(rng, 1, 512), hidden=hidden, inter=inter, experts=experts,
                    top_k=rng.choice([1, 2, 2, 2]), packed=flag(), half=rng.random() < 0.25)
    if kind == "rows":
        return dict(kind=kind, m=_log(rng, 16, 4093), hidden=_log(rng, 1000, 4096), inter=_log(rng, 1000, 14336),
                    half=rng.random() < 0.25)
    if kind == "shard":
        ranks = rng.choice([2, 4, 8])
        return dict(kind=kind, m=_log(rng, 1, 256), n=_log(rng, 500, 4096), k=128 * ranks * rng.randint(4, 112 // ranks),
                    ranks=ranks, packed=flag(), half=rng.random() < 0.25)
    return dict(kind=kind, n=_log(rng, 500, 28672), k=_of128(rng, 512, 4096))


# ---- inputs ---------------------------------------------------------------------------------


def _weight(gen, n, k):
    """Trained-like weights: N(0, 0.02) with 5% of the 128 x 128 blocks eight times larger, quantized per block."""
    nb, g = -(-n // 128), -(-k // 128)
    w = torch.zeros(nb * 128, g * 128, device=DEV)
    w[:n, :k] = torch.randn(n, k, generator=gen, device=DEV) * 0.02
    big = torch.rand(nb, 1, g, 1, generator=gen, device=DEV) < 0.05
    w = w.view(nb, 128, g, 128)
    w *= torch.where(big, 8.0, 1.0)
    s = w.abs().amax(dim=(1, 3)) / 448.0
    s = torch.where(s > 0, s, torch.ones_like(s))
    q = (w / s[:, None, :, None]).clamp_(-448.0, 448.0).view(nb * 128, g * 128)[:n, :k]
    return q.to(torch.float8_e4m3fn).contiguous(), s.contiguous()


def _acts(gen, m, k):
    """Hidden states: N(0, 1) with 1% of the channels twenty times larger."""
    x = torch.randn(m, k, generator=gen, device=DEV)
    return (x * torch.where(torch.rand(k, generator=gen, device=DEV) < 0.01, 20.0, 1.0)).bfloat16()


def _bias(gen, n):
    return torch.randn(n, generator=gen, device=DEV) * 0.1


def _inputs(c, seed):
    """The case's inputs, made from the seed alone."""
    gen = torch.Generator(device=DEV).manual_seed(int(seed))
    kind = c["kind"]
    if kind == "gemm":
        w, s = _weight(gen, c["n"], c["k"])
        return dict(x=_acts(gen, c["m"], c["k"]), w=w, s=s, bias=_bias(gen, c["n"]) if c["bias"] else None)
    if kind == "layer":
        h, qkv, inter = c["hidden"], c["hidden"] + 2 * c["kv"], c["inter"]
        d = dict(x=_acts(gen, c["m"], h), res=_acts(gen, c["m"], h))
        for name in ("g1", "g2"):
            d[name] = (1.0 + 0.1 * torch.randn(h, generator=gen, device=DEV)).bfloat16()
        for name, n, k in (("qkv", qkv, h), ("o", h, h), ("gu", 2 * inter, h), ("dn", h, inter)):
            d["w_" + name], d["s_" + name] = _weight(gen, n, k)
        return d
    if kind == "channel":
        w = torch.randn(c["n"], c["k"], generator=gen, device=DEV) * 0.02
        sw = w.abs().amax(dim=1) / 448.0
        return dict(x=_acts(gen, c["m"], c["k"]), w=(w / sw[:, None]).to(torch.float8_e4m3fn), sw=sw,
                    bias=_bias(gen, c["n"]) if c["bias"] else None)
    if kind == "moe":
        d = dict(x=torch.randn(c["t"], c["hidden"], generator=gen, device=DEV).bfloat16(),
                 logits=torch.randn(c["t"], c["experts"], generator=gen, device=DEV))
        for name, n, k in (("gu", 2 * c["inter"], c["hidden"]), ("dn", c["hidden"], c["inter"])):
            d["w_" + name] = torch.empty(c["experts"], n, k, dtype=torch.float8_e4m3fn, device=DEV)
            d["s_" + name] = torch.empty(c["experts"], -(-n // 128), -(-k // 128), device=DEV)
            for e in range(c["experts"]):
                d["w_" + name][e], d["s_" + name][e] = _weight(gen, n, k)
        return d
    if kind == "rows":
        return dict(x=_acts(gen, c["m"], c["hidden"]), res=_acts(gen, c["m"], c["hidden"]),
                    g=(1.0 + 0.1 * torch.randn(c["hidden"], generator=gen, device=DEV)).bfloat16(),
                    gu=_acts(gen, c["m"], 2 * c["inter"]))
    if kind == "shard":
        w, s = _weight(gen, c["n"], c["k"])
        gathered = torch.randn(c["ranks"] * c["m"] * c["n"], generator=gen, device=DEV)
        return dict(x=_acts(gen, c["m"], c["k"]), w=w, s=s, gathered=gathered, bias=_bias(gen, c["n"]))
    w, s = _weight(gen, c["n"], c["k"])
    return dict(w=w, s=s)


def _layer(d, m):
    q, sa, r1 = ops.rms_norm_quant(d["x"], d["g1"], 1e-5, residual=d["res"], decode_layout=True)
    qkv = ops.block_fp8_gemm_q(q, sa, m, d["w_qkv"], d["s_qkv"], decode_layout=True)
    o = ops.block_fp8_gemm(qkv[:, : d["x"].shape[1]], d["w_o"], d["s_o"], workspace=d["ws"])
    q, sa, r2 = ops.rms_norm_quant(o, d["g2"], 1e-5, residual=r1, decode_layout=True)
    gu = ops.block_fp8_gemm_q(q, sa, m, d["w_gu"], d["s_gu"], decode_layout=True)
    q, sa = ops.silu_mul_quant(gu, decode_layout=True)
    return qkv, o, r2, gu, ops.block_fp8_gemm_q(q, sa, m, d["w_dn"], d["s_dn"], decode_layout=True)


def prepare(case, seed):
    d = _inputs(case, seed)
    kind = case["kind"]
    if kind == "layer":
        for name in ("w_qkv", "w_o", "w_gu", "w_dn"):
            d[name] = ops.pack_weight(d[name])
        d["ws"] = ops.make_workspace(case["m"], case["hidden"], case["hidden"])
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):  # a first pass outside the graph, as capture asks for
            _layer(d, case["m"])
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        d["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(d["graph"]):
            d["out"] = _layer(d, case["m"])
    elif kind == "moe":
        if case["packed"]:
            d["w_gu"], d["w_dn"] = ops.pack_experts(d["w_gu"]), ops.pack_experts(d["w_dn"])
    elif case.get("packed"):
        d["w"] = ops.pack_weight(d["w"])
    return case, d


def run(state):
    case, d = state
    kind = case["kind"]
    if kind == "gemm":
        return ops.block_fp8_gemm(d["x"], d["w"], d["s"], d["bias"], native_half=case["half"])
    if kind == "layer":
        d["graph"].replay()
        return d["out"]
    if kind == "channel":
        return ops.token_channel_gemm(d["x"], d["w"], d["sw"], d["bias"])
    if kind == "moe":
        return ops.moe_block_fp8(d["x"], d["logits"], d["w_gu"], d["s_gu"], d["w_dn"], d["s_dn"],
                                 top_k=case["top_k"], native_half=case["half"])
    if kind == "rows":
        return (ops.rms_norm_quant(d["x"], d["g"], 1e-5, residual=d["res"], native_half=case["half"])
                + ops.silu_mul_quant(d["gu"], native_half=case["half"]))
    if kind == "shard":
        step = case["k"] // case["ranks"]
        part = ops.block_fp8_gemm_kslice(d["x"], d["w"], d["s"], step * (case["ranks"] - 1), step,
                                         native_half=case["half"])
        total = ops.rank_sum(d["gathered"], case["ranks"]).view(case["m"], case["n"])
        return part, ops.partial_finish(total, d["bias"])
    half, s2, rounded = ops.codec_ocp_to_half(d["w"], d["s"])
    back, s1 = ops.codec_half_to_ocp(half, s2)
    return half, s2, rounded, back, s1, ops.weights_finite(d["w"], d["s"]), ops.pack_weight(d["w"]).data


# ---- what a pass cannot do without --------------------------------------------------------------


def _linear(m, n, k, x=2, y=2):
    """Bytes of one block-scaled linear layer: weights, scales, activations in, outputs out."""
    return n * k + 4 * -(-n // 128) * -(-k // 128) + x * m * k + y * m * n


def work(case):
    c, kind = case, case["kind"]
    if kind == "gemm":
        return dict(bytes=_linear(c["m"], c["n"], c["k"]) + (4 * c["n"] if c["bias"] else 0),
                    flops=2 * c["m"] * c["n"] * c["k"])
    if kind == "layer":
        m, h, i = c["m"], c["hidden"], c["inter"]
        shapes = ((h + 2 * c["kv"], h), (h, h), (2 * i, h), (h, i))
        # the residual stream in and out once, the returned outputs out once
        nbytes = sum(_linear(m, n, k, x=0) for n, k in shapes) + 2 * m * h * 3 + 4 * h
        return dict(bytes=nbytes, flops=sum(2 * m * n * k for n, k in shapes))
    if kind == "channel":
        nbytes = c["n"] * c["k"] + 4 * c["n"] * (2 if c["bias"] else 1) + 2 * c["m"] * (c["k"] + c["n"])
        return dict(bytes=nbytes, flops=2 * c["m"] * c["n"] * c["k"])
    if kind == "moe":
        t, h, i, e = c["t"], c["hidden"], c["inter"], min(c["experts"], c["t"] * c["top_k"])
        if t * c["top_k"] < 4 * c["experts"]:  # a small batch leaves experts out: their expected number
            e = round(c["experts"] * (1 - (1 - c["top_k"] / c["experts"]) ** t))
        nbytes = e * (3 * i * h + 4 * 3 * (i // 128) * (h // 128)) + 4 * t * h + 4 * t * c["experts"]
        return dict(bytes=nbytes, flops=2 * t * c["top_k"] * 3 * i * h)
    if kind == "rows":
        m, h, i = c["m"], c["hidden"], c["inter"]
        gh, gi = -(-h // 128), -(-i // 128)
        return dict(bytes=m * (6 * h + gh * 132) + 2 * h + m * (4 * i + gi * 132), flops=0)
    if kind == "shard":
        m, n, step = c["m"], c["n"], c["k"] // c["ranks"]
        nbytes = _linear(m, n, step, y=4) + 4 * m * n * c["ranks"] + 2 * m * n + 4 * n
        return dict(bytes=nbytes, flops=2 * m * n * step)
    # one weight in, the half-range, the OCP and the packed codes out, and its three scale grids
    return dict(bytes=4 * c["n"] * c["k"] + 12 * -(-c["n"] // 128) * (c["k"] // 128), flops=0)


def tolerance(case):
    """What another correct implementation at the same precision may differ by.  Measured against exact(): one linear
    layer 1.7e-3 (its bf16 rounding; 4.1e-3 at most; another order of the sums moves 1e-4 of the values by one bf16
    ulp), the MoE layer 2.8e-3 (5.3e-2 at most: an intermediate value that rounds the other way moves an E4M3 code by
    up to 6%), the decoder layer's chain 5.7e-3 to 2.9e-2 (0.15 at most) by the same cause over four linear layers,
    the row operations' scales 2.1e-5 (5.1e-3 at most) and 2.6e-6 of their codes."""
    kind = case["kind"]
    if kind == "load":
        return "exact"
    if kind == "rows":
        return {"rel": 1e-4, "max": 0.02, "differ": 1e-4}
    if kind == "moe":
        return {"rel": 0.011, "max": 0.25}
    if kind == "layer":
        return {"rel": 0.03, "max": 0.6}
    return {"rel": 3e-3, "max": 0.016}  # two bf16 roundings apart


# ---- the same passes in plain torch, 64-bit products and sums ---------------------------------------


def _e4m3(v):
    return v.clamp(-448.0, 448.0).to(torch.float8_e4m3fn).double()


def _quant(x, half=False):
    """bf16 [m, k] -> (dequantized fp64 [m, k], scales fp64 [groups, m]): the 1 x 128 activation quantizer."""
    m, k = x.shape
    g = -(-k // 128)
    xp = torch.zeros(m, g * 128, device=DEV)
    xp[:, :k] = x.float()
    xp = xp.view(m, g, 128)
    s = xp.abs().amax(dim=2).clamp_min(1e-10) * torch.tensor(1.0 / 448.0, device=DEV)
    v = _e4m3(xp / s[:, :, None])
    if half:
        v, s = _e4m3((v * 0.5).float()), s * 2.0
    return (v * s.double()[:, :, None]).reshape(m, g * 128)[:, :k], s.t().double()


def _deq(w, s, half=False):
    v = _e4m3(w.float() * 0.5) * 2.0 if half else w.double()
    n, k = w.shape
    return v * s.double().repeat_interleave(128, 0)[:n].repeat_interleave(128, 1)[:, :k]


def _swiglu(gu):
    g, u = gu.double().chunk(2, dim=1)
    return (torch.nn.functional.silu(g) * u).bfloat16()


def _norm(x, res, gamma):
    r = (x.float() + res.float()).bfloat16()
    v = r.double()
    return r, (v * torch.rsqrt(v.square().mean(dim=1, keepdim=True) + 1e-5) * gamma.double()).bfloat16()


def exact(case, seed):
    d, kind = _inputs(case, seed), case["kind"]
    half = case.get("half", False)
    if kind == "gemm":
        y = _quant(d["x"], half)[0] @ _deq(d["w"], d["s"], half).t()
        return y if d["bias"] is None else y + d["bias"].double()
    if kind == "layer":
        lin = lambda x, name: _quant(x)[0] @ _deq(d["w_" + name], d["s_" + name]).t()  # noqa: E731
        r1, n1 = _norm(d["x"], d["res"], d["g1"])
        qkv = lin(n1, "qkv")
        o = lin(qkv[:, : case["hidden"]].bfloat16(), "o")
        r2, n2 = _norm(o.bfloat16(), r1, d["g2"])
        gu = lin(n2, "gu")
        return qkv, o, r2.double(), gu, lin(_swiglu(gu.bfloat16()), "dn")
    if kind == "channel":
        x = d["x"].float()
        m = x.abs().amax(dim=1, keepdim=True)
        s = (torch.where(m > 0, m, torch.ones_like(m)).double() / 448.0).float()
        half_codes = _e4m3((_e4m3(x / s) * 0.5).float())  # the token quantizer's half-range codes
        y = (half_codes * (2.0 * s.double())) @ (d["w"].double() * d["sw"].double()[:, None]).t()
        return y if d["bias"] is None else y + d["bias"].double()
    if kind == "moe":
        k = case["top_k"]
        top, ids = torch.sort(d["logits"].double(), dim=1, descending=True, stable=True)
        wts = torch.softmax(top[:, :k], dim=1)
        xq = _quant(d["x"], half)[0]
        y = torch.zeros(case["t"], case["hidden"], dtype=torch.float64, device=DEV)
        for e in range(case["experts"]):
            t, slot = (ids[:, :k] == e).nonzero(as_tuple=True)
            if t.numel():
                gu = xq[t] @ _deq(d["w_gu"][e], d["s_gu"][e], half).t()
                z = _quant(_swiglu(gu.bfloat16()), half)[0] @ _deq(d["w_dn"][e], d["s_dn"][e], half).t()
                y.index_add_(0, t, z * wts[t, slot][:, None])
        return y
    if kind == "rows":
        r, n = _norm(d["x"], d["res"], d["g"])
        return None, _quant(n, half)[1], r.double(), None, _quant(_swiglu(d["gu"]), half)[1]
    if kind == "shard":
        step = case["k"] // case["ranks"]
        k0 = step * (case["ranks"] - 1)
        part = _quant(d["x"][:, k0:], half)[0] @ _deq(d["w"][:, k0:], d["s"][:, k0 // 128:], half).t()
        total = d["gathered"].double().view(case["ranks"], case["m"], case["n"]).sum(dim=0)
        return part, total + d["bias"].double()
    return None, d["s"].double() * 2.0, None, None, d["s"].double(), None, None
