"""Performance cases of the quantized-GEMM library: what a serving program has
it do, one pass at a time, through the public layer `hkq` (torch tensors over
the C ABI).

A transformer layer in this library is a chain of quantizers and GEMMs, so most
cases are single linear layers whose activations and weights are quantized
already, from one decoded token to a whole prefill, in each operand format:
per-token FP8 (A8W8), block-scaled FP8 (1x128 activations, 128x128 weights),
MXFP4 and bf16. The mixture-of-experts cases are whole layers (quantizer,
router metadata, gate/up, SwiGLU with quantization, down) or one grouped GEMM.

`prepare` keeps what a program keeps between steps: weights, output buffers, a
split workspace, bound calls. `exact` repeats the arithmetic in float64.
"""
from __future__ import annotations

import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "amd-kernels_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import hkq  # noqa: E402

DEV = "cuda"
FP8 = torch.float8_e4m3fn
BF16 = torch.bfloat16

# (N, K) of the linear layers that the benchmark and the tests use
A8W8_NK = [(6144, 4096), (4096, 4096), (28672, 4096), (4096, 14336), (14336, 4096)]
BLOCKSCALE_NK = [(24576, 1536), (7168, 18432), (7168, 2048), (2112, 7168)]
MXFP4_NK = [(8192, 8192), (8192, 4096), (4096, 8192)]
BF16_NK = [(4096, 4096), (6144, 4096), (14336, 4096)]
# (experts, top-k, hidden, ffn): the benchmark's mixture and two generic
# fine-grained ones (many small experts)
MOE = [(8, 2, 4096, 14336), (32, 4, 2048, 2816), (64, 8, 2048, 1408)]


def listed():
    return [
        # one decode step of four sequences through an attention output projection: launch latency counts
        {"name": "a8w8_decode", "kind": "a8w8", "M": 4, "N": 4096, "K": 4096},
        # continuous batching: one token of each of 96 running sequences, down projection
        {"name": "a8w8_batch", "kind": "a8w8", "M": 96, "N": 4096, "K": 14336},
        # a prefill chunk of odd length, fused query/key/value projection
        {"name": "a8w8_chunk", "kind": "a8w8", "M": 601, "N": 6144, "K": 4096},
        # a long prefill, gate projection: the benchmark's headline shape
        {"name": "a8w8_prefill", "kind": "a8w8", "M": 4096, "N": 14336, "K": 4096},
        # decode of 24 sequences, block-scaled down projection
        {"name": "blockscale_decode", "kind": "blockscale", "M": 24, "N": 7168, "K": 18432},
        # a prefill chunk through the block-scaled output projection
        {"name": "blockscale_chunk", "kind": "blockscale", "M": 500, "N": 7168, "K": 2048},
        # decode of 64 sequences with MXFP4 weights and activations
        {"name": "mxfp4_batch", "kind": "mxfp4", "M": 64, "N": 8192, "K": 8192},
        # a long prefill in MXFP4: the benchmark's second shape
        {"name": "mxfp4_prefill", "kind": "mxfp4", "M": 4096, "N": 8192, "K": 8192},
        # an unquantized linear layer during decode of 64 sequences
        {"name": "bf16_batch", "kind": "bf16", "M": 64, "N": 4096, "K": 4096},
        # a whole FP8 mixture-of-experts layer over a prefill
        {"name": "moe_a8w8_prefill", "kind": "moe_a8w8", "T": 4096, "E": 8, "topk": 2, "hidden": 4096, "ffn": 14336},
        # a whole block-scaled mixture-of-experts layer, decode of 64 sequences
        {"name": "moe_blockscale_batch", "kind": "moe_blockscale", "T": 64, "E": 8, "topk": 2, "hidden": 4096,
         "ffn": 14336},
        # the gate/up grouped GEMM in MXFP4 over a short chunk
        {"name": "moe_mxfp4_chunk", "kind": "moe_mxfp4", "T": 300, "E": 8, "topk": 2, "hidden": 4096, "ffn": 14336},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choice(["a8w8"] * 4 + ["blockscale"] * 3 + ["mxfp4"] * 2 + ["bf16", "moe_a8w8", "moe_blockscale", "moe_mxfp4"])
    if kind.startswith("moe"):
        E, topk, hidden, ffn = rng.choice(MOE)
        return {"kind": kind, "T": _log_int(rng, 1, 2048), "E": E, "topk": topk, "hidden": hidden, "ffn": ffn}
    nk = {"a8w8": A8W8_NK, "blockscale": BLOCKSCALE_NK, "mxfp4": MXFP4_NK, "bf16": BF16_NK}[kind]
    if rng.random() < 0.7:
        N, K = rng.choice(nk)
    else:  # generic sizes, ragged in N
        N, K = 4 * _log_int(rng, 256, 4096), 128 * _log_int(rng, 8, 64)
    return {"kind": kind, "M": _log_int(rng, 1, 4096), "N": N, "K": K}


# ---------------------------------------------------------------------------
# inputs (from the seed alone)
# ---------------------------------------------------------------------------
def _gen(seed, salt=0):
    return torch.Generator(device=DEV).manual_seed(1000 * (int(seed) % (1 << 40)) + salt)


def _randn(shape, g, std=1.0):
    return (torch.randn(shape, generator=g, device=DEV, dtype=torch.float32) * std).to(BF16)


def _weight_codes(rows, cols, g):
    """E4M3FN codes of normal weights, as an amax quantization leaves them (4.3 sigma at the top code)."""
    return torch.randn((rows, cols), generator=g, device=DEV).mul_(104.0).clamp_(-448.0, 448.0).to(FP8)


def _scales(shape, g, level):
    return (0.75 + 0.5 * torch.rand(shape, generator=g, device=DEV)) * level


def _quant(x, group):
    """The library's dynamic FP8 rule over groups of a row: (codes, scales)."""
    M, K = x.shape
    v = x.float().view(M, K // group, group)
    s = (v.abs().amax(dim=-1) / 448.0).clamp_min(1e-10)
    q = (v * (1.0 / s).unsqueeze(-1)).clamp(-448.0, 448.0).to(FP8)
    return q.view(M, K), s


def _fp4(rows, K, g):
    """Packed E2M1 codes of normal values [rows, K/2] and e8m0 scales [rows, K/32]."""
    q = torch.empty((rows, K // 2), dtype=torch.uint8, device=DEV)
    edges = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device=DEV)
    step = max(1, (1 << 27) // K)
    for r in range(0, rows, step):
        n = min(step, rows - r)
        v = torch.randn((n, K), generator=g, device=DEV).mul_(2.0)
        c = torch.bucketize(v.abs(), edges).to(torch.uint8) | ((v < 0).to(torch.uint8) << 3)
        q[r:r + n] = c[:, 0::2] | (c[:, 1::2] << 4)
    s = torch.randint(0, 2, (rows, K // 32), generator=g, device=DEV)
    return q, s


_E2M1 = [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0]


def _fp4_values(q, s):
    """float64 values of packed codes and e8m0 scales."""
    lut = torch.tensor(_E2M1, device=DEV, dtype=torch.float64)
    rows, half = q.shape
    v = torch.stack([lut[(q & 15).long()], lut[(q >> 4).long()]], dim=-1).view(rows, half // 16, 32)
    return (v * torch.exp2(s.double() - 127.0).unsqueeze(-1)).view(rows, 2 * half)


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _workspace(name, M, N, K):
    n = int(getattr(hkq.lib(), name)(M, N, K))
    return torch.empty(n, dtype=torch.uint8, device=DEV) if n else None


def _inputs(c, seed):
    k, g = c["kind"], _gen(seed)
    if k == "a8w8":
        M, N, K = c["M"], c["N"], c["K"]
        qa, sa = _quant(_randn((M, K), g), K)
        return {"qa": qa, "sa": sa.view(M).contiguous(), "qb": _weight_codes(N, K, g), "sb": _scales((N,), g, 0.02 / 104)}
    if k == "blockscale":
        M, N, K = c["M"], c["N"], c["K"]
        qa, sa = _quant(_randn((M, K), g), 128)
        return {"qa": qa, "sa": sa.contiguous(), "qb": _weight_codes(N, K, g),
                "sb": _scales((K // 128, (N + 127) // 128), g, 0.02 / 104)}
    if k == "mxfp4":
        M, N, K = c["M"], c["N"], c["K"]
        qa, ea = _fp4(M, K, g)
        qb, eb = _fp4(N, K, g)
        return {"qa": qa, "sa": (ea + 126).to(torch.uint8), "qb": qb, "sb": (eb + 120).to(torch.uint8)}
    if k == "bf16":
        return {"a": _randn((c["M"], c["K"]), g), "b": _randn((c["N"], c["K"]), g, 0.02)}
    T, E, topk, H, F = c["T"], c["E"], c["topk"], c["hidden"], c["ffn"]
    d = {"logits": _randn((T, E), g)}
    if k == "moe_mxfp4":
        d["qa"], ea = _fp4(T, H, g)
        d["sa"] = (ea + 126).to(torch.uint8)
        qb, eb = _fp4(E * 2 * F, H, g)
        d["qb"] = qb.view(E, 2 * F, H // 2)
        d["sb"] = (eb + 120).to(torch.uint8).view(E, 2 * F, H // 32)
        d["tw"] = torch.softmax(_top(d["logits"], topk)[0].float(), dim=-1).contiguous().view(-1)
        return d
    d["x"] = _randn((T, H), g)
    d["w1"] = torch.empty((E, 2 * F, H), dtype=FP8, device=DEV)
    d["w2"] = torch.empty((E, H, F), dtype=FP8, device=DEV)
    for e in range(E):
        d["w1"][e] = _weight_codes(2 * F, H, g)
        d["w2"][e] = _weight_codes(H, F, g)
    if k == "moe_blockscale":
        d["norm"] = 1.0 + _randn((H,), g, 0.1)
        d["s1"] = _scales((E, H // 128, 2 * F // 128), g, 0.02 / 104)
        d["s2"] = _scales((E, F // 128, H // 128), g, 0.02 / 104)
    else:
        d["s1"] = _scales((E, 2 * F), g, 0.02 / 104)
        d["s2"] = _scales((E, H), g, 0.02 / 104)
    return d


def _top(logits, topk):
    """Top-k experts per row, ties to the lower expert: (values, indices)."""
    v, i = torch.sort(logits.float(), dim=-1, descending=True, stable=True)
    return v[:, :topk], i[:, :topk]


# ---------------------------------------------------------------------------
# what a program keeps, and one pass
# ---------------------------------------------------------------------------
def prepare(case, seed):
    c = case
    s = _inputs(c, seed)
    s["kind"] = k = c["kind"]
    p = {n: t.data_ptr() for n, t in s.items() if isinstance(t, torch.Tensor)}
    if not k.startswith("moe"):
        M, N, K = c["M"], c["N"], c["K"]
        s["C"] = C = torch.empty((M, N), dtype=BF16, device=DEV)
        ws = None
        if k == "blockscale":
            s["call"] = hkq.bind("hkq_gemm_blockscale", p["qa"], p["qb"], p["sa"], p["sb"], C.data_ptr(), M, N, K, K, K,
                                 s["sa"].stride(0), s["sb"].stride(0), N, 128, _stream())
            return s
        s["ws"] = ws = _workspace({"a8w8": "hkq_gemm_a8w8_workspace", "mxfp4": "hkq_gemm_mxfp4_workspace",
                                   "bf16": "hkq_gemm_bf16_workspace"}[k], M, N, K)
        wp, wn = (ws.data_ptr(), ws.numel()) if ws is not None else (None, 0)
        if k == "a8w8":
            s["call"] = hkq.bind("hkq_gemm_a8w8_ws", p["qa"], p["qb"], p["sa"], p["sb"], C.data_ptr(), M, N, K, K, K, N,
                                 wp, wn, _stream())
        elif k == "mxfp4":
            s["call"] = hkq.bind("hkq_gemm_mxfp4_ws", p["qa"], p["sa"], p["qb"], p["sb"], C.data_ptr(), M, N, K, K // 2,
                                 K // 2, K // 32, K // 32, N, wp, wn, _stream())
        else:
            s["call"] = hkq.bind("hkq_batched_gemm_bf16", p["a"], p["b"], None, C.data_ptr(), 1, M, N, K, K, K, N, 0, 0,
                                 0, 0, wp, wn, _stream())
        return s
    T, E, topk, H, F = c["T"], c["E"], c["topk"], c["hidden"], c["ffn"]
    s["topk"] = topk
    if k == "moe_mxfp4":
        idx = _top(s["logits"], topk)[1].to(torch.int32).contiguous()
        sids, eids, _, total = hkq.align_block_size(idx, E, 128)
        n = int(total.item())
        s["sids"], s["eids"], s["n_gates"] = sids[:n], eids[:n // 128], T * topk
        s["Y1"] = torch.empty((T * topk, 2 * F), dtype=BF16, device=DEV)
        return s
    s["plan"], s["route"] = hkq.moe_routing_plan(s["logits"], topk, 128)
    n = T * topk
    block = k == "moe_blockscale"
    s["q1"] = torch.empty((T, H), dtype=FP8, device=DEV)
    s["sq1"] = torch.empty((T, H // 128) if block else (T,), dtype=torch.float32, device=DEV)
    s["Y1"] = torch.empty((n, 2 * F), dtype=BF16, device=DEV)
    s["q2"] = torch.empty((n, F), dtype=FP8, device=DEV)
    s["sq2"] = torch.empty((n, F // 128) if block else (n,), dtype=torch.float32, device=DEV)
    s["Y2"] = torch.empty((n, H), dtype=BF16, device=DEV)
    return s


def run(state):
    s = state
    k = s["kind"]
    if not k.startswith("moe"):
        s["call"]()
        return s["C"]
    if k == "moe_mxfp4":
        return hkq.moe_mxfp4(s["qa"], s["sa"], s["qb"], s["sb"], s["sids"], s["eids"], s["n_gates"], s["topk"],
                             topk_weights=s["tw"], C=s["Y1"])
    o = s["plan"]
    s["route"]()
    r = (o["hist"], o["offs"], o["expt_data"])
    if k == "moe_blockscale":
        hkq.rmsnorm_quant(s["x"], s["norm"], q=s["q1"], s=s["sq1"])
        hkq.moe_a8w8_blockscale(s["q1"], s["w1"], *r, s["topk"], s["sq1"], s["s1"], 128, 128, gather=o["gather"],
                                Y=s["Y1"])
        hkq.swiglu_quant(s["Y1"], group=128, q=s["q2"], s=s["sq2"])
        hkq.moe_a8w8_blockscale(s["q2"], s["w2"], *r, 1, s["sq2"], s["s2"], 128, 128, Y=s["Y2"])
    else:
        hkq.per_token_quant(s["x"], q=s["q1"], s=s["sq1"])
        hkq.moe_a8w8(s["q1"], s["w1"], *r, s["topk"], gather=o["gather"], x_scale=s["sq1"], w_scale=s["s1"], Y=s["Y1"])
        hkq.swiglu_quant(s["Y1"], q=s["q2"], s=s["sq2"])
        hkq.moe_a8w8(s["q2"], s["w2"], *r, 1, x_scale=s["sq2"], w_scale=s["s2"], Y=s["Y2"])
    return s["Y2"]


# ---------------------------------------------------------------------------
# necessary work, tolerance, float64 results
# ---------------------------------------------------------------------------
def work(case):
    c, k = case, case["kind"]
    if not k.startswith("moe"):
        M, N, K = c["M"], c["N"], c["K"]
        per = {"a8w8": 1.0, "blockscale": 1.0, "mxfp4": 0.5 + 1 / 32, "bf16": 2.0}[k]
        b = (M + N) * K * per + 2 * M * N
        if k == "a8w8":
            b += 4 * (M + N)
        elif k == "blockscale":
            b += 4 * (M * (K // 128) + (K // 128) * ((N + 127) // 128))
        return {"bytes": b, "flops": 2.0 * M * N * K}
    T, E, topk, H, F = c["T"], c["E"], c["topk"], c["hidden"], c["ffn"]
    n = T * topk
    active = E * (1.0 - (1.0 - topk / E) ** T)  # experts that some token chooses
    if k == "moe_mxfp4":
        return {"bytes": (0.5 + 1 / 32) * (active * 2 * F * H + T * H) + 2 * n * 2 * F, "flops": 4.0 * n * F * H}
    # layer input and output, the active experts' weights; between the GEMMs each buffer written and read once
    b = active * 3 * F * H + T * 2 * (H + E) + 2 * T * H + 2 * 2 * n * 2 * F + 2 * n * F + 2 * n * H
    return {"bytes": b, "flops": 6.0 * n * F * H}


def tolerance(case):
    # Against float64 the bf16 result of every single GEMM is off by 1.7e-3 of
    # the 2-norm (its rounding). In a layer some FP8 codes between the GEMMs
    # fall on the other side of a rounding boundary: measured 4.0e-3 with
    # per-token scales, 7.5e-3 with 1x128 ones. Four times each.
    return {"rel": {"moe_a8w8": 1.6e-2, "moe_blockscale": 3e-2}.get(case["kind"], 7e-3)}


def _e4m3_groups(y, group):
    """FP8 codes (as float64 values) and scales of float64 rows by the library's rule."""
    M, K = y.shape
    v = y.view(M, K // group, group)
    s = (v.abs().amax(dim=-1, keepdim=True) / 448.0).clamp_min(1e-10)
    q = (v / s).clamp(-448.0, 448.0).float().to(FP8).double()
    return (q * s).view(M, K)


def exact(case, seed):
    c, k = case, case["kind"]
    d = _inputs(c, seed)
    if k == "a8w8":
        return (d["qa"].double() @ d["qb"].double().t()) * d["sa"].double()[:, None] * d["sb"].double()[None, :]
    if k == "blockscale":
        M, N, K = c["M"], c["N"], c["K"]
        a = (d["qa"].double().view(M, K // 128, 128) * d["sa"].double()[:, :, None]).view(M, K)
        sb = d["sb"].double().repeat_interleave(128, dim=1)[:, :N].t()  # [N, K/128]
        b = (d["qb"].double().view(N, K // 128, 128) * sb[:, :, None]).view(N, K)
        return a @ b.t()
    if k == "mxfp4":
        return _fp4_values(d["qa"], d["sa"]) @ _fp4_values(d["qb"], d["sb"]).t()
    if k == "bf16":
        return d["a"].double() @ d["b"].double().t()
    T, E, topk, H, F = c["T"], c["E"], c["topk"], c["hidden"], c["ffn"]
    idx = _top(d["logits"], topk)[1].reshape(-1)  # expert of gate t*topk + j
    if k == "moe_mxfp4":
        a = _fp4_values(d["qa"], d["sa"])
        out = torch.empty((T * topk, 2 * F), dtype=torch.float64, device=DEV)
        for e in range(E):
            gates = (idx == e).nonzero().view(-1)
            if gates.numel():
                out[gates] = (a[gates // topk] @ _fp4_values(d["qb"][e], d["sb"][e]).t()) * d["tw"].double()[gates][:, None]
        return out
    gates = torch.argsort(idx, stable=True)  # expert-sorted rows
    x = d["x"].double()
    if k == "moe_blockscale":
        y = x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + 1e-6) * d["norm"].double()[None, :]
        a = _e4m3_groups(y, 128)
    else:
        a = _e4m3_groups(x, H)
    rows, out = 0, torch.empty((T * topk, H), dtype=torch.float64, device=DEV)
    for e in range(E):
        mine = gates[idx[gates] == e] // topk
        if mine.numel() == 0:
            continue
        w1, w2 = d["w1"][e].double(), d["w2"][e].double()
        if k == "moe_blockscale":
            w1 *= d["s1"][e].double().t().repeat_interleave(128, 0).repeat_interleave(128, 1)
            w2 *= d["s2"][e].double().t().repeat_interleave(128, 0).repeat_interleave(128, 1)
        else:
            w1 *= d["s1"][e].double()[:, None]
            w2 *= d["s2"][e].double()[:, None]
        y1 = (a[mine] @ w1.t()).to(BF16).double()  # the layer holds it in bf16
        g, u = y1[:, :F], y1[:, F:]
        act = g / (1.0 + torch.exp(-g)) * u
        out[rows:rows + mine.numel()] = _e4m3_groups(act, 128 if k == "moe_blockscale" else F) @ w2.t()
        rows += mine.numel()
    return out
