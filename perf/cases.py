"""The work that users of this library have it do, as cases that can be timed and compared.

A case is one pass through a public entry point: an MoE layer (decode or prefill) in one of
the three weight formats, a single LUT matrix times a few vectors, a dequantisation, or an
encoding.  ``listed`` names the common ones, ``draw`` gives others of the same ranges:
1 to 4096 tokens, hidden sizes 512 to 4096, 8 to 64 experts, top-1 to top-8, shared experts
in LUT slots or dense bf16, matrices from 40 thousand to 50 million weights.  Weights are
random codes over tables of the values that k-means gives for Gaussian weights (std 0.02),
activations N(0, 1) in bf16, router logits N(0, 1) (NestedLUT layers: Zipf(1.1) popularity).
"""
import math

import numpy as np
import torch

from block_lut_amd import ops
from block_lut_amd.decompress import decompress_blocklut
from block_lut_amd.fast_moe import fused_lut_moe
from block_lut_amd.formats import BL4Stack, MoEWeights, NestedExpert, NestedStack, RefStack
from block_lut_amd.lut_gemv import lut_gemv
from block_lut_amd.moe_layer import LUTMoELayer
from block_lut_amd.quant_method import LUTConfig, LUTFusedMoEMethod

DEV = "cuda"
STD = 0.02

# layer shapes: hidden, intermediate, routed experts, top-k
QWEN = dict(H=2048, I=1408, E=60, k=4)        # Qwen1.5-MoE-A2.7B
DEEPSEEK = dict(H=2048, I=1408, E=64, k=6)    # DeepSeek-V2-Lite
MIXTRAL = dict(H=4096, I=14336, E=8, k=2)     # Mixtral-8x7B


def _layer(fmt, entry, T, shape, S=0, dense=0, renorm=False, f32_out=False, **more):
    """fmt: ref / bl4 / nested weights.  entry: "logits" (moe_forward_logits with the
    caller's buffers), "apply" (the quant method), "fused" (fused_lut_moe), "module"
    (LUTMoELayer).  S: shared experts as LUT slots, dense: width of a dense shared expert."""
    return dict(kind="layer", fmt=fmt, entry=entry, T=T, S=S, dense=dense, renorm=renorm, f32_out=f32_out,
                **shape, **more)


def listed():
    return [
        # one token of one sequence: the latency of a chat on one GPU
        _layer("bl4", "logits", 1, QWEN, name="qwen_bl4_decode_t1"),
        # a small serving batch; fp32 results, as a caller that adds the residual in fp32 asks for
        _layer("bl4", "logits", 8, QWEN, f32_out=True, name="qwen_bl4_decode_t8_f32"),
        # the reference's own weight format behind its quant method, an odd batch
        _layer("ref", "apply", 19, QWEN, name="qwen_ref_decode_t19"),
        # experts at mixed 2/3/4-bit tiers, popularity as tiers are chosen by: decode and prefill
        _layer("nested", "logits", 16, QWEN, name="qwen_nested_decode_t16"),
        _layer("nested", "logits", 1024, QWEN, name="qwen_nested_prefill_t1024"),
        # few large experts, a full decode batch
        _layer("bl4", "logits", 64, MIXTRAL, renorm=True, name="mixtral_bl4_decode_t64"),
        # the reference's format through its fused function: a ragged prompt
        _layer("ref", "fused", 1531, DEEPSEEK, name="deepseek_ref_prefill_t1531"),
        # a whole block, router and dense shared expert with its gate included: a short prompt
        _layer("bl4", "module", 333, QWEN, dense=5632, name="qwen_block_prefill_t333"),
        # a long prompt, two shared experts as LUT slots
        _layer("bl4", "logits", 2048, DEEPSEEK, S=2, name="deepseek_bl4_prefill_t2048"),
        # the reference's single-matrix GEMV at the shape it quotes (the smallest call)
        dict(kind="gemv", entry="lut_gemv", fmt="ref", M=2816, K=2048, T=1, x32=False, name="ref_gemv_2816x2048"),
        # an expert's matrix expanded to bf16, as the reference's decompressor does it
        dict(kind="dequant", entry="decompress", fmt="ref", M=2816, K=2048, name="ref_dequant_2816x2048"),
        # the same matrix quantised (the reference's encoder)
        dict(kind="encode", fmt="ref", M=2816, K=2048, name="ref_encode_2816x2048"),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["layer"] * 8 + ["gemv", "dequant", "encode"])
    if kind == "gemv":
        entry = rng.choice(["lut_gemv", "stack"])
        fmt = "ref" if entry == "lut_gemv" else rng.choice(["bl4", "ref", "nested"])
        K = 64 * _log(rng, 8, 64)
        if entry == "lut_gemv" and rng.random() < 0.25:
            K += rng.randrange(1, 64)
        return dict(kind=kind, entry=entry, fmt=fmt, M=_log(rng, 256, 6000), K=K, T=_log(rng, 1, 8),
                    x32=entry == "stack" and fmt != "nested" and rng.random() < 0.4)
    if kind == "dequant":
        entry = rng.choice(["decompress", "stack"])
        fmt = "ref" if entry == "decompress" else rng.choice(["bl4", "nested"])
        return dict(kind=kind, entry=entry, fmt=fmt, M=_log(rng, 80, 12000), K=64 * _log(rng, 8, 64))
    if kind == "encode":
        return dict(kind=kind, fmt="ref", M=_log(rng, 80, 2816), K=64 * _log(rng, 8, 32))
    fmt = rng.choice(["bl4", "ref", "nested"])
    family = rng.choice(["qwen", "deepseek", "mixtral", "other", "other"])
    if family == "mixtral":
        shape, top = MIXTRAL, 96
    elif family == "other":
        H, inter, E = 64 * _log(rng, 8, 64), 64 * _log(rng, 4, 44), _log(rng, 8, 64)
        shape = dict(H=H, I=inter, E=E, k=rng.randint(1, min(8, E)))
        top = 4096
    else:
        shape, top = (QWEN if family == "qwen" else DEEPSEEK), 4096
    S = rng.choice([0, 0, 1, 2]) if family != "mixtral" else 0
    dense = 64 * _log(rng, 8, 88) if S == 0 and family != "mixtral" and rng.random() < 0.3 else 0
    entries = ["logits", "module"]
    if fmt == "ref" and S == 0 and dense == 0:
        entries += ["apply", "fused"]
    # no more multiplications than the long prompt's: 2048 tokens x (6 + 2) experts
    most = 2048 * 8 * 2048 * 1408 // (shape["H"] * (shape["I"] * (shape["k"] + S) + dense))
    return _layer(fmt, rng.choice(entries), _log(rng, 1, max(1, min(top, most))), shape, S=S, dense=dense,
                  renorm=rng.random() < 0.3, f32_out=False)


# ------------------------------------------------------------------ inputs

def _levels(n):
    """n sorted quantisation levels of a unit Gaussian (quantile midpoints)."""
    q = (torch.arange(n, dtype=torch.float64) + 0.5) / n
    return (math.sqrt(2) * torch.erfinv(2 * q - 1)).to(torch.float32)


def _codebook():
    """The global 256-entry codebook of weights divided by their block's largest."""
    return (_levels(256) / 2.9).clamp(-1, 1).to(torch.bfloat16).to(DEV)


def _tables(g, lead, n):
    """Per-block tables [*lead, n], bf16: each block's k-means levels."""
    t = torch.randn(lead + (n,), generator=g, device=DEV)
    t.mul_(0.04).add_(_levels(n).to(DEV)).mul_(torch.rand(lead + (1,), generator=g, device=DEV).mul_(0.4).add_(0.8))
    return t.mul_(STD).to(torch.bfloat16)


def _bytes(g, *shape):
    return torch.randint(0, 256, shape, dtype=torch.uint8, generator=g, device=DEV)


def _ref_tensors(g, E, M, K):
    am = (torch.rand((E, -(-M * K // 128)), generator=g, device=DEV) * 0.6 + 0.8) * (2.9 * STD)
    return _bytes(g, E, M, K), am.to(torch.bfloat16)


def _bits(E):
    """A third of the experts at each tier."""
    return [(2, 3, 4)[(e * 7) % 3] for e in range(E)]


def _stack(g, fmt, E, M, K):
    if fmt == "ref":
        codes, am = _ref_tensors(g, E, M, K)
        return RefStack(codes, am, _codebook(), 128)
    if fmt == "bl4":
        return BL4Stack(_bytes(g, E, M, K // 2), _tables(g, (E, M, K // 64), 16))
    return NestedStack([NestedExpert(b, _bytes(g, M * K * b // 8), _tables(g, (M, K // 64), 1 << b))
                        for b in _bits(E)], M, K)


def _popularity(c):
    """Log popularity of the experts (NestedLUT layers), in an order that mixes the tiers."""
    E = c["E"]
    if c["fmt"] != "nested":
        return np.zeros(E, np.float32)
    rank = np.array([(e * 11) % E if math.gcd(11, E) == 1 else e for e in range(E)]) + 1
    return (-1.1 * np.log(rank)).astype(np.float32)


def _logits(c, g):
    T, E = c["T"], c["E"]
    if c["fmt"] == "nested":   # popularity + Gumbel noise: top-k samples without replacement
        u = torch.rand((T, E), generator=g, device=DEV).clamp_(1e-6, 1 - 1e-6)
        return torch.from_numpy(_popularity(c)).to(DEV) - torch.log(-torch.log(u))
    return torch.randn((T, E), generator=g, device=DEV)


def _route(c, logits):
    ids = torch.sort(logits, dim=-1, descending=True, stable=True).indices[:, :c["k"]]   # ties to the lower id
    w = torch.softmax(logits if logits.dtype == torch.float64 else logits.float(), dim=-1).gather(1, ids)
    if c["renorm"]:
        w = w / w.sum(-1, keepdim=True)
    return w.contiguous(), ids.to(torch.int32).contiguous()


def _prepare_layer(c, g):
    T, H, I, E, S = c["T"], c["H"], c["I"], c["E"], c["S"]
    s = dict(case=c, x=torch.randn((T, H), generator=g, device=DEV).to(torch.bfloat16), logits=_logits(c, g))
    if c["entry"] in ("apply", "fused"):
        w13, a13 = _ref_tensors(g, E, 2 * I, H)
        w2, a2 = _ref_tensors(g, E, H, I)
        s["topk"] = _route(c, s["logits"])
        s["raw"] = (w13, a13, w2, a2, _codebook())
        if c["entry"] == "apply":
            method = LUTFusedMoEMethod(LUTConfig())
            layer = torch.nn.Module()
            method.create_weights(layer, E, H, I, device=DEV)
            for name, t in (("w13_weight", w13), ("w13_absmax", a13), ("w2_weight", w2), ("w2_absmax", a2),
                            ("_codebook", s["raw"][4])):
                getattr(layer, name).data = t.view(getattr(layer, name).shape)
            method.process_weights_after_loading(layer)
            s["method"], s["layer"] = method, layer
        return s
    w13, w2 = _stack(g, c["fmt"], E + S, 2 * I, H), _stack(g, c["fmt"], E + S, H, I)
    dense = gate = None
    if c["dense"]:
        dense = tuple((torch.randn(sh, generator=g, device=DEV) * STD).to(torch.bfloat16)
                      for sh in ((2 * c["dense"], H), (H, c["dense"])))
        gate = (torch.randn(H, generator=g, device=DEV) * STD).to(torch.bfloat16)
    s["moe"] = MoEWeights(w13, w2, H, I, E, S, shared_gate=gate, dense_shared=dense)
    if c["entry"] == "module":
        router = (torch.randn((E, H), generator=g, device=DEV) * STD).to(torch.bfloat16)
        s["block"] = LUTMoELayer(s["moe"], router, c["k"], renormalize=c["renorm"])
    else:
        s["out"] = torch.empty((T, H), dtype=torch.float32 if c["f32_out"] else torch.bfloat16, device=DEV)
        s["ws"] = ops.new_workspace(s["moe"], T, c["k"], DEV)
    return s


def prepare(case, seed):
    c = dict(case)
    g = torch.Generator(device=DEV).manual_seed(seed)
    if c["kind"] == "layer":
        return _prepare_layer(c, g)
    M, K = c["M"], c["K"]
    if c["kind"] == "gemv":
        x = torch.randn((c["T"], K), generator=g, device=DEV)
        x = x if c["x32"] else x.to(torch.bfloat16)
        if c["entry"] == "lut_gemv":
            codes, am = _ref_tensors(g, 1, M, K)
            return dict(case=c, x=x, codes=codes[0], absmax=am[0], codebook=_codebook())
        return dict(case=c, x=x, stack=_stack(g, c["fmt"], 1, M, K))
    if c["kind"] == "dequant":
        if c["entry"] == "decompress":
            codes, am = _ref_tensors(g, 1, M, K)
            return dict(case=c, codes=codes.reshape(-1), absmax=am[0], codebook=_codebook())
        return dict(case=c, stack=_stack(g, c["fmt"], 1, M, K))
    w = (torch.randn((M, K), generator=g, device=DEV) * STD).to(torch.bfloat16)
    return dict(case=c, weight=w, codebook=_codebook().float())


# ------------------------------------------------------------------ one pass

def run(s):
    c = s["case"]
    if c["kind"] == "layer":
        if c["entry"] == "logits":
            return ops.moe_forward_logits(s["moe"], s["x"], s["logits"], c["k"], renormalize=c["renorm"],
                                          out=s["out"], workspace=s["ws"])
        if c["entry"] == "module":
            return s["block"](s["x"])
        w, ids = s["topk"]
        if c["entry"] == "apply":
            return s["method"].apply(s["layer"], s["x"], w, ids)
        w13, a13, w2, a2, cb = s["raw"]
        return fused_lut_moe(s["x"], ids, w, w13, a13, w2, a2, cb)
    if c["kind"] == "gemv":
        if c["entry"] == "lut_gemv":
            return lut_gemv(s["x"], s["codes"], s["codebook"], s["absmax"])
        return ops.gemv(s["stack"], s["x"])
    if c["kind"] == "dequant":
        if c["entry"] == "decompress":
            return decompress_blocklut(s["codes"], s["absmax"], s["codebook"])
        return ops.dequant(s["stack"])
    return ops.ref_encode(s["weight"], s["codebook"])


# ------------------------------------------------------------------ what a pass cannot do without

def _weight_bytes(fmt, n, bits=4):
    if fmt == "ref":
        return n * (1 + 2 / 128)
    return n * bits / 8 + n / 64 * 2 ** bits * 2 if fmt == "nested" else n * 1.0


def _expected_experts(c):
    """Share of passes that touch each expert: the routing simulated for 64 passes (one for long ones)."""
    rng = np.random.default_rng(1)
    passes = max(1, 64 // c["T"])
    lg = _popularity(c) + rng.gumbel(size=(passes, c["T"], c["E"]))
    top = np.argpartition(-lg, c["k"] - 1, axis=-1)[..., :c["k"]].reshape(passes, -1)
    return np.mean([np.bincount(t, minlength=c["E"]) > 0 for t in top], axis=0)


def work(case):
    c = dict(case)
    if c["kind"] == "layer":
        T, H, I, k, S = c["T"], c["H"], c["I"], c["k"], c["S"]
        share = list(_expected_experts(c)) + [1.0] * S
        byte = sum(p * _weight_bytes(c["fmt"], 3 * H * I, b) for p, b in zip(share, _bits(c["E"] + S)))
        byte += 3 * H * c["dense"] * 2 + T * H * (2 + (4 if c["f32_out"] else 2))
        flops = 6 * T * H * (I * (k + S) + c["dense"])
        if c["entry"] == "module":
            byte += c["E"] * H * 2
            flops += 2 * T * H * c["E"]
        else:
            byte += T * c["E"] * 4 if c["entry"] == "logits" else T * k * 8
        return dict(bytes=byte, flops=flops)
    n = c["M"] * c["K"]
    if c["kind"] == "gemv":
        return dict(bytes=_weight_bytes(c["fmt"], n, 2) + c["T"] * (c["K"] * (4 if c["x32"] else 2) + c["M"] * 2),
                    flops=2 * n * c["T"])
    if c["kind"] == "dequant":
        return dict(bytes=_weight_bytes(c["fmt"], n, 2) + 2 * n, flops=0)
    return dict(bytes=3 * n + 2 * n / 128, flops=0)


def tolerance(case):
    if case["kind"] in ("dequant", "encode"):
        return "exact"
    if case["kind"] == "gemv":
        # fp32 sums rounded to bf16: 1.6e-3 against 64 bits
        return dict(rel=6e-3)
    # fp32 sums: 1.7e-5 against 64 bits (some of the activations between the two projections
    # round to the neighbouring bf16 value), 1.7e-3 once the result is rounded to bf16
    return dict(rel=1e-4) if case["f32_out"] else dict(rel=7e-3)


# ------------------------------------------------------------------ the same in 64 bits

def _dequant64(stack, e, rounded=True):
    """float64 [M, K] of expert e, by the format's definition."""
    M, K = stack.rows, stack.cols
    if isinstance(stack, RefStack):
        cb = stack.codebook.double()
        am = stack.absmax[e].double().repeat_interleave(stack.block_size)[:M * K].view(M, K)
        w = cb[stack.codes[e].int()] * am      # products of two bf16 are exact in fp32
        return w.float().to(torch.bfloat16).double() if rounded else w
    if isinstance(stack, BL4Stack):
        b = stack.codes[e]
        code = torch.stack([b & 15, b >> 4], dim=-1).view(M, K // 64, 64).long()
        return stack.tables[e].double().gather(2, code).view(M, K)
    ex, n = stack.experts[e], M * K
    p = ex.planes
    shifts = torch.arange(4, device=DEV, dtype=torch.uint8) * 2
    code = ((p[:n // 4, None] >> shifts) & 3).view(-1)
    one = torch.arange(8, device=DEV, dtype=torch.uint8)
    for bit, at in ((2, n // 4), (3, n // 4 + n // 8)):
        if ex.bits > bit:
            code = code | (((p[at:at + n // 8, None] >> one) & 1).view(-1) << bit)
    return ex.table.double().gather(2, code.view(M, K // 64, 64).long()).view(M, K)


def _mlp64(x, w13, w2):
    h = x @ w13.T
    half = h.shape[1] // 2
    act = torch.nn.functional.silu(h[:, :half]) * h[:, half:]
    return act.to(torch.bfloat16).double() @ w2.T     # the layer's definition rounds it


def exact(case, seed):
    c = dict(case)
    s = prepare(c, seed)
    if c["kind"] == "encode":
        w = s["weight"].double().view(-1)
        w = torch.nn.functional.pad(w, (0, -w.numel() % 128)).view(-1, 128)
        return [None, w.abs().amax(1).clamp_min(1e-10)]
    if c["kind"] == "dequant":
        if c["entry"] == "stack":
            return _dequant64(s["stack"], 0)[None]
        st = RefStack(s["codes"].view(1, c["M"], c["K"]), s["absmax"], s["codebook"])
        return _dequant64(st, 0).view(-1)
    if c["kind"] == "gemv":
        st = s.get("stack") or RefStack(s["codes"], s["absmax"], s["codebook"])
        return s["x"].double() @ _dequant64(st, 0, rounded=False).T
    T, H, I, E = c["T"], c["H"], c["I"], c["E"]
    x = s["x"].double()
    if c["entry"] in ("apply", "fused"):
        w13, a13, w2, a2, cb = s["raw"]
        st13, st2 = RefStack(w13, a13, cb), RefStack(w2, a2, cb)
        wts, ids = s["topk"]
    else:
        st13, st2 = s["moe"].w13, s["moe"].w2
        logits = s["logits"]
        if c["entry"] == "module":
            logits = torch.nn.functional.linear(s["x"], s["block"].gate)   # bf16, as the block defines it
        wts, ids = _route(c, logits.double() if c["entry"] == "logits" else logits)
        if c["entry"] == "module":
            wts = wts.to(torch.bfloat16)
    rounded = T > 1      # the reference dequantises to bf16 for two and more tokens
    out = torch.zeros((T, H), dtype=torch.float64, device=DEV)
    for e in range(E):
        tok, slot = torch.nonzero(ids == e, as_tuple=True)
        if tok.numel():
            y = _mlp64(x[tok], _dequant64(st13, e, rounded), _dequant64(st2, e, rounded))
            out.index_add_(0, tok, y * wts[tok, slot].double()[:, None])
    for e in range(E, E + c["S"]):
        out += _mlp64(x, _dequant64(st13, e, rounded), _dequant64(st2, e, rounded))
    if c["dense"]:
        d13, d2 = s["moe"].dense_shared
        out += _mlp64(x, d13.double(), d2.double()) * torch.sigmoid(x @ s["moe"].shared_gate.double())[:, None]
    return out
