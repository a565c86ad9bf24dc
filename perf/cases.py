"""What a user of this framework has it do: MoE expert-FFN layers through the package's entry
points, one token at a time (decode) and many (batched, prefill).

Layer shapes are the configured workloads' (moe_rocm/workloads.py: gpt_oss, qwen3_30b, coder_next)
and, in draw(), generic ones around them. The weights are random blocks in the native GGUF layouts
with the magnitudes of trained weights (rms 0.02 .. 0.05), activations N(0, 1).
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "moe-stream_amd"))
import moe_rocm as M  # noqa: E402

EPS = 1e-5
DEVICE = "cuda"

# Layer shapes: GPT-OSS is MXFP4 with biases, softmax after top-k and the clamped SwiGLU; the
# other two are Q4_K with renormalised top-k and SiLU, coder_next with a shared expert.
GPT_OSS = {"type": "mxfp4", "hidden": 2880, "inter": 2880, "experts": 32, "top_k": 4, "shared": 0}
QWEN3 = {"type": "q4_k", "hidden": 2048, "inter": 768, "experts": 128, "top_k": 8, "shared": 0}
CODER = {"type": "q4_k", "hidden": 2048, "inter": 512, "experts": 512, "top_k": 10, "shared": 512}


def listed():
    def case(name, shape, call, layers=1, tokens=1, skew=0.0, **kw):
        return dict(shape, name=name, call=call, layers=layers, tokens=tokens, skew=skew, **kw)

    return [
        # the smallest call: one layer, one token, launched eagerly
        case("layer_qwen3_t1", QWEN3, "forward"),
        # batch-1 decode of a whole stack, one graph per token, as the benchmark and an engine run it
        case("decode_gpt_oss", GPT_OSS, "forward_graph", layers=24),
        # the same with the post-attention norm and the residual fused in (the engine's layer)
        case("decode_qwen3_residual", QWEN3, "residual_graph", layers=48),
        # pruned stack: 256 .. 512 experts by layer, and a shared expert
        case("decode_coder_next", CODER, "forward_graph", layers=12, experts_least=256),
        # a handful of sequences decoded together
        case("batch_gpt_oss_t4", GPT_OSS, "batched_residual", tokens=4),
        case("batch_qwen3_t16", QWEN3, "batched", tokens=16),
        # experts only: the caller routed by itself
        case("experts_gpt_oss_t8", GPT_OSS, "experts", tokens=8),
        # prompts: a batch with skewed routing, ragged lengths, a long one
        case("prefill_gpt_oss_512_skewed", GPT_OSS, "batched", tokens=512, skew=1.1),
        case("prefill_gpt_oss_2039", GPT_OSS, "batched_residual", tokens=2039),
        case("prefill_qwen3_511", QWEN3, "batched_residual", tokens=511),
        case("prefill_coder_next_384", CODER, "batched", tokens=384),
        case("prefill_qwen3_4096", QWEN3, "batched", tokens=4096),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: another call, token count and skew on one of the shapes, or on a generic shape
    around them (other widths, expert counts, top-k, shared experts of both types)."""
    call = rng.choice(["forward", "forward_graph", "residual_graph", "batched", "batched", "batched_residual",
                       "batched_residual", "noalloc", "experts"])
    if rng.random() < 0.5:
        shape = dict(rng.choice([GPT_OSS, QWEN3, CODER]))
        if shape["type"] == "q4_k" and shape["shared"]:
            shape["experts"] = rng.randint(256, 512)
    elif rng.random() < 0.5:
        inter = 32 * rng.randint(16, 92)
        shape = {"type": "mxfp4", "hidden": 32 * rng.randint(32, 92), "inter": inter,
                 "experts": rng.randint(8, 64), "top_k": rng.randint(1, 6), "shared": rng.choice([0, 0, 0, inter])}
    else:
        inter = 256 * rng.randint(1, 4)
        shape = {"type": "q4_k", "hidden": 256 * rng.randint(4, 12), "inter": inter,
                 "experts": rng.randint(16, 256), "top_k": rng.randint(2, 10), "shared": rng.choice([0, 0, inter])}
    decode = call in ("forward", "forward_graph", "residual_graph")
    layers, tokens = 1, 1
    if call == "noalloc":  # as many tokens as its fixed scratch holds at every shape here
        tokens = _log_int(rng, 1, 200)
    elif call == "experts":
        tokens = _log_int(rng, 1, 16)
    elif not decode:
        tokens = _log_int(rng, 2, 3000 if shape["type"] == "q4_k" else 2000)
    elif call != "forward":
        layers = rng.randint(2, 12)
    skew = 0.0 if decode else rng.choice([0.0, round(rng.uniform(0.6, 1.3), 2)])
    return dict(shape, call=call, layers=layers, tokens=tokens, skew=skew)


def _layer_experts(case, li):
    """Experts of layer li: all, or spread between experts_least and experts (a pruned stack)."""
    lo, hi = case.get("experts_least", case["experts"]), case["experts"]
    return lo + (hi - lo) * ((7 * li + 3) % case["layers"]) // max(1, case["layers"] - 1)


def _seed(seed, *ids):
    for i in ids:
        seed = (seed * 1000003 + i + 1) % (1 << 62)
    return seed


def _gen(seed, *ids):
    return torch.Generator(device=DEVICE).manual_seed(_seed(seed, *ids))


def _blocks(gtype, rows, cols, gen, n_mat):
    """Random blocks [n_mat, rows, blocks, block bytes] and 64 readable bytes after them."""
    size, elems = (17, 32) if gtype == "mxfp4" else (144, 256)
    n = n_mat * rows * (cols // elems)
    words = torch.randint(-(1 << 63), (1 << 63) - 1, ((n * size + 64 + 7) // 8,), generator=gen, device=DEVICE)
    flat = words.view(torch.uint8)
    b = flat[: n * size].view(n, size)
    if gtype == "mxfp4":  # block scales 2^-9 .. 2^-4
        b[:, 0] = 118 + b[:, 0] % 6
    else:  # d about 1e-4, dmin 7.5 d: the quants' mean is about taken out
        d = 6e-5 + 1.2e-4 * torch.rand(n, generator=gen, device=DEVICE)
        b[:, :4] = torch.stack([d, 7.5 * d], 1).to(torch.float16).view(torch.uint8)
    return flat, b.view(n_mat, rows, cols // elems, size)


def _normal(gen, shape, std=1.0):
    return std * torch.randn(shape, generator=gen, device=DEVICE)


def _tensors(case, seed, li):
    """One layer's weights and its input rows [tokens, hidden], from the seed alone."""
    H, I, Ish, T, E = case["hidden"], case["inter"], case["shared"], case["tokens"], _layer_experts(case, li)
    g, t = _gen(seed, li), {}
    for name, rows, cols, n in (("gate", I, H, E), ("up", I, H, E), ("down", H, I, E), ("sh_gate", Ish, H, 1),
                                ("sh_up", Ish, H, 1), ("sh_down", H, Ish, 1)):
        if rows and cols:
            t[name + "_bytes"], t[name] = _blocks(case["type"], rows, cols, g, n)
    t["router_w"] = _normal(g, (E, H), 0.02)
    if case["type"] == "mxfp4":
        t["gate_b"], t["up_b"], t["down_b"] = (_normal(g, (E, n), 0.1) for n in (I, I, H))
    if case["type"] == "mxfp4" or case["skew"]:
        t["router_b"] = _normal(g, (E,), 0.01)
        if case["skew"]:  # expert popularity ~ rank^-skew over a random ranking
            rank = 1.0 + torch.randperm(E, generator=g, device=DEVICE)
            t["router_b"] = t["router_b"] - case["skew"] * torch.log(rank)
    if Ish:
        t["sh_gate_inp"] = _normal(g, (H,), 0.02)
    t["x"] = _normal(g, (T, H))
    t["norm_w"] = 1.0 + _normal(g, (H,), 0.1)
    return t


_ctx = None


def _context():
    """The program's one context."""
    global _ctx
    if _ctx is None:
        _ctx = M.Context(0)
    return _ctx


class _Layer:
    """One layer's handles; the tensors stay alive with it."""

    def __init__(self, case, t):
        ctx, self.t, self.packs = _context(), t, {}
        gtype = M.GGML_MXFP4 if case["type"] == "mxfp4" else M.GGML_Q4_K
        H, I, Ish, E = case["hidden"], case["inter"], case["shared"], t["gate"].shape[0]
        for name, rows, cols, n in (("gate", I, H, E), ("up", I, H, E), ("down", H, I, E), ("sh_gate", Ish, H, 1),
                                    ("sh_up", Ish, H, 1), ("sh_down", H, Ish, 1)):
            if name in t:
                self.packs[name] = M.ExpertPack.wrap(ctx, gtype, t[name + "_bytes"].data_ptr(), t[name].numel(), n,
                                                     rows, cols)
        floats = {k: t[v].data_ptr() for k, v in (("router_b", "router_b"), ("gate_bias", "gate_b"), ("up_bias", "up_b"),
                                                  ("down_bias", "down_b"), ("sh_gate_inp", "sh_gate_inp")) if v in t}
        mx = case["type"] == "mxfp4"
        self.layer = M.MoeLayer(ctx, self.packs["gate"], self.packs["up"], self.packs["down"],
                                router_w=t["router_w"].data_ptr(), top_k=case["top_k"],
                                route_flags=M.ROUTE_SOFTMAX_AFTER_TOPK if mx else M.ROUTE_NORM_TOPK,
                                act=M.ACT_SWIGLU_OAI if mx else M.ACT_SILU,
                                **{k: self.packs[k] for k in ("sh_gate", "sh_up", "sh_down") if k in self.packs}, **floats)

    def close(self):
        self.layer.close()
        for p in self.packs.values():
            p.close()


class _State:
    def __init__(self, case, seed):
        self.call, self.tokens = case["call"], case["tokens"]
        ts = [_tensors(case, seed, li) for li in range(case["layers"])]
        self.layers = [_Layer(case, t) for t in ts]
        self.x = torch.stack([t["x"] for t in ts])  # [layers, tokens, hidden]
        self.y = torch.zeros_like(self.x)
        self.graph = None
        if self.call == "experts":
            self.idx, self.w = _route(case, ts[0], self.x[0].double())
            self.idx, self.w = self.idx.to(torch.int32).contiguous(), self.w.float().contiguous()
        torch.cuda.synchronize()
        for a in self.layers:
            a.layer.reserve(self.tokens)
        if self.call.endswith("_graph"):
            n = len(self.layers)
            for li, a in enumerate(self.layers):  # each layer reads the next one's router rows ahead
                a.layer.set_next(self.layers[(li + 1) % n].layer)
                if self.call == "residual_graph":
                    a.layer.set_norm(a.t["norm_w"].data_ptr())
            ctx = _context()
            ctx.graph_begin()
            for li, a in enumerate(self.layers):
                x, y = self.x[li].data_ptr(), self.y[li].data_ptr()
                if self.call == "residual_graph":
                    a.layer.forward_residual(x, a.t["norm_w"].data_ptr(), EPS, y)
                else:
                    a.layer.forward(x, y)
            self.graph = ctx.graph_end()

    def __del__(self):
        try:
            if self.graph is not None:
                self.graph.close()
            for a in self.layers:
                a.close()
        except (AttributeError, TypeError):  # half-made, or at the interpreter's end
            pass


def prepare(case, seed):
    return _State(case, seed)


def run(s):
    a = s.layers[0]
    x, y, T = s.x.data_ptr(), s.y.data_ptr(), s.tokens
    if s.graph is not None:
        s.graph.launch()
    elif s.call == "forward":
        a.layer.forward(x, y)
    elif s.call == "batched":
        a.layer.forward_batched(x, T, y)
    elif s.call == "noalloc":
        a.layer.forward_batched_noalloc(x, T, y)
    elif s.call == "batched_residual":
        a.layer.forward_batched_residual(x, T, a.t["norm_w"].data_ptr(), EPS, y)
    else:
        a.layer.experts(x, T, s.idx.data_ptr(), s.w.data_ptr(), y)
    return s.y


def _matrix_bytes(case, rows, cols):
    return rows * (cols // 32) * 17 if case["type"] == "mxfp4" else rows * (cols // 256) * 144


def work(case):
    """The experts that the tokens select (their expected number) and the router read once, each
    token's input read and its output written once; two operations per weight used."""
    H, I, Ish, T, k = case["hidden"], case["inter"], case["shared"], case["tokens"], case["top_k"]
    nbytes = flops = 0.0
    for li in range(case["layers"]):
        E = _layer_experts(case, li)
        p = (1.0 + np.arange(E)) ** -case["skew"]
        p = np.minimum(1.0, k * p / p.sum())
        used = float((1.0 - (1.0 - p) ** T).sum()) if T > 1 else float(k)
        expert = 2 * _matrix_bytes(case, I, H) + _matrix_bytes(case, H, I)
        nbytes += used * (expert + (4 * (2 * I + H) if case["type"] == "mxfp4" else 0)) + 8.0 * T * H
        flops += 6.0 * T * k * H * I + 6.0 * T * H * Ish
        if Ish:
            nbytes += 2 * _matrix_bytes(case, Ish, H) + _matrix_bytes(case, H, Ish)
        if case["call"] != "experts":
            nbytes += 4.0 * E * H
            flops += 2.0 * T * E * H
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times the error against 64 bits: the MFMA kernels take the f32 activations apart
    into short terms (three or four 8-bit floats per 32 elements, two 8-bit integers per 16 or 256)
    and sum in f32; experts() multiplies and sums in f32."""
    if case["call"] == "experts":
        return {"rel": 2e-6}
    return {"rel": 2.5e-4 if case["type"] == "mxfp4" else 1e-3}


# ---- the same in 64 bits, plain torch ----------------------------------------------------------
def _dequant(case, b):
    """[rows, blocks, block bytes] -> [rows, cols] float64."""
    rows = b.shape[0]
    if case["type"] == "mxfp4":
        kv = torch.tensor([0, .5, 1, 1.5, 2, 3, 4, 6, 0, -.5, -1, -1.5, -2, -3, -4, -6], dtype=torch.float64, device=DEVICE)
        q = b[..., 1:]
        v = torch.cat([kv[(q & 15).long()], kv[(q >> 4).long()]], -1)
        return (v * torch.exp2(b[..., :1].double() - 127.0)).reshape(rows, -1)
    dd = b[..., :4].contiguous().view(torch.float16).double()
    s = b[..., 4:16].int()
    lo, hi, top = s[..., 0:4], s[..., 4:8], s[..., 8:12]
    sc = torch.cat([lo & 63, (top & 15) | ((lo >> 6) << 4)], -1).double()
    mn = torch.cat([hi & 63, (top >> 4) | ((hi >> 6) << 4)], -1).double()
    q = b[..., 16:].reshape(rows, -1, 4, 1, 32)
    q = torch.cat([q & 15, q >> 4], -2).reshape(rows, -1, 8, 32).double()
    return ((dd[..., :1] * sc)[..., None] * q - (dd[..., 1:] * mn)[..., None]).reshape(rows, -1)


def _route(case, t, x):
    logits = x @ t["router_w"].double().T
    if "router_b" in t:
        logits = logits + t["router_b"].double()
    top, idx = torch.topk(logits, case["top_k"], dim=1)
    return idx, torch.softmax(top, dim=1)  # renormalised top-k is the same softmax


def _ffn(case, x, gate, up, down, bias, clamped):
    g, u = x @ _dequant(case, gate).T, x @ _dequant(case, up).T
    if bias:
        g, u = g + bias[0].double(), u + bias[1].double()
    if clamped:
        g, u = g.clamp(max=7.0), u.clamp(-7.0, 7.0) + 1.0
    o = (g * torch.sigmoid((1.702 if clamped else 1.0) * g) * u) @ _dequant(case, down).T
    return o + bias[2].double() if bias else o


def exact(case, seed):
    ys = []
    for li in range(case["layers"]):
        t = _tensors(case, seed, li)
        h = t["x"].double()
        residual = case["call"] in ("residual_graph", "batched_residual")
        x = h * torch.rsqrt(h.square().mean(1, keepdim=True) + EPS) * t["norm_w"].double() if residual else h
        idx, w = _route(case, t, x)
        y = torch.zeros_like(x)
        mx = case["type"] == "mxfp4"
        for e in torch.unique(idx).tolist():
            tok, slot = torch.nonzero(idx == e, as_tuple=True)
            bias = [t[b][e] for b in ("gate_b", "up_b", "down_b")] if mx else None
            y[tok] += w[tok, slot, None] * _ffn(case, x[tok], t["gate"][e], t["up"][e], t["down"][e], bias, mx)
        if case["shared"]:
            gate = torch.sigmoid(x @ t["sh_gate_inp"].double())[:, None]
            y += gate * _ffn(case, x, t["sh_gate"][0], t["sh_up"][0], t["sh_down"][0], None, False)
        ys.append(h + y if residual else y)
    return torch.stack(ys)
