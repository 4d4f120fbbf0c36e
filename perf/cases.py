"""The work a user of this framework has it do, as cases that can be timed and checked.

A case is a dict of plain values. `kind` says which entry point it goes through:

  linear      one MatMulNBits on device buffers (NBitsWeights.gemm_dev, or gemm_dev_f16 for
              fp16 activations), every weight format the operator takes
  w4a8        the same projection with the opt-in int8 activations (MODELSHARP_W4A8)
  layer       one decode step of a decoder layer, device-resident: the norm and q/k/v in one
              call, attention over the cached history, o, the norm with gate/up/SiLU in one
              call, down
  attention   GroupQueryAttention: a decode step over a cache, or a prompt over itself
  mlp         the MLP block of a decoder layer as a model graph run by the engine
              (pipeline.build and Engine.run, with the fusions pipeline.load applies)

Weights, caches and workspaces are what a serving program keeps between calls; activations
have the distributions the layers see (unit normal, or rows of unit RMS with a few outlier
channels, as behind an RMSNorm).
"""
from __future__ import annotations

import math

import torch

from modelsharp_amd import native, pipeline
from modelsharp_amd.decoder_kernels import fuse_gate_up_silu, fuse_silu_mul, fuse_skipnorm
from modelsharp_amd.graph import GraphNode, ModelGraph

EPS = 1e-6


def linear(name, M, K, N, block=32, zp="packed", bits=4, act="f32", kind="linear"):
    case = {"kind": kind, "M": M, "K": K, "N": N, "block": block, "zp": zp, "bits": bits, "act": act}
    return {"name": name, **case} if name else case


def attention(name, batch, heads, kv_heads, dim, q_seq, past):
    case = {"kind": "attention", "batch": batch, "heads": heads, "kv_heads": kv_heads, "dim": dim, "q_seq": q_seq,
            "past": past}
    return {"name": name, **case} if name else case


def listed():
    return [
        # the smallest call: one projection of a 0.5B-class model for one token
        linear("decode_small", 1, 896, 4864),
        # a 7B-class model's decode step, one layer: what a chat user waits for at every token
        {"name": "decode_layer_7b", "kind": "layer", "hidden": 3584, "inter": 18944, "heads": 28, "kv_heads": 4,
         "dim": 128, "past": 2047},
        # a few sequences decoded together, 7B-class MLP, larger blocks without zero points
        linear("small_batch", 8, 4096, 11008, block=128, zp="none"),
        # decode and prompt with fractional zero points (float zero-point exports)
        linear("float_zp_decode", 2, 4096, 11008, block=64, zp="float"),
        linear("float_zp_prefill", 512, 4096, 4096, block=64, zp="float"),
        # a short prompt through the down projection
        linear("prefill_short", 128, 11008, 4096),
        # a long prompt through the up projection
        linear("prefill_long", 2048, 4096, 11008),
        # a prompt of odd length on 8-bit weights
        linear("prefill_8bit", 500, 4096, 11008, bits=8),
        # the opt-in int8-activation product on a prompt
        linear("w4a8_prefill", 256, 4096, 11008, kind="w4a8"),
        # eight sequences decoded together over a few thousand cached tokens
        attention("attention_decode", 8, 28, 4, 128, 1, 4095),
        # a prompt of 2048 tokens over itself
        attention("attention_prefill", 1, 28, 4, 128, 2048, 0),
        # the MLP block of a 7B-class layer over a prompt, run from its graph
        {"name": "mlp_graph", "kind": "mlp", "M": 512, "hidden": 3584, "inter": 18944},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _dim(rng, lo, hi, step):
    return max(step, _log(rng, lo, hi) // step * step)


def draw(rng):
    kind = rng.choice(["linear"] * 10 + ["w4a8"] * 2 + ["layer"] * 2 + ["attention"] * 5 + ["mlp"])
    if kind in ("linear", "w4a8"):
        block = rng.choice([32, 32, 32, 128, 64, 16, 256] if kind == "linear" else [32, 32, 64, 128])
        zp = rng.choice(["packed", "packed", "none", "float"] if kind == "linear" else ["packed", "none"])
        bits = rng.choice([4, 4, 4, 8]) if kind == "linear" else 4
        # mostly whole multiples of 128, now and then a last block that is not full
        step = rng.choice([128, 128, 128, 128, 32, 8])
        K, N = _dim(rng, 512, 12288, step), _log(rng, 256, 20000)
        if rng.random() < 0.6:
            N = max(64, N // 64 * 64)
        most = 180e9 if kind == "linear" and zp != "float" and block >= 32 and K % 128 == 0 else 18e9
        M = _log(rng, 1, 2048) if rng.random() < 0.7 else rng.randint(1, 16)
        M = max(1, min(M, int(most / (2.0 * K * N))))
        act = "f16" if kind == "linear" and rng.random() < 0.2 else "f32"
        return linear(None, M, K, N, block, zp, bits, act, kind)
    if kind == "layer":
        dim, kv = rng.choice([64, 128]), rng.choice([2, 4, 8])
        heads = kv * rng.choice([1, 2, 4, 7])
        hidden = min(4096, max(512, heads * dim))
        return {"kind": "layer", "hidden": hidden, "inter": _dim(rng, 2 * hidden, 5 * hidden, 128), "heads": heads,
                "kv_heads": kv, "dim": dim, "past": _log(rng, 1, 4000)}
    if kind == "attention":
        kv = rng.choice([2, 4, 8])
        heads, dim = kv * rng.choice([1, 4, 7, 8]), rng.choice([64, 128, 128, 96, 256])
        if rng.random() < 0.5:   # decode, alone or in a batch
            past = _log(rng, 16, 8000)
            return attention(None, max(1, min(rng.choice([1, 2, 5, 8, 16]), 40000 // past)), heads, kv, dim, 1, past)
        most = 28 * 128 * 2048 * 2048   # the listed prompt's
        S = min(_log(rng, 9, 2048), int(math.sqrt(most / (heads * dim))))
        past = rng.choice([0, 0, 0, _log(rng, 1, S)])
        S = min(S, int(most / (heads * dim * (S + 2 * past)))) if past else S
        return attention(None, 1, heads, kv, dim, max(9, S), past)
    hidden = rng.choice([896, 1536, 2048, 3584])
    return {"kind": "mlp", "M": _log(rng, 1, 700), "hidden": hidden, "inter": _dim(rng, 3 * hidden, 5 * hidden, 128)}


# ---- inputs --------------------------------------------------------------------------------------

class _Weight:
    """A quantized weight as the operator takes it, on the device: codes [N, nb * blob], scales
    [N * nb], zero points packed [N, zrb], fp32 [N * nb], or None."""

    def __init__(self, gen, K, N, block, zp, bits):
        self.K, self.N, self.block, self.bits, self.kind = K, N, block, bits, zp
        self.nb = (K + block - 1) // block
        self.b = torch.randint(0, 256, (N, self.nb * block * bits // 8), dtype=torch.uint8, device="cuda", generator=gen)
        self.scales = torch.rand(N * self.nb, device="cuda", generator=gen) * 0.009 + 0.001
        if bits == 8:
            self.scales /= 16
        self.zp = None
        if zp == "packed":
            self.zp = torch.randint(0, 256, (N, (self.nb * bits + 7) // 8), dtype=torch.uint8, device="cuda",
                                    generator=gen)
        elif zp == "float":
            self.zp = (torch.rand(N * self.nb, device="cuda", generator=gen) + 0.5) * 2.0 ** (bits - 1)

    def handle(self):
        if self.kind == "float":
            return native.NBitsWeights(self.b.cpu().numpy(), self.scales.cpu().numpy(), self.zp.cpu().numpy(), self.N,
                                       self.K, self.bits, self.block)
        torch.cuda.synchronize()
        return native.NBitsWeights.from_device(self.b.data_ptr(), self.scales.data_ptr(),
                                               None if self.zp is None else self.zp.data_ptr(), self.N, self.K,
                                               self.bits, self.block)

    def bytes(self):
        return weight_bytes(self.K, self.N, self.block, self.kind, self.bits)

    def codes(self, lo, hi):
        """q - zp of rows [lo, hi) in 64 bits, [rows, nb, block]."""
        b = self.b[lo:hi]
        if self.bits == 4:
            b = torch.stack([b & 15, b >> 4], dim=-1)
        q = b.reshape(hi - lo, self.nb, self.block).double()
        if self.zp is None:
            return q - 2.0 ** (self.bits - 1)
        if self.kind == "float":
            return q - self.zp.reshape(self.N, self.nb)[lo:hi].double()[:, :, None]
        z = self.zp[lo:hi]
        if self.bits == 4:
            z = torch.stack([z & 15, z >> 4], dim=-1).reshape(hi - lo, -1)
        return q - z[:, :self.nb].double()[:, :, None]

    def product(self, a, rows=2048):
        """a [M, K] times the dequantized weights, in 64 bits."""
        out = []
        for lo in range(0, self.N, rows):
            hi = min(self.N, lo + rows)
            w = self.codes(lo, hi) * self.scales.reshape(self.N, self.nb)[lo:hi].double()[:, :, None]
            out.append(a.double() @ w.reshape(hi - lo, -1)[:, :self.K].t())
        return torch.cat(out, dim=1)


def weight_bytes(K, N, block, zp, bits):
    nb = (K + block - 1) // block
    return N * nb * (block * bits // 8 + 4) + {"packed": N * ((nb * bits + 7) // 8), "float": 4 * N * nb, "none": 0}[zp]


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(gen, *shape):
    return torch.randn(*shape, device="cuda", generator=gen)


def _rows(gen, M, K):
    """Activations: unit normal for a few tokens; for a prompt, rows of unit RMS in which one
    channel of a hundred is twenty times the others, as behind an RMSNorm."""
    a = _normal(gen, M, K)
    if M > 16:
        a[:, torch.randperm(K, device="cuda", generator=gen)[:max(1, K // 100)]] *= 20.0
        a /= a.square().mean(dim=1, keepdim=True).sqrt()
    return a


def _rotary(rows, dim):
    ang = torch.outer(torch.arange(rows, dtype=torch.float64),
                      1.0 / 10000 ** (torch.arange(dim // 2, dtype=torch.float64) / (dim // 2)))
    return torch.cos(ang).float().cuda(), torch.sin(ang).float().cuda()


def _stream():
    return torch.cuda.current_stream().cuda_stream


class _Attention:
    """GroupQueryAttention's inputs and buffers: the cache holds `past` rows, appended in place."""

    def __init__(self, gen, batch, heads, kv_heads, dim, q_seq, past, qkv=True):
        total = past + q_seq
        self.pk, self.pv = _normal(gen, batch, kv_heads, total, dim), _normal(gen, batch, kv_heads, total, dim)
        if qkv:
            self.q = _normal(gen, batch, q_seq, heads * dim)
            self.k, self.v = _normal(gen, batch, q_seq, kv_heads * dim), _normal(gen, batch, q_seq, kv_heads * dim)
        self.cos, self.sin = _rotary(total, dim)
        self.seqlens = torch.full((batch,), total - 1, dtype=torch.int32, device="cuda")
        self.out = torch.empty(batch, q_seq, heads * dim, device="cuda")
        self.desc = native.GqaDesc(batch=batch, q_seq=q_seq, kv_seq=q_seq, num_heads=heads, kv_num_heads=kv_heads,
                                   head_dim=dim, packed_qkv=0, past_seq=past, past_in_present=int(past > 0),
                                   present_capacity=total, do_rotary=1, rotary_interleaved=0, cos_rows=total,
                                   cos_cols=dim // 2, local_window_size=-1, scale=0.0, seqlens_len=batch)
        self.ws_bytes = native.gqa_workspace_size(self.desc)
        self.ws = torch.empty(max(4, self.ws_bytes), dtype=torch.uint8, device="cuda")

    def run(self, q, k, v, stream):
        native.gqa(self.desc, q.data_ptr(), k.data_ptr(), v.data_ptr(), None, None, self.seqlens.data_ptr(),
                   self.cos.data_ptr(), self.sin.data_ptr(), self.out.data_ptr(), self.pk.data_ptr(),
                   self.pv.data_ptr(), self.ws.data_ptr(), self.ws_bytes, stream)

    def product(self, q, k, v):
        """(out, present K, present V) in 64 bits."""
        d = self.desc
        B, S, H, G, D, past = d.batch, d.q_seq, d.num_heads, d.kv_num_heads, d.head_dim, d.past_seq
        cos, sin = self.cos[past:].double(), self.sin[past:].double()

        def rotate(x):   # [B, heads, S, D], half-split pairs
            a, b = x[..., :D // 2], x[..., D // 2:]
            return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1)

        q = rotate(q.double().reshape(B, S, H, D).transpose(1, 2))
        pk, pv = self.pk.double(), self.pv.double()
        pk[:, :, past:] = rotate(k.double().reshape(B, S, G, D).transpose(1, 2))
        pv[:, :, past:] = v.double().reshape(B, S, G, D).transpose(1, 2)
        keep = torch.arange(past + S, device="cuda")[None, :] <= torch.arange(past, past + S, device="cuda")[:, None]
        out = torch.empty(B, H, S, D, dtype=torch.float64, device="cuda")
        for b in range(B):
            for h in range(H):
                s = (q[b, h] @ pk[b, h // (H // G)].t().contiguous()) / math.sqrt(D)
                out[b, h] = torch.softmax(s.masked_fill(~keep, -math.inf), dim=-1) @ pv[b, h // (H // G)]
        return out.transpose(1, 2).reshape(B, S, H * D), pk, pv


def _norm64(x, skip, gamma):
    """(normed rows, x + skip) in 64 bits."""
    t = x.double() + skip.double()
    return t / torch.sqrt(t.square().mean(dim=-1, keepdim=True) + EPS) * gamma.double(), t


def _silu64(g, u):
    return g / (1.0 + torch.exp(-g)) * u


def _inputs(case, seed):
    """The tensors of a case from the seed alone."""
    gen = _generator(seed)
    kind = case["kind"]
    if kind in ("linear", "w4a8"):
        w = _Weight(gen, case["K"], case["N"], case["block"], case["zp"], case["bits"])
        a = _rows(gen, case["M"], case["K"])
        return {"w": w, "a": a.half() if case["act"] == "f16" else a}
    if kind == "attention":
        return {"att": _Attention(gen, case["batch"], case["heads"], case["kv_heads"], case["dim"], case["q_seq"],
                                  case["past"])}
    E, I = case["hidden"], case["inter"]
    s = {"w": {"gate": _Weight(gen, E, I, 32, "packed", 4), "up": _Weight(gen, E, I, 32, "packed", 4),
               "down": _Weight(gen, I, E, 32, "packed", 4)}}
    M = case.get("M", 1)
    s["x"], s["skip"] = _normal(gen, M, E), _normal(gen, M, E)
    s["gamma"] = torch.rand(E, device="cuda", generator=gen) + 0.5
    if kind == "layer":
        Q, KV = case["heads"] * case["dim"], case["kv_heads"] * case["dim"]
        for name, K, N in (("q", E, Q), ("k", E, KV), ("v", E, KV), ("o", Q, E)):
            s["w"][name] = _Weight(gen, K, N, 32, "packed", 4)
        s["gamma2"] = torch.rand(E, device="cuda", generator=gen) + 0.5
        s["att"] = _Attention(gen, 1, case["heads"], case["kv_heads"], case["dim"], 1, case["past"], qkv=False)
    return s


def _mlp_graph(s):
    """The MLP block as an exporter writes it: SkipSimplifiedLayerNormalization, the gate and up
    projections, Sigmoid-Mul-Mul, down."""
    init = {"gamma": s["gamma"].cpu().numpy()}
    for n, w in s["w"].items():
        init.update({n + ".b": w.b.cpu().numpy().reshape(w.N, w.nb, -1), n + ".s": w.scales.cpu().numpy(),
                     n + ".z": w.zp.cpu().numpy()})

    def mm(n, x, y):
        w = s["w"][n]
        return GraphNode("MatMulNBits", n, [x, n + ".b", n + ".s", n + ".z"], [y],
                         {"K": w.K, "N": w.N, "bits": w.bits, "block_size": w.block})

    nodes = [GraphNode("SkipSimplifiedLayerNormalization", "norm", ["x", "skip", "gamma"], ["n", "", "", "t"],
                       {"epsilon": EPS}),
             mm("gate", "n", "g"), mm("up", "n", "u"), GraphNode("Sigmoid", "sig", ["g"], ["s"]),
             GraphNode("Mul", "mul1", ["g", "s"], ["a"]), GraphNode("Mul", "mul2", ["a", "u"], ["h"]),
             mm("down", "h", "y")]
    return ModelGraph(nodes, init, ["x", "skip"], ["y", "t"])


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    kind = case["kind"]
    if kind in ("linear", "w4a8"):
        s["h"] = s["w"].handle()
        s["y"] = torch.empty(case["M"], case["N"], device="cuda")
    elif kind == "layer":
        s["h"] = {n: w.handle() for n, w in s["w"].items()}
        e = lambda n: torch.empty(1, n, device="cuda")   # noqa: E731
        E, I, Q, KV = case["hidden"], case["inter"], case["heads"] * case["dim"], case["kv_heads"] * case["dim"]
        s.update(n1=e(E), t1=e(E), q=e(Q), k=e(KV), v=e(KV), o=e(E), n2=e(E), t2=e(E), act=e(I), y=e(E))
    elif kind == "mlp":
        graph = _mlp_graph(s)
        fuse_silu_mul(graph)
        fuse_gate_up_silu(graph)
        fuse_skipnorm(graph)
        s["engine"] = pipeline.build(graph)
    if kind != "attention":
        del s["w"]   # the handles and the engine hold their own copy
    torch.cuda.synchronize()
    return s


# ---- one pass ------------------------------------------------------------------------------------

def run(s):
    case = s["case"]
    kind = case["kind"]
    st = _stream()
    if kind == "linear":
        call = s["h"].gemm_dev_f16 if case["act"] == "f16" else s["h"].gemm_dev
        call(s["a"].data_ptr(), s["y"].data_ptr(), case["M"], st)
        return s["y"]
    if kind == "w4a8":
        s["h"].gemm_dev_w4a8(s["a"].data_ptr(), s["y"].data_ptr(), case["M"], st)
        return s["y"]
    if kind == "attention":
        att = s["att"]
        att.run(att.q, att.k, att.v, st)
        return {"out": att.out, "present_k": att.pk, "present_v": att.pv}
    if kind == "mlp":
        return s["engine"].run({"x": s["x"], "skip": s["skip"]})
    h, att = s["h"], s["att"]
    native.gemm_dev_skipnorm([h["q"], h["k"], h["v"]], s["x"].data_ptr(), s["skip"].data_ptr(), s["gamma"].data_ptr(),
                             EPS, s["n1"].data_ptr(), s["t1"].data_ptr(),
                             [s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr()], 1, st)
    att.run(s["q"], s["k"], s["v"], st)
    h["o"].gemm_dev(att.out.data_ptr(), s["o"].data_ptr(), 1, st)
    native.gemm_dev_skipnorm_swiglu(h["gate"], h["up"], s["o"].data_ptr(), s["t1"].data_ptr(), s["gamma2"].data_ptr(),
                                    EPS, s["n2"].data_ptr(), s["t2"].data_ptr(), s["act"].data_ptr(), 1, st)
    h["down"].gemm_dev(s["act"].data_ptr(), s["y"].data_ptr(), 1, st)
    return {"y": s["y"], "residual": s["t2"], "present_k": att.pk, "present_v": att.pv}


# ---- what a pass cannot do without ---------------------------------------------------------------

def _attention_work(case):
    B, H, G, D, S, past = (case[k] for k in ("batch", "heads", "kv_heads", "dim", "q_seq", "past"))
    pairs = S * past + S * (S + 1) // 2
    return {"bytes": 4 * B * (2 * S * H * D + 4 * S * G * D + 2 * past * G * D), "flops": 4 * B * H * D * pairs}


def work(case):
    kind = case["kind"]
    if kind in ("linear", "w4a8"):
        M, K, N = case["M"], case["K"], case["N"]
        return {"bytes": weight_bytes(K, N, case["block"], case["zp"], case["bits"])
                + M * K * (2 if case["act"] == "f16" else 4) + 4 * M * N, "flops": 2 * M * K * N}
    if kind == "attention":
        return _attention_work(case)
    E, I, M = case["hidden"], case["inter"], case.get("M", 1)
    shapes = [(E, I), (E, I), (I, E)]
    w = {"bytes": 4 * M * E * 4, "flops": 0}   # x, skip, the sum, y
    if kind == "layer":
        Q, KV = case["heads"] * case["dim"], case["kv_heads"] * case["dim"]
        shapes += [(E, Q), (E, KV), (E, KV), (Q, E)]
        a = _attention_work({**case, "batch": 1, "q_seq": 1})
        w = {"bytes": w["bytes"] + a["bytes"] - 4 * (2 * Q + 2 * KV), "flops": a["flops"]}
    for K, N in shapes:
        w["bytes"] += weight_bytes(K, N, 32, "packed", 4)
        w["flops"] += 2 * M * K * N
    return w


# ---- how far another correct implementation may be off -------------------------------------------

def tolerance(case):
    kind = case["kind"]
    if kind == "w4a8":
        return "exact"   # integer block dots and fp32 block terms added in block order: every bit is defined
    # fp32 throughout: about four times the distance from exact() that the largest sizes show
    if kind in ("attention", "layer") or (kind == "mlp" and case["M"] <= 16):
        return {"rel": 2e-6}
    # fp16 operands with fp32 sums, once (3.6e-4 from exact()) or through two layers (6.3e-4)
    if kind == "mlp":
        return {"rel": 2.5e-3}
    if case["M"] > 16 and case["zp"] != "float":
        return {"rel": 1.5e-3}
    return {"rel": 2e-6} if case["M"] <= 16 else {"rel": 4e-6}


def exact(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind == "linear":
        return s["w"].product(s["a"])
    if kind == "w4a8":
        return _w4a8_64(s["a"], s["w"])
    if kind == "attention":
        att = s["att"]
        out, pk, pv = att.product(att.q, att.k, att.v)
        return {"out": out, "present_k": pk, "present_v": pv}
    w = s["w"]
    if kind == "mlp":
        n, t = _norm64(s["x"], s["skip"], s["gamma"])
        return {"y": w["down"].product(_silu64(w["gate"].product(n), w["up"].product(n))), "t": t}
    n, t1 = _norm64(s["x"], s["skip"], s["gamma"])
    out, pk, pv = s["att"].product(*(w[i].product(n) for i in ("q", "k", "v")))
    n, t2 = _norm64(w["o"].product(out.reshape(1, -1)), t1, s["gamma2"])
    y = w["down"].product(_silu64(w["gate"].product(n), w["up"].product(n)))
    return {"y": y, "residual": t2, "present_k": pk, "present_v": pv}


def _w4a8_64(a, w):
    """Activations quantized per (row, block) in fp32 as the operator defines it (scale
    max|a| / 127, codes rint(a / scale)), the rest in 64 bits."""
    pad = torch.zeros(a.shape[0], w.nb * w.block, device="cuda")
    pad[:, :w.K] = a
    blocks = pad.reshape(a.shape[0], w.nb, w.block)
    sa = blocks.abs().amax(dim=2) / 127.0
    inv = torch.where(sa > 0, 1.0 / sa, torch.zeros_like(sa))
    q = torch.clamp(torch.round(blocks * inv[:, :, None]), -127, 127)
    a64 = (q.double() * sa.double()[:, :, None]).reshape(a.shape[0], -1)
    out = []
    for lo in range(0, w.N, 2048):
        hi = min(w.N, lo + 2048)
        c = w.codes(lo, hi).clamp(-127, 127)
        c = c * w.scales.reshape(w.N, w.nb)[lo:hi].double()[:, :, None]
        out.append(a64 @ c.reshape(hi - lo, -1).t())
    return torch.cat(out, dim=1)
