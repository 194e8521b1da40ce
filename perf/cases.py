"""Performance cases of the forward, decode and training paths.

Each case is one call (or one short loop of calls) that a program using this
library makes through its public entry points: the C ABI of
include/hip_bridge.h over rustane_amd.hip_bridge, or rustane_amd.engine. The
shapes are the presets of rustane_amd.engine.ModelConfig (7B, 5B, 600M, 48M)
and one generic grouped-query shape; single-layer cases use one layer of such
a model. Weights are the library's seeded N(0, 0.02) values, which a program
writes with Model.init_synthetic; `exact` recomputes them from their published
definition (csrc/synth.hpp) and the whole path in 64-bit torch.
"""
import math

import numpy as np
import torch

from rustane_amd import engine as E
from rustane_amd import hip_bridge as hb

STD = 0.02
LOSS_SCALE = 256.0

# name: dim, hidden, heads, kv_heads, hd, layers of the whole model
SHAPES = {
    "7b": (4096, 11008, 32, 32, 128, 32),
    "5b": (2560, 6912, 20, 20, 128, 60),
    "600m": (1536, 4096, 12, 12, 128, 20),
    "48m": (512, 1536, 8, 8, 64, 8),
    "gqa": (2048, 5632, 32, 8, 64, 24),
}
VOCAB = 32000


def listed():
    return [
        # the input norm of one ragged prompt: the smallest call of the layer split
        {"name": "norm_prompt", "kind": "norm", "dim": 2560, "T": 333},
        # attention block (QKV + RoPE + causal attention) of one layer: one
        # 512-token sequence, the benchmark's prefill
        {"name": "attn_b1", "kind": "attn", "shape": "7b", "B": 1, "S": 512},
        # the same for two long prompts
        {"name": "attn_long", "kind": "attn", "shape": "7b", "B": 2, "S": 2048},
        # grouped-query heads of 64 features, three prompts of a ragged length
        {"name": "attn_gqa", "kind": "attn", "shape": "gqa", "B": 3, "S": 777},
        # FFN block of one layer: a short chat turn, one sequence, a full batch
        {"name": "ffn_chat", "kind": "ffn", "shape": "7b", "T": 45},
        {"name": "ffn_b1", "kind": "ffn", "shape": "7b", "T": 512},
        {"name": "ffn_b8", "kind": "ffn", "shape": "7b", "T": 4096},
        # whole forward with logits and losses: the headline prefill workload
        {"name": "forward_7b", "kind": "forward", "shape": "7b", "layers": 32, "B": 1, "S": 512},
        # a chat completion on one sequence: prompt, then token by token
        {"name": "decode_b1", "kind": "decode", "shape": "600m", "layers": 20, "B": 1, "S": 1000, "steps": 32},
        # sixteen sequences served together, four layers of the large shape
        {"name": "decode_b16", "kind": "decode", "shape": "7b", "layers": 4, "B": 16, "S": 200, "steps": 32},
        # one micro-batch of a data-parallel training rank (forward + backward
        # into the gradient arena that the all-reduce then reads): four
        # sequences of 512 on two layers of the large shape, ...
        {"name": "train_b4", "kind": "train", "shape": "7b", "layers": 2, "B": 4, "S": 512},
        # ... and one long sequence
        {"name": "train_long", "kind": "train", "shape": "5b", "layers": 2, "B": 1, "S": 2048},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choice(["norm", "attn", "attn", "ffn", "ffn", "wo", "head", "forward", "decode", "train", "train"])
    shape = rng.choice(list(SHAPES))
    if kind == "norm":
        return {"kind": kind, "dim": 64 * _log(rng, 4, 128), "T": _log(rng, 1, 4096)}
    if kind == "attn":
        S = _log(rng, 1, 2048)
        return {"kind": kind, "shape": shape, "B": _log(rng, 1, max(1, min(16, 4096 // S))), "S": S}
    if kind in ("ffn", "wo"):
        return {"kind": kind, "shape": shape, "T": _log(rng, 1, 4096)}
    if kind == "head":
        return {"kind": kind, "shape": shape, "T": _log(rng, 1, 1024)}
    small = rng.choice(["48m", "600m", "gqa"])
    if kind == "forward":
        S = _log(rng, 8, 512)
        return {"kind": kind, "shape": small, "layers": rng.choice([4, SHAPES[small][5]]),
                "B": _log(rng, 1, max(1, min(8, 2048 // S))), "S": S}
    if kind == "decode":
        return {"kind": kind, "shape": small, "layers": rng.choice([4, 8]), "B": _log(rng, 1, 16),
                "S": _log(rng, 1, 256), "steps": rng.randint(8, 32)}
    S = _log(rng, 32, 1024)
    return {"kind": "train", "shape": rng.choice(["48m", "600m", "gqa", "5b"]), "layers": 2,
            "B": _log(rng, 1, max(1, min(8, 2048 // S))), "S": S}


# ---------------------------------------------------------------------------
# what a program holds before the call
# ---------------------------------------------------------------------------
def _config(case, layers, seq, vocab):
    dim, hidden, heads, kv_heads, hd, full = SHAPES[case["shape"]]
    # a slice of a model keeps the whole model's residual scale
    return E.ModelConfig.make(dim, hidden, heads, layers, seq, vocab, hd=hd, kv_heads=kv_heads,
                              residual_alpha=float(np.float32(1.0 / math.sqrt(2.0 * full))))


def _randn(seed, shape, dtype, scale=1.0):
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    return (torch.randn(shape, generator=g, device="cuda") * scale).to(dtype)


def _tokens(seed, n, salt=0):
    return np.random.RandomState((int(seed) * 7919 + salt) % (1 << 32)).randint(0, VOCAB, n).astype(np.uint32)


def _device_ids(ids):
    return torch.from_numpy(ids.view(np.int32).copy()).cuda()


class _Floats:
    """n floats of device memory at an address, for torch.as_tensor, whose
    tensor keeps this object and so the memory's owner alive."""

    def __init__(self, address, n, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "<f4", "data": (address, False), "version": 2}


def _packed_views(flat, cfg):
    """The gradient arena's tensors in its packed order (output-major rows,
    W1 and W3 interleaved in pairs of rows)."""
    d, h, q, kv = cfg.dim, cfg.hidden, cfg.q_dim, cfg.kv_dim
    out, at = {}, 0
    for l in range(cfg.nlayers):
        for name, shape in (("wqkv", (q + 2 * kv, d)), ("wo", (d, q)), ("w13", (2 * h, d)), ("w2", (d, h)),
                            ("g1", (d,)), ("g2", (d,))):
            n = math.prod(shape)
            out["l%d.%s" % (l, name)] = flat[at:at + n].view(shape)
            at += n
    out["embed"] = flat[at:at + cfg.vocab * d].view(cfg.vocab, d)
    at += cfg.vocab * d
    out["gamma"] = flat[at:at + d]
    return out


def _layer_inputs(case, seed):
    """Device inputs of a single-layer case: normalised rows are N(0, 1) as a
    norm leaves them, residual rows carry the stream of a deep layer."""
    dim, hidden, heads, kv_heads, hd, _ = SHAPES[case["shape"]]
    kind = case["kind"]
    if kind == "attn":
        return {"xn": _randn(seed, (case["B"] * case["S"], dim), torch.float16)}
    if kind == "ffn":
        return {"xn": _randn(seed, (case["T"], dim), torch.float16),
                "x": _randn(seed + 1, (case["T"], dim), torch.float32)}
    if kind == "wo":
        return {"attn": _randn(seed, (case["T"], heads * hd), torch.float16, 0.5),
                "x": _randn(seed + 1, (case["T"], dim), torch.float32)}
    return {"xn": _randn(seed, (case["T"], dim), torch.float16)}  # head


def prepare(case, seed):
    kind = case["kind"]
    if kind == "norm":
        T, d = case["T"], case["dim"]
        return {"case": case, "ctx": hb.Context(0),
                "x": _randn(seed, (T, d), torch.float32), "gamma": 1 + _randn(seed + 1, (d,), torch.float32, 0.1),
                "out": torch.empty((T, d), dtype=torch.float16, device="cuda"),
                "rinv": torch.empty(T, device="cuda")}
    if kind in ("attn", "ffn", "wo", "head"):
        vocab = VOCAB if kind == "head" else 64
        cfg = _config(case, 1, case.get("S", 64), vocab)
        k = E.CompiledKernels.compile(cfg)
        k.init_synthetic(seed, STD)
        st = {"case": case, "k": k, **_layer_inputs(case, seed)}
        T = case.get("T") or case["B"] * case["S"]
        if kind == "attn":
            st["out"] = torch.empty((T, cfg.q_dim), dtype=torch.float16, device="cuda")
        elif kind == "head":
            st["targets"] = _device_ids(_tokens(seed, T))
            st["logits"] = torch.empty((T, vocab), device="cuda")
            st["losses"] = torch.empty(T, device="cuda")
        else:
            st["out"] = torch.empty((T, cfg.dim), device="cuda")
        return st
    B, S = case["B"], case["S"]
    steps = case.get("steps", 0)
    cfg = _config(case, case["layers"], S + steps, VOCAB)
    k = E.CompiledKernels.compile(cfg)
    k.init_synthetic(seed, STD)
    st = {"case": case, "k": k}
    if kind == "decode":
        st["dec"] = E.Decoder(k, B, S + steps)
        st["prompt"] = _tokens(seed, B * S)
        st["next"] = _tokens(seed, steps * B, 1).reshape(steps, B)
        return st
    st["tok"], st["tgt"] = _device_ids(_tokens(seed, B * S)), _device_ids(_tokens(seed, B * S, 1))
    st["losses"], st["mean"] = torch.empty(B * S, device="cuda"), torch.empty(1, device="cuda")
    if kind == "forward":
        st["logits"] = torch.empty((B * S, VOCAB), device="cuda")
    else:
        st["opt"] = hb.Optimizer(k.model, E.TrainConfig())
        address, n = st["opt"].grad_arena()
        st["grads"] = _packed_views(torch.as_tensor(_Floats(address, n, st["opt"]), device="cuda"), cfg)
    return st


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind = case["kind"]
    p = hb.ptr
    if kind == "norm":
        hb.call("hb_op_rmsnorm", state["ctx"].handle, p(state["x"]), p(state["gamma"]), case["T"], case["dim"],
                1e-5, p(state["out"]), p(state["rinv"]))
        return {"out": state["out"], "rms_inv": state["rinv"]}
    m = state["k"].model.handle
    if kind == "attn":
        hb.call("hb_op_sdpa_fwd", m, 0, p(state["xn"]), case["B"], case["S"], p(state["out"]), None)
        return state["out"]
    if kind == "ffn":
        hb.call("hb_op_ffn_fused", m, 0, p(state["xn"]), p(state["x"]), case["T"], p(state["out"]), None, None)
        return state["out"]
    if kind == "wo":
        hb.call("hb_op_wo_fwd", m, 0, p(state["attn"]), p(state["x"]), case["T"], p(state["out"]))
        return state["out"]
    if kind == "head":
        hb.call("hb_op_logits_ce", m, p(state["xn"]), p(state["targets"]), case["T"], p(state["logits"]),
                p(state["losses"]))
        return {"logits": state["logits"], "losses": state["losses"]}
    B, S = case["B"], case["S"]
    if kind == "forward":
        hb.call("hb_forward_device", m, p(state["tok"]), p(state["tgt"]), B, S, p(state["losses"]),
                p(state["logits"]), p(state["mean"]))
        return {"logits": state["logits"], "losses": state["losses"], "mean": state["mean"]}
    if kind == "decode":
        dec = state["dec"]
        dec.kv.reset()
        logits = [dec.prefill(state["prompt"])[0]]
        for tokens in state["next"]:
            logits.append(dec.step(tokens)[0])
        return {"prefill": logits[0], "steps": np.stack(logits[1:])}
    opt = state["opt"]
    opt.zero_grads()
    opt.forward_backward_device(p(state["tok"]), p(state["tgt"]), B, S, LOSS_SCALE, p(state["losses"]),
                                p(state["mean"]))
    return {"grads": state["grads"], "losses": state["losses"], "mean": state["mean"]}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "norm":
        n = case["T"] * case["dim"]
        return {"bytes": 6 * n + 4 * case["dim"] + 4 * case["T"], "flops": 4 * n}
    d, h, heads, kv_heads, hd, _ = SHAPES[case["shape"]]
    q, kv = heads * hd, kv_heads * hd

    def attention(B, S0, S1):  # causal scores and outputs of positions S0 .. S1-1
        keys = (S1 * (S1 + 1) - S0 * (S0 + 1)) // 2
        return 4 * B * heads * hd * keys

    if kind == "attn":
        B, S = case["B"], case["S"]
        T, w = B * S, d * (q + 2 * kv)
        return {"bytes": 2 * (w + T * (d + q)), "flops": 2 * T * w + attention(B, 0, S)}
    if kind == "ffn":
        T, w = case["T"], 3 * d * h
        return {"bytes": 2 * w + T * d * (2 + 4 + 4), "flops": 2 * T * w}
    if kind == "wo":
        T, w = case["T"], d * q
        return {"bytes": 2 * w + T * (2 * q + 8 * d), "flops": 2 * T * w}
    if kind == "head":
        T, w = case["T"], VOCAB * d
        return {"bytes": 2 * w + T * (2 * d + 4 * VOCAB), "flops": 2 * T * w}
    B, S, L = case["B"], case["S"], case["layers"]
    layer = d * (q + 2 * kv) + d * q + 3 * d * h
    mats = L * layer + VOCAB * d
    T = B * S
    if kind == "forward":
        return {"bytes": 2 * mats + 4 * T * VOCAB, "flops": 2 * T * mats + L * attention(B, 0, S)}
    if kind == "decode":
        n = case["steps"]
        rows = B * (sum(range(S + 1, S + n + 1)))
        return {"bytes": 2 * mats * (n + 1) + rows * L * 2 * kv * 2 + 4 * B * VOCAB * (n + 1),
                "flops": 2 * T * L * layer + 2 * B * VOCAB * d + 2 * B * n * mats + L * attention(B, 0, S + n)}
    # training: weights read for the forward and for the input gradients, fp32 gradients written once
    return {"bytes": 2 * 2 * mats + 4 * mats, "flops": 6 * T * mats + 3.5 * L * attention(B, 0, S)}


def tolerance(case):
    """About four times what the path measures against the 64-bit result: a
    norm 2.1e-4 (fp16 output), attention 5.4e-4 (fp16 operands and output), an
    FFN 5.4e-5 (fp16 gate under the fp32 residual), one projection or the head
    1e-7 (fp32 sums; 1e-5 allows any order), whole forwards 1.8e-3 (32 layers)
    and 9e-4 (decode), gradients 1.7e-3."""
    return {"rel": {"norm": 1e-3, "attn": 2e-3, "ffn": 2e-4, "wo": 1e-5, "head": 1e-5, "forward": 8e-3,
                    "decode": 4e-3, "train": 7e-3}[case["kind"]]}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
_M64 = (1 << 64) - 1


def _signed(v):
    v &= _M64
    return v - (1 << 64) if v >> 63 else v


def _mix_int(z):
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & _M64
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & _M64
    return z ^ (z >> 31)


def _shr(z, n):  # logical shift of int64 lanes
    return (z >> n) & ((1 << (64 - n)) - 1)


def _mix(z):
    z = (z ^ _shr(z, 30)) * _signed(0xBF58476D1CE4E5B9)
    z = (z ^ _shr(z, 27)) * _signed(0x94D049BB133111EB)
    return z ^ _shr(z, 31)


def _weights(seed, tensor, rows, cols):
    """The library's synthetic matrix [rows, cols], rounded to fp16 as it is stored."""
    key = _mix_int(((seed * 0x9E3779B97F4A7C15) & _M64) ^ (((tensor + 0x632BE59BD9B4E019) * 0xC2B2AE3D27D4EB4F) & _M64))
    scale = np.float32(float(np.float32(STD)) / math.sqrt(8.0 * (65536.0 * 65536.0 - 1.0) / 12.0))
    n = rows * cols
    out = torch.empty(n, dtype=torch.float16, device="cuda")
    step = 1 << 25
    for a in range(0, n, step):
        i = torch.arange(a, min(n, a + step), dtype=torch.int64, device="cuda")
        s = torch.full_like(i, -262140)
        for j in (0, 1):
            z = _mix((2 * i + j) * _signed(0x9E3779B97F4A7C15) + _signed(key))
            for b in range(4):
                s += (z >> (16 * b)) & 0xFFFF
        out[a:a + i.numel()] = (s.to(torch.float32) * float(scale)).to(torch.float16)
    return out.view(rows, cols).double()


def _layer_weights(case, seed, l):
    """Output-major matrices: qkv, wo, w1, w3, w2."""
    d, h, heads, kv_heads, hd, _ = SHAPES[case["shape"]]
    q, kv, b = heads * hd, kv_heads * hd, 16 * l
    w = lambda t, r, c: _weights(seed, b + t, r, c)  # noqa: E731
    qkv = torch.cat([w(0, d, q).t(), w(1, d, kv).t(), w(2, d, kv).t()]).contiguous()
    return [qkv, w(3, q, d).t().contiguous(), w(4, d, h).t().contiguous(), w(5, d, h).t().contiguous(), w(6, d, h)]


def _norm(x, gamma=None):
    y = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-5)
    return y if gamma is None else y * gamma


def _attention(case, xn, qkv, B, S):
    d, h, heads, kv_heads, hd, _ = SHAPES[case["shape"]]
    q, kv = heads * hd, kv_heads * hd
    y = xn @ qkv.t()
    i = torch.arange(hd // 2, dtype=torch.float64, device="cuda")
    ang = torch.arange(S, dtype=torch.float64, device="cuda")[:, None] / 10000.0 ** (2 * i / hd)
    c, s = torch.cos(ang), torch.sin(ang)

    def rope(v):  # [B, n, S, hd], interleaved pairs
        a, b = v[..., 0::2], v[..., 1::2]
        return torch.stack([a * c - b * s, a * s + b * c], -1).flatten(-2)

    def split(v, n):
        return v.reshape(B, S, n, hd).transpose(1, 2)

    Q = rope(split(y[:, :q], heads))
    K = rope(split(y[:, q:q + kv], kv_heads)).repeat_interleave(heads // kv_heads, 1)
    V = split(y[:, q + kv:], kv_heads).repeat_interleave(heads // kv_heads, 1)
    later = torch.ones(S, S, dtype=torch.bool, device="cuda").triu(1)
    out = []
    for b in range(B):
        sc = Q[b] @ K[b].transpose(-1, -2).contiguous() / math.sqrt(hd)
        out.append((torch.softmax(sc.masked_fill(later, -math.inf), -1) @ V[b]).transpose(0, 1).reshape(S, q))
    return torch.cat(out)


def _ffn(xn, w1, w3, w2):
    return (torch.nn.functional.silu(xn @ w1.t()) * (xn @ w3.t())) @ w2.t()


def _alpha(case):
    return float(np.float32(1.0 / math.sqrt(2.0 * SHAPES[case["shape"]][5])))


def _layer(case, x, w, g, B, S):
    qkv, wo, w1, w3, w2 = w
    x = x + _alpha(case) * _attention(case, _norm(x, g[0]), qkv, B, S) @ wo.t()
    return x + _alpha(case) * _ffn(_norm(x, g[1]), w1, w3, w2)


def _losses(logits, targets):
    t = torch.from_numpy(targets.astype(np.int64)).cuda()
    return torch.logsumexp(logits, -1) - logits.gather(1, t[:, None])[:, 0]


def exact(case, seed):
    kind = case["kind"]
    if kind == "norm":
        x = _randn(seed, (case["T"], case["dim"]), torch.float32).double()
        gamma = (1 + _randn(seed + 1, (case["dim"],), torch.float32, 0.1)).double()
        r = torch.rsqrt((x * x).mean(-1) + 1e-5)
        return {"out": x * r[:, None] * gamma, "rms_inv": r}
    d, h, heads, kv_heads, hd, _ = SHAPES[case["shape"]]
    with torch.no_grad():
        if kind in ("attn", "ffn", "wo"):
            st = {n: t.double() for n, t in _layer_inputs(case, seed).items()}
            qkv, wo, w1, w3, w2 = _layer_weights(case, seed, 0)
            if kind == "attn":
                return _attention(case, st["xn"], qkv, case["B"], case["S"])
            if kind == "wo":
                return st["x"] + _alpha(case) * st["attn"] @ wo.t()
            return st["x"] + _alpha(case) * _ffn(st["xn"], w1, w3, w2)
        embed = _weights(seed, hb.HB_SYNTH_EMBED_ID, VOCAB, d)
        if kind == "head":
            logits = _layer_inputs(case, seed)["xn"].double() @ embed.t()
            return {"logits": logits, "losses": _losses(logits, _tokens(seed, case["T"]))}
    B, S, L = case["B"], case["S"], case["layers"]
    if kind == "decode":
        n = case["steps"]
        ids = np.concatenate([_tokens(seed, B * S).reshape(B, S), _tokens(seed, n * B, 1).reshape(n, B).T], 1)
        S += n
    else:
        ids = _tokens(seed, B * S)
    ids = torch.from_numpy(ids.reshape(-1).astype(np.int64)).cuda()
    ones = torch.ones(d, dtype=torch.float64, device="cuda")
    if kind != "train":
        with torch.no_grad():
            x = embed[ids]
            for l in range(L):
                x = _layer(case, x, _layer_weights(case, seed, l), (ones, ones), B, S)
            logits = _norm(x) @ embed.t() if kind == "forward" else _norm(x.view(B, S, d)[:, case["S"] - 1:]) @ embed.t()
            if kind == "forward":
                losses = _losses(logits, _tokens(seed, B * S, 1))
                return {"logits": logits, "losses": losses, "mean": losses.mean().reshape(1)}
            return {"prefill": logits[:, 0], "steps": logits[:, 1:].transpose(0, 1).contiguous()}
    embed.requires_grad_()
    gf = ones.clone().requires_grad_()
    ws, gs = [], []
    x = embed[ids]
    for l in range(L):
        ws.append([w.requires_grad_() for w in _layer_weights(case, seed, l)])
        gs.append([ones.clone().requires_grad_(), ones.clone().requires_grad_()])
        x = _layer(case, x, ws[-1], gs[-1], B, S)
    losses = _losses(_norm(x, gf) @ embed.t(), _tokens(seed, B * S, 1))
    (losses.sum() * (LOSS_SCALE / S)).backward()
    grads = {"embed": embed.grad, "gamma": gf.grad}
    for l in range(L):
        qkv, wo, w1, w3, w2 = [w.grad for w in ws[l]]
        pairs = torch.stack([w1.view(h // 2, 2, d), w3.view(h // 2, 2, d)], 1).reshape(2 * h, d)
        for name, t in (("wqkv", qkv), ("wo", wo), ("w13", pairs), ("w2", w2), ("g1", gs[l][0].grad),
                        ("g2", gs[l][1].grad)):
            grads["l%d.%s" % (l, name)] = t
    losses = losses.detach()
    return {"grads": grads, "losses": losses, "mean": losses.mean().reshape(1)}
