"""The work a program has this framework do, as measurable cases.

A case is a dict of plain values.  ``kind`` selects the path:

  decode   one token per sequence against a KV cache (generation, serving)
  prefill  QK-Norm + RoPE of the keys, then causal attention of a prompt
  chunk    a continuation of a prompt into a paged cache
  masked   an ``Attention`` layer under a general attention mask
  model    a whole ``Qwen3Model`` call that returns logits
  train    attention forward and backward, as a training step runs it
  block    a ``TransformerBlock`` forward and backward

Head counts are those of the framework's own configurations: 8/2 (debug),
16/8, 32/8, 32/4 and 64/4 query / kv heads, head_dim 64 or 128.
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

import nano_qwen_amd as nq

DEV = "cuda"
EPS = 1e-6
THETA = 1e6
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}
ORIGINAL_POSITIONS = 32768  # positions before YaRN scaling


def listed():
    return [
        # the smallest call: one chat user's next token, short history
        dict(name="decode_one", kind="decode", B=1, Hq=32, Hkv=8, D=128, lo=1500, hi=1500, dtype="bf16", page=64),
        # a serving step: 32 users of very different histories on a page pool
        dict(name="decode_serving", kind="decode", B=32, Hq=32, Hkv=8, D=128, lo=200, hi=8192, dtype="bf16", page=64),
        # long-context serving at 16 query heads per kv head, dense per-row cache
        dict(name="decode_long", kind="decode", B=64, Hq=64, Hkv=4, D=128, lo=1024, hi=32768, dtype="bf16", page=0),
        # generation with the debug-sized fp32 model (torch's default dtype)
        dict(name="decode_f32", kind="decode", B=4, Hq=8, Hkv=2, D=64, lo=300, hi=2048, dtype="f32", page=0),
        # a short prompt through a whole small model
        dict(name="model_prompt", kind="model", B=1, S=173, hidden=1024, inter=3072, layers=4, vocab=8192,
             Hq=16, Hkv=8, D=128, dtype="bf16"),
        # a batch of ordinary sequences
        dict(name="prefill_batch", kind="prefill", B=8, S=2048, Hq=16, Hkv=8, D=128, dtype="bf16", yarn=False),
        # the longest context the framework is built for
        dict(name="prefill_yarn", kind="prefill", B=1, S=131072, Hq=32, Hkv=4, D=128, dtype="bf16", yarn=True),
        # the next turn of a long conversation: a few hundred new tokens on a long history
        dict(name="chunk_turn", kind="chunk", B=1, S=500, past=12345, Hq=32, Hkv=8, D=128, dtype="bf16", page=64),
        # a left-padded batch under a causal + padding mask
        dict(name="masked_layer", kind="masked", B=4, S=1024, hidden=2048, Hq=16, Hkv=8, D=128, dtype="bf16"),
        # the attention of a training step, long sequences
        dict(name="train_attention", kind="train", B=2, S=4096, Hq=32, Hkv=8, D=128, dtype="bf16"),
        # the attention of an fp32 training step at the debug configuration's heads
        dict(name="train_f32", kind="train", B=2, S=1000, Hq=8, Hkv=2, D=64, dtype="f32"),
        # a whole block of a training step
        dict(name="train_block", kind="block", B=2, S=2048, hidden=2048, inter=6144, Hq=16, Hkv=8, D=128,
             dtype="bf16"),
    ]


def _log(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "chunk", "chunk", "masked", "model",
                       "train", "train", "block"])
    if kind == "decode":
        if rng.random() < 0.3:
            Hq, Hkv, D = rng.choice([(8, 2, 64), (8, 2, 64), (16, 8, 128)])
            hi = _log(rng, 64, 4096)
            return dict(kind=kind, B=_log(rng, 1, 8), Hq=Hq, Hkv=Hkv, D=D, lo=max(1, hi // rng.randint(1, 8)), hi=hi,
                        dtype="f32", page=rng.choice([0, 64]))
        Hq, Hkv = rng.choice([(16, 8), (32, 8), (32, 4), (64, 4)])
        hi = _log(rng, 100, 32768)
        B = _log(rng, 1, max(1, min(64, 2 ** 21 // hi)))
        return dict(kind=kind, B=B, Hq=Hq, Hkv=Hkv, D=128, lo=max(1, hi // rng.randint(1, 32)), hi=hi, dtype="bf16",
                    page=rng.choice([0, 32, 64, 128]))
    if kind == "prefill":
        Hq, Hkv, D = rng.choice([(16, 8, 128), (32, 8, 128), (32, 4, 128), (8, 2, 64)])
        S = _log(rng, 30, 65536)
        B = _log(rng, 1, max(1, min(16, 32768 // S)))
        return dict(kind=kind, B=B, S=S, Hq=Hq, Hkv=Hkv, D=D, dtype="bf16", yarn=S > ORIGINAL_POSITIONS)
    if kind == "chunk":
        Hq, Hkv = rng.choice([(16, 8), (32, 8), (32, 4)])
        return dict(kind=kind, B=rng.choice([1, 1, 2, 4]), S=_log(rng, 16, 2048), past=_log(rng, 100, 30000), Hq=Hq,
                    Hkv=Hkv, D=128, dtype="bf16", page=rng.choice([32, 64, 128]))
    if kind == "masked":
        hidden, Hq, Hkv, D = rng.choice([(2048, 16, 8, 128), (4096, 32, 8, 128), (256, 8, 2, 64)])
        S = _log(rng, 50, 2048)
        return dict(kind=kind, B=_log(rng, 1, max(1, min(8, 4096 // S))), S=S, hidden=hidden, Hq=Hq, Hkv=Hkv, D=D,
                    dtype="bf16")
    if kind == "model":
        hidden, inter, Hq, Hkv, D = rng.choice([(1024, 3072, 16, 8, 128), (256, 1024, 8, 2, 64)])
        S = _log(rng, 10, 1500)
        return dict(kind=kind, B=_log(rng, 1, max(1, min(8, 2048 // S))), S=S, hidden=hidden, inter=inter,
                    layers=rng.randint(2, 4), vocab=8192, Hq=Hq, Hkv=Hkv, D=D, dtype="bf16")
    if kind == "train":
        if rng.random() < 0.4:
            S = _log(rng, 60, 2048)
            return dict(kind=kind, B=_log(rng, 1, max(1, min(8, 4096 // S))), S=S, Hq=8, Hkv=2, D=64, dtype="f32")
        Hq, Hkv = rng.choice([(16, 8), (32, 8)])
        S = _log(rng, 128, 4096)
        return dict(kind=kind, B=_log(rng, 1, max(1, min(8, 8192 // S))), S=S, Hq=Hq, Hkv=Hkv, D=128, dtype="bf16")
    hidden, inter, Hq, Hkv, D = rng.choice([(2048, 6144, 16, 8, 128), (1024, 3072, 16, 8, 128), (256, 1024, 8, 2, 64)])
    S = _log(rng, 100, 2048)
    return dict(kind="block", B=_log(rng, 1, max(1, min(8, 4096 // S))), S=S, hidden=hidden, inter=inter, Hq=Hq,
                Hkv=Hkv, D=D, dtype="bf16")


# ---------------------------------------------------------------------------
# inputs, from the seed alone
# ---------------------------------------------------------------------------

class _Inputs:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(seed)

    def normal(self, *shape, dtype=torch.float32, std=1.0):
        t = torch.randn(*shape, generator=self.g, device=DEV, dtype=dtype)
        return t.mul_(std) if std != 1.0 else t

    def norm_weight(self, n, dtype):
        return (1 + 0.02 * self.normal(n)).to(dtype)


def _tables(D, n, yarn=False):
    """fp32 cos and sin tables (n, D/2), on the host as a model builds them."""
    expo = torch.arange(0, D, 2, dtype=torch.float32) / D
    inv = 1.0 / (THETA ** expo)
    if yarn:
        def dim_at(turns):
            return D * math.log(ORIGINAL_POSITIONS / (turns * 2 * math.pi)) / (2 * math.log(THETA))
        low, high = max(math.floor(dim_at(32.0)), 0), min(math.ceil(dim_at(1.0)), D - 1)
        ramp = ((torch.arange(D // 2, dtype=torch.float32) - low) / (high - low)).clamp(0, 1)
        inv = inv / 4.0 * ramp + inv * (1 - ramp)
    ang = torch.outer(torch.arange(n, dtype=torch.float32), inv)
    return ang.cos().to(DEV), ang.sin().to(DEV)


def _lengths(case):
    """Rows already cached per sequence: spread evenly from lo to hi (the seed only orders them)."""
    B, lo, hi = case["B"], case["lo"], case["hi"]
    return [hi if B == 1 else lo + (hi - lo) * i // (B - 1) for i in range(B)]


def _decode_inputs(case, seed):
    B, Hq, Hkv, D, dt = case["B"], case["Hq"], case["Hkv"], case["D"], DTYPES[case["dtype"]]
    r = _Inputs(seed)
    lens = torch.tensor(_lengths(case), dtype=torch.int32, device=DEV)[torch.randperm(B, generator=r.g, device=DEV)]
    rows = case["hi"] + 1  # the new token's row included
    page = case["page"] or (rows + 63) // 64 * 64
    per = -(-rows // page)
    if case["page"]:
        bt = torch.randperm(B * per, generator=r.g, device=DEV).to(torch.int32).view(B, per)
    else:  # a dense cache is one page per sequence
        bt = torch.arange(B, dtype=torch.int32, device=DEV).view(B, 1)
    cos, sin = _tables(D, rows)
    return dict(q=r.normal(B, Hq, 1, D, dtype=dt), k_new=r.normal(B, Hkv, 1, D, dtype=dt),
                v_new=r.normal(B, Hkv, 1, D, dtype=dt), qw=r.norm_weight(D, dt), kw=r.norm_weight(D, dt),
                kp=r.normal(B * per, Hkv, page, D, dtype=dt), vp=r.normal(B * per, Hkv, page, D, dtype=dt),
                bt=bt, lens=lens, cos=cos, sin=sin, max_len=rows, page=page)


def _prefill_inputs(case, seed, positions):
    B, S, Hq, Hkv, D, dt = case["B"], case["S"], case["Hq"], case["Hkv"], case["D"], DTYPES[case["dtype"]]
    r = _Inputs(seed)
    cos, sin = _tables(D, positions, case.get("yarn", False))
    # the projections' storage is (B, S, H, D)
    return r, dict(q=r.normal(B, S, Hq, D, dtype=dt).transpose(1, 2), k=r.normal(B, S, Hkv, D, dtype=dt).transpose(1, 2),
                   v=r.normal(B, S, Hkv, D, dtype=dt).transpose(1, 2), qw=r.norm_weight(D, dt),
                   kw=r.norm_weight(D, dt), cos=cos, sin=sin)


def _chunk_inputs(case, seed):
    B, Hkv, D, dt, page = case["B"], case["Hkv"], case["D"], DTYPES[case["dtype"]], case["page"]
    T = case["past"] + case["S"]
    r, s = _prefill_inputs(case, seed, T)
    per = -(-T // page)
    s.update(bt=torch.randperm(B * per, generator=r.g, device=DEV).to(torch.int32).view(B, per),
             kp=r.normal(B * per, Hkv, page, D, dtype=dt), vp=r.normal(B * per, Hkv, page, D, dtype=dt))
    return s


def _config(case):
    return nq.ModelConfig(hidden_size=case["hidden"], num_attention_heads=case["Hq"],
                          num_key_value_heads=case["Hkv"], head_dim=case["D"], max_position_embeddings=4096,
                          rms_norm_eps=EPS, rope_theta=THETA, vocab_size=case.get("vocab", 64),
                          num_hidden_layers=case.get("layers", 1), intermediate_size=case.get("inter", 64))


def _module(case, seed, make):
    """A module with weights from the seed: matrices N(0, 0.02), norm weights about 1."""
    with torch.device(DEV):
        m = make(_config(case)).to(DTYPES[case["dtype"]])
    r = _Inputs(seed)
    with torch.no_grad():
        for name, p in m.named_parameters():
            p.copy_(r.norm_weight(p.shape[0], p.dtype) if p.dim() == 1 else r.normal(*p.shape, dtype=p.dtype, std=0.02))
    return r, m


def _mask(case, r):
    """(B, 1, S, S) bool: causal, and each sequence's left padding (up to half of it) masked."""
    B, S = case["B"], case["S"]
    pad = torch.randint(0, S // 2 + 1, (B,), generator=r.g, device=DEV)
    i = torch.arange(S, device=DEV)
    return (i[None, :] <= i[:, None])[None, None] & (i[None, :] >= pad[:, None])[:, None, None, :]


def prepare(case, seed):
    kind, dt = case["kind"], DTYPES[case["dtype"]]
    if kind == "decode":
        s = _decode_inputs(case, seed)
        s["lens_out"] = torch.empty_like(s["lens"])
        s["ws"] = None
        if dt == torch.bfloat16:
            n = nq.decode_workspace_bytes(case["B"], case["Hq"], case["Hkv"], case["D"], s["max_len"])
            s["ws"] = torch.empty(n, dtype=torch.uint8, device=DEV)
    elif kind == "prefill":
        s = _prefill_inputs(case, seed, case["S"])[1]
    elif kind == "chunk":
        s = _chunk_inputs(case, seed)
    elif kind == "train":
        r, s = _prefill_inputs(case, seed, case["S"])
        for n in ("q", "k", "v", "qw", "kw"):
            s[n].requires_grad_()
        s["do"] = r.normal(case["B"], case["S"], case["Hq"], case["D"], dtype=dt).transpose(1, 2)
    elif kind == "masked":
        r, m = _module(case, seed, nq.Attention)
        s = dict(m=m.eval(), x=r.normal(case["B"], case["S"], case["hidden"], dtype=dt), mask=_mask(case, r))
    elif kind == "model":
        r, m = _module(case, seed, nq.Qwen3Model)
        s = dict(m=m.eval(), ids=torch.randint(0, case["vocab"], (case["B"], case["S"]), generator=r.g, device=DEV))
    else:
        r, m = _module(case, seed, nq.TransformerBlock)
        x = r.normal(case["B"], case["S"], case["hidden"], dtype=dt).requires_grad_()
        s = dict(m=m.train(), x=x, params=[x] + list(m.parameters()),
                 do=r.normal(case["B"], case["S"], case["hidden"], dtype=dt))
    s["case"] = case
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "decode":
        # QK-Norm + RoPE, the new token's append and its attention
        with torch.no_grad():
            o = nq.attention_decode_paged(s["q"], s["kp"], s["vp"], s["bt"], s["lens"], max_len=s["max_len"],
                                          k_new=s["k_new"], v_new=s["v_new"], k_weight=s["kw"],
                                          lens_out=s["lens_out"], q_weight=s["qw"], eps=EPS, cos=s["cos"],
                                          sin=s["sin"], workspace=s["ws"])
        return [o, s["lens_out"], s["kp"], s["vp"]]
    if kind == "prefill":
        with torch.no_grad():
            _, k_hat, _ = nq.qk_norm_rope(k=s["k"], k_weight=s["kw"], eps=EPS, cos=s["cos"], sin=s["sin"])
            o = nq.attention_prefill(s["q"], k_hat, s["v"], q_weight=s["qw"], eps=EPS, cos=s["cos"], sin=s["sin"])
        return [o, k_hat]
    if kind == "chunk":
        past, T = case["past"], case["past"] + case["S"]
        with torch.no_grad():
            nq.kv_append_paged(s["k"], s["v"], s["kp"], s["vp"], s["bt"], k_weight=s["kw"], eps=EPS, cos=s["cos"],
                               sin=s["sin"], row_offset=past, pos_offset=past)
            o = nq.attention_prefill_paged(s["q"], s["kp"], s["vp"], s["bt"], T=T, q_weight=s["qw"], eps=EPS,
                                           cos=s["cos"], sin=s["sin"], pos_offset=past)
        return [o, s["kp"], s["vp"]]
    if kind == "train":
        o = nq.attention_core(s["q"], s["k"], s["v"], s["qw"], s["kw"], cos=s["cos"], sin=s["sin"], eps=EPS)
        return [o, *torch.autograd.grad(o, (s["q"], s["k"], s["v"], s["qw"], s["kw"]), s["do"])]
    if kind == "masked":
        with torch.no_grad():
            return [s["m"](s["x"], attention_mask=s["mask"])]
    if kind == "model":
        with torch.no_grad():
            return [s["m"](s["ids"])["logits"]]
    y, _ = s["m"](s["x"])
    return [y, *torch.autograd.grad(y, s["params"], s["do"])]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def work(case):
    B, Hq, Hkv, D = case["B"], case["Hq"], case["Hkv"], case["D"]
    es = 2 if case["dtype"] == "bf16" else 4
    if case["kind"] == "decode":
        keys = sum(n + 1 for n in _lengths(case))
        return {"bytes": 2 * Hkv * D * es * (keys + B) + 2 * B * Hq * D * es, "flops": 4 * D * Hq * keys}
    S = case["S"]
    past = case.get("past", 0)
    pairs = B * Hq * (S * past + S * (S + 1) // 2)
    qo, kv = B * S * Hq * D * es, B * S * Hkv * D * es
    if case["kind"] == "prefill":  # q, k, v in; o and the rotated keys out
        return {"bytes": 2 * qo + 3 * kv, "flops": 4 * D * pairs}
    if case["kind"] == "chunk":  # q and the new k, v in; the cached rows in; o and the new rows out
        return {"bytes": 2 * qo + 4 * kv + 2 * B * past * Hkv * D * es, "flops": 4 * D * pairs}
    if case["kind"] == "train":  # q, k, v, dO in; o, dq, dk, dv out
        return {"bytes": 4 * qo + 4 * kv, "flops": 14 * D * pairs}
    hid = case["hidden"]
    attn_w = hid * D * (2 * Hq + 2 * Hkv)
    ffn_w = 3 * hid * case.get("inter", 0)
    tok = B * S
    if case["kind"] == "masked":
        # padding of 0 to S/2 leaves 7/12 of the causal pairs on average
        return {"bytes": es * (attn_w + 2 * tok * hid) + B * S * S,
                "flops": 2 * tok * attn_w + 4 * D * pairs * 7 // 12}
    if case["kind"] == "model":
        L, V = case["layers"], case["vocab"]
        return {"bytes": es * (L * (attn_w + ffn_w) + V * hid + tok * (hid + V)),
                "flops": L * (2 * tok * (attn_w + ffn_w) + 4 * D * pairs) + 2 * tok * V * hid}
    return {"bytes": es * (2 * (attn_w + ffn_w) + 4 * tok * hid),
            "flops": 6 * tok * (attn_w + ffn_w) + 14 * D * pairs}


def tolerance(case):
    # about four times what a pass differs from 64-bit arithmetic by: 1.3e-6 in
    # fp32; in bf16 0.3% for one attention, 0.4% with its gradients or the
    # projections around it, 1% for a block's gradients and the logits
    if case["dtype"] == "f32":
        return {"rel": 6e-6}
    return {"rel": {"decode": 1.2e-2, "prefill": 1.2e-2, "chunk": 1.2e-2, "masked": 1.7e-2, "model": 4e-2,
                    "train": 1.7e-2, "block": 4e-2}[case["kind"]]}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------

def _rms(x, w):
    x = x.double()
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _rope(x, cos, sin):
    """x (..., S, D) at the positions of the table rows given."""
    a, b = x.chunk(2, -1)
    c, n = cos.double(), sin.double()
    return torch.cat((a * c - b * n, b * c + a * n), -1)


def _attend(q, k, v, keep=None, past=0, block=1024):
    """Causal attention after `past` keys (or under keep (S, T)) of q (Hq, S, D), k / v (Hkv, T, D)."""
    Hq, S, D = q.shape
    Hkv, T = k.shape[:2]
    G = Hq // Hkv
    heads = []
    for j in range(Hkv):
        kt, vj = k[j].t().contiguous(), v[j]
        parts = []
        for i in range(0, S, block):
            n = min(block, S - i)
            end = T if keep is not None else min(T, past + i + n)
            x = (q[j * G:(j + 1) * G, i:i + n].reshape(G * n, D) @ kt[:, :end]).view(G, n, end) / math.sqrt(D)
            m = keep[i:i + n] if keep is not None else (torch.arange(end, device=DEV)[None, :]
                                                        <= past + torch.arange(i, i + n, device=DEV)[:, None])
            x = x.masked_fill(~m, float("-inf"))
            p = torch.softmax(x, -1)
            if keep is not None:  # a row that keeps no key gives zeros
                p = p.masked_fill(~m.any(-1)[None, :, None], 0.0)
            parts.append((p.view(G * n, end) @ vj[:end]).view(G, n, D))
        heads.append(torch.cat(parts, 1))
    return torch.cat(heads, 0)


def _layer(w, x, case, cos, sin, keep=None):
    """The attention layer of parameters w on x (B, S, hidden)."""
    B, S, Hq, Hkv, D = case["B"], case["S"], case["Hq"], case["Hkv"], case["D"]

    def split(name, H):
        return F.linear(x, w[name + ".weight"]).view(B, S, H, D).transpose(1, 2)
    q = _rope(_rms(split("q_proj", Hq), w["q_norm.weight"]), cos, sin)
    k = _rope(_rms(split("k_proj", Hkv), w["k_norm.weight"]), cos, sin)
    v = split("v_proj", Hkv)
    o = torch.stack([_attend(q[b], k[b], v[b], None if keep is None else keep[b, 0]) for b in range(B)])
    return F.linear(o.transpose(1, 2).reshape(B, S, Hq * D), w["o_proj.weight"])


def _block(w, x, case, cos, sin):
    x = x + _layer({n[len("attention."):]: p for n, p in w.items() if n.startswith("attention.")},
                   _rms(x, w["input_layernorm.weight"]), case, cos, sin)
    h = _rms(x, w["post_attention_layernorm.weight"])
    g = F.silu(F.linear(h, w["feed_forward.gate_proj.weight"])) * F.linear(h, w["feed_forward.up_proj.weight"])
    return x + F.linear(g, w["feed_forward.down_proj.weight"])


def _doubles(m):
    return {n: p.detach().double().requires_grad_(p.requires_grad) for n, p in m.named_parameters()}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("prefill", "chunk", "train") and work(case)["flops"] > 3e13:
        return None  # over about 20 seconds in 64 bits
    if kind == "decode":
        s = _decode_inputs(case, seed)
        page, outs = s["page"], []
        kp, vp = s["kp"].clone(), s["vp"].clone()
        for b, n in enumerate(s["lens"].tolist()):
            c, sn = s["cos"][n], s["sin"][n]
            q = _rope(_rms(s["q"][b, :, 0], s["qw"]), c, sn)
            kn = _rope(_rms(s["k_new"][b, :, 0], s["kw"]), c, sn)
            pages = s["bt"][b, :n // page + 1].long()
            k = s["kp"][pages].transpose(0, 1).flatten(1, 2)[:, :n].double()
            v = s["vp"][pages].transpose(0, 1).flatten(1, 2)[:, :n].double()
            k, v = torch.cat((k, kn[:, None]), 1), torch.cat((v, s["v_new"][b].double()), 1)
            outs.append(_attend(q[:, None], k, v, past=n)[:, 0])
            kp[pages[-1], :, n % page], vp[pages[-1], :, n % page] = kn.to(kp.dtype), s["v_new"][b, :, 0]
        # the pools hold 16- or 32-bit copies of what was given, and rounded rows
        return [torch.stack(outs), s["lens"] + 1, None, None]
    if kind in ("prefill", "chunk"):
        past = case.get("past", 0)
        s = _chunk_inputs(case, seed) if past else _prefill_inputs(case, seed, case["S"])[1]
        T = past + case["S"]
        c, sn = s["cos"][past:T], s["sin"][past:T]
        outs, khat = [], []
        for b in range(case["B"]):
            q, k = _rope(_rms(s["q"][b], s["qw"]), c, sn), _rope(_rms(s["k"][b], s["kw"]), c, sn)
            v = s["v"][b].double()
            khat.append(k)
            if past:
                pages = s["bt"][b].long()
                k = torch.cat((s["kp"][pages].transpose(0, 1).flatten(1, 2)[:, :past].double(), k), 1)
                v = torch.cat((s["vp"][pages].transpose(0, 1).flatten(1, 2)[:, :past].double(), v), 1)
            outs.append(_attend(q, k, v, past=past))
        return [torch.stack(outs), None, None] if past else [torch.stack(outs), torch.stack(khat)]
    if kind == "train":
        r, s = _prefill_inputs(case, seed, case["S"])
        do = r.normal(case["B"], case["S"], case["Hq"], case["D"], dtype=DTYPES[case["dtype"]]).transpose(1, 2)
        leaves = [s[n].double().requires_grad_() for n in ("q", "k", "v", "qw", "kw")]
        q, k = _rope(_rms(leaves[0], leaves[3]), s["cos"], s["sin"]), _rope(_rms(leaves[1], leaves[4]), s["cos"], s["sin"])
        o = torch.stack([_attend(q[b], k[b], leaves[2][b]) for b in range(case["B"])])
        return [o.detach(), *torch.autograd.grad(o, leaves, do.double())]
    cos, sin = _tables(case["D"], case["S"])
    if kind == "masked":
        r, m = _module(case, seed, nq.Attention)
        x = r.normal(case["B"], case["S"], case["hidden"], dtype=DTYPES[case["dtype"]])
        with torch.no_grad():
            return [_layer(_doubles(m), x.double(), case, cos, sin, _mask(case, r))]
    if kind == "model":
        r, m = _module(case, seed, nq.Qwen3Model)
        ids = torch.randint(0, case["vocab"], (case["B"], case["S"]), generator=r.g, device=DEV)
        w = _doubles(m)
        with torch.no_grad():
            x = w["embed.embed_tokens.weight"][ids]
            for i in range(case["layers"]):
                pre = "layers.%d." % i
                x = _block({n[len(pre):]: p for n, p in w.items() if n.startswith(pre)}, x, case, cos, sin)
            return [F.linear(_rms(x, w["norm.weight"]), w["lm_head.weight"])]
    r, m = _module(case, seed, nq.TransformerBlock)
    dt = DTYPES[case["dtype"]]
    x = r.normal(case["B"], case["S"], case["hidden"], dtype=dt).double().requires_grad_()
    do = r.normal(case["B"], case["S"], case["hidden"], dtype=dt)
    w = _doubles(m)
    y = _block(w, x, case, cos, sin)
    return [y.detach(), *torch.autograd.grad(y, [x] + list(w.values()), do.double())]
