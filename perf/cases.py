"""The work this library is measured on: attention and Gated DeltaNet calls through the Python
binding, as a program that serves or evaluates a model makes them.

A case is a dict of plain values; `kind` names the entry points it goes through:

  attn       tsa.attn_fwd, equal query and K/V heads
  gqa        tsa.attn_gqa_fwd with the output gate (grouped query heads)
  prefill    tsa.gdn_chunked_fwd, the state carried in place, the workspace kept by the caller
  layer      tsa.gdn_chunked_fused_fwd on raw projections, then tsa.gdn_gated_rmsnorm
  serial     tsa.gdn_recurrent_fwd
  decode     tsa.gdn_decode_step, or with `fused` tsa.gdn_decode_fused_step
  ggml       tsa.ggml_gated_delta_net on strided fp32 views of one projection, a state of its
             own for the result
"""
import math
import os
import sys

import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "turing-sm75_amd"))
import tsa  # noqa: E402

DK = 128
EPS = 1e-6


def listed():
    return [
        # a short batch at the small head size: a few prompts of a small model, latency counts
        {"name": "attn_b2h8_s512_d64", "kind": "attn", "B": 2, "H": 8, "S": 512, "D": 64, "causal": True},
        # an ordinary prompt of odd length
        {"name": "attn_h32_s2001_d128", "kind": "attn", "B": 1, "H": 32, "S": 2001, "D": 128, "causal": True},
        # a long prompt: the largest call
        {"name": "attn_h32_s8192_d128", "kind": "attn", "B": 1, "H": 32, "S": 8192, "D": 128, "causal": True},
        # the gated grouped-query layer (24 query / 4 K/V heads, D = 256) on an ordinary prompt
        {"name": "gqa_24_4_s3000_d256", "kind": "gqa", "B": 1, "Hq": 24, "Hkv": 4, "S": 3000, "D": 256, "causal": True},
        # chunked prefill of a 4096-token prompt, 16 QK / 32 V heads
        {"name": "prefill_t4096_hv32", "kind": "prefill", "B": 1, "T": 4096, "Hq": 16, "Hv": 32, "f32": False},
        # the share of it that one of eight GPUs holds under head sharding
        {"name": "prefill_t4096_hv4", "kind": "prefill", "B": 1, "T": 4096, "Hq": 2, "Hv": 4, "f32": False},
        # fp32 I/O at 512 tokens and 48 V-heads, the lab driver's default run
        {"name": "prefill_f32_t512_hv48", "kind": "prefill", "B": 1, "T": 512, "Hq": 16, "Hv": 48, "f32": True},
        # a whole layer from raw projections on a prompt of odd length
        {"name": "layer_t1000_hv48", "kind": "layer", "B": 1, "T": 1000, "Hq": 16, "Hv": 48},
        # the token-serial recurrence at the lab driver's default run
        {"name": "serial_f32_t512_hv48", "kind": "serial", "B": 1, "T": 512, "Hq": 16, "Hv": 48, "f32": True},
        # one decode step of a batch of 16 sequences
        {"name": "decode_b16_hv32", "kind": "decode", "B": 16, "Hq": 16, "Hv": 32, "f32": False, "fused": False},
        # one decode step of one sequence from raw projections: the smallest call
        {"name": "decode_fused_b1_hv48", "kind": "decode", "B": 1, "Hq": 16, "Hv": 48, "f32": False, "fused": True},
        # one token for each of 8 server slots through the ggml views
        {"name": "ggml_b8_t1_hv48", "kind": "ggml", "B": 8, "T": 1, "Hq": 16, "Hv": 48},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["attn", "attn", "gqa", "prefill", "prefill", "layer", "serial", "decode", "ggml"])
    heads = rng.choice([(2, 4), (4, 8), (16, 16), (16, 32), (16, 48), (3, 7)])
    if kind == "attn":
        D = rng.choice([64, 128])
        c = {"B": rng.choice([1, 1, 2, 3]), "H": rng.choice([4, 8, 12, 32]), "S": _log_int(rng, 60, 6000), "D": D,
             "causal": rng.random() < 0.75}
    elif kind == "gqa":
        g = rng.choice([(24, 4), (16, 2), (6, 1), (8, 8)])
        c = {"B": rng.choice([1, 1, 2]), "Hq": g[0], "Hkv": g[1], "S": _log_int(rng, 60, 4000),
             "D": rng.choice([128, 256, 256]), "causal": rng.random() < 0.9}
    elif kind == "prefill":
        c = {"B": rng.choice([1, 1, 1, 2, 3]), "T": _log_int(rng, 33, 5000), "Hq": heads[0], "Hv": heads[1],
             "f32": rng.random() < 0.4}
    elif kind == "layer":
        c = {"B": rng.choice([1, 1, 2]), "T": _log_int(rng, 33, 4000), "Hq": heads[0], "Hv": heads[1]}
    elif kind == "serial":
        c = {"B": rng.choice([1, 2, 4]), "T": _log_int(rng, 2, 600), "Hq": heads[0], "Hv": heads[1],
             "f32": rng.random() < 0.5}
    elif kind == "decode":
        fused = rng.random() < 0.5
        c = {"B": _log_int(rng, 1, 40), "Hq": heads[0], "Hv": heads[1], "f32": not fused and rng.random() < 0.4,
             "fused": fused}
    else:
        c = {"B": _log_int(rng, 1, 16), "T": _log_int(rng, 1, 60), "Hq": heads[0], "Hv": heads[1]}
    c = {"kind": kind, **c}
    # no call larger than the largest listed ones
    while kind in ("attn", "gqa") and work(c)["flops"] > 5e11:
        c["S"] = c["S"] * 3 // 4 + 1
    while kind in ("prefill", "layer") and c["B"] * c["T"] * c["Hv"] > 200000:
        c["T"] = c["T"] * 3 // 4 + 1
    return c


class _Draw:
    """Seeded tensors on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed))

    def normal(self, *shape):
        return torch.randn(*shape, generator=self.g, device="cuda", dtype=torch.float32)

    def uniform(self, *shape):
        return torch.rand(*shape, generator=self.g, device="cuda", dtype=torch.float32)


def _attn_inputs(c, d):
    Hq, Hkv = c.get("Hq", c.get("H")), c.get("Hkv", c.get("H"))

    def tensor(h):
        x = 0.5 * d.normal(c["B"], h, c["S"], c["D"])
        if c["kind"] == "attn" and c["S"] > 4096:  # long context: 1 % outliers, eight times as large
            x = torch.where(d.uniform(*x.shape) < 0.01, 8 * x, x)
        return x.half()

    s = {"q": tensor(Hq), "k": tensor(Hkv), "v": tensor(Hkv)}
    if c["kind"] == "gqa":
        s["gate"] = d.normal(c["B"], Hq, c["S"], c["D"]).half()
    return s


def _gdn_inputs(c, d):
    B, T, Hq, Hv = c["B"], c.get("T", 1), c["Hq"], c["Hv"]
    fused = c["kind"] == "layer" or c.get("fused", False)
    io = torch.float32 if c.get("f32", False) or c["kind"] == "ggml" else torch.float16
    q, k, v = d.normal(B, T, Hq, DK), d.normal(B, T, Hq, DK), d.normal(B, T, Hv, DK)
    s = {"state": 0.02 * d.normal(B, Hv, DK, DK)}
    if fused:  # raw rows; the decay projections in the ranges such a layer is initialised to
        s.update(a=d.normal(B, T, Hv), b=d.normal(B, T, Hv))
        s["A"] = -(1 + 15 * d.uniform(Hv))
        s["dt_bias"] = torch.log(torch.expm1(0.001 + 0.1 * d.uniform(Hv)))
    else:
        q, k = F.normalize(q, dim=-1), F.normalize(k, dim=-1)
        s.update(g=-F.softplus(d.normal(B, T, Hv)), beta=torch.sigmoid(d.normal(B, T, Hv)))
    s.update(q=q.to(io), k=k.to(io), v=v.to(io))
    if c["kind"] == "layer":
        s.update(z=d.normal(B, T, Hv, DK).half(), w=1 + 0.1 * d.normal(DK))
    if c["kind"] == "decode":  # one token: no T dimension
        for n in ("q", "k", "v", "a", "b", "g", "beta"):
            if n in s:
                s[n] = s[n][:, 0].contiguous()
    return s


def prepare(case, seed):
    c, d = case, _Draw(seed)
    if c["kind"] in ("attn", "gqa"):
        return {"case": c, **_attn_inputs(c, d)}
    s = {"case": c, **_gdn_inputs(c, d)}
    if c["kind"] in ("prefill", "layer"):
        n = tsa.gdn_chunked_workspace_bytes(c["B"], c["T"], c["Hq"], c["Hv"], f32=c.get("f32", False))
        s["ws"] = torch.empty(n, dtype=torch.uint8, device="cuda")
    elif c["kind"] == "decode":  # a serving loop keeps its output buffer
        s["out"] = torch.empty_like(s["v"])
    elif c["kind"] == "ggml":  # q, k and v side by side in one projection's rows
        B, T, Hq, Hv = c["B"], c["T"], c["Hq"], c["Hv"]
        proj = torch.cat([s["q"].flatten(2), s["k"].flatten(2), s["v"].flatten(2)], dim=2)
        n = Hq * DK
        s["q"] = proj[:, :, :n].unflatten(2, (Hq, DK))
        s["k"] = proj[:, :, n:2 * n].unflatten(2, (Hq, DK))
        s["v"] = proj[:, :, 2 * n:].unflatten(2, (Hv, DK))
        s["out"] = torch.empty(B, T, Hv, DK, device="cuda")
        s["state_out"] = torch.empty_like(s["state"])
        s["ws"] = torch.empty(tsa.ggml_gdn_workspace_bytes(s["q"], s["v"]), dtype=torch.uint8, device="cuda")
    return s


def run(s):
    c = s["case"]
    if c["kind"] == "attn":
        return tsa.attn_fwd(s["q"], s["k"], s["v"], causal=c["causal"])
    if c["kind"] == "gqa":
        return tsa.attn_gqa_fwd(s["q"], s["k"], s["v"], s["gate"], causal=c["causal"])
    if c["kind"] == "prefill":
        return tsa.gdn_chunked_fwd(s["q"], s["k"], s["v"], s["g"], s["beta"], s["state"], ws=s["ws"]), s["state"]
    if c["kind"] == "layer":
        o = tsa.gdn_chunked_fused_fwd(s["q"], s["k"], s["v"], s["a"], s["b"], s["dt_bias"], s["A"], s["state"],
                                      eps=EPS, ws=s["ws"])
        return tsa.gdn_gated_rmsnorm(o, s["z"], s["w"], eps=EPS), s["state"]
    if c["kind"] == "serial":
        return tsa.gdn_recurrent_fwd(s["q"], s["k"], s["v"], s["g"], s["beta"], s["state"]), s["state"]
    if c["kind"] == "decode":
        if c["fused"]:
            o = tsa.gdn_decode_fused_step(s["q"], s["k"], s["v"], s["a"], s["b"], s["dt_bias"], s["A"], s["state"],
                                          out=s["out"], eps=EPS)
        else:
            o = tsa.gdn_decode_step(s["q"], s["k"], s["v"], s["g"], s["beta"], s["state"], out=s["out"])
        return o, s["state"]
    o = tsa.ggml_gated_delta_net(s["q"], s["k"], s["v"], s["g"], s["beta"], s["state"], s["out"], s["state_out"],
                                 ws=s["ws"])
    return o, s["state_out"]


def work(case):
    c = case
    if c["kind"] in ("attn", "gqa"):
        Hq, Hkv = c.get("Hq", c.get("H")), c.get("Hkv", c.get("H"))
        pairs = c["S"] * (c["S"] + 1) // 2 if c["causal"] else c["S"] * c["S"]
        rows = 2 * Hkv + (3 if c["kind"] == "gqa" else 2) * Hq
        return {"bytes": 2 * c["B"] * rows * c["S"] * c["D"], "flops": 4 * c["B"] * Hq * pairs * c["D"]}
    B, T, Hq, Hv = c["B"], c.get("T", 1), c["Hq"], c["Hv"]
    e = 4 if c.get("f32", False) or c["kind"] == "ggml" else 2
    rows = e * B * T * DK * (2 * Hq + 2 * Hv) + 8 * B * T * Hv
    state = 2 * 4 * B * Hv * DK * DK
    # per token and V-head: S^T k, the rank-1 update, S^T q
    flops = 6 * B * T * Hv * DK * DK
    if c["kind"] == "layer":
        rows += 2 * 2 * B * T * Hv * DK
        flops += 10 * B * T * Hv * DK
    return {"bytes": rows + state, "flops": flops}


def tolerance(case):
    # about four times the difference from exact(): 2.3e-4 to 3e-4 in attention (fp16 P and
    # output), 3.6e-4 to 4.4e-4 in the chunked recurrence (fp16 operands), 2.1e-4 where only the
    # output is rounded to fp16, 1e-7 where all is fp32
    if case["kind"] in ("attn", "gqa"):
        return {"rel": 1e-3}
    if case["kind"] in ("prefill", "layer") or (case["kind"] == "ggml" and case["T"] >= 32):
        return {"rel": 1.6e-3}
    return {"rel": 1e-5 if case["kind"] == "ggml" or case["f32"] else 8e-4}


# ---- the same values in float64, by plain torch ----
def _exact_attn(c, s):
    Hq, Hkv, S = s["q"].shape[1], s["k"].shape[1], c["S"]
    out = torch.empty(s["q"].shape, dtype=torch.float64, device="cuda")
    for b in range(c["B"]):
        for h in range(Hq):
            q = s["q"][b, h].double() / math.sqrt(c["D"])
            k, v = (s[n][b, h // (Hq // Hkv)].double() for n in ("k", "v"))
            for r0 in range(0, S, 2048):
                r1 = min(S, r0 + 2048)
                n = r1 if c["causal"] else S
                x = q[r0:r1] @ k[:n].t()
                if c["causal"]:
                    x.masked_fill_(torch.arange(n, device="cuda")[None, :] > torch.arange(r0, r1, device="cuda")[:, None],
                                   -math.inf)
                out[b, h, r0:r1] = torch.softmax(x, dim=-1) @ v[:n]
    if c["kind"] == "gqa":
        out *= torch.sigmoid(s["gate"].double())
    return out


def _exact_gdn(c, s):
    d = {n: x.double() for n, x in s.items() if isinstance(x, torch.Tensor)}
    if c["kind"] == "decode":
        for n in ("q", "k", "v", "a", "b", "g", "beta"):
            if n in d:
                d[n] = d[n][:, None]
    if "a" in d:
        d["g"] = F.softplus(d["a"] + d["dt_bias"], threshold=20.0) * d["A"]
        d["beta"] = torch.sigmoid(d["b"])
        d["q"], d["k"] = (d[n] / d[n].norm(dim=-1, keepdim=True).clamp_min(EPS) for n in ("q", "k"))
    B, T, Hq, Hv = c["B"], c.get("T", 1), c["Hq"], c["Hv"]
    head = torch.arange(Hv, device="cuda") % Hq
    st = d["state"].clone()  # [B, Hv, dv, dk]
    out = torch.empty(B, T, Hv, DK, dtype=torch.float64, device="cuda")
    decay = d["g"].exp()
    for t in range(T):
        k, q = d["k"][:, t][:, head, None, :], d["q"][:, t][:, head, None, :]
        st *= decay[:, t, :, None, None]
        delta = (d["v"][:, t] - (st * k).sum(-1)) * d["beta"][:, t, :, None]
        st += delta[..., None] * k
        out[:, t] = (st * q).sum(-1) / math.sqrt(DK)
    if c["kind"] == "decode":
        out = out[:, 0]
    if c["kind"] == "layer":
        rms = (out.square().mean(-1, keepdim=True) + EPS).sqrt()
        out = out / rms * d["w"] * F.silu(d["z"])
    return out, st


def exact(case, seed):
    """What run() returns for a new state of this seed, in float64."""
    c, d = case, _Draw(seed)
    if c["kind"] in ("attn", "gqa"):
        return _exact_attn(c, _attn_inputs(c, d))
    return _exact_gdn(c, _gdn_inputs(c, d))
