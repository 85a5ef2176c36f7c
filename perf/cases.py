"""The calls a user of the framework makes, as measurable cases.

Every case goes through a public entry point (a `torch.library` operator of
`rldx_amd.ops`, or one of the graph executors) at sizes a robot policy meets:
the release configuration of the RLDX-1 action head, the synthetic 608-token
action step, and the single operators of the VLM backbone, vision tower,
cognition memory and MSAT blocks from their smallest to their largest sizes.

`exact` evaluates the same inputs in float64 with plain torch.
"""

from __future__ import annotations

import math
import os
import sys

import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.getcwd(), "rldx-1_amd"))

import rldx_amd.ops  # noqa: E402,F401  (registers the operators)
from rldx_amd import msat_step as MS  # noqa: E402
from rldx_amd import rldx_msat as RM  # noqa: E402

BF16, F32, F64 = torch.bfloat16, torch.float32, torch.float64
DEV = "cuda"


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # One whole action inference of the RLDX-1 release: 64 cognition tokens, 17 state / action tokens,
        # 4 denoising steps, batch 1: the control loop's call on a robot.
        {"name": "head_release", "kind": "head", "n_vl": 64},
        # The synthetic 16-block triple-stream action step (512 cognition, 64 action, 32 physics tokens),
        # the benchmark's default workload.
        {"name": "step_608", "kind": "step", "blocks": 16, "n_vl": 512, "n_sa": 64, "n_p": 32},
        # VLM decoder attention of one layer: the backbone's own prompt of one camera image ...
        {"name": "gqa_169", "kind": "gqa", "seq": 169, "q_heads": 32, "kv_heads": 8},
        # ... a prompt with several camera images (7 query heads per KV head) ...
        {"name": "gqa_1280", "kind": "gqa", "seq": 1280, "q_heads": 28, "kv_heads": 4},
        # ... and a long one: video history from several cameras.
        {"name": "gqa_4096", "kind": "gqa", "seq": 4096, "q_heads": 32, "kv_heads": 8},
        # Vision tower attention of one layer: two 224-pixel camera images ...
        {"name": "vit_2x196", "kind": "vit", "lengths": "196,196", "heads": 16, "head_dim": 72},
        # ... and a ragged batch of larger images.
        {"name": "vit_ragged", "kind": "vit", "lengths": "1024,1600,484,2304,196", "heads": 16, "head_dim": 72},
        # MSAT joint attention operator over cognition, action and physics tokens, 8 physics tokens padded.
        {"name": "joint_608", "kind": "joint", "n_vl": 512, "n_sa": 64, "n_p": 32, "pad": 8, "heads": 16,
         "head_dim": 128},
        # Fused SwiGLU MLP of a single-stream block at the release shape ...
        {"name": "mlp_82", "kind": "mlp", "tokens": 82, "k": 1536, "n_half": 6144},
        # ... and over many tokens (a batch of robots, a prefill).
        {"name": "mlp_2048", "kind": "mlp", "tokens": 2048, "k": 4096, "n_half": 11008},
        # Cognition memory attention: 4 timesteps of 16 tokens, the smallest call.
        {"name": "memory_64", "kind": "memory", "length": 4, "block": 16, "heads": 16, "head_dim": 256},
        # Residual add + RMSNorm between the VLM's layers, prefill.
        {"name": "add_norm_1280", "kind": "norm", "rows": 1280, "dim": 4096},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["head", "step", "gqa", "gqa", "vit", "vit", "joint", "joint", "mlp", "mlp", "memory", "norm"])
    if kind == "head":
        return {"kind": kind, "n_vl": rng.randint(16, 64)}
    if kind == "step":
        return {"kind": kind, "blocks": rng.randint(2, 12), "n_vl": 32 * rng.randint(2, 16),
                "n_sa": 32 * rng.randint(1, 2), "n_p": 32}
    if kind == "gqa":
        hq, hkv = rng.choice([(32, 8), (28, 4), (16, 8)])
        return {"kind": kind, "seq": _log(rng, 64, 4096), "q_heads": hq, "kv_heads": hkv}
    if kind == "vit":
        lengths = [_log(rng, 64, 2304) for _ in range(rng.randint(1, 5))]
        return {"kind": kind, "lengths": ",".join(map(str, lengths)), "heads": 16, "head_dim": rng.choice([64, 72, 80])}
    if kind == "joint":
        heads, dim = rng.choice([(16, 128), (24, 64), (12, 128)])
        n_p = rng.randint(8, 48)
        return {"kind": kind, "n_vl": _log(rng, 48, 1024), "n_sa": rng.randint(17, 96), "n_p": n_p,
                "pad": rng.randint(0, n_p - 1), "heads": heads, "head_dim": dim}
    if kind == "mlp":
        k, n_half = rng.choice([(1536, 6144), (1536, 4096), (2048, 6144), (4096, 11008)])
        return {"kind": kind, "tokens": _log(rng, 18, 2048), "k": k, "n_half": n_half}
    if kind == "memory":
        return {"kind": kind, "length": _log(rng, 2, 64), "block": 16, "heads": 16, "head_dim": rng.choice([128, 256])}
    return {"kind": "norm", "rows": _log(rng, 16, 8192), "dim": rng.choice([2048, 3584, 4096])}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
class _Rand:
    """Seeded normal tensors on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(seed)

    def __call__(self, *shape, std=1.0, mean=0.0):
        return (mean + std * torch.randn(*shape, generator=self.g, device=DEV, dtype=F32)).to(BF16)


def _half_rope(seq, dim, theta):
    """Rotate-half tables [seq, dim] in float32."""
    inv = 1.0 / theta ** (torch.arange(0, dim, 2, device=DEV, dtype=F32) / dim)
    f = torch.outer(torch.arange(seq, device=DEV, dtype=F32), inv)
    f = torch.cat([f, f], dim=-1)
    return f.cos(), f.sin()


def _signed(sin):
    h = sin.shape[-1] // 2
    return torch.cat([-sin[:, :h], sin[:, h:]], dim=-1).contiguous()


def _pair_rope(rows, dim, axis0, theta=10000.0):
    """Two-axis interleaved tables [rows, dim / 2]: dim / 4 on axis 0, 3 dim / 4 on axis 1."""
    parts = []
    for ad, pos in ((dim // 4, torch.full((rows,), float(axis0), device=DEV)),
                    (dim - dim // 4, torch.arange(rows, device=DEV, dtype=F32))):
        parts.append(torch.outer(pos, 1.0 / theta ** (torch.arange(0, ad, 2, device=DEV, dtype=F32) / ad)))
    f = torch.cat(parts, dim=-1)
    return f.cos().contiguous(), f.sin().contiguous()


def _head_cfgs(c):
    return RM.RldxMsatCfg(n_vl=c["n_vl"]), RM.RldxHeadCfg(num_embodiments=4)


def _head_data(c, seed):
    """Weights under the reference's names, and one observation."""
    mc, hc = _head_cfgs(c)
    r = _Rand(seed)
    sd = {k: r(*s, std=0.02, mean=1.0 if "norm" in k else 0.0) for k, s in mc.param_shapes().items()}
    E, d, hs, A = hc.num_embodiments, mc.sa_dim, hc.hidden_size, hc.action_dim
    head = {}
    for name, (i, o) in {"state_encoder.layer1": (hc.state_dim, hs), "state_encoder.layer2": (hs, d),
                         "action_encoder.W1": (A, d), "action_encoder.W2": (2 * d, d), "action_encoder.W3": (d, d),
                         "action_decoder.layer1": (mc.output_dim, hs), "action_decoder.layer2": (hs, A)}.items():
        head[name + ".W"], head[name + ".b"] = r(E, i, o, std=0.02), r(E, o, std=0.02)
    head["position_embedding.weight"] = r(hc.action_horizon, d, std=0.02)
    head["static_tembs"] = r(hc.steps, 1, mc.inner, std=0.5)
    head["static_time_tokens"] = r(hc.steps, 1, mc.num_temb_tokens, d, std=0.5)
    obs = {"vl": r(1, mc.n_vl, mc.vl_dim), "state": r(1, 1, hc.state_dim), "x0": r(1, hc.action_horizon, A)}
    return mc, hc, sd, head, obs


def _step_cfg(c, seed):
    return MS.MsatStepCfg(blocks=c["blocks"], n_vl=c["n_vl"], n_sa=c["n_sa"], n_p=c["n_p"], seed=seed)


def _gqa_data(c, seed):
    r, D = _Rand(seed), 128
    cos, sin = _half_rope(c["seq"], D, 1e6)
    return {"qkv": r(c["seq"], (c["q_heads"] + 2 * c["kv_heads"]) * D), "qw": r(D, std=0.02, mean=1.0),
            "kw": r(D, std=0.02, mean=1.0), "cos": cos.to(BF16), "sin": _signed(sin.to(BF16))}


def _vit_data(c, seed):
    r = _Rand(seed)
    lens, D = [int(x) for x in c["lengths"].split(",")], c["head_dim"]
    # row-major patch coordinates, half of the rotary pairs per axis
    pos = torch.cat([torch.stack((torch.arange(n) // math.isqrt(n), torch.arange(n) % math.isqrt(n)), -1)
                     for n in lens]).to(DEV, F32)
    inv = 1.0 / 10000.0 ** (torch.arange(0, D // 2, 2, device=DEV, dtype=F32) / (D // 2))
    f = (pos[:, :, None] * inv).flatten(1)
    f = torch.cat([f, f], dim=-1)
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32).to(DEV)
    return {"qkv": r(sum(lens), 3 * c["heads"] * D), "cos": f.cos().contiguous(), "sin": _signed(f.sin()), "cu": cu,
            "lens": lens}


def _joint_data(c, seed):
    r, H, D = _Rand(seed), c["heads"], c["head_dim"]
    d = {s: r(n, 3 * H * D) for s, n in (("vl", c["n_vl"]), ("sa", c["n_sa"]), ("p", c["n_p"]))}
    for s in ("vl", "sa", "p"):
        d["q_" + s], d["k_" + s] = r(D, std=0.02, mean=1.0), r(D, std=0.02, mean=1.0)
    d["sa_cos"], d["sa_sin"] = _pair_rope(c["n_sa"], D, 0)
    d["p_cos"], d["p_sin"] = _pair_rope(c["n_p"], D, 1)
    n = c["n_vl"] + c["n_sa"] + c["n_p"]
    d["mask"] = torch.ones(1, n, device=DEV)
    d["mask"][:, n - c["pad"]:] = 0
    return d


def _mlp_data(c, seed):
    r = _Rand(seed)
    return {"x": r(c["tokens"], c["k"]), "w": r(2 * c["n_half"], c["k"], std=0.02), "b": r(2 * c["n_half"], std=0.02)}


def _memory_data(c, seed):
    m, D = c["length"] * c["block"], c["head_dim"]
    cos, sin = _half_rope(c["length"], D, 10000.0)  # one position per timestep
    cos, sin = (t.repeat_interleave(c["block"], 0).to(BF16) for t in (cos, sin))
    return {"qkv": _Rand(seed)(m, 3 * c["heads"] * D), "cos": cos.contiguous(), "sin": _signed(sin)}


def _norm_data(c, seed):
    r = _Rand(seed)
    return {"x": r(c["rows"], c["dim"]), "res": r(c["rows"], c["dim"]), "w": r(c["dim"], std=0.1, mean=1.0)}


_DATA = {"gqa": _gqa_data, "vit": _vit_data, "joint": _joint_data, "mlp": _mlp_data, "memory": _memory_data,
         "norm": _norm_data}


# ---------------------------------------------------------------------------
# the calls
# ---------------------------------------------------------------------------
def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "head":
        mc, hc, sd, head_sd, obs = _head_data(c, seed)
        head = RM.RldxActionHead(RM.RldxMsat(sd, mc, DEV), head_sd, hc)
        head.set_embodiment(1)
        _load_obs(head, obs)
        head.capture()
        return {"c": c, "head": head, "obs": obs}
    if kind == "step":
        cfg = _step_cfg(c, seed)
        step = MS.MsatActionStep(cfg, MS.make_weights(cfg, DEV), MS.make_inputs(cfg, DEV))
        step.capture()
        return {"c": c, "step": step}
    return {"c": c, "d": _DATA[kind](c, seed)}


def _load_obs(head, obs):
    head.vl.copy_(obs["vl"])
    head.state.copy_(obs["state"])
    head.x0.copy_(obs["x0"])


def run(state):
    c = state["c"]
    kind = c["kind"]
    if kind == "head":  # a new observation into the head's buffers, then the captured call
        _load_obs(state["head"], state["obs"])
        return state["head"].replay()
    if kind == "step":
        return state["step"].replay()
    d = state["d"]
    if kind == "gqa":
        return torch.ops.rldx_backbone.fused_attention(d["qkv"], d["qw"], d["qw"], d["kw"], d["kw"], d["cos"],
                                                       d["sin"], c["q_heads"], c["kv_heads"], 128)
    if kind == "vit":
        D = c["head_dim"]
        return torch.ops.rldx_backbone.vision_attention(d["qkv"], d["cos"], d["sin"], d["cu"], D ** -0.5, c["heads"], D)
    if kind == "joint":
        return torch.ops.ds.fused_attention_3way(
            d["sa"], d["vl"], d["p"], d["q_sa"], d["k_sa"], d["q_vl"], d["k_vl"], d["q_p"], d["k_p"], d["sa_cos"],
            d["sa_sin"], d["p_cos"], d["p_sin"], c["n_sa"], c["n_vl"], c["n_p"], c["heads"], c["head_dim"], d["mask"])
    if kind == "mlp":
        return torch.ops.ss.fused_mlp_swiglu(d["x"], d["w"], d["b"])
    if kind == "memory":
        return torch.ops.mem.fused_attention(d["qkv"], d["cos"], d["sin"], c["heads"], c["head_dim"], c["block"])
    return torch.ops.rldx_backbone.fused_epilogue_add2_rmsnorm(d["x"], d["res"], d["w"])


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    c, kind = case, case["kind"]
    if kind == "head":  # the weights of every step: more than any cache holds from one step to the next
        mc, hc = _head_cfgs(c)
        shapes = mc.param_shapes()
        n = c["n_vl"] + mc.n_sa
        mats = {k: s for k, s in shapes.items() if len(s) == 2 and not k.startswith("proj_out_1")}
        flops = 0
        for k, (o, i) in mats.items():
            rows = c["n_vl"] if ".vl_" in k or k.startswith("vl_") else mc.n_sa if ".sa_" in k else n
            flops += 2 * rows * o * i
        flops += (mc.ds_blocks + mc.ss_blocks) * 4 * mc.inner * n * n
        return {"bytes": hc.steps * 2 * sum(math.prod(s) for s in shapes.values()), "flops": hc.steps * flops}
    if kind == "step":
        cfg = _step_cfg(c, 0)
        return {"bytes": cfg.steps * cfg.weight_bytes(), "flops": cfg.flops_per_step()}
    if kind == "gqa":
        s, hq, hkv, D = c["seq"], c["q_heads"], c["kv_heads"], 128
        return {"bytes": 2 * s * D * (2 * hq + 2 * hkv + 2), "flops": 2 * hq * D * s * (s + 1)}
    if kind == "vit":
        lens, w = [int(x) for x in c["lengths"].split(",")], c["heads"] * c["head_dim"]
        return {"bytes": sum(lens) * (8 * w + 8 * c["head_dim"]), "flops": 4 * w * sum(n * n for n in lens)}
    if kind == "joint":
        n, w = c["n_vl"] + c["n_sa"] + c["n_p"], c["heads"] * c["head_dim"]
        return {"bytes": 8 * n * w, "flops": 4 * w * n * (n - c["pad"])}
    if kind == "mlp":
        m, k, h = c["tokens"], c["k"], c["n_half"]
        return {"bytes": 2 * (m * k + 2 * h * k + 2 * h + m * h), "flops": 4 * m * k * h}
    if kind == "memory":
        m, b, w = c["length"] * c["block"], c["block"], c["heads"] * c["head_dim"]
        pairs = b * b * c["length"] * (c["length"] + 1) // 2
        return {"bytes": 8 * m * w + 4 * m * c["head_dim"], "flops": 4 * w * pairs}
    return {"bytes": 8 * c["rows"] * c["dim"] + 2 * c["dim"], "flops": 8 * c["rows"] * c["dim"]}


def tolerance(case):
    """bf16 in and out, float32 sums: about four times the distance measured to float64, 2e-3 .. 4.3e-3
    (2-norm) for the operators and 5e-3 / 7e-3 for the whole calls, where a rounding travels through
    48 or 64 block applications."""
    if case["kind"] in ("head", "step"):
        return {"rel": 0.03}
    return {"rel": 0.012, "max": 0.08}


# ---------------------------------------------------------------------------
# the same in float64
# ---------------------------------------------------------------------------
def _rms(x, w, eps=1e-6):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w


def _rotate(x, cos, signed_sin):
    h = x.shape[-1] // 2
    return x * cos + torch.cat([x[..., h:], x[..., :h]], -1) * signed_sin


def _rotate_pairs(x, cos, sin):
    re, im = x[..., 0::2], x[..., 1::2]
    return torch.stack([re * cos - im * sin, re * sin + im * cos], -1).flatten(-2)


def _attend(q, k, v, bias=None):
    """[H, N, D] operands, head by head."""
    out = torch.empty_like(q)
    for h in range(q.shape[0]):
        s = q[h] @ k[h].t() / math.sqrt(q.shape[-1])
        out[h] = torch.softmax(s if bias is None else s + bias, -1) @ v[h]
    return out


def _heads(x, H):
    return x.reshape(x.shape[0], H, -1).transpose(0, 1)


def _flat(x):
    return x.transpose(0, 1).reshape(x.shape[1], -1)


def _ln(x, eps=1e-6):
    return F.layer_norm(x, x.shape[-1:], eps=eps)


def _silu_mul(x):
    g, u = x.chunk(2, -1)
    return F.silu(g) * u


def _joint(streams, H, bias=None):
    """streams: (qkv rows, q norm, k norm, cos or None, sin) in joint order -> [N, H D]."""
    qs, ks, vs = [], [], []
    for qkv, qw, kw, cos, sin in streams:
        q, k, v = (_heads(t, H) for t in qkv.chunk(3, -1))
        q, k = _rms(q, qw), _rms(k, kw)
        if cos is not None:
            q, k = _rotate_pairs(q, cos, sin), _rotate_pairs(k, cos, sin)
        qs.append(q)
        ks.append(k)
        vs.append(v)
    return _flat(_attend(torch.cat(qs, 1), torch.cat(ks, 1), torch.cat(vs, 1), bias))


def _exact_msat(mc, sd, sa, vl, temb, token):
    H = mc.heads
    lin = lambda x, n: F.linear(x, sd[n + ".weight"].to(F64), sd[n + ".bias"].to(F64))  # noqa: E731
    wt = lambda n: sd[n + ".weight"].to(F64)  # noqa: E731

    def tables(pos):  # a model in bf16 keeps the cosines in bf16 and loses the sines
        f = []
        for ad, p in ((mc.head_dim // 4, torch.zeros_like(pos)), (mc.head_dim - mc.head_dim // 4, pos)):
            f.append(torch.outer(p.float(), 1.0 / mc.rope_theta ** (torch.arange(0, ad, 2, device=DEV).float() / ad)))
        cos = torch.cat(f, -1).cos().to(BF16).to(F64)
        return cos, torch.zeros_like(cos)

    nt, nv = mc.num_temb_tokens, vl.shape[0]
    sa = torch.cat([token, sa])
    ns = sa.shape[0]
    low = tables(torch.arange(ns, device=DEV))
    up = tables(torch.cat([torch.arange(nt, device=DEV), torch.arange(nt + 1, ns + 1, device=DEV)]))
    for b in range(mc.ds_blocks):
        p = f"double_blocks.{b}."
        o = _joint([(lin(_ln(vl), p + "vl_qkv"), wt(p + "q_norm_vl"), wt(p + "k_norm_vl"), None, None),
                    (lin(_ln(sa), p + "sa_qkv"), wt(p + "q_norm_sa"), wt(p + "k_norm_sa"), *low)], H)
        sa, vl = sa + lin(o[nv:], p + "sa_proj"), vl + lin(o[:nv], p + "vl_proj")
        sa = sa + lin(_silu_mul(lin(_ln(sa), p + "sa_mlp.w12")), p + "sa_mlp.w3")
        vl = vl + lin(_silu_mul(lin(_ln(vl), p + "vl_mlp.w12")), p + "vl_mlp.w3")
    x = torch.cat([lin(vl, "vl_proj_to_sa"), sa])
    for b in range(mc.ss_blocks):
        p = f"single_blocks.{b}."
        h = lin(_ln(x), p + "linear1")
        qkv, mlp = h[:, :3 * mc.inner], h[:, 3 * mc.inner:]
        qw, kw = wt(p + "q_norm"), wt(p + "k_norm")
        o = _joint([(qkv[:nv], qw, kw, None, None), (qkv[nv:], qw, kw, *up)], H)
        x = x + lin(torch.cat([o, lin(_silu_mul(mlp), p + "mlp_proj")], -1), p + "linear2")
    shift, scale = lin(F.silu(temb), "proj_out_1").chunk(2, -1)
    return lin(_ln(x[nv + nt:]) * (1 + scale) + shift, "proj_out_2")


def _exact_head(c, seed):
    mc, hc, sd, head, obs = _head_data(c, seed)
    cat = lambda x, n: x @ head[n + ".W"][1].to(F64) + head[n + ".b"][1].to(F64)  # noqa: E731
    obs = {k: v[0].to(F64) for k, v in obs.items()}
    st = cat(torch.relu(cat(obs["state"], "state_encoder.layer1")), "state_encoder.layer2")
    act, width = obs["x0"].clone(), mc.sa_dim
    ex = torch.exp(-torch.arange(width // 2, device=DEV).float() * (math.log(10000.0) / (width // 2)))
    for i in range(hc.steps):
        f = torch.full((act.shape[0], 1), i / hc.steps, device=DEV) * ex
        tau = torch.cat([f.sin(), f.cos()], -1).to(BF16).to(F64)
        h = cat(torch.cat([cat(act, "action_encoder.W1"), tau], -1), "action_encoder.W2")
        feat = cat(F.silu(h), "action_encoder.W3") + head["position_embedding.weight"].to(F64)
        out = _exact_msat(mc, sd, torch.cat([st, feat]), obs["vl"], head["static_tembs"][i].to(F64),
                          head["static_time_tokens"][i, 0].to(F64))
        v = cat(torch.relu(cat(out, "action_decoder.layer1")), "action_decoder.layer2")[-act.shape[0]:]
        act = act + v / hc.steps
    return act[None]


def _exact_step(c, seed):
    cfg = _step_cfg(c, seed)
    w, inp = MS.make_weights(cfg, DEV), MS.make_inputs(cfg, DEV)
    lin = lambda x, n, L: F.linear(x, w[n + ".w"][L].to(F64), w[n + ".b"][L].to(F64))  # noqa: E731
    i64 = {k: v.to(F64) for k, v in inp.items()}
    tab = {"vl": (None, None), "sa": (i64["sa_cos"], i64["sa_sin"]), "p": (i64["p_cos"], i64["p_sin"])}
    cuts = [cfg.n_vl, cfg.n_sa, cfg.n_p]
    act = i64["x0"].clone()
    for t in range(cfg.steps):
        sa = F.linear(act, w["act_in.w"].to(F64), w["act_in.b"].to(F64)) + i64["temb"][t] + i64["pos"]
        xs = {"vl": i64["vl"], "sa": sa, "p": i64["p"]}
        for L in range(cfg.blocks):
            o = _joint([(lin(_ln(xs[s]), s + ".qkv", L), w[s + ".q_norm"][L].to(F64), w[s + ".k_norm"][L].to(F64),
                         *tab[s]) for s in ("vl", "sa", "p")], cfg.heads, i64["key_bias"])
            for s, part in zip(("vl", "sa", "p"), o.split(cuts)):
                x = xs[s] + lin(part, s + ".proj", L)
                xs[s] = x + lin(_silu_mul(lin(_ln(x), s + ".w12", L)), s + ".w3", L)
        act = act + F.linear(_ln(xs["sa"]), w["act_out.w"].to(F64), w["act_out.b"].to(F64)) / cfg.steps
    return act


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "head":
        return _exact_head(c, seed)
    if kind == "step":
        return _exact_step(c, seed)
    raw = _DATA[kind](c, seed)
    d = {k: v.to(F64) if torch.is_tensor(v) and v.is_floating_point() else v for k, v in raw.items()}
    if kind == "gqa":
        s, hq, hkv = c["seq"], c["q_heads"], c["kv_heads"]
        q, k, v = d["qkv"].split([hq * 128, hkv * 128, hkv * 128], -1)
        q = _rotate(_rms(_heads(q, hq), d["qw"]), d["cos"], d["sin"])
        k = _rotate(_rms(_heads(k, hkv), d["kw"]), d["cos"], d["sin"]).repeat_interleave(hq // hkv, 0)
        v = _heads(v, hkv).repeat_interleave(hq // hkv, 0)
        return _flat(_attend(q, k, v, torch.full((s, s), -math.inf, device=DEV, dtype=F64).triu(1)))
    if kind == "vit":
        q, k, v = (_heads(t, c["heads"]) for t in d["qkv"].chunk(3, -1))
        q, k = _rotate(q, d["cos"], d["sin"]), _rotate(k, d["cos"], d["sin"])
        parts = zip(*(t.split(d["lens"], 1) for t in (q, k, v)))
        return torch.cat([_flat(_attend(*p)) for p in parts])
    if kind == "joint":
        bias = torch.where(d["mask"][0] == 0, -math.inf, 0.0)
        o = _joint([(d["vl"], d["q_vl"], d["k_vl"], None, None), (d["sa"], d["q_sa"], d["k_sa"], d["sa_cos"], d["sa_sin"]),
                    (d["p"], d["q_p"], d["k_p"], d["p_cos"], d["p_sin"])], c["heads"], bias)
        return o[None]
    if kind == "mlp":
        return _silu_mul(F.linear(d["x"], d["w"], d["b"]))
    if kind == "memory":
        q, k, v = (_heads(t, c["heads"]) for t in d["qkv"].chunk(3, -1))
        q, k = _rotate(q, d["cos"], d["sin"]), _rotate(k, d["cos"], d["sin"])
        at = torch.arange(q.shape[1], device=DEV) // c["block"]
        bias = torch.where(at[None, :] <= at[:, None], 0.0, -math.inf).to(F64)
        return _flat(_attend(q, k, v, bias))
    x = d["x"] + d["res"]
    return (x, _rms(x, d["w"]))
