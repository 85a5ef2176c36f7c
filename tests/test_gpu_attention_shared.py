"""The attention kernel with K/V tiles shared through LDS (launches that fill the
chip), at the edges of its query blocks, key tiles and key groups, against the
CPU oracle; tolerances of the bf16 attention tests."""

import pytest
import torch

from oracle import cpu_reference as ref
from rldx_amd import functional as Fn
from rldx_amd import workloads as W
from tolerances import assert_bf16_close

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return torch.device("cuda:0")


def _inputs(B, Hq, Hkv, Sq, Sk, D, bias):
    g = torch.Generator().manual_seed(Hq * 100 + Sq + Sk + D)
    q, k, v = (torch.randn(B, h, s, D, generator=g).to(torch.bfloat16) for h, s in ((Hq, Sq), (Hkv, Sk), (Hkv, Sk)))
    kb = None
    if bias:
        kb = torch.zeros(B, Sk)
        kb[0, ::3] = 0.5 * torch.randn((Sk + 2) // 3, generator=g)  # every tile
        if B > 1:  # whole tiles masked, one raised key, the rest zero
            kb[1, 64:161] = float("-inf")
            kb[1, 7] = 1.5
    return q, k, v, kb


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,D,causal,bias", [
    # 128 queries per workgroup
    (1, 128, 16, 417, 417, 128, True, False),
    (1, 135, 135, 417, 417, 128, True, False),   # heads not divisible over the XCDs
    (1, 251, 251, 513, 513, 64, True, False),
    (1, 128, 16, 513, 300, 128, True, True),     # queries past the last key
    (2, 130, 10, 400, 500, 64, True, True),
    (4, 32, 8, 290, 333, 128, False, True),
    (4, 32, 32, 384, 32, 128, False, False),     # one key tile
    (2, 64, 64, 257, 97, 128, False, True),
    # 64 queries and two key groups per workgroup
    (1, 64, 16, 449, 449, 128, True, False),
    (1, 220, 4, 64, 64, 64, True, False),        # one query block: the second group's only tile is the diagonal
    (2, 30, 10, 449, 449, 128, True, True),
    (2, 32, 8, 400, 33, 128, False, True),       # a second key group with one partial tile
    (1, 64, 64, 400, 31, 64, False, False),      # a second key group without a tile
    (2, 32, 32, 400, 545, 64, False, True),
    (4, 32, 16, 333, 290, 64, False, True),      # head_dim 64: also beyond one round of workgroups
    (1, 280, 4, 64, 64, 64, True, False),
    # either side of the lines for few query rows and partly filled blocks
    (2, 64, 16, 128, 500, 128, False, True), (1, 400, 80, 33, 70, 128, False, True), (4, 110, 10, 64, 160, 128, False, False),
    (13, 32, 8, 32, 600, 128, False, False), (20, 32, 8, 1, 290, 128, False, True), (20, 28, 28, 40, 97, 128, False, False),
    (1, 260, 4, 33, 33, 128, True, False), (1, 220, 4, 64, 64, 128, True, True), (17, 16, 4, 32, 32, 128, True, False),
    (33, 16, 16, 7, 7, 64, True, False), (24, 16, 8, 50, 50, 64, True, True), (20, 16, 16, 64, 64, 64, True, False),
    (7, 16, 4, 280, 280, 128, True, True), (1, 260, 4, 70, 70, 64, True, False), (13, 12, 4, 78, 78, 128, True, False),
    (4, 32, 16, 384, 290, 64, False, True), (8, 28, 28, 79, 97, 64, False, False), (8, 28, 28, 120, 97, 64, False, True),
])
def test_attention_shared_tiles(dev, B, Hq, Hkv, Sq, Sk, D, causal, bias):
    q, k, v, kb = _inputs(B, Hq, Hkv, Sq, Sk, D, bias)
    o = Fn.attention(q.to(dev), k.to(dev), v.to(dev), key_bias=None if kb is None else kb.to(dev), causal=causal)
    r = ref.sdpa(q, ref.repeat_kv(k, Hq // Hkv), ref.repeat_kv(v, Hq // Hkv), key_bias=kb, causal=causal)
    assert_bf16_close(o, r, "attention, shared tiles")


@pytest.mark.parametrize("Hq,Hkv,Sq,D", [(400, 4, 33, 128), (3, 1, 17000, 128)])
def test_shared_tiles_bias_past_the_flags(dev, Hq, Hkv, Sq, D):
    """Tiles after the 2048 that have a flag: their bias decides the result (two key groups, one key group)."""
    Sk = 2048 * 32 + 77
    q, k, v, kb = _inputs(1, Hq, Hkv, Sq, Sk, D, True)
    kb[0, 2048 * 32 - 5:] += 6.0
    kb[0, -9:-3] = float("-inf")
    o = Fn.attention(q.to(dev), k.to(dev), v.to(dev), key_bias=kb.to(dev))
    for h in (0, Hq - 1):
        kv = h // (Hq // Hkv)
        rows = slice(max(0, Sq - 40), Sq)
        r = ref.sdpa(q[:, h:h + 1, rows], k[:, kv:kv + 1], v[:, kv:kv + 1], key_bias=kb)
        assert_bf16_close(o[:, h:h + 1, rows], r, "attention, bias past the flags")


@pytest.mark.parametrize("Hq,Hkv,S,D,causal,part", [
    (400, 400, 128, 128, False, 80), (416, 416, 64, 64, False, 104), (64, 16, 600, 128, False, 4),  # part: heads per unshared launch
    (32, 8, 800, 128, True, 8), (300, 60, 128, 128, True, 40), (32, 8, 2100, 128, True, 4), (40, 8, 1100, 64, True, 10)])
@pytest.mark.parametrize("sharp", [1.0, 2.0])
def test_shared_tiles_lose_no_precision(dev, Hq, Hkv, S, D, causal, part, sharp):
    """The error against float64 is not above that of the kernel without shared tiles
    (the same heads in launches too small to share).  Both round P and O to bf16 and add
    in fp32, so equal errors are equal up to a few values on a rounding edge: 0.1 %."""
    g = torch.Generator(device=dev).manual_seed(S + Hq)
    rnd = lambda h, x=1.0: (x * torch.randn(1, h, S, D, generator=g, device=dev)).to(torch.bfloat16)  # noqa: E731
    q, k, v = rnd(Hq, sharp), rnd(Hkv), rnd(Hkv)
    n = Hq // Hkv
    whole = Fn.attention(q, k, v, causal=causal)
    parts = torch.cat([Fn.attention(q[:, h:h + part], k[:, h // n:(h + part + n - 1) // n], v[:, h // n:(h + part + n - 1) // n],
                                    causal=causal) for h in range(0, Hq, part)], dim=1)
    err, norm = [0.0, 0.0], 0.0
    for h in range(Hq):
        p = q[0, h].double() @ k[0, h // n].double().t() * D ** -0.5
        if causal:
            p.masked_fill_(torch.ones(S, S, dtype=torch.bool, device=dev).triu(1), float("-inf"))
        r = torch.softmax(p, -1) @ v[0, h // n].double()
        norm += float(r.square().sum())
        for i, o in enumerate((whole, parts)):
            err[i] += float((o[0, h].double() - r).square().sum())
    err = [(e / norm) ** 0.5 for e in err]
    assert err[0] <= 1.001 * err[1], f"shared {err[0]:.4e}, unshared {err[1]:.4e}"


@pytest.mark.parametrize("H,S,causal", [(400, 128, False), (64, 600, False), (32, 800, True), (300, 128, True)])
def test_shared_tiles_infinite_scores(dev, H, S, causal):
    """Keys that score -inf are ignored, a query with a score of +inf is NaN as in softmax,
    and the other queries and heads are untouched by it."""
    g = torch.Generator().manual_seed(S)
    q, k, v = (torch.randn(1, H, S, 128, generator=g).to(torch.bfloat16) for _ in range(3))
    clean = Fn.attention(q.to(dev), k.to(dev), v.to(dev), causal=causal)
    q[0, 3] = q[0, 3].abs()
    k[0, 3, 40] = -3e38       # -inf for every query of positive elements ...
    q[0, 3, 90] = -q[0, 3, 90]  # ... and +inf for this one
    o = Fn.attention(q.to(dev), k.to(dev), v.to(dev), causal=causal)
    r = ref.sdpa(q[:, 3:4].float(), k[:, 3:4].float(), v[:, 3:4].float(), causal=causal)
    nan = torch.isnan(r[0, 0]).all(dim=-1)
    assert nan.nonzero().tolist() == [[90]] and bool(torch.isnan(o[0, 3, 90]).all())
    assert_bf16_close(o[0, 3].cpu()[~nan], r[0, 0][~nan], "the other queries")
    rest = [h for h in range(H) if h != 3]
    assert torch.equal(o[:, rest], clean[:, rest])


@pytest.mark.parametrize("B,H,S,D", [(4, 32, 290, 128), (2, 32, 400, 64)])
def test_attention_shared_outputs(dev, B, H, S, D):
    """Rows of 8-byte alignment, and the packed output by row segments: the same bits as contiguous rows."""
    q, k, v, kb = (t.to(dev) for t in _inputs(B, H, H, S, S, D, True))
    kvp = Fn.kv_pack(k, v)
    o = Fn.attention_packed(q, kvp, S, key_bias=kb)
    wide = torch.zeros(B, H, S, D + 4, dtype=torch.bfloat16, device=dev)
    Fn.attention_packed(q, kvp, S, key_bias=kb, out=wide[..., :D])
    assert torch.equal(wide[..., :D], o) and not wide[..., D:].any()
    cut = 96  # rows [0, cut) of every batch entry, then rows [cut + 5, S); the 5 between are not stored
    n1 = S - cut - 5
    packed = Fn.PackedAct.empty(B * (cut + n1), H * D, dev)
    Fn.attention_packed(q, kvp, S, key_bias=kb, out=packed, segments=[(0, cut, 0), (cut + 5, n1, B * cut)])
    rows = o.permute(0, 2, 1, 3).reshape(B, S, H * D)
    want = torch.cat([rows[:, :cut].reshape(-1, H * D), rows[:, cut + 5:].reshape(-1, H * D)])
    assert torch.equal(packed.unpack(), want)


@pytest.mark.parametrize("M,Hq,Hkv,D", [(449, 64, 16, 128), (417, 128, 16, 128), (385, 140, 4, 64), (449, 300, 4, 64), (70, 200, 8, 64), (70, 260, 4, 64),
                                        (280, 112, 28, 128), (20, 640, 32, 128), (64, 400, 40, 64)])
def test_gqa_operator_shared_tiles(dev, M, Hq, Hkv, D):
    """The fused Q norm + RoPE of a wave's own rows."""
    inp = W.gqa_inputs(W.GqaCfg(q_heads=Hq, kv_heads=Hkv, head_dim=D, seq=M, seed=M))
    o = Fn.llm_fused_attention(*(inp[n].to(dev) for n in ("qkv", "q_norm_w", "k_norm_w", "cos")),
                               W.signed_sin(inp["sin"]).to(dev), Hq, Hkv, D)
    r = ref.llm_fused_attention(inp["qkv"], inp["q_norm_w"], inp["k_norm_w"], inp["cos"], inp["sin"], Hq, Hkv, D)
    assert_bf16_close(o, r, "GQA operator, shared tiles")


@pytest.mark.parametrize("lengths,H,D", [
    ((300, 1, 0, 450, 129), 48, 72), ((300, 1, 0, 450, 129), 48, 88), ((300, 1, 0, 450, 129), 48, 64),
    ((300, 1, 0, 450, 129), 48, 120), ((300, 1, 0, 450, 129), 24, 72), ((300, 1, 0, 450, 129), 24, 96),
    ((300, 1, 0, 450, 129), 24, 64), ((65, 448, 64), 48, 128),
    (tuple((37 * i) % 50 for i in range(70)), 8, 80),  # binary-search lookup
    # enough rows, not only blocks, for 128 and 64 queries per workgroup
    ((300, 1, 0, 450, 129), 64, 72), ((300, 1, 0, 450, 129), 64, 120), ((300, 1, 0, 450, 129), 28, 72),
    ((300, 1, 0, 450, 129), 28, 96), ((300, 1, 0, 450, 129), 56, 64), ((65, 448, 64), 48, 96), ((65, 700, 64), 32, 64),
    (tuple((37 * i) % 50 for i in range(70)), 32, 80), (tuple((37 * i) % 50 for i in range(70)), 32, 64),
])
def test_vision_attention_shared_tiles(dev, lengths, H, D):
    inp = W.vit_attention_inputs(W.VitAttnCfg(lengths=lengths, heads=H, head_dim=D, seed=len(lengths) * 100 + D))
    t = {k: (v.to(dev) if torch.is_tensor(v) else v) for k, v in inp.items()}
    o = Fn.vision_attention(t["qkv"], t["rope_cos"], t["rope_sin"], t["cu_seqlens"], t["scaling"], H, D)
    assert_bf16_close(o, ref.vision_attention(**inp), f"vision attention {lengths} H={H} D={D}")


@pytest.mark.parametrize("B,H,S,D", [(1, 4, 77, 64), (2, 3, 1, 128), (4, 32, 290, 128), (2, 32, 400, 64), (1, 2, 2200, 128)])
def test_attention_key_mask(dev, B, H, S, D):
    """A key mask read by the kernel: the bits of the 0 / -inf bias built from it (2200 keys: past the flag scan)."""
    q, k, v, _ = (t if t is None else t.to(dev) for t in _inputs(B, H, H, S, S, D, False))
    kvp = Fn.kv_pack(k, v)
    g = torch.Generator().manual_seed(S)
    mask = (torch.rand(B, S, generator=g) > 0.3).float()
    mask[:, 0] = float("nan")  # not zero: visible
    mask[:, S // 2:S // 2 + 40] = -0.0
    mask = mask.to(dev)
    for m in (mask, mask[:1]):
        bias = torch.where(m == 0, float("-inf"), 0.0).float()
        o = Fn.attention_packed(q, kvp, S, key_mask=m)
        assert torch.equal(o, Fn.attention_packed(q, kvp, S, key_bias=bias))


def test_joint_operator_mask_types(dev):
    """kv_mask of other types, shapes and strides gives the fp32 mask's result."""
    import rldx_amd.ops  # noqa: F401

    H, D, sizes = 4, 64, (40, 18, 9)
    g = torch.Generator().manual_seed(5)
    sa, vl, p = (torch.randn(n, 3 * H * D, generator=g).to(torch.bfloat16).to(dev) for n in (18, 40, 9))
    w = [(1 + 0.1 * torch.randn(D, generator=g)).to(torch.bfloat16).to(dev) for _ in range(6)]
    cs = [torch.randn(n, D // 2, generator=g).to(dev) for n in (18, 18, 9, 9)]
    mask = torch.ones(1, sum(sizes))
    mask[:, 30:34] = 0
    mask[:, -3:] = 0
    mask = mask.to(dev)
    call = lambda m: torch.ops.ds.fused_attention_3way(sa, vl, p, *w, *cs, 18, 40, 9, H, D, m)  # noqa: E731
    want = call(mask)
    wide = torch.zeros(1, 2 * sum(sizes), device=dev)
    wide[:, ::2] = mask
    for m in (mask[0], mask.bool(), mask.long(), mask.bfloat16(), mask.double(), wide[:, ::2]):
        assert torch.equal(call(m), want)
    for bad in (mask[:, 1:], mask.expand(2, -1)):
        with pytest.raises(RuntimeError):
            call(bad)
