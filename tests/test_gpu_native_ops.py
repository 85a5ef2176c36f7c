"""The operators' native dispatch: the bits of the Python implementations in the
forms it takes, the Python implementations' behaviour in the others."""

import gc

import pytest
import torch

from rldx_amd import workloads as W

ops = pytest.importorskip("rldx_amd.ops")
pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


@pytest.fixture(scope="module")
def dev():
    return torch.device("cuda:0")


def _rnd(dev, *shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed + len(shape))).to(BF16).to(dev)


def _calls(dev):
    """(operator, Python implementation, args): every native operator in its common form."""
    H, D = 4, 64
    sa, vl, p = (_rnd(dev, n, 3 * H * D, seed=n) for n in (18, 40, 9))
    w = [1 + 0.1 * _rnd(dev, D, seed=i) for i in range(6)]
    cs = [torch.randn(n, D // 2).to(dev) for n in (18, 18, 9, 9)]
    mask = torch.ones(1, 67, device=dev)
    mask[:, -3:] = 0
    x = _rnd(dev, 58, 3 * H * D + 128)
    g = {k: v.to(dev) for k, v in W.gqa_inputs(W.GqaCfg(q_heads=4, kv_heads=2, seq=70)).items()}
    vi = W.vit_attention_inputs(W.VitAttnCfg(lengths=(33, 50), heads=2))
    mi = W.memory_attention_inputs(W.MemAttnCfg(heads=2))
    t = lambda d, *n: [d[k].to(dev) for k in n]  # noqa: E731
    h, r, ds, nw = (_rnd(dev, 2, 5, 256, seed=i) for i in range(3)), None, None, _rnd(dev, 256)
    h, r, ds = h
    return {
        "gqa": (torch.ops.rldx_backbone.fused_attention, ops.rldx_backbone_fused_attention,
                [g["qkv"], g["q_norm_w"], g["q_norm_w"], g["k_norm_w"], g["k_norm_w"], g["cos"], g["sin"], 4, 2, 128]),
        "vit": (torch.ops.rldx_backbone.vision_attention, ops.rldx_backbone_vision_attention,
                [*t(vi, "qkv", "rope_cos", "rope_sin", "cu_seqlens"), 72 ** -0.5, 2, 72]),
        "mem": (torch.ops.mem.fused_attention, ops.mem_fused_attention, [*t(mi, "qkv", "cos", "signed_sin"), 2, 256, 16]),
        "ds2": (torch.ops.ds.fused_attention_2way, ops.ds_fused_attention_2way,
                [sa, vl, *w[:4], *cs[:2], 18, 40, H, D]),
        "ds3": (torch.ops.ds.fused_attention_3way, ops.ds_fused_attention_3way,
                [sa, vl, p, *w, *cs, 18, 40, 9, H, D, mask]),
        "ds3 unmasked": (torch.ops.ds.fused_attention_3way, ops.ds_fused_attention_3way,
                         [sa[None], vl, p, *w, *cs, 17, 33, 9, H, D]),
        "ss2": (torch.ops.ss.fused_attention_2way, ops.ss_fused_attention_2way, [x, *w[:2], *cs[:2], 18, H, D]),
        "ss3": (torch.ops.ss.fused_attention_3way, ops.ss_fused_attention_3way,
                [x, p, *w[:4], *cs, 58, 18, 9, H, D, mask[0]]),
        "swiglu": (torch.ops.rldx_amd.swiglu, ops.swiglu_op, [_rnd(dev, 3, 7, 48)]),
        "mlp": (torch.ops.ss.fused_mlp_swiglu, ops.ss_fused_mlp_swiglu,
                [_rnd(dev, 19, 256)[:, :128], _rnd(dev, 128, 128), _rnd(dev, 128)]),
        "add2": (torch.ops.rldx_backbone.fused_epilogue_add2_rmsnorm, ops.rldx_backbone_fused_epilogue_add2_rmsnorm,
                 [h, r, nw]),
        "add3": (torch.ops.rldx_backbone.fused_epilogue_add3_rmsnorm, ops.rldx_backbone_fused_epilogue_add3_rmsnorm,
                 [h, r, ds, nw]),
        "mem add2": (torch.ops.mem.fused_epilogue_add2_rmsnorm, ops.mem_fused_epilogue_add2_rmsnorm, [h, r, nw]),
    }


def _same(a, b):
    for x, y in zip(a if isinstance(a, tuple) else (a,), b if isinstance(b, tuple) else (b,)):
        assert x.shape == y.shape and x.dtype == y.dtype and x.stride() == y.stride()
        assert torch.equal(x.view(torch.int16), y.view(torch.int16))


def test_native_library_is_built():
    assert ops._native, "librldx_torch.so missing: build with make -C rldx-1_amd"


def test_native_calls_match_python(dev):
    for name, (op, impl, args) in _calls(dev).items():
        want = impl._init_fn(*args)
        side = torch.cuda.Stream()
        for _ in range(2):  # (the second MLP call finds its packed weight)
            _same(op(*args), want)
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            got = op(*args)
        side.synchronize()
        _same(got, want)


def test_other_forms_reach_python(dev):
    """Strided and differently typed arguments give the same values; wrong ones raise the Python errors."""
    for name, (op, impl, args) in _calls(dev).items():
        spread = [torch.stack([a, a], -1)[..., 0] if torch.is_tensor(a) and a.dim() >= 2 else a for a in args]
        try:
            want = impl._init_fn(*spread)
        except RuntimeError as e:
            with pytest.raises(RuntimeError, match="rldx_amd"):
                op(*spread)
            assert "rldx_amd" in str(e), name
        else:
            _same(op(*spread), want)
        wrong = [a.half() if torch.is_tensor(a) and a.dtype == BF16 else a for a in args]
        with pytest.raises(RuntimeError, match="rldx_amd"):
            op(*wrong)
        with pytest.raises((RuntimeError, NotImplementedError)):
            op(*[a.cpu() if torch.is_tensor(a) else a for a in args])


def test_inputs_with_gradients(dev):
    """As for a custom operator without a backward: the call runs, the backward pass raises."""
    for name, (op, impl, args) in _calls(dev).items():
        args = [a.clone().requires_grad_() if i == 0 else a for i, a in enumerate(args)]
        out = op(*args)
        first = out[0] if isinstance(out, tuple) else out
        assert first.requires_grad, name
        with pytest.raises(RuntimeError, match="no autograd formula"):
            first.float().sum().backward()
        with torch.no_grad():
            _same(op(*args), impl._init_fn(*args))


def test_forward_mode_tangents(dev):
    """An input with a tangent goes to the Python implementation, as one that needs a
    gradient: no formula, so the call raises or its result carries no tangent."""
    from torch.autograd import forward_ad as fw

    for name, (op, impl, args) in _calls(dev).items():
        with fw.dual_level():
            dual = [fw.make_dual(a, torch.ones_like(a)) if i == 0 else a for i, a in enumerate(args)]
            try:
                out = op(*dual)
            except (RuntimeError, NotImplementedError):
                continue
            first = out[0] if isinstance(out, tuple) else out
            assert fw.unpack_dual(first).tangent is None, name


def test_vmap(dev):
    """Mapped over the first argument: each slice's own result, or the refusal of an operator without a
    batching rule."""
    for name, (op, impl, args) in _calls(dev).items():
        pair = torch.stack([args[0], args[0] * 0.5])
        try:
            out = torch.vmap(lambda a: op(a, *args[1:]))(pair)
        except RuntimeError as e:
            assert "batching rule" in str(e) or "vmap" in str(e), name
            continue
        for i in range(2):
            one = impl._init_fn(pair[i].clone(), *args[1:])
            for got, want in zip(out if isinstance(out, tuple) else (out,), one if isinstance(one, tuple) else (one,)):
                assert torch.equal(got[i].view(torch.int16), want.view(torch.int16)), name


def test_mlp_weight_updates_and_lifetime(dev):
    op, impl, (x, w, b) = _calls(dev)["mlp"]
    op(x, w, b)
    w.mul_(0.5)  # a new version
    _same(op(x, w, b), impl._init_fn(x, w.clone(), b))
    w.data = _rnd(dev, 128, 128, seed=9)  # new storage
    _same(op(x, w, b), impl._init_fn(x, w.clone(), b))
    whole = w.data  # the same storage under other shapes: fewer rows, all of them again, transposed
    for data in (whole[:64], whole, whole.t(), whole[64:]):
        w.data = data
        for _ in range(2):
            _same(op(x, w, b[:len(data)].clone()), impl._init_fn(x, data.contiguous().clone(), b[:len(data)].clone()))
    w.data = whole
    # weights that come and go, at addresses used before; nothing packed is kept
    n = len(ops._packed_weights)
    for i in range(5):
        wi = _rnd(dev, 128, 128, seed=20 + i)
        _same(op(x, wi, b), impl._init_fn(x, wi.clone(), b))
        _same(op(x, wi, b), impl._init_fn(x, wi.clone(), b))
        del wi
    gc.collect()
    big = torch.zeros(4096, 4096, dtype=BF16, device=dev)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    op(torch.zeros(4, 4096, dtype=BF16, device=dev), big, torch.zeros(4096, dtype=BF16, device=dev))
    del big
    gc.collect()
    assert torch.cuda.memory_allocated() < before  # the weight and its packed copy are both freed
    assert len(ops._packed_weights) <= n


def _busy(dev, seconds=0.02):
    """Work that keeps the current stream busy for a while (bf16 products of about 0.1 ms each)."""
    a = torch.ones(4096, 4096, dtype=BF16, device=dev)
    for _ in range(int(seconds / 1e-4)):
        a @ a


def test_mlp_weight_packed_on_another_stream(dev):
    """A copy that one stream is still to pack is waited for by the stream that finds it."""
    op, impl, (x, _, b) = _calls(dev)["mlp"]
    one, two = torch.cuda.Stream(), torch.cuda.Stream()
    for trial in range(3):
        w = _rnd(dev, 128, 128, seed=40 + trial)
        want, want2 = (impl._init_fn(x, w.clone(), b, n) for n in (1, 2))
        torch.cuda.synchronize()
        with torch.cuda.stream(one):
            _busy(dev)
            first = op(x, w, b)
        with torch.cuda.stream(two):
            second = op(x, w, b)
            split = op(x, w, b, 2)  # (the Python path)
        torch.cuda.synchronize()
        _same(first, want)
        _same(second, want)
        _same(split, want2)


@pytest.mark.parametrize("split", [1, 2])
def test_mlp_weight_packed_in_a_capture(dev, split):
    """The first call with a weight inside a capture only records its packing: calls before
    the first replay, other graphs and later updates of the weight are right all the same."""
    op, impl, (x, _, b) = _calls(dev)["mlp"]
    x = x.contiguous()
    w = _rnd(dev, 128, 128, seed=50)
    op(x, w.clone(), b, split)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = op(x, w, b, split)
    _same(op(x, w, b, split), impl._init_fn(x, w.clone(), b, split))  # before any replay
    for step in range(4):
        x.copy_(_rnd(dev, 19, 128, seed=60 + step))
        if step == 2:
            w.mul_(0.5)
        graph.replay()
        want = impl._init_fn(x, w.clone(), b, split)
        _same(out, want)
        _same(op(x, w, b, split), want)


def test_mlp_weight_updated_after_a_capture(dev):
    """A graph that reads a weight's packed copy: after an in-place update and one call
    outside the graph its replays see the new weight."""
    op, impl, (x, _, b) = _calls(dev)["mlp"]
    x = x.contiguous()
    w = _rnd(dev, 128, 128, seed=90)
    op(x, w, b)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = op(x, w, b)
    for step in range(4):
        x.copy_(_rnd(dev, 19, 128, seed=91 + step))
        w.mul_(0.75)
        want = impl._init_fn(x, w.clone(), b)
        _same(op(x, w, b), want)
        junk = [torch.full((128 * 128,), 7.0, dtype=BF16, device=dev) for _ in range(4)]  # memory a freed copy would give
        graph.replay()
        _same(out, want)
        del junk


def test_mlp_weight_packed_before_a_capture(dev):
    """A capture takes a copy that is complete, and packs for itself beside one that is not."""
    op, impl, (x, _, b) = _calls(dev)["mlp"]
    x = x.contiguous()
    for busy in (False, True):
        w = _rnd(dev, 128, 128, seed=70 + busy)
        side = torch.cuda.Stream()
        torch.cuda.synchronize()
        graph, capture = torch.cuda.CUDAGraph(), torch.cuda.Stream()
        op(x, _rnd(dev, 128, 128, seed=80), b)
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            if busy:
                _busy(dev)
            op(x, w, b)
        if not busy:
            torch.cuda.synchronize()
        with torch.cuda.stream(capture):
            graph.capture_begin()
            out = op(x, w, b)
            graph.capture_end()
            graph.replay()
        capture.synchronize()
        _same(out.clone(), impl._init_fn(x, w.clone(), b))
        torch.cuda.synchronize()
