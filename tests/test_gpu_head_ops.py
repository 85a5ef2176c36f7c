"""GPU tests of the action head's small launches: the strided row copies, the
gather of stacked parameters and the output modulation with its packing, all bit
for bit those of the eager chain."""

import pytest
import torch
import torch.nn.functional as F

from rldx_amd import functional as Fn

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def rnd(*shape, seed=0, dtype=BF16):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(dtype).cuda()


@pytest.mark.parametrize("batch", [1, 3])
def test_copy_rows_many(batch):
    """1 unit, one workgroup exactly (1024 units), one past it, strided and broadcast
    sources; nothing outside the destination rows changes.  A row of 12 bytes and a
    source of another type take torch's copy."""
    srcs = [rnd(batch, 1, 8, seed=1), rnd(batch, 16, 1024, seed=2)[:, ::2, :512], rnd(1, 41, 200, seed=3).expand(batch, 41, 200),
            rnd(batch, 18, 1536, seed=4)]
    buf = [torch.full((batch, s.shape[1] + 2, s.shape[2] + 8), 7.0, dtype=BF16, device="cuda") for s in srcs]
    Fn.copy_rows_many([(s, b[:, 1:-1, :-8]) for s, b in zip(srcs, buf)])
    for s, b in zip(srcs, buf):
        assert torch.equal(b[:, 1:-1, :-8], s)
        assert bool((b[:, 0] == 7).all() and (b[:, -1] == 7).all() and (b[:, :, -8:] == 7).all())
    odd = [(rnd(batch, 5, 6), torch.zeros(batch, 5, 6, dtype=BF16, device="cuda")),
           (rnd(batch, 5, 16, dtype=torch.float32), torch.zeros(batch, 5, 16, dtype=BF16, device="cuda"))]
    Fn.copy_rows_many(odd)
    assert all(torch.equal(d, s.to(BF16)) for s, d in odd)
    with pytest.raises(Exception):
        Fn.copy_rows_many([(srcs[0], buf[1])])


@pytest.mark.parametrize("ids", [[2], [0, 4, 4]])
def test_gather_slabs(ids):
    """Slabs of one unit, of 1024 units and of one more, and in 2-byte units: one of 14
    bytes, one of 1025 units, one that is not 16-byte aligned; a strided stack takes
    torch's index_select.  An id outside the stacks makes its slabs NaN and leaves the
    other robots' right, whatever was there before."""
    idx = torch.tensor(ids, device="cuda")
    stacks = [rnd(5, 8, seed=1), rnd(5, 64, 128, seed=2), rnd(5, 8200, seed=3), rnd(5, 7, seed=4), rnd(5, 1025, seed=5),
              rnd(1 + 5 * 16, seed=6)[1:].view(5, 16), rnd(5, 6, dtype=torch.float32, seed=7), rnd(10, 40, seed=8)[::2]]
    outs = [torch.zeros(len(ids), 1, *s.shape[1:], dtype=s.dtype, device="cuda") for s in stacks]
    Fn.gather_slabs(list(zip(stacks, outs)), idx)
    for s, o in zip(stacks, outs):
        assert torch.equal(o[:, 0], s[idx])
    for bad in (5, -1, 2**40):
        mixed = idx.clone()
        mixed[0] = bad
        Fn.gather_slabs(list(zip(stacks, outs))[:-1], mixed)
        for s, o in zip(stacks[:-1], outs):
            assert bool(torch.isnan(o[0]).all()) and torch.equal(o[1:, 0], s[idx[1:]])


@pytest.mark.parametrize("batch,rows,d", [(1, 1, 16), (1, 17, 1536), (3, 31, 1040), (2, 33, 2064), (1, 3, 8192), (4, 17, 1536)])
def test_adaln_pack(batch, rows, d):
    """The bits of the eager chain (torch's LayerNorm, then three rounded steps), at rows
    across 32-row blocks and partial workgroups, for values over the range of bf16."""
    x = rnd(batch, rows + 2, d, seed=d)[:, 1:-1] * 3 + 1
    x[:, -1] *= 1e-3
    shift, scale = rnd(batch, 2 * d, seed=d + 1).chunk(2, dim=1)
    scale[:, ::7] *= 100
    m = batch * rows
    for s in (scale, scale.float()):  # (a scale of another type takes the eager chain)
        want = (F.layer_norm(x, (d,), eps=1e-6) * (1 + s[:, None]) + shift[:, None]).to(BF16).view(m, d)
        out = Fn.PackedAct.empty(m, d, "cuda")
        Fn.adaln_pack(x, shift, s, out)
        assert torch.equal(out.unpack().view(torch.int16), want.view(torch.int16))
