"""Host tests of the packed-weight cache of ss::fused_mlp_swiglu (rldx_amd/ops.py and its
copy in csrc/torch_ops.cpp): a packed copy serves a weight only as it was when packed."""

import os
import subprocess
import sys
from pathlib import Path

import pytest
import torch

from rldx_amd import functional as Fn

ops = pytest.importorskip("rldx_amd.ops")
BF16 = torch.bfloat16


@pytest.fixture
def packs(monkeypatch):
    """pack_weight without a GPU: the packed copy is a copy; the list holds the weights' shapes as packed."""
    seen = []

    def pack(w, swiglu_pairs=False, row_sums=True, out=None):
        seen.append(tuple(w.shape))
        data = torch.empty(w.numel(), dtype=BF16) if out is None else out
        return Fn.PackedWeight(data.copy_(w.reshape(-1)), *w.shape, swiglu_pairs)

    monkeypatch.setattr(Fn, "pack_weight", pack)
    return seen


def _w(*shape):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(sum(shape))).to(BF16)


@pytest.mark.parametrize("change", [lambda t: t[:64], lambda t: t.t(), lambda t: t[:, :64], lambda t: t.view(256, 64),
                                    lambda t: t.view(64, 2, 128)[:, 0]], ids=["rows", "transposed", "columns", "view", "strided"])
def test_storage_of_another_shape_is_packed_again(packs, change):
    """`w.data = view of the same storage` keeps the tensor, its version and its data
    pointer; only the shape and the strides tell it from the packed one."""
    w = _w(128, 128)
    before = ops._packed_weight(w, True)
    assert ops._packed_weight(w, True) is before and len(packs) == 1
    state = (w._version, w.data_ptr())
    w.data = change(w.data)
    assert (w._version, w.data_ptr()) == state
    after = ops._packed_weight(w, True)
    assert after is not before and (after.n, after.k) == tuple(w.shape)
    assert torch.equal(after.data.view(w.shape), w) and len(packs) == 2


def test_update_in_place_is_packed_over_the_old_copy(packs):
    """A captured graph holds the copy's address: it must stay the copy of this weight."""
    w = _w(128, 128)
    before = ops._packed_weight(w, True)
    address = before.data.data_ptr()
    w.mul_(0.5)
    after = ops._packed_weight(w, True)
    assert after.data.data_ptr() == address and len(packs) == 2
    assert torch.equal(after.data.view(w.shape), w)
    w.data = w.data.clone()  # other storage, to which nobody ordered the old copy's readers
    assert ops._packed_weight(w, True).data.data_ptr() != address and len(packs) == 3


def test_storage_grown_in_place_is_packed_again(packs):
    base = _w(256, 128)
    w = base[:128].detach()
    small = ops._packed_weight(w, True)
    w.data = base
    grown = ops._packed_weight(w, True)
    assert (small.n, grown.n) == (128, 256) and packs == [(128, 128), (256, 128)]


@pytest.mark.skipif(not ops._native, reason="librldx_torch.so was not built")
def test_native_copy_serves_the_packed_shape_only():
    native = torch.ops.rldx_native
    w, packed = _w(128, 128), torch.zeros(128 * 128, dtype=BF16)
    whole = w.data
    assert native.packed_of(w) is None
    native.remember_packed(w, packed)
    try:
        for other in (whole[:64], whole.t(), whole[:, :64], whole.view(256, 64)):
            assert native.packed_of(w).data_ptr() == packed.data_ptr()
            w.data = other
            assert native.packed_of(w) is None
            w.data = whole
        w.add_(1)  # a new version
        assert native.packed_of(w) is None
    finally:
        native.forget_packed(int(w._cdata))
    assert native.packed_of(w) is None


_LOCK_ORDER = """
import threading, torch
import rldx_amd.ops
native = torch.ops.rldx_native
w = torch.zeros(64, 64, dtype=torch.bfloat16)

class Noted(torch.Tensor):  # a Python object whose end runs Python code
    def __del__(self):
        for _ in range(1000):
            native.packed_of(w)

for _ in range(200):
    native.remember_packed(w, torch.zeros(64 * 64, dtype=torch.bfloat16).as_subclass(Noted))
native.forget_packed(int(w._cdata))
print("done")
"""


@pytest.mark.skipif(not ops._native, reason="librldx_torch.so was not built")
def test_replaced_copies_are_freed_outside_the_lock():
    """A packed tensor may be Python's last one, and its end may run Python code that calls
    the operator again: with the table's lock held that would never return."""
    env = {**os.environ, "PYTHONPATH": str(Path(ops.__file__).resolve().parents[1])}
    r = subprocess.run([sys.executable, "-c", _LOCK_ORDER], env=env, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "done", r.stderr[-2000:]
