"""Host side of a call, on the CPU: switches are read as they are at the call, scale preparation gives the same views
through its short and its general path, and a weight's stamp follows its tensors."""
from __future__ import annotations

import os

import pytest
import torch

from forge_amd import layouts as L
from forge_amd import ops_gemm as ops
from tests._util import w4_parts


def test_switches_follow_the_environment(monkeypatch):
    assert not ops.force_ref() and ops.forced_impl() is None and not ops.kernel_debug()
    monkeypatch.setenv("FORGE_FORCE_REF", "1")
    monkeypatch.setenv("FORGE_W4_IMPL", " Prefill ")
    monkeypatch.setenv("FORGE_KERNEL_DEBUG", "1")
    assert ops.force_ref() and ops.forced_impl() == "prefill" and ops.kernel_debug()
    os.environ["FORGE_W4_IMPL"] = "unheard-of"
    assert ops.forced_impl() is None
    monkeypatch.delenv("FORGE_FORCE_REF")
    assert not ops.force_ref()


def test_switches_follow_an_environment_put_in_its_place(monkeypatch):
    monkeypatch.setattr(os, "environ", {**os.environ, "FORGE_FORCE_REF": "1", "FORGE_W4_IMPL": "gemv"})
    assert ops.force_ref() and ops.forced_impl() == "gemv" and not ops.kernel_debug()
    monkeypatch.undo()
    assert not ops.force_ref() and ops.forced_impl() is None


def _view(side, strides, i, kb):
    return side.as_strided((1,), (1,), side.storage_offset() + i * strides[0] + kb * strides[1]).item()


@pytest.mark.parametrize("m", [1, 2, 5])
@pytest.mark.parametrize("n", [1, 2, 7])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_vector_scales_short_path_equals_general(m, n, dt):
    sx, sw = torch.rand(m).to(dt), torch.rand(n).to(dt)
    wide = torch.stack([sx, sx], 1)[:, 0], torch.stack([sw, sw], 1)[:, 0]  # strided: the general path
    short, general = ops.prepare_fp8_scales(sx, sw, m, n, 256, 128), ops.prepare_fp8_scales(*wide, m, n, 256, 128)
    assert short[0] == general[0] and short[4] == general[4]
    for i in range(m):
        assert _view(short[1], short[3][:2], i, 1) == _view(general[1], general[3][:2], i, 1) == sx[i].float().item()
    for i in range(n):
        assert _view(short[2], short[3][2:], i, 1) == _view(general[2], general[3][2:], i, 1) == sw[i].float().item()


def test_block_scales_are_read_through_their_strides():
    sx, sw = torch.rand(3, 5), torch.rand(2, 3)
    dense, turned = (ops.prepare_fp8_scales(a, sw, 5, 256, 300, 128) for a in (sx.t().contiguous(), sx.t()))
    assert dense[0] == turned[0] == 2 and turned[3][:2] == (1, 5)
    for i in range(5):
        for kb in range(3):
            assert _view(dense[1], dense[3][:2], i, kb) == _view(turned[1], turned[3][:2], i, kb) == sx[kb, i].item()


@pytest.mark.parametrize("sym,act_order", [(True, False), (False, False), (True, True), (False, True)])
def test_stamp_changes_with_every_tensor(sym, act_order):
    q, s, z = w4_parts(16, 64, 32, sym)
    p = L.pack_w4(q, s, z, 32, g_idx=torch.arange(64) // 32 if act_order else None)
    seen = {ops._stamp(p)}
    for t in p.tensors().values():
        t.add_(0)
        seen.add(ops._stamp(p))
    p.scales = p.scales.clone()
    seen.add(ops._stamp(p))
    assert len(seen) == len(p.tensors()) + 2


@pytest.mark.parametrize("name", ["qweight", "scales"])
@pytest.mark.parametrize("cls", [ops.KernelW4A16Linear, ops.KernelW8A16Linear])
def test_packed_follows_a_parameter_in_a_buffers_place(cls, name):
    mod = cls.from_dense(torch.nn.Linear(64, 16, bias=False))
    setattr(mod, name, torch.nn.Parameter(getattr(mod, name).clone(), requires_grad=False))
    assert getattr(mod.packed(), name) is getattr(mod, name) is mod._parameters[name]
