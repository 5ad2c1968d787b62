"""The workspace a W4A16 / W8A16 caller is told to bring covers what the launch writes, whatever the configuration asks for:
host code only, no kernel runs."""
from __future__ import annotations

import ctypes
import random

import pytest
import torch

from forge_amd import _lib

ODD_WIDTHS = (8, 16, 32, 96, 192, 320)  # tile_n values that name no tile kernel (they are widths of the GEMV's)
SHAPES = [(m, n, k) for m in (5, 20, 33, 64, 100, 256, 300, 700, 1111, 1409, 2304) for n in (520, 2816, 4096, 6144, 28672)
          for k in (1056, 4096, 4160, 14336)]


def _w4(m, n, k, gs=128, **kw):
    return _lib.lib().fg_w4a16_workspace_bytes(m, n, k, gs, 1, 1, 0, ctypes.byref(_config(**kw)))


def _w8(m, n, k, gs=-1, **kw):
    return _lib.lib().fg_w8a16_workspace_bytes(m, n, k, gs, ctypes.byref(_config(**kw)))


def _config(impl=None, tile_m=0, split_k=0, tile_n=0):
    return _lib.W4Config(_lib.W4_IMPL[impl], 0, 0, tile_m, split_k, tile_n, 0)


@pytest.mark.parametrize("query", [_w4, _w8])
@pytest.mark.parametrize("impl", [None, "prefill"])
def test_a_width_that_names_no_kernel_leaves_the_choice_and_the_size_to_the_policy(query, impl):
    for m, n, k in SHAPES:
        if impl == "prefill" and k % 64:
            continue
        for split in (0, 5, 13):
            policy = query(m, n, k, impl=impl, split_k=split)
            for width in ODD_WIDTHS:
                assert query(m, n, k, impl=impl, split_k=split, tile_n=width) == policy, (m, n, k, split, width)


def test_three_way_split_of_65_to_85_tiles_is_sized():
    for m, n in ((1111, 4096), (1281, 3072), (1409, 2816), (1280, 4352)):  # 80, 72, 66 and 85 tiles of 256 x 256
        for width in (0, 256, *ODD_WIDTHS):
            assert _w4(m, n, 4096, tile_n=width) >= 3 * m * n * 4


@pytest.mark.skipif(torch.cuda.is_available(), reason="the operands are addresses of nothing: only without a GPU, where no "
                                                      "launch can follow the checks")
@pytest.mark.parametrize("bits", [4, 8])
def test_every_launch_fits_the_workspace_it_asked_for(bits):
    """Calls over shapes, alignments, perms and configurations, each with exactly the bytes it was told to bring: the entry
    point compares them with the need of the kernel it chose, and only the launch itself fails (no device)."""
    lib, rng, addr = _lib.lib(), random.Random(7), 1 << 20
    seen = 0
    for _ in range(3000):
        m, n = int(2 ** rng.uniform(0, 12)), max(8, int(2 ** rng.uniform(6, 15)) // 8 * 8)
        k = max(32, int(2 ** rng.uniform(7, 14)) // 32 * 32)
        gs = rng.choice([g for g in (32, 64, 128, -1) if k % max(g, 1) == 0])
        g = 1 if gs < 0 else k // gs
        cfg = _config(rng.choice((None, None, "mfma", "prefill")), rng.choice((0, 0, 0, 64)), rng.choice((0, 0, 3, 13)),
                      rng.choice((0, 0, 64, 128, 256, *ODD_WIDTHS)))
        x, perm, sdt = addr + rng.choice((0, 0, 0, 2)), None, rng.choice((_lib.F16, _lib.F16, _lib.F32))
        if bits == 4:
            perm = rng.choice((None, None, None, addr))
            need = lib.fg_w4a16_workspace_bytes(m, n, k, gs, int(x % 16 == 0), 1, 0, ctypes.byref(cfg))
            args = (x, k, _lib.BF16, addr, k // 8, addr, sdt, n, addr, n // 8, perm, None, None, 0, addr, n, m, n, k, gs, g)
            call = lib.fg_w4a16_gemm
        else:
            need = lib.fg_w8a16_workspace_bytes(m, n, k, gs, ctypes.byref(cfg))
            args = (x, k, _lib.BF16, addr, k, addr, sdt, n, None, 0, addr, n, m, n, k, gs, g)
            call = lib.fg_w8a16_gemm
        status = call(*args, ctypes.byref(cfg), addr if need else None, need, None)
        assert status in (_lib.EHIP, _lib.EUNSUPPORTED), (m, n, k, gs, x, cfg.impl, cfg.split_k, cfg.tile_n, _lib.last_error())
        seen += status == _lib.EHIP
        if bits == 4 and need and status == _lib.EHIP:
            assert call(*args, ctypes.byref(cfg), addr, need - 1, None) == _lib.EINVAL
    assert seen > 1500


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,tile_n", [(1111, 4096, 4096, 32), (1409, 2816, 4160, 96), (20, 1032, 4128, 64)])
def test_odd_widths_run_as_the_policy_does(m, n, k, tile_n):
    """Through the public op, with nothing past the workspace written: 80 and 66 tiles split three ways, and few rows over a
    K that ends inside a slice."""
    from forge_amd import layouts as L
    from forge_amd import ops_gemm as ops
    from tests._util import w4_parts, x_act

    gs = 64 if k % 64 == 0 else 32
    p = L.pack_w4(*w4_parts(n, k, gs, False, seed=m), gs).to("cuda")
    x = x_act(m, k, torch.bfloat16, seed=m).to("cuda")
    y = ops.w4a16_linear(x, p)
    kern = ops.last_kernel()
    guard = 1 << 20
    lib, cfg = _lib.lib(), _config(tile_n=tile_n)
    need = lib.fg_w4a16_workspace_bytes(m, n, k, gs, 1, 1, 0, ctypes.byref(cfg))
    ws = torch.full((need + guard,), 0x5A, dtype=torch.uint8, device="cuda")
    out = torch.empty_like(y)
    _lib.check(lib.fg_w4a16_gemm(
        _lib.ptr(x), x.stride(0), _lib.BF16, _lib.ptr(p.qweight), p.qweight.stride(0), _lib.ptr(p.scales), _lib.F16,
        p.scales.stride(0), _lib.ptr(p.zeros), p.zeros.stride(0), None, None, None, 0, _lib.ptr(out), n, m, n, k, gs,
        p.num_groups, ctypes.byref(cfg), _lib.ptr(ws), need, _lib.stream_of(x)), "fg_w4a16_gemm")
    assert _lib.last_kernel() == kern and torch.equal(out, y)
    assert (ws[need:] == 0x5A).all()
    assert torch.equal(ops.w4a16_linear(x, p, config={"tile_n": tile_n}), y)
