"""The W8A8 tiles of the automatic policy, each reached at a ragged output size, with K of one slice, of more slices than
the ring has stages, and ending inside a slice (K % 128 != 0): FP8, FP8 with K-blocked scales, INT8.  The same operands
eight bytes off 16-byte alignment run in the register-staged kernel, which multiplies and adds in the same order, so
results agree bit for bit; INT8 is also compared with an exact product."""
from __future__ import annotations

import pytest
import torch

from forge_amd import ops_gemm as ops
from tests._util import assert_close, gen
from tests.test_isa_waits import _check_ring_loops, kernels  # noqa: F401  (fixture)

DEV = "cuda"
# (m, n) whose cheapest tile is rows x columns
TILES = [(1, 96, "64x32"), (33, 8200, "64x64"), (70, 9000, "128x64"), (17, 16392, "64x128"), (70, 16392, "128x128"),
         (130, 12296, "192x64"), (130, 16392, "192x128"), (200, 16392, "256x128"), (385, 16392, "256x256"),
         (513, 16390, "256x256")]
KS = [16, 128, 160, 1264]


def _off(t: torch.Tensor) -> torch.Tensor:
    wide = torch.zeros(t.shape[0], t.shape[1] + 8, dtype=torch.uint8, device=t.device)
    wide[:, 8:] = t.view(torch.uint8)
    return wide.view(t.dtype)[:, 8:]


def _codes(m: int, k: int, dt: torch.dtype, seed: int) -> torch.Tensor:
    x = torch.randn(m, k, generator=gen(seed)) * 40
    return (x.clamp(-127, 127).round().to(dt) if dt == torch.int8 else x.to(dt)).to(DEV)


@pytest.mark.gpu
@pytest.mark.parametrize("k", KS)
@pytest.mark.parametrize("m,n,tile", TILES)
def test_fp8_tiles(m, n, tile, k):
    a, w = _codes(m, k, torch.float8_e4m3fn, m + k), _codes(n, k, torch.float8_e4m3fn, n + k)
    sx, sw = torch.rand(m, generator=gen(1)).to(DEV), torch.rand(n, generator=gen(2)).to(DEV)
    b = torch.randn(n, generator=gen(3)).to(torch.bfloat16).to(DEV)
    for odt, bias in ((torch.bfloat16, b), (torch.float32, None)):
        y = ops.fp8_linear(a, w, sw, bias, x_scale=sx, out_dtype=odt)
        assert tile in ops.last_kernel(), ops.last_kernel()
        ref = ops.fp8_linear(_off(a), _off(w), sw, bias, x_scale=sx, out_dtype=odt)
        assert ops.last_kernel().startswith("mm_kernel") and torch.equal(y, ref)


@pytest.mark.gpu
@pytest.mark.parametrize("k,per_row_weight", [(k, r) for k in KS for r in (False, True)
                                              if k > 128 or not r])  # one block of per-row scales is a per-channel scale
@pytest.mark.parametrize("m,n,tile", TILES)
def test_fp8_block_scale_tiles(m, n, tile, k, per_row_weight):
    a, w = _codes(m, k, torch.float8_e4m3fn, m + k), _codes(n, k, torch.float8_e4m3fn, n + k)
    kb = -(-k // 128)
    sx = torch.rand(kb, m, generator=gen(1)).to(DEV).t()  # block-major, and row-major below
    sw = torch.rand(n if per_row_weight else -(-n // 128), kb, generator=gen(2)).to(DEV)
    b = torch.randn(n, generator=gen(3)).to(torch.bfloat16).to(DEV)
    ref = {}
    for odt, bias in ((torch.bfloat16, b), (torch.float32, None)):
        ref[odt] = ops.fp8_linear(_off(a), _off(w), sw, bias, x_scale=sx, out_dtype=odt)
        assert ops.last_kernel().startswith("mm_kernel")
        for scale in (sx, sx.contiguous()):
            y = ops.fp8_linear(a, w, sw, bias, x_scale=scale, out_dtype=odt)
            assert ops.last_kernel().startswith(f"mm_blk_kernel {tile}"), ops.last_kernel()
            assert torch.equal(y, ref[odt])


@pytest.mark.gpu
@pytest.mark.parametrize("k", KS)
@pytest.mark.parametrize("m,n,tile", [t for t in TILES if t[0] > 2])
def test_int8_tiles(m, n, tile, k):
    a, w = _codes(m, k, torch.int8, m + k), _codes(n, k, torch.int8, n + k)
    acc = ops.int8_gemm(a, None, w, None, out_dtype=torch.int32)
    assert tile in ops.last_kernel(), ops.last_kernel()
    assert torch.equal(acc.double(), a.double() @ w.double().t())
    sx, sw = torch.rand(m, generator=gen(1)).to(DEV), torch.rand(n, generator=gen(2)).to(DEV)
    y = ops.int8_gemm(a, sx, w, sw, out_dtype=torch.float16)
    assert torch.equal(y, ((acc.float() * sx.view(-1, 1)) * sw).half())


# K of whole 256-column steps: the skinny kernel's lines on both sides (256 CUs: 8192 channels are one 64 x 32 tile each)
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,expect", [
    (8, 8192, 256, "w8_skinny"), (8, 8224, 256, "mm_ring"), (9, 8192, 1024, "mm_ring"), (9, 8160, 1024, "w8_skinny"),
    (16, 8160, 256, "w8_skinny"), (17, 8160, 256, "mm_ring"), (17, 4096, 1024, "w8_skinny"), (32, 4096, 256, "w8_skinny"),
    (32, 4128, 256, "mm_ring"), (33, 4096, 1024, "mm_ring"), (16, 8224, 16384, "w8_skinny"), (17, 8224, 16384, "mm_ring")])
def test_skinny_kernel_lines(m, n, k, expect):
    a, w = _codes(m, k, torch.int8, m + k), _codes(n, k, torch.int8, n + k)
    acc = ops.int8_gemm(a, None, w, None, out_dtype=torch.int32)
    assert ops.last_kernel().startswith(expect), ops.last_kernel()
    assert torch.equal(acc.double(), a.double() @ w.double().t())
    a, w = _codes(m, k, torch.float8_e4m3fn, m + k), _codes(n, k, torch.float8_e4m3fn, n + k)
    sx, sw = torch.rand(m, generator=gen(1)).to(DEV), torch.rand(n, generator=gen(2)).to(DEV)
    y = ops.fp8_linear(a, w, sw, x_scale=sx, out_dtype=torch.float32)
    assert ops.last_kernel().startswith(expect), ops.last_kernel()
    ref = (a.double() @ w.double().t()) * sx.double().view(-1, 1) * sw.double()
    assert_close(y.cpu(), ref.cpu().float().numpy(), "float32", what=ops.last_kernel())


@pytest.mark.gpu
@pytest.mark.parametrize("m,k", [(5, 1024), (70, 1000), (3, 777)])
def test_block_linear_quantises_like_the_quantiser(m, k):
    """fp8_linear on float x with block scales: the codes and scales of quantize_act_fp8, whatever their layout."""
    x = torch.randn(m, k, generator=gen(k)).to(torch.bfloat16).to(DEV)
    w = _codes(520, k, torch.float8_e4m3fn, 1)
    sw = torch.rand(5, -(-k // 128), generator=gen(2)).to(DEV)
    q, s = ops.quantize_act_fp8(x, granularity="block")
    assert torch.equal(ops.fp8_linear(x, w, sw), ops.fp8_linear(q, w, sw, x_scale=s))


def test_block_kernel_loop_issues_one_slice_and_waits_for_the_next(kernels):  # noqa: F811
    """The load accounting of mm_blk_kernel in the built code: the ring kernel's, with one more load per slice (scales)."""
    import re
    found = 0
    for name, code in kernels.items():
        if "mm_blk_kernel" not in name:
            continue
        bm, bn, wm, wn, s = (int(v) for v in re.findall(r"Li(\d+)E", name)[:5])
        if s > 2:
            found += _check_ring_loops(name, code, (bm + bn) * 128 // 16 // (wm * wn * 64) + 1, s)
    assert found >= 9, f"expected the block-scale instances' loops, checked {found}"
