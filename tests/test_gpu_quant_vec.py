"""The 16-byte activation quantisers against the element-wise ones: rows one element longer than they need send the same
values to the element-wise kernels, so codes and scales have to agree bit for bit."""
from __future__ import annotations

import pytest
import torch

from forge_amd import ops_gemm as ops
from tests._util import gen

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _values(m: int, k: int, dt: torch.dtype, seed: int) -> torch.Tensor:
    """Rows of ordinary values, and (from four rows) rows of zeros of both signs, of the type's smallest and largest
    magnitudes, and with a NaN and infinities."""
    g = gen(seed)
    x = torch.randn(m, k, generator=g) * torch.exp2(torch.randint(-20, 10, (m, 1), generator=g).float())
    x = x.to(dt)
    x[:, ::7] = -0.0
    if m >= 8:
        x[1] = 0.0
        x[1, ::2] = -0.0
        x[2] = torch.finfo(dt).smallest_normal / 64 * torch.randint(-9, 10, (k,), generator=g)
        x[3] = torch.finfo(dt).max * (torch.rand(k, generator=g) * 2 - 1)
        x[4, k // 2] = float("nan")
        x[5, 0], x[5, k - 1] = float("inf"), -1.0
        x[6, k - 1] = -float("nan")
        x[7] = torch.finfo(dt).tiny * 2.0 ** -5
    return x.to(DEV)


def _strided(x: torch.Tensor) -> torch.Tensor:
    wide = torch.zeros(x.shape[0] + 1, x.shape[1] + 1, dtype=x.dtype, device=x.device)
    wide[:-1, :-1] = x
    return wide[:-1, :-1] if x.shape[0] > 1 else wide[0, 1:].copy_(x[0]).reshape(1, -1)  # one row: off by one element


def _same(a, b):
    assert torch.equal(a[0].view(torch.uint8), b[0].view(torch.uint8)), "codes differ"
    assert torch.equal(a[1].view(torch.int32), b[1].view(torch.int32)), "scales differ"


# one unit per row; under, at and over a wavefront of units; 1, 2, 4 and 8 units per thread; the largest row and past it
ROWS = [(1, 8), (8, 504), (9, 512), (9, 520), (8, 8192), (600, 4096), (600, 1032), (16, 14336), (3, 32768), (2, 65536),
        (2, 65544)]


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,k", ROWS)
def test_rowwise_equals_elementwise(m, k, dt):
    x = _values(m, k, dt, m + k)
    _same(ops.quantize_act_int8(x), ops.quantize_act_int8(_strided(x)))
    _same(ops.quantize_act_fp8(x), ops.quantize_act_fp8(_strided(x)))


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("block", [8, 64, 128, 512])
@pytest.mark.parametrize("m,k", [(1, 8), (9, 520), (33, 1000), (600, 4096)])
def test_row_blocks_equal_elementwise(m, k, block, dt):
    x = _values(m, k, dt, m + k + block)
    _same(ops.quantize_act_fp8(x, granularity="block", block=block),
          ops.quantize_act_fp8(_strided(x), granularity="block", block=block))


# one wavefront per row and more, one to eight units per thread, the largest row in LDS and past it
@pytest.mark.parametrize("wdt", [None, torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,k", [(1, 8), (8, 504), (9, 520), (600, 512), (600, 1032), (600, 4096), (1024, 14336), (3, 28672),
                                 (9, 32000), (3, 32008)])
def test_norm_rowwise_equals_elementwise(m, k, dt, wdt):
    """The sum of squares runs in the element-wise kernel's order, so codes and scales agree bit for bit here too."""
    x = _values(m, k, dt, m + k) if m == 9 else torch.randn(m, k, generator=gen(k)).to(dt).to(DEV)
    w = None if wdt is None else (1 + 0.1 * torch.randn(k, generator=gen(1))).to(wdt).to(DEV)
    _same(ops.quantize_act_fp8(x, rms_weight=w, rms_eps=1e-5),
          ops.quantize_act_fp8(_strided(x), rms_weight=w, rms_eps=1e-5))


@pytest.mark.parametrize("wdt", [None, torch.bfloat16])
@pytest.mark.parametrize("m,k", [(8, 504), (9, 520), (600, 1032), (9, 8192)])
def test_norm_of_rows_whose_squares_underflow(m, k, wdt):
    """eps = 0 and a row whose mean square is zero: the row is multiplied by infinity, and the threads that hold no unit
    of it must not add a NaN of their own."""
    x = _values(m, k, torch.bfloat16, m + k)
    w = None if wdt is None else (1 + 0.1 * torch.randn(k, generator=gen(1))).to(wdt).to(DEV)
    a = ops.quantize_act_fp8(x, rms_weight=w, rms_eps=0.0)
    _same(a, ops.quantize_act_fp8(_strided(x), rms_weight=w, rms_eps=0.0))
    assert torch.isinf(a[1][7])
