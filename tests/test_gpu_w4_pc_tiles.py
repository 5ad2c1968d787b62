"""The producer / consumer kernel's row tiles, groups and K tails, reached through the policy: 64-, 128- and 256-row tiles
with and without K splits, groups of 32 / 64 / 96 / one, K that ends inside a 64-column slice, fp16 and bf16 x with scales
of either type (packed fp16 dequantisation and the fp32 one), against the CPU oracle."""
from __future__ import annotations

import pytest
import torch

from forge_amd import layouts as L
from forge_amd import ops_gemm as ops
from oracle import gemm as og
from tests._util import assert_close, gen, oracle_packed, to_f32, w4_parts, x_act

pytestmark = pytest.mark.gpu
DEV = "cuda"
BF, HF = torch.bfloat16, torch.float16
CASES = [  # m, n, k, group, sym, x, scales, bias, tile rows
    (5, 136, 512, 64, False, HF, HF, None, 64),
    (17, 1032, 1056, 32, True, BF, HF, BF, 64),       # K % 64 == 32
    (64, 2048, 96, 96, False, HF, BF, HF, 64),        # one group, one slice and a half
    (65, 1024, 2048, 64, False, HF, HF, HF, 64),
    (128, 6144, 4096, 64, True, HF, HF, HF, 128),     # splits
    (127, 16392, 1056, 32, False, BF, BF, None, 128),
    (200, 6144, 2048, 32, False, BF, HF, None, 256),
    (129, 6144, 4128, 96, True, HF, HF, BF, 256),
    (256, 20488, 544, -1, False, HF, HF, None, 256),
    (33, 20488, 160, 32, False, HF, HF, None, 64),    # tiles cover the CUs: no split
]


@pytest.mark.parametrize("m,n,k,gs,sym,xdt,sdt,bdt,bm", CASES)
def test_tiles_groups_and_tails(m, n, k, gs, sym, xdt, sdt, bdt, bm):
    q, s, z = w4_parts(n, k, gs, sym, seed=m + k, scale_dtype=sdt)
    p = L.pack_w4(q, s, z, gs).to(DEV)
    x = x_act(m, k, xdt, seed=m)
    b = None if bdt is None else torch.randn(n, generator=gen(3)).to(bdt)
    y = ops.w4a16_linear(x.to(DEV), p, None if b is None else b.to(DEV))
    kern = ops.last_kernel()
    assert kern.startswith("w4_pc_kernel") and f" {bm}x128" in kern, kern
    ref = og.w4a16_gemm_ref(to_f32(x), oracle_packed(q, s, z, gs), None if b is None else to_f32(b))
    assert_close(y.cpu(), ref, "bfloat16" if xdt == BF else "float16", what=kern)
    assert torch.equal(y, ops.w4a16_linear(x.to(DEV), p, None if b is None else b.to(DEV)))


def test_packed_fp16_dequantisation_equals_the_fp32_form():
    """Every code, zero-point and a spread of fp16 scales (subnormal products among them): x picks single weights, so
    the outputs are the dequantised weights themselves, equal to ((q - z) * s) rounded once to fp16."""
    n, k = 256, 64
    q = torch.arange(16, dtype=torch.uint8).repeat(n, k // 16)
    z = (torch.arange(n) % 16).to(torch.uint8).view(n, 1)
    s = torch.exp2(torch.linspace(-24, 10, n)).mul(1 + torch.rand(n, generator=gen(1))).half().view(n, 1)
    p = L.pack_w4(q, s, z, k).to(DEV)
    y = ops.w4a16_linear(torch.eye(k).half().to(DEV), p)
    assert ops.last_kernel().startswith("w4_pc_kernel") or ops.last_kernel().startswith("w4_skinny"), ops.last_kernel()
    y = ops.w4a16_linear(torch.eye(k).half().to(DEV), p, config={"impl": "prefill", "tile_n": 128})
    assert ops.last_kernel().startswith("w4_pc_kernel"), ops.last_kernel()
    want = ((q.float() - z.float()) * s.float()).half()
    assert torch.equal(y.cpu(), want.t())


def test_forced_prefill_still_refuses_what_it_refused():
    q, s, z = w4_parts(128, 96, 32, False)
    p = L.pack_w4(q, s, z, 32).to(DEV)
    from forge_amd import _lib
    with pytest.raises(_lib.KernelLaunchError, match="K%64"):
        ops.w4a16_linear(x_act(70, 96).to(DEV), p, config={"impl": "prefill"})


@pytest.mark.parametrize("m,n,k,gs,xdt,bdt", [
    (3, 130, 96, -1, BF, None), (6, 3072, 1376, -1, HF, BF), (64, 4096, 160, 32, BF, BF), (70, 6144, 4096, -1, BF, None),
    (128, 1030, 1056, 96, HF, HF), (200, 4096, 2048, 64, HF, None), (256, 520, 4096, 32, BF, BF), (700, 3074, 1376, -1, BF, None)])
def test_int8_weights(m, n, k, gs, xdt, bdt):
    """W8A16 in the same kernel: groups of 32 / 64 / 96 / one, K tails, splits; |q| up to 128."""
    q = torch.randint(-128, 128, (n, k), generator=gen(m + k), dtype=torch.int8)
    s = (torch.rand(n, L.num_groups(k, gs), generator=gen(1)) * 0.01).half()
    p = L.pack_w8(q, s, gs).to(DEV)
    x = x_act(m, k, xdt, seed=m)
    b = None if bdt is None else torch.randn(n, generator=gen(3)).to(bdt)
    y = ops.w8a16_linear(x.to(DEV), p, None if b is None else b.to(DEV))
    assert ops.last_kernel().startswith("w4_pc_kernel<") and ",w8>" in ops.last_kernel(), ops.last_kernel()
    w = q.double() * s.double().repeat_interleave(k if gs < 0 else gs, 1)[:, :k]
    ref = x.double() @ w.t() + (0 if b is None else b.double())
    assert_close(y.cpu(), ref.float().numpy(), "bfloat16" if xdt == BF else "float16", what=ops.last_kernel())


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("m", [20, 100])
@pytest.mark.parametrize("k,gs", [(1056, 32), (96, 96), (4128, -1)])
def test_overflowing_weights_before_a_k_tail_give_infinity(m, k, gs, bits):
    """Weights of the last 32 columns that round to an fp16 infinity: the columns past K hold nothing, so y is infinite (x
    is positive) and not a NaN."""
    n = 136
    g = 1 if gs < 0 else k // gs
    s = torch.full((n, g), 0.01).half()
    s[:, -1] = 8000.0
    q = torch.full((n, k), 9 if bits == 4 else 1, dtype=torch.uint8 if bits == 4 else torch.int8)
    q[:, -32:] = 15 if bits == 4 else 100
    x = torch.ones(m, k).half().to(DEV)
    if bits == 4:
        y = ops.w4a16_linear(x, L.pack_w4(q, s, torch.full((n, g), 1, dtype=torch.uint8), gs).to(DEV))
    else:
        y = ops.w8a16_linear(x, L.pack_w8(q, s, gs).to(DEV))
    assert ops.last_kernel().startswith("w4_pc_kernel"), ops.last_kernel()
    assert torch.isposinf(y).all()


@pytest.mark.parametrize("m,n,k,gs,xdt,expect", [
    (16, 20480, 2048, 64, BF, "w4_big_kernel<64"),    # 80 wide tiles: three K splits in a round, against one
    (5, 43016, 1024, 32, BF, "w4_big_kernel<64"),
    (16, 4096, 2048, 64, BF, "w4_pc_kernel"),
    (300, 20480, 576, 32, BF, "w4_big_kernel<128"),
    (509, 28680, 1024, 32, BF, "w4_big_kernel<256"),
    (513, 4104, 1152, 96, HF, "w4_pc_kernel"),
    (300, 20480, 576, 64, BF, "w4_pp_kernel"),        # groups of 64 from 256 rows: by the other rules
])
def test_all_rounder_where_it_costs_less(m, n, k, gs, xdt, expect):
    q, s, z = w4_parts(n, k, gs, False, seed=m)
    p = L.pack_w4(q, s, z, gs).to(DEV)
    x = x_act(m, k, xdt, seed=m)
    y = ops.w4a16_linear(x.to(DEV), p)
    assert ops.last_kernel().startswith(expect), ops.last_kernel()
    ref = og.w4a16_gemm_ref(to_f32(x), oracle_packed(q, s, z, gs))
    assert_close(y.cpu(), ref, "bfloat16" if xdt == BF else "float16", what=expect)


@pytest.mark.parametrize("m,n,k,gs,xdt,expect", [
    (129, 8192, 2048, -1, BF, "w4_pc_kernel"), (129, 5120, 8192, 64, BF, "w4_big_kernel"), (70, 4096, 4096, -1, BF, "w4_pc_kernel"),
    (173, 9608, 8192, -1, HF, "w4_big_kernel"), (256, 2048, 8192, -1, BF, "w4_pc_kernel")])
def test_all_rounder_on_int8_weights_where_it_costs_less(m, n, k, gs, xdt, expect):
    q = torch.randint(-128, 128, (n, k), generator=gen(m + k), dtype=torch.int8)
    s = (torch.rand(n, L.num_groups(k, gs), generator=gen(1)) * 0.01).half()
    x = x_act(m, k, xdt, seed=m)
    y = ops.w8a16_linear(x.to(DEV), L.pack_w8(q, s, gs).to(DEV))
    assert ops.last_kernel().startswith(expect), ops.last_kernel()
    ref = x.double() @ (q.double() * s.double().repeat_interleave(k if gs < 0 else gs, 1)).t()
    assert_close(y.cpu(), ref.float().numpy(), "bfloat16" if xdt == BF else "float16", what=ops.last_kernel())


@pytest.mark.parametrize("xdt", [BF, HF])
@pytest.mark.parametrize("m,n,k,gs", [(6, 1032, 4128, 32), (40, 264, 1056, 96), (100, 1024, 4128, -1), (513, 520, 1376, 32)])
def test_int8_weights_stay_exact_before_a_k_tail(m, n, k, gs, xdt):
    """No weight is rounded to 16 bits: the distance to the 64-bit product is that of its rounding to x's type, and the
    fp32 sum's, K terms of 2^-24 at most, here within a hundredth of the former."""
    q = torch.randint(-128, 128, (n, k), generator=gen(m + k), dtype=torch.int8)
    s = (torch.rand(n, L.num_groups(k, gs), generator=gen(1)) * 0.002 + 0.0002).half()
    x = x_act(m, k, xdt, seed=m)
    y = ops.w8a16_linear(x.to(DEV), L.pack_w8(q, s, gs).to(DEV)).cpu().double()
    assert ops.last_kernel().startswith("w4_pc_kernel<") and ",w8>" in ops.last_kernel(), ops.last_kernel()
    ref = x.double() @ (q.double() * s.double().repeat_interleave(k if gs < 0 else gs, 1)).t()
    assert (y - ref).norm() <= 1.01 * (ref.to(xdt).double() - ref).norm()
