"""The ping-pong kernel below 160 tiles, reached through the policy: K split three ways on W4 and W8A16 weights, the
neighbours of that range on both sides, short K, ragged rows and channels, against the CPU oracle."""
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


@pytest.mark.parametrize("m,n,k,gs,xdt,expect", [
    (1111, 4096, 4096, 128, BF, "w4_pp_kernel<bf16,w4> 256x256 splits=3"),   # 80 tiles
    (1409, 2816, 4160, 64, HF, "w4_pp_kernel<f16,w4> 256x256 splits=3"),     # 66 tiles, an uneven last split
    (1153, 4104, 4096, -1, BF, "w4_pp_kernel<bf16,w4> 256x256 splits=3"),    # 85 tiles, the last 8 channels wide
    (1111, 4096, 4032, 64, BF, "w4_pc_kernel"),                           # K below the line
    (600, 6144, 4096, 128, HF, "w4_pc_kernel"),                           # 128-row tiles of that kernel fit one round
    (1280, 4608, 4096, 128, BF, "w4_pc_kernel"),                          # 90 tiles
])
def test_w4(m, n, k, gs, xdt, expect):
    q, s, z = w4_parts(n, k, gs, False, seed=m)
    p = L.pack_w4(q, s, z, gs).to(DEV)
    x = x_act(m, k, xdt, seed=m)
    y = ops.w4a16_linear(x.to(DEV), p)
    assert ops.last_kernel().startswith(expect), ops.last_kernel()
    ref = og.w4a16_gemm_ref(to_f32(x), oracle_packed(q, s, z, gs))
    assert_close(y.cpu(), ref, "bfloat16" if xdt == BF else "float16", what=expect)
    assert torch.equal(y, ops.w4a16_linear(x.to(DEV), p))


@pytest.mark.parametrize("m,n,k,gs,xdt,split", [
    (1111, 4096, 4096, -1, BF, 3), (600, 6144, 2048, 128, HF, 3), (1153, 4104, 1600, -1, BF, 3), (1111, 4096, 1024, -1, BF, 2),
    (1111, 4096, 512, -1, HF, 1), (2304, 4096, 1088, 64, BF, 1), (1500, 4096, 1024, -1, HF, 2)])
def test_int8_weights(m, n, k, gs, xdt, split):
    q = torch.randint(-128, 128, (n, k), generator=gen(m + k), dtype=torch.int8)
    s = (torch.rand(n, L.num_groups(k, gs), generator=gen(1)) * 0.01).half()
    p = L.pack_w8(q, s, gs).to(DEV)
    x = x_act(m, k, xdt, seed=m)
    y = ops.w8a16_linear(x.to(DEV), p)
    assert ops.last_kernel().startswith("w4_pp_kernel<") and f"256x256 splits={split}" in ops.last_kernel(), ops.last_kernel()
    ref = og.w8a16_gemm_ref(to_f32(x), og.pack_w8(q.numpy(), s.float().numpy(), gs))
    assert_close(y.cpu(), ref, "bfloat16" if xdt == BF else "float16", what=f"w8a16 m={m} n={n} k={k}")
    assert torch.equal(y, ops.w8a16_linear(x.to(DEV), p))


@pytest.mark.parametrize("m,n,k,gs,xdt,split", [
    (600, 4096, 1024, -1, BF, 4), (600, 4096, 512, 128, HF, 1), (1024, 4096, 1024, -1, BF, 2), (1024, 4096, 1984, 64, BF, 3),
    (700, 3592, 1088, -1, HF, 4)])
def test_int8_weights_of_40_to_64_tiles(m, n, k, gs, xdt, split):
    test_int8_weights(m, n, k, gs, xdt, split)
