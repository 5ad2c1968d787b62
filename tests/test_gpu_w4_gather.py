"""The column gather in front of act-order weights: every element in place, and the whole call against the oracle in the
kernels it now reaches."""
from __future__ import annotations

import pytest
import torch

from forge_amd import _lib
from forge_amd import layouts as L
from forge_amd import ops_gemm as ops
from oracle import gemm as og
from tests._util import assert_close, gen, oracle_packed, to_f32, w4_parts, x_act

pytestmark = pytest.mark.gpu
DEV = "cuda"


# direct form up to 64 rows and past 32768 columns; LDS form with 1, 2, 4 and 8 units per thread; K off the 8-column unit
@pytest.mark.parametrize("m,k", [(1, 8), (64, 4096), (65, 1), (65, 4093), (65, 4096), (70, 8192), (66, 14336),
                                 (65, 32768), (65, 32776), (1500, 520)])
@pytest.mark.parametrize("pad", [0, 3])
def test_gather_moves_every_element(m, k, pad):
    x = torch.randint(-30000, 30000, (m, k + pad), generator=gen(k), dtype=torch.int16).view(torch.bfloat16)
    x = x.to(DEV)[:, :k]
    perm = torch.randperm(k, generator=gen(m)).to(torch.int32).to(DEV)
    out = ops._gather_columns(x, perm)
    assert torch.equal(out.view(torch.int16), x[:, perm.long()].view(torch.int16)) and out.stride(0) % 8 == 0


# the GEMV on blocked scales, the CDNA4 copies, the prefill kernels, and (groups of 16) the tiled kernel
@pytest.mark.parametrize("m,n,k,gs,kernel", [(1, 1024, 2048, 128, "w4_gemv_split"), (16, 1024, 2048, 128, "w4_frag"),
                                             (100, 1024, 2048, 64, "w4_pc"), (300, 1030, 2048, 128, "w4_big"),
                                             (9, 520, 1056, 16, "w4_mfma")])
@pytest.mark.parametrize("xdt", [torch.bfloat16, torch.float16])
def test_act_order_module_reaches_the_policy_kernels(m, n, k, gs, kernel, xdt):
    q, s, z = w4_parts(n, k, gs, False, seed=m)
    g_idx = (torch.arange(k) // gs)[torch.randperm(k, generator=gen(k))].to(torch.int32)
    mod = ops.make_packed_linear("w4a16", packed=L.pack_w4(q, s, z, gs, g_idx=g_idx).to(DEV))
    x = x_act(m, k, xdt, seed=m + 1)
    y = mod(x.to(DEV))
    assert ops.last_kernel().startswith(f"gather_columns + {kernel}"), ops.last_kernel()
    ref = og.w4a16_gemm_ref(to_f32(x), oracle_packed(q, s, z, gs, g_idx))
    assert_close(y.cpu(), ref, "bfloat16" if xdt == torch.bfloat16 else "float16", what=f"act-order {kernel}")
    mod.scales.mul_(2)  # the copies of the sorted weight follow the weight's own tensors
    assert_close(mod(x.to(DEV)).cpu(), 2 * ref, "bfloat16" if xdt == torch.bfloat16 else "float16", what="scaled")


def test_a_forced_kernel_still_refuses_unaligned_rows():
    """config names a kernel that needs 16-byte aligned x: refused on an act-order weight as on a plain one, not served by
    the gather's aligned copy; the policy serves both."""
    m, n, k = 20, 512, 1024
    q, s, z = w4_parts(n, k, 128, False, seed=1)
    g_idx = (torch.arange(k) // 128)[torch.randperm(k, generator=gen(2))].to(torch.int32)
    x = x_act(m, k + 1, torch.bfloat16, seed=3).to(DEV)[:, 1:]
    for packed in (L.pack_w4(q, s, z, 128).to(DEV), L.pack_w4(q, s, z, 128, g_idx=g_idx).to(DEV)):
        for impl in ("mfma", "prefill", "dequant_gemm"):
            with pytest.raises(_lib.KernelLaunchError, match="aligned"):
                ops.w4a16_linear(x, packed, config={"impl": impl})
    y = ops.w4a16_linear(x, packed)
    ref = og.w4a16_gemm_ref(to_f32(x.cpu()), oracle_packed(q, s, z, 128, g_idx))
    assert_close(y.cpu(), ref, "bfloat16", what="act-order, unaligned x")


@pytest.mark.parametrize("m", [2, 9, 100])
def test_unaligned_rows_keep_fp32_weights(m):
    """The kernels for rows that are not 16-byte aligned multiply dequantised weights in fp32, with act order as without:
    the distance to the 64-bit product is that of its rounding to bf16 (and a hundredth for the fp32 sum)."""
    n, k = 520, 1024
    q, s, z = w4_parts(n, k, 128, False, seed=1)
    g_idx = (torch.arange(k) // 128)[torch.randperm(k, generator=gen(2))].to(torch.int32)
    x = x_act(m, k + 1, torch.bfloat16, seed=3)[:, 1:]
    y = ops.w4a16_linear(torch.nn.functional.pad(x, (1, 0)).to(DEV)[:, 1:], L.pack_w4(q, s, z, 128, g_idx=g_idx).to(DEV))
    w = (q.double() - z.double()[:, g_idx.long()]) * s.double()[:, g_idx.long()]
    ref = x.double() @ w.t()
    assert (y.cpu().double() - ref).norm() <= 1.01 * (ref.bfloat16().double() - ref).norm(), ops.last_kernel()


def test_the_gathers_label_ends_with_its_op():
    """A gather that no product followed (a failed allocation in between) does not name the next op's kernel."""
    x = x_act(20, 512, torch.bfloat16, seed=1).to(DEV)
    ops._gather_columns(x, torch.randperm(512, generator=gen(1)).to(torch.int32).to(DEV))
    assert ops.last_kernel() == "gather_columns"
    a = torch.ones(64, 256, dtype=torch.int8, device=DEV)
    ops.int8_gemm(a, None, a, None, out_dtype=torch.int32)
    assert "gather" not in ops.last_kernel(), ops.last_kernel()


def _act_order(m, n, k, gs, xdt, seed):
    q, s, z = w4_parts(n, k, gs, False, seed=seed)
    g_idx = (torch.arange(k) // gs)[torch.randperm(k, generator=gen(seed))].to(torch.int32)
    x = x_act(m, k, xdt, seed=seed + 1)
    return q, s, z, g_idx, x, og.w4a16_gemm_ref(to_f32(x), oracle_packed(q, s, z, gs, g_idx))


# the kernels that read the permutation themselves, which a C caller may hand over with the sorted weight
@pytest.mark.parametrize("m,n,k,gs,gemv,kernel", [
    (1, 1024, 2048, 128, "split", "w4_gemv_split"), (4, 1024, 2048, 64, "tile", "w4_gemv_tile"), (2, 1024, 2048, 128, "wave", "w4_gemv"),
    (1, 4096, 4096, 128, None, "w4_gemv"), (4, 4096, 4096, 128, None, "w4_"), (16, 1024, 2048, 128, None, "w4_mfma"),
    (128, 520, 1024, 64, None, "w4_mfma"), (9, 520, 1056, 16, None, "w4_mfma"), (9, 520, 1056, 16, "unaligned", "w4_generic")])
@pytest.mark.parametrize("xdt", [torch.bfloat16, torch.float16])
def test_permutation_in_the_kernel(m, n, k, gs, gemv, kernel, xdt):
    q, s, z, g_idx, x, ref = _act_order(m, n, k, gs, xdt, m + n)
    packed = L.pack_w4(q, s, z, gs, g_idx=g_idx).to(DEV)
    w, perm = L.cached_group_sort(packed, compute=True)
    xd, y = x.to(DEV), torch.empty(m, n, dtype=xdt, device=DEV)
    if gemv == "unaligned":
        xd, gemv = torch.nn.functional.pad(xd, (1, 0))[:, 1:], None
    config = None if gemv is None else {"impl": "gemv", "gemv_kernel": gemv}
    ops._w4_call(xd, ops._W4Operands(w, perm=perm), None, y, ops._w4_config(config))
    assert _lib.last_kernel().startswith(kernel), _lib.last_kernel()
    assert_close(y.cpu(), ref, "bfloat16" if xdt == torch.bfloat16 else "float16", what=_lib.last_kernel())


@pytest.mark.parametrize("m", [1, 16, 100])
def test_act_order_weight_in_the_cdna4_layout(m):
    """Its portable_row copy, sorted, serves it, the permutation read in the kernel."""
    n, k = 1024, 2048
    q, s, z, g_idx, x, ref = _act_order(m, n, k, 128, torch.bfloat16, m)
    packed = L.pack_w4(q, s, z, 128, L.CDNA4_W4, g_idx=g_idx).to(DEV)
    y = ops.w4a16_linear(x.to(DEV), packed)
    assert "gather" not in ops.last_kernel()
    assert_close(y.cpu(), ref, "bfloat16", what=f"cdna4 act-order {ops.last_kernel()}")
