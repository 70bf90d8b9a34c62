"""The 8-row form's workgroups that stay (wide matrices with a packed copy) against those of a tile each, bit for bit, and against 64 bits."""

from __future__ import annotations

import pytest
import torch

from tinyserve_llm_amd.ops import hip

BF = torch.bfloat16
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 3, 4, 8])
@pytest.mark.parametrize("n,k", [(32768, 256), (32776, 1024), (34816, 2048), (33000, 3072), (32768, 4096), (32768, 8192)])      # (8,192: a tile each)
@pytest.mark.parametrize("out_dtype", [torch.float32, BF])
def test_workgroups_that_stay_add_up_as_those_of_a_tile_each(rows, n, k, out_dtype):
    g = torch.Generator(device="cuda").manual_seed(rows + n + k)
    x = torch.randn(rows, k, generator=g, device="cuda").to(BF)
    w = (torch.randn(n, k, generator=g, device="cuda") / 16).to(BF)
    packed = hip.pack_weight8(w)
    got = hip.gemm_skinny8(x, w, out_dtype, packed)
    assert torch.equal(got, hip.gemm_skinny8(x, w, out_dtype))                                       # (without the copy: a tile a workgroup)
    assert torch.equal(got[:, 1024:2048], hip.gemm_skinny8(x, w[1024:2048], out_dtype, packed[128:256]))
    assert torch.equal(got, hip.gemm_skinny8(hip.pack_rows8(x, hip.skinny8_steps(k)), w, out_dtype, packed))
    want = x.double() @ w[-64:].double().t()
    torch.testing.assert_close(got[:, -64:].double(), want, rtol=2e-5 if out_dtype is torch.float32 else 2.0 ** -8, atol=1e-4 * k ** 0.5)
