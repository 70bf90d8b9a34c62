"""The 8-row form's workgroups that stay (wide matrices with a packed copy) against those of a tile each, bit for bit, and against 64 bits."""

from __future__ import annotations

import pytest
import torch

from tinyserve_llm_amd.ops import hip

BF = torch.bfloat16
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 3, 4, 8])
@pytest.mark.parametrize("n,k", [(32768, 1792), (34816, 2048), (33000, 3072), (32768, 3584), (98304, 4096),      # (the smallest reduction and the fewest rows that stay)
                                 (32768, 256), (32776, 1024), (128256, 1536), (32760, 2048), (32768, 4096), (98296, 4096), (32768, 8192)])      # (a tile each)
@pytest.mark.parametrize("out_dtype", [torch.float32, BF])
def test_workgroups_that_stay_add_up_as_those_of_a_tile_each(rows, n, k, out_dtype):
    g = torch.Generator(device="cuda").manual_seed(rows + n + k)
    x = torch.randn(rows, k, generator=g, device="cuda").to(BF)
    w = (torch.randn(n, k, generator=g, device="cuda") / 16).to(BF)
    packed = hip.pack_weight8(w)
    assert hip.skinny8_stays(n, k) == ((n, k) in ((32768, 1792), (34816, 2048), (33000, 3072), (32768, 3584), (98304, 4096)))
    got = hip.gemm_skinny8(x, w, out_dtype, packed)
    assert torch.equal(got, hip.gemm_skinny8(x, w, out_dtype))                                       # (without the copy: a tile a workgroup)
    assert torch.equal(got[:, 1024:2048], hip.gemm_skinny8(x, w[1024:2048], out_dtype, packed[128:256]))
    assert torch.equal(got, hip.gemm_skinny8(hip.pack_rows8(x, hip.skinny8_steps(k)), w, out_dtype, packed))
    want = x.double() @ w[-64:].double().t()
    torch.testing.assert_close(got[:, -64:].double(), want, rtol=2e-5 if out_dtype is torch.float32 else 2.0 ** -8, atol=1e-4 * k ** 0.5)


@pytest.mark.parametrize("rows", [1, 3, 4, 5, 8, 16, 17, 32, 33, 64, 65, 130])
@pytest.mark.parametrize("n,k", [(32832, 2048), (128256, 1024), (32768, 8192), (2048, 1024), (40000, 96)])
def test_capped_logits_have_the_bits_of_the_product_and_the_cap(rows, n, k, monkeypatch):
    """By the kernel that makes the product where it caps its sums itself, by a kernel of its own elsewhere."""
    from tinyserve_llm_amd.parts.ends import ProjectionHead
    g = torch.Generator(device="cuda").manual_seed(rows + n)
    x, w = torch.randn(rows, k, generator=g, device="cuda").to(BF), (torch.randn(n, k, generator=g, device="cuda") * 4 * k ** -0.5).to(BF)
    x[0, 3], w[5] = 0.0, 0.0
    if rows > 1:
        x[1] *= 1e3      # (sums far beyond the cap)
    head = ProjectionHead(n, k, softcap=20.0)
    head.bind({"weight": w})
    head.keep_streaming_copies()
    want = hip.soft_cap(hip.linear_bf16(x, w, torch.float32, head.weight_packed), 20.0)
    got = head.forward(x)
    assert torch.equal(got, want) and float(got.abs().max()) <= 20.0
    apart, general, made, run = [], [], hip.soft_cap, hip._run
    monkeypatch.setattr(hip, "soft_cap", lambda *args: apart.append(args) or made(*args))
    monkeypatch.setattr(hip, "_run", lambda name, rc: general.append(name) or run(name, rc))
    head.forward(x)
    first = {(32832, 2048): 1, (128256, 1024): 5}.get((n, k), 65)      # (1,024: too short a reduction for workgroups that stay, which up to 4 rows would be given to)
    assert (not apart) == (first <= rows <= 64) and (apart or not general)      # (capped: one call of the module, which refused nothing)
