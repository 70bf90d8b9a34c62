"""The experts' products of narrow tiles by whole lines (`moe_gemm_lines_kernel`): reductions of one stage to many, columns that end inside a
workgroup's, tiles of 1 to 16 rows, against 64 bits, a row's bits whatever its batch, and those of the kernel for other reductions."""

from __future__ import annotations

import pytest
import torch

from tinyserve_llm_amd.ops import hip

BF, F32 = torch.bfloat16, torch.float32
pytestmark = pytest.mark.gpu
E = 5


def present(experts):
    return [p for p, e in enumerate(experts) if e < E]


@pytest.mark.parametrize("once", [False, True])
@pytest.mark.parametrize("n,k", [(16, 256), (40, 512), (24, 768), (72, 1024), (33, 1280), (64, 3072)])
@pytest.mark.parametrize("tokens", [1, 3, 7, 19])
def test_products_by_lines(monkeypatch, tokens, n, k, once):
    monkeypatch.setattr(hip, "moe_weights_once", lambda pairs, experts: once)
    g = torch.Generator(device="cuda").manual_seed(tokens + n + k)
    top = 2
    ids = torch.randint(0, E + 1, (tokens, top), generator=g, device="cuda", dtype=torch.int32)      # (E: an identity expert, in no tile)
    ids[:, 1] = (ids[:, 0] + 1 + ids[:, 1] % E) % (E + 1)
    grouped = hip.moe_group(ids, E)
    x = torch.randn(tokens, k, generator=g, device="cuda").to(BF)
    rows = torch.randn(tokens * top, k, generator=g, device="cuda").to(BF)
    w = (torch.randn(E, 2 * n, k, generator=g, device="cuda") / k ** 0.5).to(BF)
    flat = ids.flatten().tolist()
    gated = hip.moe_gemm(x, w, grouped, BF, per_token=True, glu=(5.0, 1.0, 0.5))
    plain = hip.moe_gemm(rows, w[:, :n].contiguous(), grouped, F32, per_token=False)
    squared = hip.moe_gemm(rows, w[:, :n].contiguous(), grouped, BF, per_token=False, activation="relu2")
    for p, e in enumerate(flat):
        if e >= E:
            continue
        sums = w[e].double() @ x[p // top].double()
        gate, up = sums[:n].clamp(max=5.0), sums[n:].clamp(-5.0, 5.0)
        torch.testing.assert_close(gated[p].double(), gate * torch.sigmoid(gate) * (up + 0.5), rtol=2.0 ** -8, atol=1e-4)
        want = w[e, :n].double() @ rows[p].double()
        torch.testing.assert_close(plain[p].double(), want, rtol=1e-5, atol=2e-6 * k ** 0.5)
        torch.testing.assert_close(squared[p].double(), want.clamp(min=0.0) ** 2, rtol=2.0 ** -8, atol=1e-4)
    # a step of zeros behind each quarter of the reduction makes it the other kernel's, whose sums are the same, bit for bit
    spread = lambda t: torch.nn.functional.pad(t.reshape(*t.shape[:-1], 4, k // 4), (0, 32)).flatten(-2).contiguous()
    assert (k + 128) % 256
    assert torch.equal(gated[present(flat)], hip.moe_gemm(spread(x), spread(w), grouped, BF, per_token=True, glu=(5.0, 1.0, 0.5))[present(flat)])
    assert torch.equal(plain[present(flat)], hip.moe_gemm(spread(rows), spread(w[:, :n]), grouped, F32, per_token=False)[present(flat)])
    # a token by itself: the same bits
    alone = hip.moe_group(ids[-1:].contiguous(), E)
    last = hip.moe_gemm(x[-1:].contiguous(), w, alone, BF, per_token=True, glu=(5.0, 1.0, 0.5))
    for j in range(top):
        if flat[-top + j] < E:
            assert torch.equal(last[j], gated[(tokens - 1) * top + j])
