"""Head norms and turns by whole pieces of four numbers, against the kernels that take them one by one (which a start that no piece lies at goes to)."""

from __future__ import annotations

import pytest
import torch

from tinyserve_llm_amd.ops import hip

BF = torch.bfloat16


def askew(t: torch.Tensor) -> torch.Tensor:
    """The same numbers from a start that is one number off a 16-byte border."""
    return torch.cat([t.new_zeros(1), t.flatten()])[1:].view(t.shape)


@pytest.mark.gpu
@pytest.mark.parametrize("heads, kv_heads, hd, vd", [(32, 8, 64, 64), (1, 1, 4, 8), (3, 2, 20, 24), (5, 1, 80, 160), (7, 3, 256, 256), (6, 2, 128, 512), (2, 2, 64, 12)])
@pytest.mark.parametrize("interleaved", [False, True])
@pytest.mark.parametrize("which", ["qkv", "q", "k", "v", "qk"])
def test_prepared_heads(heads, kv_heads, hd, vd, interleaved, which):
    """A norm's squares are added in another order: at most (hd / 4 + 8) roundings of 2^-24 in the mean square, half of that in its root, and two more."""
    gen = torch.Generator().manual_seed(hd + vd)
    positions = torch.tensor([0, 1, 63, 700, 70000], dtype=torch.int32).cuda()
    rows = (torch.randn(5, (heads + kv_heads) * hd + kv_heads * vd, generator=gen) * 3).cuda()
    wq, wk = ((1 + 0.2 * torch.randn(hd, generator=gen)).cuda() for _ in range(2))
    freqs = (9000.0 ** (-torch.arange(vd // 2, dtype=torch.float64) * 2 / vd)).cuda()
    got, want = rows.clone(), askew(rows)
    for at in (got, want):
        hip.qkv_prepare(at, positions, heads, kv_heads, hd, vd, q_weight=wq if "q" in which else None, k_weight=wk if "k" in which else None, eps=1e-5,
                        value_freqs=freqs if "v" in which else None, value_interleaved=interleaved)
    normed = (heads + kv_heads) * hd
    assert torch.equal(got[:, normed:], want[:, normed:])
    torch.testing.assert_close(got[:, :normed], want[:, :normed], rtol=(hd / 8 + 8) * 2.0 ** -24, atol=0.0)
    for cut, changed in ((slice(0, heads * hd), "q" in which), (slice(heads * hd, normed), "k" in which), (slice(normed, None), "v" in which)):
        assert torch.equal(got[:, cut], rows[:, cut]) != changed


@pytest.mark.gpu
@pytest.mark.parametrize("heads, rot, width", [(32, 64, 64), (3, 40, 48), (5, 32, 64), (6, 128, 128), (3, 24, 40), (9, 16, 16)])
@pytest.mark.parametrize("interleaved", [False, True])
@pytest.mark.parametrize("src_type, dst_type", [(torch.float32, torch.float32), (torch.float32, BF), (BF, BF)])
def test_turned_heads(heads, rot, width, interleaved, src_type, dst_type):
    gen = torch.Generator().manual_seed(heads + rot)
    n = -(-(1 << 20) // (heads * rot // 2))      # (fewer pairs go to the other kernel)
    positions = torch.randint(0, 70000, (n,), generator=gen, dtype=torch.int32).cuda()
    src = (torch.randn(n, heads, width, generator=gen) * 3).to(src_type).cuda()
    freqs, gate = (9000.0 ** (-torch.arange(rot // 2, dtype=torch.float64) * 2 / rot)).cuda(), torch.randn(n, heads + 3, generator=gen).cuda()[:, 3:]
    for back, g in ((False, None), (True, gate)):
        got, want = torch.zeros(n, heads, width, dtype=dst_type, device="cuda"), torch.zeros(n, heads, width, dtype=dst_type, device="cuda")
        hip.rotate_heads(got, src, freqs, 1.25, positions, interleaved=interleaved, back=back, gate=g)
        hip.rotate_heads(want, askew(src), freqs, 1.25, positions, interleaved=interleaved, back=back, gate=g)
        assert torch.equal(got, want) and bool(got[:, :, :rot].any()) and not bool(got[:, :, rot:].any())
        if src_type == dst_type:
            inside = src.clone()
            hip.rotate_heads(inside, inside, freqs, 1.25, positions, interleaved=interleaved, back=back, gate=g)
            assert torch.equal(inside[:, :, :rot], got[:, :, :rot]) and torch.equal(inside[:, :, rot:], src[:, :, rot:])
