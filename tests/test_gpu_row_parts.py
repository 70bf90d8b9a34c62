"""Rows in parts (`hip.RowParts`) through the stream's kernels: the bits of the sum made first by a kernel of its own."""

from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch

from tinyserve_llm_amd.ops import hip
from tinyserve_llm_amd.parts.gated_delta import GatedDelta
from tinyserve_llm_amd.parts.norm import RMSNorm
from tinyserve_llm_amd.parts.stream import ResidualStream

BF, F32 = torch.bfloat16, torch.float32
pytestmark = pytest.mark.gpu


def make(n, width, count):
    g = torch.Generator(device="cuda").manual_seed(n + width + 7 * count)

    def r(*shape):
        return torch.randn(*shape, generator=g, device="cuda")
    parts = hip.RowParts((r(n, width), r(n, width)), (0.7, -1.1)) if count == 0 else hip.RowParts(r(count, n, width))
    return r(n, width), parts, r(n, width), r


@pytest.mark.parametrize("count", [0, 1, 2, 3, 4, 5, 9])      # (0: two mixers' rows with their factors)
@pytest.mark.parametrize("n,width", [(1, 64), (3, 1020), (5, 1024), (7, 1028), (130, 2048), (2, 2052), (3, 4096), (2, 4100)])
def test_parts_are_added_up_where_the_stream_takes_them(n, width, count):
    x, parts, a, r = make(n, width, count)
    post, scale, w = r(width), r(width), r(width)
    for out_dtype, weight, sc in ((BF, w, scale), (F32, w, None), (BF, None, None), (None, None, scale)):
        got, want = x.clone(), x.clone()
        rows = hip.stream_post_norm(got, parts, post, sc, 1e-5, weight, 1e-6, out_dtype)
        rows_want = hip.stream_post_norm(want, parts.rows(), post, sc, 1e-5, weight, 1e-6, out_dtype)
        assert torch.equal(got, want) and (rows is None) == (rows_want is None) and (rows is None or torch.equal(rows, rows_want))
    for first, weight, out_dtype in ((None, w, BF), (a, w.to(BF), BF), (a, w, F32), (a.to(BF), w, BF)):
        got, want = x.clone(), x.clone()
        rows, _ = hip.stream_update_norm(got, first, parts, None, 0.5, (weight, None), 1e-5, out_dtype=out_dtype)
        rows_want, _ = hip.stream_update_norm(want, first, parts.rows(), None, 0.5, (weight, None), 1e-5, out_dtype=out_dtype)
        assert torch.equal(got, want) and torch.equal(rows, rows_want)
    for first in (None, a, a.to(BF)):
        assert torch.equal(hip.stream_join(x, first, parts, a, BF), hip.stream_join(x, first, parts.rows(), a, BF))


def test_a_stream_keeps_parts_pending_in_either_place():
    x, parts, a, r = make(9, 256, 3)
    norm = RMSNorm(256, 1e-5)
    norm.bind({"weight": r(256).to(BF)})
    for one, other in ((parts, None), (None, parts), (a, parts), (parts, a), (parts, parts)):
        got, rows = ResidualStream(x.clone(), one, other).take(norm)
        want, rows_want = ResidualStream(x.clone(), hip.added_up(one), hip.added_up(other)).take(norm)
        assert torch.equal(got, want) and torch.equal(rows, rows_want)
        assert torch.equal(ResidualStream(x.clone(), one, other).joined_with(a, BF), ResidualStream(x.clone(), hip.added_up(one), hip.added_up(other)).joined_with(a, BF))
        assert torch.equal(ResidualStream(x.clone(), one, other).settle()[0], ResidualStream(x.clone(), hip.added_up(one), hip.added_up(other)).settle()[0])


@pytest.mark.parametrize("rows,n,k", [(160, 2048, 8192), (700, 2048, 8192), (1000, 1024, 4096), (2048, 2048, 8192), (129, 1032, 2112)])
def test_a_product_in_slices_leaves_its_parts(rows, n, k):
    g = torch.Generator(device="cuda").manual_seed(rows)
    x, w = torch.randn(rows, k, generator=g, device="cuda").to(BF), torch.randn(n, k, generator=g, device="cuda").to(BF)
    plan = hip.many_rows_plan(rows, n, k, "f32")
    parts = hip.linear_parts(x, w)
    assert (parts is not None) == (plan is not None and plan[1] > 1)
    if parts is not None:
        assert torch.equal(parts.rows(), hip.linear_bf16(x, w, F32))
    assert hip.linear_parts(x[:, ::2], w[:, : k // 2]) is None      # (rows that are not dense)


@pytest.mark.parametrize("rows", [300, 999, 1280, 2048])
def test_a_part_that_leaves_parts_leaves_those_of_its_own_rows(rows, monkeypatch):
    """The delta rule's output projection (4,096 into 2,048): in parts only where the product made whole is in the same slices, so the bits are those of its rows."""
    g = torch.Generator(device="cuda").manual_seed(rows)
    mixer = GatedDelta(hidden_size=2048, num_heads=32, groups=16, head_dim=128, value_dim=128, conv_taps=4, norm_eps=1e-5)
    mixer.proj = torch.randn(64, 2048, generator=g, device="cuda").to(BF)
    mixer.o = torch.randn(2048, 4096, generator=g, device="cuda").to(BF)
    gated = torch.randn(rows, 4096, generator=g, device="cuda").to(BF)
    for name, made in (("delta_prepare", None), ("delta_scan", None), ("mlstm_finish", gated)):
        monkeypatch.setattr(hip, name, lambda *args, _made=made, **options: _made)
    memory = SimpleNamespace(state=None)
    x = torch.randn(rows, 2048, generator=g, device="cuda").to(BF)
    assert torch.equal(hip.added_up(mixer.forward(x, None, memory, parts=True)), mixer.forward(x, None, memory))


@pytest.mark.parametrize("top,identity,shared", [(1, False, None), (2, True, "gated"), (4, True, "plain"), (4, False, "gated"), (5, True, None), (9, True, "plain")])
@pytest.mark.parametrize("n,width", [(1, 64), (7, 1028), (48, 2048), (130, 2052), (3, 4096), (2, 4100)])
def test_experts_rows_are_added_up_where_the_stream_takes_them(n, width, top, identity, shared):
    g = torch.Generator(device="cuda").manual_seed(n + width + top)

    def r(*shape):
        return torch.randn(*shape, generator=g, device="cuda")
    ids = torch.randint(0, 6, (n, top), generator=g, device="cuda", dtype=torch.int32)
    pairs = r(n * top, width)
    if identity:
        pairs[ids.view(-1) >= 4] = float("nan")      # (an identity expert's pairs are in no tile)
    x, post, scale, w = r(n, width), r(width), r(width), r(width)
    for kind in (BF, F32):      # (a 32-bit input of identity experts is added up before)
        left = hip.ExpertRows(pairs, r(n, top), r(n, width) if shared else None, (ids, 4, r(n, width).to(kind)) if identity else None, r(n, 1) if shared == "gated" else None)
        for out_dtype, weight, sc in ((BF, w, scale), (F32, w, None), (BF, None, None), (None, None, scale)):
            got, want = x.clone(), x.clone()
            rows = hip.stream_post_norm(got, left, post, sc, 1e-5, weight, 1e-6, out_dtype)
            rows_want = hip.stream_post_norm(want, left.rows(), post, sc, 1e-5, weight, 1e-6, out_dtype)
            assert torch.equal(got, want) and (rows is None) == (rows_want is None) and (rows is None or torch.equal(rows, rows_want))
    assert not torch.isnan(left.rows()).any()
    norm = RMSNorm(width, 1e-5)
    norm.bind({"weight": w.to(BF)})
    for one, other in ((left, None), (None, left), (x, left)):
        got, rows = ResidualStream(x.clone(), one, other).take(norm)
        want, rows_want = ResidualStream(x.clone(), hip.added_up(one), hip.added_up(other)).take(norm)
        assert torch.equal(got, want) and torch.equal(rows, rows_want)
