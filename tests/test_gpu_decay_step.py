"""A step of one token a request through the decay states' own kernel: the bits of the kernel that walks requests of any length."""

from __future__ import annotations

import pytest
import torch

from tinyserve_llm_amd.ops import hip

F32 = torch.float32
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form,bonus", [("sigmoid_root", False), ("double_exponent", True), ("double_exponent", False)])
@pytest.mark.parametrize("dim,vdim", [(64, 64), (64, 128), (64, 192), (64, 256), (128, 64), (128, 128), (128, 256), (128, 512), (128, 320)])
@pytest.mark.parametrize("requests,heads", [(1, 1), (5, 3), (48, 2)])
def test_one_token_a_request(requests, heads, dim, vdim, form, bonus):
    g = torch.Generator(device="cuda").manual_seed(requests + dim + vdim)

    def r(*shape):
        return torch.randn(*shape, generator=g, device="cuda")
    fused = r(requests, 2 * heads * dim + heads * vdim + 4)      # (rows that lie apart, as columns of one product)
    q, k, v = fused[:, :heads * dim], fused[:, heads * dim:2 * heads * dim], fused[:, 2 * heads * dim:-4]
    z, z_bias = r(requests, heads * dim) * 3, r(heads * dim)
    if requests == 1:
        z[0, :2] = torch.tensor([100.0, -100.0])
    state = r(requests + 2, heads * dim * vdim + 8)
    slots = torch.randperm(requests + 2, generator=g, device="cuda")[:requests].to(torch.int32)
    cu = torch.arange(requests + 1, dtype=torch.int32, device="cuda")
    made = []
    for longest in (1, 2):      # (2: the walk)
        kept = state.clone()
        o = hip.decay_scan(q, k, v, z, z_bias, kept, cu, slots, heads, dim, vdim, form=form, tau=16.0, q_scale=dim ** -0.5,
                           bonus=state[0, :heads * dim].clone().view(heads, dim) if bonus else None, longest=longest)
        made.append((o, kept))
    assert torch.equal(made[0][0], made[1][0]) and torch.equal(made[0][1], made[1][1])
    assert not torch.equal(made[0][1], state)


@pytest.mark.parametrize("form,bonus", [("sigmoid_root", False), ("double_exponent", True)])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, F32])
@pytest.mark.parametrize("dim,vdim,shared,takes", [(64, 64, True, True), (64, 128, False, True), (64, 256, None, True), (128, 64, False, True), (128, 128, True, True),
                                                   (128, 256, False, True), (128, 512, False, False), (128, 192, True, False)])
@pytest.mark.parametrize("requests,heads", [(1, 1), (7, 3), (48, 2)])
def test_one_token_a_request_with_the_heads_norm_and_gate(requests, heads, dim, vdim, shared, takes, out_dtype, form, bonus):
    """The finishing kernel's bits of the sums that are left without it; weights of all heads, shared and none, rows of the gate that lie apart."""
    g = torch.Generator(device="cuda").manual_seed(requests + dim + vdim)

    def r(*shape):
        return torch.randn(*shape, generator=g, device="cuda")
    q, k, v, z, z_bias = r(requests, heads * dim), r(requests, heads * dim), r(requests, heads * vdim), r(requests, heads * dim) * 3, r(heads * dim)
    gate = r(requests, heads * vdim + 8)[:, 4:-4] * 4
    weight = None if shared is None else r(vdim if shared else heads * vdim)
    state = r(requests + 2, heads * dim * vdim)
    slots = torch.randperm(requests + 2, generator=g, device="cuda")[:requests].to(torch.int32)
    cu = torch.arange(requests + 1, dtype=torch.int32, device="cuda")
    kw = dict(form=form, tau=16.0, q_scale=dim ** -0.5, bonus=r(heads, dim) if bonus else None, longest=1)
    kept, other = state.clone(), state.clone()
    assert hip._decay_step_finishes(weight, gate, 1e-6, out_dtype, requests, heads, vdim) == takes
    got = hip.decay_scan(q, k, v, z, z_bias, kept, cu, slots, heads, dim, vdim, finish=(weight, gate, 1e-6, out_dtype), **kw)
    o = hip.decay_scan(q, k, v, z, z_bias, other, cu, slots, heads, dim, vdim, **kw)
    want = hip.mlstm_finish(o, weight, gate, heads, vdim, 1e-6, out_dtype, silu_gate=True)
    assert torch.equal(got, want) and torch.equal(kept, other)


@pytest.mark.parametrize("finish", [False, True])
def test_a_portion_in_chunks_beside_requests_that_feed_nothing(finish):
    """As many tokens as requests, and one the most of those that are not in chunks, but no step of a token a request. The bound: a number is a sum of some
    dim + 64 products beside what the state's 32-bit numbers carry; the norm divides by a root that is no less than the eps's."""
    from tests.test_gpu_fanotar import step_context
    least, dim = hip.DECAY_CHUNKS_FROM, 64
    lengths = [least, 1] + [0] * (least - 1)
    tokens = requests = sum(lengths)
    assert len(lengths) == requests
    g = torch.Generator(device="cuda").manual_seed(3)
    q, k, v, z, gate = (torch.randn(tokens, dim, generator=g, device="cuda") for _ in range(5))
    z_bias, start = torch.randn(dim, generator=g, device="cuda"), torch.randn(requests, dim * dim, generator=g, device="cuda")
    cu = torch.tensor([0, least] + [tokens] * requests, dtype=torch.int32, device="cuda")[:requests + 1]
    slots, made = torch.arange(requests, dtype=torch.int32, device="cuda"), []
    for ctx in (step_context([[0]] * requests, 4096, [0] * requests, lengths, slots=list(range(requests))), None):
        state = start.clone()
        o = hip.decay_scan(q, k, v, z, z_bias, state, cu, slots, 1, dim, dim, form="sigmoid_root", tau=16.0, q_scale=dim ** -0.5, longest=least, ctx=ctx,
                           finish=(None, gate, 1.0, F32) if finish else None)
        made.append((o, state))
    for got, want in zip(*made):
        torch.testing.assert_close(got, want, atol=4 * (dim + 64) * 2.0 ** -24 * float(want.abs().max()), rtol=1e-4)
