"""What goes by the caches in large steps has the results of smaller ones, where it goes through them: decode attention over many keys and values
(DEC_ONCE_BYTES of attention_decode.hip), whether a request's pages are its own or shared, and experts' products (`hip.moe_weights_once`)."""

from __future__ import annotations

import pytest
import torch

from tinyserve_llm_amd.ops import hip

BF, I32 = torch.bfloat16, torch.int32
TOKENS, KEYS, KV, ONCE_BYTES = 32, 2048, 8, 48 << 20


def tables(layout, page, pages_per_entry):
    """[TOKENS, entries]: every request's own pages, everyone's the first's, or the first three entries shared by neighbours and the rest their own."""
    entries = -(-KEYS // (page * pages_per_entry))
    own = torch.randperm(TOKENS * entries, generator=torch.Generator().manual_seed(page)).view(TOKENS, entries).to(I32)
    if layout == "shared":
        return own[:1].expand(TOKENS, entries).contiguous()
    if layout == "begun together":
        own[1::2, :3] = own[::2, :3]
    return own


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["own", "shared", "begun together"])
@pytest.mark.parametrize("hd, page, pages_per_entry", [(64, 256, 1), (128, 128, 2), (32, 24, 1), (96, 64, 1)])
@pytest.mark.parametrize("chunk, waves", [(0, 0), (1024, 4), (2048, 2)])      # (0: a single step a wave)
@pytest.mark.parametrize("form", ["plain", "window", "capped", "sinks and gates"])
def test_a_token_s_result_does_not_depend_on_how_its_keys_come(layout, hd, page, pages_per_entry, chunk, waves, form):
    heads = 2 * KV
    if chunk == 0:
        waves = hip.decode_waves(hd, one_step=True)
        chunk = 32 * waves
    g = torch.Generator(device="cuda").manual_seed(hd + page)
    table = tables(layout, page, pages_per_entry).cuda()
    pool = (int(table.max()) + 1) * pages_per_entry
    k = torch.randn(pool, KV, page, hd, generator=g, device="cuda", dtype=BF).permute(0, 2, 1, 3)
    v = torch.randn(pool, KV, hd, page, generator=g, device="cuda", dtype=BF).permute(0, 3, 1, 2)
    q = torch.randn(TOKENS, heads, hd, generator=g, device="cuda").to(BF)
    positions = torch.tensor([KEYS - 1 - 37 * i for i in range(TOKENS - 4)] + [0, 31, 32, 700], dtype=I32, device="cuda")
    requests = torch.arange(TOKENS, dtype=I32, device="cuda")
    more = {"plain": {}, "window": dict(window=1024), "capped": dict(softcap=20.0), "sinks and gates": dict(sink=True, sinks=torch.randn(heads, generator=g, device="cuda"))}[form]
    gate = torch.randn(TOKENS, heads * hd, generator=g, device="cuda") if form == "sinks and gates" else None

    def attend(tokens):
        keys = min(-(-KEYS // chunk) * chunk, more.get("window", 1 << 30))
        assert (len(tokens) * KV * hd * 4 * keys >= ONCE_BYTES) == (len(tokens) == TOKENS)
        given = dict(more, gate=gate[tokens]) if gate is not None else more
        return hip.paged_attention_decode(q[tokens].contiguous(), k, v, table, requests[tokens].contiguous(), positions[tokens].contiguous(), hd ** -0.5, chunk=chunk, waves=waves,
                                          pages_per_entry=pages_per_entry, **given)
    if form == "window" and hd == 32:
        pytest.skip("the window keeps this step below the limit")
    everyone = attend(list(range(TOKENS)))
    for first in range(0, TOKENS, 5):
        part = list(range(first, min(first + 5, TOKENS)))
        assert torch.equal(attend(part), everyone[part])


@pytest.mark.gpu
@pytest.mark.parametrize("experts, top, tokens", [(4, 1, 4), (4, 1, 5), (4, 2, 31), (4, 2, 32), (16, 4, 4), (16, 4, 5), (16, 4, 63), (16, 4, 64)])
@pytest.mark.parametrize("n, k", [(48, 512), (131, 1120)])
def test_an_expert_s_rows_do_not_depend_on_how_its_matrices_come(experts, top, tokens, n, k):
    g = torch.Generator().manual_seed(experts + tokens + n)
    ids = torch.stack([torch.randperm(experts, generator=g)[:top] for _ in range(tokens)]).to(I32).cuda()
    x, w = torch.randn(tokens, k, generator=g).to(BF).cuda(), (torch.randn(experts, 2 * n, k, generator=g) * k ** -0.5).to(BF).cuda()
    assert hip.moe_weights_once(tokens * top, experts) == (experts < tokens * top < 16 * experts)
    for args in (dict(out_dtype=torch.float32), dict(out_dtype=BF, glu=(1.2, 1.702, 1.0)), dict(out_dtype=BF, activation="relu2")):
        together = hip.moe_gemm(x, w, hip.moe_group(ids, experts), per_token=True, **args).view(tokens, top, -1)
        for t in range(tokens):
            assert not hip.moe_weights_once(top, experts)
            assert torch.equal(hip.moe_gemm(x[t:t + 1], w, hip.moe_group(ids[t:t + 1].contiguous(), experts), per_token=True, **args), together[t])


def test_experts_matrices_go_by_the_caches_between_a_pair_and_a_tile_an_expert():
    once = hip.moe_weights_once
    assert not once(16, 16) and once(17, 16) and once(255, 16) and not once(256, 16) and not once(4, 128) and once(384, 64)
