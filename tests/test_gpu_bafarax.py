"""The Bafarax decoder on the GPU against the plain implementation in tests/plain/bafarax.py: each
mechanism's kernel alone (with inputs made so that a fault shows: a far key whose score stands out, keys
just inside and just outside a chunk or a window, at page borders, the first tokens where the sink weighs
most, gates at their caps, states carried over steps and slots), then whole models of four small
configurations through trace replay (layer by layer, whole, token by token, in portions down to two
tokens, mixed batches on pages and state slots that are used again, long decoding), and greedy
generation through `LLM.generate` and the scheduler. float32 and bfloat16."""

from __future__ import annotations

import itertools
import math

import pytest
import torch

from tests.helpers import bafarax_configs, prompt
from tests.plain import bafarax as plain
from tests.test_gpu_fanotar import paged, rounded, step_context, tolerance

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
F64 = torch.float64


def hip():
    from tinyserve_llm_amd.ops import hip as h
    return h


# ---- the norm with 1 + weight, norms over stretches of a row, rotations ----------------------------

@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("width", [80, 99, 256])
def test_norm_stored_around_zero_on_the_stream(dtype, width):
    from tinyserve_llm_amd.parts.norm import RMSNorm
    from tinyserve_llm_amd.parts.stream import ResidualStream
    n, eps = 7, 1e-5
    x = torch.randn(n, width) * 3
    a, a64 = rounded(torch.randn(n, width), dtype)
    w, w64 = rounded(torch.randn(width) * 0.2, dtype)                     # stored around zero, in the weights' type
    norm = RMSNorm(width, eps, one_plus=True)
    norm.bind({"weight": w})
    xd = x.to(DEV)
    h, _ = norm(ResidualStream(xd, a))
    want = x.to(F64) + a64
    torch.testing.assert_close(xd.cpu().to(F64), want, atol=2e-6, rtol=1e-6)
    assert h.dtype == dtype
    torch.testing.assert_close(h.cpu().to(F64), plain.layer_norm(want, w64, eps), **tolerance(dtype))
    rows = torch.tensor([5, 0, 5], dtype=torch.int32, device=DEV)
    picked, _ = norm(ResidualStream(xd), None, rows)
    torch.testing.assert_close(picked.cpu().to(F64), plain.layer_norm(want[[5, 0, 5]], w64, eps), **tolerance(dtype))
    with pytest.raises(TypeError):
        norm(a)                                                            # (only a 32-bit stream)


@pytest.mark.parametrize("sizes", [(128, 64, 96), (60, 60, 84), (22, 40, 6), (2048, 512, 512)])
def test_norm_over_a_whole_projection_in_place(sizes):
    h = hip()
    q, k, v = sizes
    rows = torch.randn(9, q + k + v) * 2
    wq, wk = 1 + 0.1 * torch.randn(q), 1 + 0.1 * torch.randn(k)
    d = rows.to(DEV)
    h.segment_rmsnorm(d, 0, q, wq.to(DEV), 1e-5, out=d[:, :q])
    h.segment_rmsnorm(d, q, k, wk.to(DEV), 1e-5, out=d[:, q:q + k])
    r = rows.to(F64)
    torch.testing.assert_close(d[:, :q].cpu().to(F64), plain.unit_rms(r[:, :q], 1e-5) * wq.to(F64), atol=5e-6, rtol=1e-5)
    torch.testing.assert_close(d[:, q:q + k].cpu().to(F64), plain.unit_rms(r[:, q:q + k], 1e-5) * wk.to(F64), atol=5e-6, rtol=1e-5)
    assert torch.equal(d[:, q + k:].cpu(), rows[:, q + k:]), "the values are left as they are"
    both = rows.to(DEV)
    h.segment_rmsnorm_pair(both, (0, q, wq.to(DEV)), (q, k, wk.to(DEV)), 1e-5)              # the two in one launch
    assert torch.equal(both, d)
    out = h.segment_rmsnorm(rows.to(DEV), q, k, None, 0.0, out_dtype=torch.bfloat16)
    torch.testing.assert_close(out.cpu().to(F64), plain.unit_rms(r[:, q:q + k], 0.0), atol=2e-2, rtol=1e-2)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shape", [(4, 2, 32, 48, 16, None), (3, 1, 20, 12, 10, None), (8, 2, 64, 64, 64, (4.0, 64.0, 16.0, 1.0)),
                                   (2, 2, 16, 16, 0, None)])
def test_heads_turn_in_halves_with_an_amplitude_and_reach_the_cache(dtype, shape):
    """q | k | v rows to rotated query heads and the cache: pairs (i, i + rot/2), only the first `rot` dimensions of a head,
    far positions (the angle is taken in 64-bit), a frequency ramp's amplitude on cosine and sine."""
    h = hip()
    H, G, D, V, rot, ramp = shape
    ramp = dict(zip(("factor", "original", "fast", "slow"), ramp)) if ramp else None
    page, positions = 16, [0, 1, 15, 16, 17, 700, 70000]
    freqs, amp = plain.rotary_frequencies(rot, 9000.0, ramp) if rot else (None, 1.0)
    rows = torch.randn(len(positions), (H + G) * D + G * V)
    k, v = paged(6, page, G, D, V, dtype)
    slots = [3 * page + 1, 0, 5 * page + 15, 17, 2 * page, 4 * page + 7, 4 * page + 8]
    dev = lambda t: torch.tensor(t, dtype=torch.int32, device=DEV)
    q = h.qkv_finish(rows.to(DEV), freqs.to(DEV) if rot else None, dev(positions), dev(slots), k, v, H, G, D, V, dtype,
                     interleaved=False, amplitude=amp)
    r = rows.to(F64)
    pos = torch.tensor(positions)
    f = freqs if rot else torch.zeros(0, dtype=F64)
    want_q = plain.rotate(r[:, :H * D].reshape(-1, H, D), pos, f, amp, False)
    want_k = plain.rotate(r[:, H * D:(H + G) * D].reshape(-1, G, D), pos, f, amp, False)
    tol = dict(atol=2e-5, rtol=1e-5) if dtype == torch.float32 else dict(atol=3e-2, rtol=1e-2)
    torch.testing.assert_close(q.cpu().to(F64), want_q, **tol)
    for i, s in enumerate(slots):
        torch.testing.assert_close(k[s // page, s % page].cpu().to(F64), want_k[i], **tol)
        torch.testing.assert_close(v[s // page, s % page].cpu().to(F64), r[i, (H + G) * D:].reshape(G, V), **tol)


@pytest.mark.parametrize("shape", [(1, 1, 32, 16, 32, False), (4, 2, 64, 64, 64, False), (8, 2, 64, 32, 48, True), (5, 1, 96, 128, 64, False),
                                   (2, 1, 256, 256, 256, True), (3, 1, 40, 8, 0, False), (16, 16, 24, 32, 6, True)])
@pytest.mark.parametrize("few", [1, 3, 23, 127])
def test_a_step_of_few_tokens_finishes_like_one_of_many(few, shape):
    """The kernel for few tokens against the one for many on the same rows: every head, tokens that share a workgroup, a last
    workgroup that is not full. The same 32-bit operations; a product and a sum may be contracted in either order, half a
    step of the larger term each, beside the root's."""
    h = hip()
    H, G, D, V, rot, inter = shape
    page, many = 16, 1100
    gen = torch.Generator().manual_seed(few + D)
    rows = torch.randn(many, (H + G) * D + G * V, generator=gen).to(DEV)
    positions = torch.randint(0, 90000, (many,), generator=gen, dtype=torch.int32).to(DEV)
    slots = torch.randperm(70 * page, generator=gen)[:many].to(torch.int32)
    slots[1::7] = -1                                                       # (rows that leave nothing in the cache)
    slots = slots.to(DEV)
    freqs = plain.rotary_frequencies(rot, 9000.0, None)[0].to(DEV) if rot else None
    found = []
    for n in (few, many):
        k, v = paged(70, page, G, D, V, torch.float32)
        k.zero_(), v.zero_()
        q = h.qkv_finish(rows[:n], freqs, positions[:n].contiguous(), slots[:n].contiguous(), k, v, H, G, D, V, torch.float32,
                         interleaved=inter, qk_norm_eps=1e-5 if D != 96 else None, amplitude=1.25)
        at = slots[:few][slots[:few] >= 0].long()
        found.append((q[:few], k[at // page, at % page], v[at // page, at % page], k.count_nonzero() if n == few else None))
    for a, b in zip(found[0][:3], found[1][:3]):
        torch.testing.assert_close(a, b, rtol=0.0, atol=2.0 ** -21 * 8)
    assert int(found[0][3]) <= found[0][1].numel(), "nothing but the step's own slots is written"


@pytest.mark.parametrize("few", [256, 257, 700, 1023])
@pytest.mark.parametrize("shape", [(1, 1, 32, 32, 32, False), (1, 1, 24, 32, 24, True), (2, 1, 32, 8, 16, False)])
def test_steps_of_few_tokens_whose_values_leave_apart(few, shape):
    """From 256 tokens on the values leave through their own kernel, and a token of one query and one key head gives a
    workgroup of the kernel for few tokens 32 tokens' angles at once, the most that its table must hold."""
    test_a_step_of_few_tokens_finishes_like_one_of_many(few, shape)


# ---- attention inside chunks with learned sinks -----------------------------------------------------

def chunk_case(dtype, H, G, D, V, page, length, queries, stand_out, scale, chunk, seed=0, sink_value=None, portion_from=None):
    """Keys and values of one request of `length` tokens on shuffled pages, queries at the positions `queries`, each a
    decoded token of a request of its own over the same pages; with `portion_from`, one request instead that feeds the
    positions from there to the end as one portion of a prompt (0: the whole prompt), every position a query.
    `stand_out` maps a query's position to the key position whose score is made to stand out for it. Returns
    (kernel output, oracle output, values, query positions)."""
    h = hip()
    if portion_from is not None:
        queries = list(range(portion_from, length))
        stand_out = {q: key for q, key in stand_out.items() if q >= portion_from}
    gen = torch.Generator().manual_seed(seed)
    k64 = plain.unit_rms(torch.randn(length, G, D, generator=gen, dtype=F64), 0.0)
    v64 = torch.randn(length, G, V, generator=gen, dtype=F64)
    q64 = plain.unit_rms(torch.randn(len(queries), H, D, generator=gen, dtype=F64), 0.0)
    for i, p in enumerate(queries):
        if p in stand_out:
            g_dir = plain.unit_rms(torch.randn(G, D, generator=gen, dtype=F64), 0.0)
            for hh in range(H):
                q64[i, hh] = g_dir[hh // (H // G)]
            k64[stand_out[p]] = 11.0 / (D * scale) * g_dir                     # q.k * scale = 11
    sinks = torch.randn(H, generator=gen, dtype=F64) if sink_value is None else torch.full((H,), sink_value, dtype=F64)
    pages = -(-length // page)
    table = torch.randperm(pages + 3, generator=gen)[:pages].tolist()
    k, v = paged(pages + 3, page, G, D, V, dtype)
    kr, vr = k64.to(dtype), v64.to(dtype)
    at = torch.arange(length)
    pg, off = torch.tensor(table)[at // page].to(DEV), (at % page).to(DEV)
    k[pg, off], v[pg, off] = kr.to(DEV), vr.to(DEV)
    q = q64.to(dtype).to(DEV)
    if portion_from is None:
        ctx = step_context([table] * len(queries), page, queries, [1] * len(queries))
    else:
        ctx = step_context([table], page, [portion_from], [len(queries)])
    out = h.paged_attention(q, k, v, ctx, 0, scale, 0, sinks=sinks.float().to(DEV), chunk_mask=chunk)
    want = plain.masked_attention(q.cpu().to(F64), kr.to(F64), vr.to(F64), torch.tensor(queries), scale,
                                  "chunk" if chunk else "full", chunk, sinks.float().to(F64))
    return out.cpu().to(F64), want, vr.to(F64), queries


FORMS = {"decoded": None, "prompt": 0, "portion": 130}       # (a portion that starts inside a page)


def decides(want_row, value_row) -> bool:
    return float((want_row - value_row).abs().max()) < 0.2 * float(value_row.abs().max())


@pytest.mark.parametrize("form", sorted(FORMS))
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("chunk, sizes", [(1, (4, 2, 32, 40)), (7, (4, 2, 32, 40)), (16, (4, 2, 32, 40)), (24, (4, 2, 32, 40)),
                                          (64, (8, 2, 64, 64)), (100, (4, 2, 32, 40)), (33, (8, 2, 64, 64)), (65, (4, 4, 64, 64)),
                                          (130, (4, 1, 64, 64)), (96, (2, 2, 128, 128)), (257, (6, 2, 32, 32)), (3, (3, 1, 20, 12))])
def test_chunk_edges(dtype, chunk, sizes, form):
    """The key that stands out is the first of the query's chunk for some queries (the farthest key they see) and the last
    of the chunk before for others (then it must not count at all): at chunks shorter and longer than a page, than a wave's
    stretch of keys and than a matrix-core tile, for decoded tokens, a whole prompt and a portion of one. Chunks count from
    position 0 of the request wherever the portion starts."""
    (H, G, D, V), page = sizes, 16
    length = max(600, 8 * chunk + 15)
    # (queries whose key stands out lie in chunks of their own, so that none sees another's)
    inside = {(c + 1) * chunk - 1: c * chunk for c in (1, 3)}              # the chunk's last position and its first key
    outside = {c * chunk + chunk // 2: c * chunk - 1 for c in (5, 7)}      # the last key of the chunk before
    queries = sorted({0, 127, 128, 129, *inside, *outside})
    out, want, v, queries = chunk_case(dtype, H, G, D, V, page, length, queries, {**inside, **outside}, D ** -0.5, chunk,
                                       sink_value=-3.0, portion_from=FORMS[form])
    torch.testing.assert_close(out, want, **tolerance(dtype))
    # the test is sharp: an inside key decides its row, an outside key leaves the row to the others
    for q, key in inside.items():
        if q in queries:
            assert decides(want[queries.index(q), 0], v[key, 0]), (q, key)
    for q, key in outside.items():
        if q in queries and chunk > 1:
            assert not decides(want[queries.index(q), 0], v[key, 0]), (q, key)


@pytest.mark.parametrize("form", sorted(FORMS))
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("sizes", [(4, 2, 32, 48), (2, 2, 16, 16), (6, 1, 24, 8), (8, 4, 64, 64), (4, 4, 128, 128)])
def test_far_keys_and_page_borders_without_chunks_and_inside_a_long_chunk(dtype, sizes, form):
    H, G, D, V = sizes
    page, length = 16, 700
    stand_out = {699: 3, 650: 15, 651: 16, 652: 17, 653: 653, 500: 255, 501: 256, 31: 0}
    queries = [0, 1, 2, 3, 15, 16, 17, 31, 500, 501, 650, 651, 652, 653, 699]
    for chunk in (0, 1000):
        out, want, v, qs = chunk_case(dtype, H, G, D, V, page, length, queries, stand_out, D ** -0.5, chunk, portion_from=FORMS[form])
        torch.testing.assert_close(out, want, **tolerance(dtype))
        assert decides(want[qs.index(699), 0], v[3, 0]), "the far key decides the row"


def test_the_learned_sink_weighs_most_on_the_first_tokens_of_every_chunk():
    # a large sink takes nearly all the weight where there are few keys: at position 0 and again where a chunk starts
    out, want, v, _ = chunk_case(torch.float32, 4, 2, 32, 32, 16, 40, [0, 1, 19, 20, 39], {}, 32 ** -0.5, 20, sink_value=6.0)
    torch.testing.assert_close(out, want, atol=2e-5, rtol=1e-5)
    assert float(out[0].abs().max()) < 0.02 * float(v[0].abs().max()) and float(out[3].abs().max()) < 0.02 * float(v[20].abs().max())
    # and a sink far below the scores changes nothing: the weights sum to one
    out, _, v, _ = chunk_case(torch.float32, 4, 2, 32, 32, 16, 40, [0, 20], {}, 32 ** -0.5, 20, sink_value=-40.0)
    torch.testing.assert_close(out[0, 0], v[0, 0], atol=1e-5, rtol=1e-5)
    torch.testing.assert_close(out[1, 3], v[20, 1], atol=1e-5, rtol=1e-5)


# ---- attention through a latent ----------------------------------------------------------------------

@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("sizes", [(36, 40, 8, None), (16, 16, 16, None), (22, 34, 6, (8.0, 32.0, 4.0, 1.0)), (192, 256, 32, None),
                                   (96, 128, 0, None), (7, 512, 128, (3.0, 64.0, 16.0, 2.0))])
def test_latent_norms_shared_key_part_and_cache_rows(dtype, sizes):
    h = hip()
    q_rank, rank, rot, ramp = sizes
    ramp = dict(zip(("factor", "original", "fast", "slow"), ramp)) if ramp else None
    page, positions = 16, [0, 1, 15, 16, 17, 700, 70000]
    freqs, amp = plain.rotary_frequencies(rot, 5000.0, ramp) if rot else (None, 1.0)
    extra = 11                                                              # (a gate's columns behind: left alone)
    down = torch.randn(len(positions), q_rank + rank + rot + extra) * 2
    wq, wc = 1 + 0.1 * torch.randn(q_rank), 1 + 0.1 * torch.randn(rank)
    cache = torch.zeros(6, page, 1, rank + rot, dtype=dtype, device=DEV)
    values = torch.zeros(6, 1, rank, page, dtype=dtype, device=DEV).permute(0, 3, 1, 2)      # transposed inside a page
    slots = [3 * page + 1, 0, 5 * page + 15, 17, 2 * page, 4 * page + 7, 4 * page + 8]
    dev = lambda t: torch.tensor(t, dtype=torch.int32, device=DEV)
    d = down.to(DEV)
    cq = h.latent_finish(d, 0, q_rank, q_rank, rank, rot, wq.to(DEV), wc.to(DEV), 1e-5, freqs.to(DEV) if rot else None, amp,
                         dev(positions), dev(slots), cache, dtype, v_cache=values)
    r = down.to(F64)
    tol = dict(atol=2e-5, rtol=1e-5) if dtype == torch.float32 else dict(atol=3e-2, rtol=1e-2)
    torch.testing.assert_close(cq.cpu().to(F64), plain.unit_rms(r[:, :q_rank], 1e-5) * wq.to(F64), **tol)
    c = plain.unit_rms(r[:, q_rank:q_rank + rank], 1e-5) * wc.to(F64)
    kr = plain.rotate(r[:, q_rank + rank:q_rank + rank + rot], torch.tensor(positions), freqs if rot else torch.zeros(0, dtype=F64), amp, True)
    for i, s in enumerate(slots):
        torch.testing.assert_close(cache[s // page, s % page, 0].cpu().to(F64), torch.cat([c[i], kr[i]]), **tol)
        assert torch.equal(values[s // page, s % page, 0], cache[s // page, s % page, 0, :rank]), "the values are the latent once more"
    assert int((values != 0).any(-1).sum()) == len(slots), "no other slot was written"
    assert torch.equal(d.cpu(), down), "the projected rows stay as they were (the gate is read from them later)"


@pytest.mark.parametrize("interleaved", [True, False])
def test_a_stretch_of_every_head_turns_to_a_place_of_its_own(interleaved):
    h = hip()
    T, H, D, rot = 6, 3, 20, 8
    freqs, amp = plain.rotary_frequencies(rot, 300.0, dict(factor=5.0, original=16.0, fast=4.0, slow=1.0))
    src = torch.randn(T, H, D + rot)
    dst = torch.full((T, H, 30 + rot), 7.0, device=DEV)
    pos = [0, 3, 64, 65, 1000, 12345]
    h.rotate_heads(dst[:, :, 30:], src.to(DEV)[:, :, D:], freqs.to(DEV), amp, torch.tensor(pos, dtype=torch.int32, device=DEV), interleaved=interleaved)
    want = plain.rotate(src.to(F64)[:, :, D:], torch.tensor(pos), freqs, amp, interleaved)
    torch.testing.assert_close(dst[:, :, 30:].cpu().to(F64), want, atol=1e-5, rtol=1e-5)
    assert float((dst[:, :, :30] - 7.0).abs().max()) == 0.0


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("sizes", [(1, 3, 24, 40), (5, 3, 20, 34), (23, 2, 16, 16), (70, 8, 64, 256), (130, 4, 128, 512), (300, 2, 33, 65),
                                   (2, 5, 24, 40), (64, 3, 256, 64), (200, 2, 40, 70)])
def test_products_per_head_as_stored_and_transposed_with_a_gate(dtype, sizes):
    h = hip()
    T, H, K, N = sizes
    x = torch.randn(T, H, K + (8 if T % 2 == 0 else 5))     # (rows at 16-byte borders, which the matrix cores want, or not)
    w, w64 = rounded(torch.randn(H, K, N) * K ** -0.5, dtype)
    wt, wt64 = rounded(torch.randn(H, N, K) * K ** -0.5, dtype)
    gate = torch.randn(T, H * N + 3) * 2
    xd, gd = x.to(DEV), gate.to(DEV)
    tol = dict(atol=2e-5, rtol=1e-5) if dtype == torch.float32 else dict(atol=2e-2, rtol=1e-2)
    out = torch.zeros(T, H, N + 2, device=DEV)
    h.heads_gemm(xd[:, :, :K], w, out[:, :, :N])
    torch.testing.assert_close(out[:, :, :N].cpu().to(F64), torch.einsum("thk,hkn->thn", x.to(F64)[:, :, :K], w64), atol=2e-5, rtol=1e-5)
    assert float(out[:, :, N:].abs().max()) == 0.0
    y = torch.empty(T, H, N, dtype=dtype, device=DEV)
    # bfloat16 matrices whose k runs along memory, k in 16-byte pieces, aligned rows: the matrix cores
    assert h.heads_gemm_mfma_takes(xd[:, :, :K], wt.transpose(1, 2), y) == (dtype == torch.bfloat16 and T % 2 == 0 and K % 8 == 0)
    h.heads_gemm(xd[:, :, :K], wt.transpose(1, 2), y, gate=gd[:, :H * N])
    want = torch.einsum("thk,hnk->thn", x.to(F64)[:, :, :K], wt64) * torch.sigmoid(gate.to(F64)[:, :H * N]).view(T, H, N)
    torch.testing.assert_close(y.cpu().to(F64), want, **tol)


def latent_case(dtype, H, rank, rot, page, length, queries, stand_out, scale, window, seed=0, portion_from=None, mfma=None):
    """Cached rows [c | r] of one request on shuffled pages; queries as in `chunk_case`. The key that stands out has its
    whole row along the query's direction. The oracle sees one key/value head: keys the rows, values their first `rank`."""
    h = hip()
    row = rank + rot
    if portion_from is not None:
        queries = list(range(portion_from, length))
        stand_out = {q: key for q, key in stand_out.items() if q >= portion_from}
    gen = torch.Generator().manual_seed(seed)
    rows64 = plain.unit_rms(torch.randn(length, row, generator=gen, dtype=F64), 0.0)
    q64 = plain.unit_rms(torch.randn(len(queries), H, row, generator=gen, dtype=F64), 0.0)
    for i, p in enumerate(queries):
        if p in stand_out:
            g_dir = plain.unit_rms(torch.randn(row, generator=gen, dtype=F64), 0.0)
            q64[i] = g_dir
            rows64[stand_out[p]] = 11.0 / (row * scale) * g_dir
    pages = -(-length // page)
    table = torch.randperm(pages + 3, generator=gen)[:pages].tolist()
    cache = torch.zeros(pages + 3, page, 1, row, dtype=dtype, device=DEV)
    values = torch.zeros(pages + 3, 1, rank, page, dtype=dtype, device=DEV).permute(0, 3, 1, 2)
    rr = rows64.to(dtype)
    at = torch.arange(length)
    pg, off = torch.tensor(table)[at // page].to(DEV), (at % page).to(DEV)
    cache[pg, off, 0] = rr.to(DEV)
    values[pg, off, 0] = rr[:, :rank].to(DEV)
    q = q64.float().to(DEV)                                                 # (queries stay 32-bit up to the scores)
    if portion_from is None:
        ctx = step_context([table] * len(queries), page, queries, [1] * len(queries))
    else:
        ctx = step_context([table], page, [portion_from], [len(queries)])
    out = h.paged_attention_latent(q, cache, rank, ctx, 0, scale, window, 0, out_dtype=dtype, v_cache=values)
    if mfma is not None:
        assert h.latent_mfma_takes(q, cache, values, rank) == mfma, "the case was made for the other kernel"
    keys = rr.to(F64)
    want = plain.masked_attention(q.cpu().to(F64), keys[:, None, :], keys[:, None, :rank], torch.tensor(queries), scale,
                                  "window" if window else "full", window, None)
    return out.cpu().to(F64), want, keys[:, :rank], queries


@pytest.mark.parametrize("form", sorted(FORMS))
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("page", [16, 32])
@pytest.mark.parametrize("window, sizes", [(1, (3, 40, 8)), (7, (3, 34, 6)), (16, (2, 16, 16)), (50, (3, 48, 8)), (64, (4, 96, 16)),
                                           (70, (5, 16, 16)), (96, (6, 128, 32)), (130, (8, 256, 32)), (257, (2, 512, 64)), (65, (4, 64, 0)),
                                           (33, (24, 32, 8)), (100, (32, 256, 64)), (31, (16, 80, 24)), (200, (40, 64, 8))])
def test_latent_attention_window_edges(dtype, window, sizes, form, page):
    """Pages of 16 keys go to the kernel that is 32-bit throughout, as float32 always does; pages of 32 in bfloat16 go to
    the matrix cores where the sizes allow: tokens of fewer than 32 heads share a tile, heads beyond 32 take a second one;
    steps of few tiles cut a tile's keys into stretches that a second kernel adds up."""
    H, rank, rot = sizes
    mfma = dtype == torch.bfloat16 and page == 32 and rank % 16 == 0 and rot % 8 == 0
    if window > 100:
        length = 4 * window + 15
        inside = {q: q - window + 1 for q in (window - 1, 3 * window + 9)}
        outside = {q: q - window for q in (2 * window + 4, 4 * window + 14)}
    else:
        length = 600
        inside = {q: q - window + 1 for q in (window - 1, 400)}
        outside = {q: q - window for q in (200, 599)}
    queries = sorted({0, 127, 128, 129, *inside, *outside})
    out, want, v, queries = latent_case(dtype, H, rank, rot, page, length, queries, {**inside, **outside}, (rank + rot) ** -0.5,
                                        window, portion_from=FORMS[form], mfma=mfma)
    torch.testing.assert_close(out, want, **tolerance(dtype))
    for q, key in inside.items():
        if q in queries:
            assert decides(want[queries.index(q), 0], v[key]), (q, key)
    for q, key in outside.items():
        if q in queries and window > 1:
            assert not decides(want[queries.index(q), 0], v[key]), (q, key)


@pytest.mark.parametrize("mask", [("full", 0), ("window", 100), ("chunk", 128)])
@pytest.mark.parametrize("sizes", [(32, 256, 0), (16, 256, 128), (40, 96, 24), (130, 64, 16), (32, 128, 0)])
def test_latent_attention_of_several_requests_in_wide_tiles(sizes, mask, monkeypatch):
    """Requests of uneven lengths and starts in one list of tiles of 128 rows, decoded tokens beside them, tiles cut at the requests'
    borders, heads beyond 128, pages of the pool in runs, sinks and a gate per head. Scores spread over +-10, so that a key
    more or less at an edge shows. The same requests with many more decoded tokens are the other kernel's where heads are few."""
    h = hip()
    (H, rank, rot), (kind, size) = sizes, mask
    row, page, scale = rank + rot, 64, 3.0 * (rank + rot) ** -0.5
    gen = torch.Generator().manual_seed(H + row + size)
    ran, plain_run = [], h._run
    monkeypatch.setattr(h, "_run", lambda name, code: ran.append(name) or plain_run(name, code))
    for decoding in (3, 1200):
        starts = [40, 333, 700] * (decoding // 3) + [0, 77, 500, 0, 130]
        counts = [1] * decoding + [290, 129, 1, 5, 160]
        ends = [a + b for a, b in zip(starts, counts)]
        pages = [-(-n // page) for n in ends]
        order = torch.randperm(sum(pages) + 5, generator=gen).tolist()
        tables = [order[sum(pages[:i]):sum(pages[:i + 1])] for i in range(len(pages))]
        cache = torch.zeros(2 * len(order), 32, 1, row, dtype=torch.bfloat16, device=DEV)
        values = torch.zeros(2 * len(order), 1, rank, 32, dtype=torch.bfloat16, device=DEV).permute(0, 3, 1, 2)
        kept = []
        for table, n in zip(tables, ends):
            rows, at = torch.randn(n, row, generator=gen).bfloat16().to(DEV), torch.arange(n)
            pg, off = (2 * torch.tensor(table)[at // page] + at % page // 32).to(DEV), (at % 32).to(DEV)
            cache[pg, off, 0], values[pg, off, 0] = rows, rows[:, :rank]
            kept.append(rows.cpu().to(F64))
        q = torch.randn(sum(counts), H, row, generator=gen).bfloat16().float().to(DEV)
        sinks, gates = torch.linspace(-3.0, 8.0, H, device=DEV), torch.randn(sum(counts), H + 3, generator=gen).to(DEV)
        ctx = step_context(tables, page, starts, counts)
        ran.clear()
        out = h.paged_attention_latent(q, cache, rank, ctx, 0, scale, size if kind == "window" else 0, size if kind == "chunk" else 0,
                                       out_dtype=torch.float32, v_cache=values, sinks=sinks, head_gate=gates[:, 1:1 + H])
        assert ran == ["paged_attention_latent_tiles" if decoding == 3 or H > 32 else "paged_attention_latent_mfma"]
        picked = range(len(counts)) if decoding == 3 else [0, 1, decoding - 1, decoding, decoding + 4]
        for i in picked:
            mine = slice(sum(counts[:i]), sum(counts[:i + 1]))
            positions = torch.arange(starts[i], ends[i])
            want = plain.masked_attention(q[mine].cpu().to(F64), kept[i][:, None], kept[i][:, None, :rank], positions, scale, kind, size, sinks.cpu().to(F64))
            want = want * torch.sigmoid(gates[mine, 1:1 + H].cpu().to(F64))[:, :, None]
            # (weights are kept as two bfloat16 terms, 2^-16 of each; scores of up to 15 good to 2^-21 of that over 384 products)
            torch.testing.assert_close(out[mine].cpu().to(F64), want, atol=1e-4, rtol=1e-4)


@pytest.mark.parametrize("sizes", [(32, 256, 0), (16, 256, 32), (40, 128, 64)])
@pytest.mark.parametrize("sharp", [1.0, 3.0])
def test_wide_latent_tiles_are_as_close_to_64_bits_as_narrow_ones(sizes, sharp, monkeypatch):
    """Softmaxes that a few keys decide as well as flat ones: the error's root mean square is that of the kernel of 32 rows (the
    same scores and weights; the sums of the weights are made in another order: a hundredth of it)."""
    h = hip()
    H, rank, rot = sizes
    row, n = rank + rot, 520
    gen = torch.Generator().manual_seed(H + rot)
    rows = torch.randn(544, row, generator=gen).bfloat16().to(DEV)
    cache, values = rows.view(17, 32, 1, row), rows[:, :rank].reshape(17, 32, 1, rank).permute(0, 2, 3, 1).contiguous().permute(0, 3, 1, 2)
    q = torch.randn(n, H, row, generator=gen).bfloat16().float().to(DEV)
    scores = torch.einsum("thd,kd->htk", q.double().cpu(), rows.double().cpu()) * (sharp * row ** -0.5)
    scores = scores.masked_fill(torch.arange(544)[None, None] > torch.arange(n)[None, :, None], float("-inf"))
    want = torch.einsum("htk,kd->thd", torch.softmax(scores, dim=-1), rows[:, :rank].double().cpu())
    off = []
    for wide in (False, True):
        monkeypatch.setattr(h, "latent_wide_tiles", lambda *a: wide)
        out = h.paged_attention_latent(q, cache, rank, step_context([list(range(17))], 32, [0], [n]), 0, sharp * row ** -0.5, out_dtype=torch.float32, v_cache=values)
        off.append(float((out.cpu().double() - want).norm() / want.norm()))
    assert 0.0 < off[1] <= 1.01 * off[0] < 1e-5, off


@pytest.mark.parametrize("listed", [False, True])
def test_a_step_recorded_before_its_wide_tiles_are_listed(listed, monkeypatch):
    """From 32 heads on the kernel of 32 rows needs no list of tiles, so a step is recorded as its context comes; where an eager step
    listed the wide tiles before, they are recorded. Replays with the inputs changed and eager work in between."""
    h = hip()
    H, rank, n = 32, 128, 300
    gen = torch.Generator().manual_seed(5)
    rows = torch.randn(320, rank, generator=gen).bfloat16().to(DEV)
    cache, values = rows.view(10, 32, 1, rank), rows.reshape(10, 32, 1, rank).permute(0, 2, 3, 1).contiguous().permute(0, 3, 1, 2)
    queries = [torch.randn(n, H, rank, generator=gen).bfloat16().float().to(DEV) for _ in range(4)]
    attend = lambda q, ctx: h.paged_attention_latent(q, cache, rank, ctx, 0, 0.1, out_dtype=torch.float32, v_cache=values)
    ctx, q = step_context([list(range(10))], 32, [0], [n]), queries[0].clone()
    if listed:
        attend(q, ctx)
    ran, plain_run = [], h._run
    monkeypatch.setattr(h, "_run", lambda name, code: ran.append(name) or plain_run(name, code))
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = attend(q, ctx)
    assert ran == ["paged_attention_latent_tiles" if listed else "paged_attention_latent_mfma"]
    monkeypatch.setattr(h, "latent_wide_tiles", lambda *a: listed)
    for given in queries:
        want = attend(given, step_context([list(range(10))], 32, [0], [n]))
        q.copy_(given)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


@pytest.mark.parametrize("form", sorted(FORMS))
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("page", [16, 32])
@pytest.mark.parametrize("sizes", [(3, 48, 8), (2, 16, 16), (8, 256, 32), (5, 34, 6), (20, 128, 16)])
def test_latent_attention_far_keys_and_page_borders(dtype, sizes, form, page):
    H, rank, rot = sizes
    stand_out = {699: 3, 650: 15, 651: 16, 652: 17, 653: 653, 500: 255, 501: 256, 31: 0, 32: 31, 33: 32}
    queries = [0, 1, 2, 3, 15, 16, 17, 31, 32, 33, 500, 501, 650, 651, 652, 653, 699]
    out, want, v, qs = latent_case(dtype, H, rank, rot, page, 700, queries, stand_out, (rank + rot) ** -0.5, 0, portion_from=FORMS[form])
    torch.testing.assert_close(out, want, **tolerance(dtype))
    assert decides(want[qs.index(699), 0], v[3]), "the far key decides the row"


# ---- the matrix memory ---------------------------------------------------------------------------------

def mlstm_weights(H, D, V, cap):
    """Projections that pick coordinates of the input, so that the plain mixer can be fed a projected row itself."""
    width = 2 * H * D + H * V + 2 * H + H * V
    eye = torch.eye(width, dtype=F64)
    at, W = 0, {}
    for name, rows in (("q", H * D), ("k", H * D), ("v", H * V), ("i", H), ("f", H), ("g", H * V)):
        W[name] = eye[at:at + rows]
        at += rows
    W["o"] = torch.eye(H * V, dtype=F64)
    return W, dict(heads=H, dim=D, vdim=V, gate_cap=cap), width


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("sizes", [(3, 20, 28, 8.0), (1, 16, 16, 15.0), (2, 18, 270, 5.0), (4, 64, 128, 12.0), (2, 32, 40, 10.0),
                                   (1, 1, 1, 2.0), (2, 128, 64, 6.0), (1, 300, 20, 4.0)])
@pytest.mark.parametrize("portions", [[1, 2, 13, 1, 5, 31, 3], [1, 2, 13, 1, 5, 64, 3], [200, 1, 32]])
def test_matrix_memory_over_steps_slots_and_gates_at_their_caps(dtype, sizes, portions):
    """Three requests of unequal length in packed steps of changing portions (one token, two, many), each with its state in
    a slot of its own among slots that hold another request's leftovers until they are cleared; gate sums far beyond the
    cap on either side; heads whose values span several workgroups, and heads of one dimension. Steps in which every
    request feeds few tokens walk token by token; a step in which one feeds 32 or more is worked in chunks of 64 (whole
    chunks, a chunk's rest, single tokens of other requests beside them)."""
    h = hip()
    H, D, V, cap = sizes
    W, m, width = mlstm_weights(H, D, V, cap)
    gen = torch.Generator().manual_seed(H * 1000 + D)
    lengths = [37, 1, 90] if portions[0] < 100 else [150, 1, 333]
    bi, bf = torch.randn(H, generator=gen), torch.randn(H, generator=gen) + 1
    W["i.b"], W["f.b"] = bi.to(F64), bf.to(F64)
    norm_w = 1 + 0.1 * torch.randn(H * V, generator=gen)
    W["norm"] = norm_w.to(F64)
    gates_at = 2 * H * D + H * V
    rows = []
    for n in lengths:
        r = torch.randn(n, width, generator=gen)
        r[:, gates_at:gates_at + 2 * H] *= 4.0
        if n > 10:
            r[3, gates_at:gates_at + H] = 60.0                              # an input gate at its cap,
            r[5, gates_at + H:gates_at + 2 * H] = -60.0                     # a forget gate that forgets all it can,
            r[7, gates_at:gates_at + H] = -60.0                             # an input gate that takes next to nothing
            r[20:30, gates_at + H:gates_at + 2 * H] = 60.0                  # and a stretch that forgets nothing
        rows.append(r)
    want = [plain.mlstm(r.to(F64), W, m, 1e-5, {}) for r in rows]
    state = torch.randn(5, h.mlstm_state_size(H, D, V), device=DEV)        # leftovers everywhere
    slots = [4, 0, 2]
    state[slots] = 0.0                                                      # (what the manager does when it hands a slot out)
    cursors, got, tick = [0, 0, 0], [[], [], []], 0
    while any(c < n for c, n in zip(cursors, lengths)):
        live = [i for i in range(3) if cursors[i] < lengths[i]]
        counts = [min(portions[(tick + 2 * i) % len(portions)], lengths[i] - cursors[i]) for i in live]
        tick += 1
        proj = torch.cat([rows[i][cursors[i]:cursors[i] + n] for i, n in zip(live, counts)]).to(DEV)
        cu = torch.tensor([0] + list(itertools.accumulate(counts)), dtype=torch.int32, device=DEV)
        o = h.mlstm_scan(proj, bi.to(DEV), bf.to(DEV), state, cu, torch.tensor([slots[i] for i in live], dtype=torch.int32, device=DEV), H, D, V, cap,
                         host_cu_seqlens=[0] + list(itertools.accumulate(counts)))
        y = h.mlstm_finish(o, norm_w.to(DEV), proj[:, gates_at + 2 * H:], H, V, 1e-5, dtype)
        at = 0
        for i, n in zip(live, counts):
            got[i].append(y[at:at + n])
            at += n
            cursors[i] += n
    tol = dict(atol=1e-4, rtol=1e-4) if dtype == torch.float32 else dict(atol=2e-2, rtol=2e-2)
    for i in range(3):
        torch.testing.assert_close(torch.cat(got[i]).cpu().to(F64), want[i], **tol)
    # the state left behind is the plain one's: S, n and m of the longest request
    st = {}
    plain.mlstm(rows[2].to(F64), W, m, 1e-5, st)
    left = state[2].cpu().to(F64).view(H, D * V + D + 1)
    torch.testing.assert_close(left[:, :D * V].reshape(H, D, V), st["S"], atol=1e-4, rtol=1e-4)
    torch.testing.assert_close(left[:, D * V:D * V + D], st["n"], atol=1e-4, rtol=1e-4)
    torch.testing.assert_close(left[:, -1], st["m"], atol=1e-5, rtol=1e-5)
    assert float((state[[1, 3]].cpu() - 0).abs().max()) > 0, "slots of other requests are left alone"


def test_matrix_memory_starts_at_a_maximum_of_zero():
    # a first token whose input gate is far below zero: with m starting at 0 the read-out's floor exp(-m) is about 2, not huge
    h = hip()
    H, D, V, cap = 1, 4, 4, 50.0
    W, m, width = mlstm_weights(H, D, V, cap)
    W.update({"i.b": torch.zeros(1, dtype=F64), "f.b": torch.zeros(1, dtype=F64), "norm": torch.ones(4, dtype=F64)})
    r = torch.randn(1, width)
    r[0, 2 * D + V] = -30.0
    r[0, 2 * D + V + 1] = 0.0
    state = torch.zeros(1, h.mlstm_state_size(H, D, V), device=DEV)
    dev = lambda t: torch.tensor(t, dtype=torch.int32, device=DEV)
    o = h.mlstm_scan(r.to(DEV), torch.zeros(1, device=DEV), torch.zeros(1, device=DEV), state, dev([0, 1]), dev([0]), H, D, V, cap)
    assert float(state[0, -1]) == pytest.approx(-math.log(2.0), abs=1e-6)
    st = {}
    plain.mlstm(r.to(F64), W, m, 0.0, st)
    q = r[0, :D].to(F64) * D ** -0.5
    want = torch.einsum("dv,d->v", st["S"][0], q) / (max(abs(float(st["n"][0] @ q)), 2.0) + 1e-6)
    torch.testing.assert_close(o[0].cpu().to(F64), want, atol=1e-18, rtol=1e-4)


# ---- the router and the ungated experts ------------------------------------------------------------------

@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("sizes", [(6, 3, 80, 40, 23), (4, 1, 48, 20, 1), (3, 3, 99, 17, 9), (12, 2, 64, 24, 70), (8, 2, 512, 128, 40),
                                   (5, 2, 99, 17, 60), (4, 2, 64, 32, 170), (3, 2, 128, 192, 300)])
def test_softmax_over_the_chosen_and_experts_with_a_squared_relu(dtype, sizes):
    h = hip()
    E, top, W, F, n = sizes
    x, x64 = rounded(torch.randn(n, W), dtype)
    router = (torch.randn(E, W) * 0.3).to(DEV)
    ids, weights = h.moe_route(x, router, None, top, 1.0, True, softmax_chosen=True)
    z = x64 @ router.cpu().to(F64).T
    chosen, w64 = plain.chosen_experts(z, top)
    for t in range(n):
        ranked = torch.sort(z[t], descending=True).values
        if top < E and float(ranked[top - 1] - ranked[top]) < 1e-3:
            continue                                                         # (no close calls are made)
        assert sorted(ids[t].tolist()) == sorted(chosen[t].tolist())
        got = dict(zip(ids[t].tolist(), weights[t].tolist()))
        for e, w in zip(chosen[t].tolist(), w64[t].tolist()):
            assert got[e] == pytest.approx(w, rel=1e-4, abs=1e-5)
        assert sum(got.values()) == pytest.approx(1.0, abs=1e-5)
    up, up64 = rounded(torch.randn(E, F, W) * W ** -0.5 * 2, dtype)
    down, d64 = rounded(torch.randn(E, W, F) * F ** -0.5, dtype)
    grouped = h.moe_group(ids, E, h.moe_tile_rows(n * top, E, dtype, (W, F)))
    act = h.moe_gemm(x, up, grouped, dtype, per_token=True, activation="relu2")
    out = h.moe_combine(h.moe_gemm(act, down, grouped, torch.float32, per_token=False), weights, None)
    picked = list(range(0, n, max(1, n // 40)))
    want = torch.zeros(len(picked), W, dtype=F64)
    flat = ids.cpu().view(-1).tolist()
    for row, t in enumerate(picked):
        for j in range(top):
            e = flat[t * top + j]
            y = torch.relu(x64[t] @ up64[e].T) ** 2
            torch.testing.assert_close(act[t * top + j].cpu().to(F64), y, **(dict(atol=1e-4, rtol=1e-4) if dtype == torch.float32 else dict(atol=3e-2, rtol=2e-2)))
            want[row] += float(weights[t, j]) * (act[t * top + j].cpu().to(F64) @ d64[e].T)
    torch.testing.assert_close(out[picked].cpu().to(F64), want, **(dict(atol=1e-4, rtol=1e-4) if dtype == torch.float32 else dict(atol=2e-2, rtol=1e-2)))


# ---- whole models through trace replay ---------------------------------------------------------------

LENGTHS = {"P": [1, 23, 97, 200], "Q": [1, 30, 75, 150], "R": [2, 19, 66, 131], "S": [1, 40, 140]}
TOL = {"float32": 2e-4, "bfloat16": 6e-2}       # of the spread of the oracle's logits


@pytest.fixture(scope="module", params=["P", "Q", "R", "S"])
def case(request, tmp_path_factory):
    from tinyserve_llm_amd.weights.random_init import write_random_model
    name = request.param
    config, seed = bafarax_configs()[name]
    folder = str(tmp_path_factory.mktemp(f"bafarax_{name}"))
    write_random_model(folder, config, seed, torch.bfloat16)
    oracle = plain.PlainBafarax.from_folder(folder)
    prompts = [prompt(500 + i, n, config.vocab) for i, n in enumerate(LENGTHS[name])]
    return name, folder, config, prompts, oracle, [oracle.logits(p) for p in prompts]


def replayer(folder, dtype, max_tokens):
    from tinyserve_llm_amd.engine.replay import Replay
    return Replay(folder, dtype, max_tokens)


def check(got, oracle_rows, dtype):
    assert got, "nothing was compared"
    spread = float(torch.cat([o.flatten() for o in oracle_rows]).std())
    worst = 0.0
    for (r, pos), row in got.items():
        want = oracle_rows[r][pos]
        torch.testing.assert_close(row.double().cpu(), want, atol=TOL[dtype] * spread, rtol=0.0,
                                   msg=lambda m: f"request {r} position {pos}: {m}")
        worst = max(worst, float((row.double().cpu() - want).abs().max()))
    print(f"[{dtype}] worst logit error {worst / spread:.3e} of the logits' spread ({spread:.2f}) over {len(got)} rows")


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_layer_streams_and_whole_requests(case, dtype):
    name, folder, config, prompts, oracle, rows = case
    rep = replayer(folder, dtype, 256)
    got = {}
    for r, p in enumerate(prompts):
        logits = rep.step([{"id": f"r{r}", "tokens": p, "want": list(range(len(p)))}], [f"r{r}"])
        assert logits.shape == (len(p), config.vocab) and logits.dtype == torch.float32
        for pos in range(len(p)):
            got[(r, pos)] = logits[pos]
    check(got, rows, dtype)
    assert rep.manager.num_available_blocks() == rep.manager.num_blocks, "every page came back"
    assert len(rep.manager.free_state_slots) == 4, "every state slot came back"
    if dtype == "float32":
        # the residual stream after every run of a layer, one by one (a layer that runs twice counts twice)
        from tinyserve_llm_amd.engine.runner import StepEntry
        from tinyserve_llm_amd.parts import base
        from tinyserve_llm_amd.parts.stream import ResidualStream
        p = prompts[2]
        want = oracle.streams(p)
        assert len(want) == len(config.layers) == len(rep.model.spec.order)
        rep.manager.allocate(77, p)
        ctx, _, _ = rep.runner.prepare([StepEntry(77, p, 0, [])])
        ctx.position_encodings = rep.model.position_encodings
        hidden, residual = rep.model.embedding.forward(ctx), None
        for i, (run, mem) in enumerate(zip(rep.model.spec.order, rep.runner.memory)):
            layer = rep.model.layers[run.layer]
            hidden, residual = base.BLOCKS[layer.block](layer, hidden, residual, ctx, mem)
            now = ResidualStream(hidden.x.clone(), hidden.a).take()[0]
            scale = float(want[i].abs().max())
            torch.testing.assert_close(now.cpu().double(), want[i], atol=2e-5 * max(1.0, scale), rtol=1e-5, msg=lambda m: f"after layer {i}: {m}")


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_prompt_then_token_by_token(case, dtype):
    """The last tokens one by one: more of them than a page, most chunks and most windows hold."""
    name, folder, config, prompts, oracle, rows = case
    rep = replayer(folder, dtype, 256)
    got = {}
    for r, p in enumerate(prompts):
        head = max(0, len(p) - 80)
        if head:
            got[(r, head - 1)] = rep.step([{"id": f"r{r}", "tokens": p[:head], "want": [head - 1]}], [])[0]
        for pos in range(head, len(p)):
            got[(r, pos)] = rep.step([{"id": f"r{r}", "tokens": [p[pos]], "want": [0]}], [f"r{r}"] if pos == len(p) - 1 else [])[0]
    check(got, rows, dtype)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_portions_down_to_two_tokens(case, dtype):
    name, folder, config, prompts, oracle, rows = case
    rep = replayer(folder, dtype, 256)
    sizes = [2, 7, 3, 16, 2, 5, 31, 2, 64, 9, 1, 33]
    got = {}
    for r, p in enumerate(prompts):
        pos, i = 0, r
        while pos < len(p):
            n = min(sizes[i % len(sizes)], len(p) - pos)
            i += 1
            want = sorted({0, n - 1})
            logits = rep.step([{"id": f"r{r}", "tokens": p[pos:pos + n], "want": want}], [f"r{r}"] if pos + n == len(p) else [])
            for j, w in enumerate(want):
                got[(r, pos + w)] = logits[j]
            pos += n
    check(got, rows, dtype)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_mixed_batches_on_pages_and_slots_used_again(case, dtype):
    """Nine unequal requests, at most four live, on a pool that holds the first four: later requests start on pages and in
    state slots that earlier ones have written and given back, beside others that are in the middle of theirs. A matrix
    memory that is not cleared, or a stale page, shows in the logits."""
    name, folder, config, _, oracle, _ = case
    lengths = [129, 70, 40, 1, 65, 100, 128, 30, 150]
    prompts = [prompt(900 + i, n, config.vocab) for i, n in enumerate(lengths)]
    rows = [oracle.logits(p) for p in prompts]
    pool = sum(-(-n // 64) for n in lengths[:4])
    rep = replayer(folder, dtype, 64 * pool)
    assert rep.manager.num_blocks == pool and len(rep.manager.free_state_slots) == 4
    chunk = [13, 2, 1, 7, 1, 1, 30, 1, 3, 1]
    cursors, pages = [0] * len(prompts), [-(-n // 64) for n in lengths]
    waiting, live, tick, got, slots_used = list(range(len(prompts))), [], 0, {}, []
    while waiting or live:
        while waiting and len(live) < 4 and sum(pages[r] for r in live) + pages[waiting[0]] <= pool:
            live.append(waiting.pop(0))
        batch, end, wanted = [], [], []
        new = [r for r in live if cursors[r] == 0]
        for r in live:
            n = min(lengths[r] - cursors[r], chunk[(tick + 3 * r) % len(chunk)])
            batch.append({"id": f"q{r}", "tokens": prompts[r][cursors[r]:cursors[r] + n], "want": [n - 1]})
            wanted.append((r, cursors[r] + n - 1))
            cursors[r] += n
            if cursors[r] == lengths[r]:
                end.append(r)
        logits = rep.step(batch, [])
        slots_used += [rep.manager.state_slot(rep.ids[f"q{r}"]) for r in new]
        for j, key in enumerate(wanted):
            got[key] = logits[j]
        rep.step([], [f"q{r}" for r in end])
        live = [r for r in live if r not in end]
        tick += 1
    assert len(slots_used) > len(set(slots_used)), "state slots were used again"
    check(got, rows, dtype)
    assert rep.manager.num_available_blocks() == rep.manager.num_blocks


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_long_prompts_whole_and_in_long_portions(case, dtype):
    """Steps of hundreds of tokens take kernels of their own: a prompt of 520 tokens whole, and cut where the second
    portion starts in the middle of a page, of a chunk and of a window, beside a short request."""
    name, folder, config, _, oracle, _ = case
    long, short = prompt(321, 520, config.vocab), prompt(322, 40, config.vocab)
    rows = [oracle.logits(long), oracle.logits(short)]
    rep = replayer(folder, dtype, 640)
    marks = [0, 1, 255, 256, 257, 300, 518, 519]
    got = {}
    logits = rep.step([{"id": "w", "tokens": long, "want": marks}], ["w"])
    for j, pos in enumerate(marks):
        got[(0, pos)] = logits[j]
    check(got, rows, dtype)
    got = {}
    logits = rep.step([{"id": "a", "tokens": long[:263], "want": [0, 262]}, {"id": "b", "tokens": short[:7], "want": [6]}], [])
    got[(0, 0)], got[(0, 262)], got[(1, 6)] = logits[0], logits[1], logits[2]
    logits = rep.step([{"id": "b", "tokens": short[7:], "want": [0, 32]}, {"id": "a", "tokens": long[263:], "want": [0, 1, 37, 256]}], ["a", "b"])
    got[(1, 7)], got[(1, 39)] = logits[0], logits[1]
    for j, pos in enumerate([263, 264, 300, 519]):
        got[(0, pos)] = logits[2 + j]
    check(got, rows, dtype)
    assert rep.manager.num_available_blocks() == rep.manager.num_blocks


def test_a_batch_equals_each_request_alone_in_float32(case):
    """float32: the logits of a request do not depend on what else is in the batch, beyond rounding."""
    name, folder, config, prompts, oracle, rows = case
    rep = replayer(folder, "float32", 1024)
    alone = [rep.step([{"id": f"a{r}", "tokens": p, "want": [len(p) - 1]}], [f"a{r}"])[0] for r, p in enumerate(prompts)]
    together = rep.step([{"id": f"b{r}", "tokens": p, "want": [len(p) - 1]} for r, p in enumerate(prompts)],
                        [f"b{r}" for r in range(len(prompts))])
    for r in range(len(prompts)):
        torch.testing.assert_close(together[r], alone[r], atol=2e-6, rtol=1e-6)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_long_decoding(case, dtype):
    """300 tokens fed one by one after a prompt of five: the matrix memory is carried through every step, chunks start and
    windows pass over decoded tokens, latents and keys fill page after page."""
    name, folder, config, _, oracle, _ = case
    p = prompt(77, 305, config.vocab)
    rows = oracle.logits(p)
    rep = replayer(folder, dtype, 320)
    rep.step([{"id": "d", "tokens": p[:5], "want": []}], [])
    got = {}
    for pos in range(5, len(p)):
        logits = rep.step([{"id": "d", "tokens": [p[pos]], "want": [0]}], [])
        if pos % 7 == 0 or pos >= 300:
            got[(0, pos)] = logits[0]
    check(got, [rows], dtype)


# ---- generation through the engine's entry point -----------------------------------------------------

def test_greedy_generation_through_the_scheduler(case):
    from tinyserve_llm_amd.engine.llm import LLM, CacheConfig
    from tinyserve_llm_amd.engine.scheduler import SchedulerConfig
    from tinyserve_llm_amd.engine.sequence import SamplingParams
    name, folder, config, prompts, oracle, _ = case
    prompts = [p for p in prompts if len(p) <= 75] + [prompt(42, 90, config.vocab)]
    want = [oracle.greedy(p, 12) for p in prompts]
    sc = SchedulerConfig(max_model_len=256, max_num_seqs=4, max_num_batched_tokens=48, max_prefill_chunk=32)
    llm = LLM(folder, sc, CacheConfig(block_size=32), dtype=torch.float32, num_blocks=24)
    got = llm.generate(prompts, SamplingParams(max_tokens=12, temperature=0.0, ignore_eos=True))
    assert [r.token_ids[0] for r in got] == want
    # bfloat16 may flip a near-tie: its tokens are judged by the plain model's logits for the same history
    llm16 = LLM(folder, sc, CacheConfig(block_size=32), dtype=torch.bfloat16, num_blocks=24)
    got16 = llm16.generate(prompts[:2], SamplingParams(max_tokens=8, temperature=0.0, ignore_eos=True))
    spread = float(oracle.logits(prompts[1]).std())
    for p, r in zip(prompts, got16):
        ids = list(p)
        for tok in r.token_ids[0]:
            row = oracle.logits(ids)[-1]
            assert float(row.max() - row[tok]) <= 0.15 * spread, "a bfloat16 token far from the plain model's best"
            ids.append(tok)


def test_forked_continuations_and_preemption(case):
    """n = 3 at temperature 0: the continuations part after the prompt, each with a copy of the matrix memory and the
    prompt's pages shared; all three must be the oracle's greedy continuation. And a pool so small that requests are
    preempted and fed again from their first token."""
    from tinyserve_llm_amd.engine.llm import LLM, CacheConfig
    from tinyserve_llm_amd.engine.scheduler import SchedulerConfig
    from tinyserve_llm_amd.engine.sequence import SamplingParams
    name, folder, config, prompts, oracle, _ = case
    p = prompt(11, 45, config.vocab)
    want = oracle.greedy(p, 10)
    sc = SchedulerConfig(max_model_len=128, max_num_seqs=4, max_num_batched_tokens=64, max_prefill_chunk=16)
    llm = LLM(folder, sc, CacheConfig(block_size=16), dtype=torch.float32, num_blocks=24)
    got = llm.generate([p], SamplingParams(max_tokens=10, temperature=0.0, n=3, ignore_eos=True))
    assert got[0].token_ids == [want, want, want]
    many = [prompt(20 + i, 60 + 3 * i, config.vocab) for i in range(4)]
    wants = [oracle.greedy(q, 30) for q in many]
    small = LLM(folder, sc, CacheConfig(block_size=16, caching=False), dtype=torch.float32, num_blocks=14)
    out = small.generate(many, SamplingParams(max_tokens=30, temperature=0.0, ignore_eos=True))
    assert [r.token_ids[0] for r in out] == wants


def test_command_line_generates_from_a_model_folder(case, tmp_path):
    import json
    import os
    import subprocess
    import sys
    name, folder, config, prompts, oracle, _ = case
    if name != "P":
        pytest.skip("one configuration through the command line is enough")
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    p = prompts[2]
    out = tmp_path / "record.json"
    cmd = [sys.executable, "-m", "tinyserve_llm_amd.generate", "--model", folder, "--prompt-ids", ",".join(map(str, p)),
           "--max-tokens", "6", "--temperature", "0", "--ignore-eos", "--dtype", "float32", "--block-size", "32",
           "--num-blocks", "16", "--max-model-len", "256", "--max-num-seqs", "4", "--out", str(out)]
    r = subprocess.run(cmd, cwd=root, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    record = json.loads(out.read_text())
    text = json.dumps(record)
    assert json.dumps(oracle.greedy(p, 6)).replace(" ", "") in text.replace(" ", ""), text[:500]
