"""Steps of many rows: products with the reduction in slices (gemm_slices.hip) against 64 bits, their endings against the kernels
they stand in for and the rule that chooses them; the gated product in every tile; values on their way into transposed pages;
prompts' attention; walks over chunks of the state-space recurrence; products per head."""

from __future__ import annotations

import types

import pytest
import torch

from tinyserve_llm_amd.ops import hip
from tinyserve_llm_amd.parts.linear import DeferredNorm, NormRequest, linear

BF = torch.bfloat16


def operands(rows, n, k, seed=0, x_skew=0):
    g = torch.Generator().manual_seed(1000 * rows + n + k + seed)
    x = torch.randn(rows, k + x_skew, generator=g).to(BF).cuda()[:, :k]
    return x, (torch.randn(n, k, generator=g) * k ** -0.5).to(BF).cuda()


# (edges of the tiles' rows and columns, uneven slices, the fewest steps a slice, one slice, rows of x apart)
FORMS = [(t, s, rows, n, k, skew) for t, (bm, bn, *_) in enumerate(hip.SLICES_TILES)
         for s, rows, n, k, skew in ((3, bm, bn, 640, 0), (2, bm + 1, bn + 8, 448, 8), (1, 1, 8, 192, 0), (5, 2 * bm - 1, 2 * bn - 8, 1024, 64),
                                     (16, 37, bn + 64, 3072, 0))]


@pytest.mark.gpu
@pytest.mark.parametrize("tile, slices, rows, n, k, skew", FORMS)
def test_a_product_in_slices(tile, slices, rows, n, k, skew):
    """32-bit sums of k products: (k + slices) 2^-24 of the sum of their sizes at most; in bfloat16 half a unit in the last place more."""
    x, w = operands(rows, n, k, x_skew=skew)
    want, sizes = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    wide = hip.gemm_slices(x, w, tile, slices, torch.float32)
    bound = (k + slices) * 2.0 ** -24 * sizes
    assert wide.shape == want.shape and bool(((wide.double() - want).abs() <= bound).all())
    assert torch.equal(hip.gemm_slices(x, w, tile, slices), wide.to(BF))


@pytest.mark.gpu
@pytest.mark.parametrize("rows, n, residual", [(129, 2048, True), (3, 8192, True), (200, 1032, False), (33, 264, True)])
def test_the_norm_that_follows_has_the_bits_of_its_own_kernel(rows, n, residual):
    x, w = operands(rows, n, 512)
    g = torch.Generator().manual_seed(n)
    res = torch.randn(rows, n, generator=g).to(BF).cuda() if residual else None
    nw = torch.randn(n, generator=g).to(BF).cuda()
    got, total = hip.gemm_slices(x, w, 0, 2, next_norm=(res, nw, 1e-5))
    product = hip.gemm_slices(x, w, 0, 2)
    want, want_total = hip.rmsnorm(product, nw, 1e-5, res)
    assert torch.equal(got, want) and torch.equal(total, want_total)


@pytest.mark.gpu
def test_numbers_that_are_none_stay_in_their_rows_and_columns():
    x, w = operands(150, 1024, 2048)
    x[7, 2000], w[5, 3] = float("nan"), float("inf")
    y = hip.gemm_slices(x, w, 4, 4, torch.float32)
    odd = torch.zeros_like(y, dtype=torch.bool)
    odd[7], odd[:, 5] = True, True
    assert bool((~torch.isfinite(y) == odd).all())


@pytest.mark.gpu
def test_linear_takes_the_slices_where_the_rule_says_so_and_hands_the_norm_on(monkeypatch):
    rows, n, k = 160, 2048, 8192
    assert hip.slices_plan(rows, n, k, "bf16") and hip.slices_plan(rows, n, k, "norm")
    x, w = operands(rows, n, k)
    res, nw = torch.randn(rows, n, device="cuda").to(BF), torch.randn(n, device="cuda").to(BF)
    plan = hip.slices_plan(rows, n, k, "f32")
    assert torch.equal(linear(x, w, torch.float32), hip.gemm_slices(x, w, *plan, torch.float32))
    d = linear(x, w, then=NormRequest(nw, 1e-5, res))
    assert isinstance(d, DeferredNorm) and d.done is not None and d.rows == rows
    want, total = hip.gemm_slices(x, w, *hip.slices_plan(rows, n, k, "norm"), next_norm=(res, nw, 1e-5))
    assert torch.equal(d.materialize(), want) and torch.equal(d.residual_out, total)
    narrow = torch.randn(64, n, device="cuda").to(BF)
    assert torch.equal(linear(d, narrow), linear(want, narrow))


@pytest.mark.gpu
def test_what_the_slices_do_not_take_is_refused_before_anything_runs():
    x, w = operands(130, 1024, 2048)
    nw, res = torch.ones(1024, dtype=BF, device="cuda"), torch.zeros(130, 1024, dtype=BF, device="cuda")
    for args, kwargs in [((x[:, :2000], w[:, :2000], 0, 2), {}), ((x, w, 5, 2), {}), ((x, w, 0, 11), {}), ((x, w, 0, 0), {}), ((x.float(), w, 0, 2), {}),
                         ((x, w[:1020], 0, 2), {}), ((x[:, 1:], w[:, 1:], 0, 2), {}), ((x, w, 0, 2, torch.float16), {}),
                         ((x, w, 0, 2, torch.float32), {"next_norm": (res, nw, 1e-5)}), ((x, w, 0, 2), {"next_norm": (res[:129], nw, 1e-5)}),
                         ((x, w, 0, 2), {"next_norm": (res, None, 1e-5)}), ((x, w, 0, 2), {"next_norm": (res, nw.float(), 1e-5)})]:
        with pytest.raises(hip.KernelError):
            hip.gemm_slices(*args, **kwargs)


@pytest.mark.gpu
def test_a_recorded_product_in_slices_is_replayed():
    x, w = operands(140, 1024, 2048)
    want = hip.gemm_slices(operands(140, 1024, 2048, seed=1)[0], w, 0, 4)
    hip.gemm_slices(x, w, 0, 4)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = hip.gemm_slices(x, w, 0, 4)
    x.copy_(operands(140, 1024, 2048, seed=1)[0])
    for _ in range(3):
        got.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)


def test_the_rule_keeps_to_what_was_measured():
    for ending in ("bf16", "f32", "norm"):
        for rows, n, k in ((128, 2048, 8192), (2049, 2048, 8192), (256, 8192, 8192), (256, 512, 8192), (256, 2048, 1024), (256, 2048, 8160), (256, 2044, 8192)):
            assert hip.slices_plan(rows, n, k, ending) is None
        for rows in range(129, 2049, 37):
            for n in (1024, 2048, 3072, 4096):
                for k in (2048, 4096, 8192, 14336):
                    plan = hip.slices_plan(rows, n, k, ending)
                    if plan is not None:
                        bm, bn = hip.SLICES_TILES[plan[0]][:2]
                        assert k // 64 // plan[1] >= hip.SLICES_MIN_STEPS and -(-rows // bm) * -(-n // bn) * plan[1] <= hip.COMPUTE_UNITS


def test_the_rule_leaves_to_the_library_what_the_library_is_faster_at():
    """Products that slices took 1.04 to 1.15 times the library's time for, and some that they take 0.72 to 0.95 of it for."""
    for rows, n, k, ending in ((513, 1536, 8192, "bf16"), (900, 1024, 8192, "bf16"), (850, 1024, 8192, "bf16"), (1999, 4096, 4096, "norm"), (2048, 4096, 4096, "norm"),
                               (450, 2048, 6144, "bf16"), (1514, 4096, 3072, "norm"), (320, 3072, 6144, "bf16"), (1501, 4096, 4096, "f32"), (2048, 4096, 5120, "bf16")):
        assert hip.slices_plan(rows, n, k, ending) is None
    for rows, n, k, ending in ((160, 2048, 8192, "bf16"), (512, 2048, 8192, "f32"), (1514, 3072, 8192, "norm"), (2048, 2048, 8192, "norm"), (300, 2048, 4096, "norm"),
                               (160, 2048, 4096, "norm")):
        assert hip.slices_plan(rows, n, k, ending) is not None


@pytest.mark.gpu
@pytest.mark.parametrize("tile", range(len(hip.GLU_TILES)))
@pytest.mark.parametrize("over", [-1, 0, 1])
def test_the_gated_product_is_the_same_in_every_tile(tile, over, monkeypatch):
    """A row more and less than one and two tiles, columns that hang over: each sum adds up in the order of K in every tile."""
    rows, f, k = 2 * hip.GLU_TILES[tile][0] + over, 136, 192
    x, w = operands(rows, 2 * f, k)
    want = [hip.gemm_glu(x, w, form, 5.0, 1.5, 0.5) for form in ("silu_rounded", "sigmoid")]
    one = hip.gemm_glu(x[:hip.GLU_TILES[tile][0] + over], w, "relu")
    monkeypatch.setattr(hip, "glu_plan", lambda rows, n: (tile, 0))
    assert all(torch.equal(hip.gemm_glu(x, w, form, 5.0, 1.5, 0.5), y) for form, y in zip(("silu_rounded", "sigmoid"), want))
    assert torch.equal(hip.gemm_glu(x[:hip.GLU_TILES[tile][0] + over], w, "relu"), one)


@pytest.mark.gpu
@pytest.mark.parametrize("heads, dim", [(2, 64), (8, 128), (3, 80)])
@pytest.mark.parametrize("portions", [
    [(40, 0)], [(13, None), (50, 0)], [(5, None), (3, 13), (20, 21), (9, 7)], [(17, 5), (1, -1), (30, 8)], [(7, 1), (8, 8), (8, 15), (16, 16)], [(9, -1), (23, 6)]])
def test_values_reach_their_slots_wherever_a_run_of_eight_begins(heads, dim, portions):
    """Steps of portions (tokens, their first slot on a page of its own; None: single tokens on pages of their own; -1: no slots):
    aligned, behind decoding requests, ends of portions, over a page's edge. Every slot holds its token, all others stay."""
    page, slots, next_page = 16, [], 0
    for n, first in portions:
        if first is None:
            slots += [(next_page + i) * page + (5 * i) % page for i in range(n)]
            next_page += n
        else:
            slots += [-1 if first < 0 else next_page * page + first + i for i in range(n)]
            next_page += 0 if first < 0 else -(-(first + n) // page)
    g = torch.Generator().manual_seed(len(slots))
    qkv = torch.randn(len(slots), 3 * heads * dim, generator=g).to(BF).cuda()
    k, v = torch.zeros(next_page, page, heads, dim, dtype=BF, device="cuda"), torch.full((next_page, heads, dim, page), 7.0, dtype=BF, device="cuda")
    where = torch.tensor(slots, dtype=torch.int32, device="cuda")
    hip.rope_store(qkv, None, torch.zeros_like(where), where, k, v.permute(0, 3, 1, 2), heads, heads, dim)
    want = torch.full((next_page * page, heads, dim), 7.0, dtype=BF)
    for t, s in enumerate(slots):
        if s >= 0:
            want[s] = qkv[t, 2 * heads * dim:].view(heads, dim).cpu()
    assert torch.equal(v.permute(0, 3, 1, 2).reshape(-1, heads, dim).cpu(), want)


def attended(q, k, v, starts, lens, scale, window, softcap):
    """float64, one request after the other; k, v [requests][keys, kv heads, dim]."""
    out, at = [], 0
    for i, n in enumerate(lens):
        group = q.shape[1] // k[i].shape[1]
        x, kk, vv = q[at:at + n].double(), k[i].double().repeat_interleave(group, 1), v[i].double().repeat_interleave(group, 1)
        score = torch.einsum("thd,shd->hts", x.cpu(), kk.cpu()).cuda() * scale
        if softcap:
            score = softcap * torch.tanh(score / softcap)
        gap = (torch.arange(n, device="cuda") + starts[i])[:, None] - torch.arange(k[i].shape[0], device="cuda")[None]
        score = score.masked_fill((gap < 0) | ((gap >= window) if window else False), float("-inf"))
        p = torch.softmax(score, -1)
        out.append(torch.stack([p[h] @ vv[:, h] for h in range(q.shape[1])], 1))
        at += n
    return torch.cat(out)


@pytest.mark.gpu
@pytest.mark.parametrize("heads, kv, dim, waves, tiles", [(8, 2, 64, 4, 1), (8, 2, 64, 8, 1), (4, 4, 64, 4, 4), (6, 2, 128, 4, 1), (6, 2, 128, 8, 1), (4, 1, 96, 4, 2),
                                                          (2, 2, 32, 4, 1), (4, 2, 64, 8, 2)])
@pytest.mark.parametrize("page, lens, starts, window, softcap", [(32, (300, 5, 77), (0, 40, 31), 0, 0.0), (64, (33, 257), (600, 1), 100, 0.0),
                                                                 (256, (31, 190), (8500, 0), 0, 20.0), (32, (1, 64), (0, 9000), 8400, 0.0)])
def test_prompts_attend_to_their_keys(heads, kv, dim, waves, tiles, page, lens, starts, window, softcap):
    """Tiles in several rounds and a partial one, walks of fewer steps than LDS holds and of more than the ring of places, steps that
    begin inside a window; slots past a request's last hold numbers that must not count (and no number at all in a page's keys)."""
    g = torch.Generator().manual_seed(dim + sum(lens))
    pages = [-(-(s + n) // page) for s, n in zip(starts, lens)]
    total = sum(lens)
    q = torch.randn(total, heads, dim, generator=g).to(BF).cuda()
    k_pool = torch.full((sum(pages), page, kv, dim), float("nan"), dtype=BF, device="cuda")
    v_pool = torch.full((sum(pages), kv, dim, page), 1e4, dtype=BF, device="cuda")
    tables = torch.zeros(len(lens), max(pages), dtype=torch.int32)
    order, at, ks, vs = torch.randperm(sum(pages), generator=g), 0, [], []
    for i, (s, n) in enumerate(zip(starts, lens)):
        mine = order[at:at + pages[i]]
        at += pages[i]
        tables[i, :pages[i]] = mine.int()
        ks.append(torch.randn(s + n, kv, dim, generator=g).to(BF).cuda())
        vs.append(torch.randn(s + n, kv, dim, generator=g).to(BF).cuda())
        for t0 in range(0, s + n, page):
            cut = ks[i][t0:t0 + page]
            k_pool[mine[t0 // page], :cut.shape[0]] = cut
            v_pool[mine[t0 // page], :, :, :cut.shape[0]] = vs[i][t0:t0 + page].permute(1, 2, 0)
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    tokens = waves * tiles * (16 // (heads // kv))
    where = torch.tensor(hip.attention_tiles(cu, list(starts), tokens), dtype=torch.int32).view(-1, 2).cuda()
    seq = torch.cat([torch.full((n,), i) for i, n in enumerate(lens)]).int().cuda()
    pos = torch.cat([torch.arange(s, s + n) for s, n in zip(starts, lens)]).int().cuda()
    got = hip.paged_attention_prefill(q, k_pool, v_pool.permute(0, 3, 1, 2), tables.cuda(), seq, pos, where, dim ** -0.5, window, tile_tokens=tokens, waves=waves, softcap=softcap)
    want = attended(q, ks, vs, starts, lens, dim ** -0.5, window, softcap)
    # weights and output in bfloat16: 2^-8 of the values' size a weight (they add up to 1), 2^-8 of the output
    bound = (2.0 ** -7) * max(float(v.abs().max()) for v in vs)
    assert bool(((got.double() - want).abs() <= bound).all()), float((got.double() - want).abs().max())
    assert float((got.double() - want).norm() / want.norm()) < 0.01


def test_heads_of_128_take_eight_waves_where_these_fill_the_chip_and_the_general_variant_keeps_single_tiles():
    shape = hip.prefill_shape
    assert shape(1501, 20, 4, 8, 3, 128, 500.0, False) == (40, 8) and shape(1024, 20, 4, 8, 3, 128, 512.0, False) == (20, 4)
    assert shape(1501, 20, 4, 8, 3, 128, 2000.0, False) == (20, 4) and shape(1501, 20, 4, 8, 3, 128, 500.0, True) == (20, 4)
    assert shape(2048, 32, 8, 8, 4, 64, 1024.0, True) == (16, 4) and shape(2048, 32, 8, 8, 4, 64, 1024.0, False) == (32, 8)


def test_wide_tiles_of_eight_waves_are_for_long_walks_and_whole_tiles_and_are_not_cut():
    """Steps that were measured (24 heads of 128 over 8, and 16 over 2): a short window, requests whose ends leave the wide tiles
    open, and a context long enough that so few workgroups would have their keys cut in chunks."""
    def plan(nh, nkv, lens, window=0):
        cu = [0]
        for n in lens:
            cu.append(cu[-1] + n)
        ctx = types.SimpleNamespace(scratch={}, host_cu_seqlens=cu, host_starts=[0] * len(lens), host_context_lens=lens)
        lead, tile_tokens, waves, _, splits, _ = hip._prefill_plan(torch.empty(cu[-1], nh, 128, dtype=BF), torch.empty(1, 32, nkv, 128, dtype=BF), ctx, True, False, window)
        assert lead == 0
        return tile_tokens, waves, splits
    assert plan(24, 8, [600, 901]) == plan(24, 8, [1500], 1024) == (40, 8, 1)
    assert plan(24, 8, [1500], 128) == plan(24, 8, [1500], 512) == plan(24, 8, [1500], -2048) == (20, 4, 1)
    assert plan(24, 8, [100] * 16) == (20, 4, 1) and plan(16, 16, [300] * 8) == (64, 4, 1)
    assert plan(16, 2, [3000]) == (16, 8, 1) and plan(16, 2, [2000]) == (8, 4, 1)


def test_requests_of_few_chunks_are_walked_only_where_the_chip_holds_them_at_once():
    """Sizes measured on both sides: 16 requests of a chunk each, of five, one and two requests; states of 32 places."""
    def walks(heads, vp, np, lens):
        chunks = [-(-n // 64) for n in lens]
        return hip.ssd_walks(sum(chunks), max(chunks), type("Z", (), dict(np=np, matrix=heads * vp * np)), len(lens))
    assert not walks(64, 64, 128, [64] * 16) and not walks(32, 128, 32, [64] * 16) and not walks(32, 128, 32, [128] * 8) and not walks(16, 64, 32, [30] * 24)
    assert walks(64, 64, 128, [300] * 16) and walks(64, 64, 128, [64]) and walks(64, 64, 128, [64] * 2) and walks(16, 64, 32, [64] * 8)
    assert not walks(32, 128, 32, [300] * 16) and walks(32, 128, 32, [304]) and walks(4, 64, 128, [300] * 16) and not walks(4, 64, 128, [2048])


def test_chunks_are_walked_where_their_states_are_many():
    def z(heads, vp, np):
        return type("Z", (), dict(np=np, matrix=heads * vp * np))
    assert hip.ssd_walks(32, 32, z(64, 64, 128)) and hip.ssd_walks(5, 5, z(64, 64, 128)) and hip.ssd_walks(17, 7, z(16, 128, 128))
    assert hip.ssd_walks(80, 5, z(4, 64, 128)) and hip.ssd_walks(1, 1, z(4, 64, 32))
    assert not hip.ssd_walks(32, 32, z(4, 64, 128)) and not hip.ssd_walks(32, 32, z(16, 128, 128)) and not hip.ssd_walks(32, 32, z(64, 64, 160))


@pytest.mark.gpu
@pytest.mark.parametrize("heads, vdim, groups, places", [(2, 16, 1, 32), (3, 37, 3, 64), (4, 64, 2, 96), (8, 80, 4, 128), (1, 130, 1, 100)])
@pytest.mark.parametrize("lengths", [[64], [1, 65, 130], [200, 37, 300], [128, 448]])
@pytest.mark.parametrize("one_decay", [False, True])
def test_a_walk_over_the_chunks_leaves_what_the_chunks_do(heads, vdim, groups, places, lengths, one_decay, monkeypatch):
    """The same states, bit for bit (the sums are the same), and outputs a rounding apart: two 32-bit sums of at most 64 and `places`
    terms that are added once more, so 2^-22 of what goes into them; channels that are no fours, places of none, a chunk's rest."""
    g = torch.Generator().manual_seed(sum(lengths) + heads)
    z = hip.SsdSizes(heads, vdim, groups, places, 4)
    total, slots = sum(lengths), list(range(len(lengths)))[::-1]
    mixed = torch.zeros(total, z.row)
    x, bc = mixed[:, :heads * z.vp].view(total, heads, z.vp), mixed[:, heads * z.vp:].view(total, 2 * groups, z.np)
    x[:, :, :vdim] = torch.randn(total, heads, vdim, generator=g)
    bc[:, :, :places] = torch.randn(total, 2 * groups, places, generator=g)
    shape = (heads,) if one_decay else (total, heads)
    steps, logs = (torch.rand(shape, generator=g) + 0.1).cuda(), -(torch.rand(shape, generator=g) ** 4 * 30).cuda()
    skip, start = torch.randn(heads, generator=g).cuda(), torch.randn(len(lengths), z.matrix + z.kept, generator=g).cuda()
    start[:, :z.matrix].view(-1, heads, z.vp, z.np)[:, :, vdim:] = 0.0
    mixed = mixed.to(BF).cuda()
    cu = [0]
    for n in lengths:
        cu.append(cu[-1] + n)
    found = []
    for walks in (True, False):
        ctx = type("Ctx", (), dict(num_seqs=len(lengths), num_tokens=total, max_query_len=max(lengths), host_cu_seqlens=cu, scratch={},
                                   cu_seqlens=torch.tensor(cu, dtype=torch.int32).cuda(), state_slots=torch.tensor(slots, dtype=torch.int32).cuda(),
                                   seq_of_token=torch.cat([torch.full((n,), i) for i, n in enumerate(lengths)]).int().cuda()))
        monkeypatch.setattr(hip, "ssd_walks", lambda *a, w=walks: w)
        state = start.clone()
        y = hip.ssd_scan(mixed, steps, logs, skip, state, ctx, z, chunks_from=1, keeps=torch.exp(logs) if one_decay else None)
        found.append((y, state))
    (y, state), (want, want_state) = found
    assert torch.equal(state, want_state)
    size = float(want.abs().max()) + float(start.abs().max()) * places ** 0.5 + 64.0
    assert float((y - want).abs().max()) <= 2.0 ** -22 * 8 * size


# (tokens at the edges of two and four blocks of 16 a wave, a block that ends early; columns in fours or not; a ragged reduction)
@pytest.mark.gpu
@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("heads, k, n", [(32, 72, 100), (32, 64, 256), (128, 128, 62)])
@pytest.mark.parametrize("x_type, y_type", [(torch.float32, torch.float32), (torch.float32, BF), (BF, torch.float32), (BF, BF)])
@pytest.mark.parametrize("tokens", [257, 512, 1000, 2065])
def test_products_per_head_are_the_same_bits_whatever_the_tokens(tokens, x_type, y_type, heads, k, n, gated):
    """Against the same rows 48 at a time (one block of tokens a wave), and against 64 bits: sums of k products good to k 2^-24 of the
    sum of their sizes, the gate to 2^-21, in bfloat16 half a unit in the last place more. Rows lie apart, what is beside them stays."""
    g = torch.Generator().manual_seed(tokens + n)
    x = torch.randn(tokens, heads, k, generator=g).to(x_type).cuda()
    w = (torch.randn(heads, n, k, generator=g) * k ** -0.5).to(BF).cuda().transpose(1, 2)
    gate = torch.randn(tokens, heads * n + 4, generator=g).cuda()[:, :heads * n] if gated else None
    kept = torch.full((tokens + 1, heads, n + 4), 7.0, dtype=y_type, device="cuda")
    out = hip.heads_gemm(x, w, kept[:tokens, :, :n], gate)
    few = torch.empty(tokens, heads, n, dtype=y_type, device="cuda")
    for a in range(0, tokens, 48):
        hip.heads_gemm(x[a:a + 48], w, few[a:a + 48], None if gate is None else gate[a:a + 48])
    assert torch.equal(out, few) and torch.all(kept[tokens] == 7.0) and torch.all(kept[:, :, n:] == 7.0)
    picked = [0, tokens // 2, tokens - 17, tokens - 1]
    xs, ws = x[picked].to(BF).double().cpu().transpose(0, 1), w.double().cpu()
    want, size = torch.bmm(xs, ws.contiguous()).transpose(0, 1), torch.bmm(xs.abs(), ws.abs().contiguous()).transpose(0, 1)
    if gated:
        turn = torch.sigmoid(gate[picked].double().cpu().view(len(picked), heads, n))
        want, size = want * turn, size * turn
    bound = size * (k * 2.0 ** -24 + (2.0 ** -21 if gated else 0.0)) + (want.abs() * 2.0 ** -8 if y_type == BF else 0.0)
    assert torch.all((out[picked].double().cpu() - want).abs() <= bound + 1e-30)


@pytest.mark.gpu
@pytest.mark.parametrize("x_type, y_type", [(torch.float32, torch.float32), (torch.float32, BF), (BF, BF)])
@pytest.mark.parametrize("heads, k, n", [(5, 72, 100), (32, 256, 64), (64, 64, 62), (130, 128, 192)])
@pytest.mark.parametrize("tokens", [1, 16, 17, 33])
def test_products_per_head_of_few_tokens_share_out_the_columns(tokens, x_type, y_type, heads, k, n):
    """A block of 16 tokens a workgroup and 16 columns a wave (up to 384 workgroups, and any number of them up to 16 tokens), with a gate: the bits of
    the same rows among 700, whose waves take all 64 columns; nothing beside them."""
    g = torch.Generator().manual_seed(tokens + heads)
    x = torch.randn(700, heads, k, generator=g).to(x_type).cuda()
    w = (torch.randn(heads, n, k, generator=g) * k ** -0.5).to(BF).cuda().transpose(1, 2)
    gate = torch.randn(700, heads * n, generator=g).cuda()
    whole, few = (torch.full((m + 1, heads, n + 4), 7.0, dtype=y_type, device="cuda") for m in (700, tokens))
    hip.heads_gemm(x, w, whole[:700, :, :n], gate)
    hip.heads_gemm(x[:tokens], w, few[:tokens, :, :n], gate[:tokens])
    assert torch.equal(few[:tokens], whole[:tokens]) and torch.all(few[tokens] == 7.0) and torch.all(few[:, :, n:] == 7.0)


def test_the_blocks_of_tokens_a_wave_takes_are_blocks_that_have_tokens():
    """Sizes that were measured on both sides of the rule's lines (latent_mfma.hip): few tokens of many heads keep one block a wave."""
    blocks = hip.library().ts_heads_gemm_blocks
    for x_type in (0, 1):
        assert [blocks(t, 128, 512, 128, x_type) for t in (1, 5, 48, 64)] == [1] * 4
        assert [blocks(t, 32, 256, 64, x_type) for t in (8, 64, 129, 200, 304)] == [1, 1, 1, 2, 2]
        assert blocks(1000, 24, 100, 40, x_type) == 1 and blocks(2048, 32, 256, 64, x_type) == 4
        assert blocks(100, 128, 512, 128, x_type) == 4 and blocks(2048, 32, 64, 256, x_type) == (4 if x_type else 2)


@pytest.mark.gpu
@pytest.mark.parametrize("x_type, y_type", [(torch.float32, torch.float32), (BF, BF), (BF, torch.float32)])
@pytest.mark.parametrize("tokens", [1, 17, 63, 64, 65])
def test_products_per_head_of_few_tokens_are_stored_as_those_of_many(tokens, x_type, y_type):
    """Results stored as they are (below 64 tokens, and 16-bit ones of one block) and turned: the same bits, nothing beside them."""
    g = torch.Generator().manual_seed(tokens)
    x = torch.randn(320, 64, 64, generator=g).to(x_type).cuda()
    w = (torch.randn(64, 132, 64, generator=g) / 8).to(BF).cuda().transpose(1, 2)
    whole, few = (torch.full((n + 1, 64, 136), 7.0, dtype=y_type, device="cuda") for n in (320, tokens))
    hip.heads_gemm(x, w, whole[:320, :, :132])
    hip.heads_gemm(x[:tokens], w, few[:tokens, :, :132])
    assert torch.equal(few[:tokens], whole[:tokens]) and torch.all(few[tokens] == 7.0) and torch.all(few[:, :, 132:] == 7.0)
