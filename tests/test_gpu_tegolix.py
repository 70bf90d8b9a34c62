"""The Tegolix decoder on the GPU against the plain implementation in tests/plain/tegolix.py: each mechanism's kernel
alone (with inputs made so that a fault shows: a token far back whose k v^T is the only thing a query finds in the
state, keys just inside and just outside a window at page borders, first tokens that read the kept row, states carried
over steps and slots that are used again), then whole models of four small configurations through trace replay (layer by
layer, whole, token by token, in portions down to two tokens, mixed batches on pages and state slots that are used
again, long decoding), and greedy generation through `LLM.generate` and the scheduler. float32 and bfloat16."""

from __future__ import annotations

import math

import pytest
import torch

from tests.helpers import prompt, tegolix_configs
from tests.plain import tegolix as plain
from tests.test_gpu_fanotar import paged, rounded, step_context, tolerance

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
F64 = torch.float64


def hip():
    from tinyserve_llm_amd.ops import hip as h
    return h


def dev(values):
    return torch.tensor(values, dtype=torch.int32, device=DEV)


# ---- the stream: a branch through an RMS norm and a scale per channel, the next norm on the way out ----------------

@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("width", [80, 99, 512, 4100])
def test_branch_through_its_norm_and_scale_into_the_stream(dtype, width):
    from tinyserve_llm_amd.parts.norm import ChannelScale, RMSNorm
    from tinyserve_llm_amd.parts.stream import ResidualStream
    n, eps = 6, 1e-5
    x = torch.randn(n, width) * 3
    a = torch.randn(n, width) * 0.01                                       # small rows: the norm, not the rows, sets the size
    wb, wb64 = rounded(torch.randn(width) * 0.2, dtype)
    wn, wn64 = rounded(torch.randn(width) * 0.2, dtype)
    ls, ls64 = rounded(torch.randn(width), dtype)
    post, nxt, scale = RMSNorm(width, eps, one_plus=True), RMSNorm(width, eps, one_plus=True), ChannelScale(width)
    post.bind({"weight": wb}), nxt.bind({"weight": wn}), scale.bind({"weight": ls})
    xd = x.to(DEV)
    stream = ResidualStream(xd, a.to(DEV), post=post, scale=scale.weight32)
    _, h = stream.take(nxt)
    want = x.to(F64) + plain.layer_norm(a.to(F64), wb64, eps) * ls64
    torch.testing.assert_close(xd.cpu().to(F64), want, atol=1e-5, rtol=1e-5)
    assert h.dtype == dtype and not stream.pending
    torch.testing.assert_close(h.cpu().to(F64), plain.layer_norm(want, wn64, eps), **tolerance(dtype))
    # the rows as an operand, without a norm; a plain weight and no scale; picked rows after a pending sum
    plain_post = RMSNorm(width, eps)
    plain_post.bind({"weight": wb})
    stream = ResidualStream(xd, a.to(DEV), post=plain_post)
    _, rows = stream.rows_as(dtype)
    want = want + plain.unit_rms(a.to(F64), eps) * wb64
    torch.testing.assert_close(rows.cpu().to(F64), want, **tolerance(dtype))
    stream = ResidualStream(xd, a.to(DEV), post=post, scale=scale.weight32)
    picked, _ = nxt(stream, None, dev([4, 0, 4]))
    want = want + plain.layer_norm(a.to(F64), wb64, eps) * ls64
    torch.testing.assert_close(picked.cpu().to(F64), plain.layer_norm(want[[4, 0, 4]], wn64, eps), **tolerance(dtype))


def test_two_mixers_sum_with_their_factors_and_the_gated_table_rows():
    h = hip()
    a, b = torch.randn(5, 70), torch.randn(5, 70)
    out = h.scaled_sum(a.to(DEV), 0.6, b.to(DEV), -1.1)
    torch.testing.assert_close(out.cpu().to(F64), 0.6 * a.to(F64) - 1.1 * b.to(F64), atol=1e-6, rtol=1e-6)
    sums = torch.randn(9, 7) * 2
    for dtype in (torch.float32, torch.bfloat16):
        table, t64 = rounded(torch.randn(30, 21), dtype)
        ids = [3, 29, 0, 3, 17, 5, 5, 28, 1]
        got = h.gather_gate(sums.to(DEV), table, 14, dev(ids), "gelu_tanh", dtype)
        want = plain.gelu_tanh(sums.to(F64)) * t64[ids][:, 14:21]
        torch.testing.assert_close(got.cpu().to(F64), want, **tolerance(dtype))


# ---- decays, the scan, the token shift ---------------------------------------------------------------------------------

def scan_case(read_first: bool, H: int, D: int, V: int, counts_by_step, slots, tau=3.0, seed=0, far=None, chunked=False):
    """Requests fed in unequal portions over several steps, each on its state slot; returns (kernel rows, oracle rows) per
    request. `far` = (request, position): that token's k and v are made large and the decays near 1, and every later
    query of the request is aligned with that k, so what it reads is what the state has kept of one token far back."""
    h = hip()
    gen = torch.Generator().manual_seed(seed)
    R = len(slots)
    totals = [sum(step[r] for step in counts_by_step) for r in range(R)]
    rnd = lambda *s: torch.randn(*s, generator=gen)
    q = [rnd(n, H * D) for n in totals]
    k = [rnd(n, H * D) for n in totals]
    v = [rnd(n, H * V) for n in totals]
    z = [rnd(n, H * D) * 2 for n in totals]
    bias = rnd(H * D)
    bonus = rnd(H, D) if read_first else None
    if far is not None:
        r, p = far
        bias = bias + (9.0 if not read_first else -9.0)                     # decays near 1 in either form
        k[r][p] *= 30.0
        v[r][p] *= 30.0
        q[r][p + 1:] = k[r][p] / 30.0 + 0.05 * q[r][p + 1:]
    state = torch.full((max(slots) + 2, H * D * V + 5), 7.0, device=DEV)        # (leftovers, and room behind S)
    state[slots] = 0.0
    got = [[] for _ in range(R)]
    fed = [0] * R
    for step in counts_by_step:
        live = [r for r in range(R) if step[r]]
        cat = lambda parts: torch.cat([parts[r][fed[r]:fed[r] + step[r]] for r in live]).to(DEV)
        cu = [0]
        for r in live:
            cu.append(cu[-1] + step[r])
        fused = torch.cat([cat(q), cat(k), cat(v)], dim=1).contiguous()           # columns of one projection, rows apart
        K = H * D
        o = h.decay_scan(fused[:, :K], fused[:, K:2 * K], fused[:, 2 * K:], cat(z), bias.to(DEV), state, dev(cu), dev([slots[r] for r in live]),
                         H, D, V, form="double_exponent" if read_first else "sigmoid_root", tau=tau, q_scale=1.0 if read_first else D ** -0.5,
                         bonus=None if bonus is None else bonus.to(DEV), longest=max(step),
                         ctx=step_context([[0]] * len(live), 4096, [0] * len(live), [step[r] for r in live], slots=[slots[r] for r in live]) if chunked else None)
        for i, r in enumerate(live):
            got[r].append(o[cu[i]:cu[i + 1]].cpu())
            fed[r] += step[r]
    assert torch.all(state[max(slots) + 1] == 7.0) and torch.all(state[slots][:, H * D * V:] == 0.0), "nothing beside the states is written"
    want = []
    for r in range(R):
        S = torch.zeros(H, D, V, dtype=F64)
        rows = []
        for t in range(totals[r]):
            qq, kk, vv = q[r][t].to(F64).reshape(H, D), k[r][t].to(F64).reshape(H, D), v[r][t].to(F64).reshape(H, V)
            zz = (z[r][t].to(F64) + bias.to(F64)).reshape(H, D)
            kv = kk[:, :, None] * vv[:, None, :]
            if read_first:
                w = torch.exp(-torch.exp(zz))
                rows.append(torch.einsum("hkv,hk->hv", S + bonus.to(F64)[:, :, None] * kv, qq).reshape(-1))
                S = w[:, :, None] * S + kv
            else:
                w = torch.exp(torch.nn.functional.logsigmoid(zz) / tau)
                S = w[:, :, None] * S + kv
                rows.append(torch.einsum("hkv,hk->hv", S, qq * D ** -0.5).reshape(-1))
        want.append(torch.stack(rows))
    return [torch.cat(g) for g in got], want


@pytest.mark.parametrize("read_first", [False, True])
@pytest.mark.parametrize("sizes", [(3, 20, 28), (1, 16, 16), (2, 4, 70), (2, 18, 270), (1, 300, 12), (4, 64, 128), (2, 128, 64), (1, 256, 16)])
def test_decay_scan_over_unequal_requests_in_unequal_portions(read_first, sizes):
    H, D, V = sizes
    steps = [[5, 1, 0], [1, 40, 2], [17, 1, 1], [0, 2, 33], [1, 1, 1]]
    got, want = scan_case(read_first, H, D, V, steps, slots=[2, 0, 3], seed=D + V)
    for g, w in zip(got, want):
        torch.testing.assert_close(g.to(F64), w, atol=2e-4 * float(w.abs().max()), rtol=1e-4)


@pytest.mark.parametrize("read_first", [False, True])
@pytest.mark.parametrize("sizes", [(3, 32, 64), (2, 64, 128), (5, 64, 64), (2, 128, 64), (1, 128, 256), (2, 32, 320)])
def test_long_portions_in_chunks(read_first, sizes):
    """Portions from the shortest that is worked in chunks on, whole chunks and ragged ends (one token, a block's edge), beside
    requests that are walked, states handed from chunks to walk and back. The bound: a number is a sum of at most
    D + 64 products beside what the state's 32-bit numbers carry, each rounding good to 2^-24."""
    H, D, V = sizes
    least = hip().DECAY_CHUNKS_FROM
    steps = [[least, 3, 0], [1, least + 129, least + 16], [least + 63, 1, least + 47], [70, 0, 2]]
    got, want = scan_case(read_first, H, D, V, steps, slots=[2, 0, 3], seed=D + V, chunked=True)
    for g, w in zip(got, want):
        torch.testing.assert_close(g.to(F64), w, atol=(D + 64) * 2.0 ** -24 * float(w.abs().max()), rtol=1e-5)


@pytest.mark.parametrize("read_first", [False, True])
@pytest.mark.parametrize("sizes", [(8, 64, 64), (4, 128, 128), (2, 128, 256)])
def test_chunks_are_no_further_from_64_bits_than_the_walk(read_first, sizes):
    """Read-outs and states of both against the recurrence in 64 bits from the same 32-bit inputs, root mean square: the
    chunks' order of sums costs no precision."""
    h = hip()
    H, D, V = sizes
    n, gen = 1030, torch.Generator().manual_seed(D + V)
    rand = lambda *shape: torch.randn(*shape, generator=gen).to(DEV)
    q, k, v, z, bias, start = rand(n, H * D), rand(n, H * D), rand(n, H * V), rand(n, H * D) * 1.5, rand(H * D) + (-1.0 if read_first else 2.0), rand(1, H * D * V)
    bonus, q_scale = (rand(H, D) * 0.5, 1.0) if read_first else (None, D ** -0.5)
    zz = (z + bias).to(F64)
    w = (torch.exp(-torch.exp(zz)) if read_first else torch.exp(torch.nn.functional.logsigmoid(zz) / 16.0)).view(n, H, D, 1)
    S, rows = start.to(F64).view(H, D, V), []
    for t in range(n):
        kv = k[t].to(F64).view(H, D, 1) * v[t].to(F64).view(H, 1, V)
        if not read_first:
            S = w[t] * S + kv
        read = S + bonus.to(F64)[:, :, None] * kv if read_first else S
        rows.append((q[t].to(F64).view(H, 1, D) * q_scale @ read).view(-1))
        if read_first:
            S = w[t] * S + kv
    want, off = torch.stack(rows), []
    for ctx in (None, step_context([[0]], 4096, [0], [n], slots=[0])):
        state, dev = start.clone(), lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
        out = h.decay_scan(q, k, v, z, bias, state, dev([0, n]), dev([0]), H, D, V, form="double_exponent" if read_first else "sigmoid_root", tau=16.0,
                           q_scale=q_scale, bonus=bonus, longest=n, ctx=ctx)
        off.append([float((a.to(F64) - b).norm() / b.norm()) for a, b in ((out, want), (state.view(H, D, V), S))])
    (walk, walk_state), (chunks, chunk_state) = off
    assert 0.0 < chunks <= walk and 0.0 < chunk_state <= walk_state, off      # (the walk is the measure; a state's error grows with its memory)


@pytest.mark.parametrize("chunked", [False, True])
@pytest.mark.parametrize("read_first", [False, True])
def test_a_token_far_back_is_still_in_the_state(read_first, chunked):
    """Position 3 of 700 (or 2,400) stands out; the request is fed in portions and then token by token. A state that is dropped between
    steps, decayed in the wrong order, or read from the wrong slot loses it."""
    steps = [[1300 if chunked else 300], [64], [2], [900 if chunked else 200]] + [[1]] * 134
    got, want = scan_case(read_first, 2, 32, 64 if chunked else 48, steps, slots=[1], far=(0, 3), seed=5, chunked=chunked)
    assert float(want[0][-1].abs().max()) > 50 * float(want[0][2].abs().max()), "the far token dominates the last read-out"
    torch.testing.assert_close(got[0].to(F64), want[0], atol=3e-4 * float(want[0].abs().max()), rtol=2e-4)


def test_the_bonus_is_for_the_current_token_only_and_tau_roots_the_decay():
    h = hip()
    # one head, one channel each: numbers that can be followed by hand
    one = lambda x: torch.tensor([[x]], dtype=torch.float32, device=DEV)
    state = torch.zeros(1, 1, device=DEV)
    args = dict(cu_seqlens=dev([0, 1]), state_slots=dev([0]), heads=1, dim=1, vdim=1)
    o1 = h.decay_scan(one(2.0), one(3.0), one(5.0), one(0.0), torch.zeros(1, device=DEV), state, **args, form="double_exponent",
                      bonus=torch.full((1, 1), 0.5, device=DEV))
    assert float(o1) == pytest.approx(2.0 * 0.5 * 15.0) and float(state) == pytest.approx(15.0)
    o2 = h.decay_scan(one(1.0), one(0.0), one(0.0), one(0.0), torch.zeros(1, device=DEV), state, **args, form="double_exponent",
                      bonus=torch.full((1, 1), 0.5, device=DEV))
    assert float(o2) == pytest.approx(15.0), "the state is read before it decays, and without the bonus"
    assert float(state) == pytest.approx(15.0 * math.exp(-1.0))
    state.zero_()
    h.decay_scan(one(1.0), one(1.0), one(8.0), one(0.0), torch.zeros(1, device=DEV), state, **args, form="sigmoid_root", tau=2.0)
    o = h.decay_scan(one(1.0), one(0.0), one(0.0), one(0.0), torch.zeros(1, device=DEV), state, **args, form="sigmoid_root", tau=2.0)
    assert float(o) == pytest.approx(8.0 * math.sqrt(0.5), rel=1e-6), "sigmoid(0)^(1/2), applied before the read-out"


@pytest.mark.parametrize("listed", [False, True])
def test_a_step_recorded_before_its_chunks_are_listed(listed):
    """A long portion is recorded as its context comes, as the walk; where an eager step listed the chunks before, as the
    chunks. Replays from fresh states with the inputs changed and eager work in between."""
    h = hip()
    H, D, V, n = 2, 64, 64, 800
    gen = torch.Generator().manual_seed(3)
    rand = lambda *shape: torch.randn(*shape, generator=gen).to(DEV)
    k, v, z, bias, start = rand(n, H * D), rand(n, H * V), rand(n, H * D), rand(H * D) + 2.0, rand(1, H * D * V)
    queries, cu, slots = [rand(n, H * D) for _ in range(4)], dev([0, n]), dev([0])
    scan = lambda q, state, ctx: h.decay_scan(q, k, v, z, bias, state, cu, slots, H, D, V, form="sigmoid_root", tau=2.0, longest=n, ctx=ctx)
    ctx, q, state = step_context([[0]], 4096, [0], [n], slots=[0]), queries[0].clone(), start.clone()
    if listed:
        scan(q, start.clone(), ctx)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = scan(q, state, ctx)
    for given in queries:
        want_state = start.clone()
        want = scan(given, want_state, step_context([[0]], 4096, [0], [n], slots=[0]) if listed else None)
        q.copy_(given)
        state.copy_(start)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(state, want_state)


@pytest.mark.parametrize("read_first", [False, True])
@pytest.mark.parametrize("sizes", [(2, 64, 128), (3, 20, 64), (1, 256, 256), (2, 128, 72)])
def test_wide_and_narrow_slices_of_the_columns_give_the_same_bits(read_first, sizes):
    """Steps of few tokens a request give a wave 64 value columns, steps of many 16: a request decoded token by token and the
    same request fed whole must not differ by a bit."""
    h = hip()
    H, D, V = sizes
    gen = torch.Generator().manual_seed(D)
    n = 9
    q, k, z = (torch.randn(n, H * D, generator=gen).to(DEV) for _ in range(3))
    v = torch.randn(n, H * V, generator=gen).to(DEV)
    bias, bonus = torch.randn(H * D, generator=gen).to(DEV), torch.randn(H, D, generator=gen).to(DEV)
    kw = dict(heads=H, dim=D, vdim=V, form="double_exponent" if read_first else "sigmoid_root", tau=2.0, bonus=bonus if read_first else None)
    whole_state, stepped_state = torch.zeros(1, H * D * V, device=DEV), torch.zeros(1, H * D * V, device=DEV)
    whole = h.decay_scan(q, k, v, z, bias, whole_state, dev([0, n]), dev([0]), **kw, longest=n)
    stepped = torch.cat([h.decay_scan(q[t:t + 1], k[t:t + 1], v[t:t + 1], z[t:t + 1], bias, stepped_state, dev([0, 1]), dev([0]), **kw, longest=1)
                         for t in range(n)])
    assert torch.equal(whole, stepped) and torch.equal(whole_state, stepped_state)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_token_shift_reads_the_kept_row_and_leaves_the_last(dtype):
    h = hip()
    W, mixes = 70, 5
    mu = torch.rand(mixes, W)
    kept = torch.randn(6, W + 3, device=DEV)[:, 3:]                          # rows apart, as inside a wider state
    before = kept.clone()
    x, x64 = rounded(torch.randn(9, W), dtype)
    ctx = step_context([[0], [0], [0]], 16, [4, 0, 9], [3, 1, 5], slots=[4, 1, 2])
    out = h.token_shift(x, mu.to(DEV), kept, ctx)
    h.token_shift_keep(kept, x, ctx)
    first = {0: 4, 3: 1, 4: 2}
    for t in range(9):
        prev = before[first[t]].cpu().to(F64) if t in first else x64[t - 1]
        for s in range(mixes):
            torch.testing.assert_close(out[s, t].cpu().to(F64), x64[t] + (prev - x64[t]) * mu[s].to(F64), **tolerance(dtype))
    for slot, last in ((4, 2), (1, 3), (2, 8)):
        torch.testing.assert_close(kept[slot].cpu().to(F64), x64[last], atol=0, rtol=0)
    assert torch.equal(kept[[0, 3, 5]], before[[0, 3, 5]])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,width,mixes", [(65540, 8, 1), (7400, 72, 5), (523, 1024, 3), (259, 2056, 5)])
def test_token_shift_in_whole_pieces(dtype, n, width, mixes):
    """Many rows of whole 16-byte pieces take eight elements a thread; kept rows that begin elsewhere take one. The same bits."""
    from types import SimpleNamespace
    h = hip()
    mu = torch.rand(mixes, width, device=DEV)
    wide = torch.randn(6, width + 8, device=DEV)
    apart = torch.empty(6, width + 8, device=DEV)
    apart[:, 3:3 + width] = wide[:, 4:4 + width]
    x, _ = rounded(torch.randn(n, width), dtype)
    ints = lambda t: torch.tensor(t, dtype=torch.int32, device=DEV)
    ctx = SimpleNamespace(cu_seqlens=ints([0, 1, n - 7, n]), seq_of_token=ints([0] + [1] * (n - 8) + [2] * 7), state_slots=ints([4, 1, 2]))
    assert torch.equal(h.token_shift(x, mu, wide[:, 4:4 + width], ctx), h.token_shift(x, mu, apart[:, 3:3 + width], ctx))


@pytest.mark.parametrize("n,width,mixes", [(76804, 8, 1), (8540, 72, 5), (601, 1024, 3), (300, 2056, 5)])
def test_token_shift_of_enough_pieces(n, width, mixes):
    """The least numbers of rows that go in pieces (76,800 of them in bfloat16), a last workgroup that is not full."""
    test_token_shift_in_whole_pieces(torch.bfloat16, n, width, mixes)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("lengths,width", [([1], 70), ([1] * 48, 2048), ([1] * 299, 2056), ([1, 1, 3], 264), ([1, 0, 2], 72)])
def test_token_shift_keeps_the_rows_of_a_decode_step(dtype, lengths, width):
    """One launch for a step of one token a request (up to 614,400 numbers), two for others: the bits of the two calls, other slots as they were."""
    from types import SimpleNamespace
    h = hip()
    n, requests = sum(lengths), len(lengths)
    mu, state = torch.rand(5, width, device=DEV), torch.randn(requests + 2, width + 3, device=DEV)
    x, _ = rounded(torch.randn(n, width), dtype)
    ints = lambda t: torch.tensor(t, dtype=torch.int32, device=DEV)
    cu = [sum(lengths[:i]) for i in range(requests + 1)]
    ctx = SimpleNamespace(cu_seqlens=ints(cu), seq_of_token=ints([i for i, m in enumerate(lengths) for _ in range(m)]), num_seqs=requests,
                          max_query_len=max(lengths), state_slots=torch.randperm(requests + 2, device=DEV)[:requests].int())
    one, two = state.clone(), state.clone()
    got = h.token_shift(x, mu, one[:, 3:], ctx, keep=True)
    want = h.token_shift(x, mu, two[:, 3:], ctx)
    h.token_shift_keep(two[:, 3:], x, ctx)
    assert torch.equal(got, want) and torch.equal(one, two) and not torch.equal(one, state)


@pytest.mark.parametrize("shared", [True, False])
def test_heads_norm_weight_and_silu_gate(shared):
    h = hip()
    H, V, n, eps = 3, 28, 5, 1e-5
    o, gate = torch.randn(n, H * V) * 4, torch.randn(n, H * V + 9)
    w = torch.randn(V if shared else H * V)
    got = h.mlstm_finish(o.to(DEV), w.to(DEV), gate.to(DEV)[:, 9:], H, V, eps, torch.float32, silu_gate=True)
    g64 = gate[:, 9:].to(F64)
    weight = (w.to(F64).repeat(H) if shared else w.to(F64))
    want = plain.unit_rms(o.to(F64).reshape(n, H, V), eps).reshape(n, H * V) * weight * g64 * torch.sigmoid(g64)
    torch.testing.assert_close(got.cpu().to(F64), want, atol=1e-5, rtol=1e-5)


# ---- the attention side: weighted head norms before the turn, values that turn, the window, the gate per head ---------

@pytest.mark.parametrize("shape", [(4, 2, 32, 48), (3, 1, 20, 12), (2, 2, 16, 16), (5, 1, 80, 160)])
def test_head_norms_and_turned_values_in_place(shape):
    h = hip()
    H, G, D, V = shape
    positions, eps = [0, 1, 15, 16, 700, 70000], 1e-5
    rows = torch.randn(len(positions), (H + G) * D + G * V) * 3
    wq, wk = 1 + 0.2 * torch.randn(D), 1 + 0.2 * torch.randn(D)
    freqs, _ = plain.rotary_frequencies(V, 9000.0, None)
    d = rows.to(DEV)
    h.qkv_prepare(d, dev(positions), H, G, D, V, q_weight=wq.to(DEV), k_weight=wk.to(DEV), eps=eps, value_freqs=freqs.to(DEV))
    r, pos = rows.to(F64), torch.tensor(positions)
    want_q = plain.unit_rms(r[:, :H * D].reshape(-1, H, D), eps) * wq.to(F64)
    want_k = plain.unit_rms(r[:, H * D:(H + G) * D].reshape(-1, G, D), eps) * wk.to(F64)
    want_v = plain.rotate_halves(r[:, (H + G) * D:].reshape(-1, G, V), pos, freqs)
    torch.testing.assert_close(d[:, :H * D].cpu().to(F64).reshape(-1, H, D), want_q, atol=2e-5, rtol=1e-5)
    torch.testing.assert_close(d[:, H * D:(H + G) * D].cpu().to(F64).reshape(-1, G, D), want_k, atol=2e-5, rtol=1e-5)
    torch.testing.assert_close(d[:, (H + G) * D:].cpu().to(F64).reshape(-1, G, V), want_v, atol=5e-5, rtol=1e-5)
    # turned back by the same positions, with a gate per head
    for dtype in (torch.float32, torch.bfloat16):
        o, o64 = rounded(torch.randn(len(positions), H, V), dtype)
        gate = torch.randn(len(positions), H + 2)
        h.rotate_heads(o, o, freqs.to(DEV), 1.0, dev(positions), interleaved=False, back=True, gate=gate.to(DEV)[:, 2:])
        want = plain.rotate_halves(o64, pos, freqs, back=True) * torch.sigmoid(gate[:, 2:].to(F64))[:, :, None]
        torch.testing.assert_close(o.cpu().to(F64), want, **tolerance(dtype))


def attention_mixer(dtype, m: dict, width: int, eps: float, seed: int):
    """The engine's attention part with the design's options and random weights, and the same weights for the oracle."""
    from tinyserve_llm_amd.parts.attention import GeneralAttention
    from tinyserve_llm_amd.parts.rope import RotaryFrequencies
    rot = m["rot"]
    enc = {"qk": RotaryFrequencies(rot["dims"], rot["base"], interleaved=False, ramp=rot.get("scaling")),
           "v": RotaryFrequencies(m["vdim"], rot["base"], interleaved=False)}
    for e in enc.values():
        e.prepare(torch.device(DEV))
    part = GeneralAttention(width, m["heads"], m["kv_heads"], m["dim"], m["vdim"], position="qk" if rot["dims"] else None, scale=m["scale"],
                            softcap=m.get("softcap", 0.0), window=m["mask"]["size"] if m.get("mask") else 0, head_norm_eps=eps,
                            value_position="v", head_gate=True)
    gen = torch.Generator().manual_seed(seed)
    H, G, D, V = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
    shapes = {"q": (H * D, width), "k": (G * D, width), "v": (G * V, width), "g": (H, width), "o": (width, H * V)}
    W = {n: torch.randn(s, generator=gen) * s[1] ** -0.5 for n, s in shapes.items()}
    W["q.norm"], W["k.norm"] = 1 + 0.2 * torch.randn(D, generator=gen), 1 + 0.2 * torch.randn(D, generator=gen)
    stored = {n: (t.to(dtype) if t.dim() == 2 else t) for n, t in W.items()}
    part.bind({"qkv": torch.cat([stored["q"], stored["k"], stored["v"]]).to(DEV), "o": stored["o"].to(DEV), "gate": stored["g"].to(DEV),
               "q_norm": W["q.norm"].to(DEV), "k_norm": W["k.norm"].to(DEV)})
    return part, enc, {n: t.to(F64) for n, t in stored.items()}


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("case", [
    dict(heads=4, kv_heads=2, dim=32, vdim=48, scale=0.5, softcap=6.0, mask={"size": 24}, rot={"dims": 16, "base": 10000.0,
         "scaling": {"factor": 3.0, "original": 64.0, "fast": 16.0, "slow": 2.0}}),
    dict(heads=2, kv_heads=2, dim=16, vdim=16, scale=0.7, mask={"size": 1}, rot={"dims": 16, "base": 700.0}),
    dict(heads=4, kv_heads=1, dim=8, vdim=24, scale=0.6, softcap=30.0, rot={"dims": 0, "base": 300.0}),
    dict(heads=8, kv_heads=2, dim=64, vdim=64, scale=0.3, softcap=15.0, mask={"size": 33}, rot={"dims": 32, "base": 250000.0}),
    dict(heads=3, kv_heads=1, dim=80, vdim=160, scale=0.2, softcap=12.0, mask={"size": 17}, rot={"dims": 40, "base": 20000.0}),
])
def test_attention_side_in_portions_over_shuffled_pages(dtype, case):
    """The whole left mixer against the oracle: a request of 83 tokens fed as 40 + 2 + 1 + 1 + 39 on pages of 16 in a
    shuffled order, beside a second request that starts later on pages the first has not got. Sharp scores (large query
    and key weights) make every position's output hang on few keys, so a window that is one off, a value turned by the
    wrong position or a page read at the wrong place shows."""
    from tinyserve_llm_amd.parts.base import LayerMemory
    width, eps, page = 72, 1e-5, 16
    part, enc, W = attention_mixer(dtype, case, width, eps, seed=case["dim"])
    gen = torch.Generator().manual_seed(1)
    lengths = [83, 30]
    hs = [rounded(torch.randn(n, width, generator=gen), dtype) for n in lengths]
    k, v = paged(12, page, case["kv_heads"], case["dim"], case["vdim"], dtype)
    tables = [[7, 2, 9, 0, 5, 11], [4, 10]]
    mem = LayerMemory(k_cache=k, v_cache=v, space=0, store=True)
    cuts = [[40, 2, 1, 1, 39], [0, 0, 7, 1, 22]]
    fed = [0, 0]
    got = [[], []]
    for step in range(5):
        live = [r for r in range(2) if cuts[r][step]]
        counts = [cuts[r][step] for r in live]
        ctx = step_context([tables[r] for r in live], page, [fed[r] for r in live], counts)
        ctx.position_encodings = enc
        x = torch.cat([hs[r][0][fed[r]:fed[r] + n] for r, n in zip(live, counts)])
        out = part.forward(x, ctx, mem)
        at = 0
        for r, n in zip(live, counts):
            got[r].append(out[at:at + n].cpu())
            at += n
            fed[r] += n
    for r in range(2):
        want = plain.left_attention(hs[r][1], torch.arange(lengths[r]), W, case, eps, {})
        tol = dict(atol=1e-4, rtol=1e-4) if dtype == torch.float32 else dict(atol=6e-2, rtol=3e-2)
        torch.testing.assert_close(torch.cat(got[r]).to(F64), want, **tol)


@pytest.mark.parametrize("window", [1, 2, 15, 16, 17, 40, 64, 65])
@pytest.mark.parametrize("decoded", [False, True])
def test_keys_just_inside_and_just_outside_the_window(window, decoded):
    """One key stands out for every query: the oldest one the window keeps, or the one just before it, which must not be
    seen at all. Values of a size of their own, capped scores, pages of 16; prompts and single decoded tokens."""
    h = hip()
    H, G, D, V, page, length = 2, 1, 24, 40, 16, 150
    gen = torch.Generator().manual_seed(window)
    k64 = plain.unit_rms(torch.randn(length, G, D, generator=gen, dtype=F64), 0.0)
    v64 = torch.randn(length, G, V, generator=gen, dtype=F64)
    k, v = paged(10, page, G, D, V, torch.float32)
    table = [3, 8, 0, 5, 9, 1, 7, 2, 6, 4]
    for j in range(length):
        k[table[j // page], j % page] = k64[j].float().to(DEV)
        v[table[j // page], j % page] = v64[j].float().to(DEV)
    for inside in (True, False):
        queries = list(range(length)) if not decoded else [0, window - 1, window, window + 1, 2 * window, 99, 149]
        queries = [i for i in queries if i < length]
        q64 = torch.randn(len(queries), H, D, generator=gen, dtype=F64) * 0.1
        for n, i in enumerate(queries):
            j = i - window + 1 if inside else i - window
            if j >= 0:
                q64[n] += 40.0 * k64[j, 0]
        if decoded:
            ctx = step_context([table] * len(queries), page, queries, [1] * len(queries))
        else:
            ctx = step_context([table], page, [0], [length])
        out = h.paged_attention(q64.float().to(DEV), k, v, ctx, 0, 1.0, window, softcap=25.0)
        want = plain.window_attention(q64.float().to(F64), k64.float().to(F64), v64.float().to(F64), torch.tensor(queries), 1.0, 25.0, window)
        torch.testing.assert_close(out.cpu().to(F64), want, atol=2e-4, rtol=1e-4)


# ---- the router over all outputs, identity experts, the shared expert's gate ---------------------------------------

@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("sizes", [(6, 2, 3, 80, 40, 23), (4, 0, 1, 48, 20, 5), (3, 3, 6, 99, 17, 9), (8, 4, 3, 256, 64, 70), (8, 2, 2, 512, 128, 300)])
def test_softmax_over_all_outputs_identity_experts_and_a_gated_shared_expert(dtype, sizes):
    from tinyserve_llm_amd.parts.moe import RoutedExperts
    E, I, top, W, F, n = sizes
    part = RoutedExperts(W, E, top, F, limit=0.0, slope=1.0, up_shift=0.0, router_scale=1.0, normalize=False, correction=True,
                         shared=dict(intermediate_size=F + 8, limit=0.0, slope=1.0, up_shift=0.0), scoring="softmax_all", identity=I, shared_gate=True)
    gen = torch.Generator().manual_seed(E * 10 + I)
    router = torch.randn(E + I + 1, W, generator=gen) * 0.3
    correction = torch.randn(E + I, generator=gen) * 0.1
    mats = {name: rounded(torch.randn(*shape, generator=gen) * shape[-1] ** -0.5 * 1.5, dtype)
            for name, shape in (("gate_up", (E, 2 * F, W)), ("down", (E, W, F)), ("shared_gate_up", (2 * (F + 8), W)), ("shared_down", (W, F + 8)))}
    part.bind({"router": router.to(DEV), "correction": correction.to(DEV), **{k: t[0] for k, t in mats.items()}})
    x, x64 = rounded(torch.randn(n, W, generator=gen), dtype)
    out = part.forward(x, None)
    Wd = {"router": router[:E + I].to(F64), "correction": correction.to(F64), "shared.sg": router[E + I:].to(F64)}
    for e in range(E):
        Wd[f"e{e}.gate"], Wd[f"e{e}.up"], Wd[f"e{e}.down"] = mats["gate_up"][1][e, :F], mats["gate_up"][1][e, F:], mats["down"][1][e]
    Wd["shared.gate"], Wd["shared.up"], Wd["shared.down"] = mats["shared_gate_up"][1][:F + 8], mats["shared_gate_up"][1][F + 8:], mats["shared_down"][1]
    mlp = {"router": {"experts": E, "identity": I, "top": top}, "shared": {"ff": F + 8}}
    want = plain.expert_mixture(x64, Wd, mlp)
    s = torch.softmax(x64 @ Wd["router"].T, -1) + Wd["correction"]
    ranked = torch.sort(s, descending=True).values
    sure = [t for t in range(n) if top >= E + I or float(ranked[t, top - 1] - ranked[t, top]) > 1e-3]      # (no close calls are made)
    assert len(sure) > n // 2
    tol = dict(atol=1e-4, rtol=1e-4) if dtype == torch.float32 else dict(atol=5e-2, rtol=3e-2)
    torch.testing.assert_close(out[sure].cpu().to(F64), want[sure], **tol)


def test_relu_gated_unit():
    h = hip()
    sums = torch.randn(6, 2 * 37) * 2
    got = h.capped_glu(sums.to(DEV), 0.0, 1.0, 0.0, torch.float32, activation="relu")
    torch.testing.assert_close(got.cpu(), torch.relu(sums[:, :37]) * sums[:, 37:], atol=1e-6, rtol=1e-6)


# ---- whole models through trace replay ---------------------------------------------------------------

LENGTHS = {"P": [1, 23, 97, 200], "Q": [1, 30, 75, 150], "R": [2, 19, 66, 131], "S": [1, 40, 140], "T": [3, 50, 120]}
TOL = {"float32": 2e-4, "bfloat16": 6e-2}       # of the spread of the oracle's logits
# A router's choice is discrete: where the oracle's last chosen expert leads the best one left out by less than the
# engine's rounding of the scores, either choice is right, and what follows in the request (the states carry it on) is
# no longer comparable. Positions from a request's first such close call on are left out of the comparison.
CLOSE_CALL = {"float32": 2e-6, "bfloat16": 4e-3}


def oracle_rows(oracle, prompts):
    """The oracle's logits per prompt, each with the first position at which a router's choice is a close call for every type."""
    rows = []
    for p in prompts:
        logits = oracle.logits(p)
        first = {d: next((i for i, m in enumerate(oracle.margins.tolist()) if m < c), len(p)) for d, c in CLOSE_CALL.items()}
        rows.append(Rows(logits, first))
    return rows


class Rows:
    def __init__(self, logits, comparable):
        self.logits, self.comparable = logits, comparable

    def __getitem__(self, pos):
        return self.logits[pos]


@pytest.fixture(scope="module", params=["P", "Q", "R", "S", "T"])
def case(request, tmp_path_factory):
    from tinyserve_llm_amd.weights.random_init import write_random_model
    name = request.param
    config, seed = tegolix_configs()[name]
    folder = str(tmp_path_factory.mktemp(f"tegolix_{name}"))
    write_random_model(folder, config, seed, torch.bfloat16)
    oracle = plain.PlainTegolix.from_folder(folder)
    prompts = [prompt(500 + i, n, config.vocab) for i, n in enumerate(LENGTHS[name])]
    return name, folder, config, prompts, oracle, oracle_rows(oracle, prompts)


def replayer(folder, dtype, max_tokens):
    from tinyserve_llm_amd.engine.replay import Replay
    return Replay(folder, dtype, max_tokens)


def check(got, oracle_rows, dtype):
    """float32: every row within the tolerance. bfloat16: the design has places where a rounding decides something
    discrete (a router's choice that `CLOSE_CALL` does not catch because the stream before it has drifted; the sign of
    q.k where a head's state holds one token and the head's norm then makes a unit row of either sign), and the
    states carry what follows from it through the rest of the request. So in bfloat16 the typical row has to be
    within the tolerance and four rows of five as well; a fault of a bfloat16 kernel moves most rows."""
    assert got, "nothing was compared"
    spread = float(torch.cat([o.logits.flatten() for o in oracle_rows]).std())
    errors = []
    for (r, pos), row in got.items():
        if pos >= oracle_rows[r].comparable[dtype]:
            continue
        want = oracle_rows[r][pos]
        if dtype == "float32":
            torch.testing.assert_close(row.double().cpu(), want, atol=TOL[dtype] * spread, rtol=0.0,
                                       msg=lambda m: f"request {r} position {pos}: {m}")
        errors.append(float((row.double().cpu() - want).abs().max()) / spread)
    assert errors, "every position lies behind a close call of a router"
    errors.sort()
    if dtype != "float32" and len(errors) < 5:
        assert errors[0] <= TOL[dtype], f"the best of {len(errors)} rows is off by {errors[0]:.3f} of the logits' spread"
    elif dtype != "float32":
        assert errors[len(errors) // 2] <= TOL[dtype], f"the median row is off by {errors[len(errors) // 2]:.3f} of the logits' spread"
        over = sum(e > TOL[dtype] for e in errors)
        assert over <= len(errors) // 5, f"{over} of {len(errors)} rows are off by more than {TOL[dtype]} of the logits' spread"
    print(f"[{dtype}] worst logit error {errors[-1]:.3e}, median {errors[len(errors) // 2]:.3e} of the logits' spread ({spread:.2f}) over {len(errors)} of {len(got)} rows")


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
        # the residual stream after every layer, one by one
        from tinyserve_llm_amd.engine.runner import StepEntry
        from tinyserve_llm_amd.parts import base
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
            now = hidden.settle()[0]
            scale = float(want[i].abs().max())
            torch.testing.assert_close(now.cpu().double(), want[i], atol=2e-5 * max(1.0, scale), rtol=1e-5, msg=lambda m: f"after layer {i}: {m}")


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_prompt_then_token_by_token(case, dtype):
    """The last tokens one by one: more of them than a page and than most windows hold."""
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
    state slots that earlier ones have written and given back, beside others that are in the middle of theirs. A state or
    a kept row that is not cleared, or a stale page, shows in the logits."""
    name, folder, config, _, oracle, _ = case
    lengths = [129, 70, 40, 1, 65, 100, 128, 30, 150]
    prompts = [prompt(900 + i, n, config.vocab) for i, n in enumerate(lengths)]
    rows = oracle_rows(oracle, prompts)
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
    """Steps of hundreds of tokens: a prompt of 520 tokens whole, and cut where the second portion starts in the middle of
    a page and of a window, beside a short request."""
    name, folder, config, _, oracle, _ = case
    long, short = prompt(321, 520, config.vocab), prompt(322, 40, config.vocab)
    rows = oracle_rows(oracle, [long, short])
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
    """300 tokens fed one by one after a prompt of five: the states are carried through every step, windows pass over
    decoded tokens, keys fill page after page."""
    name, folder, config, _, oracle, _ = case
    p = prompt(77, 305, config.vocab)
    rows = oracle_rows(oracle, [p])
    rep = replayer(folder, dtype, 320)
    rep.step([{"id": "d", "tokens": p[:5], "want": []}], [])
    got = {}
    for pos in range(5, len(p)):
        logits = rep.step([{"id": "d", "tokens": [p[pos]], "want": [0]}], [])
        if pos % 7 == 0 or pos >= 300:
            got[(0, pos)] = logits[0]
    check(got, rows, dtype)


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
    """n = 3 at temperature 0: the continuations part after the prompt, each with a copy of the states and the prompt's
    pages shared; all three must be the oracle's greedy continuation. And a pool so small that requests are preempted and
    fed again from their first token."""
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
