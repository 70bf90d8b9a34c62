"""A step's decoding tokens and prompts attended to in one launch: the bits of the two launches."""

from __future__ import annotations

import ctypes

import pytest
import torch

from tinyserve_llm_amd.ops import hip

BF, I32 = torch.bfloat16, torch.int32
pytestmark = pytest.mark.gpu


REFUSED = 2      # the launchers' answer to operands that they do not take


def one_launch(q, k, v, tables, seq, pos, lead, chunk, dwaves, tiles, tile, waves, window, softcap=0.0, sink=False, sinks=None, slopes=None, gate=None):
    """(the answer of the launcher of both in one, what it made): the module goes to two launches where it refuses."""
    p, i, i64, f = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64, ctypes.c_float
    launch = hip.library().ts_paged_attention_step
    launch.argtypes = [p] * 9 + [i] * 4 + [p] + [i] * 7 + [i64] * 6 + [i, f, i, i, i, f, i, p, p, p, i64, p]
    heads, dim, page = q.shape[1], q.shape[2], k.shape[1]
    splits = -(-tables.shape[1] * page // chunk)
    out = torch.zeros_like(q)
    parts = torch.empty(lead, heads, splits, dim, device="cuda"), torch.empty(lead, heads, splits, 2, device="cuda")
    at = lambda t: None if t is None else t.data_ptr()
    rc = launch(at(out), *map(at, parts), at(q), at(k), at(v), at(tables), at(seq), at(pos), lead, splits, chunk, dwaves, at(tiles), tiles.shape[0], tile, waves, heads,
                k.shape[2], dim, page, *k.stride()[:3], v.stride(0), v.stride(2), v.stride(3), tables.shape[1], dim ** -0.5, window, 0,
                int(bool(softcap or sink or sinks is not None or slopes is not None or gate is not None)), softcap, int(sink), at(sinks), at(slopes), at(gate),
                0 if gate is None else gate.stride(0), torch.cuda.current_stream().cuda_stream)
    return rc, out


@pytest.mark.parametrize("extra", ["plain", "cap", "sinks", "gate", "window", "chunks"])
@pytest.mark.parametrize("heads,kv,dim", [(8, 2, 64), (3, 1, 64), (16, 1, 64), (6, 2, 128), (4, 4, 128)])
@pytest.mark.parametrize("rt,waves,chunk,dwaves,lead,page", [(1, 4, 128, 4, 33, 64), (1, 4, 256, 8, 1, 32), (1, 8, 256, 8, 5, 256), (2, 4, 256, 8, 33, 96),
                                                             (1, 4, 256, 4, 5, 256), (1, 8, 512, 8, 33, 32), (2, 4, 1024, 8, 1, 256)])
def test_one_launch_has_the_bits_of_two(rt, waves, chunk, dwaves, lead, page, heads, kv, dim, extra):
    if dim == 128 and chunk != 32 * dwaves:
        chunk, dwaves = chunk // 2, 4          # (wide heads decode in up to four waves where a wave has several steps)
    g = torch.Generator().manual_seed(lead + heads + chunk)
    prompts = [70, 1, 33]
    lengths = [int(n) for n in torch.randint(1, 700, (lead,), generator=g)]
    lengths[0] = 700
    starts = [n - 1 for n in lengths] + [0, 5, 64]
    ends = lengths + [s + n for s, n in zip(starts[lead:], prompts)]
    per = [-(-n // page) for n in ends]
    pages, width = sum(per) + 1, max(per)
    tables, at, order = torch.zeros(len(ends), width, dtype=I32), 0, torch.randperm(pages, generator=g)
    for i, n in enumerate(per):
        tables[i, :n] = order[at:at + n]
        at += n
    tables = tables.cuda()
    k = torch.randn(pages, kv, page, dim, generator=g).to(BF).cuda().permute(0, 2, 1, 3)
    v = torch.randn(pages, kv, dim, page, generator=g).to(BF).cuda().permute(0, 3, 1, 2)
    total = lead + sum(prompts)
    q = torch.randn(total, heads, dim, generator=g).to(BF).cuda()
    seq = torch.tensor(list(range(lead)) + [lead + i for i, n in enumerate(prompts) for _ in range(n)], dtype=I32).cuda()
    pos = torch.tensor(starts[:lead] + [s + j for s, n in zip(starts[lead:], prompts) for j in range(n)], dtype=I32).cuda()
    cu = list(range(lead + 1))
    for n in prompts:
        cu.append(cu[-1] + n)
    tile = rt * waves * (16 // (heads // kv))
    tiles = torch.tensor(hip.attention_tiles(cu, starts, tile, lead), dtype=I32).view(-1, 2).cuda()
    window = {"window": 100, "chunks": -96}.get(extra, 0)
    more = dict(softcap=30.0 if extra == "cap" else 0.0, sink=False, sinks=torch.randn(heads, generator=g).cuda() if extra == "sinks" else None, slopes=None,
                gate=torch.randn(total, heads * dim, generator=g).cuda() if extra == "gate" else None)
    one = hip._native().attention_step(q, k, v, tables, seq, pos, tiles, dim ** -0.5, window, *more.values(), 1, lead, chunk, dwaves, tile, waves, 1, 0, lead)
    # in two launches go: wide heads of the general kind, chunks for fewer waves than a tile's, and sums that a tile's LDS does not hold
    rc, alone = one_launch(q, k, v, tables, seq, pos, lead, chunk, dwaves, tiles, tile, waves, window, **more)
    assert rc == (REFUSED if (dim == 128 and extra in ("cap", "sinks", "gate")) or dwaves < waves or (heads == 16 and dwaves == 8) else 0)
    assert rc or torch.equal(alone, one)
    two = torch.zeros_like(q)
    hip.paged_attention_prefill(q, k, v, tables, seq, pos, tiles, dim ** -0.5, window, tile, two, waves=waves, first_token=lead, **more)
    if more["gate"] is not None:
        more["gate"] = more["gate"][:lead]
    hip.paged_attention_decode(q[:lead], k, v, tables, seq[:lead], pos[:lead], dim ** -0.5, window, chunk, dwaves, two[:lead], **more)
    assert torch.equal(one, two)


@pytest.mark.parametrize("shared", ["own", "pairs", "all"])
@pytest.mark.parametrize("extra", ["plain", "cap", "window"])
@pytest.mark.parametrize("dim,kv,group,rt,waves,chunk,dwaves", [(64, 8, 4, 1, 8, 256, 8), (64, 8, 4, 2, 4, 256, 8), (64, 8, 1, 1, 4, 128, 4), (64, 8, 4, 1, 8, 512, 8), (64, 8, 2, 1, 4, 512, 4),
                                                                (128, 8, 3, 1, 8, 256, 8), (128, 8, 3, 2, 4, 256, 4)])
def test_one_launch_of_walks_past_the_caches(dim, kv, group, rt, waves, chunk, dwaves, extra, shared):
    """More keys and values than DEC_ONCE_BYTES of the decode kernel (48 MB): values past the caches, and with one step a wave of heads of 64 keys too, but not of
    pages that the next token's request has as well (the token before, of the last). Requests with pages of their own, pairs that share all but the last, and one table for all."""
    if extra == "cap" and dim == 128:
        pytest.skip("wide heads of the general kind go in two launches")
    g, made, lead, page, width = torch.Generator().manual_seed(chunk + group), torch.Generator(device="cuda").manual_seed(chunk + group), 33, 256, 6
    assert lead * kv * dim * 4 * (1024 if extra == "window" else width * page) >= 48 << 20
    prompts, heads = [70, 33], kv * group
    lengths = [int(n) for n in torch.randint(1, width * page + 1, (lead,), generator=g)]
    lengths[0], lengths[-1], lengths[-2] = width * page, width * page - 1, 1
    starts = [n - 1 for n in lengths] + [0, 700]
    tables = torch.randperm((lead + 2) * width, generator=g).to(I32).view(lead + 2, width)
    if shared == "pairs":
        tables[1:lead:2, :-1] = tables[0:lead - 1:2, :-1]
    elif shared == "all":
        tables[1:lead] = tables[0]
    tables = tables.cuda()
    k = torch.randn((lead + 2) * width, kv, page, dim, generator=made, device="cuda").to(BF).permute(0, 2, 1, 3)
    v = torch.randn((lead + 2) * width, kv, dim, page, generator=made, device="cuda").to(BF).permute(0, 3, 1, 2)
    q = torch.randn(lead + sum(prompts), heads, dim, generator=g).to(BF).cuda()
    seq = torch.tensor(list(range(lead)) + [lead + i for i, n in enumerate(prompts) for _ in range(n)], dtype=I32).cuda()
    pos = torch.tensor(starts[:lead] + [s + j for s, n in zip(starts[lead:], prompts) for j in range(n)], dtype=I32).cuda()
    cu = list(range(lead + 1)) + [lead + 70, lead + 103]
    tile = rt * waves * (16 // group)
    tiles = torch.tensor(hip.attention_tiles(cu, starts, tile, lead), dtype=I32).view(-1, 2).cuda()
    window, softcap = 1024 if extra == "window" else 0, 30.0 if extra == "cap" else 0.0
    rc, one = one_launch(q, k, v, tables, seq, pos, lead, chunk, dwaves, tiles, tile, waves, window, softcap)
    assert rc == 0
    assert torch.equal(one, hip._native().attention_step(q, k, v, tables, seq, pos, tiles, dim ** -0.5, window, softcap, False, None, None, None, 1, lead, chunk, dwaves, tile,
                                                         waves, 1, 0, lead))
    two = torch.zeros_like(q)
    hip.paged_attention_prefill(q, k, v, tables, seq, pos, tiles, dim ** -0.5, window, tile, two, waves=waves, first_token=lead, softcap=softcap)
    hip.paged_attention_decode(q[:lead], k, v, tables, seq[:lead], pos[:lead], dim ** -0.5, window, chunk, dwaves, two[:lead], softcap=softcap)
    assert torch.equal(one, two)


@pytest.mark.parametrize("splits", [1, 2, 7, 8, 9, 16, 17, 70])
@pytest.mark.parametrize("heads,dim", [(3, 64), (2, 96), (5, 128), (2, 32)])
@pytest.mark.parametrize("window", [0, 40, -64])
def test_chunks_are_combined_whatever_the_ones_without_a_visible_key_hold(splits, heads, dim, window):
    """Against 64 bits: a bfloat16 rounding (2^-8 with room for the 32-bit sums' own error, which is splits + 3 roundings of 2^-22 of the terms' sizes)."""
    g, chunk = torch.Generator().manual_seed(100 * splits + dim), 32
    positions = [0, 31, 32, splits * chunk // 2, splits * chunk - 1, splits * chunk - 33]
    positions = torch.tensor([min(max(p, 0), splits * chunk - 1) for p in positions], dtype=I32)
    tokens = len(positions)
    o, ml = torch.randn(tokens, heads, splits, dim, generator=g), torch.rand(tokens, heads, splits, 2, generator=g) * 3 + 0.1
    want, size = torch.empty(tokens, heads, dim, dtype=torch.float64), torch.empty(tokens, heads, dim, dtype=torch.float64)
    for t, p in enumerate(positions.tolist()):
        first = max(p - window + 1, 0) if window > 0 else p // -window * -window if window else 0
        seen = slice(first // chunk, p // chunk + 1)
        w = torch.exp2(ml[t, :, seen, 0].double())
        total = (ml[t, :, seen, 1].double() * w).sum(1)[:, None]
        want[t], size[t] = (o[t, :, seen].double() * w[..., None]).sum(1) / total, (o[t, :, seen].double().abs() * w[..., None]).sum(1) / total
        hidden = [s for s in range(splits) if not seen.start <= s < seen.stop]
        o[t, :, hidden], ml[t, :, hidden] = float("nan"), float("nan")
    got = hip.SplitAttention(o.cuda(), ml.cuda(), positions.cuda(), chunk, window).combined().view(tokens, heads, dim).cpu().double()
    assert bool(((got - want).abs() <= 2.0 ** -8 * want.abs() + (splits + 3) * 2.0 ** -22 * size).all())


@pytest.mark.parametrize("splits", [1, 2, 4, 5, 8, 9, 12, 16])
@pytest.mark.parametrize("heads,dim", [(3, 64), (5, 128), (2, 256), (2, 32)])
@pytest.mark.parametrize("window", [0, 40, 200, -64])
def test_few_chunks_have_the_bits_of_the_kernel_for_many(splits, heads, dim, window):
    """The same chunks with more behind them that no token sees go to the kernel that takes any number of them."""
    g, chunk = torch.Generator(device="cuda").manual_seed(splits + dim), 32
    positions = torch.arange(0, splits * chunk, 13, dtype=I32, device="cuda")
    tokens = len(positions)
    o, ml = torch.randn(tokens, heads, splits, dim, generator=g, device="cuda"), torch.rand(tokens, heads, splits, 2, generator=g, device="cuda") * 9 + 0.1
    beyond = lambda t: torch.cat([t, t.new_full((tokens, heads, 17 - splits, t.shape[3]), float("nan"))], 2)
    few, many = (hip.SplitAttention(a, b, positions, chunk, window).combined() for a, b in ((o, ml), (beyond(o), beyond(ml))))
    assert torch.equal(few, many)
