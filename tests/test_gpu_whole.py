"""Products of whole tiles (gemm_whole.hip): against 64 bits, several in one launch, and the q|k|v projection through the rotation
into q and the cache against a product and the rotation's kernel."""

from __future__ import annotations

import types

import pytest
import torch

from tinyserve_llm_amd.ops import hip

BF, I32 = torch.bfloat16, torch.int32


def operands(rows, n, k, seed=0, x_skew=0):
    g = torch.Generator().manual_seed(1000 * rows + n + k + seed)
    x = torch.randn(rows, k + x_skew, generator=g).to(BF).cuda()[:, :k]
    return x, (torch.randn(n, k, generator=g) * k ** -0.5).to(BF).cuda()


@pytest.mark.gpu
@pytest.mark.parametrize("tile", range(len(hip.SLICES_TILES)))
@pytest.mark.parametrize("over", [-1, 0, 1])
def test_several_products_of_one_launch(tile, over):
    """32-bit sums of k products: k 2^-24 of the sum of their sizes at most; in bfloat16 those sums rounded. Widths of several tiles, of a
    part of one, and rows of x apart."""
    bm, bn = hip.SLICES_TILES[tile][:2]
    rows, k = 2 * bm + over, 192 + 64 * (over + 1)
    pairs = [operands(rows, n, k, seed=n, x_skew=16) for n in (bn + 8 * over, 8, 2 * bn + 72)]
    xs, ws = [p[0] for p in pairs], [p[1] for p in pairs]
    wide, narrow = hip.gemm_whole(xs, ws, tile, torch.float32), hip.gemm_whole(xs, ws, tile)
    for x, w, y, z in zip(xs, ws, wide, narrow):
        want, sizes = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
        assert y.shape == want.shape and bool(((y.double() - want).abs() <= k * 2.0 ** -24 * sizes).all())
        assert torch.equal(z, y.to(BF)) and torch.equal(hip.gemm_slices(x, w, tile, 1, torch.float32), y)


@pytest.mark.gpu
@pytest.mark.parametrize("tile, rows, n", [(1, 1000, 6144), (1, 1000, 6152), (1, 1200, 8192), (1, 127, 8), (2, 768, 10304), (2, 769, 10304), (2, 1792, 9280), (2, 193, 200),
                                           (3, 1000, 12288), (3, 1000, 12296), (3, 2048, 4160), (3, 257, 184)])
def test_tiles_are_narrow_or_wide_with_the_same_bits(tile, rows, n):
    """Up to and past the last width that 192 columns take no more rounds of the chip for, in one round and in two; a tile's sums are those of tiles of
    128 x 128, whole and in each slice."""
    x, w = operands(rows, n, 448, x_skew=8)
    for out in (torch.float32, BF):
        assert torch.equal(hip.gemm_whole([x], [w], tile, out)[0], hip.gemm_whole([x], [w], 0, out)[0])
    assert torch.equal(hip.gemm_slices(x, w, tile, 2, torch.float32), hip.gemm_slices(x, w, 0, 2, torch.float32))


@pytest.mark.gpu
def test_what_the_whole_tiles_do_not_take_is_refused():
    x, w = operands(130, 64, 256)
    for bad in (lambda: hip.gemm_whole([x] * 9, [w] * 9, 0), lambda: hip.gemm_whole([x, x[:129]], [w, w], 0), lambda: hip.gemm_whole([x], [w[:, :192]], 0),
                lambda: hip.gemm_whole([x], [w], 5), lambda: hip.gemm_whole([x[:, :128]], [w[:, :128].contiguous()], 0), lambda: hip.gemm_whole([x.float()], [w], 0),
                lambda: hip.gemm_whole([x], [w[:60]], 0), lambda: hip.gemm_whole([], [], 0)):
        with pytest.raises(hip.KernelError):
            bad()


def caches(pages, page, heads, dim, transposed=True):
    k = torch.zeros(pages, heads, page, dim, dtype=BF, device="cuda").permute(0, 2, 1, 3)
    v = torch.zeros(pages, heads, dim, page, dtype=BF, device="cuda").permute(0, 3, 1, 2) if transposed else torch.zeros(pages, page, heads, dim, dtype=BF, device="cuda")
    return k, v


def places(rows, how, held):
    """A prompt from the start of a page on; requests that decode ahead of a prompt that goes on in the middle of one; tokens anywhere, some nowhere."""
    if how == "prompt":
        s = torch.arange(rows)
    elif how == "beside":
        s = torch.cat([torch.arange(min(rows, 13)) * 37 + 5, torch.arange(max(rows - 13, 0)) + 523])
    else:
        s = torch.randperm(held, generator=torch.Generator().manual_seed(rows))[:rows]
        s[::5] = -1
    return s.to(I32).cuda()


@pytest.mark.gpu
@pytest.mark.parametrize("tile", range(len(hip.WHOLE_ROPE_TILES)))
@pytest.mark.parametrize("heads, kv, dim", [(6, 2, 64), (3, 1, 128), (2, 1, 256), (5, 3, 64), (2, 0, 64)])
@pytest.mark.parametrize("how, page, transposed", [("prompt", 32, True), ("beside", 32, True), ("anywhere", 40, True), ("beside", 24, False), ("prompt", 20, True)])
def test_a_projection_has_the_bits_of_the_product_and_the_rotation(tile, heads, kv, dim, how, page, transposed):
    n, k = (heads + 2 * kv) * dim, 256
    bm = hip.WHOLE_ROPE_TILES[tile][0]
    g = torch.Generator().manual_seed(dim)
    table = torch.randn(700, dim, generator=g).cuda()
    for rows in (1, bm - 1, bm + 17, 2 * bm):
        x, w = operands(rows, n, k, x_skew=8)
        pos = torch.randint(0, 700, (rows,), generator=g).to(I32).cuda()
        pages = -(-(rows + 700) // page)
        slots = places(rows, how, pages * page) if kv else None
        for cs in (table, None):
            got_kv = caches(pages, page, kv, dim, transposed) if kv else (None, None)
            want_kv = caches(pages, page, kv, dim, transposed) if kv else (None, None)
            q = hip.qkv_rope_store_whole(x, w, tile, cs, pos, slots, *got_kv, heads, kv, dim)
            want = hip.rope_store(hip.gemm_whole([x], [w], 0)[0], cs, pos, slots, *want_kv, heads, kv, dim)
            assert torch.equal(q, want)
            assert not kv or (torch.equal(got_kv[0], want_kv[0]) and torch.equal(got_kv[1], want_kv[1]))
    if kv:      # a layer that reads another's cache: only its queries are made
        assert torch.equal(hip.qkv_rope_store_whole(x, w, tile, table, pos, None, None, None, heads, kv, dim),
                           hip.rope_store(hip.gemm_whole([x], [w], 0)[0], table, pos, None, None, None, heads, kv, dim))


@pytest.mark.gpu
@pytest.mark.parametrize("heads, kv, dim", [(38, 5, 64), (14, 5, 128), (48, 9, 64)])
@pytest.mark.parametrize("rows", [1921, 2048, 2200])
def test_the_second_tile_is_narrow_or_wide_with_the_same_bits(rows, heads, kv, dim):
    """3,072 columns in 256 workgroups of 192 columns (1,921 and 2,048 rows) and in wide ones (2,200 rows); 4,224 columns in wide ones."""
    n, k, page = (heads + 2 * kv) * dim, 256, 32
    assert (-(-rows // 128) * -(-n // 192) <= hip.COMPUTE_UNITS) == (n == 3072 and rows < 2200)
    x, w = operands(rows, n, k)
    pages = -(-(rows + 700) // page)
    table, pos, slots = torch.randn(rows, dim, device="cuda"), torch.arange(rows, dtype=I32, device="cuda"), places(rows, "beside", pages * page)
    got_kv, want_kv = caches(pages, page, kv, dim, True), caches(pages, page, kv, dim, True)
    q = hip.qkv_rope_store_whole(x, w, 1, table, pos, slots, *got_kv, heads, kv, dim)
    want = hip.rope_store(hip.gemm_whole([x], [w], 0)[0], table, pos, slots, *want_kv, heads, kv, dim)
    assert torch.equal(q, want) and torch.equal(got_kv[0], want_kv[0]) and torch.equal(got_kv[1], want_kv[1])


@pytest.mark.gpu
def test_the_module_and_the_general_function_give_the_same_and_refuse_the_same(monkeypatch):
    x, w = operands(300, 4 * 64, 256)
    table, pos, slots = torch.randn(400, 64, device="cuda"), torch.arange(300, dtype=I32, device="cuda"), torch.arange(300, dtype=I32, device="cuda")

    def run(x=x, w=w, tile=0, table=table, pos=pos, slots=slots, dim=64):
        k, v = caches(12, 32, 1, dim)
        try:
            return [hip.qkv_rope_store_whole(x, w, tile, table, pos, slots, k, v, 2, 1, dim), k, v]
        except hip.KernelError as e:
            return str(e)
    forms = [{}, dict(table=None), dict(tile=4), dict(dim=32), dict(x=x[:, :192]), dict(pos=pos[:9]), dict(slots=None), dict(table=table[:, :32].contiguous()), dict(x=x.float()),
             dict(w=w[:, :192])]
    got = [run(**f) for f in forms]
    monkeypatch.setattr(hip, "_native", lambda: types.SimpleNamespace(qkv_rope_store_sliced=lambda *a: None))
    for g, w_ in zip(got, [run(**f) for f in forms]):
        assert g == w_ if isinstance(w_, str) else all(torch.equal(a, b) for a, b in zip(g, w_))
    assert sum(isinstance(g, str) for g in got) == 8


@pytest.mark.gpu
def test_an_attention_layer_takes_it_where_the_rule_says_so(monkeypatch):
    """And has the keys, values and outputs of the way apart, up to the roundings of a product summed in another order."""
    from tinyserve_llm_amd.parts.attention import Attention
    from tinyserve_llm_amd.parts.linear import DeferredNorm

    layer, rows = Attention(2048, 32, 8, 64), 300
    _, layer.qkv = operands(1, 3072, 2048)
    x, _ = operands(rows, 8, 2048)
    nw = torch.rand(2048, generator=torch.Generator().manual_seed(5)).to(BF).cuda()
    table, pos = torch.randn(rows, 64, device="cuda"), torch.arange(rows, dtype=I32, device="cuda")
    taken = []
    real = hip.qkv_rope_store_whole
    monkeypatch.setattr(hip, "qkv_rope_store_whole", lambda *a: taken.append(a[2]) or real(*a))
    monkeypatch.setattr(hip, "paged_attention", lambda q, *a, **k: q)
    layer.o = torch.eye(2048, dtype=BF, device="cuda")

    def forward(given):
        k, v = caches(10, 32, 8, 64)
        mem = types.SimpleNamespace(store=True, space=0, k_cache=k, v_cache=v)
        ctx = types.SimpleNamespace(position_encodings={"rope": types.SimpleNamespace(rotary_table=lambda: table)}, slot_mapping=[pos], positions=pos, num_tokens=rows)
        return layer.forward(given, ctx, mem), k, v
    got = forward(x)
    assert taken == [hip.qkv_rope_whole_plan(rows, 3072, 2048)]
    normed = DeferredNorm(x, None, nw, 1e-5)
    through = forward(normed)
    assert len(taken) == 2 and torch.equal(normed.residual_out, x)
    assert all(torch.equal(a, b) for a, b in zip(through, forward(hip.rmsnorm(x, nw, 1e-5)[0])))
    taken.clear()
    hip.many_rows_products("tiled")
    try:
        want = forward(x)
    finally:
        hip.many_rows_products("library")
    assert not taken
    for a, b in zip(got, want):
        assert float((a.float() - b.float()).norm() / b.float().norm()) < 2.0 ** -8      # half a unit in the last place, and the numbers a pair turns into


def test_the_rule_keeps_to_what_was_measured():
    plan = hip.qkv_rope_whole_plan
    tiles = [t[:2] for t in hip.WHOLE_ROPE_TILES]
    for rows, n, k, tile in ((160, 3072, 2048, (64, 128)), (513, 3072, 2048, (64, 128)), (2048, 3072, 2048, (128, 256)), (1514, 5120, 3072, (128, 256)), (700, 5120, 3072, (128, 128)), (3000, 3072, 2048, (192, 256))):
        assert tiles[plan(rows, n, k)] == tile
    assert plan(128, 3072, 2048) is None and plan(3073, 3072, 2048) is None and plan(170, 5120, 3072) is None
    assert plan(512, 3072, 2080) is None and plan(512, 1536, 128) is None


def test_a_product_that_goes_in_slices_by_itself_is_left_apart():
    sliced = [(rows, n, k) for n in (2048, 3072, 4096) for k in (5376, 6144, 8192) for rows in range(129, 2049, 13) if hip.slices_plan(rows, n, k, "bf16") is not None]
    assert len(sliced) > 500 and all(hip.qkv_rope_whole_plan(*size) is None for size in sliced)


def test_whole_tiles_are_taken_where_they_were_the_faster_way():
    for rows, n, k, ending, tile in ((999, 12352, 2048, "f32", (256, 256)), (2048, 10304, 2048, "f32", (192, 256)), (2048, 2048, 2048, "bf16", (128, 128)), (720, 2048, 2048, "f32", (64, 128))):
        plan, slices = hip.many_rows_plan(rows, n, k, ending)
        assert hip.SLICES_TILES[plan][:2] == tile and slices == 1
    for rows, n, k in ((257, 2048, 2048), (128, 12352, 2048), (3073, 12352, 2048), (999, 16384, 2048), (999, 1024, 2048), (999, 12352, 960), (999, 12356, 2048)):
        assert hip.many_rows_plan(rows, n, k, "f32") is None
    assert hip.many_rows_plan(1024, 2048, 8192, "f32") == hip.slices_plan(1024, 2048, 8192, "f32") != None      # noqa: E711 (a long reduction is cut as before)


def test_wide_products_of_even_columns_are_the_library_s_where_it_was_as_fast():
    for n in (8192, 10240, 12288, 12800):
        for rows in range(129, 3073, 7):
            assert all(hip.whole_plan(rows, n, k, "bf16") is None for k in (1024, 2048, 4096, 5120))
            assert rows >= 960 or all(hip.whole_plan(rows, n, k, "f32") is None for k in (1024, 2048, 4096, 5120))
    for rows, n, k, ending, taken in ((1280, 10304, 2048, "bf16", True), (1150, 12288, 2048, "bf16", False), (1514, 7168, 2048, "bf16", True), (999, 12288, 2048, "f32", False),
                                      (1514, 10240, 2048, "f32", True), (800, 12352, 4096, "f32", False), (640, 12352, 4096, "f32", True)):
        assert (hip.whole_plan(rows, n, k, ending) is not None) == taken


@pytest.mark.gpu
@pytest.mark.parametrize("rows, n, k, out", [(720, 2048, 2048, torch.float32), (999, 12352, 2048, BF)])
def test_linear_takes_them_by_the_module_and_by_the_general_function(rows, n, k, out, monkeypatch):
    x, w = operands(rows, n, k)
    want = hip.gemm_whole([x], [w], hip.whole_plan(rows, n, k, "f32" if out is torch.float32 else "bf16"), out)[0]
    assert torch.equal(hip.linear_bf16(x, w, out), want)
    monkeypatch.setattr(hip, "_native", lambda: types.SimpleNamespace(gemm_slices=lambda *a: None, gemm_library=lambda *a: None))
    assert torch.equal(hip.linear_bf16(x, w, out), want)
