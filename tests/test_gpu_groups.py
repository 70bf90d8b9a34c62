"""Several products in one launch: the kernel for few rows against 64 bits, the rule that chooses, and two mixers side by side whose
products are made together against the same mixers one by one."""

from __future__ import annotations

import pytest
import torch

from tests.test_gpu_parts import context
from tinyserve_llm_amd.ops import hip
from tinyserve_llm_amd.parts.base import LayerMemory, PartSpec, make

BF = torch.bfloat16


def group(rows, widths, k, seed=0, skew=0):
    g = torch.Generator().manual_seed(1000 * rows + k + seed)
    xs = list(torch.randn(len(widths), rows, k + skew, generator=g).to(BF).cuda()[:, :, :k])
    return xs, [(torch.randn(n, k, generator=g) * k ** -0.5).to(BF).cuda() for n in widths]


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 15, 16, 17, 63, 64, 65, 127, 128])
@pytest.mark.parametrize("widths, k, skew", [([64, 16, 80, 32], 1024, 0), ([16], 2048, 8), ([48, 128, 2000, 64, 16, 16, 112, 64], 2048, 0)])
def test_products_of_few_rows_in_one_launch(rows, widths, k, skew):
    """32-bit sums of k products: 128 + k / 128 roundings, those within a stretch of 128 and of the stretches' sums, each at most 2^-24 of the sum of the products' sizes."""
    xs, ws = group(rows, widths, k, skew=skew)
    ys = hip.gemm_rows64_group(xs, torch.cat([hip.pack_weight(w) for w in ws]), widths)
    for x, w, y in zip(xs, ws, ys):
        want, sizes = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
        assert y.shape == want.shape and y.is_contiguous() and bool(((y.double() - want).abs() <= (128 + k / 128) * 2.0 ** -24 * sizes).all())


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 8, 16, 32, 48, 64])
@pytest.mark.parametrize("n, k", [(2048, 2048), (3104, 2048), (1024, 1024), (2048, 4096)])
def test_they_are_as_near_to_64_bits_as_one_by_one(rows, n, k):
    """The mean error over n columns and all rows varies by less than a tenth between one order of the sums and another that is as good."""
    from tinyserve_llm_amd.parts.linear import linear, streaming_copy
    xs, ws = group(rows, [n], k)
    want = xs[0].double() @ ws[0].double().T
    apart = linear(xs[0], ws[0], out_dtype=torch.float32, packed=streaming_copy(ws[0]))
    (together,) = hip.gemm_rows64_group(xs, hip.pack_weight(ws[0]), [n])
    assert float((together.double() - want).norm()) <= 1.1 * float((apart.double() - want).norm())


@pytest.mark.gpu
def test_numbers_that_are_none_stay_in_their_rows_and_columns():
    xs, ws = group(20, [64, 32], 1024)
    xs[0][7, 1000], ws[1][5, 3] = float("nan"), float("inf")
    a, b = hip.gemm_rows64_group(xs, torch.cat([hip.pack_weight(w) for w in ws]), [64, 32])
    assert bool(a[7].isnan().all()) and bool(a[:7].isfinite().all()) and bool(a[8:].isfinite().all())
    assert not bool(b[:, 5].isfinite().any()) and bool(b[:, :5].isfinite().all()) and bool(b[:, 6:].isfinite().all())


@pytest.mark.gpu
def test_what_a_group_does_not_take_is_refused_and_gemm_group_leaves_it():
    xs, ws = group(9, [64, 64], 1024)
    packed = torch.cat([hip.pack_weight(w) for w in ws])
    for bad in (lambda: hip.gemm_rows64_group(xs, packed, [64, 48]), lambda: hip.gemm_rows64_group(xs, packed, [128]), lambda: hip.gemm_rows64_group([xs[0], xs[1][:8]], packed, [64, 64]),
                lambda: hip.gemm_rows64_group([x.float() for x in xs], packed, [64, 64]), lambda: hip.gemm_rows64_group([x[:, :512] for x in xs], packed, [64, 64]),
                lambda: hip.gemm_rows64_group([], packed, [])):
        with pytest.raises(hip.KernelError):
            bad()
    assert hip.gemm_group(xs, ws, packed) is not None
    for given in ((xs, ws, None), ([x.float() for x in xs], ws, packed), ([xs[0], xs[1][:8]], ws, packed), (xs, [ws[0], ws[1].t().contiguous().t()], packed),
                  ([x[:0] for x in xs], ws, packed)):
        assert hip.gemm_group(*given) is None


@pytest.mark.gpu
def test_a_recorded_group_is_replayed():
    xs, ws = group(12, [64, 144], 1024)
    packed = torch.cat([hip.pack_weight(w) for w in ws])
    many = [group(130, [2048, 64], 1024, seed=s) for s in range(2)]
    hip.gemm_group(xs, ws, packed), hip.gemm_group(*many[0], None)
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        got, far = hip.gemm_group(xs, ws, packed), hip.gemm_group(*many[0], None)
    for seed in range(3):
        for old, new in zip(xs, group(12, [64, 144], 1024, seed=seed)[0]):
            old.copy_(new)
        for old, new in zip(many[0][0], group(130, [2048, 64], 1024, seed=seed)[0]):
            old.copy_(new)
        graph.replay()
        torch.cuda.synchronize()
        want, wide = hip.gemm_group(xs, ws, packed), hip.gemm_group(*many[0], None)
        assert all(torch.equal(a, b) for a, b in zip(got, want)) and all(torch.equal(a, b) for a, b in zip(far, wide))


def test_the_rule_takes_what_was_measured_faster():
    shift, pair, lasts = (2048,) * 4 + (64,), (3104, 8192), (2048, 2048)
    for rows in (1, 8, 48, 64):
        assert hip.group_plan(rows, shift, 2048, True) == -1 and hip.group_plan(rows, shift, 2048, False) is None
    for widths, rows, taken in ((pair, 4, False), (pair, 5, True), (lasts, 8, False), (lasts, 9, True)):
        assert (hip.group_plan(rows, widths, 2048, True) == -1) == taken
    for widths, rows in ((shift, 65), (shift, 2048), (pair, 1000), (pair, 2048), (lasts, 65), (lasts, 1024)):
        assert hip.group_plan(rows, widths, 2048, True) >= 0
    assert hip.group_plan(1500, pair, 2048, True) is None and hip.group_plan(4000, shift, 2048, True) is None
    assert hip.group_plan(48, (2048,), 2048, True) is None and hip.group_plan(48, (64,) * 9, 2048, True) is None
    assert hip.group_plan(48, (2048, 24), 2048, True) is None and hip.group_plan(48, lasts, 1536, True) is None and hip.group_plan(100, (2048, 20), 2048, True) is None


@pytest.mark.parametrize("widths, k", [((2048, 2048), 5120), ((2048, 2048), 8192), ((1536, 1536), 8192), ((4096,) * 4, 5120), ((4096,) * 4, 6144), ((2048,) * 4 + (64,), 8192)])
def test_products_that_go_in_slices_by_themselves_are_not_grouped(widths, k):
    """Their reductions' shorter chains are nearer to 64 bits than a whole one, and faster."""
    sliced = [rows for rows in range(129, 2049) if any(hip.slices_plan(rows, n, k, "f32") is not None for n in widths)]
    assert len(sliced) > 200 and all(hip.group_plan(rows, widths, k, True) is None for rows in sliced)


@pytest.mark.parametrize("rows, widths, inside, outside", [
    (9, (1024, 1024), 1024, 2048), (9, (2304, 768), 1024, 2048), (9, (64, 64), 1024, 2048), (16, (1024, 1024), 2048, 3072), (9, (2048, 2048), 3072, 4096), (48, (2048, 2048), 4096, 8192), (17, (4096, 4096), 8192, 9216), (1, (1024,) * 3, 2048, 3072),
    (5, (1024,) * 3, 4096, 5120), (64, (2048,) * 4 + (64,), 8192, 9216), (16, (64,) * 3, 4096, 16384), (9, (4096, 64), 4096, 5120), (128, (2048, 2048), 3072, 4096), (200, (2048, 2048), 3072, 4096)])
def test_groups_of_few_columns_are_left_over_long_reductions(rows, widths, inside, outside):
    """A workgroup walks all of k, however few of them there are."""
    assert hip.group_plan(rows, widths, inside, True) is not None and hip.group_plan(rows, widths, outside, True) is None


def test_wide_groups_of_many_rows_promise_more_than_the_estimates_err_by():
    for rows, k in ((1500, 1024), (1500, 2048), (1500, 4096)):
        assert hip.group_plan(rows, (3104, 8192), k, True) is None
    assert hip.group_plan(2048, (6144, 8192), 4096, True) is None and hip.group_plan(900, (3104, 8192), 4096, True) is not None


def test_small_results_go_along_in_chains_or_by_themselves():
    parts = hip.group_parts
    for rows in (130, 600, 1600):
        assert parts(rows, (3072,) + (2048,) * 4 + (64, 32), 2048, True)[1:] == ((5, 6), ())
        assert parts(rows, (2048, 64), 2048, True) == (None, (), ()) and parts(rows, (2048, 64), 1024, True)[1:] == ((), ())
    assert parts(2048, (2048,) * 4 + (64,), 2048, True) == (hip.group_plan(2048, (2048,) * 4, 2048, False), (), (4,))
    for rows in (129, 200, 330, 700, 1229, 2048):
        for widths in ((512, 2048, 1024), (2048,) * 4 + (64,), (32, 2048, 2048)):
            small = tuple(i for i, n in enumerate(widths) if rows * n <= 1 << 17)
            assert parts(rows, widths, 2048, False)[1:] in ((small, ()), ((), small))
    for rows in (65, 80, 128):
        assert parts(rows, (2048,) * 4 + (64,), 2048, True) == parts(rows, (1024,) * 3, 2048, True) == (-1, (), ())
        assert parts(rows, (1024,) * 3, 2048, False) == (None, (), ()) and parts(rows, (1024,) * 3, 4096, True) == (None, (), ())
    assert parts(80, (3104, 8192), 2048, True) == (-1, (), ()) and parts(80, (3104, 8192), 2048, False) == (None, (), ())
    assert parts(96, (3104, 8192), 2048, True) == (hip.group_plan(96, (3104, 8192), 2048, True), (), ())


@pytest.mark.gpu
@pytest.mark.parametrize("tile", range(5))
@pytest.mark.parametrize("rows, widths, k, chained", [(1, (8, 64), 768, (0,)), (130, (72, 264, 32), 832, (0, 2)), (300, (128, 64), 2048, (0, 1)), (257, (2048, 64), 1984, (1,))])
def test_products_in_chains(tile, rows, widths, k, chained):
    """A product cut into four is the four added up, bit for bit, and the others are what they were."""
    xs, ws = group(rows, widths, k)
    plain, got = hip.gemm_whole(xs, ws, tile, torch.float32), hip.gemm_whole(xs, ws, tile, torch.float32, chained)
    ends = [0]
    for i in range(4):
        ends.append(ends[-1] + 64 * (k // 64 // 4 + (i < k // 64 % 4)))
    for i, (x, w) in enumerate(zip(xs, ws)):
        want = plain[i]
        if i in chained:
            parts = [hip.gemm_whole([x[:, a:b].contiguous()], [w[:, a:b].contiguous()], tile, torch.float32)[0] for a, b in zip(ends, ends[1:])]
            want = ((parts[0] + parts[1]) + parts[2]) + parts[3]
        assert torch.equal(got[i], want)
    for bad in (lambda: hip.gemm_whole(xs, ws, tile, BF, chained), lambda: hip.gemm_whole(xs, ws, tile, torch.float32, (len(xs),)),
                lambda: hip.gemm_whole([x[:, :704].contiguous() for x in xs], [w[:, :704].contiguous() for w in ws], tile, torch.float32, chained)):
        with pytest.raises(hip.KernelError):
            bad()


@pytest.mark.gpu
def test_a_group_with_small_results_by_the_module_and_by_the_general_function(monkeypatch):
    import types
    groups = [(300, (2048, 64, 2048, 32)), (2048, (2048, 2048, 64, 2048, 2048))]
    assert [hip.group_parts(rows, widths, 2048, False)[1:] for rows, widths in groups] == [((1, 3), ()), ((), (2,))]
    made = [group(rows, widths, 2048) for rows, widths in groups]
    got = [hip.gemm_group(xs, ws, None) for xs, ws in made]
    monkeypatch.setattr(hip, "_native", lambda: types.SimpleNamespace(gemm_slices=lambda *a: None, gemm_library=lambda *a: None))
    for ys, (xs, ws) in zip(got, made):
        assert all(torch.equal(a, b) for a, b in zip(ys, hip.gemm_group(xs, ws, None)))
    assert torch.equal(got[1][2], hip.linear_bf16(made[1][0][2], made[1][1][2], torch.float32))


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [66, 88, 96, 129, 200, 330, 700])
@pytest.mark.parametrize("widths, k", [((2048, 2048, 64), 2048), ((1536, 1536), 2048), ((1024, 1024, 1024), 3072), ((3104, 8192), 2048), ((512, 2048, 1024), 1536)])
def test_no_product_of_a_group_of_many_rows_is_further_from_64_bits_than_by_itself(rows, widths, k):
    """The mean error over a result's numbers varies by less than a tenth between one order of the sums and another that is as good."""
    xs, ws = group(rows, widths, k)
    copies = torch.cat([hip.pack_weight(w) for w in ws]) if k % 1024 == 0 else None
    for packed in (copies, None):
        ys = hip.gemm_group(xs, ws, packed)
        for x, w, y in zip(xs, ws, ys or ()):
            want = x.double() @ w.double().T
            assert y.shape == want.shape and float((y.double() - want).norm()) <= 1.1 * float((hip.linear_bf16(x, w, torch.float32).double() - want).norm())


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [BF, torch.float32])
@pytest.mark.parametrize("right", ["shifted_decay_recurrence", "retention"])
@pytest.mark.parametrize("lengths", [[1], [1, 1, 1, 1, 1, 1, 1, 1, 1], [40, 1, 7], [70, 3], [300]])
def test_two_mixers_side_by_side_are_the_mixers_one_by_one(dtype, right, lengths, monkeypatch):
    """And leave the same keys, values and states; up to the roundings of 32-bit sums in another order, where the products are made together."""
    width, n = 1024, len(lengths)
    specs = {"shifted_decay_recurrence": dict(hidden_size=width, num_heads=16, head_dim=64, decay_rank=64, norm_eps=1e-6),
             "retention": dict(hidden_size=width, num_heads=8, head_dim=64, value_dim=128, decay=[0.9 + 0.01 * i for i in range(8)], norm_eps=1e-6)}
    left = dict(hidden_size=width, num_heads=16, num_kv_heads=4, head_dim=64, position=None, window=256)
    pair = make("mixer", PartSpec("side_by_side", dict(left=PartSpec("attention_general", left), right=PartSpec(right, specs[right]), left_scale=0.6, right_scale=1.1)))
    g = torch.Generator().manual_seed(len(right))
    pair.bind({name: (torch.randn(ps.shape, generator=g) * (ps.shape[-1] ** -0.5 if len(ps.shape) == 2 else 0.3)).to(torch.float32 if ps.storage == "float32" else dtype).cuda()
               for name, ps in pair.param_specs().items()})
    held = pair.keep_streaming_copies() if dtype == BF else 0
    assert (held > 0) == (dtype == BF)
    if dtype == BF:      # every packed copy of a first or last product is a part of one tensor
        together = pair.first_together.untyped_storage().data_ptr()
        assert all(c is None or c.by16 is None or c.by16.untyped_storage().data_ptr() == together for _, c in pair.left.first_weights() + pair.right.first_weights())
        assert pair.left.o_packed.by16.untyped_storage().data_ptr() == pair.last_together.untyped_storage().data_ptr()
    x = torch.randn(sum(lengths), width, generator=g).to(dtype).cuda()
    tables = [[3 * i + j for j in range(3)] for i in range(n)]
    calls = []
    real = hip.gemm_group
    monkeypatch.setattr(hip, "gemm_group", lambda *a: calls.append(real(*a)) or calls[-1])

    def forward(mixers):
        k = torch.zeros(3 * n, 4, 128, 64, dtype=dtype, device="cuda").permute(0, 2, 1, 3)
        v = torch.zeros(3 * n, 4, 64, 128, dtype=dtype, device="cuda").permute(0, 3, 1, 2)
        state = torch.randn(n, *pair.state_spec().shape, generator=torch.Generator().manual_seed(7)).cuda() * 0.1
        mem, ctx = LayerMemory(k_cache=k, v_cache=v, space=0, store=True, state=state), context(lengths, [0] * n, 128, tables)
        return [mixers(x, ctx, mem), k, v, state]
    got = forward(pair.forward)
    made = [c is not None for c in calls]
    want = forward(lambda *a: hip.scaled_sum(pair.left.forward(*a), 0.6, pair.right.forward(*a), 1.1))
    if dtype == torch.float32:
        assert not any(made) and all(torch.equal(a, b) for a, b in zip(got, want))
        return
    assert any(made) or len(x) <= 8
    for a, b in zip(got, want):
        assert float((a.float() - b.float()).norm()) <= 2.0 ** -7 * float(b.float().norm()) + 1e-6      # (a rounding of bfloat16 rows, and what follows of it)
