"""The launches that the library's own module makes (calls.cpp) against the functions of ops/hip.py that they stand in for:
the same bits for every form that both take, and the same refusals."""

from __future__ import annotations

import types

import pytest
import torch

from tinyserve_llm_amd.ops import hip

BF, F32, I32 = torch.bfloat16, torch.float32, torch.int32


class NoCalls:
    """The module as it answers operands that it does not take."""

    def __getattr__(self, name):
        return lambda *args: None


class Recorded:
    """The module with a list of its answers: (function, whether it made the call)."""

    def __init__(self, module):
        self.module, self.answers = module, []

    def __getattr__(self, name):
        def call(*args):
            result = getattr(self.module, name)(*args)
            self.answers.append((name, result is not None))
            return result
        return call


# forms that are not plain: refused by everyone, or served by the functions of ops/hip.py alone (picked rows, two norms, empty
# products, rows that no 16-byte piece fits, head sizes of other kernels, steps that only decode)
NOT_PLAIN = {"rmsnorm-strided", "rmsnorm-weight", "rmsnorm-residual", "rmsnorm-picked", "linear-odd-k", "linear-odd-stride", "linear-shapes", "linear-types", "linear-out-type",
             "linear-transposed", "glu-0-64-64-relu", "glu-k", "glu-form", "rows64-rows", "rows64-unit-scaled", "sliced-slices", "sliced-weight", "rope-row", "update-two",
             "update-shapes", "capped-odd", "heads-norm-gate", "attention-(60,)-48-{}", "attention-(1, 1)-64-{}"}


def plain(name):
    return name not in NOT_PLAIN and not (name.startswith("post") and name.endswith("None")) and not (name.startswith("slices") and name.endswith("float32-True"))


def test_operands_that_are_not_on_a_gpu_are_left_to_the_general_functions():
    x, w = torch.zeros(4, 64, dtype=BF), torch.zeros(64, dtype=BF)
    native = hip._native()
    assert native.rmsnorm(x, w, 1e-5, None, True) is None
    assert native.gemm_library(x, torch.zeros(8, 64, dtype=BF), False) is None
    assert native.rmsnorm(x, w, 1e-5, None) is None and native.rmsnorm("x", w, 1e-5, None, True) is None and native.rmsnorm() is None
    assert native.capped_glu(x, "limit", 1.0, 0.0, 1, 0) is None and native.capped_glu(x, 1.0, 1.0, 0.0, 1 << 40, 0) is None
    with pytest.raises(hip.KernelError, match="GPU"):
        hip.rmsnorm(x, w, 1e-5)


def rows(n, width, dtype=BF, skew=0, seed=0):
    g = torch.Generator(device="cuda").manual_seed(1000 * n + width + seed)
    return torch.randn(n, width + skew, generator=g, device="cuda").to(dtype)[:, :width]


def vec(n, dtype=BF, seed=3):
    return rows(1, n, dtype, seed=seed)[0].contiguous()


def caches(pages, page, heads, dim, vdim=None, dtype=BF):
    """Key pages as they are, value pages transposed, as the engine's pools lay them out."""
    k = torch.zeros(pages, page, heads, dim, dtype=dtype, device="cuda")
    v = torch.zeros(pages, heads, vdim or dim, page, dtype=dtype, device="cuda").permute(0, 3, 1, 2)
    return k, v


def ints(*values):
    return torch.tensor(values, dtype=I32, device="cuda")


def forms():
    """(name, function, arguments made anew for each side: they may be written to)."""
    out = []

    def add(name, fn, make):
        out.append(pytest.param(fn, make, plain(name), id=name))
    for n, width, dtype, wdtype in ((1, 64, BF, BF), (37, 1028, BF, BF), (5, 96, F32, F32), (9, 256, BF, F32), (0, 64, BF, BF)):
        for res in (False, True):
            for want in (True, False):
                add(f"rmsnorm-{n}-{width}-{dtype}-{wdtype}-{res}-{want}", hip.rmsnorm, lambda n=n, width=width, dtype=dtype, wdtype=wdtype, res=res, want=want:
                    ((rows(n, width, dtype), vec(width, wdtype), 1e-5, rows(n, width, dtype, seed=7) if res else None), dict(want_residual=want)))
    add("rmsnorm-strided", hip.rmsnorm, lambda: ((rows(4, 64, skew=8), vec(64), 1e-5), {}))
    add("rmsnorm-weight", hip.rmsnorm, lambda: ((rows(4, 64), vec(60), 1e-5), {}))
    add("rmsnorm-residual", hip.rmsnorm, lambda: ((rows(4, 64), vec(64), 1e-5, rows(4, 64, F32)), {}))
    add("rmsnorm-picked", hip.rmsnorm, lambda: ((rows(4, 64), vec(64), 1e-5), dict(rows=ints(3, 1))))
    for m, n, k, skew in ((1, 64, 64, 0), (130, 192, 96, 8), (77, 40, 200, 0), (300, 1000, 512, 16)):
        for out_dtype in (BF, F32):
            add(f"linear-{m}-{n}-{k}-{skew}-{out_dtype}", hip.linear_bf16, lambda m=m, n=n, k=k, skew=skew, out_dtype=out_dtype: ((rows(m, k, skew=skew), rows(n, k), out_dtype), {}))
            add(f"library-{m}-{n}-{k}-{skew}-{out_dtype}", hip.gemm_library, lambda m=m, n=n, k=k, skew=skew, out_dtype=out_dtype: ((rows(m, k, skew=skew), rows(n, k), out_dtype), {}))
    for m, n, k, skew in ((130, 1024, 2048, 0), (200, 2048, 4096, 16), (40, 72, 384, 8)):
        for out_dtype, norm in ((BF, None), (F32, None), (BF, True), (BF, False), (F32, True)):
            add(f"slices-{m}-{n}-{k}-{skew}-{out_dtype}-{norm}", hip.gemm_slices, lambda m=m, n=n, k=k, skew=skew, out_dtype=out_dtype, norm=norm: (
                (rows(m, k, skew=skew), rows(n, k), 4, 2, out_dtype, None if norm is None else (rows(m, n) if norm else None, vec(n), 1e-5)), {}))
        add(f"linear-deep-{m}-{n}-{k}", hip.linear_bf16, lambda m=m, n=n, k=k, skew=skew: ((rows(m, k, skew=skew), rows(n, k), F32), {}))
    add("linear-odd-k", hip.linear_bf16, lambda: ((rows(50, 100), rows(40, 100)), {}))
    add("linear-odd-stride", hip.linear_bf16, lambda: ((rows(50, 64, skew=3), rows(40, 64)), {}))
    add("linear-shapes", hip.linear_bf16, lambda: ((rows(50, 64), rows(40, 72)), {}))
    add("linear-types", hip.linear_bf16, lambda: ((rows(50, 64, F32), rows(40, 64)), {}))
    add("linear-out-type", hip.linear_bf16, lambda: ((rows(50, 64), rows(40, 64), torch.float16), {}))
    add("linear-transposed", hip.linear_bf16, lambda: ((rows(64, 50).t(), rows(40, 64)), {}))
    for m, f, k, form in ((1, 64, 64, "silu_rounded"), (200, 72, 192, "sigmoid"), (33, 512, 64, "relu"), (0, 64, 64, "relu"), (70, 64, 64, "gelu_tanh")):
        add(f"glu-{m}-{f}-{k}-{form}", hip.gemm_glu, lambda m=m, f=f, k=k, form=form: ((rows(m, k, skew=8), rows(2 * f, k), form, 5.0, 1.5, 0.5), {}))
    add("glu-k", hip.gemm_glu, lambda: ((rows(9, 72), rows(64, 72), "relu"), {}))
    add("glu-form", hip.gemm_glu, lambda: ((rows(9, 64), rows(64, 64), "tanh"), {}))
    for m in (1, 4, 5, 64, 65, 128):
        add(f"rows64-{m}", hip.gemm_rows64, lambda m=m: ((rows(m, 1024, skew=8), hip.pack_weight(rows(256, 1024)), F32), {}))
        add(f"rows64-glu-{m}", hip.gemm_rows64, lambda m=m: ((rows(m, 1024), hip.pack_weight(rows(256, 1024))), dict(glu=True, squares=rows(m, 3, F32).abs(), eps=1e-5)))
        add(f"rows64-unit-{m}", hip.gemm_rows64, lambda m=m: ((rows(m, 1024), hip.pack_weight(rows(256, 1024))), dict(glu=True, unit=("relu", 2.0, 1.0, 0.25))))
        add(f"sliced-{m}", hip.gemm_rows64_sliced, lambda m=m: ((rows(m, 1024, skew=8), hip.pack_weight(rows(192, 1024)), 2), {}))
        add(f"sliced-norm-{m}", hip.gemm_rows64_sliced, lambda m=m: ((rows(m, 1024), hip.pack_weight(rows(192, 1024)), 2), dict(next_norm=(rows(m, 192), vec(192)))))
        add(f"sliced-norm-alone-{m}", hip.gemm_rows64_sliced, lambda m=m: ((rows(m, 1024), hip.pack_weight(rows(192, 1024)), 1), dict(next_norm=(None, vec(192)))))
    add("rows64-rows", hip.gemm_rows64, lambda: ((rows(129, 1024), hip.pack_weight(rows(256, 1024))), {}))
    add("rows64-unit-scaled", hip.gemm_rows64, lambda: ((rows(4, 1024), hip.pack_weight(rows(256, 1024))), dict(glu=True, squares=rows(4, 1, F32).abs(), unit=("relu", 2.0, 1.0, 0.25))))
    add("sliced-slices", hip.gemm_rows64_sliced, lambda: ((rows(9, 1024), hip.pack_weight(rows(192, 1024)), 3), {}))
    add("sliced-weight", hip.gemm_rows64_sliced, lambda: ((rows(9, 1024), hip.pack_weight(rows(192, 1024)), 2), dict(next_norm=(None, vec(64)))))
    for t, heads, kv, dim, rot, dtype in ((1, 4, 2, 32, 32, BF), (70, 6, 2, 64, 64, BF), (33, 2, 2, 16, 8, F32), (9, 4, 1, 48, None, BF)):
        def stored(t=t, heads=heads, kv=kv, dim=dim, rot=rot, dtype=dtype, slots=True):
            table = None if rot is None else rows(256, rot, F32).contiguous()
            k, v = caches(4, 32, kv, dim, dtype=dtype) if slots else (None, None)
            where = torch.arange(t, dtype=I32, device="cuda") - 1 if slots else None
            return ((rows(t, (heads + 2 * kv) * dim, dtype), table, torch.arange(t, dtype=I32, device="cuda"), where, k, v, heads, kv, dim), {})
        add(f"rope-{t}-{dim}-{rot}-{dtype}", hip.rope_store, stored)
        add(f"rope-q-{t}-{dim}-{rot}-{dtype}", hip.rope_store, lambda stored=stored: stored(slots=False))
    add("rope-row", hip.rope_store, lambda: ((rows(3, 100), None, ints(0, 1, 2), None, None, None, 1, 1, 32), {}))
    for m, slices, sq in ((1, 1, False), (40, 2, True), (128, 2, False)):
        def sliced_rope(m=m, slices=slices, sq=sq, hd=64):
            k, v = caches(8, 32, 2, hd)
            return ((rows(m, 1024, skew=8), hip.pack_weight_rope(rows(8 * hd, 1024), hd), slices, rows(256, hd, F32).contiguous(), torch.arange(m, dtype=I32, device="cuda"),
                     torch.arange(m, dtype=I32, device="cuda"), k, v, 4, 2, hd), dict(eps=1e-5, squares=rows(m, 2, F32).abs() if sq else None))
        add(f"sliced-rope-{m}-{slices}-{sq}", hip.qkv_rope_store_sliced, sliced_rope)
    for t, hd, vd, rot, norm, inner, dtype in ((1, 64, 64, 32, None, False, BF), (50, 48, 32, 48, 1e-6, True, BF), (7, 64, 64, 0, 1e-6, False, F32)):
        def finished(t=t, hd=hd, vd=vd, rot=rot, norm=norm, inner=inner, dtype=dtype):
            k, v = caches(4, 32, 2, hd, vd, dtype=dtype)
            freqs = torch.rand(rot // 2, dtype=torch.float64, device="cuda") * 0 + 0.1 if rot else None
            return ((rows(t, 6 * hd + 2 * vd + 8, F32), freqs, torch.arange(t, dtype=I32, device="cuda"), torch.arange(t, dtype=I32, device="cuda"), k, v, 4, 2, hd, vd, dtype),
                    dict(interleaved=inner, qk_norm_eps=norm, v_norm_eps=norm, amplitude=1.25))
        add(f"finish-{t}-{hd}-{vd}-{rot}", hip.qkv_finish, finished)
    for n, width in ((1, 64), (45, 1028), (0, 64)):
        for scaled in (False, True):
            for out_dtype in (BF, F32, None):
                add(f"post-{n}-{width}-{scaled}-{out_dtype}", hip.stream_post_norm, lambda n=n, width=width, scaled=scaled, out_dtype=out_dtype:
                    ((rows(n, width, F32), rows(n, width, F32, seed=5), vec(width, F32), vec(width, F32, 4) if scaled else None, 1e-6, None if scaled else vec(width, F32, 6), 1e-5 if out_dtype else 0.0, out_dtype), {})
                    if out_dtype or scaled else ((rows(n, width, F32), rows(n, width, F32, seed=5), vec(width, F32), None, 1e-6), {}))
        for a, b in ((BF, None), (F32, BF), (None, None)):
            add(f"update-{n}-{width}-{a}-{b}", hip.stream_update_norm, lambda n=n, width=width, a=a, b=b:
                ((rows(n, width, F32), None if a is None else rows(n, width, a, seed=5), None if b is None else rows(n, width, b, seed=6)), dict(mult=0.5, weights=(vec(width), None), eps=1e-5, out_dtype=BF)))
    add("update-two", hip.stream_update_norm, lambda: ((rows(3, 64, F32), rows(3, 64)), dict(weights=(vec(64), vec(64, seed=8)), eps=1e-5)))
    add("update-shapes", hip.stream_update_norm, lambda: ((rows(3, 64, F32), rows(3, 60)), dict(weights=(vec(64), None))))
    for n, width, dtype in ((1, 8, F32), (33, 1030, F32), (9, 64, BF)):
        add(f"capped-{n}-{width}-{dtype}", hip.capped_glu, lambda n=n, width=width, dtype=dtype: ((rows(n, width, dtype, skew=4), 3.0, 1.7, 0.5, BF, "gelu_tanh"), {}))
    add("capped-odd", hip.capped_glu, lambda: ((rows(4, 7, F32), 3.0, 1.7, 0.5, BF), {}))
    for t, heads, vdim, shared, silu in ((1, 4, 32, True, False), (21, 3, 40, False, True)):
        add(f"heads-norm-{t}-{vdim}", hip.mlstm_finish, lambda t=t, heads=heads, vdim=vdim, shared=shared, silu=silu:
            ((rows(t, heads * vdim, F32), vec(vdim if shared else heads * vdim, F32), rows(t, heads * vdim, F32, skew=4), heads, vdim, 1e-6, BF), dict(silu_gate=silu)))
    add("heads-norm-gate", hip.mlstm_finish, lambda: ((rows(3, 64, F32), None, rows(3, 60, F32), 2, 32, 1e-6, BF), {}))
    for lens, before, dim, opts in (((40,), (0,), 64, {}), ((1, 1, 33, 70), (300, 9, 0, 40), 64, {}), ((1, 50), (700, 0), 128, dict(softcap=20.0)), ((90, 17), (3, 0), 32, dict(window=24)),
                                    ((1, 64), (500, 0), 64, dict(gate=True, sinks=True)), ((1, 64), (500, 0), 64, dict(gate="heads", slopes=True, window=100)), ((60,), (0,), 48, {}), ((1, 1), (40, 90), 64, {})):
        add(f"attention-{lens}-{dim}-{opts}", step_attention, lambda lens=lens, before=before, dim=dim, opts=opts: ((lens, before, dim, opts), {}))
    return out


def step_attention(lens, before, dim, opts, heads=8, kv=2, page=32):
    """A step of requests that feed `lens` tokens behind `before` cached ones, twice (the second call finds the step's plan)."""
    total = sum(lens)
    width = max(-(-(a + b) // page) for a, b in zip(lens, before))
    tables = torch.arange(len(lens) * width, dtype=I32, device="cuda").view(len(lens), width)
    k, v = caches(len(lens) * width, page, kv, dim)
    g = torch.Generator(device="cuda").manual_seed(5)
    k.copy_(torch.randn(k.shape, generator=g, device="cuda"))
    v.copy_(torch.randn(v.shape, generator=g, device="cuda"))
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    ctx = types.SimpleNamespace(block_tables=[tables], page_size=page, scratch={}, max_query_len=max(lens), host_cu_seqlens=cu, host_starts=list(before),
                                host_context_lens=[a + b for a, b in zip(lens, before)],
                                seq_of_token=ints(*[s for s, n in enumerate(lens) for _ in range(n)]), positions=ints(*[b + j for n, b in zip(lens, before) for j in range(n)]))
    opts = dict(opts)
    if "gate" in opts:
        opts["gate"] = rows(total, heads if opts["gate"] == "heads" else heads * dim, F32, skew=4)
    for name in ("sinks", "slopes"):
        if name in opts:
            opts[name] = vec(heads, F32).abs()
    q = rows(total, heads * dim).contiguous().view(total, heads, dim)
    return [hip.paged_attention(q, k, v, ctx, 0, dim ** -0.5, **opts) for _ in range(2)]


def tensors(value):
    if isinstance(value, torch.Tensor):
        return [value]
    if isinstance(value, hip.PreparedNorm):
        return [value.summed, value.operand, value.squares]
    if isinstance(value, (list, tuple)):
        return [t for v in value for t in tensors(v)]
    return []


def run(fn, make):
    args, kwargs = make()
    try:
        result = fn(*args, **kwargs)
    except Exception as e:       # (a refusal, to be compared)
        return type(e), str(e)
    kept = [a for a in args if isinstance(a, torch.Tensor)]
    return [(t.dtype, t.shape, t.stride(), t.clone()) for t in tensors(result) + kept]


@pytest.mark.gpu
@pytest.mark.parametrize("fn, make, served", forms() if torch.cuda.is_available() else [pytest.param(None, None, None)])
def test_a_call_gives_the_bits_of_the_general_function(fn, make, served, monkeypatch):
    """And a plain form is served by the module: an attention step twice, in the layer that makes its plan and in the one that finds it."""
    calls = Recorded(hip._native())
    monkeypatch.setattr(hip, "_native", lambda: calls)
    got = run(fn, make)
    made = [name for name, done in calls.answers if done]
    assert len(made) == served * (2 if fn is step_attention else 1)
    if served and fn not in (step_attention, hip.linear_bf16):
        assert made == [fn.__name__]
    monkeypatch.setattr(hip, "_native", NoCalls)
    want = run(fn, make)
    if isinstance(want, tuple):
        assert got == want
        return
    assert not isinstance(got, tuple), got
    assert len(got) == len(want)
    for (gd, gs, gt, g), (wd, ws, wt, w) in zip(got, want):
        assert (gd, gs, gt) == (wd, ws, wt)
        assert torch.equal(g.contiguous().view(torch.uint8), w.contiguous().view(torch.uint8))


@pytest.mark.gpu
def test_calls_go_to_the_current_stream_and_can_be_recorded():
    """On a stream of its own and replayed from a graph, on values that came after the recording."""
    x, w = rows(40, 512), vec(512)
    want = hip.rmsnorm(rows(40, 512, seed=9), w, 1e-5)[0]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        hip.rmsnorm(x, w, 1e-5)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = hip.rmsnorm(x, w, 1e-5)[0]
    x.copy_(rows(40, 512, seed=9))
    for _ in range(3):
        got.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("place", [0, 1])
def test_a_projection_into_a_norm_has_one_route(place, monkeypatch):
    """`linear` with a request asks `hip.linear_into_norm` and nothing beside it: what that leaves (here a weight that begins between two 16-byte pieces, and
    nothing is launched) is the general way's."""
    from tinyserve_llm_amd.parts.linear import DeferredNorm, NormRequest, linear, streaming_copy
    whole = torch.zeros(2048 * 8192 + 8, dtype=torch.bfloat16, device="cuda")
    weight = whole[place:place + 2048 * 8192].view(2048, 8192)
    packed = streaming_copy(whole[:2048 * 8192].view(2048, 8192))
    x, then = torch.zeros(48, 8192, dtype=torch.bfloat16, device="cuda"), NormRequest(torch.ones(2048, dtype=torch.bfloat16, device="cuda"), 1e-5, None)
    asked, made = [], torch.zeros(48, 2048, dtype=torch.bfloat16, device="cuda")
    prepared = hip.PreparedNorm(made, made, torch.ones(48, 1, device="cuda"))
    for name, answer in (("gemm_rows64_sliced", prepared), ("linear_through_norm", None), ("linear_bf16", made)):
        monkeypatch.setattr(hip, name, lambda *args, _name=name, _answer=answer, **options: asked.append(_name) or _answer)
    assert isinstance(linear(x, weight, packed=packed, then=then), DeferredNorm)
    assert asked == (["linear_through_norm", "linear_bf16"] if place else ["gemm_rows64_sliced"])
