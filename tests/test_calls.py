"""The library's own module (calls.cpp) over launchers that only answer: what it does with each answer, on tensors in host memory."""

from __future__ import annotations

import ctypes
import importlib.machinery
import importlib.util
import os
import re
import subprocess

import pytest
import torch

from tinyserve_llm_amd.csrc import build
from tinyserve_llm_amd.ops import hip

BF, F32, I32 = torch.bfloat16, torch.float32, torch.int32
OK, BAD_DTYPE, BAD_SHAPE, LAUNCH_FAILED, TOO_LARGE = range(5)

STUB = """
#include <map>
#include <string>
namespace c10::hip { struct NoStream { hipStream_t stream() const { return nullptr; } }; inline NoStream no_stream() { return {}; } }
#define is_cuda is_cpu
#define getCurrentHIPStream no_stream
static std::map<std::string, int> answers;
static std::string called;
static int locked = 0;
static int answer(const char* name) { locked += PyGILState_Check(); called += std::string(name) + " "; return answers[name]; }
extern "C" int stub_locked() { const int n = locked; locked = 0; return n; }
extern "C" void stub_answer(const char* name, int rc) { answers[name] = rc; }
extern "C" const char* stub_called() { static std::string last; last = called; called.clear(); return last.c_str(); }
"""


@pytest.fixture(scope="session")
def stub(tmp_path_factory):
    """(the module, answer(launcher, rc), called() -> the launchers called since it was last asked), none of them with Python's lock held."""
    folder = tmp_path_factory.mktemp("calls")
    with open(os.path.join(build.HERE, "calls.cpp")) as f:
        source = f.read()
    with open(os.path.join(build.HERE, "entry_points.h")) as f:
        points = re.findall(r"^int (ts_\w+)(\([^;]*\));", f.read(), re.M)
    headers = re.findall(r'^#include .*$', source, re.M)
    launchers = [f'extern "C" int {name}{parameters} {{ return answer("{name}"); }}' for name, parameters in points]
    code, lib = folder / "stub.cpp", folder / "stub.so"
    code.write_text("\n".join([*headers, STUB, *launchers, f'#include "{build.HERE}/calls.cpp"\n']))
    links = [flag for flag in build.LINK if flag != "-lhipblaslt"]
    subprocess.run([build._hipcc(), *build._compile_flags("calls.cpp"), f"-I{build.HERE}", "-shared", "-Wl,-Bsymbolic", str(code), "-x", "none",
                    f"-L{build._torch_folder()}/lib", *links, "-o", str(lib)], check=True)
    loader = importlib.machinery.ExtensionFileLoader("tinyserve_hip_calls", str(lib))
    module = importlib.util.module_from_spec(importlib.util.spec_from_loader(loader.name, loader))
    loader.exec_module(module)
    c = ctypes.CDLL(str(lib))
    c.stub_called.restype = ctypes.c_char_p
    def called():
        assert c.stub_locked() == 0
        return c.stub_called().decode().split()
    return module, lambda name, rc: c.stub_answer(name.encode(), rc), called


def ints(*values):
    return torch.tensor(values, dtype=I32)


def caches(pages=4, page=32, heads=2, dim=64):
    return torch.zeros(pages, page, heads, dim, dtype=BF), torch.zeros(pages, heads, dim, page, dtype=BF).permute(0, 3, 1, 2)


def bf(*shape):
    return torch.zeros(*shape, dtype=BF)


def step(lead, softcap=0.0):
    """`attention_step` of `lead` decoding requests beside a prompt of 40 tokens; a few keys a workgroup of the decoding part."""
    T = lead + 40
    k, v = caches()
    return (bf(T, 4, 64), k, v, torch.zeros(lead + 1, 2, dtype=I32), torch.zeros(T, dtype=I32), torch.zeros(T, dtype=I32), torch.zeros(5, 2, dtype=I32), 0.125, 0,
            softcap, False, None, None, None, 1, lead, 64 if lead else 0, 2 if lead else 0, 32, 4, 1, 0, lead)


# a plain call of every function, and the launchers that it makes
PLAIN = {
    "rmsnorm": (lambda: (bf(3, 64), bf(64), 1e-5, bf(3, 64), True), ["ts_rmsnorm"]),
    "stream_post_norm": (lambda: (torch.zeros(3, 64), torch.zeros(3, 64), torch.zeros(64), None, 1e-6, torch.zeros(64), 1e-5, 1), ["ts_stream_post_norm"]),
    "stream_update_norm": (lambda: (torch.zeros(3, 64), bf(3, 64), None, 0.5, bf(64), 1e-5, 1), ["ts_stream_update_norm"]),
    "gemm_library": (lambda: (bf(9, 64), bf(16, 64), True), ["ts_gemm_library_bf16"]),
    "gemm_slices": (lambda: (bf(9, 384), bf(16, 384), 0, 2, False, bf(9, 16), bf(16), 1e-5), ["ts_gemm_slices_bf16"]),
    "gemm_glu": (lambda: (bf(9, 64), bf(32, 64), 0, 0, 0.0, 1.0, 0.0), ["ts_gemm_glu_bf16"]),
    "gemm_rows64": (lambda: (bf(9, 1024), bf(8, 32, 64, 8), False, 1, None, 0.0, 0.0, 0.0, 0.0), ["ts_gemm_rows64_bf16"]),
    "gemm_rows64_sliced": (lambda: (bf(9, 1024), bf(4, 32, 64, 8), 2, None, bf(64)), ["ts_gemm_rows64_sliced_bf16"]),
    "rope_store": (lambda: (bf(3, 8 * 64), torch.zeros(9, 64), ints(0, 1, 2), ints(0, 1, 2), *caches(), 4, 2, 64), ["ts_rope_store"]),
    "qkv_rope_store_sliced": (lambda: (bf(3, 1024), bf(32, 32, 64, 8), 2, torch.zeros(9, 64), ints(0, 1, 2), ints(0, 1, 2), *caches(), 4, 2, 64, 0.0, None),
                              ["ts_gemm_rows64_sliced_rope_bf16"]),
    "qkv_finish": (lambda: (torch.zeros(3, 8 * 64), torch.zeros(16, dtype=torch.float64), ints(0, 1, 2), ints(0, 1, 2), *caches(), 4, 2, 64, 64, 1, False, None, 1e-6, 1.0),
                   ["ts_qkv_finish"]),
    "attention_step": (lambda: step(0), ["ts_paged_attention_prefill"]),
    "capped_glu": (lambda: (torch.zeros(3, 64), 3.0, 1.0, 0.0, 1, 0), ["ts_capped_glu"]),
    "mlstm_finish": (lambda: (torch.zeros(3, 64), None, torch.zeros(3, 64), 2, 32, 1e-6, 1, False), ["ts_mlstm_finish"]),
}


def test_every_function_is_here(stub):
    assert sorted(PLAIN) == sorted(n for n in dir(stub[0]) if not n.startswith("_"))


@pytest.mark.parametrize("name", PLAIN)
def test_a_refusal_is_left_to_the_general_function_and_a_failed_launch_is_raised(stub, name):
    """A launch that failed may have run, and written to what it updates in place: it is not to be made once more."""
    module, answer, called = stub
    args, launchers = PLAIN[name]
    assert getattr(module, name)(*args()) is not None and called() == launchers
    for rc in (BAD_DTYPE, BAD_SHAPE, TOO_LARGE):
        answer(launchers[0], rc)
        assert getattr(module, name)(*args()) is None and called() == launchers
    answer(launchers[0], LAUNCH_FAILED)
    with pytest.raises(hip.KernelError, match=hip._ERRORS[LAUNCH_FAILED]):
        getattr(module, name)(*args())
    assert called() == launchers
    answer(launchers[0], OK)


@pytest.mark.parametrize("softcap", [0.0, 20.0])
def test_a_step_whose_decoding_part_has_run_is_not_made_again(stub, softcap):
    module, answer, called = stub
    general = "_general" if softcap else ""
    decode, prefill = f"ts_paged_attention_decode{general}", f"ts_paged_attention_prefill{general}"
    assert module.attention_step(*step(2, softcap)) is not None and called() == [decode, prefill]
    answer(decode, BAD_SHAPE)
    assert module.attention_step(*step(2, softcap)) is None and called() == [decode]
    answer(decode, OK)
    for rc in (BAD_SHAPE, LAUNCH_FAILED):
        answer(prefill, rc)
        with pytest.raises(hip.KernelError, match=f"paged_attention_prefill{general}: {re.escape(hip._ERRORS[rc])}"):
            module.attention_step(*step(2, softcap))
        assert called() == [decode, prefill]
    answer(prefill, BAD_SHAPE)
    assert module.attention_step(*step(0, softcap)) is None and called() == [prefill]
    answer(prefill, OK)


@pytest.mark.parametrize("softcap", [0.0, 20.0])
def test_a_step_of_decoding_tokens_and_prompts_is_one_launch_or_two(stub, softcap):
    module, answer, called = stub
    general = "_general" if softcap else ""
    both, decode, prefill = "ts_paged_attention_step", f"ts_paged_attention_decode{general}", f"ts_paged_attention_prefill{general}"
    change = lambda **other: [other.get(f"a{i}", a) for i, a in enumerate(step(2, softcap))]
    wide = dict(a16=128, a17=4)      # (chunks for as many waves as the prompts' tiles have)
    assert module.attention_step(*change(**wide)) is not None and called() == [both]
    for rc in (BAD_DTYPE, BAD_SHAPE, TOO_LARGE):
        answer(both, rc)
        assert module.attention_step(*change(**wide)) is not None and called() == [both, decode, prefill]
    answer(both, LAUNCH_FAILED)
    with pytest.raises(hip.KernelError, match=f"paged_attention_step: {re.escape(hip._ERRORS[LAUNCH_FAILED])}"):
        module.attention_step(*change(**wide))
    assert called() == [both]
    answer(both, OK)
    # fewer waves than a tile's, tiles of four rows of 16 a wave, prompts in parts
    for other in (dict(a16=64, a17=2), dict(wide, a18=128), dict(wide, a20=2, a21=64)):
        assert module.attention_step(*change(**other)) is not None and called() == [decode, prefill]


def test_a_stream_is_updated_by_one_launch(stub, monkeypatch):
    module, answer, called = stub
    monkeypatch.setattr(hip, "_native", lambda: module)
    answer("ts_stream_update_norm", LAUNCH_FAILED)
    with pytest.raises(hip.KernelError, match="stream_update_norm"):
        hip.stream_update_norm(torch.zeros(3, 64), bf(3, 64), weights=(bf(64), None), eps=1e-5, out_dtype=BF)
    assert called() == ["ts_stream_update_norm"]
    answer("ts_stream_update_norm", OK)


def test_the_limits_are_those_of_the_general_functions():
    """The numbers that calls.cpp holds for itself, by which it takes or leaves a call."""
    with open(os.path.join(build.HERE, "calls.cpp")) as f:
        held = dict(re.findall(r"\b([A-Z][A-Z0-9_]+) = (\d+)[,;]", f.read()))
    assert {name: int(value) for name, value in held.items()} == {
        "DECODE_MAX_TOKENS": hip.MAX_DECODE_TOKENS, "MAX_SPLITS": hip.MAX_DECODE_SPLITS, "ROWS64_MAX_ROWS": hip.ROWS64_MAX_ROWS, "ROWS64_SLICE_K": hip.ROWS64_SLICE_K,
        "ROW_SKEW": hip.OPERAND_ROW_SKEW, "GATED_SKEW_MIN_ROWS": hip.GATED_SKEW_MIN_ROWS}


def test_a_group_of_products(stub):
    """`gemm_slices` with tuples of operands: in whole tiles, or with packed copies by the kernel that streams them; anything another way is left alone."""
    module, answer, called = stub
    xs, ws, packed = (bf(9, 1024), bf(9, 1024)), (bf(64, 1024), bf(32, 1024)), bf(6, 32, 64, 8)
    for copies, launcher in ((None, "ts_gemm_whole_bf16"), (packed, "ts_gemm_rows64_group_bf16")):
        ys = module.gemm_slices(xs, ws, 0, copies)
        assert [(y.dtype, tuple(y.shape)) for y in ys] == [(F32, (9, 64)), (F32, (9, 32))] and called() == [launcher]
        answer(launcher, BAD_SHAPE)
        assert module.gemm_slices(xs, ws, 0, copies) is None and called() == [launcher]
        answer(launcher, LAUNCH_FAILED)
        with pytest.raises(hip.KernelError, match=hip._ERRORS[LAUNCH_FAILED]):
            module.gemm_slices(xs, ws, 0, copies)
        answer(launcher, OK)
        called()
        for other in ((list(xs), ws), (xs, ws[:1]), ((), ()), (xs * 5, ws * 5), ((xs[0], None), ws), ((xs[0], bf(8, 1024)), ws), ((xs[0], xs[1].float()), ws),
                      ((xs[0], bf(9, 1032)[:, :1024]), ws), ((xs[0], bf(9 * 1024 + 1)[1:].view(9, 1024)), ws), (xs, (ws[0], bf(1024, 32).t())), (xs, (ws[0], bf(28, 1024))),
                      (xs, (ws[0], bf(32, 512))), (tuple(x[:0] for x in xs), ws), (tuple(x[:, :128] for x in xs), tuple(w[:, :128] for w in ws))):
            assert module.gemm_slices(*other, 0, copies) is None and called() == []
    many = tuple(bf(129, 1024) for _ in xs)
    assert module.gemm_slices(many, ws, 0, None) is not None and called() and module.gemm_slices(many, ws, 0, packed) is None
    for other in (bf(6, 16, 64, 8), bf(5, 32, 64, 8), packed.float()):
        assert module.gemm_slices(xs, ws, 0, other) is None and called() == []


def test_the_two_meanings_of_a_q_k_v_call_are_kept_apart(stub, monkeypatch):
    """The module tells a packed weight from one as it is; neither general function takes the other's."""
    module, answer, called = stub
    monkeypatch.setattr(hip, "_native", lambda: module)
    weight, packed, rest = bf(512, 1024), bf(32, 32, 64, 8), (torch.zeros(9, 64), ints(0, 1, 2), ints(0, 1, 2), *caches(), 4, 2, 64)
    hip.qkv_rope_store_sliced(bf(3, 1024), packed, 2, *rest), hip.qkv_rope_store_whole(bf(3, 1024), weight, 2, *rest)
    assert called() == ["ts_gemm_rows64_sliced_rope_bf16", "ts_gemm_whole_rope_bf16"]
    for bad in (lambda: hip.qkv_rope_store_sliced(bf(3, 1024), weight, 2, *rest), lambda: hip.qkv_rope_store_whole(bf(3, 1024), packed, 2, *rest)):
        with pytest.raises(hip.KernelError):
            bad()
    assert called() == []


def test_calls_of_few_rows_reach_the_kernels_that_stream_the_copies(stub):
    """The forms of three calls that lead to another kernel: no slices, and the 8-row form's copy."""
    module, answer, called = stub
    rope = lambda slices, heads=4: (bf(3, 1024), bf(32, 32, 64, 8), slices, torch.zeros(9, 64), ints(0, 1, 2), ints(0, 1, 2), *caches(), heads, 2, 64, 1e-5, torch.zeros(3, 2))
    into = lambda res=bf(3, 64), nw=bf(64): (bf(3, 1024), bf(4, 32, 64, 8), 0, res, nw)
    few = lambda x=bf(8, 1024), p=bf(4, 4, 4, 64, 8), unit=0, squares=None: (x, p, True, unit, squares, 0.0, 0.0, 0.0, 0.0)
    for call, plain, refused, launcher, shape in (
            (module.qkv_rope_store_sliced, rope(0), [rope(-1), rope(0, 5)], "ts_gemm_skinny_rope_bf16", (3, 4, 64)),
            (module.gemm_rows64_sliced, into(), [into(None, None), into(bf(3, 32)), into(nw=bf(32))], "ts_gemm_skinny_bf16", (3, 64)),
            (module.gemm_rows64, few(), [few(bf(9, 1024)), few(bf(8, 1032)), few(unit=1), few(squares=torch.zeros(8, 1)), few(p=bf(4, 4, 4, 64, 8).float())],
             "ts_gemm_skinny8_bf16", (8, 32))):
        y = call(*plain)
        y = y[0] if isinstance(y, tuple) else y
        assert called()[-1] == launcher and tuple(y.shape) == shape
        assert [call(*args) for args in refused] == [None] * len(refused) and called() == []
        answer(launcher, BAD_SHAPE)
        assert call(*plain) is None and called()[-1] == launcher
        answer(launcher, OK)


def test_the_general_functions_of_few_rows_take_what_they_say(stub, monkeypatch):
    """What the module's forms that share a name would take of another function's operands, or without a look at the weight that a copy is of."""
    module, _, called = stub
    monkeypatch.setattr(hip, "_native", lambda: module)
    x, w, w512, p16, p16q, p8 = bf(3, 1024), bf(64, 1024), bf(512, 1024), bf(4, 32, 64, 8), bf(32, 32, 64, 8), bf(8, 4, 4, 64, 8)
    rope = (torch.zeros(9, 64), ints(0, 1, 2), ints(0, 1, 2), *caches(), 4, 2, 64)
    away = lambda t: torch.empty_like(t, device="meta")
    into = dict(packed=p16, next_norm=(None, bf(64)))
    for good, launcher in ((lambda: hip.gemm_rows64(x, p16), "ts_gemm_rows64_bf16"), (lambda: hip.gemm_rows64_sliced(x, p16, 2), "ts_gemm_rows64_sliced_bf16"),
                           (lambda: hip.qkv_rope_store_sliced(x, p16q, 2, *rope), "ts_gemm_rows64_sliced_rope_bf16"),
                           (lambda: hip.gemm_skinny8(x, w, BF, p8), "ts_gemm_skinny8_bf16"), (lambda: hip.gemm_skinny(x, w, **into), "ts_gemm_skinny_bf16"),
                           (lambda: hip.qkv_rope_store(x, w512, *rope, packed=p16q), "ts_gemm_skinny_rope_bf16"),
                           (lambda: hip.stream_update_norm(torch.zeros(3, 64), None, hip.RowParts(torch.zeros(2, 3, 64)), weights=(bf(64), None), out_dtype=BF), "ts_stream_update_norm_parts"),
                           (lambda: hip.stream_post_norm(torch.zeros(3, 64), hip.RowParts(torch.zeros(2, 3, 64)), torch.zeros(64), None, 1e-6, out_dtype=BF), "ts_stream_post_norm_parts")):
        good()
        assert called()[-1] == launcher
    for bad in (lambda: hip.gemm_rows64(x, p8), lambda: hip.gemm_rows32(x, p8), lambda: hip.gemm_rows64_sliced(x, p16, 0, next_norm=(None, bf(64))),
                lambda: hip.qkv_rope_store_sliced(x, p16q, 0, *rope), lambda: hip.gemm_skinny8(x, away(w), BF, p8), lambda: hip.gemm_skinny8(x, bf(64), BF, p8),
                lambda: hip.gemm_skinny8(x, w, F32, p8, cap=-1.0), lambda: hip.gemm_skinny8(x, w, F32, p8, cap=float("nan")), lambda: hip.gemm_rows64(x, p16, F32, cap=-1.0),
                lambda: hip.gemm_rows64(x, p16, cap=1.0), lambda: hip.gemm_skinny(x, away(w), **into), lambda: hip.gemm_skinny(x, w, unit=("sigmoid", 0.0, 1.0, 0.0), **into),
                lambda: hip.qkv_rope_store(x, away(w512), *rope, packed=p16q),
                lambda: hip.stream_update_norm(torch.zeros(3, 64), None, (torch.zeros(2, 3, 64),), weights=(bf(64), None), out_dtype=BF),
                lambda: hip.stream_post_norm(torch.zeros(3, 64), (torch.zeros(2, 3, 64),), torch.zeros(64), None, 1e-6, out_dtype=BF)):
        with pytest.raises((hip.KernelError, AttributeError)):      # (a tuple is no tensor)
            bad()
        assert called() == []
    plain = lambda copy: module.gemm_rows64(x, copy, True, 0, None, 0.0, 0.0, 0.0, 0.0)
    assert plain(p8) is not None and called() == ["ts_gemm_skinny8_bf16"]
    assert plain(bf(8, 2, 8, 64, 8)) is None and plain(bf(8, 1, 16, 64, 8)) is None and called() == []      # (copies for a reader of other steps)


@pytest.mark.parametrize("k", [256, 512, 1024, 2048, 2304, 4096, 8192, 1024 * 16, 1024 * 17, 96, 5120])
def test_the_steps_of_the_8_row_form_are_the_same_on_both_sides(stub, k):
    module, _, called = stub
    steps = hip.skinny8_steps(k)
    for tried in (4, 8, 16):
        taken = k % (64 * tried) == 0 and module.gemm_rows64(bf(1, k), bf(1, k // (64 * tried), tried, 64, 8), True, 0, None, 0.0, 0.0, 0.0, 0.0) is not None
        assert taken == (tried == steps)
    called()
