"""Up to 32 rows by the kernel that shares x among 64 rows of W: the bits of the 16-row weight-streaming form, which served them before, and the
rule that chooses."""

from __future__ import annotations

import pytest
import torch

from tinyserve_llm_amd.ops import hip
from tinyserve_llm_amd.parts.linear import few_rows_unit, linear, streaming_copy

BF = torch.bfloat16


def operands(rows, n, k, skew=0):
    g = torch.Generator().manual_seed(rows + n + k)
    x = torch.randn(rows, k + skew, generator=g).to(BF).cuda()[:, :k]
    return x, (torch.randn(n, k, generator=g) * k ** -0.5).to(BF).cuda()


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 2, 5, 8, 9, 15, 16, 17, 31, 32])
@pytest.mark.parametrize("n, k, skew", [(128, 1024, 0), (640, 2048, 8), (256, 3072, 0), (384, 4096, 0)])
def test_the_sums_are_the_16_row_forms(rows, n, k, skew):
    x, w = operands(rows, n, k, skew)
    packed = hip.pack_weight(w)
    for dtype in (torch.float32, BF):
        assert torch.equal(hip.gemm_rows32(x, packed, dtype), hip.gemm_skinny(x, w, dtype)[0])
    if hip.skinny_fuses(rows, k, False, True):
        gated, unit = hip.gemm_rows32(x, packed, glu=True), hip.gemm_rows32(x, packed, glu=True, unit=("relu", 0.5, 1.0, 0.25))
        assert torch.equal(gated, hip.gemm_skinny(x, w, glu=True)[0]) and torch.equal(unit, hip.gemm_skinny(x, w, glu=True, unit=("relu", 0.5, 1.0, 0.25))[0])
        if rows <= 8 and n // 2 % 256 == 0:
            for u in (None, ("relu", 0.5, 1.0, 0.25)):
                handed = hip.gemm_rows32(x, packed, glu=True, unit=u, pack8_steps=4)
                assert isinstance(handed, hip.PackedRows8) and torch.equal(handed.rows(), gated if u is None else unit)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 8, 16, 17, 32])
@pytest.mark.parametrize("parts", [1, 2, 63, 64, 256, 257, 300])
def test_a_prepared_norms_parts_are_added_up(rows, parts):
    """The scale of a row from `parts` sums of squares: those sums' roundings, at most parts + 6 of 2^-24, halve in the root, and two more follow."""
    x, w = operands(rows, 128, 1024)
    sq = torch.rand(rows, parts, generator=torch.Generator().manual_seed(parts)).cuda() * 16
    sums = hip.gemm_rows32(x, hip.pack_weight(w), torch.float32)
    got = hip.gemm_rows32(x, hip.pack_weight(w), torch.float32, squares=sq, eps=1e-5)
    want = sums.double() * torch.rsqrt(sq.double().sum(1, keepdim=True) / 1024 + 1e-5)
    torch.testing.assert_close(got.double(), want, rtol=(parts + 10) * 2.0 ** -24, atol=0.0)
    if rows > 1:
        assert torch.equal(hip.gemm_rows32(x[rows - 1:], hip.pack_weight(w), torch.float32, squares=sq[rows - 1:].contiguous(), eps=1e-5)[0], got[rows - 1])


@pytest.mark.gpu
def test_wide_products_of_few_rows_go_there(monkeypatch):
    """Through the parts, with the packed copy and without it: the same numbers."""
    went, real = [], hip.gemm_rows32
    monkeypatch.setattr(hip, "gemm_rows32", lambda *a, **k: went.append(a[0].shape[0]) or real(*a, **k))
    for rows, n, k in ((5, 10304, 2048), (16, 5120, 2048), (8, 16384, 1024)):
        x, w = operands(rows, n, k)
        assert torch.equal(linear(x, w, torch.float32, packed=streaming_copy(w)), linear(x, w, torch.float32)) and went.pop() == rows and not went
    for rows in (5, 8, 16, 32):
        x, w = operands(rows, 16384, 2048)
        assert torch.equal(linear(x, w, glu=True, packed=streaming_copy(w)), linear(x, w, glu=True)) and went.pop() == rows and not went
        down = torch.empty(2048, 8192, dtype=BF, device="cuda")
        handed = few_rows_unit(x, w, streaming_copy(w), down, ("gelu_tanh", 0.0, 1.0, 0.0))
        assert isinstance(handed, hip.PackedRows8) == (2 <= rows <= 8) and went.pop() == rows and not went
    x, w = operands(4, 16384, 2048)
    assert torch.equal(linear(x, w, torch.float32, packed=streaming_copy(w)), hip.gemm_skinny8(x, w, torch.float32)) and not went


@pytest.mark.gpu
def test_packed_rows_are_refused_where_no_reader_takes_them():
    x, w = operands(33, 1024, 1024)
    packed = hip.pack_weight(w)
    for bad in (lambda: hip.gemm_rows32(x, packed), lambda: hip.gemm_rows32(x[:9], packed, glu=True, pack8_steps=4), lambda: hip.gemm_rows32(x[:8], packed, pack8_steps=4),
                lambda: hip.gemm_rows32(x[:8], packed, glu=True, pack8_steps=16), lambda: hip.gemm_rows32(x[:8], packed, glu=True, pack8_steps=5)):
        with pytest.raises(hip.KernelError):
            bad()


def test_the_rule_takes_what_was_measured_faster():
    few = hip.rows64_few
    assert few(5, 128256, 2048) and few(32, 128256, 4096) and few(5, 10304, 1024) and few(9, 5120, 3072) and few(17, 5120, 2048) and few(24, 8192, 3072)
    assert few(5, 16384, 2048, True) and few(5, 8192, 2048, True) and few(32, 8192, 2048, True) and few(8, 16384, 1024, True)
    for rows, n, k in ((4, 128256, 2048), (8, 8192, 2048), (16, 4096, 2048), (9, 8192, 4096), (17, 8192, 1024), (17, 8192, 4096), (24, 5120, 3072), (33, 16384, 2048),
                       (0, 16384, 2048), (8, 16392, 2048), (8, 16384, 2560), (8, 16384, 5120)):
        assert not few(rows, n, k)
    for rows, n, k in ((1, 16384, 2048), (4, 16384, 4096), (8, 8192, 3072), (32, 8192, 3072), (16, 4096, 2048), (8, 16448, 2048), (33, 16384, 2048)):
        assert not few(rows, n, k, True)


def test_the_gate_s_line_is_a_bound_on_the_reduction():
    few = hip.rows64_few
    for rows in (5, 8, 9, 16):
        assert few(rows, 8192, 2048, True) and not few(rows, 8192, 3072, True) and not few(rows, 8192, 4096, True)
        assert all(few(rows, 8320, k, True) for k in (2048, 3072, 4096)) and not any(few(rows, 8064, k, True) for k in (1024, 2048, 3072, 4096))
    for rows, n, taken in ((5, 16384, False), (7, 28672, False), (8, 8192, False), (8, 16384, True), (9, 8192, True), (16, 8192, True), (17, 11264, False), (17, 16384, True), (32, 8192, False)):
        assert few(rows, n, 1024, True) == taken
    assert few(17, 8192, 2048, True) and few(32, 8192, 2048, True)
