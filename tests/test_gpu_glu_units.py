"""The gated units' forms (glu_unit.h) against 64 bits, at ordinary gates and at the ends of the type's range."""

from __future__ import annotations

import math

import pytest
import torch

from tinyserve_llm_amd.ops import hip

F32, F64 = torch.float32, torch.float64
pytestmark = pytest.mark.gpu


def gate(form, g, slope):
    g = g.to(F64)
    if form == "relu":
        return g.clamp_min(0.0)
    return g * torch.sigmoid(slope * g if form == "sigmoid" else 2.0 * math.sqrt(2.0 / math.pi) * (g + 0.044715 * g ** 3))


@pytest.mark.parametrize("form,slope", [("sigmoid", 1.0), ("sigmoid", 1.702), ("sigmoid", -0.5), ("gelu_tanh", 1.0)])
@pytest.mark.parametrize("size", [0.5, 3.0, 20.0])
def test_units_are_32_bit_numbers_near_their_64_bit_values(form, slope, size):
    g = torch.randn(64, 4096, generator=torch.Generator().manual_seed(1)) * size
    u = torch.ones_like(g)
    y = hip.capped_glu(torch.cat([g, u], 1).cuda(), 0.0, slope, 0.0, F32, activation=form).cpu().to(F64)
    want = gate(form, g, slope)
    # two units in the last place of 2^-24 for the quotient and the exponential, and of the exponent's own size for what is rounded in it; gelu's 1 + tanh is
    # of numbers up to 1, so what is rounded in it counts against the gate itself: four units, a product's, a cube's and the tangent's two
    if form == "gelu_tanh":
        bound = 4.0 * 2.0 ** -23 * g.abs().to(F64) + 1e-36
    else:
        bound = (2.0 + (slope * g).abs().to(F64)) * 2.0 ** -23 * want.abs() + 1e-36
    assert bool(((y - want).abs() <= bound).all())


@pytest.mark.parametrize("form,slope", [("sigmoid", 1.0), ("sigmoid", 1.702), ("gelu_tanh", 1.0)])
def test_units_at_the_ends_of_the_range(form, slope):
    inf = math.inf
    g = torch.tensor([[inf, -inf, math.nan, 0.0, -0.0, 88.0, -89.0, -100.0, 1e30, -1e30, 3e38, -3e38, 1e-40]])
    y = hip.capped_glu(torch.cat([g, torch.ones_like(g)], 1).cuda(), 0.0, slope, 0.0, F32, activation=form).cpu()[0]
    assert y[0] == inf and y[1].isnan() and y[2].isnan()      # (as the library's exponential and a division have them)
    assert y[3] == 0 and y[4] == 0 and y[5] == 88.0 and y[8] == 1e30 and y[10] == torch.tensor(3e38)
    assert bool((y[[6, 7, 9, 11]].abs() < 1e-35).all()) and y[12].abs() < 1e-39
    capped = hip.capped_glu(torch.cat([g, torch.full_like(g, 9.0)], 1).cuda(), 7.0, slope, 0.5, F32, activation=form).cpu()[0]
    top = gate(form, torch.tensor(7.0), slope).item() * 7.5
    torch.testing.assert_close(capped[[0, 5, 8, 10]], torch.full((4,), top, dtype=F32), rtol=1e-6, atol=0.0)


@pytest.mark.parametrize("rows", [3, 20, 200])
@pytest.mark.parametrize("form", ["sigmoid", "gelu_tanh"])
def test_a_unit_does_not_depend_on_the_kernel_that_makes_it(rows, form):
    g = torch.Generator(device="cuda").manual_seed(rows)
    x = torch.randn(rows, 1024, generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randn(512, 1024, generator=g, device="cuda") / 16).to(torch.bfloat16)
    made = [hip.gemm_glu(x, w, form, 5.0, 1.3, 0.25)]
    if rows <= 128:
        made.append(hip.gemm_rows64(x, hip.pack_weight(w), glu=True, unit=(form, 5.0, 1.3, 0.25)))
    if rows <= 32:
        made.append(hip.gemm_skinny(x, w, glu=True, unit=(form, 5.0, 1.3, 0.25))[0])
    sums = (x.to(F64) @ w.to(F64).t()).to(F32)
    apart = hip.capped_glu(sums, 5.0, 1.3, 0.25, torch.bfloat16, activation=form).to(F32)
    for y in made:      # (their sums are in orders of their own: a bfloat16 place apart at most)
        assert bool(((y.to(F32) - apart).abs() <= 2.0 ** -7 * apart.abs() + 1e-6).all())


def test_the_sigmoid_keeps_what_is_left_of_large_negative_gates():
    """g e^g down to the smallest normal numbers, by every kernel that makes the unit: g is one product, exact in bfloat16."""
    gates = torch.tensor([-80.0, -87.0, -87.5, -88.0, -88.5], device="cuda")
    want = gate("sigmoid", gates.cpu(), 1.0)
    apart = hip.capped_glu(torch.cat([gates, torch.ones_like(gates)])[None], 0.0, 1.0, 0.0, F32, activation="sigmoid").cpu().to(F64)[0]
    assert bool(((apart - want).abs() <= 91 * 2.0 ** -23 * want.abs()).all())      # (the exponent's rounding, and two places)
    w = torch.zeros(128, 1024, device="cuda")
    w[:5, 0], w[64:69, 0] = gates, 1.0
    w = w.to(torch.bfloat16)
    for rows in (1, 3, 20, 200):
        x = torch.zeros(rows, 1024, device="cuda", dtype=torch.bfloat16)
        x[:, 0] = 1.0
        made = [hip.gemm_glu(x, w, "sigmoid", 0.0, 1.0, 0.0)]
        if rows <= 128:
            made.append(hip.gemm_rows64(x, hip.pack_weight(w), glu=True, unit=("sigmoid", 0.0, 1.0, 0.0)))
        if rows <= 32:
            made.append(hip.gemm_skinny(x, w, glu=True, unit=("sigmoid", 0.0, 1.0, 0.0))[0])
        for y in made:
            y = y[:, :5].cpu().to(F64)
            assert bool(((y - want).abs() <= 2.0 ** -8 * want.abs()).all())
