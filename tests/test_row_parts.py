"""Who is asked to leave rows in parts to a 32-bit stream."""

from __future__ import annotations

import pytest

from tinyserve_llm_amd.parts import block
from tinyserve_llm_amd.parts.gated_delta import GatedDelta
from tinyserve_llm_amd.parts.mlp import CappedGLU
from tinyserve_llm_amd.parts.moe import RoutedExperts
from tinyserve_llm_amd.parts.side_by_side import SideBySide


@pytest.mark.parametrize("base", [GatedDelta, CappedGLU, RoutedExperts, SideBySide])
def test_a_class_with_a_forward_of_its_own_is_asked_for_parts_only_if_it_says_so(base):
    class Plain(base):
        def __init__(self):
            pass

        def forward(self, x, rest):
            return x, rest

    class Leaves(Plain):
        leaves_parts = True

        def forward(self, x, rest, parts=False):
            return x, rest, parts

    class Below(Leaves):
        pass
    assert base.leaves_parts and not Plain.leaves_parts and Leaves.leaves_parts and Below.leaves_parts
    assert block._into_stream(Plain(), 1, 2) == (1, 2)
    assert block._into_stream(Leaves(), 1, 2) == (1, 2, True)
    assert block._into_stream(Below(), 1, 2) == (1, 2, True)
