"""Two mixers side by side: both read the same input, and the result is left_scale * left + right_scale * right. Each is a
mixer of its own kind with its own parameters (`left_...`, `right_...`); at most one of them keeps a cache and at most
one keeps per-request state, which the pair passes on as its own. Where both offer their products apart (`Mixer.in_three`), the
first ones of both are made together, and so are the last ones (`products`): seven products of 48 rows that a pair of attention and
shifted decay begins with took 74 µs one by one and take 15."""

from __future__ import annotations

import torch

from tinyserve_llm_amd.ops import hip
from tinyserve_llm_amd.parts.base import KVSpec, LayerMemory, Mixer, ParamSpec, PartSpec, StateSpec, StepContext, make, register
from tinyserve_llm_amd.parts.linear import packed_together, products


@register("mixer", "side_by_side")
class SideBySide(Mixer):
    leaves_parts = True

    def __init__(self, left: PartSpec, right: PartSpec, left_scale: float = 1.0, right_scale: float = 1.0) -> None:
        self.left, self.right = make("mixer", left), make("mixer", right)
        self.left_scale, self.right_scale = float(left_scale), float(right_scale)
        self.in_threes = self.left.in_three and self.right.in_three
        self.first_together: torch.Tensor | None = None      # `packed_together` of both mixers' first products, and of their last ones
        self.last_together: torch.Tensor | None = None
        if self.left.kv_spec() is not None and self.right.kv_spec() is not None:
            raise ValueError("of two mixers side by side at most one keeps a cache")
        if self.left.state_spec() is not None and self.right.state_spec() is not None:
            raise ValueError("of two mixers side by side at most one keeps per-request state")

    @property
    def graph_safe(self) -> bool:
        return self.left.graph_safe and self.right.graph_safe

    def param_specs(self) -> dict[str, ParamSpec]:
        specs = {f"left_{n}": ps for n, ps in self.left.param_specs().items()}
        specs.update({f"right_{n}": ps for n, ps in self.right.param_specs().items()})
        return specs

    def bind(self, params) -> None:
        self.left.bind({n[len("left_"):]: t for n, t in params.items() if n.startswith("left_")})
        self.right.bind({n[len("right_"):]: t for n, t in params.items() if n.startswith("right_")})

    def kv_spec(self) -> KVSpec | None:
        return self.left.kv_spec() or self.right.kv_spec()

    def state_spec(self) -> StateSpec | None:
        return self.left.state_spec() or self.right.state_spec()

    def widest_activation(self) -> int:
        return max(self.left.widest_activation(), self.right.widest_activation())

    def keep_streaming_copies(self) -> int:
        if not self.in_threes:
            return self.left.keep_streaming_copies() + self.right.keep_streaming_copies()
        held = self.left.keep_product_copies() + self.right.keep_product_copies()
        self.first_together, first = packed_together(self.left.first_weights() + self.right.first_weights())
        self.last_together, last = packed_together([(m.o, m.o_packed) for m in (self.left, self.right)])
        return held + first + last

    def forward(self, x: torch.Tensor, ctx: StepContext, mem: LayerMemory, parts: bool = False) -> "torch.Tensor | hip.RowParts":
        if not self.in_threes:
            a = self.left.forward(x, ctx, mem)
            b = self.right.forward(x, ctx, mem)
        else:
            pairs = [(self.left, self.left.first_weights()), (self.right, self.right.first_weights())]
            sums = products([(rows, w, c) for m, weights in pairs for rows, (w, c) in zip(m.first_rows(x, ctx, mem), weights)], self.first_together)
            at = len(pairs[0][1])
            lasts = [m.between(part, x, ctx, mem) for m, part in ((self.left, sums[:at]), (self.right, sums[at:]))]
            a, b = products([(rows, m.o, m.o_packed) for m, rows in zip((self.left, self.right), lasts)], self.last_together)
        sides = hip.RowParts((a, b), (self.left_scale, self.right_scale))
        return sides if parts else sides.rows()
