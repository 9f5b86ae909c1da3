"""The host side of a routed layer's device routing (kernels.moe_routing), on the CPU."""

from __future__ import annotations

import pytest
import torch

from kernels import moe_grouped, moe_routing
from serve import quantize


class _FakeRoute:
    made = []
    seg_off = pos = token_of_slot = None

    def __init__(self, idx, n):
        self.calls = []
        _FakeRoute.made.append(self)

    @staticmethod
    def takes(idx, n):
        return True

    def wait(self):
        self.calls.append("wait")

    def check(self):
        self.calls.append("check")


@pytest.mark.parametrize("fails", [False, True])
def test_the_routing_launch_has_ended_when_its_pinned_word_goes(monkeypatch, fails):
    """The routing kernel writes a pinned word that the host allocator does not know to be in use:
    a layer that raises between the launch and the check waits for it all the same."""
    def layer(*a, **k):
        if fails:
            raise ValueError("refused")
        return "out"

    slots = {n: (None, None) for n in ("w_gate", "w_up", "w_down")}
    monkeypatch.setattr(quantize, "stacked_int4_experts", lambda experts: {**slots, "group_size": 32})
    monkeypatch.setattr(moe_grouped, "int4_expert_mlp_combine", layer)
    monkeypatch.setattr(moe_routing, "_Route", _FakeRoute)
    x = torch.zeros(2, 4, dtype=torch.bfloat16)
    if fails:
        with pytest.raises(ValueError, match="refused"):
            moe_routing.moe_dispatch_combine(x, None, torch.zeros(2, 1, dtype=torch.int64), [None])
        assert _FakeRoute.made[-1].calls == ["wait"]
    else:
        assert moe_routing.moe_dispatch_combine(x, None, torch.zeros(2, 1, dtype=torch.int64), [None]) == "out"
        assert _FakeRoute.made[-1].calls == ["check"]
