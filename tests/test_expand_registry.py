"""The grouped-expansion registry of claudemaxing_amd/expand.py on the host (no GPU): an
expansion left for a weight is handed out once, only in fp16, and dropped with its device's
entries; a weight with no recorded group gets no backward group; a layer without NF4
projections is left alone."""

import torch

from claudemaxing_amd import expand


def test_take_hands_an_expansion_out_once():
    packed = torch.zeros(8, dtype=torch.uint8)
    w = torch.ones(2, 2, dtype=torch.float16)
    expand._READY[packed.device.index] = {packed.data_ptr(): w}
    try:
        assert expand.take(packed, torch.float32) is None  # another dtype: not this expansion
        assert expand.take(packed, torch.float16) is w
        assert expand.take(packed, torch.float16) is None  # once
    finally:
        expand.drop(packed.device)


def test_take_pair_and_drop():
    gate, up = torch.zeros(8, dtype=torch.uint8), torch.zeros(8, dtype=torch.uint8)

    class Proj:
        def __init__(self, packed):
            self.packed = packed

    w2 = torch.ones(4, 2, dtype=torch.float16)
    key = ("pair", gate.data_ptr(), up.data_ptr())
    expand._READY[gate.device.index] = {key: w2}
    assert expand.take_pair(Proj(up), Proj(gate)) is None  # the order matters: [Wg; Wu]
    expand.drop(gate.device)
    assert expand.take_pair(Proj(gate), Proj(up)) is None  # dropped
    expand._READY[gate.device.index] = {key: w2}
    assert expand.take_pair(Proj(gate), Proj(up)) is w2
    expand.drop(gate.device)


def test_no_group_without_a_recorded_layer():
    packed = torch.zeros(8, dtype=torch.uint8)
    assert expand.backward_group(packed, torch.float16) is None


def test_layer_without_nf4_projections_is_left_alone():
    layer = torch.nn.Module()
    layer.self_attn = torch.nn.Module()
    layer.self_attn.o_proj = torch.nn.Linear(4, 4)
    layer.mlp = torch.nn.Module()
    for name in ("gate_proj", "up_proj", "down_proj"):
        setattr(layer.mlp, name, torch.nn.Linear(4, 4))
    hidden = torch.zeros(1, 3, 4)
    expand.expand_layer(layer, hidden)
    assert not expand._READY.get(hidden.device.index)


class State:
    def __init__(self):
        self.absmax = torch.zeros(1)


def _left(*keys_pairs):
    left = expand._Left(torch.device("cpu"))
    for key, pairs in keys_pairs:
        left.leave(key, torch.ones(2, 2, dtype=torch.float16), pairs)
    expand._READY[None] = left
    return left


def test_take_rows_is_handed_out_once_in_its_order():
    q, k, v = ((torch.zeros(8, dtype=torch.uint8), State()) for _ in range(3))
    key = expand._rows_key([q[0], k[0], v[0]])
    try:
        w = _left((key, [q, k, v]))[key][0]
        assert expand.take_rows([k, q, v]) is None  # the order of the stacked rows
        assert expand.take_rows([q, k, v]) is w
        assert expand.take_rows([q, k, v]) is None  # once
        _left((key, [q, k, v]))
        expand.drop(q[0].device)
        assert expand.take_rows([q, k, v]) is None  # dropped
    finally:
        expand.drop(q[0].device)


def test_left_expansions_are_of_the_weights_as_they_are():
    """Not handed out for a weight written to since, a replaced QuantState, or rewritten scales."""
    def changed(write):
        packed, state = torch.zeros(8, dtype=torch.uint8), State()
        _left((packed.data_ptr(), [(packed, state)]))
        try:
            state = write(packed, state) or state
            return expand.take(packed, torch.float16, state)
        finally:
            expand.drop(packed.device)

    assert changed(lambda p, s: None) is not None
    assert changed(lambda p, s: (p.add_(1), None)[1]) is None
    assert changed(lambda p, s: State()) is None
    assert changed(lambda p, s: (s.absmax.add_(1), None)[1]) is None


def test_left_expansions_end_with_their_backward():
    """What a backward pass leaves is not handed out after it, nor in another one."""
    packed, state = torch.zeros(8, dtype=torch.uint8), State()
    seen = []

    class Leaves(torch.autograd.Function):
        @staticmethod
        def forward(ctx, x, leave):
            ctx.leave = leave
            return x * 1

        @staticmethod
        def backward(ctx, g):
            if ctx.leave:
                _left((packed.data_ptr(), [(packed, state)]))
            else:
                seen.append(expand.take(packed, torch.float16, state))
            return g, None

    x = torch.ones(1, requires_grad=True)
    try:
        Leaves.apply(Leaves.apply(x, False), True).backward()
        assert seen[0] is not None  # the same pass
        Leaves.apply(x, True).backward()
        assert expand.take(packed, torch.float16, state) is None  # after it
        Leaves.apply(x, False).backward()
        assert seen[1] is None  # another pass
    finally:
        expand.drop(packed.device)
