"""Mixers side by side whose branches are not the ones that start and end together: they run by the plain contract."""
import pytest
import torch

from atoma_infer_amd.parts import GatedDeltaRule, TiedValueAttention
from atoma_infer_amd.parts.parallel import ParallelMixer


class OwnAttention(TiedValueAttention):
    def forward(self, x, ctx, cache, sink=None):
        return x + 1


class OwnRecurrence(GatedDeltaRule):
    def forward(self, x, ctx, cache):
        return 2 * x


class Plain:
    """Not a part at all, only what a branch needs."""
    def cache_spec(self):
        return None

    def state_spec(self):
        return None

    def forward(self, x, ctx, cache):
        return x - 1


def attention(cls):
    part = cls(32, 2, 1, 16, 1.0, 1e-6, 1e4, 16)
    part.w_qk = torch.ones(48, 32)
    return part


def recurrence(cls):
    part = cls(32, 2, 1, 16, 16, 4, 1e-6)
    part.w_in = torch.ones(64, 32)
    return part


def _run(branches):
    x = torch.arange(96.0).view(3, 32)
    return x, [t for t, _ in ParallelMixer(branches, [0.5, 0.5], ["a", "b"]).forward(x, None, None).terms]


def test_branches_with_a_forward_of_their_own_keep_the_plain_contract():
    x, outs = _run([attention(OwnAttention), recurrence(OwnRecurrence)])
    assert torch.equal(outs[0], x + 1) and torch.equal(outs[1], 2 * x)


def test_a_branch_that_is_no_mixer_keeps_the_plain_contract():
    x, outs = _run([Plain(), recurrence(OwnRecurrence)])
    assert torch.equal(outs[0], x - 1) and torch.equal(outs[1], 2 * x)


def test_a_forward_put_in_the_place_of_one_instance_keeps_the_plain_contract(monkeypatch):
    a, b = attention(TiedValueAttention), recurrence(GatedDeltaRule)
    assert a.first_weight() is a.w_qk and b.first_weight() is b.w_in
    monkeypatch.setattr(a, "forward", lambda x, ctx, cache: x + 1)
    monkeypatch.setattr(b, "forward", lambda x, ctx, cache: 2 * x)
    x, outs = _run([a, b])
    assert torch.equal(outs[0], x + 1) and torch.equal(outs[1], 2 * x)
