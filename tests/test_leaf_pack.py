"""The native evaluation's packed weights under another thread's rebuild (CPU:
the device call is replaced by the other thread's step).

One Prepared serves every thread that evaluates a model.  The native call runs
without the interpreter lock and reads the pack's memory until it returns."""

from __future__ import annotations

import gc
import weakref
from types import SimpleNamespace

import pytest
import torch

from mantisnet import PRODUCTION, MantisNet, forward, ops


@pytest.fixture()
def net():
    torch.manual_seed(3)
    return MantisNet(PRODUCTION).eval()


def _train_step(net):
    with torch.no_grad():
        net.mlp_v[0].weight.mul_(1.5)


@pytest.mark.parametrize("full", [True, False])
def test_a_rebuild_during_the_native_call_frees_nothing_it_reads(net, monkeypatch, full):
    W, pack_leaf, refs, alive = forward._prepared(net), forward._pack_leaf, [], []

    def pack(*args):
        out = pack_leaf(*args)
        refs.append([weakref.ref(x) for x in out[2]])
        return out

    def call(struct, *args):
        _train_step(net)  # the other thread's step, check and evaluation
        assert W.rebuild_if_changed()
        W.leaf()
        gc.collect()
        alive.extend(r() is not None for r in refs[0])
        return torch.zeros(1, 4)

    monkeypatch.setattr(forward, "_pack_leaf", pack)
    monkeypatch.setattr(ops, "leaf_forward", call)
    monkeypatch.setattr(forward, "_supported", lambda m: torch.device("cpu"))
    monkeypatch.setattr(forward, "_speculative", lambda m, b, evaluate, native: native(None, W))
    batch = SimpleNamespace(stone_own=torch.zeros(1))
    forward.forward(net, batch, 0.2) if full else forward.policy_q(net, batch)
    assert len(refs) == 2 and alive and all(alive)


def test_a_pack_of_replaced_operands_is_not_kept(net, monkeypatch):
    W, packed = forward._prepared(net), []

    def pack(cfg, t, params):
        if not packed:
            _train_step(net)  # the other thread's step and check, while this one packs
            assert W.rebuild_if_changed()
        packed.append(t)
        return None, None, []

    monkeypatch.setattr(forward, "_pack_leaf", pack)
    W.leaf()
    W.leaf()
    W.leaf()
    assert len(packed) == 2 and packed[-1] is W.t
