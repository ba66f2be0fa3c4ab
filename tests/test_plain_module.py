"""Which modules a fused call may stand in for: none whose own call would do anything else."""

import pytest
import torch
from torch import nn

from atma_amd.kernel.train_glue import plain_module
from atma_amd.layers.global_attention import Linear


def test_plain():
    assert plain_module(Linear(8, 8), Linear)


class Sub(Linear):
    pass


def _own_forward(m):
    m.forward = lambda x: x


def _parametrised(m):
    nn.utils.parametrize.register_parametrization(m, "weight", nn.Identity())


@pytest.mark.parametrize("change", [
    lambda m: m.register_forward_hook(lambda *a: None), lambda m: m.register_forward_pre_hook(lambda *a: None),
    lambda m: m.register_full_backward_hook(lambda *a: None), lambda m: m.register_full_backward_pre_hook(lambda *a: None),
    _own_forward, _parametrised])
def test_changed_module_is_not_plain(change):
    m = Linear(8, 8)
    change(m)
    assert not plain_module(m, Linear)
    assert not plain_module(Sub(8, 8), Linear) and not plain_module(nn.Linear(8, 8), Linear)


@pytest.mark.parametrize("register", ["register_module_forward_hook", "register_module_forward_pre_hook",
                                      "register_module_full_backward_hook", "register_module_full_backward_pre_hook"])
def test_a_hook_on_every_module(register):
    m = Linear(8, 8)
    handle = getattr(nn.modules.module, register)(lambda *a: None)
    try:
        assert not plain_module(m, Linear)
    finally:
        handle.remove()
    assert plain_module(m, Linear)
