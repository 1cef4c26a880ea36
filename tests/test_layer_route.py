"""Which of W8A8LlamaLayer.forward's two routes a call takes (no GPU: the
modules are stand-ins on the host).  Past 64 rows the residual adds go into
the epilogues of o_proj and down, which does not call o_proj, down or
``mlp.forward_residual_rmsnorm``; so whatever replaces or observes one of
these has to be called at every row count."""
from __future__ import annotations

import pytest
import torch
import torch.nn as nn

from nanopointllm_amd.linear import PackedW8A8Weight, W8A8Linear, W8A8MLP
from nanopointllm_amd.runner import W8A8LlamaLayer

HIDDEN = 16
CORE = 2.0


def _linear(n: int, k: int) -> W8A8Linear:
    return W8A8Linear(PackedW8A8Weight(torch.zeros(0, dtype=torch.int8), torch.zeros(n), None, n, k))


class _QKV(nn.Module):
    def project_rmsnorm(self, rows, norm):
        return rows, rows, rows


def _layer(mlp_type=W8A8MLP) -> W8A8LlamaLayer:
    layer = W8A8LlamaLayer.__new__(W8A8LlamaLayer)
    nn.Module.__init__(layer)
    layer.layer_index = 0
    layer.input_layernorm = layer.post_attention_layernorm = nn.Identity()
    layer.qkv, layer.o_proj = _QKV(), _linear(HIDDEN, HIDDEN)
    layer.mlp = mlp_type.__new__(mlp_type)
    nn.Module.__init__(layer.mlp)
    layer.mlp.down, layer.mlp.h_scale = _linear(HIDDEN, 32), None
    layer.attention_core = lambda q, k, v, i, state: q * CORE
    return layer


def _x(rows: int, dtype=torch.float16) -> torch.Tensor:
    return torch.ones(rows, HIDDEN, dtype=dtype)


def _epilogues(layer, rows, dtype=torch.float16) -> bool:
    return layer._adds_in_epilogues(_x(rows, dtype), _x(rows, dtype))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_plain_modules(dtype):
    layer = _layer()
    assert [_epilogues(layer, m, dtype) for m in (1, 64, 65, 200)] == [False, False, True, True]
    assert not _epilogues(layer, 200, torch.float32)
    assert not layer._adds_in_epilogues(_x(200, torch.float32), _x(200))


@pytest.mark.parametrize("which", ["o_proj", "down"])
def test_hooks_and_other_activations(which):
    layer = _layer()
    mod = layer.o_proj if which == "o_proj" else layer.mlp.down
    for register in (mod.register_forward_hook, mod.register_forward_pre_hook):
        handle = register(lambda *a: None)
        assert not _epilogues(layer, 200)
        handle.remove()
    handle = nn.modules.module.register_module_forward_hook(lambda *a: None)
    assert not _epilogues(layer, 200)
    handle.remove()
    assert _epilogues(layer, 200)
    mod.static_scale = torch.ones(1)
    assert not _epilogues(layer, 200)


class _OwnMLP(W8A8MLP):
    def forward_residual_rmsnorm(self, hidden_states, residual, norm):
        self.seen = hidden_states.shape[0]
        return hidden_states + residual, hidden_states


@pytest.mark.parametrize("rows", [64, 65, 200])
def test_own_methods_are_called_at_every_row_count(rows):
    layer = _layer(_OwnMLP)
    seen = []
    layer.o_proj.forward = lambda x: seen.append(x.shape[0]) or x + 1
    out = layer(_x(rows))
    assert layer.mlp.seen == rows and seen == [rows]
    # context 2, o_proj 3, residual 1 + 3, mlp 3
    assert torch.equal(out, torch.full_like(out, 7.0))


@pytest.mark.parametrize("name", ["forward", "forward_i8"])
def test_down_replaced_on_the_instance(name):
    layer = _layer()
    setattr(layer.mlp.down, name, lambda *a, **k: None)
    assert not _epilogues(layer, 200)
    layer = _layer()
    layer.mlp.forward_residual_rmsnorm = lambda *a: None
    assert not _epilogues(layer, 200)


def test_other_modules_need_no_w8a8_attributes():
    layer = _layer()
    layer.o_proj = nn.Identity()
    assert not _epilogues(layer, 200)
    layer = _layer()
    layer.mlp.down = nn.Identity()
    assert not _epilogues(layer, 200)
