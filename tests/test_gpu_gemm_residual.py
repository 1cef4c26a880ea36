"""The residual add in the GEMM's own epilogue (``w8a8_linear_residual`` /
``w8a8_linear_i8in_residual`` past 64 rows without the RMSNorm chunk sums) and
the decoder layer that uses it.  Bit-equal to the plain linear followed by
torch's 16-bit add (one rounding of the sum): pipelined and ring tiles,
one-pass and several-pass staging, ragged N, and residual rows that are
strided or off the 16-byte grid."""
from __future__ import annotations

import sys

import pytest
import torch
import torch.nn as nn

pytestmark = pytest.mark.gpu


def note(msg: str) -> None:
    sys.__stderr__.write(f"[gpu-case] {msg}\n")
    sys.__stderr__.flush()


# ring mid / small / t112x96 / w256sq (K < 1024), then pipelined tiles
@pytest.mark.parametrize("m,n,k", [
    (65, 1000, 520), (300, 3001, 520), (560, 4096, 520), (2040, 16380, 136), (200, 12288, 1040),
    (300, 12295, 1040), (2048, 4096, 1100), (520, 12000, 1040), (1024, 22016, 1024), (201, 4100, 1040), (350, 4096, 1100)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_residual_in_gemm_epilogue(cuda, m, n, k, dtype):
    from nanopointllm_amd import w8a8
    from nanopointllm_amd.linear import PackedW8A8Weight

    note(f"gemm residual m={m} n={n} k={k} {dtype}")
    g = torch.Generator(device=cuda).manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g, device=cuda).to(dtype)
    p = PackedW8A8Weight.from_float((torch.randn(n, k, generator=g, device=cuda) * 0.02).to(dtype))
    wide = torch.randn(m, n + 9, generator=g, device=cuda).to(dtype)
    plain = w8a8.linear_dynamic(x, p.packed, p.scale, None, n)
    q, s = w8a8.quant_rows(x)
    for res in (wide[:, :n].contiguous(), wide[:, :n], wide[:, 1:n + 1]):
        want = (plain + res).view(torch.int16)
        got = w8a8.linear_residual(x, p.packed, p.scale, None, n, res, ss_parts=False)
        assert got.ss_parts is None and torch.equal(got.y.view(torch.int16), want)
        got = w8a8.linear_i8in_residual(q, s.reshape(-1), p.packed, p.scale, None, n, res,
                                        ss_parts=False)
        assert torch.equal(got.y.view(torch.int16), want)


@pytest.mark.parametrize("rows", [64, 65, 200])
def test_layer_bits_do_not_depend_on_the_route(cuda, rows):
    """A forward hook on o_proj sees its call, and the layer takes the route
    that makes it; without one the adds run in the epilogues."""
    from nanopointllm_amd.runner import W8A8LlamaRunner

    h, inter = 256, 704
    g = torch.Generator(device=cuda).manual_seed(rows)

    def linear(n, k):
        mod = nn.Linear(k, n, bias=False, device="meta")
        mod.weight = nn.Parameter((torch.randn(n, k, generator=g, device=cuda) * 0.05).half(),
                                  requires_grad=False)
        return mod

    class Norm(nn.Module):
        def __init__(self):
            super().__init__()
            self.weight = nn.Parameter(torch.ones(h, device=cuda).half(), requires_grad=False)
            self.variance_epsilon = 1e-6

    layer = nn.Module()
    layer.input_layernorm, layer.post_attention_layernorm = Norm(), Norm()
    layer.self_attn, layer.mlp = nn.Module(), nn.Module()
    layer.self_attn.num_heads = layer.self_attn.num_key_value_heads = 2
    layer.self_attn.head_dim = 128
    for name in ("q_proj", "k_proj", "v_proj", "o_proj"):
        setattr(layer.self_attn, name, linear(h, h))
    for name, n, k in (("gate_proj", inter, h), ("up_proj", inter, h), ("down_proj", h, inter)):
        setattr(layer.mlp, name, linear(n, k))
    model = nn.Module()
    model.model = nn.Module()
    model.model.embed_tokens, model.model.norm = nn.Embedding(1, 1), Norm()
    model.model.layers = nn.ModuleList([layer])
    model.lm_head = linear(32, h)
    runner = W8A8LlamaRunner(model, lambda q, k, v, i, state: q.reshape(q.shape[0], -1))
    mod = runner.layers[0]
    x = torch.randn(rows, h, generator=g, device=cuda).half()
    route = lambda: mod._adds_in_epilogues(x, x)  # noqa: E731
    assert route() == (rows > 64)
    out = mod(x)
    seen = []
    handle = mod.o_proj.register_forward_hook(lambda m, a, y: seen.append(tuple(y.shape)))
    assert not route()
    hooked = mod(x)
    handle.remove()
    assert seen == [(rows, h)]
    assert torch.equal(out.view(torch.int16), hooked.view(torch.int16))
