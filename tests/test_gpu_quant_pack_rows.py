"""Weight quantization straight into the packed tiles (``w8a8_quant_pack_rows``)
against the two-kernel path (``w8a8_quant_rows`` + ``w8a8_pack_rows``), bit for
bit, padding bytes included: every register variant and its edges, ragged rows
and columns, one to three matrices, both row layouts, unaligned and strided
rows, and non-finite weights.  The packed gate/up and QKV modules equal the
packing of their concatenated weights (llama/lightweight_runner.py:81-92,
llama/paged_attention.py:1242-1262).
"""
from __future__ import annotations

import ctypes
import sys

import pytest
import torch
import torch.nn as nn

from nanopointllm_amd import _lib

DTYPES = (torch.float16, torch.bfloat16, torch.float32)


def note(msg: str) -> None:
    sys.__stderr__.write(f"[gpu-case] {msg}\n")
    sys.__stderr__.flush()


def weight(n, k, dtype, seed, device):
    w = torch.randn(n, k, generator=torch.Generator().manual_seed(seed)) * 0.05
    w[:, :: 29] *= 8.0
    w[n // 2] = 0.0
    return w.to(dtype).to(device)


def two_kernels(w, layout):
    from nanopointllm_amd import w8a8

    q, s = w8a8.quant_rows(w)
    if layout == _lib.ROWS_INTERLEAVE_HALVES:
        s = torch.stack(s.chunk(2), dim=1).reshape(-1)
    return w8a8.pack_rows(q, layout), s


@pytest.mark.gpu
@pytest.mark.parametrize("k", [1, 7, 64, 100, 520, 2048, 2056, 4096, 4104, 8192, 8200, 11264, 11272,
                               13824])
@pytest.mark.parametrize("n", [1, 16, 34])
@pytest.mark.parametrize("dtype", DTYPES, ids=str)
def test_equals_quantize_then_pack(cuda, n, k, dtype):
    from nanopointllm_amd import w8a8

    note(f"quant_pack {n}x{k} {dtype}")
    w = weight(n, k, dtype, n + k, cuda)
    for layout in (_lib.ROWS_AS_IS, _lib.ROWS_INTERLEAVE_HALVES):
        if layout and n % 2:
            continue
        want, ws = two_kernels(w, layout)
        parts = [[w]]
        if n > 2:
            parts.append([w[: n // 2], w[n // 2:]])
            if not layout:
                parts.append([w[:1], w[1: n - 3], w[n - 3:]])
        for p in parts:
            got, s = w8a8.quant_pack_rows(p, layout)
            assert torch.equal(got, want) and torch.equal(s, ws)


# Rows read twice: odd and even numbers of 512-column chunks around the groups
# of four and the passes of two, a partial last tile, unaligned rows.
@pytest.mark.gpu
@pytest.mark.parametrize("k", [11776, 12288, 12296, 13312, 14336, 14400, 20000, 13825, 14335])
@pytest.mark.parametrize("dtype", DTYPES, ids=str)
def test_long_rows_equal_quantize_then_pack(cuda, k, dtype):
    from nanopointllm_amd import w8a8

    note(f"quant_pack long rows k={k} {dtype}")
    w = weight(50, k, dtype, k, cuda)
    w[:, k - 1] = 3.0   # the last column holds the scales
    for layout in (_lib.ROWS_AS_IS, _lib.ROWS_INTERLEAVE_HALVES):
        want, ws = two_kernels(w, layout)
        for parts in ([w], [w[:25], w[25:]]):
            got, s = w8a8.quant_pack_rows(parts, layout)
            assert torch.equal(got, want) and torch.equal(s, ws)


@pytest.mark.gpu
@pytest.mark.parametrize("n,k,dtype,parts,one", [
    (2048, 11264, torch.float16, 1, True), (2048, 11272, torch.bfloat16, 1, False),
    (2048, 11272, torch.bfloat16, 2, True), (1040, 16384, torch.float16, 1, False),
    (1040, 16392, torch.float16, 1, True), (1024, 16392, torch.float16, 1, False),
    (1024, 16392, torch.float16, 2, False), (64, 4096, torch.float32, 1, True),
    (2048, 4104, torch.float32, 1, False), (2048, 4104, torch.float32, 2, True),
    (2, 1 << 28, torch.bfloat16, 1, False)])
def test_one_kernel_or_two(cuda, monkeypatch, n, k, dtype, parts, one):
    """The rule that keeps quantizing and packing apart, at its edges, and at a
    width that the one kernel refuses; the same bytes either way."""
    from nanopointllm_amd import w8a8
    from nanopointllm_amd.linear import PackedW8A8Weight

    note(f"quant_pack route {n}x{k} {dtype} in {parts}")
    calls = []
    kernel = w8a8.quant_pack_rows
    monkeypatch.setattr(w8a8, "quant_pack_rows", lambda *a: calls.append(1) or kernel(*a))
    w = torch.empty((n, k), dtype=dtype, device=cuda)
    w.normal_(generator=torch.Generator(device=cuda).manual_seed(k))
    got = PackedW8A8Weight.from_parts(list(w.chunk(parts)))
    assert bool(calls) == one
    want, s = two_kernels(w, _lib.ROWS_AS_IS)
    assert torch.equal(got.packed, want) and torch.equal(got.scale, s)


@pytest.mark.gpu
def test_strided_unaligned_and_non_finite_rows(cuda):
    from nanopointllm_amd import w8a8

    big = weight(40, 1200, torch.float16, 5, cuda)
    big[3, 40], big[5, 41], big[7, 42] = float("inf"), float("-inf"), float("nan")
    note("quant_pack views")
    for view in (big[:, 8:1008], big[:, 3:1003], big[::2, :1000], big.t()):
        want, ws = two_kernels(view.contiguous(), _lib.ROWS_AS_IS)
        got, s = w8a8.quant_pack_rows([view])
        assert torch.equal(got, want) and torch.equal(s, ws)


@pytest.mark.gpu
@pytest.mark.parametrize("bias", [False, True])
def test_modules_equal_the_concatenated_weight(cuda, bias):
    from nanopointllm_amd.linear import PackedW8A8Weight, W8A8GateUpSiluMul, W8A8PackedQKV

    def linear(n, k, seed, dtype=torch.float16):
        mod = nn.Linear(k, n, bias=bias, device=cuda, dtype=dtype)
        mod.weight.data.copy_(weight(n, k, dtype, seed, cuda))
        return mod

    def same(a, b):
        assert torch.equal(a.packed, b.packed) and torch.equal(a.scale, b.scale)
        assert (a.bias is None and b.bias is None) or torch.equal(a.bias, b.bias)
        assert (a.out_features, a.in_features, a.layout) == (b.out_features, b.in_features, b.layout)

    def cat_path(mods, layout):
        w = torch.cat([m.weight.detach() for m in mods])
        b = torch.cat([m.bias.detach() for m in mods]) if bias else None
        q, s = two_rows(w)
        return PackedW8A8Weight.from_int8(q, s, b, layout=layout)

    def two_rows(w):
        from nanopointllm_amd import w8a8

        return w8a8.quant_rows(w)

    note(f"quant_pack modules bias={bias}")
    g, u = linear(40, 96, 1), linear(40, 96, 2)
    same(W8A8GateUpSiluMul(g, u).weight_q, cat_path([g, u], _lib.ROWS_INTERLEAVE_HALVES))
    q, k, v = linear(64, 96, 3), linear(32, 96, 4), linear(32, 96, 5)
    qkv = W8A8PackedQKV(q, k, v, num_heads=2, num_kv_heads=1, head_dim=32)
    same(qkv.linear.weight_q, cat_path([q, k, v], _lib.ROWS_AS_IS))
    # Mixed types concatenate (and promote) first.
    mixed = W8A8GateUpSiluMul(g, linear(40, 96, 6, torch.float32)).weight_q
    assert mixed.out_features == 80


def test_bad_arguments_are_refused_without_a_launch():
    lib = _lib.load()
    fake = ctypes.c_void_p(0x1000)

    def call(rows, lds, dtype=_lib.F16, k=64, layout=0, ptr=0x1000, packed=fake, scales=fake):
        n = len(rows)
        return lib.w8a8_quant_pack_rows(
            (ctypes.c_void_p * n)(*[ptr] * n), (ctypes.c_int64 * n)(*rows),
            (ctypes.c_int64 * n)(*lds), n, dtype, k, layout, packed, scales, None)

    assert call([16] * 4, [64] * 4) == _lib.ERR_SHAPE
    assert call([-1], [64]) == _lib.ERR_SHAPE
    assert call([16], [63]) == _lib.ERR_SHAPE
    assert call([16], [64], dtype=_lib.I8) == _lib.ERR_DTYPE
    assert call([16], [64], layout=2) == _lib.ERR_DTYPE
    assert call([15], [64], layout=1) == _lib.ERR_SHAPE
    assert call([16, 18], [64, 64], layout=1) == _lib.ERR_SHAPE
    assert call([16], [64], ptr=0x1001) == _lib.ERR_ALIGN
    assert call([16], [64], packed=ctypes.c_void_p(0x1008)) == _lib.ERR_ALIGN
    assert call([16], [64], scales=None) == _lib.ERR_NULL
    assert call([0], [64]) == _lib.OK
