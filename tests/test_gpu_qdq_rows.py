"""The one-pass quantize-dequantize kernels (``w8a8_qdq_rows``) behind
``dynamic_per_token_activation_qdq``, ``per_output_weight_qdq`` and
``groupwise_weight_qdq`` (nanopointllm/compression/w8a8.py:53-115).

Bars: int8 values, scales and dequantized values bit-exact against the oracle
over lane-group sizes, odd groups, ragged last groups, rows past the register
variants and unaligned or strided rows; non-finite rows equal the separate
quantization kernel followed by torch's product.
"""
from __future__ import annotations

import sys

import numpy as np
import pytest
import torch

from oracle import w8a8_oracle as O

pytestmark = pytest.mark.gpu

DTYPES = (torch.float16, torch.bfloat16, torch.float32)


def note(msg: str) -> None:
    sys.__stderr__.write(f"[gpu-case] {msg}\n")
    sys.__stderr__.flush()


def rows(n, k, dtype, seed):
    x = torch.randn(n, k, generator=torch.Generator().manual_seed(seed)) * 0.3
    x[:, ::37] *= 20.0
    x[n // 2] = 0.0
    return x.to(dtype)


def rounded(values, dtype):
    return torch.from_numpy(np.ascontiguousarray(values)).to(dtype)


@pytest.mark.parametrize("k", [8, 264, 1000, 4104])
@pytest.mark.parametrize("group", [4, 8, 16, 32, 64, 128, 256, 512, 96, 100, 2000])
@pytest.mark.parametrize("dtype", DTYPES, ids=str)
def test_groups_exact(cuda, k, group, dtype):
    from nanopointllm_amd import w8a8

    w = rows(5, k, dtype, seed=k + group)
    note(f"qdq groups k={k} g={group} {dtype}")
    deq, q, s = w8a8.groupwise_weight_qdq(w.to(cuda), group_size=group)
    edeq, eq, es = O.groupwise_weight_qdq(w.float().numpy(), group_size=group)
    np.testing.assert_array_equal(q.cpu().numpy(), eq)
    np.testing.assert_array_equal(s.cpu().numpy(), es)
    assert torch.equal(deq.cpu(), rounded(edeq, dtype))


@pytest.mark.parametrize("m,k", [(1, 1), (3, 7), (2, 513), (560, 4096), (5, 11008), (2100, 2056),
                                 (2, 16392), (3, 33000)])
@pytest.mark.parametrize("dtype", DTYPES, ids=str)
def test_rows_exact(cuda, m, k, dtype):
    from nanopointllm_amd import w8a8

    x = rows(m, k, dtype, seed=m + k)
    note(f"qdq rows {m}x{k} {dtype}")
    edeq, eq, es = O.groupwise_weight_qdq(x.float().numpy(), group_size=k)
    deq, q, s = w8a8.per_output_weight_qdq(x.to(cuda))
    np.testing.assert_array_equal(q.cpu().numpy(), eq)
    np.testing.assert_array_equal(s.cpu().numpy(), es[:, 0])
    assert torch.equal(deq.cpu(), rounded(edeq, dtype))
    deq, s = w8a8.dynamic_per_token_activation_qdq(x.to(cuda))
    np.testing.assert_array_equal(s.cpu().numpy(), es)
    assert torch.equal(deq.cpu(), rounded(edeq, dtype))


# Per workgroup size (256, 512, 1024 threads): the last columns that stay in
# registers, the first that are read twice, one whole round of four chunks a
# thread and the columns behind it, aligned and not.
@pytest.mark.parametrize("m,k", [(2049, 16384), (2049, 16392), (2049, 16391), (513, 32768),
                                 (513, 32776), (515, 32769), (512, 32776), (1, 65536), (2, 65544),
                                 (1, 65543), (2, 98304), (1, 98312), (1, 131071), (3, 300001)])
@pytest.mark.parametrize("dtype", DTYPES, ids=str)
def test_long_rows_equal_the_separate_kernels(cuda, m, k, dtype):
    from nanopointllm_amd import w8a8

    note(f"qdq long rows {m}x{k} {dtype}")
    g = torch.Generator(device=cuda).manual_seed(m + k)
    x = torch.empty((m, k), device=cuda, dtype=dtype).normal_(generator=g)
    x[:, k - 1] = 9.0   # the last column holds the scale
    q, s = w8a8.quant_rows(x)
    deq, q2, s2 = w8a8.per_output_weight_qdq(x)
    assert torch.equal(q2, q) and torch.equal(s2, s)
    assert torch.equal(deq, (q.float() * s[:, None]).to(dtype))


@pytest.mark.parametrize("group", [64, 96, 4096])
def test_strided_and_unaligned_rows(cuda, group):
    from nanopointllm_amd import w8a8

    big = rows(9, 1100, torch.float16, seed=3).to(cuda)
    note(f"qdq views g={group}")
    for view in (big[:, 3:1003], big[:, 8:1008], big[::2, 16:1016], big.t(), big[:1].expand(4, -1)):
        want = w8a8.groupwise_weight_qdq(view.contiguous().clone(), group_size=group)
        for a, b in zip(w8a8.groupwise_weight_qdq(view, group_size=group), want):
            assert torch.equal(a, b)
    x = rows(6, 40, torch.float16, seed=4).reshape(2, 3, 40).to(cuda)
    deq, s = w8a8.dynamic_per_token_activation_qdq(x, axis=1)
    want, ws = w8a8.dynamic_per_token_activation_qdq(x.movedim(1, -1).contiguous())
    assert torch.equal(deq, want.movedim(-1, 1)) and torch.equal(s, ws.movedim(-1, 1))


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
def test_non_finite_rows_equal_the_separate_kernels(cuda, dtype):
    from nanopointllm_amd import w8a8

    x = rows(6, 520, dtype, seed=9)
    x[0, 5], x[1, 7], x[2, 9] = float("inf"), float("-inf"), float("nan")
    x[3, :] = float("nan")
    x[4, 3] = torch.finfo(dtype).max
    note(f"qdq non-finite {dtype}")
    q, s = w8a8.quant_rows(x.to(cuda))
    want = (q.float() * s[:, None]).to(dtype)
    deq, q2, s2 = w8a8.per_output_weight_qdq(x.to(cuda))
    assert torch.equal(q2, q) and torch.equal(s2, s)
    torch.testing.assert_close(deq, want, rtol=0, atol=0, equal_nan=True)


def test_other_weight_types_go_through_binary32(cuda):
    from nanopointllm_amd import w8a8

    w = rows(7, 200, torch.float32, seed=1)
    note("qdq float64 weight")
    deq, q, s = w8a8.groupwise_weight_qdq(w.double().to(cuda), group_size=64)
    want = w8a8.groupwise_weight_qdq(w.to(cuda), group_size=64)
    assert deq.dtype == torch.float64 and torch.equal(deq, want[0].double())
    assert torch.equal(q, want[1]) and torch.equal(s, want[2])


def test_rows_past_32_bit_columns(cuda):
    """One row of 2^31 + 8 columns against the same columns of a short row with
    the same scale: the first ones, those around byte 2^31, and the last, past
    element 2^31 and byte 2^32."""
    from nanopointllm_amd import w8a8

    k, n = (1 << 31) + 8, 4096
    note(f"qdq one row of {k}")
    x = torch.empty((1, k), dtype=torch.bfloat16, device=cuda)
    x.copy_(torch.arange(8191, device=cuda).sub_(4095).to(torch.bfloat16)
            .repeat(k // 8191 + 1)[None, :k])
    x[0, 5] = 6000.0  # the row's largest, in the first slice
    for group in (None, 128):
        if group is None:
            deq, s = w8a8.dynamic_per_token_activation_qdq(x)
        else:
            deq, q, s = w8a8.groupwise_weight_qdq(x, group_size=group)
        for start, end in ((0, n), ((1 << 30) - n // 2, (1 << 30) + n // 2), (k - n - 8, k)):
            part = x[:, start:end].clone()
            if group is None:
                part = torch.cat([part, x[:, 5:6]], dim=1)
                want, ws = w8a8.dynamic_per_token_activation_qdq(part)
                assert torch.equal(s, ws)
            else:
                want, wq, ws = w8a8.groupwise_weight_qdq(part, group_size=group)
                assert torch.equal(q[:, start:end], wq)
                assert torch.equal(s[:, start // group:-(-end // group)], ws)
            assert torch.equal(deq[:, start:end], want[:, :end - start])
        del deq
    assert s.shape == (1, k // 128 + 1)
