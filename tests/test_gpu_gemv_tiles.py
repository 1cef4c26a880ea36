"""The GEMV on activations in the packed tiles (csrc/gemv.hip
``gemv_tiles_kernel``): 17..64 rows (9..16 with more output blocks than CUs),
K > 4096, at most two output blocks per CU, where the library quantizes the rows itself.  Bit-equal to the general route,
the same int8 rows handed over row-major (``gemv_kernel``), at every count of
row tiles, one and two blocks per workgroup, ragged N, K of uneven wavefront
shares and off the 64-column grid, strided x, bias, int32 and both 16-bit
outputs, with and without the residual epilogue; and to the oracle."""
from __future__ import annotations

import sys

import numpy as np
import pytest
import torch

from oracle import w8a8_oracle as O

pytestmark = pytest.mark.gpu


def note(msg: str) -> None:
    sys.__stderr__.write(f"[gpu-case] {msg}\n")
    sys.__stderr__.flush()


def _case(m, n, k, dtype, dev, pad=0):
    from nanopointllm_amd import w8a8

    g = torch.Generator().manual_seed(m * 7 + n + k)
    x = torch.randn(m, k + pad, generator=g).to(dtype).to(dev)[:, :k]
    wq = torch.randint(-127, 128, (n, k), generator=g, dtype=torch.int8)
    sw = torch.from_numpy(O.scale_from_absmax(
        np.abs(np.random.default_rng(n).standard_normal(n)) * 0.05).astype(np.float32)).to(dev)
    bias = torch.randn(n, generator=g).to(dev)
    return x, wq, w8a8.pack_rows(wq.to(dev)), sw, bias


# (m, n, k): 9 (at 5120 outputs) and 64 are the rule's ends, 16/17, 32/33 and 48/49 those of the
# row tiles; 4096 outputs give one block per CU, 4100 and 5120 two, 8192 the most.
@pytest.mark.parametrize("m,n,k", [
    (9, 5120, 11008), (16, 4096, 11008), (16, 5120, 13824), (17, 4096, 4104), (32, 4100, 4160), (33, 8192, 4168),
    (48, 4096, 11008), (49, 5120, 6400), (64, 4096, 11008), (64, 40, 8200), (12, 8, 16384)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_tiles_match_row_major_route(cuda, m, n, k, dtype):
    from nanopointllm_amd import _lib, w8a8

    note(f"gemv_tiles m={m} n={n} k={k} {dtype}")
    x, _, wp, sw, bias = _case(m, n, k, dtype, cuda, pad=8)
    q, s = w8a8.quant_rows(x)
    s = s.reshape(-1)
    for b in (None, bias):
        got = w8a8.linear_dynamic(x, wp, sw, b, n)
        want = w8a8.linear_i8in(q, s, wp, sw, b, n, out_dtype=dtype)
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    got = w8a8.linear_dynamic(x, wp, sw, None, n, epilogue=_lib.EPI_I32)
    assert torch.equal(got, w8a8.gemm_i32(q, wp, n))
    res = torch.randn(m, n, generator=torch.Generator().manual_seed(m)).to(dtype).to(cuda)
    got = w8a8.linear_residual(x, wp, sw, bias, n, res)
    want = w8a8.linear_i8in_residual(q, s, wp, sw, bias, n, res)
    for a, b in zip(got, want):
        assert torch.equal(a.float(), b.float())


@pytest.mark.parametrize("m,n,k", [(16, 5120, 4200), (50, 300, 4352)])
def test_tiles_match_oracle(cuda, m, n, k):
    from nanopointllm_amd import w8a8

    note(f"gemv_tiles oracle m={m} n={n} k={k}")
    x, wq, wp, sw, _ = _case(m, n, k, torch.float16, cuda)
    y = w8a8.linear_dynamic(x, wp, sw, None, n).cpu().numpy()
    exp, _, _, _ = O.w8a8_linear_dynamic(x.float().cpu().numpy(), wq.numpy(), sw.cpu().numpy())
    np.testing.assert_array_equal(y, exp.astype(np.float16))
