"""The pipelined GEMM tiles (csrc/gemm_pipe.hip ``gemm_pipe_kernel``), one
shape per tile that the library's own rule gives to it: ragged in M and N
(partial tiles, a partial last 16-row block), K with a partial last k-block,
and every remainder of each tile's unrolled loop (six k-blocks for the 352-wide
tiles, two for the others).  int32 products exact, the float epilogues bit-equal
to the oracle's, the integer ones exact; and the rule itself (no GPU)."""
from __future__ import annotations

import sys

import numpy as np
import pytest
import torch

from gemm_tiles import launched_tile
from oracle import w8a8_oracle as O

SHAPES = [(66, 4886, 1030, "64x64"), (65, 9858, 1100, "128x64"), (129, 8230, 1160, "128x96"),
          (130, 12400, 1250, "128x128"), (257, 12390, 1100, "192x160"),
          (195, 20588, 1160, "256x128"), (260, 21950, 1250, "256x192"),
          (515, 16350, 1030, "192x288"), (580, 18510, 1100, "256x256"),
          (577, 21800, 1160, "192x352"), (580, 22570, 1250, "256x352")]
# 16 to 21 k-blocks: what the unrolled loop of six leaves is 4, 5, 0, 1, 2, 3.
SIX_KS = (1000, 1030, 1100, 1160, 1250, 1340)
# Every remainder of each tile's unrolled loop.
REMAINDERS = [(m, n, k, t) for m, n, _, t in SHAPES
              for k in (SIX_KS if t in ("192x352", "256x352") else (1030, 1100))]
# One shape per tile of the ring kernels, at a K that leaves it to them.
RING = [(100, 1000, 900, "tiny-deep"), (300, 6000, 900, "small-deep"), (760, 4096, 900, "big-deep"),
        (567, 12288, 300, "big"), (128, 4096, 900, "mid"), (560, 12288, 300, "wd7x2"),
        (560, 4096, 900, "t112x96"), (640, 4096, 900, "t128x96")]


def note(msg: str) -> None:
    sys.__stderr__.write(f"[gpu-case] {msg}\n")
    sys.__stderr__.flush()


def pipe_config(m, n, k, cus=256):
    from nanopointllm_amd import _lib

    code = _lib.load().w8a8_gemm_pipe_config(m, n, k, cus)
    return None if code < 0 else _lib.GEMM_PIPE_NAMES[code]


@pytest.mark.parametrize("m,n,k,tile", [(m, n, k, t) for m, n, k, t in SHAPES] + [
    (560, 12288, 4096, "192x160"), (560, 22016, 4096, "192x288"), (560, 4096, 11008, "128x96"), (1024, 4096, 11008, "128x128"),
    (1024, 22016, 4096, "256x352"), (2048, 4096, 4096, "256x128"), (2048, 12288, 4096, "256x192"),
    (201, 12288, 4096, "128x96"), (201, 4096, 4096, "64x64"), (448, 4096, 4096, "128x64"),
    (768, 22016, 4096, "192x352"), (100, 4096, 11008, None), (64, 22016, 8192, None), (2048, 12288, 960, None),
    # fewer than 16 k-blocks of 64 stay on the ring tiles
    (560, 4096, 960, None), (560, 4096, 961, "128x96"), (560, 4096, 1023, "128x96"),
    (500, 12000, 1000, "192x160"),
    (0, 4096, 4096, None), (560, 4096, 0, None)])
def test_rule(m, n, k, tile):
    assert pipe_config(m, n, k) == tile


def _case(m, n, k, dev):
    g = torch.Generator().manual_seed(m + n + k)
    xq = torch.randint(-127, 128, (m, k), generator=g, dtype=torch.int8).to(dev)
    wq = torch.randint(-127, 128, (n, k), generator=g, dtype=torch.int8).to(dev)
    rng = np.random.default_rng(m + n)
    sx = O.scale_from_absmax(np.abs(rng.standard_normal((m, 1))) * 3).astype(np.float32)
    sw = O.scale_from_absmax(np.abs(rng.standard_normal(n)) * 0.05).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    acc = torch.matmul(xq.double(), wq.double().T).to(torch.int32).cpu().numpy()
    return xq, wq, acc, sx, sw, bias


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,tile", SHAPES + RING)
def test_tile_int32_and_dequant(cuda, m, n, k, tile):
    from nanopointllm_amd import w8a8

    assert launched_tile(m, n, k) == (tile if k <= 960 else f"pipe-{tile}")
    note(f"gemm {tile} m={m} n={n} k={k}")
    xq, wq, eacc, sx, sw, bias = _case(m, n, k, cuda)
    wp = w8a8.pack_rows(wq)
    np.testing.assert_array_equal(w8a8.gemm_i32(xq, wp, n).cpu().numpy(), eacc)
    sxt, swt, bt = (torch.from_numpy(a).to(cuda) for a in (sx, sw, bias))
    for dt, b in ((torch.float16, bt), (torch.bfloat16, None), (torch.float32, bt)):
        y = w8a8.linear_i8in(xq, sxt, wp, swt, b, n, out_dtype=dt)
        exp = torch.from_numpy(O.dequant_epilogue(eacc, sx, sw, None if b is None else bias))
        np.testing.assert_array_equal(y.float().cpu().numpy(), exp.to(dt).float().numpy(),
                                      err_msg=str(dt))


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,tile", REMAINDERS)
def test_every_remainder_of_the_unrolled_loop(cuda, m, n, k, tile):
    from nanopointllm_amd import w8a8

    assert pipe_config(m, n, k) == tile
    note(f"gemm pipe remainder {tile} m={m} n={n} k={k}")
    g = torch.Generator(device=cuda).manual_seed(k)
    xq = torch.randint(-127, 128, (m, k), generator=g, dtype=torch.int8, device=cuda)
    wq = torch.randint(-127, 128, (n, k), generator=g, dtype=torch.int8, device=cuda)
    want = torch.matmul(xq.double(), wq.double().T).to(torch.int32)
    assert torch.equal(w8a8.gemm_i32(xq, w8a8.pack_rows(wq), n), want)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,tile", SHAPES)
def test_pipe_tile_silu_and_integer_epilogues(cuda, m, n, k, tile):
    from nanopointllm_amd import _lib, integer_epilogues as E, w8a8

    note(f"gemm pipe epilogues {tile} m={m} n={n} k={k}")
    xq, wq, eacc, sx, sw, _ = _case(m, n, k, cuda)
    wp = w8a8.pack_rows(wq)   # the rows as they are: gate, up, gate, up, ...
    sxt, swt = torch.from_numpy(sx).to(cuda), torch.from_numpy(sw).to(cuda)
    h = w8a8.linear_i8in(xq, sxt, wp, swt, None, n, epilogue=_lib.EPI_SILU_MUL,
                         out_dtype=torch.float16)
    eh = O.gateup_silu_mul_from_acc(eacc, sx, sw, layout="interleave")
    got, want = h.cpu().numpy(), eh.astype(np.float16)
    # A binary32 SiLU may round to the other neighbour of a binary16 tie, and
    # the product then moves by as much: two steps.
    step = np.abs(np.spacing(want.astype(np.float16))).astype(np.float64)
    assert np.all(np.abs(got.astype(np.float64) - want.astype(np.float64)) <= 2 * step)
    assert np.mean(got != want) < 1e-3
    h_scale = float(O.static_activation_scale(float(h.float().abs().max().item())))
    hq = w8a8.linear_i8in(xq, sxt, wp, swt, None, n, epilogue=_lib.EPI_SILU_MUL_Q8,
                          out_dtype=torch.int8, y_scale=h_scale)
    eq = O.quantize_symmetric(got.astype(np.float32), np.float32(h_scale))
    np.testing.assert_array_equal(hq.cpu().numpy(), eq)
    comp = [O.compile_fp16_requant_scale(0.02, float(w), 0.5) for w in sw]
    mult = torch.from_numpy(np.array([c[0] for c in comp], np.uint32).view(np.int32)).to(cuda)
    shift = torch.from_numpy(np.array([c[1] for c in comp], np.int32)).to(cuda)
    bias = torch.randint(-3000, 3000, (n,), dtype=torch.int32).to(cuda)
    y = E.linear_i8in_requant(xq, wp, mult, shift, bias, n)
    ref = E.requantize_int32(torch.from_numpy(eacc).to(cuda), bias, mult, shift)
    assert torch.equal(y, ref)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n", [(100, 1000), (300, 6000), (760, 4096), (560, 12288), (560, 4096)])
def test_empty_reduction_gives_the_bias(cuda, m, n):
    """K = 0 through the C ABI: no k-block's barrier stands between the copies
    of the scales and bias to LDS and the epilogue that reads them."""
    from nanopointllm_amd import _lib

    note(f"gemm K = 0 m={m} n={n}")
    lib = _lib.load()
    xq = torch.zeros(m, 16, dtype=torch.int8, device=cuda)
    sx, sw = torch.full((m,), 0.5, device=cuda), torch.full((n,), 0.25, device=cuda)
    bias = torch.randn(n, generator=torch.Generator().manual_seed(n)).to(cuda)
    y = torch.full((m, n), 7.0, dtype=torch.float16, device=cuda)
    ws = torch.empty(max(256, lib.w8a8_workspace_bytes(m, 0)), dtype=torch.uint8, device=cuda)
    rc = lib.w8a8_linear_i8in(xq.data_ptr(), 16, sx.data_ptr(), None, sw.data_ptr(),
                              bias.data_ptr(), _lib.EPI_DEQUANT, y.data_ptr(), _lib.F16, n, 0.0,
                              _lib.F16, m, n, 0, ws.data_ptr(), ws.numel(),
                              _lib.stream_handle(cuda))
    _lib.check(rc, "w8a8_linear_i8in")
    assert torch.equal(y, bias.half().expand(m, n))
