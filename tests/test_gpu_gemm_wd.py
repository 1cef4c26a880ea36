"""The weights-direct GEMM tile (csrc/gemm.hip ``gemm_wd_kernel``): 112 x 256
(8 wavefronts of 112 x 32), taken when one round of it fills the CUs and K has
at most 15 k-blocks of 64 (longer products run on the pipelined tiles, and the
shapes here that do name the one they take).  Weight fragments go straight from
memory into registers several k-blocks ahead; only the activations pass through
LDS.

Bars as for every GEMM path: int32 accumulators bit-exact against the
oracle's integer product; dequant outputs bit-equal to the oracle's binary32
result rounded once; SiLU*mul equal to the oracle's; the int8 requant of h
and the integer requant (requant1) bit-exact; the two-phase per-block maxima
giving hq and scales bit-exact against the per-token quantization of h.
Shapes are ragged in M, N and K, including K of one or a few k-blocks (fewer
than the prefetch depth), of 11 to 15 (the unrolled loop of 10 and what is left
behind it) and K that leaves a partial one.
"""
from __future__ import annotations

import sys

import numpy as np
import pytest
import torch

from gemm_tiles import launched_tile
from oracle import w8a8_oracle as O

pytestmark = pytest.mark.gpu


def note(msg: str) -> None:
    sys.__stderr__.write(f"[gpu-case] {msg}\n")
    sys.__stderr__.flush()


def _case(m, n, k, seed):
    g = torch.Generator().manual_seed(seed)
    xq = torch.randint(-127, 128, (m, k), generator=g, dtype=torch.int8)
    wq = torch.randint(-127, 128, (n, k), generator=g, dtype=torch.int8)
    rng = np.random.default_rng(seed)
    sx = O.scale_from_absmax(np.abs(rng.standard_normal((m, 1))) * 3).astype(np.float32)
    sw = O.scale_from_absmax(np.abs(rng.standard_normal(n)) * 0.05).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    return xq, wq, sx, sw, bias


SHAPES = [
    # (m, n, k, tile): ragged rows / columns, K from one k-block to 11008
    (560, 12288, 960, "wd7x2"), (500, 12000, 641, "wd7x2"), (545, 12100, 64, "wd7x2"),
    (480, 12288, 200, "wd7x2"), (555, 11900, 700, "wd7x2"), (480, 12100, 640, "wd7x2"),
    (400, 16000, 800, "wd7x2"), (470, 11100, 64, "wd7x2"), (465, 13000, 130, "wd7x2"),
    (560, 12288, 4096, "pipe-192x160"), (500, 12000, 1000, "pipe-192x160"),
    (555, 11900, 2700, "pipe-192x160"), (400, 16000, 1111, "pipe-256x128"),
]


@pytest.mark.parametrize("m,n,k,cfg", SHAPES)
def test_wd_int32_and_dequant(cuda, m, n, k, cfg):
    from nanopointllm_amd import w8a8

    assert launched_tile(m, n, k) == cfg
    xq, wq, sx, sw, bias = _case(m, n, k, seed=m + n + k)
    note(f"gemm {cfg} m={m} n={n} k={k}")
    xd, wp = xq.to(cuda), w8a8.pack_rows(wq.to(cuda))
    eacc = O.int32_matmul_f64(xq.numpy(), wq.numpy())
    np.testing.assert_array_equal(w8a8.gemm_i32(xd, wp, n).cpu().numpy(), eacc)
    sxt, swt, bt = (torch.from_numpy(a).to(cuda) for a in (sx, sw, bias))
    for dt in (torch.float16, torch.bfloat16, torch.float32):
        for b in (None, bt):
            y = w8a8.linear_i8in(xd, sxt, wp, swt, b, n, out_dtype=dt)
            exp = O.dequant_epilogue(eacc, sx, sw, None if b is None else bias)
            got = y.float().cpu().numpy()
            if dt == torch.bfloat16:
                want = torch.from_numpy(exp).to(torch.bfloat16).float().numpy()
            else:
                want = exp.astype(np.float16).astype(np.float32) if dt == torch.float16 else exp
            np.testing.assert_array_equal(got, want, err_msg=f"{dt} bias={b is not None}")


@pytest.mark.parametrize("m,inter,k,cfg", [(520, 6100, 960, "wd7x2"), (560, 6144, 333, "wd7x2"),
                                            (470, 6000, 730, "wd7x2"), (400, 7500, 640, "wd7x2"),
                                            (520, 6100, 4096, "pipe-192x160"),
                                            (470, 6000, 1000, "pipe-192x160")])
def test_wd_silu_mul_int8_chain_and_two_phase(cuda, m, inter, k, cfg):
    from nanopointllm_amd import _lib, w8a8

    n = 2 * inter
    assert launched_tile(m, n, k) == cfg
    xq, wq, sx, sw, _ = _case(m, n, k, seed=11 + k)
    note(f"gemm {cfg} silu m={m} inter={inter} k={k}")
    wp = w8a8.pack_rows(wq.to(cuda), _lib.ROWS_INTERLEAVE_HALVES)
    sp = O.pack_gateup_rows(sw[:inter, None], sw[inter:, None], "interleave")[:, 0]
    qp = O.pack_gateup_rows(wq.numpy()[:inter], wq.numpy()[inter:], "interleave")
    xd, sxt = xq.to(cuda), torch.from_numpy(sx).to(cuda)
    spt = torch.from_numpy(np.ascontiguousarray(sp)).to(cuda)
    h = w8a8.linear_i8in(xd, sxt, wp, spt, None, n, epilogue=_lib.EPI_SILU_MUL,
                         out_dtype=torch.float16)
    eh = O.gateup_silu_mul_from_acc(O.int32_matmul_f64(xq.numpy(), qp), sx, sp,
                                    layout="interleave")
    np.testing.assert_array_equal(h.cpu().numpy(), eh.astype(np.float16))
    h_scale = float(O.static_activation_scale(float(h.float().abs().max().item())))
    hq = w8a8.linear_i8in(xd, sxt, wp, spt, None, n, epilogue=_lib.EPI_SILU_MUL_Q8,
                          out_dtype=torch.int8, y_scale=h_scale)
    eq = O.quantize_symmetric(h.cpu().numpy().astype(np.float32), np.float32(h_scale))
    np.testing.assert_array_equal(hq.cpu().numpy(), eq)
    # Two-phase per-token requant: the epilogue's per-block maxima of h.
    out = w8a8.gateup_silu_mul_two_phase(xd, wp, spt, None, n, x_scale=sxt, in_features=k)
    np.testing.assert_array_equal(out.h.cpu().numpy(), h.cpu().numpy())
    tq, ts = O.dynamic_per_token_quant(h.cpu().numpy().astype(np.float32))
    np.testing.assert_array_equal(out.hq.cpu().numpy(), tq)
    np.testing.assert_array_equal(out.scale.cpu().numpy(), ts[:, 0])


@pytest.mark.parametrize("m,n,k,cfg", [(560, 12288, 700, "wd7x2"), (400, 15000, 960, "wd7x2"),
                                       (560, 12288, 1000, "pipe-192x160"),
                                       (400, 15000, 2000, "pipe-256x128")])
def test_wd_integer_epilogues(cuda, m, n, k, cfg):
    """requant1 (multiplier / shift int8 out) and the single-rounding
    int32 -> bf16 dequant on the weights-direct tiles."""
    from nanopointllm_amd import _lib, integer_epilogues as E, w8a8

    assert launched_tile(m, n, k) == cfg
    xq, wq, sx, sw, _ = _case(m, n, k, seed=5 + k)
    comp = [O.compile_fp16_requant_scale(0.02, float(w), 0.5) for w in sw]
    mult = np.array([c[0] for c in comp], np.uint32)
    shift = np.array([c[1] for c in comp], np.int32)
    bias = np.random.default_rng(5).integers(-3000, 3000, n).astype(np.int32)
    note(f"gemm {cfg} integer epilogues m={m} n={n} k={k}")
    multt = torch.from_numpy(mult.view(np.int32)).to(cuda)
    shiftt, biast = torch.from_numpy(shift).to(cuda), torch.from_numpy(bias).to(cuda)
    xd, wp = xq.to(cuda), w8a8.pack_rows(wq.to(cuda))
    acc = O.int32_matmul_f64(xq.numpy(), wq.numpy())
    y = E.linear_i8in_requant(xd, wp, multt, shiftt, biast, n).cpu().numpy()
    ref = E.requantize_int32(torch.from_numpy(acc).to(cuda), biast, multt, shiftt)
    np.testing.assert_array_equal(y, ref.cpu().numpy())
    rng = np.random.default_rng(6)
    for i, j in zip(rng.integers(0, m, 500), rng.integers(0, n, 500)):
        assert y[i, j] == O.requantize_int32(int(acc[i, j]), int(bias[j]), int(mult[j]),
                                             int(shift[j]))
    sxt, swt = torch.from_numpy(sx).to(cuda), torch.from_numpy(sw).to(cuda)
    yb = w8a8.linear_i8in(xd, sxt, wp, swt, None, n, epilogue=_lib.EPI_DEQUANT_BF16_EXACT,
                          out_dtype=torch.bfloat16)
    sa_bits = sx[:, 0].astype(np.float16).view(np.uint16)
    sw_bits = sw.astype(np.float16).view(np.uint16)
    for i, j in zip(rng.integers(0, m, 500), rng.integers(0, n, 500)):
        want = O.dequantize_int32_to_bf16(int(acc[i, j]), int(sa_bits[i]), int(sw_bits[j]))
        got = int(yb[i, j].view(torch.int16).item()) & 0xFFFF
        assert got == want, (i, j)


@pytest.mark.parametrize("m,n,k,epi", [(8, 4096, 4096, "f16"), (96, 1000, 700, "i32"),
                                       (560, 12288, 4096, "f16"), (560, 4096, 11008, "bf16"),
                                       (567, 22016, 4096, "silu"), (1024, 4096, 4096, "f32")])
def test_linear_packed_equals_linear_i8in(cuda, m, n, k, epi):
    """w8a8_linear_packed (activations already in packed tiles, the GEMM
    alone) gives the bits of w8a8_linear_i8in on the same row-major rows."""
    from nanopointllm_amd import _lib, w8a8

    xq, wq, sx, sw, bias = _case(m, n, k, seed=31 + m)
    layout = _lib.ROWS_INTERLEAVE_HALVES if epi == "silu" else _lib.ROWS_AS_IS
    note(f"linear_packed m={m} n={n} k={k} {epi} tile={launched_tile(m, n, k)}")
    xd, wp = xq.to(cuda), w8a8.pack_rows(wq.to(cuda), layout)
    sxt, swt, bt = (torch.from_numpy(a).to(cuda) for a in (sx, sw, bias))
    code = {"i32": _lib.EPI_I32, "silu": _lib.EPI_SILU_MUL}.get(epi, _lib.EPI_DEQUANT)
    dt = {"i32": torch.int32, "f16": torch.float16, "bf16": torch.bfloat16,
          "f32": torch.float32, "silu": torch.float16}[epi]
    b = bt if epi in ("f16", "f32") else None
    ref = w8a8.linear_i8in(xd, sxt, wp, swt, b, n, epilogue=code, out_dtype=dt)
    got = w8a8.linear_packed(w8a8.pack_rows(xd), sxt, m, k, wp, swt, b, n, epilogue=code,
                             out_dtype=dt)
    assert torch.equal(got, ref)
    with pytest.raises(ValueError, match="packed tiles"):
        w8a8.linear_packed(xd[: m // 2], sxt, m, k, wp, swt, b, n, epilogue=code, out_dtype=dt)
