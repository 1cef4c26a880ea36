"""How the eager linears reach the library (no GPU: its entry points are
recorded).  Up to 16 rows, where a call is bound by the host, the entry point
is called straight from the wrapper's own frame, first without a workspace;
past them once, with one."""
from __future__ import annotations

import sys

import pytest
import torch

from nanopointllm_amd import _lib, w8a8

N, K = 32, 64


class Recorder:
    """Stands for the loaded library: entry points note their caller and
    whether they got a workspace, and ask for one when ``needs`` says so."""

    def __init__(self, needs: bool) -> None:
        self.needs = needs
        self.calls: list[tuple[str, str, bool]] = []
        self.real = _lib.load()

    def __getattr__(self, name):
        if name not in ("w8a8_linear", "w8a8_linear_residual", "w8a8_rmsnorm_linear",
                        "w8a8_rmsnorm_linear_ss"):
            return getattr(self.real, name)

        def entry(*args):
            assert len(args) == len(_lib._SIGNATURES[name][1])
            workspace = args[-3] is not None
            assert (args[-2] > 0) == workspace
            self.calls.append((name, sys._getframe(1).f_code.co_name, workspace))
            return _lib.ERR_WORKSPACE if self.needs and not workspace else _lib.OK

        return entry


def _record(monkeypatch, needs: bool) -> Recorder:
    lib = Recorder(needs)
    monkeypatch.setattr(_lib, "load", lambda path=None: lib)
    monkeypatch.setattr(_lib, "require_cuda", lambda *t: torch.device("cpu"))
    monkeypatch.setattr(_lib, "stream_handle", lambda device: 0)
    return lib


def _linear(x, w, s):
    w8a8.linear_dynamic(x, w, s, None, N)


def _rmsnorm(x, w, s):
    w8a8.rmsnorm_linear(x, torch.ones(K, dtype=x.dtype), 1e-6, w, s, None, N)


def _rmsnorm_ss(x, w, s):
    w8a8.rmsnorm_linear(x, torch.ones(K, dtype=x.dtype), 1e-6, w, s, None, N,
                        ss_parts=torch.zeros(len(x), K // 8))


def _residual(x, w, s):
    w8a8.linear_residual(x, w, s, None, N, torch.zeros(len(x), N, dtype=x.dtype))


@pytest.mark.parametrize("needs", [False, True])
@pytest.mark.parametrize("m", [1, 16, 17, 300])
@pytest.mark.parametrize("call,entry,frame", [
    (_linear, "w8a8_linear", "linear_dynamic"),
    (_rmsnorm, "w8a8_rmsnorm_linear", "rmsnorm_linear"),
    (_rmsnorm_ss, "w8a8_rmsnorm_linear_ss", "rmsnorm_linear"),
    (_residual, "w8a8_linear_residual", "_residual_call")])
def test_calls_into_the_library(monkeypatch, call, entry, frame, m, needs):
    w = torch.zeros(w8a8.packed_bytes(N, K), dtype=torch.int8)
    lib = _record(monkeypatch, needs)
    call(torch.zeros(m, K, dtype=torch.float16), w, torch.ones(N))
    tries = [True] if m > 16 else ([False, True] if needs else [False])
    assert lib.calls == [(entry, frame, t) for t in tries]
