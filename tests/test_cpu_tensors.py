"""Entry points refuse CPU tensors on the host, before a kernel gets their addresses (CPU)."""

from __future__ import annotations

import pytest
import torch

from dionw_amd import _lib
from dionw_amd._adamw import adamw_step
from dionw_amd._kernels import accumulate_copy_decay, accumulate_row_l1, gemm_nt, ns_line_1, ns_line_2
from dionw_amd.newton_schulz import NewtonSchulz, newton_schulz_fn


@pytest.fixture(autouse=True)
def _no_launches(monkeypatch: pytest.MonkeyPatch) -> None:
    """No GPU is touched, whatever the machine: a current device, a stream, and a
    library call that fails the test instead of launching."""
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda index: 0, raising=False)
    monkeypatch.setattr(_lib, "call", lambda name, *args: pytest.fail(f"{name} was launched"))


def _adamw() -> None:
    param = torch.nn.Parameter(torch.ones(8))
    param.grad = torch.ones(8)
    adamw_step({"params": [param], "lr": 1e-3, "betas": (0.9, 0.95), "eps": 1e-8,
                "weight_decay": 0.0}, {param: {}})


@pytest.mark.parametrize("call", [
    lambda: _lib.stream_handle(torch.device("cpu")),
    lambda: gemm_nt(torch.ones(8, 64).half(), torch.ones(8, 64).half()),
    lambda: gemm_nt(torch.ones(2, 8, 64), torch.ones(2, 8, 64)),
    lambda: ns_line_1(torch.ones(8, 64).half()),
    lambda: ns_line_2(torch.ones(64, 64).half(), 1.0, 2.0),
    lambda: accumulate_row_l1(torch.ones(4, 8), torch.ones(4, 8), torch.ones(4), 8),
    lambda: accumulate_copy_decay(torch.ones(4, 8), torch.ones(4, 8), torch.ones(4, 8), 0.9,
                                  nesterov=False),
    lambda: newton_schulz_fn(NewtonSchulz.GRAM)(torch.ones(4, 8), 1e-8),
    _adamw,
], ids=["stream", "gemm_nt", "gemm_nt f32", "ns_line_1", "ns_line_2", "row_l1", "copy_decay",
        "newton_schulz", "adamw"])
def test_cpu_tensors_are_refused(call) -> None:
    with pytest.raises(ValueError):
        call()
