"""Row sums of short rows (a wave per row) against the oracle's fixed-order sums (GPU)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from dionw_amd import _lib
from oracle.dion_ref import row_l1_scores

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


def _pointers(tensors):
    return _lib.ptr_array(tensors)


@pytest.mark.parametrize("cols", [4, 64, 252, 256, 260, 508, 512, 516, 768, 1020, 1024, 1028])
@pytest.mark.parametrize("rows", [1, 3, 5, 130])
def test_short_row_sums(rows: int, cols: int) -> None:
    """Two tensors of ``rows`` rows, not a multiple of a workgroup's four: momentum and
    scores bit for bit, sums of squares (with and without momentum, heavy ball and
    Nesterov) within float32 rounding of a sum of ``cols`` terms."""
    print(f"{rows}x{cols}", flush=True)
    g = torch.Generator().manual_seed(rows * 4099 + cols)
    grads = [torch.randn(rows, cols, generator=g) for _ in range(2)]
    m0 = torch.randn(2 * rows, cols, generator=g)
    grad = torch.cat(grads)
    on_gpu = [x.to(DEV) for x in grads]
    m = m0.to(DEV)
    scores, rowsq = (torch.full((2 * rows + 1,), -1.0, device=DEV) for _ in range(2))
    stream = _lib.stream_handle(DEV)
    _lib.call("dionw_accumulate_scores", _pointers(on_gpu), 2, rows, cols, m.data_ptr(),
              scores.data_ptr(), rowsq.data_ptr(), _lib.F32, stream)
    total = m0 + grad
    assert torch.equal(m.cpu(), total)
    assert np.array_equal(scores[:-1].cpu().numpy(), row_l1_scores(total.numpy()))
    assert scores[-1] == -1 and rowsq[-1] == -1
    tight = cols * 2.0 ** -24

    def close(u: torch.Tensor) -> None:
        want = u.double().square().sum(1)
        assert ((rowsq[:-1].cpu().double() - want).abs() <= tight * want).all()

    close(total)
    mu = 0.95
    old = m0.to(DEV)
    for momentum, nesterov, u in ((old, 0, total), (None, 0, grad),
                                  (old, 1, grad + total * np.float32(mu))):
        _lib.call("dionw_full_sumsq", _pointers(on_gpu), 2, rows, cols,
                  None if momentum is None else momentum.data_ptr(), mu, nesterov,
                  rowsq.data_ptr(), _lib.F32, stream)
        close(u)
        assert rowsq[-1] == -1
