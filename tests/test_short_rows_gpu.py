"""Row sums of short rows (a wave per row) against the oracle's fixed-order sums (GPU)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from dionw_amd import _lib
from dionw_amd.newton_schulz import _INPUT_ELEMS
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


def _extended(x: torch.Tensor, to: int) -> torch.Tensor:
    """``x`` with zero columns appended: they change no sum, but rows past the short
    ones' 1024 columns take the workgroup per row."""
    out = torch.zeros(x.shape[0], to, dtype=x.dtype)
    out[:, :x.shape[1]] = x
    return out


@pytest.mark.parametrize("elem", [_lib.F32, _lib.F16, _lib.BF16])
@pytest.mark.parametrize("cols", [4, 64, 252, 256, 260, 508, 512, 768, 1020, 1024])
def test_short_row_sums_have_the_bits_of_long_rows(cols: int, elem: int) -> None:
    """Sums of squares of rows in a wave each, bit for bit those of the same rows in a
    workgroup each: with scores, and alone with and without momentum, heavy ball and
    Nesterov, rounded to bf16 first or not (``elem``: the iteration's type)."""
    rows, mu = 37, 0.95
    print(f"{rows}x{cols} {elem}", flush=True)
    g = torch.Generator().manual_seed(cols)
    grad, m0 = torch.randn(rows, cols, generator=g), torch.randn(rows, cols, generator=g)
    stream = _lib.stream_handle(DEV)

    def sums(width: int) -> list[torch.Tensor]:
        x, m = (_extended(t, width).to(DEV) for t in (grad, m0))
        out = []
        for momentum, nesterov in ((None, 0), (m, 0), (m, 1)):
            rowsq = torch.full((rows,), -1.0, device=DEV)
            _lib.call("dionw_full_sumsq", _pointers([x]), 1, rows, width,
                      None if momentum is None else momentum.data_ptr(), mu, nesterov,
                      rowsq.data_ptr(), elem, stream)
            out.append(rowsq)
        scores, rowsq = (torch.full((rows,), -1.0, device=DEV) for _ in range(2))
        _lib.call("dionw_accumulate_scores", _pointers([x]), 1, rows, width, m.data_ptr(),
                  scores.data_ptr(), rowsq.data_ptr(), elem, stream)
        return [*out, rowsq, scores]

    for i, (short, long) in enumerate(zip(sums(cols), sums(2048), strict=True)):
        assert torch.equal(short, long), f"pass {i}"


@pytest.mark.parametrize("elem", [_lib.F16, _lib.BF16])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("cols", [8, 260, 576, 1024])
def test_short_rows_of_an_input_have_the_bits_of_long_rows(cols: int, dtype: torch.dtype,
                                                           elem: int) -> None:
    """The same for the row sums of ``dionw_normalize_input``, on each input type."""
    rows = 13
    print(f"{rows}x{cols} {dtype} {elem}", flush=True)
    source = torch.randn(rows, cols, generator=torch.Generator().manual_seed(cols)).to(dtype)
    stream = _lib.stream_handle(DEV)

    def sums(width: int) -> torch.Tensor:
        x = _extended(source, width).to(DEV)
        rowsq, den = torch.full((rows,), -1.0, device=DEV), torch.zeros(1, device=DEV)
        pad = (width + 7) // 8 * 8
        out = torch.empty(16, pad, dtype=torch.int16, device=DEV)
        _lib.call("dionw_normalize_input", x.data_ptr(), _INPUT_ELEMS[dtype], 1, rows, width, 1.0,
                  1e-8, rowsq.data_ptr(), den.data_ptr(), 16, pad, elem, out.data_ptr(), None,
                  stream)
        return rowsq

    assert torch.equal(sums(cols), sums(2048))
