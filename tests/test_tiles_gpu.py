"""The products' tiles at the sizes where they can go wrong (GPU).

``dionw_gemm_nt`` against float64 on shapes around the edges of the 128x128 and
256x256 tiles and their halves, with the fewest and an odd number of 64-deep
stages, with and without an addend (whole 16-byte rows or not), with padded
leading dimensions, symmetric and not, and with the transposed output. The bar
per element: half a unit of the output type at the result, plus float32 rounding
of a sum of k products.
"""

from __future__ import annotations

import pytest
import torch

from dionw_amd._kernels import gemm_nt

pytestmark = pytest.mark.gpu
DEV = "cuda"
HALF_ULP = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


def _strided(shape: tuple[int, int, int], pad: int, dtype: torch.dtype, g) -> torch.Tensor:
    """Random entries in rows of ``cols + pad`` elements."""
    b, rows, cols = shape
    store = torch.randn(b, rows, cols + pad, device=DEV, generator=g).to(dtype)
    return store[:, :, :cols]


def _check(got: torch.Tensor, product: torch.Tensor, scale: torch.Tensor, k: int, what: str) -> None:
    unit = HALF_ULP[got.dtype]
    bound = unit * product.abs() * 1.01 + (k + 4) * 2.0 ** -23 * scale + 2.0 ** -24
    excess = ((got.double() - product).abs() - bound).max()
    assert excess <= 0, f"{what}: {float(excess):.3g} past the bound"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize(("batch", "m", "n", "k", "addend", "pad"), [
    (1, 64, 72, 128, True, 0),       # one small tile, two stages
    (1, 129, 200, 192, True, 8),     # a row past a half, three stages, padded rows
    (2, 127, 257, 128, False, 0),
    (1, 384, 128, 320, True, 0),     # half tiles exactly
    (3, 136, 132, 128, True, 4),     # addend rows that are not 16-byte chunks
    (40, 256, 512, 128, True, 0),    # enough tiles for 256x256: whole,
    (40, 264, 520, 192, True, 8),    # a few rows and columns past,
    (40, 385, 640, 128, True, 0),    # and half of the last tile used
    (40, 392, 633, 256, False, 0),
    (64, 513, 248, 64, False, 0),    # one stage: the 32-deep kernel
])
def test_product_at_tile_edges(batch, m, n, k, addend, pad, dtype) -> None:
    print(f"{batch} x {m}x{n}x{k} addend {addend} pad {pad} {dtype}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(m * n + k)
    a = _strided((batch, m, k), 8 * (pad > 0), dtype, g)
    b = _strided((batch, n, k), 16 * (pad > 0), dtype, g)
    d = _strided((batch, m, n), pad, dtype, g) if addend else None
    out = torch.full((batch, m, n + pad), 7.0, device=DEV, dtype=dtype)
    out_t = torch.full((batch, n, m + pad), 7.0, device=DEV, dtype=dtype)
    gemm_nt(a, b, d=d, alpha=0.5, beta=-1.25 if addend else 0.0, out=out[:, :, :n],
            out_t=out_t[:, :, :m])
    product = 0.5 * torch.matmul(a.double(), b.double().mT.contiguous())
    scale = 0.5 * torch.matmul(a.double().abs(), b.double().abs().mT.contiguous())
    if addend:
        product -= 1.25 * d.double()
        scale += 1.25 * d.double().abs()
    _check(out[:, :, :n], product, scale, k, "out")
    assert torch.equal(out_t[:, :, :m], out[:, :, :n].mT), "the transposed output differs"
    assert (out[:, :, n:] == 7).all() and (out_t[:, :, m:] == 7).all(), "wrote past the rows"


@pytest.mark.parametrize(("batch", "n", "k", "addend"), [
    (1, 64, 128, True), (2, 136, 192, True), (1, 200, 256, False), (3, 384, 384, True),
    (40, 264, 128, False), (40, 512, 512, True), (40, 392, 448, True),
])
def test_symmetric_product_at_tile_edges(batch, n, k, addend) -> None:
    """A symmetric product against the full one, bit for bit above the diagonal,
    and exactly symmetric."""
    print(f"{batch} x {n}x{n}x{k} addend {addend}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(n + k)
    a = torch.randn(batch, n, k, device=DEV, generator=g).half()
    d = torch.randn(batch, n, n, device=DEV, generator=g).half() if addend else None
    if addend:
        d = (d + d.mT).contiguous()
    beta = 0.75 if addend else 0.0
    got = gemm_nt(a, a, d=d, alpha=2.0, beta=beta, symmetric=True,
                  out=torch.empty(batch, n, n, device=DEV, dtype=a.dtype))
    full = gemm_nt(a, a, d=d, alpha=2.0, beta=beta)
    assert torch.equal(torch.triu(got), torch.triu(full))
    assert torch.equal(got, got.mT)
