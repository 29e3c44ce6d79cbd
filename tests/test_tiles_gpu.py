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
from dionw_amd.newton_schulz import NewtonSchulz, newton_schulz_fn

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
    (64, 513, 248, 64, False, 0),    # one stage and many tiles: the 32-deep kernel
    (2, 100, 72, 64, True, 8),       # 64x64 tiles: one stage,
    (1, 65, 130, 576, True, 0),      # more stages than the ring holds,
    (3, 40, 24, 1024, False, 8),     # less than a tile
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
    (1, 64, 128, True), (1, 64, 64, True), (2, 136, 192, True), (1, 200, 256, False), (3, 384, 384, True),
    (40, 264, 128, False), (40, 512, 512, True), (40, 392, 448, True),
    (2, 640, 128, True), (1, 1090, 128, False), (8, 1300, 128, True),  # several column strips
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


@pytest.mark.parametrize(("blocks", "r", "c"), [
    (1, 64, 72), (2, 128, 200), (60, 192, 264), (3, 320, 1000), (40, 512, 776),
])
def test_left_products_read_the_iterate_as_it_lies(blocks: int, r: int, c: int) -> None:
    """The products that read X as a [k, n] operand, on each tile and with columns
    that end inside a tile: five Keller steps against the same polynomials in
    float64 (bf16 rounding: within 0.03, as the quintics' oracle is)."""
    print(f"{blocks} x {r}x{c}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(r + c)
    x = torch.randn(blocks, r, c, device=DEV, generator=g)
    got = newton_schulz_fn(NewtonSchulz.KELLER_TRITON)(x, 1e-8).double()
    y = x.double()
    y = y / y.flatten(1).norm(dim=1).view(-1, 1, 1)
    for _ in range(5):
        gram = torch.matmul(y, y.mT.contiguous())
        y = 3.4445 * y + torch.matmul(2.0315 * torch.matmul(gram, gram) - 4.7750 * gram, y)
    for b in range(blocks):
        assert (got[b] - y[b]).norm() <= 0.03 * y[b].norm(), f"block {b}"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("k", [128, 192, 448])
@pytest.mark.parametrize(("batch", "m", "n"), [
    (40, 512, 640),  # 256x256 tiles, the last column's half empty
    (40, 256, 192),  # 128x128 tiles, the same
])
def test_addend_in_tiles_without_a_right_half(batch, m, n, k, dtype) -> None:
    """The addend's last rows go to the slot of the row operand's second half while
    that half is still to be multiplied: against float64, and the same bits again."""
    print(f"{batch} x {m}x{n}x{k} {dtype}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    a, b, d = (_strided(shape, 0, dtype, g)
               for shape in ((batch, m, k), (batch, n, k), (batch, m, n)))
    got = gemm_nt(a, b, d=d, alpha=0.5, beta=-1.25)
    product = 0.5 * torch.matmul(a.double(), b.double().mT.contiguous()) - 1.25 * d.double()
    scale = (0.5 * torch.matmul(a.double().abs(), b.double().abs().mT.contiguous())
             + 1.25 * d.double().abs())
    _check(got, product, scale, k, "out")
    for _ in range(3):
        assert torch.equal(gemm_nt(a, b, d=d, alpha=0.5, beta=-1.25), got)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize(("batch", "m", "n", "k", "symmetric"), [
    (1, 130, 72, 128, False),    # 128x128 tiles of the ring of two 64-deep stages,
    (3, 392, 385, 448, False),   # with ragged rows and columns,
    (36, 768, 768, 192, False),
    (36, 768, 760, 64, False),   # one stage;
    (40, 520, 520, 320, False),  # 256x256 tiles,
    (64, 500, 500, 64, False),   # one stage
    (2, 264, 264, 192, True), (36, 520, 520, 128, True),
])
def test_addend_in_rows_that_are_no_chunks(batch, m, n, k, symmetric, dtype) -> None:
    """An addend whose rows are not 16-byte chunks, at depths that are a multiple of 64."""
    print(f"{batch} x {m}x{n}x{k} symmetric {symmetric} {dtype}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    a = _strided((batch, m, k), 0, dtype, g)
    b = a if symmetric else _strided((batch, n, k), 8, dtype, g)
    d = _strided((batch, m, n), 4 if n % 2 == 0 else 3, dtype, g)
    if symmetric:
        d.copy_(d + d.mT)
    got = gemm_nt(a, b, d=d, alpha=0.5, beta=-1.25, symmetric=symmetric,
                  out=torch.empty(batch, m, n, device=DEV, dtype=dtype))
    product = 0.5 * torch.matmul(a.double(), b.double().mT.contiguous()) - 1.25 * d.double()
    scale = (0.5 * torch.matmul(a.double().abs(), b.double().abs().mT.contiguous())
             + 1.25 * d.double().abs())
    _check(got, product, scale, k, "out")


@pytest.mark.parametrize("wide", [False, True])
def test_operand_past_2_gb(wide) -> None:
    """Rows past the 2 GB that a tile's byte offsets reach, read and multiplied in place:
    the first and last rows against float64."""
    m, n, k = 65600, 136, 16384
    print(f"{m}x{n}x{k} wide {wide}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(7)
    long = torch.randn(m, k, device=DEV, generator=g, dtype=torch.float16)
    short = torch.randn(n, k, device=DEV, generator=g, dtype=torch.float16)
    got = gemm_nt(short, long) if wide else gemm_nt(long, short)
    got = got.mT if wide else got
    for rows in (slice(0, 64), slice(m - 200, m)):
        a, b = long[rows].double(), short.double()
        _check(got[rows], a @ b.T.contiguous(), a.abs() @ b.T.abs().contiguous(), k, str(rows))


@pytest.mark.parametrize(("batch", "m", "n", "addend"), [
    (257, 64, 64, True), (300, 50, 72, True), (3000, 64, 64, False), (90, 130, 88, True),
    (40, 513, 64, True),
])
def test_one_stage_on_many_small_tiles(batch, m, n, addend) -> None:
    """Depth 64 on more 64x64 tiles than CUs, whose workgroups hold one stage and share
    a CU."""
    print(f"{batch} x {m}x{n}x64 addend {addend}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(m + n)
    a = _strided((batch, m, 64), 0, torch.bfloat16, g)
    b = _strided((batch, n, 64), 8, torch.bfloat16, g)
    d = _strided((batch, m, n), 8, torch.bfloat16, g) if addend else None
    out = torch.full((batch, m, n + 8), 7.0, device=DEV, dtype=torch.bfloat16)
    out_t = torch.full((batch, n, m + 8), 7.0, device=DEV, dtype=torch.bfloat16)
    gemm_nt(a, b, d=d, alpha=0.5, beta=-1.25 if addend else 0.0, out=out[:, :, :n],
            out_t=out_t[:, :, :m])
    product = 0.5 * torch.matmul(a.double(), b.double().mT.contiguous())
    scale = 0.5 * torch.matmul(a.double().abs(), b.double().abs().mT.contiguous())
    if addend:
        product -= 1.25 * d.double()
        scale += 1.25 * d.double().abs()
    _check(out[:, :, :n], product, scale, 64, "out")
    assert torch.equal(out_t[:, :, :m], out[:, :, :n].mT)
    assert (out[:, :, n:] == 7).all() and (out_t[:, :, m:] == 7).all(), "wrote past the rows"


@pytest.mark.parametrize("kind", [NewtonSchulz.GRAM, NewtonSchulz.KELLER, NewtonSchulz.POLAR_EXPRESS_TRITON])
@pytest.mark.parametrize(("rows", "cols"), [(48, 192), (64, 130), (200, 60)])
def test_many_thin_blocks_are_iterated_alike(rows: int, cols: int, kind) -> None:
    """A block of a batch of 300 thin blocks, whose products take several rounds of
    one-stage tiles, has the bits that it has alone."""
    print(f"300 x {rows}x{cols} {kind}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(rows + cols)
    x = torch.randn(300, rows, cols, device=DEV, generator=g)
    f = newton_schulz_fn(kind)
    got = f(x, 1e-8)
    for b in (0, 7, 255, 256, 299):
        assert torch.equal(got[b], f(x[b:b + 1], 1e-8)[0]), f"block {b}"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize(("batch", "m", "n", "k", "symmetric"), [
    (1, 64, 64, 64, False), (3, 65, 129, 192, False), (300, 64, 72, 64, False),  # 64x64 tiles
    (40, 256, 257, 128, False), (40, 250, 250, 128, True),  # 128x128
    (40, 512, 513, 128, False), (40, 512, 512, 192, True), (40, 515, 515, 128, True),  # 256x256
])
@pytest.mark.parametrize("offset", [1, 3, 4])
def test_outputs_in_rows_that_start_anywhere(batch, m, n, k, symmetric, offset, dtype) -> None:
    """Outputs whose rows start at any element have the bits of aligned ones, and nothing
    beside them is written."""
    print(f"{batch} x {m}x{n}x{k} symmetric {symmetric} offset {offset} {dtype}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    a = _strided((batch, m, k), 0, dtype, g)
    b = a if symmetric else _strided((batch, n, k), 8, dtype, g)

    def outputs(rows: int, cols: int, start: int, pad: int) -> tuple[torch.Tensor, torch.Tensor]:
        store = torch.full((start + batch * rows * (cols + pad) + 8,), 7.0, device=DEV, dtype=dtype)
        whole = store[start:start + batch * rows * (cols + pad)].view(batch, rows, cols + pad)
        return store, whole[:, :, :cols]

    results = []
    for start, pad in ((0, -n % 8 + 8), (offset, (-n % 8 + 8) + offset)):
        store, out = outputs(m, n, start, pad)
        store_t, out_t = outputs(n, m, start, (-m % 8 + 8) + (offset if start else 0))
        gemm_nt(a, b, alpha=0.5, out=out, out_t=None if symmetric else out_t, symmetric=symmetric)
        results.append(out.clone())
        if not symmetric:
            assert torch.equal(out_t, out.mT)
        for written, s in ((out, store), (out_t, store_t)):
            written.fill_(7.0)
            assert (s == 7).all(), "wrote beside the rows"
    assert torch.equal(*results)
