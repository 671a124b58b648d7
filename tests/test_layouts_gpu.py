"""The tile kernels on every storage order of their operands, against the product in 64 bits: sizes at the edges of the tiles and of
the 16-byte copies, and few enough tiles or many enough for each depth of the copy pipeline.

Tolerances: half a unit in the last place of the result's type per element bounds the rounding (in the 2-norm at most eps / 2), and
single-precision sums of k terms add about sqrt(k) * 2**-24; twice that sum is allowed."""
import math

import pytest
import torch

import tritonblas_amd as tb
from tritonblas_amd.matmul import streamk_matmul_lt

pytestmark = pytest.mark.gpu


def _stored(gen, rows, cols, order, dtype):
    x = torch.randn((rows, cols) if order == "T" else (cols, rows), device="cuda", generator=gen).to(dtype)
    return x if order == "T" else x.T


def _check(c, a, b):
    want = a.double() @ b.double()
    tol = 2 * (torch.finfo(c.dtype).eps / 2 + math.sqrt(a.shape[1]) * 2.0 ** -24)
    err = ((c.double() - want).norm() / want.norm()).item()
    assert err <= tol, f"relative error {err:.3e} > {tol:.3e}"


@pytest.mark.parametrize("ta,tb_", [("T", "T"), ("T", "N"), ("N", "T"), ("N", "N")])
@pytest.mark.parametrize("dtype,tile", [(d, t) for d in (torch.bfloat16, torch.float16, torch.float32) for t in ((256, 256), (128, 128), (64, 64))] +
                         [(torch.bfloat16, (32, 128)), (torch.float16, (32, 128))])
def test_every_tile_and_storage_order(dtype, tile, ta, tb_):
    bk = (256 if tile[0] == 32 else 128) // dtype.itemsize
    gen = torch.Generator(device="cuda").manual_seed(tile[0])
    # one K step, fewer than the pipeline is deep, more; one row chunk, a tile and a chunk, several tiles
    for m, n, k in [(8, 8, bk), (tile[0] + 8, tile[1] - 8, 3 * bk), (2 * tile[0] - 16, 3 * tile[1] + 24, 7 * bk), (1544, 1536, 2 * bk)]:
        a, b = _stored(gen, m, k, ta, dtype), _stored(gen, k, n, tb_, dtype)
        c = torch.full((m, n), float("nan"), dtype=dtype, device="cuda")
        sel = tb.OrigamiMatmulSelector(m, n, k, dtype, dtype, dtype, a.device)
        sel._sel.block_m, sel._sel.block_n, sel._sel.block_k = tile[0], tile[1], bk
        tb.matmul_lt(a, b, c, sel, tb.matmul_preamble(sel))
        _check(c, a, b)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("m,n,k", [(64, 72, 80), (65, 72, 83), (40, 77, 64), (1, 8, 8)])
@pytest.mark.parametrize("view", ["rows", "transposed", "offset", "strided"])
def test_gradients_for_every_way_an_operand_is_stored(view, m, n, k, dtype):
    gen = torch.Generator(device="cuda").manual_seed(m + n)

    def operand(rows, cols):
        if view == "transposed":
            return _stored(gen, rows, cols, "N", dtype)
        if view == "offset":
            return _stored(gen, rows, cols + 3, "T", dtype)[:, 3:]
        if view == "strided":
            return _stored(gen, 2 * rows, 2 * cols, "T", dtype)[::2, ::2]
        return _stored(gen, rows, cols, "T", dtype)

    a, b, g = operand(m, k).requires_grad_(), operand(k, n).requires_grad_(), operand(m, n)
    da, db = torch.autograd.grad(tb.matmul(a, b), (a, b), g)
    assert da.shape == a.shape and db.shape == b.shape
    _check(da, g, b.detach().T)
    _check(db, a.detach().T, g)


def _poisoned(gen, rows, cols, order, dtype, pad):
    """An operand whose rows (as stored) are followed by ``pad`` NaNs, for int8 by its largest value."""
    r, c = (rows, cols) if order == "T" else (cols, rows)
    x = torch.randint(-9, 9, (r, c + pad), device="cuda", generator=gen).float()
    x[:, c:] = float("nan") if dtype != torch.int8 else 127
    x = x.to(dtype)[:, :c]
    return x if order == "T" else x.T


@pytest.mark.parametrize("dtype,ta,tb_", [(d, "T", "N") for d in (torch.float8_e4m3fn, torch.float8_e5m2, torch.int8)] +
                         [(d, x, y) for d in (torch.bfloat16, torch.float32) for x in "TN" for y in "TN"])
@pytest.mark.parametrize("tile", [(256, 256), (128, 128), (64, 64)])
@pytest.mark.parametrize("schedule", ["persistent", "streamk"])
def test_k_that_is_no_multiple_of_the_k_step(schedule, tile, dtype, ta, tb_):
    chunk = 16 // dtype.itemsize
    out = torch.bfloat16 if dtype.itemsize == 1 else dtype
    gen = torch.Generator(device="cuda").manual_seed(5)
    for m, n, k in [(16, 16, chunk), (tile[0] + 16, 2 * tile[1], 8 * chunk + chunk), (272, 304, 37 * chunk), (520, 512, 63 * chunk)]:
        if (ta, tb_) == ("N", "T"):
            k -= 1                     # K along neither operand's rows: any K
        a, b = _poisoned(gen, m, k, ta, dtype, chunk), _poisoned(gen, k, n, tb_, dtype, chunk)
        c = torch.full((m, n), float("nan"), dtype=out, device="cuda")
        sel = tb.OrigamiMatmulSelector(m, n, k, dtype, dtype, out, a.device, streamk=schedule == "streamk")
        sel._sel.block_m, sel._sel.block_n, sel._sel.block_k = tile[0], tile[1], 128 // dtype.itemsize
        config = tb.matmul_preamble(sel)
        if dtype.itemsize == 1:
            one_m, one_n = torch.ones(m, device="cuda"), torch.ones(n, device="cuda")
            tb.matmul_a8w8_lt(a, b, one_m, one_n, c, sel, config, enable_streamk=schedule == "streamk")
        else:
            tb.matmul_lt(a, b, c, sel, config, enable_streamk=schedule == "streamk")
        # (whole numbers below 2**24: the sums are exact and only the result is rounded)
        assert torch.equal(c, (a.double() @ b.double()).float().to(out)), (m, n, k)


@pytest.mark.parametrize("types", [(torch.float8_e4m3fn, torch.float8_e5m2), (torch.float8_e5m2, torch.float8_e4m3fn)])
@pytest.mark.parametrize("tile", [(256, 256), (128, 128), (64, 64)])
@pytest.mark.parametrize("schedule", ["persistent", "streamk"])
def test_k_remainder_of_mixed_formats(schedule, tile, types):
    gen = torch.Generator(device="cuda").manual_seed(6)
    for m, n, k in [(16, 16, 16), (tile[0] + 16, 2 * tile[1], 144), (272, 304, 592), (520, 512, 1008)]:
        a, b = _poisoned(gen, m, k, "T", types[0], 16), _poisoned(gen, k, n, "N", types[1], 16)
        c = torch.full((m, n), float("nan"), dtype=torch.float32, device="cuda")
        sel = tb.OrigamiMatmulSelector(m, n, k, *types, c.dtype, a.device, streamk=schedule == "streamk")
        sel._sel.block_m, sel._sel.block_n, sel._sel.block_k = tile[0], tile[1], 128
        tb.matmul_a8w8_lt(a, b, torch.ones(m, device="cuda"), torch.ones(n, device="cuda"), c, sel, tb.matmul_preamble(sel), enable_streamk=schedule == "streamk")
        assert torch.equal(c, (a.double() @ b.double()).float()), (m, n, k)


@pytest.mark.parametrize("k", [16, 144, 1040, 2064])
@pytest.mark.parametrize("tile", [(None, None, None), (256, 256, 128), (128, 128, 128), (64, 64, 128)])
def test_grouped_k_remainder(tile, k):
    """Experts without rows, with one, with ragged last blocks; behind every row of both operands lie NaNs."""
    gen = torch.Generator(device="cuda").manual_seed(k)
    counts, n = [70, 0, 1, 257, 300], 200
    offsets = torch.tensor([0] + counts).cumsum(0)
    a = _poisoned(gen, sum(counts), k, "T", torch.float8_e4m3fn, 16)
    w = _poisoned(gen, len(counts) * n, k, "T", torch.float8_e4m3fn, 16).unflatten(0, (len(counts), n))
    c = torch.full((sum(counts), n), float("nan"), dtype=torch.bfloat16, device="cuda")
    tb.grouped_matmul_a8w8(a, w, None, None, c, offsets.int().cuda(), *tile)
    for e, (lo, hi) in enumerate(zip(offsets.tolist(), offsets.tolist()[1:])):
        assert torch.equal(c[lo:hi], (a[lo:hi].double() @ w[e].double().T).float().to(torch.bfloat16)), e


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_k_remainder_in_more_stream_k_pieces_than_stages(dtype):
    """A tile cut into pieces of one to three K steps: the remainder lies in one piece only, the first copy stages of the others are whole."""
    chunk = 16 // dtype.itemsize
    gen = torch.Generator(device="cuda").manual_seed(7)
    for grid in (5, 17, 64):
        m, n, k = 64, 64, 17 * 8 * chunk + 3 * chunk
        a, b = _poisoned(gen, m, k, "T", dtype, chunk), _poisoned(gen, k, n, "N", dtype, chunk)
        c = torch.full((m, n), float("nan"), dtype=dtype, device="cuda")
        sel = tb.OrigamiMatmulSelector(m, n, k, dtype, dtype, dtype, a.device, streamk=True)
        sel._sel.block_m, sel._sel.block_n, sel._sel.block_k = 64, 64, 8 * chunk
        streamk_matmul_lt(a, b, c, sel, tb.matmul_preamble(sel), sk_grid=grid)
        assert torch.equal(c, (a.double() @ b.double()).float().to(dtype)), grid
