"""The row quantiser's kernel (tb_quantize_rows) against the same recipe written as tensor operations on the same device: codes
and scales bit for bit, at the edges of its register tiles, on misaligned and strided rows, and on values that no finite code holds."""
import pytest
import torch

import tritonblas_amd.utils as U

DTYPES8 = [torch.float8_e4m3fn, torch.float8_e5m2, torch.int8]


def _by_tensor_operations(x, dtype, axis, **kw):
    """(a tensor that autograd records takes the tensor operations)"""
    q, s = U.quantize_tensor_per_channel(x.clone(memory_format=torch.preserve_format).requires_grad_(), dtype, axis, **kw)
    return q.detach(), s.detach()


def _same(x, dtype, axis, **kw):
    assert U._plain(x) and U._rows(x, axis) is not None
    q, s = U.quantize_tensor_per_channel(x, dtype, axis, **kw)
    wq, ws = _by_tensor_operations(x, dtype, axis, **kw)
    assert q.shape == wq.shape and s.shape == ws.shape and q.dtype == dtype and s.dtype == torch.float32
    nan = torch.isnan(ws)
    assert torch.equal(torch.isnan(s), nan)
    assert torch.equal(s[~nan].view(torch.int32), ws[~nan].view(torch.int32))
    a, b = q.contiguous().view(torch.uint8), wq.contiguous().view(torch.uint8)
    if dtype != torch.int8:     # (the sign of a NaN code says nothing)
        a, b = (torch.where(torch.isnan(t.float()), torch.full_like(u, 0x7f), u) for t, u in ((q.contiguous(), a), (wq.contiguous(), b)))
    assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES8)
@pytest.mark.parametrize("src", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("shape", [(1, 1), (3, 7), (5, 4096), (2049, 1024), (2050, 4096), (300, 4104), (257, 16384), (2, 16392), (3, 32776),
                                   (2, 65536), (2, 65544), (700, 999), (1, 8), (70001, 1), (5000, 8), (4099, 9), (3001, 64), (2050, 65), (40, 5)])
def test_rows_match_the_tensor_operations(shape, src, dtype):
    g = torch.Generator(device="cuda").manual_seed(shape[0] * 7 + shape[1])
    x = (torch.randn(shape, device="cuda", generator=g) * torch.logspace(-4, 3, shape[0], device="cuda").unsqueeze(1)).to(src)
    x[shape[0] // 2] = 0
    _same(x, dtype, 1)
    _same(x.T, dtype, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES8)
def test_rows_with_strides_and_offsets(dtype):
    x = torch.randn(40, 530, device="cuda").bfloat16()
    for view in (x[:, 1:513], x[:, 8:520], x[3:, :511], x[::2, 16:272], x[:1, 5:]):
        _same(view, dtype, 1)
    _same(torch.randn(3, 5, 264, device="cuda").half(), dtype, 2)
    _same(torch.randn(3, 5, 264, device="cuda").half(), dtype, -1)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES8)
def test_rows_with_infinities_nans_and_tiny_scales(dtype):
    inf, nan = float("inf"), float("nan")
    x = torch.randn(9, 512, device="cuda")
    x[0, 3], x[1, 100], x[2, 511], x[3, 5] = inf, -inf, nan, 0.0
    x[4], x[5], x[6] = 1e-38, 1e-42, -3e38
    x[7, 7], x[7, 9] = nan, inf
    _same(x, dtype, 1)
    _same(x, dtype, 1, min_scale=0.0)
    _same(x[:, :17], dtype, 1, min_scale=3.0)


def test_what_is_recorded_keeps_the_tensor_operations():
    """Without a GPU: a CPU tensor, and a gradient through the scale."""
    x = torch.randn(4, 32, requires_grad=True)
    assert not U._plain(x)
    _, s = U.quantize_tensor_per_channel(x, torch.float8_e4m3fn, 1)
    s.sum().backward()
    assert torch.count_nonzero(x.grad) == 4


@pytest.mark.parametrize("shape,axis,want", [((4, 8), 1, (4, 8, 8)), ((4, 8), 0, None), ((2, 3, 8), 2, (6, 8, 8)), ((2, 3, 8), 1, None), ((4, 1), 1, (4, 1, 1))])
def test_which_rows_the_kernel_takes(shape, axis, want):
    x = torch.zeros(shape)
    assert U._rows(x, axis) == want
    if len(shape) == 2 and want and shape[1] > 1:
        assert U._rows(x.T, 0) == want
        assert U._rows(x[:, ::2], 1) is None
        assert U._rows(x[:1].expand(4, 8), 1) is None


@pytest.mark.gpu
def test_more_rows_than_one_launch_has_threads_for():
    """2**26 rows: HIP refuses launches of 2**32 threads and more."""
    x = torch.randn(2 ** 26 + 3, 8, device="cuda", dtype=torch.bfloat16)
    q, s = U.quantize_tensor_per_channel(x, torch.int8, 1)
    for rows in (slice(0, 4096), slice(2 ** 25 - 5, 2 ** 25 + 4096), slice(2 ** 26 - 4096, None)):
        wq, ws = _by_tensor_operations(x[rows], torch.int8, 1)
        assert torch.equal(q[rows], wq) and torch.equal(s[rows], ws)
    assert bool((s > 0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES8)
@pytest.mark.parametrize("shape", [(3, 131073), (2, 131080), (255, 147456), (256, 147456), (2, 200003), (1, (1 << 22) + 5), (1, 1 << 22)])
def test_rows_in_parts(shape, dtype):
    """Several workgroups to a row: their maxima, one scale, their codes."""
    x = torch.randn(shape, device="cuda").bfloat16()
    x[0, -1] = 9.0
    if shape[0] > 1:
        x[1, 16383], x[-1, 65536:] = float("nan") if shape[0] == 3 else -7.0, 0
    _same(x, dtype, 1)
    _same(x[:, 1:], dtype, 1)
    _same(x.float(), dtype, 1, min_scale=20.0)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES8)
@pytest.mark.parametrize("n", [64, 1000, 4096, 16384])
def test_rows_at_the_edge_of_plain_rounding(n, dtype):
    """Rows whose values cannot leave the code's range are rounded without a look at it.  At that line: magnitudes up to the largest finite float beside an infinity
    and a NaN, scales around the smallest normal number, rows of nothing but the largest magnitude."""
    top = 127.0 if dtype == torch.int8 else torch.finfo(dtype).max
    huge, tiny = torch.finfo(torch.float32).max, torch.finfo(torch.float32).tiny
    peaks = [huge, float("inf"), float("nan"), tiny * top, tiny * top * 0.999, tiny * top * 1.001, tiny * 0.5, 1.0, 0.0]
    x = torch.rand(len(peaks), n, device="cuda") * 2 - 1
    for row, peak in enumerate(peaks):
        x[row] *= min(peak, huge) if peak == peak else 1.0
        x[row, n // 3] = peak
    x[7] = torch.where(x[7] < 0, -1.0, 1.0)
    _same(x, dtype, 1, min_scale=0.0)
    _same(x, dtype, 1)
