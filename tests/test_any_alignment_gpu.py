"""Operands whose rows start anywhere (16-byte loads through registers): every storage order and tile at sizes around the tiles, the 16-byte
chunks and the K steps, inside buffers whose other values are NaN.  Values are small whole numbers: the sums are exact."""
import pytest
import torch

import tritonblas_amd as tb

pytestmark = pytest.mark.gpu


def _inside_nans(gen, rows, cols, order, dtype, pad, lead):
    r, c = (rows, cols) if order == "T" else (cols, rows)
    base = torch.full((r * (c + pad) + lead + 8,), float("nan"), device="cuda", dtype=dtype)
    x = base[lead:lead + r * (c + pad)].view(r, c + pad)[:, :c]
    x.copy_(torch.randint(-9, 9, (r, c), device="cuda", generator=gen))
    return x if order == "T" else x.T


SIZES = [(8, 8, 8), (9, 11, 13), (64, 65, 63), (129, 127, 65), (130, 70, 131), (71, 257, 200), (1187, 301, 153)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("ta,tb_", [("T", "T"), ("T", "N"), ("N", "T"), ("N", "N")])
@pytest.mark.parametrize("pad,lead", [(0, 0), (3, 1), (8, 5)])
def test_any_alignment(pad, lead, ta, tb_, dtype):
    gen = torch.Generator(device="cuda").manual_seed(9)
    for m, n, k in SIZES:
        a, b = _inside_nans(gen, m, k, ta, dtype, pad, lead), _inside_nans(gen, k, n, tb_, dtype, pad, lead)
        want = (a.double() @ b.double()).float().to(dtype)
        assert torch.equal(tb.matmul(a, b), want), (m, n, k)
        assert torch.equal(tb.matmul(a, b, enable_streamk=True), want), (m, n, k, "stream-k")
        assert torch.equal(tb.matmul(a, b, work_stealing=True), want), (m, n, k, "work stealing")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (3, 5, 100), (100, 5, 3), (100, 3, 100), (7, 100, 7)])
def test_indices_shorter_than_a_chunk_and_other_strides(m, n, k, dtype):
    gen = torch.Generator(device="cuda").manual_seed(9)
    for ta in "TN":
        for tb_ in "TN":
            a, b = _inside_nans(gen, m, k, ta, dtype, 1, 1), _inside_nans(gen, k, n, tb_, dtype, 1, 1)
            assert torch.equal(tb.matmul(a, b), (a.double() @ b.double()).float().to(dtype))
    a, b = torch.ones(m, 2 * k, device="cuda", dtype=dtype)[:, ::2], torch.ones(1, n, device="cuda", dtype=dtype).expand(k, n)
    assert (tb.matmul(a, b) == k).all()


@pytest.mark.parametrize("pad,lead", [(0, 0), (3, 5)])
@pytest.mark.parametrize("m,n,k", [(1, 1, 32), (65, 63, 96), (128, 130, 480), (200, 70, 544), (33, 257, 1056), (300, 260, 4128)])
def test_mxfp4_rows_and_scales_at_any_alignment(m, n, k, pad, lead):
    from tritonblas_amd.utils import e8m0_to_f32, mxfp4_to_f32
    gen = torch.Generator(device="cuda").manual_seed(k)

    def rows(count, width, lo, hi, fill):
        base = torch.full((count * (width + pad) + lead,), fill, device="cuda", dtype=torch.uint8)
        x = base[lead:].view(count, width + pad)[:, :width]
        x.copy_(torch.randint(lo, hi, (count, width), device="cuda", generator=gen))
        return x

    # (what lies between the rows: scale byte 255 is NaN)
    a, b = rows(m, k // 2, 0, 256, 0x77), rows(n, k // 2, 0, 256, 0x77)
    sa, sb = rows(m, k // 32, 126, 129, 255), rows(n, k // 32, 126, 129, 255)
    c = torch.full((m, n), float("nan"), device="cuda", dtype=torch.bfloat16)
    tb.matmul_fp4(a, b, c, sa, sb)
    full = [mxfp4_to_f32(x.contiguous()).double() * e8m0_to_f32(s.contiguous()).double().repeat_interleave(32, 1) for x, s in ((a, sa), (b, sb))]
    # (multiples of 1/16 below 2**16 * 144: the sums are exact)
    assert torch.equal(c, (full[0] @ full[1].T).float().to(torch.bfloat16))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_operands_stored_backwards(dtype):
    """Negative strides, which the C interface takes (torch has none): the operands' K runs from the last stored row to the first."""
    import ctypes as C
    from tritonblas_amd import _lib
    m, n, k = 136, 72, 96
    gen = torch.Generator(device="cuda").manual_seed(9)
    a, b = (torch.randint(-9, 9, (k, s), device="cuda", generator=gen).to(dtype) for s in (m, n))
    c = torch.empty(m, n, device="cuda", dtype=dtype)
    d = _lib.tb_gemm_desc()
    d.struct_bytes = C.sizeof(_lib.tb_gemm_desc)
    d.a_type = d.b_type = d.c_type = _lib.tb_dtype(dtype)
    d.m, d.n, d.k = m, n, k
    d.a_stride_m, d.a_stride_k, d.b_stride_k, d.b_stride_n, d.c_stride_m, d.c_stride_n = 1, -m, n, 1, n, 1
    d.a, d.b, d.c = a[-1].data_ptr(), b.data_ptr(), c.data_ptr()
    assert _lib.load().tb_gemm(d, _lib.stream_handle()) == _lib.TB_OK
    assert torch.equal(c, (a.flip(0).double().T @ b.double()).float().to(dtype))
    d.a_stride_k, d.a, d.b_stride_k, d.b = m, a.data_ptr(), -n, b[-1].data_ptr()
    assert _lib.load().tb_gemm(d, _lib.stream_handle()) == _lib.TB_OK
    assert torch.equal(c, (a.double().T @ b.flip(0).double()).float().to(dtype))


def test_rows_further_apart_than_32_bit_offsets_reach():
    """64 rows of 32 MiB and more: the gather kernel, for bf16 and for MXFP4 (whose other operands all take 16-byte loads)."""
    from tritonblas_amd.utils import e8m0_to_f32, mxfp4_to_f32
    m, n, pitch = 66, 40, (1 << 25) + 64
    gen = torch.Generator(device="cuda").manual_seed(3)
    base = torch.empty(m * pitch, device="cuda", dtype=torch.uint8)
    k = 136
    a = base.view(torch.bfloat16).as_strided((m, k), (pitch // 2, 1))
    a.copy_(torch.randint(-9, 9, (m, k), device="cuda", generator=gen))
    b = torch.randint(-9, 9, (n, k), device="cuda", generator=gen).bfloat16().T
    assert torch.equal(tb.matmul(a, b), (a.double() @ b.double()).float().bfloat16())
    k = 544
    codes = base.as_strided((m, k // 2), (pitch, 1))
    codes.copy_(torch.randint(0, 256, (m, k // 2), device="cuda", generator=gen))
    w = torch.randint(0, 256, (n, k // 2), device="cuda", generator=gen).to(torch.uint8)
    sa, sw = (torch.randint(126, 129, (r, k // 32), device="cuda", generator=gen).to(torch.uint8) for r in (m, n))
    c = torch.full((m, n), float("nan"), device="cuda", dtype=torch.bfloat16)
    tb.matmul_fp4(codes, w, c, sa, sw)
    full = [mxfp4_to_f32(x.contiguous()).double() * e8m0_to_f32(s).double().repeat_interleave(32, 1) for x, s in ((codes, sa), (w, sw))]
    assert torch.equal(c, (full[0] @ full[1].T).float().to(torch.bfloat16))      # (exact sums, as above)
