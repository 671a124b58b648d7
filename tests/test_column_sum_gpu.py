"""Column sums (a bias gradient) against the sum in 64 bits, at the edges of the row parts, of the column blocks and of the 16-byte loads.

Tolerance: half a unit in the last place of the result's type, and an fp32 rounding of the running sum per row a lane adds; sums are
of positive values, so every running sum is at most the result."""
import pytest
import torch

import tritonblas_amd as tb
from tritonblas_amd.matmul import _bias_gradient, _column_sum


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("m,n", [(1, 1), (1, 8), (17, 127), (127, 128), (128, 136), (129, 1000), (300, 2049), (2049, 64), (8200, 12),
                                 (4096, 1024), (255, 65536)])
def test_column_sum(m, n, dtype):
    x = torch.rand((m, n), device="cuda", generator=torch.Generator(device="cuda").manual_seed(m)).to(dtype)
    got, want = _column_sum(x), x.double().sum(0)
    bound = want * (torch.finfo(dtype).eps / 2 + (m / 16 + 100) * 2.0 ** -24)
    assert got.dtype == dtype and got.shape == (n,)
    assert ((got.double() - want).abs() <= bound).all()


@pytest.mark.gpu
def test_column_sum_off_sixteen_bytes_and_with_infinities():
    base = torch.rand(100 * 64 + 1, device="cuda").bfloat16()
    x = base[1:].view(100, 64)
    assert torch.equal(_column_sum(x), _column_sum(x.clone()))
    y = torch.ones(40, 24, device="cuda")
    y[3, 1], y[4, 2], y[5, 3], y[6, 3] = float("inf"), float("nan"), float("inf"), -float("inf")
    s = _column_sum(y)
    assert s[1] == float("inf") and s[2].isnan() and s[3].isnan() and (s[4:] == 40).all()


@pytest.mark.gpu
def test_bias_gradient_can_be_differentiated_again():
    x, w = (torch.randn(s, device="cuda").requires_grad_() for s in ((24, 32), (32, 40)))
    bias, g = torch.randn(40, device="cuda").requires_grad_(), torch.randn(24, 40, device="cuda").requires_grad_()
    db, = torch.autograd.grad(tb.addmm(bias, x, w), bias, g, create_graph=True)
    v = torch.randn(40, device="cuda")
    dg, = torch.autograd.grad(db, g, v)
    assert torch.equal(dg, v.expand(24, 40))


@pytest.mark.gpu
def test_more_columns_than_one_launch_has_threads_for():
    """2**28 columns and a few, 16 to a workgroup of 256 threads: HIP refuses launches of 2**32 threads and more."""
    x = torch.rand((1, 2 ** 28 + 3), device="cuda", dtype=torch.bfloat16)
    assert torch.equal(_column_sum(x), x[0])
    x = torch.rand((2, 2 ** 27 + 64), device="cuda", dtype=torch.bfloat16)
    assert torch.equal(_column_sum(x), (x[0].float() + x[1].float()).bfloat16())


@pytest.mark.gpu
def test_column_sum_of_every_way_a_matrix_is_stored():
    base = torch.randint(-9, 9, (96, 80), device="cuda").bfloat16()        # (whole numbers: exact sums)
    for x in (base.T, base[:, ::2], base[::3, 8:72], base[:1].expand(50, 80), base[:, :1].expand(96, 33), base.T[:, :1], base[:, 5:6]):
        assert torch.equal(_column_sum(x), x.double().sum(0).bfloat16())


@pytest.mark.gpu
@pytest.mark.parametrize("m,n", [(64, 128), (2048, 2040), (2048, 2056)])
def test_bias_gradient_on_both_sides_of_its_rule(m, n):
    """Sums of whole numbers below 2**24: exact on either way."""
    g = torch.randint(-9, 9, (m, n), device="cuda").float()
    assert torch.equal(_bias_gradient(g), g.double().sum(0).float())
    bias = torch.zeros(n, device="cuda", requires_grad=True)
    db, = torch.autograd.grad(tb.addmm(bias, torch.ones(m, 8, device="cuda"), torch.ones(8, n, device="cuda")), bias, g)
    assert torch.equal(db, g.double().sum(0).float())
