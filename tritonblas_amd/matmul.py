"""GEMM entry points with the reference's Python signatures (include/tritonblas/matmul.py).

Each launcher fills one C descriptor and calls the shared library on torch's current stream; nothing
here computes.  ``a`` is (M, K), ``b`` is (K, N) with arbitrary 2-D strides (transposes are views),
``c`` is written in place and returned.
"""
from typing import Optional

import torch

from . import _lib
from ._lib import C
from .config import MatmulConfig, matmul_preamble
from .origami import OrigamiMatmulSelector
from .utils import _launch, _plain


_SELECTOR_CACHE = {}
_SELECTOR_CACHE_MAX = 4096
# Launch state for entry points that are called without a MatmulConfig (tb.matmul(..., enable_streamk=True)
# and friends): one workspace per (device, stream), grown on demand.  Epoch tags make zeroing between
# launches unnecessary, and launches on one stream are ordered, so they can share it.  Entries are never
# dropped: a launch captured into a HIP graph keeps the raw pointer of the workspace it was given.
_STREAM_CONFIGS = {}


def _stream_config(dev) -> MatmulConfig:
    key = (dev.index if dev.index is not None else torch.cuda.current_device(), torch.cuda.current_stream(dev).cuda_stream)
    cfg = _STREAM_CONFIGS.get(key)
    if cfg is None:
        cfg = MatmulConfig(device=dev, workspace=None)
        _STREAM_CONFIGS[key] = cfg
    return cfg


def _make_matmul_selector(M, N, K, a_dtype, b_dtype, c_dtype, device, mx_block_size=0, streamk=False,
                          num_stages: int = 2):
    """Reference matmul.py:42-66, which scores the tiles again on every call; here a selector is a pure
    function of its arguments and is kept (the entry points that build their own selector call this)."""
    key = (M, N, K, a_dtype, b_dtype, c_dtype, device, mx_block_size, bool(streamk), num_stages)
    sel = _SELECTOR_CACHE.get(key)
    if sel is None:
        if len(_SELECTOR_CACHE) >= _SELECTOR_CACHE_MAX:
            _SELECTOR_CACHE.clear()
        sel = OrigamiMatmulSelector(M, N, K, a_dtype, b_dtype, c_dtype, device, mx_block_size=mx_block_size,
                                    streamk=streamk, num_stages=num_stages)
        _SELECTOR_CACHE[key] = sel
    return sel


class _NoSwitch:
    def __enter__(self):
        return None

    def __exit__(self, *exc):
        return False


_NO_SWITCH = _NoSwitch()


def _on_device(dev):
    """Context that makes ``dev`` the current device for a launch; free when it already is."""
    if dev.index is None or _lib.current_device() == dev.index:
        return _NO_SWITCH
    return torch.cuda.device(dev)


def _ptr(t: Optional[torch.Tensor]):
    return None if t is None else C.c_void_p(t.data_ptr())


def _check_index(*tensors):
    """The index of the one GPU that all of them are on."""
    index = None
    for t in tensors:
        if t is None:
            continue
        if not t.is_cuda:
            raise RuntimeError("tritonblas_amd: tensors must live on a GPU (there is no CPU path)")
        if index is None:
            index = t.get_device()
        elif t.get_device() != index:
            raise RuntimeError("tritonblas_amd: tensors are on different devices")
    return index


def _check_device(*tensors):
    index = _check_index(*tensors)
    return None if index is None else torch.device("cuda", index)


def _empty_problem(M, N, K, c, bias=None) -> bool:
    """M, N or K of zero: torch.matmul's answer (nothing to write, or an empty sum = zeros plus the bias)
    without a launch.  True when the problem was such a one."""
    if M == 0 or N == 0:
        return True
    if K == 0:
        if bias is None:
            c.zero_()
        else:
            c.copy_(bias.reshape(1, N).to(torch.float32).expand(M, N))
        return True
    return False


def _flat_scales(a_scale, b_scale, M, N):
    if (a_scale is None) != (b_scale is None):
        raise RuntimeError("tritonblas_amd: a_scale and b_scale come together")
    if a_scale is None:
        return None, None
    if a_scale.dtype != torch.float32 or b_scale.dtype != torch.float32:
        raise RuntimeError("tritonblas_amd: scales must be float32")
    if a_scale.dim() != 1:
        a_scale = a_scale.reshape(-1)
    if b_scale.dim() != 1:
        b_scale = b_scale.reshape(-1)
    if not (a_scale.is_contiguous() and b_scale.is_contiguous() and a_scale.numel() == M and b_scale.numel() == N):
        raise RuntimeError("tritonblas_amd: a_scale must be contiguous (M,) and b_scale contiguous (N,)")
    return a_scale, b_scale


def _queue_tile(selector, dtype):
    """The tile that a work-stealing launch names, (0, 0, 0) where it leaves the choice to the library.

    The model that chose a selector's tile did not know that the tiles come from the queues, which 32x32 tiles of the 16- and 8-bit types do not suit (FP8
    256x256x7904 31.5 us, in 64x32 19; with a selector for 64 CUs 28.6 and 19)."""
    tile = selector.block_m, selector.block_n, selector.block_k
    if tile[1] != 32 or dtype == torch.float32:
        return tile
    if tile == getattr(selector, "_model_tile", None):
        return 0, 0, 0
    return (64, *tile[1:]) if tile == getattr(selector, "_part_tile", None) else tile


def _launch_gemm(a, b, c, selector, config, schedule, bias=None, a_scale=None, b_scale=None, sk_grid=None):
    M, K = a.shape
    K2, N = b.shape
    assert K == K2, "Incompatible Dimensions"
    c_shape = c.shape
    assert c_shape[0] == M and c_shape[1] == N, "Incompatible Dimensions"
    index = _check_index(a, b, c, bias, a_scale, b_scale)
    if _empty_problem(M, N, K, c, bias):
        return c
    lib = _lib.load()
    a_scale, b_scale = _flat_scales(a_scale, b_scale, M, N)
    bias_type = bias_stride = 0
    if bias is not None:
        if bias.numel() != N:
            raise AssertionError("Incompatible Dimensions")
        if bias.dim() != 1:
            bias = bias.reshape(-1)     # (1, N) and the like: one value per output column
        bias_type, bias_stride = _lib.tb_dtype(bias.dtype), bias.stride(0)
    streamk = schedule in (_lib.TB_SCHED_STREAMK, _lib.TB_SCHED_STREAMK_WS)
    a_sm, a_sk = a.stride()
    b_sk, b_sn = b.stride()
    block_m = block_n = block_k = group_m = num_xcds = counters = 0
    if selector is not None:
        block_m, block_n, block_k = selector.block_m, selector.block_n, selector.block_k
        group_m, num_xcds, counters = selector.group_m, selector.num_sms, selector.COUNTERS_PER_XCD
        # A selector knows sizes and types, not how the operands are stored.  That matters to the tile model only where K is no even number of K
        # steps: the hand-scheduled kernels take what is left behind them from K-contiguous operands whose rows start on 16 bytes, for others the model
        # has the eight-wave kernel's figures.  Then the library's own choice, the same model with the operands at hand, takes the place of a choice that is
        # the model's as well (bf16 3232x6880x2272 with a row-major b: 256x128 for a selector, 113 us, and 256x256 once the layout is told, 102).
        if (K % (2 * block_k) and not (a_sk == 1 == b_sk and (a_sm | b_sn) % 16 == 0) and not streamk
                and (block_m, block_n, block_k) == getattr(selector, "_model_tile", None)):
            block_m = block_n = block_k = group_m = 0
        elif schedule and not streamk:      # (work stealing)
            block_m, block_n, block_k = _queue_tile(selector, a.dtype)
            if block_m == 0:
                group_m = counters = 0
    grid = 0
    if selector is not None and not streamk and getattr(selector, "_total_cus", None) is not None:
        # a selector built for a CU partition sizes the launch (reference matmul.py:113: grid = N_CU):
        # as many workgroups as that many CUs hold at once; a mask (below) makes it one per mask entry
        grid = selector._N_CU * max(1, selector.waves_per_eu)
    c_strides = c.stride()
    desc = _lib.pack_gemm(
        _lib.GEMM_BYTES, _lib.tb_dtype(a.dtype), _lib.tb_dtype(b.dtype), _lib.tb_dtype(c.dtype), bias_type, M, N, K,
        a_sm, a_sk, b_sk, b_sn, c_strides[0], c_strides[1], a.data_ptr(), b.data_ptr(), c.data_ptr(),
        0 if a_scale is None else a_scale.data_ptr(), 0 if b_scale is None else b_scale.data_ptr(), 0 if bias is None else bias.data_ptr(),
        bias_stride, block_m, block_n, block_k, group_m, num_xcds, schedule, grid, counters, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0)
    if schedule == _lib.TB_SCHED_PERSISTENT:
        _launch(_lib.launch_gemm, desc, index, "tb_gemm")
        return c
    dev = a.device
    d = _lib.tb_gemm_desc.from_buffer_copy(desc)
    if schedule == _lib.TB_SCHED_WORK_STEALING and config is not None:
        # reference matmul.py:112-159: GLOBAL_ATOMIC from the config, the per-workgroup mask by program id
        if getattr(config, "hierarchical", False):
            # (the split is left to the library: it knows the tile the launch really runs, which is not
            # the selector's when the operands need the gather kernel)
            d.ws_mode = _lib.TB_WS_HIERARCHICAL
        elif config.global_atomic:
            d.ws_mode = _lib.TB_WS_GLOBAL_ATOMIC
        mask = config.active_mask()
        if mask is not None:
            if mask.dtype != torch.int32 or not mask.is_contiguous() or mask.device != dev:
                raise RuntimeError("tritonblas_amd: config.mask must be a contiguous int32 tensor on the GEMM's device")
            d.cu_mask, d.cu_mask_len = _ptr(mask), mask.numel()
            d.grid = 0
    if streamk:
        if sk_grid is not None:
            d.grid = int(sk_grid)
        elif selector is not None and selector.streamk:
            d.grid = selector.sk_grid
    # 0 bytes: the library runs this problem with a kernel that needs no workspace (or refuses the
    # descriptor, which the launch below reports)
    need = lib.tb_workspace_bytes(d)
    if need > 0:
        if config is None:
            config = _stream_config(dev)
        ws = config.ensure(need)
        d.workspace, d.workspace_bytes = C.c_void_p(ws.data_ptr()), ws.numel()
        # (the workspace tags Stream-K launches with its own count: nothing in the descriptor changes from
        # call to call, so a launch captured in a graph can be replayed)
        d.epoch = _lib.TB_EPOCH_ON_DEVICE
        d.spin_limit = int(getattr(config, "spin_limit", 0) or 0)
    with _on_device(dev):
        _lib.check(lib.tb_gemm(d, _lib.stream_handle(dev)), "tb_gemm")
    return c


def persistent_matmul_lt(a, b, c, selector, config: Optional[MatmulConfig] = None, bias=None, a_scale=None,
                         b_scale=None, quantized: bool = False, work_stealing: bool = False):
    """Data-parallel launch, optionally through the work-stealing queues (reference matmul.py:69-200)."""
    sched = _lib.TB_SCHED_WORK_STEALING if (work_stealing and config is not None) else _lib.TB_SCHED_PERSISTENT
    return _launch_gemm(a, b, c, selector, config, sched, bias=bias,
                        a_scale=a_scale if quantized else None, b_scale=b_scale if quantized else None)


def streamk_matmul_lt(a, b, c, selector, config: Optional[MatmulConfig] = None, bias=None, sk_grid=None,
                      a_scale=None, b_scale=None, quantized: bool = False, work_stealing: bool = False):
    """Stream-K launch (reference matmul.py:202-366).  ``work_stealing``: the whole tiles in front of the
    Stream-K tail are drawn from the XCD x slot queues instead of being dealt out by workgroup id (reference
    matmul.py:279-323, kernels/streamk_gemm_work_stealing.py); the tail itself is the same, and so are the
    results.  A launch that shares the device with other work can run into the poll bound of the partial-tile
    exchange (NaN tiles + the workspace's status word): callers in that situation should call
    ``config.check()`` after synchronising."""
    sched = _lib.TB_SCHED_STREAMK_WS if work_stealing else _lib.TB_SCHED_STREAMK
    return _launch_gemm(a, b, c, selector, config, sched, bias=bias, sk_grid=sk_grid,
                        a_scale=a_scale if quantized else None, b_scale=b_scale if quantized else None)


def matmul_lt(a, b, c, selector, config: MatmulConfig = None, enable_streamk=False, work_stealing=False):
    """Reference matmul.py:368-378."""
    assert a.shape[1] == b.shape[0], "Incompatible Dimensions"
    if enable_streamk:
        return streamk_matmul_lt(a, b, c, selector, config, work_stealing=work_stealing)
    return persistent_matmul_lt(a, b, c, selector, config, work_stealing=work_stealing)


def matmul_a8w8_lt(a, b, a_scale, b_scale, c, selector, config: MatmulConfig = None, enable_streamk=False,
                   work_stealing=False):
    """Reference matmul.py:380-390."""
    assert a.shape[1] == b.shape[0], "Incompatible Dimensions"
    if enable_streamk:
        return streamk_matmul_lt(a, b, c, selector, config, a_scale=a_scale, b_scale=b_scale, quantized=True)
    return persistent_matmul_lt(a, b, c, selector, config, a_scale=a_scale, b_scale=b_scale, quantized=True,
                                work_stealing=work_stealing)


def _run(a, b, out, bias, enable_streamk, sk_grid, work_stealing, out_dtype_for_selector):
    M, K = a.shape
    _, N = b.shape
    if _empty_problem(M, N, K, out, bias):
        return out
    selector = _make_matmul_selector(M, N, K, a.dtype, b.dtype, out_dtype_for_selector, a.device,
                                     streamk=bool(enable_streamk))
    config = matmul_preamble(selector, a.device) if work_stealing else None
    if enable_streamk:
        return streamk_matmul_lt(a, b, out, selector, config, bias=bias, sk_grid=sk_grid, work_stealing=work_stealing)
    return persistent_matmul_lt(a, b, out, selector, config, bias=bias, work_stealing=work_stealing)


# ---- torch custom operators (reference matmul.py:393-472, 628-752) ----------------------------------
# Registered with torch.library so that autograd and torch.compile (fullgraph) see one opaque operator
# with a shape rule (fake implementation) instead of a ctypes call they cannot trace.  The reference
# registers the same four operators with triton_op; the namespace differs so that both packages can be
# imported side by side.
def _fake_new_output(a, b):
    assert a.shape[1] == b.shape[0], "Incompatible A-B Dimensions"
    return a.new_empty(a.shape[0], b.shape[1])


@torch.library.custom_op("tritonblas_amd::_matmul", mutates_args=())
def _matmul(a: torch.Tensor, b: torch.Tensor, enable_streamk: Optional[bool] = False, sk_grid: Optional[int] = None,
            work_stealing: Optional[bool] = False) -> torch.Tensor:
    assert a.shape[1] == b.shape[0], "Incompatible A-B Dimensions"
    out = a.new_empty(a.shape[0], b.shape[1])
    _run(a, b, out, None, enable_streamk, sk_grid, work_stealing, out.dtype)
    return out


@_matmul.register_fake
def _(a, b, enable_streamk=False, sk_grid=None, work_stealing=False):
    return _fake_new_output(a, b)


def _matmul_setup_context(ctx, inputs, output):
    a, b, enable_streamk, sk_grid, work_stealing = inputs
    ctx.save_for_backward(a, b)
    ctx.opts = (enable_streamk, sk_grid, work_stealing)


def _transposed(t, g):
    """``t.T`` for a product with the contiguous gradient ``g``: as it is stored, or copied where the copy pays.

    The kernels take either index of a 16- or 32-bit operand as the contiguous one, so a copy of rows that start on 16 bytes only
    costs (4096x14336x4096 bf16: two copies, 0.32 of 1.6 ms).  Rows that do not are loaded through registers; a copy whose rows do start
    there saves that if the rows of ``g`` do too (a.T @ g of a 4096x4096x4099 bf16 product: 237 us as stored, 189 with the copy;
    1184x3000x1531 39 and 35) and is lost otherwise (1187x3001x1531: 47 and 58; g @ b.T 42 and 83)."""
    size = t.element_size()
    chunk = 16 // size
    for inner, outer in ((1, 0), (0, 1)):
        if size > 1 and t.stride(inner) == 1 and t.shape[inner] % chunk == 0 and t.stride(outer) % chunk == 0 and t.storage_offset() % chunk == 0:
            return t.T
    if size > 1 and 1 in t.stride() and (t.shape[0] % chunk or g.shape[1] % chunk):
        return t.T
    return t.T.contiguous()


def _product_gradients(a, b, g, opts):
    # two more library GEMMs: grad_a = g @ b^T, grad_b = a^T @ g
    sk, grid, ws = opts
    return (matmul(g, _transposed(b, g), enable_streamk=sk, sk_grid=grid, work_stealing=ws),
            matmul(_transposed(a, g), g, enable_streamk=sk, sk_grid=grid, work_stealing=ws))


def _matmul_backward(ctx, grad_output):
    a, b = ctx.saved_tensors
    g = grad_output.contiguous()
    grad_a, grad_b = _product_gradients(a, b, g, ctx.opts)
    return grad_a, grad_b, None, None, None


_matmul.register_autograd(_matmul_backward, setup_context=_matmul_setup_context)


@torch.library.custom_op("tritonblas_amd::_matmul_out", mutates_args={"out"})
def _matmul_out(a: torch.Tensor, b: torch.Tensor, out: torch.Tensor, enable_streamk: Optional[bool] = False,
                sk_grid: Optional[int] = None, work_stealing: Optional[bool] = False) -> None:
    assert a.shape[1] == b.shape[0], "Incompatible A-B Dimensions"
    _run(a, b, out, None, enable_streamk, sk_grid, work_stealing, out.dtype)


@_matmul_out.register_fake
def _(a, b, out, enable_streamk=False, sk_grid=None, work_stealing=False):
    assert a.shape[1] == b.shape[0], "Incompatible A-B Dimensions"
    return None


@torch.library.custom_op("tritonblas_amd::_column_sum", mutates_args=())
def _column_sum(x: torch.Tensor) -> torch.Tensor:
    """``x.sum(dim=0)`` of a matrix, formed in fp32 (a bias gradient)."""
    m, n = x.shape
    if m == 0 or n == 0 or not x.is_cuda or x.dtype not in (torch.bfloat16, torch.float16, torch.float32) or (n > 1 and x.stride(1) != 1):
        return x.sum(dim=0)         # (the kernel reads rows of adjacent values)
    out = x.new_empty(n)
    lib = _lib.load()
    with _on_device(x.device):
        need = lib.tb_column_sum_bytes(m, n)
        partial = torch.empty(need // 4, dtype=torch.float32, device=x.device)
        d = _lib.tb_column_sum_desc()
        d.struct_bytes = C.sizeof(_lib.tb_column_sum_desc)
        d.type, d.m, d.n, d.x, d.x_stride_m = _lib.tb_dtype(x.dtype), m, n, x.data_ptr(), x.stride(0)
        d.out, d.partial, d.partial_bytes = out.data_ptr(), partial.data_ptr() if need else None, need
        _lib.check(lib.tb_column_sum(d, _lib.stream_handle(x.device)), "tb_column_sum")
    return out


@_column_sum.register_fake
def _(x):
    return x.new_empty(x.shape[1])


def _column_sum_setup_context(ctx, inputs, output):
    ctx.rows = inputs[0].shape[0]


def _column_sum_backward(ctx, grad_output):
    return grad_output.expand(ctx.rows, -1)


_column_sum.register_autograd(_column_sum_backward, setup_context=_column_sum_setup_context)


@torch.library.custom_op("tritonblas_amd::_addmm", mutates_args=())
def _addmm(bias: torch.Tensor, a: torch.Tensor, b: torch.Tensor, enable_streamk: Optional[bool] = False,
           sk_grid: Optional[int] = None, work_stealing: Optional[bool] = False) -> torch.Tensor:
    assert a.shape[1] == b.shape[0], "Incompatible A-B Dimensions"
    out = a.new_empty(a.shape[0], b.shape[1])
    _run(a, b, out, bias, enable_streamk, sk_grid, work_stealing, bias.dtype)
    return out


@_addmm.register_fake
def _(bias, a, b, enable_streamk=False, sk_grid=None, work_stealing=False):
    return _fake_new_output(a, b)


def _addmm_setup_context(ctx, inputs, output):
    bias, a, b, enable_streamk, sk_grid, work_stealing = inputs
    ctx.save_for_backward(a, b)
    ctx.opts = (enable_streamk, sk_grid, work_stealing)
    ctx.bias_shape = tuple(bias.shape)


# From how many values on a bias gradient is formed by tb_column_sum.  Its operator costs the host 9 to 11 us more than torch's sum (16
# against 5 to 7), which a small step, bound by the host, pays in full (256x512x512 bf16 forward and backward 119 us by sum as it was, 128 by the operator, 113 now).  The kernel
# takes 4 to 12 us less than sum below 2**22 values, 10 (8192x512 bf16: 16.6 -> 6.6) to 170 (4096x14336: 194 -> 21) above.
_COLUMN_SUM_FROM = 1 << 22


def _bias_gradient(g):
    return _column_sum(g) if g.numel() >= _COLUMN_SUM_FROM else g.sum(dim=0)


def _addmm_backward(ctx, grad_output):
    a, b = ctx.saved_tensors
    g = grad_output.contiguous()
    grad_a, grad_b = _product_gradients(a, b, g, ctx.opts)
    return _bias_gradient(g).reshape(ctx.bias_shape), grad_a, grad_b, None, None, None


_addmm.register_autograd(_addmm_backward, setup_context=_addmm_setup_context)


@torch.library.custom_op("tritonblas_amd::_addmm_out", mutates_args={"out"})
def _addmm_out(bias: torch.Tensor, a: torch.Tensor, b: torch.Tensor, out: torch.Tensor,
               enable_streamk: Optional[bool] = False, sk_grid: Optional[int] = None,
               work_stealing: Optional[bool] = False) -> None:
    assert a.shape[1] == b.shape[0], "Incompatible A-B Dimensions"
    _run(a, b, out, bias, enable_streamk, sk_grid, work_stealing, bias.dtype)


@_addmm_out.register_fake
def _(bias, a, b, out, enable_streamk=False, sk_grid=None, work_stealing=False):
    assert a.shape[1] == b.shape[0], "Incompatible A-B Dimensions"
    return None


def matmul(a, b, out: Optional[torch.Tensor] = None, enable_streamk: Optional[bool] = False,
           sk_grid: Optional[int] = None, work_stealing: Optional[bool] = False) -> Optional[torch.Tensor]:
    """Reference matmul.py:475-495: out=None allocates and supports autograd; out=... writes in
    place, returns None and refuses tensors that require grad."""
    if out is None:
        if _plain(a, b):      # (the operator exists for autograd and the tracers; its way through torch's dispatcher costs more host time than many of these products take)
            assert a.shape[1] == b.shape[0], "Incompatible A-B Dimensions"
            out = a.new_empty(a.shape[0], b.shape[1])
            _run(a, b, out, None, enable_streamk, sk_grid, work_stealing, out.dtype)
            return out
        return _matmul(a, b, enable_streamk, sk_grid, work_stealing)
    if torch.is_grad_enabled() and (a.requires_grad or b.requires_grad or out.requires_grad):
        raise RuntimeError(
            "tritonblas.matmul(): functions with out=... arguments don't support "
            "automatic differentiation, but one of the arguments requires grad."
        )
    return _matmul_out(a, b, out, enable_streamk, sk_grid, work_stealing)


def addmm(bias, a, b, out: Optional[torch.Tensor] = None, enable_streamk: Optional[bool] = False,
          sk_grid: Optional[int] = None, work_stealing: Optional[bool] = False) -> Optional[torch.Tensor]:
    """Reference matmul.py:727-752; the bias is added per output column."""
    if out is None:
        if _plain(bias, a, b):
            assert a.shape[1] == b.shape[0], "Incompatible A-B Dimensions"
            out = a.new_empty(a.shape[0], b.shape[1])
            _run(a, b, out, bias, enable_streamk, sk_grid, work_stealing, bias.dtype)
            return out
        return _addmm(bias, a, b, enable_streamk, sk_grid, work_stealing)
    if torch.is_grad_enabled() and (bias.requires_grad or a.requires_grad or b.requires_grad or out.requires_grad):
        raise RuntimeError(
            "tritonblas.addmm(): functions with out=... arguments don't support "
            "automatic differentiation, but one of the arguments requires grad."
        )
    return _addmm_out(bias, a, b, out, enable_streamk, sk_grid, work_stealing)


def matmul_a8w8(a, b, a_scale, b_scale, c, enable_streamk=False, work_stealing=False, sk_grid=None):
    """Reference matmul.py:498-517."""
    assert a.shape[1] == b.shape[0], "Incompatible Dimensions"
    M, K = a.shape
    _, N = b.shape
    if _empty_problem(M, N, K, c):
        return c
    selector = _make_matmul_selector(M, N, K, a.dtype, b.dtype, c.dtype, a.device, streamk=bool(enable_streamk))
    config = matmul_preamble(selector, a.device) if work_stealing else None
    if enable_streamk:
        return streamk_matmul_lt(a, b, c, selector, config, sk_grid=sk_grid, a_scale=a_scale, b_scale=b_scale,
                                 quantized=True, work_stealing=work_stealing)
    return persistent_matmul_lt(a, b, c, selector, config, a_scale=a_scale, b_scale=b_scale, quantized=True,
                                work_stealing=work_stealing)


def matmul_fp4(a, b, c, a_scales, b_scales, block_m: int = None, block_n: int = None, block_k: int = None,
               group_size_m: int = 8, num_warps: int = 8, num_stages: int = 2):
    """MXFP4 GEMM (reference matmul.py:519-625).  a: (M, K/2) uint8, b: (N, K/2) uint8 (two e2m1
    codes per byte, low nibble first), scales (M|N, K/32) E8M0 bytes, c: (M, N) bf16/fp16.
    ``num_warps``/``num_stages`` are accepted for signature compatibility; the kernels fix them."""
    M, Kp = a.shape
    N = b.shape[0]
    K = Kp * 2
    assert b.shape[1] * 2 == K, f"Incompatible Dimensions: A has K={K}, B has K={b.shape[1] * 2}"
    for t in (a, b, a_scales, b_scales):
        if t.element_size() != 1:
            raise RuntimeError(f"tritonblas_amd: matmul_fp4 takes packed codes and E8M0 scales as one-byte elements, got {t.dtype}")
    if tuple(a_scales.shape) != (M, K // 32) or tuple(b_scales.shape) != (N, K // 32):
        raise RuntimeError(f"tritonblas_amd: matmul_fp4 scales must be (M, K/32) and (N, K/32), got {tuple(a_scales.shape)} and {tuple(b_scales.shape)}")
    index = _check_index(a, b, c, a_scales, b_scales)
    if M == 0 or N == 0:
        return c
    if a.stride(1) != 1 or b.stride(1) != 1:
        raise RuntimeError("tritonblas_amd: matmul_fp4 needs K-contiguous packed operands")
    tile = (0, 0, 0, 0)
    if block_m is not None:
        assert block_k % 64 == 0, "BLOCK_K must be multiple of 64 for FP4"
        tile = (block_m, block_n, block_k, group_size_m)
    _lib.load()
    desc = _lib.pack_gemm_fp4(
        _lib.FP4_BYTES, _lib.tb_dtype(c.dtype), M, N, K, a.data_ptr(), b.data_ptr(), c.data_ptr(), a.stride(0), b.stride(0), *c.stride()[:2],
        a_scales.data_ptr(), b_scales.data_ptr(), *a_scales.stride(), *b_scales.stride(), *tile, 0)
    _launch(_lib.launch_gemm_fp4, desc, index, "tb_gemm_fp4")
    return c


def grouped_matmul_a8w8(a, w, a_scale, w_scale, c, group_offsets, block_m: int = None, block_n: int = None,
                        block_k: int = None, small_rows: int = 0, enable_streamk: bool = False,
                        config: MatmulConfig = None):
    """Grouped (MoE) FP8 GEMM: rows ``group_offsets[e]:group_offsets[e+1]`` of ``a`` (M, K) meet expert
    weight ``w[e]`` (N, K); ``c[rows] = cast((a[rows] @ w[e].T) * a_scale[rows, None] * w_scale[e][None, :])``.
    ``group_offsets`` is an int32 device tensor of E+1 ascending row offsets.  No host sync: the row counts
    are only read on the device, and the tile is sized by what the average expert has of them.  ``small_rows`` > 0: an expert's last partial
    row block of at most that many rows goes to a second launch with a 32-row tile (-1: one launch; 0: one launch, with ``enable_streamk`` and no tile
    named as many as are cheaper by the row counts, decided on the device).
    ``enable_streamk``: the tiles that do not fill whole rounds of the launch grid are cut into K ranges when the
    row counts make that cheaper than one more round (decided on the device; only those tiles' summation order
    changes).  The flags and partial tiles live in ``config``'s workspace, by default the one this package keeps
    per device and stream.  Off by default: exchanging 256x256 partial tiles costs about as much as 50 K steps, so it
    only pays for long K (beyond about 8192 for FP8), and the kernel that can cut tiles is 2-3 % slower when it
    does not."""
    M, K = a.shape
    E, N, K2 = w.shape
    assert K == K2 and c.shape[0] == M and c.shape[1] == N, "Incompatible Dimensions"
    assert group_offsets.numel() == E + 1 and group_offsets.dtype == torch.int32
    if a.dtype != torch.float8_e4m3fn or w.dtype != torch.float8_e4m3fn:
        raise RuntimeError(f"tritonblas_amd: grouped GEMM takes float8_e4m3fn operands, got {a.dtype} and {w.dtype}")
    dev = _check_device(a, w, c, a_scale, w_scale, group_offsets)
    if M == 0 or N == 0:
        return c
    if a.stride(1) != 1 or w.stride(2) != 1:
        raise RuntimeError("tritonblas_amd: grouped GEMM needs K-contiguous operands")
    d = _lib.tb_grouped_gemm_desc()
    d.struct_bytes = C.sizeof(_lib.tb_grouped_gemm_desc)
    d.c_type = _lib.tb_dtype(c.dtype)
    d.m_total, d.n, d.k, d.num_groups = M, N, K, E
    d.a, d.w, d.c = _ptr(a), _ptr(w), _ptr(c)
    d.a_stride_m, d.w_stride_g, d.w_stride_n = a.stride(0), w.stride(0), w.stride(1)
    d.c_stride_m, d.c_stride_n = c.stride(0), c.stride(1)
    if a_scale is not None:
        a_scale, w_scale = a_scale.reshape(-1), w_scale.reshape(E, N)
        if not (a_scale.is_contiguous() and w_scale.is_contiguous()):
            raise RuntimeError("tritonblas_amd: scales must be contiguous")
        d.a_scale, d.w_scale = _ptr(a_scale), _ptr(w_scale)
    d.group_offsets = _ptr(group_offsets)
    if block_m is not None:
        d.block_m, d.block_n, d.block_k = block_m, block_n, block_k
    d.small_rows = small_rows
    with _on_device(dev):
        lib = _lib.load()
        if enable_streamk:
            d.streamk = 1
            need = lib.tb_grouped_workspace_bytes(d)
            if need:
                cfg = config if config is not None else _stream_config(dev)
                ws = cfg.ensure(need)
                d.workspace, d.workspace_bytes = ws.data_ptr(), ws.numel()
                d.epoch, d.spin_limit = _lib.TB_EPOCH_ON_DEVICE, cfg.spin_limit
            else:
                d.streamk = 0
        _lib.check(lib.tb_grouped_gemm_fp8(d, _lib.stream_handle(dev)), "tb_grouped_gemm_fp8")
    return c
