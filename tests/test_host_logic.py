"""Host-side logic that needs no GPU: the LDS model and Stream-K grid model restated from the
reference, the shared library's exports, the analytical selector, and argument validation."""
import ctypes as C
import os
import re

import pytest
import numpy as np
import torch

from oracle import selector as O

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


# --- LDS model: the reference's known answers (tests/test_lds_estimation.py:44-150) --------------
@pytest.mark.parametrize("args,want", [
    ((128, 128, 64, 2, 2, 1), 128 * 64 * 2), ((256, 64, 64, 2, 2, 1), 256 * 64 * 2), ((64, 256, 64, 2, 2, 1), 64 * 256 * 2),
    ((128, 128, 64, 2, 2, 2), 32768), ((256, 256, 64, 2, 2, 2), 65536), ((128, 128, 64, 2, 2, 3), 65536),
    ((128, 64, 64, 2, 2, 2), 24576), ((256, 128, 64, 2, 2, 2), 49152), ((64, 64, 32, 2, 2, 2), 8192),
    ((128, 256, 64, 2, 2, 2), 49152), ((64, 64, 32, 4, 4, 2), 16384), ((128, 128, 32, 4, 4, 2), 32768),
    ((128, 128, 64, 4, 4, 2), 65536), ((128, 128, 64, 1, 2, 2), 24576), ((128, 128, 64, 0.5, 0.5, 2), 8192),
])
def test_lds_known_answers(args, want):
    from tritonblas_amd.origami import estimate_triton_lds_bytes
    assert O.estimate_lds_bytes(*args) == want
    assert estimate_triton_lds_bytes(*args) == want


def test_lds_capacity_known_answers():
    from tritonblas_amd.origami import check_triton_lds_capacity
    for fn in (O.check_lds_capacity, check_triton_lds_capacity):
        assert fn(64, 64, 32, 2, 2, 65536, 2) is True
        assert fn(256, 256, 64, 4, 4, 65536, 2) is False
        assert fn(256, 256, 64, 2, 2, 65536, 2) is True
        assert fn(128, 128, 64, 2, 2, 65536, 3) is True
        assert fn(128, 128, 64, 2, 2, 65536, 4) is False
        assert fn(128, 128, 64, 0.5, 0.5, 0, 2) is False


def test_reference_sk_grid_model_hand_checked():
    # 8192^2 output with 256^2 tiles on 256 CUs: 1024 tiles, first fraction gives 256, 1024 % 256 == 0
    assert O.compute_sk_grid(8192, 8192, 8192, 256, 256, 64, 256) == 256
    # decode shape with a 256-wide tile: 32 tiles < 256 CUs, k split by 8 -> 256 (divides? 32 % 256 != 0 -> tiles)
    assert O.compute_sk_grid(32, 8192, 28672, 256, 256, 128, 256) == 32
    # a non-divisor candidate falls back to the tile count
    assert O.compute_sk_grid(4864, 8192, 4160, 256, 256, 64, 256) == 19 * 32
    # 608 tiles on 304 CUs: the first fraction gives 304, which divides the tile count
    assert O.compute_sk_grid(4864, 8192, 4160, 256, 256, 64, 304) == 304
    # gfx942-only override: 1024 tiles on 304 CUs leave a last wave of 112 (< 128) -> 256
    assert O.compute_sk_grid(8192, 8192, 8192, 256, 256, 64, 304) == 256
    assert [O.ws_counters_per_xcd(t) for t in (1, 512, 513, 1536, 1537, 2048, 2049)] == [8, 8, 4, 4, 2, 2, 1]


# --- shared library ------------------------------------------------------------------------------
def _header_symbols():
    text = open(os.path.join(ROOT, "include", "tritonblas_amd.h")).read()
    return sorted(set(re.findall(r"\b(tb_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    from tritonblas_amd import _lib
    lib = _lib.load()
    syms = _header_symbols()
    assert set(syms) == set(_lib.EXPORTED_SYMBOLS)
    for s in syms:
        assert hasattr(lib, s), s
    assert lib.tb_abi_version() == 1
    assert _lib.status_string(0) == "ok" and _lib.status_string(-2) == "Incompatible Dimensions"


def test_struct_sizes_match_the_header():
    """ctypes mirrors vs the C compiler's layout (compiled here with gcc)."""
    import subprocess
    import tempfile
    from tritonblas_amd import _lib
    src = '#include <stdio.h>\n#include "tritonblas_amd.h"\nint main(){printf("%zu %zu %zu %zu %zu %zu %zu %zu %zu %zu\\n",' \
          'sizeof(tb_hw),sizeof(tb_problem),sizeof(tb_selection),sizeof(tb_gemm_desc),sizeof(tb_gemm_fp4_desc),' \
          'sizeof(tb_grouped_gemm_desc),sizeof(tb_quant_desc),sizeof(tb_row_quant_desc),sizeof(tb_column_sum_desc),' \
          'sizeof(tb_launch_info));return 0;}'
    with tempfile.TemporaryDirectory() as td:
        open(os.path.join(td, "s.c"), "w").write(src)
        subprocess.check_call(["gcc", "-I", os.path.join(ROOT, "include"), "-o", os.path.join(td, "s"), os.path.join(td, "s.c")])
        sizes = [int(v) for v in subprocess.check_output([os.path.join(td, "s")]).split()]
    mine = [C.sizeof(t) for t in (_lib.tb_hw, _lib.tb_problem, _lib.tb_selection, _lib.tb_gemm_desc, _lib.tb_gemm_fp4_desc,
                                  _lib.tb_grouped_gemm_desc, _lib.tb_quant_desc, _lib.tb_row_quant_desc, _lib.tb_column_sum_desc, _lib.tb_launch_info)]
    assert mine == sizes


def test_default_hardware_is_mi355x():
    from tritonblas_amd import _lib
    hw = _lib.tb_hw()
    assert _lib.load().tb_device_info(-1, hw) == 0
    assert (hw.n_cu, hw.num_xcd, hw.cu_per_xcd, hw.lds_bytes, hw.arch) == (256, 8, 32, 163840, b"gfx950")


def test_selector_properties_and_lds_fit():
    """Mirror of the reference's only selector pin (tests/test_lds_estimation.py:211-228): the chosen
    tile fits the LDS of the part; plus the attribute surface the launchers read."""
    import tritonblas_amd as tb
    from tritonblas_amd import _lib
    for shape, dt, bits in [((8192, 28672, 8192), torch.float8_e4m3fn, 8), ((8192, 8192, 8192), torch.bfloat16, 16),
                            ((1024, 1024, 1024), torch.float16, 16), ((8192, 8192, 16384), "f4", 4), ((15, 17, 512), torch.bfloat16, 16)]:
        for sk in (False, True):
            s = tb.OrigamiMatmulSelector(*shape, dt, dt, torch.bfloat16, torch.device("cuda"), streamk=sk)
            assert s._hardware.N_CU == 256 and s._hardware.NUM_XCD == 8 and s._hardware.lds_capacity == 163840
            assert s._hardware.arch.name == "gfx950" and s._N_CU == 256 and s._ACTIVE_CU == 256
            assert s._sel.lds_bytes <= s._hardware.lds_capacity
            n = _lib.load().tb_list_tiles(_lib.tb_dtype(dt), None, 0)
            buf = (C.c_int32 * (3 * n))()
            _lib.load().tb_list_tiles(_lib.tb_dtype(dt), buf, n)
            tiles = {(buf[3 * i], buf[3 * i + 1], buf[3 * i + 2]) for i in range(n)}
            assert (s.block_m, s.block_n, s.block_k) in tiles
            assert s.group_m == min(8, -(-shape[0] // s.block_m)) and s.num_sms == 8
            assert s.even_k == (shape[2] % s.block_k == 0)
            assert s.sk_grid >= 1 and s.num_stages >= 2 and s.waves_per_eu >= 1
            total = -(-shape[0] // s.block_m) * -(-shape[1] // s.block_n)
            assert s.COUNTERS_PER_XCD == O.ws_counters_per_xcd(total)


def test_streamk_whole_tiles_answer_survives_the_resident_clamp():
    """FP8 2048x14336x4096 with 256x256 tiles: 448 tiles on 256 resident workgroups, and the model says
    that a second round of whole tiles beats a shared tail (its answer is the tile count, 448).  A
    launch that asks for that grid, or for none, must then run whole tiles only -- which shows as a
    Stream-K descriptor that needs no workspace -- and not a 256-workgroup grid with 192 shared tiles."""
    import tritonblas_amd as tb
    from tritonblas_amd import _lib
    m, n, k = 2048, 14336, 4096
    s = tb.OrigamiMatmulSelector(m, n, k, torch.float8_e4m3fn, torch.float8_e4m3fn, torch.bfloat16, torch.device("cuda"), streamk=True)
    assert (s.block_m, s.block_n) == (256, 256) and s.sk_grid == 448
    for grid in (0, 448):
        d = _lib.tb_gemm_desc()
        d.struct_bytes = C.sizeof(_lib.tb_gemm_desc)
        d.a_type = d.b_type = _lib.tb_dtype(torch.float8_e4m3fn)
        d.c_type = _lib.tb_dtype(torch.bfloat16)
        d.m, d.n, d.k = m, n, k
        d.a_stride_m, d.a_stride_k, d.b_stride_n, d.b_stride_k, d.c_stride_m, d.c_stride_n = k, 1, k, 1, n, 1
        d.block_m, d.block_n, d.block_k = 256, 256, 128
        d.schedule, d.grid = _lib.TB_SCHED_STREAMK, grid
        assert _lib.load().tb_workspace_bytes(d) == 0
    d.grid = 256      # an explicit resident grid still shares the 192-tile tail
    assert _lib.load().tb_workspace_bytes(d) > 256 * 256 * 256 * 4


def test_argument_validation_without_a_gpu():
    from tritonblas_amd import _lib
    lib = _lib.load()
    assert lib.tb_gemm(None, None) == _lib.TB_ERR_NULL_POINTER
    d = _lib.tb_gemm_desc()
    assert lib.tb_gemm(d, None) == _lib.TB_ERR_BAD_ARGUMENT          # struct_bytes not set
    d.struct_bytes = C.sizeof(_lib.tb_gemm_desc)
    d.a_type, d.b_type = _lib.TB_F16, _lib.TB_BF16
    assert lib.tb_gemm(d, None) == _lib.TB_ERR_BAD_DTYPE
    d.b_type = _lib.TB_F16
    assert lib.tb_gemm(d, None) == _lib.TB_ERR_NULL_POINTER
    q = _lib.tb_quant_desc()
    q.struct_bytes = C.sizeof(_lib.tb_quant_desc)
    assert lib.tb_hadamard_mxfp4_quant(q, None) == _lib.TB_ERR_NULL_POINTER
    assert lib.tb_select(None, None, None) == _lib.TB_ERR_NULL_POINTER
    with pytest.raises(AssertionError, match="Incompatible Dimensions"):
        _lib.check(_lib.TB_ERR_BAD_SHAPE)
    with pytest.raises(RuntimeError):
        _lib.check(_lib.TB_ERR_BAD_TILE)


def test_grouped_descriptor_validation_and_workspace_size_without_a_gpu():
    """The grouped entry point's checks that need no device, and the workspace a Stream-K tail asks for: the flags
    and one fp32 256x256 partial tile per workgroup of a 256-CU grid when the 4-wave kernel can take it (K a
    multiple of 512), nothing otherwise."""
    from tritonblas_amd import _lib
    lib = _lib.load()
    g = _lib.tb_grouped_gemm_desc()
    assert lib.tb_grouped_gemm_fp8(g, None) == _lib.TB_ERR_BAD_ARGUMENT    # struct_bytes not set
    g.struct_bytes = C.sizeof(_lib.tb_grouped_gemm_desc)
    assert lib.tb_grouped_gemm_fp8(g, None) == _lib.TB_ERR_NULL_POINTER
    g.a = g.w = g.c = g.group_offsets = 256                                # (never dereferenced: the checks below fail first)
    g.c_type = _lib.TB_BF16
    g.m_total, g.n, g.k, g.num_groups = 8192, 14336, 4096, 8
    g.a_stride_m, g.w_stride_g, g.w_stride_n, g.c_stride_m, g.c_stride_n = 4096, 14336 * 4096, 4096, 14336, 1
    g.streamk = 2
    assert lib.tb_grouped_gemm_fp8(g, None) == _lib.TB_ERR_BAD_ARGUMENT
    g.streamk = 0
    g.small_rows = -2
    assert lib.tb_grouped_gemm_fp8(g, None) == _lib.TB_ERR_BAD_ARGUMENT
    g.small_rows = -1
    assert lib.tb_grouped_workspace_bytes(g) == 0                          # no Stream-K tail asked for
    g.streamk = 1
    _, flags_off = _lib.workspace_layout()
    assert lib.tb_grouped_workspace_bytes(g) == flags_off + 1024 + 256 * 256 * 256 * 4
    g.k = 4096 + 128                                                       # an odd number of K steps: 8-wave kernel, whole tiles
    g.a_stride_m = g.w_stride_n = g.k
    g.w_stride_g = 14336 * g.k
    assert lib.tb_grouped_workspace_bytes(g) == 0


@pytest.mark.parametrize("a_type,m,n,k,a_pitch,n_major,tile,grid,small", [
    (1, 4352, 4096, 4104, 4104, False, (256, 256, 64), 200, True),       # bf16, a remainder of K
    (1, 4352, 4096, 4097, 4097, False, (256, 256, 64), 200, True),       # rows off 16 bytes
    (4, 4352, 4096, 4096, 4096, True, (256, 256, 32), 200, True),        # fp32, N-contiguous weight
    (1, 4352, 4096, 4096, 4096, False, (256, 256, 64), 200, False),      # whole K steps: refused by tb_gemm
])
def test_launch_info_of_stream_k_in_a_workspace_that_is_too_small(a_type, m, n, k, a_pitch, n_major, tile, grid, small):
    from tritonblas_amd import _lib
    lib = _lib.load()
    d = _lib.tb_gemm_desc()
    d.struct_bytes = C.sizeof(_lib.tb_gemm_desc)
    d.a_type = d.b_type = d.c_type = a_type
    d.m, d.n, d.k = m, n, k
    d.a_stride_m, d.a_stride_k = a_pitch, 1
    d.b_stride_k, d.b_stride_n = (n, 1) if n_major else (1, a_pitch)
    d.c_stride_m, d.c_stride_n = n, 1
    d.a = d.b = d.c = 1 << 20
    d.block_m, d.block_n, d.block_k = tile
    d.schedule, d.grid = _lib.TB_SCHED_STREAMK, grid
    info = _lib.tb_launch_info()
    assert lib.tb_gemm_launch_info(d, C.byref(info)) == _lib.TB_OK
    assert info.mode == 2 and info.block_m >= 128 and lib.tb_workspace_bytes(d) > 8 << 20
    d.workspace, d.workspace_bytes = 1 << 20, 8 << 20
    assert lib.tb_gemm_launch_info(d, C.byref(info)) == _lib.TB_OK
    assert info.mode == 2 and info.grid == grid and (info.block_m, info.block_n) == ((64, 64) if small else tile[:2])


@pytest.mark.parametrize("dtype", [0, 1, 4])
def test_operands_stored_backwards_are_planned_for_the_gather_kernel(dtype):
    """The vector loaders' lane offsets are unsigned: a negative stride belongs to the element-wise kernel (64x64), whichever operand
    and index has it."""
    from tritonblas_amd import _lib
    lib, n = _load(), 4096
    for strides in [(1, -n, 1, n), (1, n, -n, 1), (n, 1, -n, 1), (-n, 1, 1, n), (n, -1, 1, n), (-1, n, n, 1)]:
        d = _lib.tb_gemm_desc()
        d.struct_bytes = C.sizeof(_lib.tb_gemm_desc)
        d.a_type = d.b_type = d.c_type = dtype
        d.m = d.n = d.k = n
        d.a_stride_m, d.a_stride_k, d.b_stride_k, d.b_stride_n = strides
        d.c_stride_m, d.c_stride_n = n, 1
        d.a = d.b = d.c = 1 << 40
        info = _lib.tb_launch_info()
        assert lib.tb_gemm_launch_info(d, C.byref(info)) == _lib.TB_OK
        assert (info.block_m, info.block_n) == (64, 64), strides


def test_python_api_refuses_cpu_tensors():
    import tritonblas_amd as tb
    a = torch.zeros(16, 16, dtype=torch.float16)
    with pytest.raises(AssertionError, match="Incompatible Dimensions"):
        tb.matmul_lt(a, torch.zeros(8, 16, dtype=torch.float16), a, None, None)
    with pytest.raises(RuntimeError, match="GPU"):
        tb.matmul_lt(a, a, a.clone(), None, None)
    with pytest.raises(RuntimeError, match="differentiation"):
        tb.matmul(a.requires_grad_(), a, out=torch.zeros(16, 16, dtype=torch.float16))


@pytest.mark.parametrize("rows,cols,pitch,g_cols,copied", [
    (64, 72, 72, 40, False), (64, 72, 72, 41, False),      # rows on 16 bytes
    (64, 73, 73, 40, True), (64, 72, 73, 40, True),        # off them, the copy's on them, the gradient's too
    (64, 73, 73, 41, False), (65, 73, 73, 40, False),      # the gradient's or the copy's off them as well
])
def test_which_operands_of_the_backward_pass_are_copied(rows, cols, pitch, g_cols, copied):
    from tritonblas_amd.matmul import _transposed
    g = torch.zeros(3, g_cols, dtype=torch.bfloat16)
    t = torch.zeros(rows, pitch, dtype=torch.bfloat16)[:, :cols]
    assert (_transposed(t, g).data_ptr() != t.data_ptr()) == copied and torch.equal(_transposed(t, g), t.T)
    t = torch.zeros(2 * rows, 2 * pitch, dtype=torch.bfloat16)[::2, ::2]
    assert _transposed(t, g).is_contiguous()               # (no unit stride: the element-wise kernel otherwise)


# ---- tile order of the kernels (host evaluation through the C ABI) -------------------------------
import itertools


def _load():
    from tritonblas_amd import _lib
    return _lib.load()


def _coords(lib, t, tm, tn, gm, panel):
    pm, pn = C.c_int32(-1), C.c_int32(-1)
    assert lib.tb_tile_coords(t, tm, tn, gm, panel, C.byref(pm), C.byref(pn)) == 0
    return pm.value, pn.value


@pytest.mark.parametrize("tm,tn,gm", [(32, 112, 8), (4, 4, 8), (5, 7, 2), (1, 9, 8), (9, 1, 4), (13, 3, 8)])
def test_tile_order_without_panels_is_the_reference_swizzle(tm, tn, gm):
    from oracle import schedule as S
    lib = _load()
    for panel in (0, tn, tn + 5):
        assert [_coords(lib, t, tm, tn, gm, panel) for t in range(tm * tn)] == [S.tile_coords(t, tm, tn, gm) for t in range(tm * tn)]


@pytest.mark.parametrize("tm,tn,gm,panel", [(32, 112, 8, 16), (32, 112, 8, 32), (5, 7, 2, 3), (13, 30, 8, 4), (3, 9, 8, 1), (7, 10, 4, 9)])
def test_tile_order_with_panels_is_a_bijection_panel_by_panel(tm, tn, gm, panel):
    lib = _load()
    got = [_coords(lib, t, tm, tn, gm, panel) for t in range(tm * tn)]
    assert set(got) == set(itertools.product(range(tm), range(tn)))
    # panels are visited left to right, each completely before the next; inside a panel the order is
    # the reference swizzle of a (tm x width) problem
    from oracle import schedule as S
    pos = 0
    for first in range(0, tn, panel):
        width = min(panel, tn - first)
        want = [(m, first + n) for (m, n) in (S.tile_coords(t, tm, width, gm) for t in range(tm * width))]
        assert got[pos:pos + tm * width] == want
        pos += tm * width


def test_tile_coords_rejects_bad_arguments():
    from tritonblas_amd._lib import TB_ERR_BAD_ARGUMENT, TB_ERR_NULL_POINTER
    lib = _load()
    pm, pn = C.c_int32(), C.c_int32()
    assert lib.tb_tile_coords(12, 3, 4, 8, 0, C.byref(pm), C.byref(pn)) == TB_ERR_BAD_ARGUMENT
    assert lib.tb_tile_coords(0, 3, 4, 0, 0, C.byref(pm), C.byref(pn)) == TB_ERR_BAD_ARGUMENT
    assert lib.tb_tile_coords(0, 3, 4, 8, 0, None, C.byref(pn)) == TB_ERR_NULL_POINTER


def test_default_panel_is_a_near_square_multiple_of_the_xcd_block():
    lib = _load()
    assert lib.tb_default_panel(256, 32, 8) == 16     # 8 XCD blocks of 8x4 tiles -> rounds of 16x16
    assert lib.tb_default_panel(512, 64, 8) == 24
    assert lib.tb_default_panel(1, 1, 1) == 1
    assert lib.tb_default_panel(7, 1, 8) == 3


# ---- torch custom operators: registration and shape rules (no GPU needed) -------------------------
def test_custom_ops_are_registered_with_the_reference_signatures():
    import tritonblas_amd  # noqa: F401  (registers the operators)
    ops = torch.ops.tritonblas_amd
    assert str(ops._matmul.default._schema) == ("tritonblas_amd::_matmul(Tensor a, Tensor b, bool? enable_streamk=False, "
                                                "SymInt? sk_grid=None, bool? work_stealing=False) -> Tensor")
    assert "Tensor(a2!) out" in str(ops._matmul_out.default._schema) and str(ops._matmul_out.default._schema).endswith("-> ()")
    assert str(ops._addmm.default._schema).startswith("tritonblas_amd::_addmm(Tensor bias, Tensor a, Tensor b,")
    assert "Tensor(a3!) out" in str(ops._addmm_out.default._schema)


def test_custom_op_fake_implementations_propagate_shapes():
    import tritonblas_amd as tb
    from torch._subclasses.fake_tensor import FakeTensorMode
    with FakeTensorMode():
        a = torch.empty(64, 32, device="cuda", dtype=torch.bfloat16)
        b = torch.empty(32, 48, device="cuda", dtype=torch.bfloat16)
        bias = torch.empty(48, device="cuda", dtype=torch.bfloat16)
        c = tb.matmul(a, b)
        assert tuple(c.shape) == (64, 48) and c.dtype == torch.bfloat16 and c.device.type == "cuda"
        assert tuple(tb.addmm(bias, a, b, enable_streamk=True).shape) == (64, 48)
        out = torch.empty(64, 48, device="cuda", dtype=torch.bfloat16)
        assert tb.matmul(a, b, out=out) is None and tb.addmm(bias, a, b, out=out) is None
        with pytest.raises(Exception, match="Incompatible A-B Dimensions"):
            tb.matmul(a, torch.empty(31, 48, device="cuda", dtype=torch.bfloat16))


# ---- work-stealing queues (host evaluation through the C ABI) ------------------------------------
from oracle import schedule as OS

TB_WS_QUEUES, TB_WS_GLOBAL_ATOMIC, TB_WS_HIERARCHICAL = 0, 1, 2


def _queue(lib, mode, q, total, X, S, local):
    cnt, tile = C.c_int32(-1), C.c_int32(-1)
    assert lib.tb_ws_queue_tile(mode, q, 0, total, X, S, local, C.byref(cnt), C.byref(tile)) == 0
    out = []
    for i in range(cnt.value):
        c2 = C.c_int32(-1)
        assert lib.tb_ws_queue_tile(mode, q, i, total, X, S, local, C.byref(c2), C.byref(tile)) == 0
        assert c2.value == cnt.value
        out.append(tile.value)
    assert lib.tb_ws_queue_tile(mode, q, cnt.value, total, X, S, local, C.byref(c2 if cnt.value else cnt), C.byref(tile)) == 0
    assert tile.value == -1
    return out


@pytest.mark.parametrize("total,X,S", [(1, 8, 4), (7, 8, 1), (64, 8, 8), (1000, 8, 4), (3584, 8, 1), (333, 4, 2), (50, 1, 3)])
def test_ws_flat_queues_follow_the_reference_ranges_and_cover_every_tile_once(total, X, S):
    lib = _load()
    seen = []
    for pid in range(X * S):   # workgroups 0..X*S-1 sit on distinct queues
        q, first, bound = OS.ws_slot_range(pid, total, X, S)
        got = _queue(lib, TB_WS_QUEUES, q, total, X, S, 0)
        assert got == list(range(first, first + bound))
        seen += got
    assert sorted(seen) == list(range(total))


@pytest.mark.parametrize("total,X", [(1, 8), (7, 8), (64, 8), (1001, 8), (333, 4), (50, 1)])
def test_ws_global_atomic_queue_is_the_chiplet_transform_of_the_counter(total, X):
    lib = _load()
    got = _queue(lib, TB_WS_GLOBAL_ATOMIC, 0, total, X, 4, 0)
    assert got == [OS.ws_global_atomic_tile(i, total, X) for i in range(total)]
    assert sorted(got) == list(range(total))
    # workgroup ids dealt round-robin to XCDs: consecutive counter values alternate between XCD runs
    if X > 1 and total >= 2 * X and total % X == 0:
        assert got[1] - got[0] == total // X


@pytest.mark.parametrize("total,X,local", [(1024, 8, 128), (1024, 8, 100), (9, 8, 1), (5, 8, 0), (3584, 8, 224), (77, 4, 10)])
def test_ws_hierarchical_queues(total, X, local):
    lib = _load()
    seen = []
    for xcd in range(X):
        got = _queue(lib, TB_WS_HIERARCHICAL, xcd, total, X, 4, local)
        assert got == [OS.ws_hierarchical_tile(xcd, i, 1, local, X) for i in range(local)]
        seen += got
    pool = _queue(lib, TB_WS_HIERARCHICAL, X, total, X, 4, local)
    assert pool == [OS.ws_hierarchical_tile(0, i, 2, local, X) for i in range(total - X * local)]
    assert sorted(seen + pool) == list(range(total))


def test_ws_queue_tile_rejects_bad_arguments():
    lib = _load()
    cnt, tile = C.c_int32(), C.c_int32()
    TB_ERR_NULL_POINTER, TB_ERR_BAD_ARGUMENT = -1, -10
    assert lib.tb_ws_queue_tile(3, 0, 0, 10, 8, 4, 0, C.byref(cnt), C.byref(tile)) == TB_ERR_BAD_ARGUMENT
    assert lib.tb_ws_queue_tile(0, 32, 0, 10, 8, 4, 0, C.byref(cnt), C.byref(tile)) == TB_ERR_BAD_ARGUMENT
    assert lib.tb_ws_queue_tile(1, 1, 0, 10, 8, 4, 0, C.byref(cnt), C.byref(tile)) == TB_ERR_BAD_ARGUMENT
    assert lib.tb_ws_queue_tile(2, 0, 0, 10, 8, 4, 2, C.byref(cnt), C.byref(tile)) == TB_ERR_BAD_ARGUMENT   # 8*2 > 10
    assert lib.tb_ws_queue_tile(0, 0, 0, 10, 8, 4, 0, None, C.byref(tile)) == TB_ERR_NULL_POINTER


def test_hierarchical_split_known_answers():
    # <= 4 tiles per CU: everything local; 14 tiles per CU and beyond: half
    assert OS.hierarchical_split(1024, 256, 8) == (128, 0)
    assert OS.hierarchical_split(512, 256, 8) == (64, 0)
    assert OS.hierarchical_split(3584, 256, 8) == (224, 1792)          # 14 per CU -> frac 0.5
    assert OS.hierarchical_split(256 * 20, 256, 8) == (320, 2560)      # floor at one half
    lp, g = OS.hierarchical_split(2048, 256, 8)                        # 8 per CU -> frac 0.8
    assert (lp, g) == (int(2048 * 0.8) // 8, 2048 - 8 * (int(2048 * 0.8) // 8))


@pytest.mark.parametrize("m,n,k", [(8192, 8192, 8192), (8192, 28672, 8192), (4096, 4096, 4096), (256, 256, 256), (16384, 16384, 1024)])
def test_selector_hierarchical_split_matches_the_reference_formula(m, n, k):
    import tritonblas_amd as tb
    sel = tb.OrigamiMatmulSelector(m, n, k, torch.bfloat16, torch.bfloat16, torch.bfloat16, "cpu")
    total = -(-m // sel.block_m) * -(-n // sel.block_n)
    hw = sel._hardware._c.num_xcd * sel._hardware._c.cu_per_xcd
    X = sel.num_sms
    want = OS.hierarchical_split(total, hw, X)
    got = sel.hierarchical_split(X)
    assert got[0] * X + got[1] == total and got[0] >= 0 and got[1] >= 0
    if want[1] >= 0:
        assert got == want
    else:   # fewer tiles than XCDs: the reference formula overshoots, the selector keeps the split valid
        assert got == (total // X, total - X * (total // X))


@pytest.mark.parametrize("remove,X,per", [(0, 8, 32), (1, 8, 32), (5, 8, 32), (31, 8, 32), (3, 4, 20), (2, 1, 7)])
def test_balanced_cu_mask(remove, X, per):
    from tritonblas_amd.benchmarks.common import build_balanced_hex_mask
    s = build_balanced_hex_mask(remove, X, per)
    assert s == OS.build_balanced_hex_mask(remove, X, per)
    if remove == 0:
        assert s == ""
        return
    v = int(s, 16)
    assert v < (1 << (X * per))
    for xcd in range(X):   # CU bit i sits on XCD i % X: every XCD loses exactly `remove` CUs, the lowest ones
        bits = [(v >> i) & 1 for i in range(xcd, X * per, X)]
        assert bits == [0] * remove + [1] * (per - remove)


def test_matmul_config_mask_rules():
    import tritonblas_amd as tb
    from tritonblas_amd.config import MatmulConfig
    cfg = MatmulConfig(device=torch.device("cpu"), workspace=None)
    assert cfg.mask is None and cfg.active_mask() is None and not cfg.global_atomic and not cfg.hierarchical
    m = torch.ones(8, dtype=torch.int32)
    cfg.mask = m            # a mask the caller assigns is used
    assert cfg.active_mask() is m
    cfg.mask = None
    assert cfg.active_mask() is None
    cfg2 = MatmulConfig(device=torch.device("cpu"), workspace=None, mask=m, use_mask=False)   # what matmul_preamble does with all CUs active
    assert cfg2.mask is m and cfg2.active_mask() is None


@pytest.mark.parametrize("total", [1, 5, 8, 9, 63, 512, 1024, 1100, 2048, 3584, 5120, 100000])
@pytest.mark.parametrize("hw_cus,xcds", [(256, 8), (304, 8), (64, 4), (32, 1)])
def test_library_hierarchical_split(total, hw_cus, xcds):
    lib = _load()
    l, g = C.c_int32(), C.c_int32()
    assert lib.tb_hierarchical_split(total, hw_cus, xcds, C.byref(l), C.byref(g)) == 0
    want = OS.hierarchical_split(total, hw_cus, xcds)
    assert l.value * xcds + g.value == total and l.value >= 0 and g.value >= 0
    if want[1] >= 0:
        assert (l.value, g.value) == want
    else:
        assert (l.value, g.value) == (total // xcds, total - xcds * (total // xcds))
    assert lib.tb_hierarchical_split(0, hw_cus, xcds, C.byref(l), C.byref(g)) == -10
    assert lib.tb_hierarchical_split(total, hw_cus, xcds, None, C.byref(g)) == -1


def test_grouped_gemm_refuses_other_operand_types():
    """the grouped entry point computes in FP8 e4m3 whatever it is handed: other types must not be read as that"""
    import tritonblas_amd as tb
    a = torch.zeros(8, 128, dtype=torch.float8_e5m2)
    w = torch.zeros(2, 16, 128, dtype=torch.float8_e5m2)
    c = torch.zeros(8, 16, dtype=torch.bfloat16)
    offs = torch.tensor([0, 4, 8], dtype=torch.int32)
    with pytest.raises(RuntimeError, match="float8_e4m3fn"):
        tb.grouped_matmul_a8w8(a, w, None, None, c, offs)


def test_matmul_fp4_refuses_wrong_element_sizes_and_scale_shapes():
    import tritonblas_amd as tb
    a, b = torch.zeros(8, 64, dtype=torch.uint8), torch.zeros(16, 64, dtype=torch.uint8)
    c = torch.zeros(8, 16, dtype=torch.bfloat16)
    sa, sb = torch.zeros(8, 4, dtype=torch.uint8), torch.zeros(16, 4, dtype=torch.uint8)
    with pytest.raises(RuntimeError, match="one-byte"):
        tb.matmul_fp4(a.to(torch.bfloat16), b, c, sa, sb)
    with pytest.raises(RuntimeError, match="scales must be"):
        tb.matmul_fp4(a, b, c, sa.T.contiguous(), sb)


def _streamk_ranges(total, G, units, cut):
    """The K ranges the kernels give their workgroups for `cut` tiles at the end of a table (units of K per tile):
    workgroup i takes q units, the first `rem` workgroups one more, in the order of their ids."""
    first = (total - cut) * units
    q, rem = divmod(cut * units, G)
    return [(first + i * q + min(i, rem), first + (i + 1) * q + min(i + 1, rem)) for i in range(G)]


@pytest.mark.parametrize("G", [1, 5, 8, 12, 256])
def test_streamk_tail_rule_by_brute_force(G):
    """tb_streamk_tail_tiles against a walk of the ranges it implies: the answer is 0, the tail or the tail plus one
    round; the ranges cover every K unit of the cut tiles exactly once; no tile meets more ranges than the rule charged
    for; and among the three plans the answer is the cheapest by the critical path of that walk (whole rounds, then the
    longest range, then one exchange per extra piece of the most-cut tile)."""
    from tritonblas_amd import _lib
    lib = _lib.load()
    rng = np.random.default_rng(G)
    for _ in range(300):
        total = int(rng.integers(1, 6 * G + 2))
        units = int(rng.integers(1, 17))
        unit_steps = int(rng.choice([1, 4]))
        fix = int(rng.integers(0, 40))
        cut = lib.tb_streamk_tail_tiles(total, G, units, unit_steps, fix)
        tail, rounds = total % G, total // G
        assert cut in {0, tail, tail + G} and cut <= total
        if tail == 0 or units < 2:
            assert cut == 0
            continue

        def walk_cost(c):
            if c == 0:
                return (rounds + 1) * units * unit_steps
            ranges = _streamk_ranges(total, G, units, c)
            cover = np.zeros(total * units, dtype=np.int32)
            pieces = {}
            for lo, hi in ranges:
                cover[lo:hi] += 1
                for t in range(lo // units, (hi + units - 1) // units if hi > lo else lo // units):
                    pieces[t] = pieces.get(t, 0) + 1
            assert (cover[(total - c) * units:] == 1).all() and (cover[:(total - c) * units] == 0).all()
            longest = max(hi - lo for lo, hi in ranges)
            return ((total - c) // G) * units * unit_steps + longest * unit_steps, max(pieces.values())

        options = [0, tail] + ([tail + G] if rounds >= 1 else [])
        costs = {}
        for c in options:
            if c == 0:
                costs[c] = walk_cost(0)
            else:
                base, most = walk_cost(c)
                # the rule's bound on the pieces of a tile is an upper bound of what the walk shows, and tight enough
                # that both agree on the price within one exchange
                q = (c * units) // G
                bound = min(units, ((units - 2) // max(q, 1) if units >= 2 else 0) + 2)
                assert most <= bound, (total, G, units, c, most, bound)
                costs[c] = base + (bound - 1) * fix
        assert costs[cut] == min(costs.values()), (total, G, units, unit_steps, fix, cut, costs)


def test_streamk_tail_rule_known_answers():
    """8 experts' 2072 tiles of 32 K steps on 256 workgroups: 8 whole rounds and 24 tiles.  Cutting the 24 tiles alone
    means eight pieces per tile; cutting them together with one whole round means two: with exchanges at 9 K steps the
    rule takes 280, at the library's 64 K steps it leaves the tiles whole, and with four times the K it cuts again."""
    from tritonblas_amd import _lib
    lib = _lib.load()
    assert lib.tb_streamk_tail_tiles(2072, 256, 8, 4, 9) == 280
    assert lib.tb_streamk_tail_tiles(2072, 256, 8, 4, 64) == 0
    assert lib.tb_streamk_tail_tiles(2072, 256, 32, 4, 64) == 280
    assert lib.tb_streamk_tail_tiles(2048, 256, 8, 4, 9) == 0          # whole rounds only
    assert lib.tb_streamk_tail_tiles(256 + 200, 256, 8, 4, 9) == 0     # a nearly full last round is cheaper whole
    assert lib.tb_streamk_tail_tiles(256 + 128, 256, 8, 4, 0) == 128   # free exchanges: always cut
    assert lib.tb_streamk_tail_tiles(100, 256, 8, 4, 9) in (0, 100)
    assert lib.tb_streamk_tail_tiles(10, 0, 8, 4, 9) == -10 and lib.tb_streamk_tail_tiles(10, 4, 8, 0, 9) == -10


def test_packed_descriptors_fill_the_structures_field_by_field():
    """The packed form of a descriptor is the ctypes structure's bytes: every field, in order, with the structure's padding."""
    from tritonblas_amd import _lib
    for pack, struct in ((_lib.pack_gemm, _lib.tb_gemm_desc), (_lib.pack_gemm_fp4, _lib.tb_gemm_fp4_desc),
                         (_lib.pack_quant_mx, _lib.tb_quant_desc), (_lib.pack_quant_rows, _lib.tb_row_quant_desc)):
        values = [i + 3 for i in range(len(struct._fields_))]
        got = struct.from_buffer_copy(pack(*values))
        want = struct(*values)
        for name, _ in struct._fields_:
            assert getattr(got, name) == getattr(want, name), (struct.__name__, name)


def test_streaming_kernel_and_partitions():
    """A few rows go to the streaming kernel, also int8 ones and any whole number of 16-byte chunks of K; a launch that is kept to some of the CUs by a
    grid goes to tiles (unless it has 16 rows at most)."""
    import ctypes as C
    from tritonblas_amd import _lib
    lib = _lib.load()

    def streams(dtype, m, n, k, grid=0):
        d = _lib.tb_gemm_desc()
        d.struct_bytes = C.sizeof(_lib.tb_gemm_desc)
        d.a_type = d.b_type = dtype
        d.c_type = _lib.TB_BF16
        d.m, d.n, d.k = m, n, k
        d.a_stride_m, d.a_stride_k, d.b_stride_k, d.b_stride_n, d.c_stride_m, d.c_stride_n = k, 1, 1, k, n, 1
        d.grid = grid
        info = _lib.tb_launch_info()
        assert lib.tb_gemm_launch_info(d, C.byref(info)) == _lib.TB_OK
        return info.skinny == 1

    for dtype in (_lib.TB_BF16, _lib.TB_FP8_E4M3, _lib.TB_I8):
        for m in (1, 16, 32):
            assert streams(dtype, m, 4096, 14336) and streams(dtype, m, 4096, 14336 + 16)
        assert not streams(dtype, 65, 4096, 14336)
        assert not streams(dtype, 48, 4096, 14336, grid=64)
    assert streams(_lib.TB_BF16, 8, 4096, 14336, grid=64) and not streams(_lib.TB_I8, 8, 4096, 14336, grid=64)


def _job(a_type, m, n, k, schedule=0, grid=0, c_type=None, n_major=False, m_major=False, tile=None, **fields):
    """A descriptor of contiguous operands (B stored (k, n) when n_major, A stored (k, m) when m_major)."""
    import ctypes as C
    from tritonblas_amd import _lib
    d = _lib.tb_gemm_desc()
    d.struct_bytes = C.sizeof(_lib.tb_gemm_desc)
    d.a_type = d.b_type = a_type
    d.c_type = _lib.TB_BF16 if c_type is None else c_type
    d.m, d.n, d.k = m, n, k
    d.a_stride_m, d.a_stride_k = (1, m) if m_major else (k, 1)
    d.b_stride_k, d.b_stride_n = (n, 1) if n_major else (1, k)
    d.c_stride_m, d.c_stride_n = n, 1
    if tile:
        d.block_m, d.block_n, d.block_k = tile
    d.schedule, d.grid = schedule, grid
    for name, value in fields.items():
        setattr(d, name, value)
    return d


def _launch_of(d):
    import ctypes as C
    from tritonblas_amd import _lib
    info = _lib.tb_launch_info()
    assert _lib.load().tb_gemm_launch_info(d, C.byref(info)) == _lib.TB_OK
    return info


@pytest.mark.parametrize("a_type,m,n,k,schedule", [("TB_FP8_E4M3", 64, 3584, 704, "WORK_STEALING"), ("TB_I8", 32, 4096, 14336, "WORK_STEALING"),
                                                   ("TB_FP8_E4M3", 48, 8192, 28672, "STREAMK"), ("TB_FP8_E4M3", 48, 8192, 28672, "STREAMK_WS"),
                                                   ("TB_BF16", 16, 2048, 1024, "PERSISTENT"), ("TB_BF16", 4, 12416, 1024, "WORK_STEALING"),
                                                   ("TB_F16", 8, 4224, 1000, "STREAMK")])
def test_a_callers_grid_or_mask_keeps_few_rows_on_tiles(a_type, m, n, k, schedule):
    """Launches of few rows that stream over the whole device run as tiles where the caller sized the launch, under every schedule."""
    from tritonblas_amd import _lib
    a_type, schedule = getattr(_lib, a_type), getattr(_lib, "TB_SCHED_" + schedule)
    assert _launch_of(_job(a_type, m, n, k, schedule)).skinny == 1
    for grid in (32, 64):
        info = _launch_of(_job(a_type, m, n, k, schedule, grid))
        assert info.skinny == 0 and info.grid <= grid
    if schedule == _lib.TB_SCHED_WORK_STEALING:
        info = _launch_of(_job(a_type, m, n, k, schedule, cu_mask=256, cu_mask_len=64))       # (an address that nobody reads)
        assert info.skinny == 0 and info.grid == 64
    # what the device holds of any tile, and more, keeps the launch to nothing
    assert _launch_of(_job(a_type, m, n, k, schedule, 255)).skinny == 0
    assert _launch_of(_job(a_type, m, n, k, schedule, 2048)).skinny == 1


@pytest.mark.parametrize("dtype,m,n,k", [(torch.float8_e4m3fn, 64, 3584, 704), (torch.float8_e4m3fn, 32, 8192, 28672), (torch.int8, 32, 4096, 14336), (torch.bfloat16, 8, 2048, 1024)])
@pytest.mark.parametrize("schedule", ["PERSISTENT", "WORK_STEALING"])
def test_selectors_of_a_partition_and_of_the_whole_device(dtype, m, n, k, schedule):
    """The grid that a selector for so many CUs gives is what they hold of its tile: a part of the device keeps a launch on tiles, the whole of it does not."""
    import tritonblas_amd as tb
    from tritonblas_amd import _lib
    whole = tb.OrigamiMatmulSelector(m, n, k, dtype, dtype, torch.bfloat16, None)._N_CU
    for cus in (16, 64, whole - 1, whole):
        sel = tb.OrigamiMatmulSelector(m, n, k, dtype, dtype, torch.bfloat16, None, total_cus=cus)
        info = _launch_of(_job(_lib.tb_dtype(dtype), m, n, k, getattr(_lib, "TB_SCHED_" + schedule), cus * sel.waves_per_eu, tile=(sel.block_m, sel.block_n, sel.block_k)))
        assert info.skinny == (1 if cus == whole else 0), (cus, sel.waves_per_eu)


@pytest.mark.parametrize("a_type,m,n,k", [(torch.float8_e4m3fn, 32, 8192, 28672), (torch.bfloat16, 8, 14336, 4096), (torch.int8, 24, 4096, 14336)])
def test_stream_k_with_the_selectors_grid_streams(a_type, m, n, k):
    """The grid that a Stream-K launch carries by default is the selector's and keeps it to nothing; one of a selector for a CU partition does."""
    import tritonblas_amd as tb
    from tritonblas_amd import _lib
    for total_cus in (None, 40):
        sel = tb.OrigamiMatmulSelector(m, n, k, a_type, a_type, torch.bfloat16, None, streamk=True, total_cus=total_cus)
        info = _launch_of(_job(_lib.tb_dtype(a_type), m, n, k, _lib.TB_SCHED_STREAMK, sel.sk_grid, tile=(sel.block_m, sel.block_n, sel.block_k)))
        assert info.skinny == (1 if total_cus is None else 0)


@pytest.mark.parametrize("a_type,m,n,k,schedule,grid,room", [
    ("TB_I8", 7872, 272, 4288, "STREAMK", 256, 16), ("TB_FP8_E4M3", 4528, 8576, 1600, "STREAMK", 64, 16), ("TB_F32", 1536, 4224, 7808, "STREAMK_WS", 0, 16),
    ("TB_F16", 752, 6544, 384, "STREAMK", 128, 16), ("TB_F32", 304, 3568, 11968, "STREAMK", 0, 4), ("TB_BF16", 992, 1360, 704, "STREAMK_WS", 200, 4)])
def test_stream_k_without_a_named_tile_takes_one_that_fits_the_workspace(a_type, m, n, k, schedule, grid, room):
    """A tile that the model likes best and whose partial tiles outgrow the workspace gives way to the next that fits."""
    from tritonblas_amd import _lib
    a_type, schedule = getattr(_lib, a_type), getattr(_lib, "TB_SCHED_" + schedule)
    c_type = a_type if a_type == _lib.TB_F32 else _lib.TB_BF16
    assert _lib.load().tb_workspace_bytes(_job(a_type, m, n, k, schedule, grid, c_type)) > room << 20
    info = _launch_of(_job(a_type, m, n, k, schedule, grid, c_type, workspace=1 << 20, workspace_bytes=room << 20))
    _, flags = _lib.workspace_layout()
    partials = info.grid * (4 + 4 * info.block_m * info.block_n) if info.mode == 2 else 0
    assert flags + 256 + partials <= room << 20
    if grid:
        assert info.grid == grid


@pytest.mark.parametrize("dtype,c_type", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32), (torch.float8_e4m3fn, torch.bfloat16),
                                          (torch.int8, torch.int8), (torch.float32, torch.float32)])
def test_selectors_tile_is_the_one_that_the_operands_layout_asks_for(dtype, c_type):
    """What a launch with a selector names is what the library picks by itself for these operands, also where K is no even number of K steps and an operand
    is not K-contiguous, or its rows start off 16 bytes."""
    import random
    import tritonblas_amd as tb
    from tritonblas_amd import _lib
    rng = random.Random(7)
    code, c_code, step = _lib.tb_dtype(dtype), _lib.tb_dtype(c_type), 128 // dtype.itemsize
    cases = [(4136, 4296, 7584)] + [tuple(rng.randint(32, 1024) * 8 for _ in range(3)) for _ in range(60)] + [(2000, 3000, 4097), (4096, 2040, 2047)]
    told = 0
    for m, n, k in cases:
        sel = tb.OrigamiMatmulSelector(m, n, k, dtype, dtype, c_type, None)
        for n_major in (False, True):
            if n_major and dtype.itemsize == 1:
                continue
            own = _launch_of(_job(code, m, n, k, c_type=c_code, n_major=n_major))
            tile = sel.block_m, sel.block_n, sel.block_k
            assert tile == sel._model_tile
            info = own if k % (2 * sel.block_k) else _launch_of(_job(code, m, n, k, c_type=c_code, n_major=n_major, tile=tile))
            assert (info.block_m, info.block_n, info.waves, info.four_wave) == (own.block_m, own.block_n, own.waves, own.four_wave), (m, n, k, n_major)
            told += (own.block_m, own.block_n, own.block_k) != tile
    assert told or dtype.itemsize != 2
    # a tile that the caller put into the selector stays, and so does a partition's
    side = 64 if sel.block_m != 64 else 128
    sel._sel.block_m, sel._sel.block_n, sel._sel.block_k = side, side, step
    assert (sel.block_m, sel.block_n, sel.block_k) != sel._model_tile
    part = tb.OrigamiMatmulSelector(4136, 4296, 7584, dtype, dtype, c_type, None, total_cus=64)
    assert part._model_tile is None


@pytest.mark.parametrize("a_type", ["TB_FP8_E4M3", "TB_FP8_E5M2", "TB_I8", "TB_BF16", "TB_F16"])
def test_few_k_steps_and_a_rest_go_to_the_eight_wave_kernel(a_type):
    """The 256x256 tile has two kernels for K-contiguous operands; for a K that is no even number of K steps the hand-scheduled one pays from some steps on."""
    from tritonblas_amd import _lib
    code = getattr(_lib, a_type)
    width = 128 if a_type in ("TB_FP8_E4M3", "TB_FP8_E5M2", "TB_I8") else 64
    for m, n, c_type, from_even, from_odd in [
            (4096, 4096, "TB_BF16", 10, 24), (512, 512, "TB_BF16", 10, 24), (500, 512, "TB_F16", 20, 36), (512, 504, "TB_F16", 20, 36), (4096, 8192, "TB_BF16", 10, 24),
            (4000, 8184, "TB_BF16", 10, 24), (7000, 9000, "TB_BF16", 4, 12), (4096, 8448, "TB_BF16", 4, 12), (4096, 4096, "TB_F32", 32, 48),
            (7000, 9000, "TB_F32", 32, 48), (4096, 4096, "TB_FP8_E4M3", 40, 56), (4096, 8452, "TB_BF16", 99, 99)]:       # (the last: rows of C off 16 bytes)
        if c_type == "TB_FP8_E4M3" and not a_type.startswith("TB_FP8"):
            continue
        for steps in range(4, 60):
            for part in (0, 16, width - 16):
                if steps % 2 == 0 and part == 0:
                    continue
                d = _job(code, m, n, steps * width + part, c_type=getattr(_lib, c_type), tile=(256, 256, width))
                info = _launch_of(d)
                assert (info.four_wave == 1) == (steps >= (from_odd if steps % 2 else from_even)), (m, n, steps, part)
                assert info.waves == (4 if info.four_wave else 8)


@pytest.mark.parametrize("a_type", ["TB_FP8_E4M3", "TB_FP8_E5M2", "TB_I8", "TB_BF16", "TB_F16"])
def test_few_even_k_steps_go_to_the_eight_wave_kernel(a_type):
    """... and for an even number of K steps, by how many rounds of tiles there are; Stream-K launches keep the hand-scheduled kernel."""
    from tritonblas_amd import _lib
    code = getattr(_lib, a_type)
    width = 128 if a_type in ("TB_FP8_E4M3", "TB_FP8_E5M2", "TB_I8") else 64
    one_round = 32 if a_type.startswith("TB_FP8") else 24
    for m, n, start in [(4096, 4096, one_round), (500, 300, one_round), (4096, 4352, 12), (4096, 8192, 12), (4096, 8448, 4), (7000, 9000, 4)]:
        for steps in range(4, 42, 2):
            info = _launch_of(_job(code, m, n, steps * width, tile=(256, 256, width)))
            assert (info.four_wave == 1) == (steps >= start), (m, n, steps)
            assert info.waves == (4 if info.four_wave else 8)


@pytest.mark.parametrize("dtype,m,n,k", [(torch.bfloat16, 4096, 4096, 1280), (torch.bfloat16, 4096, 4096, 512), (torch.float8_e4m3fn, 4096, 4096, 3840),
                                         (torch.int8, 4096, 4096, 1024)])
def test_few_even_k_steps_in_launches_that_loop_over_tiles(dtype, m, n, k):
    """... but only where a workgroup has one tile: launches that loop, from a caller's grid or the work-stealing queues, keep the hand-scheduled kernel."""
    import tritonblas_amd as tb
    from tritonblas_amd import _lib
    code, tile = _lib.tb_dtype(dtype), (256, 256, 128 // dtype.itemsize)
    assert _launch_of(_job(code, m, n, k, tile=tile)).four_wave == 0
    for schedule in (_lib.TB_SCHED_PERSISTENT, _lib.TB_SCHED_WORK_STEALING):
        for cus in (32, 64, 128, 255):
            assert _launch_of(_job(code, m, n, k, schedule, cus, tile=tile)).four_wave == 1
            sel = tb.OrigamiMatmulSelector(m, n, k, dtype, dtype, torch.bfloat16, None, total_cus=cus)
            info = _launch_of(_job(code, m, n, k, schedule, cus * sel.waves_per_eu, tile=(sel.block_m, sel.block_n, sel.block_k)))
            assert info.four_wave == (sel.block_m == sel.block_n == 256)
    assert _launch_of(_job(code, m, n, k, _lib.TB_SCHED_WORK_STEALING, tile=tile)).four_wave == 1
    assert _launch_of(_job(code, m, n, k, _lib.TB_SCHED_WORK_STEALING, tile=tile, cu_mask=256, cu_mask_len=64)).four_wave == 1      # (an address that nobody reads)


def _split_of(d):
    """The columns of a persistent call's first launch, and what its one or two launches are."""
    import ctypes as C
    from tritonblas_amd import _lib
    columns, launches = C.c_int64(), (_lib.tb_launch_info * 2)()
    assert _lib.load().tb_gemm_split_info(d, columns, launches) == _lib.TB_OK
    return columns.value, launches


@pytest.mark.parametrize("a_type", ["TB_BF16", "TB_F16", "TB_FP8_E4M3", "TB_FP8_E5M2", "TB_I8", "TB_F32"])
def test_both_parts_of_a_column_split_add_up_k_alike(a_type):
    """The columns behind the whole rounds run a tile of the same K step as the others, and no streaming kernel: every column of C sums K in the same order."""
    from tritonblas_amd import _lib
    code, splits = getattr(_lib, a_type), 0
    for m in (64, 512, 1024, 1280, 1792, 2048, 4096):
        for n in (6656, 6912, 8448, 8704, 9472, 13312, 70000):
            for k in (256, 512, 640, 1024, 2304, 3072):
                first, (a, b) = _split_of(_job(code, m, n, k, c_type=_lib.TB_F32 if a_type == "TB_F32" else None))
                if first < n:
                    splits += 1
                    assert a.block_k == b.block_k and not a.skinny and not b.skinny, (m, n, k)
    assert splits >= 10


@pytest.mark.parametrize("a_type,m,n,steps,columns", [
    ("TB_BF16", 1280, 13312, 16, 13056), ("TB_F16", 1280, 13312, 22, 13056), ("TB_BF16", 4096, 4352, 16, 4096), ("TB_BF16", 8192, 5120, 8, 4096),
    ("TB_FP8_E4M3", 1280, 13312, 16, 13056), ("TB_FP8_E5M2", 1280, 13312, 18, 13056), ("TB_FP8_E4M3", 4096, 4352, 24, 4096), ("TB_FP8_E4M3", 8192, 2560, 30, 2048),
    ("TB_I8", 1280, 13312, 16, 13056)])
def test_a_column_split_whose_parts_run_either_kernel_of_the_tile(a_type, m, n, steps, columns):
    """Just over one or two rounds of 256x256 tiles: the whole would run the hand-scheduled kernel, the columns that fill the rounds the eight-wave one, and the
    launch is split all the same.  A K with a rest, which the two add up in another order, is split only where both run one kernel."""
    from tritonblas_amd import _lib
    code = getattr(_lib, a_type)
    step = 64 if a_type in ("TB_BF16", "TB_F16") else 128
    d = _job(code, m, n, steps * step)
    whole = _launch_of(d)
    first, (a, b) = _split_of(d)
    assert (whole.block_m, whole.block_n, whole.four_wave) == (256, 256, 1)
    assert first == columns and (a.block_m, a.block_n, a.four_wave) == (256, 256, 0) and b.total_tiles > 0
    for k in range(steps * step - 7 * step, steps * step, 16):
        d = _job(code, m, n, k)
        first, (a, _) = _split_of(d)
        if first < n and k % (2 * a.block_k):
            whole = _launch_of(d)
            assert (a.block_m, a.block_n, a.waves, a.four_wave) == (whole.block_m, whole.block_n, whole.waves, whole.four_wave)
    d.column_split = -1
    assert _split_of(d)[0] == n


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float8_e4m3fn, torch.int8])
@pytest.mark.parametrize("m,n,k", [(512, 512, 8192), (256, 256, 7904), (200, 1000, 2000)])
def test_small_tiles_are_for_cus_that_would_be_idle(dtype, m, n, k):
    """32x32 and 64x32 tiles split what leaves CUs idle in 64x64: a launch that its caller keeps to fewer workgroups than it would have of them has none idle,
    and one that draws its tiles from the work-stealing queues takes 64x32 alone."""
    import tritonblas_amd as tb
    from tritonblas_amd import _lib
    from tritonblas_amd.matmul import _queue_tile
    code, queues = _lib.tb_dtype(dtype), _lib.TB_SCHED_WORK_STEALING
    own = _launch_of(_job(code, m, n, k))
    assert own.block_n == 32
    for grid in (8, 16, 32, 64, 128, 256):
        for info in (_launch_of(_job(code, m, n, k, grid=grid)), _launch_of(_job(code, m, n, k, queues, grid)),
                     _launch_of(_job(code, m, n, k, queues, cu_mask=256, cu_mask_len=grid))):       # (an address that nobody reads)
            assert info.block_n > 32 or info.total_tiles <= grid
            assert info.block_n > 32 or info.mode != 1 or info.block_m == 64
        assert grid > 16 or (info.block_m, info.block_n) == (64, 64)
    info = _launch_of(_job(code, m, n, k, queues))
    assert (info.block_m, info.block_n) == (64, 32) and info.total_tiles <= 256
    sel = tb.OrigamiMatmulSelector(m, n, k, dtype, dtype, torch.bfloat16, None)
    assert (sel.block_m, sel.block_n) == (own.block_m, own.block_n)
    assert _queue_tile(sel, dtype) == (0, 0, 0)
    for cus in (8, 16, 64):
        sel = tb.OrigamiMatmulSelector(m, n, k, dtype, dtype, torch.bfloat16, None, total_cus=cus)
        tiles = -(-m // sel.block_m) * -(-n // sel.block_n)
        assert sel.block_n > 32 or tiles <= cus * sel.waves_per_eu
        model = sel.block_m, sel.block_n, sel.block_k
        assert _queue_tile(sel, dtype) == ((64, 32, model[2]) if model[1] == 32 else model)
        sel._sel.block_m = sel._sel.block_n = 32      # (a tile that the caller put into the selector stays)
        assert model[:2] == (32, 32) or _queue_tile(sel, dtype) == (32, 32, model[2])


def test_fp32_and_int8_tiles_of_launches_kept_to_some_workgroups():
    """The tiles that pay where the whole device would be idle else are not for a part of it, but for fp32 tiles that all run at once."""
    import tritonblas_amd as tb
    from tritonblas_amd import _lib

    def side(a_type, m, n, k, **kw):
        info = _launch_of(_job(a_type, m, n, k, c_type=_lib.TB_F32 if a_type == _lib.TB_F32 else None, **kw))
        return info.block_m, info.block_n
    for m, n, k in [(1664, 480, 5568), (512, 2048, 2848), (240, 3552, 4672)]:
        assert side(_lib.TB_F32, m, n, k) == (32, 32)
        assert side(_lib.TB_F32, m, n, k, grid=64) == (64, 64) == side(_lib.TB_F32, m, n, k, grid=128, schedule=_lib.TB_SCHED_WORK_STEALING)
        assert tb.OrigamiMatmulSelector(m, n, k, torch.float32, torch.float32, torch.float32, None, total_cus=64).block_m == 64
    assert tb.OrigamiMatmulSelector(256, 512, 2048, torch.float32, torch.float32, torch.float32, None, total_cus=32).block_m == 32
    assert side(_lib.TB_F32, 20, 4000, 512, grid=16) == (32, 32)          # (few rows: the shortest tile there is)
    sel = tb.OrigamiMatmulSelector(640, 1024, 3072, torch.int8, torch.int8, torch.bfloat16, None, total_cus=32)
    assert (sel.block_m, sel.block_n) == (128, 128)


def _grouped_job(rows, experts, n, k, **fields):
    from tritonblas_amd import _lib
    g = _lib.tb_grouped_gemm_desc()
    g.struct_bytes, g.c_type = C.sizeof(_lib.tb_grouped_gemm_desc), _lib.TB_BF16
    g.m_total, g.n, g.k, g.num_groups = rows, n, k, experts
    g.a_stride_m, g.w_stride_g, g.w_stride_n, g.c_stride_m, g.c_stride_n = k, n * k, k, n, 1
    for name, value in fields.items():
        setattr(g, name, value)
    return g


def _grouped_launches(*args, tile=None, **fields):
    from tritonblas_amd import _lib
    if tile:
        fields.update(block_m=tile[0], block_n=tile[1], block_k=tile[2])
    launches = (_lib.tb_launch_info * 2)()
    assert _lib.load().tb_grouped_launch_info(_grouped_job(*args, **fields), launches) == _lib.TB_OK
    return launches


def test_which_grouped_calls_plan_two_launches():
    """A verdict on the device about a second launch is for calls with a Stream-K tail (the 256x256 hand-scheduled kernel on K in blocks of four steps) whose short row
    blocks may take the table past its first or second round."""
    two_by_verdict = [(4096, 8, 4096, 14336), (4096, 4, 4096, 6144), (8192, 8, 4096, 8192)]
    for case in two_by_verdict:
        first, second = _grouped_launches(*case, streamk=1)
        assert (first.block_m, first.block_n, first.four_wave) == (256, 256, 1) and (second.block_m, second.block_n, second.block_k) == (32, 128, 256)
    for rows, experts, n, k in [(8192, 8, 14336, 4096), (4096, 8, 4096, 14336), (1000, 4, 1536, 7168), (1024, 16, 4096, 2048), (8192, 8, 14336, 4096 + 256)]:
        for small in (-1, 0):
            assert _grouped_launches(rows, experts, n, k, small_rows=small)[1].total_tiles == 0
        assert _grouped_launches(rows, experts, n, k, streamk=1, small_rows=-1)[1].total_tiles == 0
        assert (_grouped_launches(rows, experts, n, k, streamk=1)[1].total_tiles > 0) == ((rows, experts, n, k) in two_by_verdict)
        assert _grouped_launches(rows, experts, n, k, streamk=1, tile=(256, 256, 128))[1].total_tiles == 0       # (a tile that the caller names)
        assert _grouped_launches(rows, experts, n, k, small_rows=40, tile=(256, 256, 128))[1].total_tiles > 0
    # a short K; no tail; no round that short blocks could end; rounds enough to share one more among
    for case in [(4096, 8, 4096, 4096), (4096, 8, 4096, 14336 + 128), (6144, 8, 4096, 14336), (2048, 8, 4096, 14336), (16384, 8, 4096, 14336)]:
        assert _grouped_launches(*case, streamk=1)[1].total_tiles == 0


GROUPED_VARIANTS = [((256, 128, 128), 423), ((128, 128, 128), 222), ((128, 128, 128), 424), ((128, 64, 128), 424), ((64, 64, 128), 222), ((64, 64, 128), 223),
                    ((64, 64, 128), 224), ((32, 128, 256), 143)]


def test_grouped_kernels_of_one_tile_to_a_workgroup(tb_option):
    """Each variant that the cost model knows, but for 256x256, has the kernel of one table entry to a workgroup, and every table fits the grid: a launch has as many
    workgroups as its table can have entries, over experts without rows and more of them than a wave has lanes."""
    import random
    from oracle import schedule as S
    rng = random.Random(11)
    for tile, waves in GROUPED_VARIANTS:
        tb_option("waves", waves)
        for experts in (1, 7, 64, 65, 200):
            for _ in range(4):
                counts = [rng.choice([0, 1, rng.randint(1, tile[0]), tile[0] - 1, tile[0], tile[0] + 1, rng.randint(1, 2000)]) for _ in range(experts)]
                counts[rng.randrange(experts)] += 1
                info = _grouped_launches(sum(counts), experts, 520, 512, tile=tile)[0]
                assert (info.block_m, info.block_n) == tile[:2] and info.waves == (waves // 100) * (waves // 10 % 10)
                table = sum(-(-c // tile[0]) for c in counts) * -(-520 // tile[1])
                assert info.grid == info.total_tiles >= table, (tile, waves, experts)
                offsets = [0]
                for c in counts:
                    offsets.append(offsets[-1] + c)
                assert S.grouped_tile_lookup(table - 1, offsets, tile[0], -(-520 // tile[1])) is not None
                assert S.grouped_tile_lookup(table, offsets, tile[0], -(-520 // tile[1])) is None
        # the most entries: one row above a whole block for every expert
        rows = 65 * (tile[0] + 1)
        assert _grouped_launches(rows, 65, 520, 512, tile=tile)[0].total_tiles == 65 * 2 * -(-520 // tile[1])
    tb_option("waves", 0)
    info = _grouped_launches(8192, 8, 14336, 4096, tile=(256, 256, 128))[0]
    assert info.four_wave == 1 and info.grid == 256 < info.total_tiles


@pytest.mark.parametrize("rows,experts,n,k,want", [(8192, 8, 14336, 4096, (256, 256)), (4096, 16, 4096, 2048, (256, 128)), (1024, 8, 14336, 4096, (128, 128)),
                                                   (1000, 4, 1536, 7168, (128, 64)), (64, 8, 14336, 4096, (64, 64)), (3000, 4, 1536, 7168, (256, 128))])
def test_the_grouped_models_choice(rows, experts, n, k, want):
    info = _grouped_launches(rows, experts, n, k)[0]
    assert (info.block_m, info.block_n) == want


@pytest.mark.parametrize("a_type", ["TB_BF16", "TB_F16", "TB_F32", "TB_FP8_E4M3", "TB_FP8_E5M2", "TB_I8"])
def test_persistent_launches_have_a_workgroup_to_a_tile(a_type):
    """... whatever the tile, with fewer tiles than the device holds and with more, but for the hand-scheduled kernels; a launch that names a grid loops."""
    from tritonblas_amd import _lib
    code = getattr(_lib, a_type)
    c_type = _lib.TB_F32 if a_type == "TB_F32" else None
    buf = (C.c_int32 * 60)()
    for i in range(_lib.load().tb_list_tiles(code, buf, 20)):
        tile = tuple(buf[3 * i:3 * i + 3])
        for m, n in [(40, 520), (300, 700), (9000, 9000)]:
            info = _launch_of(_job(code, m, n, 2 * tile[2], c_type=c_type, tile=tile, column_split=-1))
            assert info.skinny == 1 or (info.block_m, info.block_n) == tile[:2]
            assert info.skinny == 1 or info.four_wave == 1 or info.grid == info.total_tiles
            info = _launch_of(_job(code, m, n, 2 * tile[2], grid=3, c_type=c_type, tile=tile))
            assert info.skinny == 1 or info.grid == min(3, info.total_tiles)


@pytest.mark.parametrize("a_type", ["TB_BF16", "TB_F16", "TB_FP8_E4M3", "TB_I8"])
def test_which_problems_of_few_tiles_take_small_ones(a_type):
    """Both sides of the lines: few rows against many columns are the streaming kernel's or a taller tile's."""
    from tritonblas_amd import _lib
    for m, n, k, small in [(65, 1024, 256, True), (64, 1024, 512, False), (64, 1000, 528, True), (33, 40, 4096, True), (200, 1000, 2000, True), (256, 256, 7904, True), (31, 33, 272, True),
                           (1, 1000, 1040, True), (64, 4096, 4096, False), (2048, 2048, 2048, False)]:
        info = _launch_of(_job(getattr(_lib, a_type), m, n, k))
        assert (info.block_n == 32) == small, (m, n, k, info.block_m, info.block_n)
    # Stream-K launches have none
    assert _launch_of(_job(getattr(_lib, a_type), 256, 256, 7904, _lib.TB_SCHED_STREAMK)).block_n > 32


def test_few_even_k_steps_of_mxfp4():
    """The lines of MXFP4 for the two kernels of the 256x256 tile: 24 K steps of 256 values in one round, 16 in two, none beyond."""
    from tritonblas_amd import _lib
    for m, n, start in [(4096, 4096, 24), (7860, 1552, 24), (4096, 8192, 16), (4096, 8448, 4)]:
        for steps in range(4, 30, 2):
            g = _lib.tb_gemm_fp4_desc()
            g.struct_bytes, g.c_type = C.sizeof(_lib.tb_gemm_fp4_desc), _lib.TB_BF16
            g.m, g.n, g.k = m, n, steps * 256
            g.a_stride_m = g.b_stride_n = g.k // 2
            g.c_stride_m, g.c_stride_n = n, 1
            g.a_scales_stride_m = g.b_scales_stride_n = g.k // 32
            g.a_scales_stride_k = g.b_scales_stride_k = 1
            g.block_m, g.block_n, g.block_k = 256, 256, 256
            info = _lib.tb_launch_info()
            assert _lib.load().tb_gemm_fp4_launch_info(g, info) == _lib.TB_OK
            assert (info.four_wave == 1) == (steps >= start) and info.waves == (4 if info.four_wave else 8), (m, n, steps)


@pytest.mark.parametrize("a_type,m,n,k", [("TB_BF16", 1024, 1024, 1024), ("TB_BF16", 2048, 2048, 2048), ("TB_FP8_E4M3", 4096, 4096, 1024)])
def test_stream_k_calls_that_share_no_tile_run_as_persistent_ones(a_type, m, n, k):
    """... of the tile that they have, by a workgroup to a tile where it has that kernel, and by the same line for few even K steps."""
    from tritonblas_amd import _lib
    code = getattr(_lib, a_type)
    plan = _launch_of(_job(code, m, n, k, _lib.TB_SCHED_STREAMK))
    assert plan.mode == 0
    first, (a, b) = _split_of(_job(code, m, n, k, _lib.TB_SCHED_STREAMK))
    own = _launch_of(_job(code, m, n, k, tile=(plan.block_m, plan.block_n, plan.block_k)))
    assert first == n and (a.block_m, a.block_n, a.waves, a.four_wave, a.grid) == (own.block_m, own.block_n, own.waves, own.four_wave, own.total_tiles) and b.total_tiles == 0


def test_tiles_of_the_register_loading_kernels():
    """Rows off 16 bytes run in 128x128 or 64x64 tiles: 128 where the chosen tile has it on both sides, and where fp32 fills the CUs with them once."""
    from tritonblas_amd import _lib
    def tile(a_type, m, n, k, **kw):
        info = _launch_of(_job(a_type, m, n, k, c_type=a_type, **kw))
        return info.block_m, info.block_n
    for a_type, width in ((_lib.TB_BF16, 64), (_lib.TB_F16, 64), (_lib.TB_F32, 32)):
        for named, want in [((256, 256), 128), ((128, 128), 128), ((64, 64), 64)] + ([((256, 128), 128), ((128, 64), 64), ((32, 128), 64)] if width == 64 else []):
            named += (128 if named == (32, 128) else width,)
            assert tile(a_type, 1063, 1379, 527, tile=named) == (want, want), (a_type, named)
    assert tile(_lib.TB_BF16, 1063, 1379, 527) == (64, 64) and tile(_lib.TB_BF16, 3039, 331, 339) == (64, 64)
    assert tile(_lib.TB_F32, 5294, 658, 7306) == (128, 128) and tile(_lib.TB_F32, 1265, 2929, 1039) == (128, 128)
    assert tile(_lib.TB_F32, 1507, 1917, 305) == (64, 64) and tile(_lib.TB_F32, 2341, 4149, 5047) == (64, 64)
    # a Stream-K launch keeps what its workspace was sized for
    assert tile(_lib.TB_F32, 1265, 2929, 1039, schedule=_lib.TB_SCHED_STREAMK, tile=(64, 64, 32)) == (64, 64)
