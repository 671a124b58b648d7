"""The persistent schedule with one tile to a workgroup (a launch that names no grid) against the looping kernel (a launch with one): the same K loop and
the same store, so the results are the same bit for bit, and within the rounding of their type of the product in 64 bits."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu

TYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32, "fp8": torch.float8_e4m3fn, "i8": torch.int8}
# the rounding of a result to its type; fp32: sums of up to 1100 products of whole numbers up to 9 are exact
REL = {"bf16": 2.0 ** -8, "f16": 2.0 ** -11, "f32": 0.0, "fp8": 2.0 ** -8, "i8": 2.0 ** -8}


def _product(a, b, c, tile, grid, column_split=-1, schedule=0, workspace=None):
    from tritonblas_amd import _lib
    d = _lib.tb_gemm_desc()
    d.struct_bytes = C.sizeof(_lib.tb_gemm_desc)
    d.a_type = d.b_type = _lib.tb_dtype(a.dtype)
    d.c_type = _lib.tb_dtype(c.dtype)
    d.m, d.k = a.shape
    d.n = b.shape[1]
    d.a_stride_m, d.a_stride_k = a.stride()
    d.b_stride_k, d.b_stride_n = b.stride()
    d.c_stride_m, d.c_stride_n = c.stride()
    d.a, d.b, d.c = a.data_ptr(), b.data_ptr(), c.data_ptr()
    d.block_m, d.block_n, d.block_k = tile
    d.grid, d.column_split, d.schedule = grid, column_split, schedule
    if workspace is not None:
        d.workspace, d.workspace_bytes, d.epoch = workspace.data_ptr(), workspace.numel(), _lib.TB_EPOCH_ON_DEVICE
    assert _lib.load().tb_gemm(d, _lib.stream_handle()) == _lib.TB_OK
    return c


@pytest.mark.parametrize("kind,m,n,k,order", [
    ("bf16", 1, 1, 8, "kk"), ("bf16", 129, 191, 64, "kn"), ("bf16", 640, 1000, 1096, "mn"),      # a corner of a tile; edges; a remainder of K
    ("bf16", 131, 203, 1031, "kk"), ("f16", 257, 333, 777, "mn"),                                # rows off 16 bytes
    ("f32", 65, 72, 36, "kk"), ("f32", 300, 520, 1092, "kn"), ("f32", 127, 131, 1001, "mk"),
    ("fp8", 64, 64, 128, "kk"), ("fp8", 300, 1040, 1104, "kk"), ("i8", 33, 272, 1040, "kk"), ("i8", 100, 90, 1001, "kk"),
    ("bf16", 5000, 4000, 128, "kk"),                                                             # more tiles than the device holds at once
])
def test_one_tile_per_workgroup_matches_the_loop(kind, m, n, k, order):
    from tritonblas_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(m + n + k)

    def stored(rows, cols, contiguous):
        x = torch.randint(-3, 4, (rows, cols) if contiguous else (cols, rows), device="cuda", generator=g).to(TYPES[kind])
        return x if contiguous else x.T

    a, b = stored(m, k, order[0] == "k"), stored(k, n, order[1] == "n")
    out = TYPES[kind] if kind in ("bf16", "f16", "f32") else torch.bfloat16
    want = a.double() @ b.double()
    buf = (C.c_int32 * 60)()
    count = _lib.load().tb_list_tiles(_lib.tb_dtype(TYPES[kind]), buf, 20)
    for i in range(count):
        tile = tuple(buf[3 * i:3 * i + 3])
        got = _product(a, b, torch.full((m, n), float("nan"), device="cuda", dtype=out), tile, 0)
        loop = _product(a, b, torch.full((m, n), float("nan"), device="cuda", dtype=out), tile, 48)
        assert torch.equal(got, loop), tile
        assert ((got.double() - want).abs() <= REL[kind] * want.abs()).all(), tile


GROUPED_TILES = [((256, 128, 128), 423), ((128, 128, 128), 222), ((128, 128, 128), 424), ((128, 64, 128), 424), ((64, 64, 128), 222), ((64, 64, 128), 223),
                 ((64, 64, 128), 224), ((32, 128, 256), 143), ((256, 256, 128), 22), (None, 0)]


@pytest.mark.parametrize("counts,n,k", [
    ([1], 1, 16), ([0, 33, 0, 31, 1, 0], 130, 272), ([127, 128, 129, 0, 255, 257], 200, 1040),      # corners, empty experts, edges of the tiles, remainders of K
    ([3 * (e % 5) for e in range(131)], 96, 512),                                                   # more experts than a wave has lanes
    ([5000, 1, 700], 1100, 640),                                                                    # more tiles than the device holds at once
])
def test_grouped_one_tile_per_workgroup(counts, n, k, tb_option):
    import tritonblas_amd as tb
    g = torch.Generator(device="cuda").manual_seed(n + k)
    rows, experts = sum(counts), len(counts)
    a = torch.randint(-2, 3, (rows, k), device="cuda", generator=g).to(torch.float8_e4m3fn)
    w = torch.randint(-2, 3, (experts, n, k), device="cuda", generator=g).to(torch.float8_e4m3fn)
    at = [0]
    for c in counts:
        at.append(at[-1] + c)
    offsets = torch.tensor(at, dtype=torch.int32, device="cuda")
    want = torch.cat([a[lo:hi].double() @ w[e].double().T for e, (lo, hi) in enumerate(zip(at, at[1:]))])     # (whole numbers below 2**24: exact in fp32)
    for tile, waves in GROUPED_TILES:
        tb_option("waves", waves)
        got = torch.full((rows, n), float("nan"), device="cuda", dtype=torch.bfloat16)
        tb.grouped_matmul_a8w8(a, w, None, None, got, offsets, *(tile or (None, None, None)))
        assert ((got.double() - want).abs() <= REL["fp8"] * want.abs()).all(), (tile, waves)


@pytest.mark.parametrize("kind", ["bf16", "f16", "fp8", "i8"])
@pytest.mark.parametrize("m,n,k", [(65, 1024, 256), (64, 1024, 512), (64, 1000, 528), (33, 40, 4096), (200, 1000, 2000), (256, 256, 7904), (31, 33, 272), (1, 1000, 1040)])
def test_few_tiles(m, n, k, kind):
    """Both sides of the rule for the 32x32 and 64x32 tiles: the library's own choice, and the two named."""
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a = torch.randint(-2, 3, (m, k), device="cuda", generator=g).to(TYPES[kind])
    b = torch.randint(-2, 3, (n, k), device="cuda", generator=g).to(TYPES[kind]).T
    want = a.double() @ b.double()
    out = TYPES[kind] if kind in ("bf16", "f16") else torch.bfloat16
    step = 128 if kind in ("bf16", "f16") else 256
    for tile in ((0, 0, 0), (32, 32, step), (64, 32, step)):
        got = _product(a, b, torch.full((m, n), float("nan"), device="cuda", dtype=out), tile, 0)
        assert ((got.double() - want).abs() <= REL[kind] * want.abs()).all(), tile       # (whole numbers below 2**24: the sums are exact)


@pytest.mark.parametrize("kind", ["bf16", "f16", "fp8"])
@pytest.mark.parametrize("k", [640, 1152, 1200, 2432])
def test_order_of_k_in_small_tiles(kind, k):
    """Values that fp32 sums round.  The remainder of K is added first, and tiles whose K steps are twice as long have another one where it holds half a step: each tile
    adds up K in an order of its own, and all are within the rounding of k fp32 sums (2**-24 each of at most the sum of the magnitudes) of the product in 64 bits."""
    g = torch.Generator(device="cuda").manual_seed(k)
    a, b = (torch.randn(s, device="cuda", generator=g).to(TYPES[kind]) for s in ((200, k), (1000, k)))
    want, size = a.double() @ b.double().T, a.double().abs() @ b.double().abs().T
    unit = 64 if kind in ("bf16", "f16") else 128
    for tile in ((0, 0, 0), (32, 32, 2 * unit), (64, 32, 2 * unit), (32, 128, 2 * unit), (64, 64, unit)):
        got = _product(a, b.T, torch.full((200, 1000), float("nan"), device="cuda"), tile, 0)
        assert ((got.double() - want).abs() <= k * 2.0 ** -24 * size).all(), tile


@pytest.mark.parametrize("kind", ["bf16", "f16", "fp8", "i8"])
@pytest.mark.parametrize("m,n,k", [(33, 40, 4096), (200, 1000, 2000), (256, 256, 7904), (31, 33, 272), (353, 1264, 1552)])
def test_small_tiles_under_the_other_schedules(m, n, k, kind):
    """32x32 and 64x32 tiles from the work-stealing queues and with a Stream-K tail, named and as the library chooses, on the whole device and on 24 workgroups; one
    workspace for all launches.  Then through a selector, which has a small tile for each of these."""
    import tritonblas_amd as tb
    from tritonblas_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a = torch.randint(-2, 3, (m, k), device="cuda", generator=g).to(TYPES[kind])
    b = torch.randint(-2, 3, (n, k), device="cuda", generator=g).to(TYPES[kind]).T
    want = a.double() @ b.double()
    out = TYPES[kind] if kind in ("bf16", "f16") else torch.bfloat16
    step = 128 if kind in ("bf16", "f16") else 256
    workspace = torch.zeros(64 << 20, dtype=torch.uint8, device="cuda")
    for schedule in (_lib.TB_SCHED_WORK_STEALING, _lib.TB_SCHED_STREAMK, _lib.TB_SCHED_STREAMK_WS):
        for grid in (0, 24):
            for tile in ((0, 0, 0), (32, 32, step), (64, 32, step)):
                got = _product(a, b, torch.full((m, n), float("nan"), device="cuda", dtype=out), tile, grid, schedule=schedule, workspace=workspace)
                assert ((got.double() - want).abs() <= REL[kind] * want.abs()).all(), (schedule, grid, tile)
    selector = tb.OrigamiMatmulSelector(m, n, k, a.dtype, b.dtype, out, a.device)
    config = tb.matmul_preamble(selector, a.device)
    for streamk in (False, True):
        got = torch.full((m, n), float("nan"), device="cuda", dtype=out)
        tb.matmul_lt(a, b, got, selector, config, enable_streamk=streamk, work_stealing=True)
        assert ((got.double() - want).abs() <= REL[kind] * want.abs()).all(), streamk


def _split_and_whole(kind, m, n, k):
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    if kind == "i8":
        a, b = (torch.randint(-127, 128, s, device="cuda", generator=g).to(torch.int8) for s in ((m, k), (n, k)))
    else:
        a, b = (torch.randn(s, device="cuda", generator=g).to(TYPES[kind]) for s in ((m, k), (n, k)))
    out = TYPES[kind] if kind in ("bf16", "f16") else torch.float32
    return [_product(a, b.T, torch.full((m, n), float("nan"), device="cuda", dtype=out), (0, 0, 0), 0, column_split=c) for c in (0, -1)]


@pytest.mark.parametrize("kind,m,n,k", [("bf16", 1792, 9472, 2304), ("f16", 1024, 8448, 256), ("fp8", 1024, 8448, 640), ("i8", 1024, 8448, 640)])
def test_column_split_with_a_rest_of_few_tiles(kind, m, n, k):
    """The columns behind the whole rounds, few enough for tiles of another K step, have the bits that one launch gives them."""
    split, whole = _split_and_whole(kind, m, n, k)
    assert torch.equal(split, whole)


@pytest.mark.parametrize("kind,m,n,k", [("bf16", 1280, 13312, 1024), ("f16", 4096, 4360, 1024), ("fp8", 1280, 13312, 2048), ("i8", 1280, 13312, 2048)])
def test_column_split_over_both_kernels_of_the_tile(kind, m, n, k):
    """A split whose columns in whole rounds run the eight-wave kernel where the whole would run the hand-scheduled one (see the host test of the route): the same bits."""
    split, whole = _split_and_whole(kind, m, n, k)
    assert torch.equal(split, whole)
