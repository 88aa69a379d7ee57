"""GPU parity of the GEMM for operands that are no whole 16-byte vectors (csrc/gemm_ragged.hpp) where it can go wrong: all of
its tiles (128 x 128 from 256 C tiles on, 64 x 64, 64 x 32 or 32 x 32 below, by their rows per CU), K below, at and just past one, two, three and four K tiles of 128
bytes, extents one short of and one past a C tile, fewer elements than one vector in the contiguous direction, operands that
end at their last element, all layouts. Integer operands small enough that every fp32 partial sum is exact: the result is the
rounded exact product, whatever the order of the sum, and int8 is compared bit for bit after wrapping."""
import ctypes

import pytest

import composable_kernel_amd as ck
from composable_kernel_amd import capi

pytestmark = pytest.mark.gpu

LAYOUTS = {"mk_nk": (ck.RowMajor, ck.ColumnMajor), "km_kn": (ck.ColumnMajor, ck.RowMajor),
           "km_nk": (ck.ColumnMajor, ck.ColumnMajor), "mk_kn": (ck.RowMajor, ck.RowMajor)}


# one problem for each tile below the 128 x 128 one, one element over or under whole tiles
SMALL = {(32, 32): (67, 93), (64, 32): (705, 497), (64, 64): (1021, 1003)}


class _Tile(ctypes.Structure):
    _fields_ = [("m", ctypes.c_int), ("n", ctypes.c_int)]


def _tile(M, N, batch=1):
    """rows and columns of the C tile that the problem runs on"""
    if capi.lib()._ZN3ckx11ragged_tileEiii(M, N, batch) == 128:
        return 128, 128
    f = capi.lib()._ZN3ckx17ragged_small_tileEiii
    f.argtypes, f.restype = [ctypes.c_int] * 3, _Tile
    t = f(M, N, batch)
    return t.m, t.n


def _run(kind, layout, M, N, K, off):
    import torch
    import gpu_util
    g = torch.Generator(device="cuda").manual_seed(1000 * M + 10 * N + K)
    dt = {"i8": torch.int8, "f16": torch.float16, "bf16": torch.bfloat16}[kind]
    al, bl = LAYOUTS[layout]

    def operand(shape):
        x = torch.randint(-3, 4, shape, generator=g, device="cuda").to(dt)
        buf = torch.full((x.numel() + off,), 100 if kind == "i8" else float("nan"), dtype=dt, device="cuda")
        buf[off:] = x.reshape(-1)
        return x, buf, buf.data_ptr() + off * x.element_size()

    a, buf_a, pa = operand((K, M) if al is ck.ColumnMajor else (M, K))
    b, buf_b, pb = operand((K, N) if bl is ck.RowMajor else (N, K))
    c = torch.full((M + 1, N), 77, dtype=dt, device="cuda")
    op = {"i8": ck.DeviceGemmInt8, "f16": ck.DeviceGemmF16, "bf16": ck.DeviceGemmBF16}[kind](ALayout=al, BLayout=bl)
    arg = op.MakeArgumentPointer(pa, pb, c, M, N, K, a.shape[1], b.shape[1], N)
    assert op.IsSupportedArgument(arg), capi.last_error()
    op.MakeInvokerPointer().Run(arg, ck.StreamConfig(gpu_util.stream()))
    torch.cuda.synchronize()
    a_mk = (a.T if al is ck.ColumnMajor else a).float().contiguous()
    b_kn = (b if bl is ck.RowMajor else b.T).float().contiguous()
    want = a_mk @ b_kn  # |sum| <= 9 K < 2^24: exact in fp32
    want = want.to(torch.int32).to(torch.int8) if kind == "i8" else want.to(dt)
    assert torch.equal(c[:M], want), f"{kind} {layout} {M} x {N} x {K}: {int((c[:M] != want).sum())} elements differ"
    assert bool((c[M] == 77).all()), "wrote past the last row"


@pytest.mark.parametrize("layout", sorted(LAYOUTS))
@pytest.mark.parametrize("kind", ["i8", "f16", "bf16"])
@pytest.mark.parametrize("tile", sorted(SMALL))
def test_k_around_the_k_tiles(kind, layout, tile):
    kt = 128 if kind == "i8" else 64
    M, N = SMALL[tile]
    assert _tile(M, N) == tile
    for tiles in range(0, 7):
        for d in (-1, 0, 1):
            K = tiles * kt + d
            if K > 0:
                _run(kind, layout, M, N, K, 1)


@pytest.mark.parametrize("layout", sorted(LAYOUTS))
@pytest.mark.parametrize("kind", ["i8", "f16", "bf16"])
@pytest.mark.parametrize("shape", [(63, 65, 131), (65, 63, 200), (1, 127, 129), (129, 1, 127), (5, 7, 300), (15, 17, 9), (2, 3, 1),
                                   (2047, 2049, 195), (2049, 2047, 321), (2000, 2001, 64)])
def test_tile_edges(kind, layout, shape):
    _run(kind, layout, *shape, off=0)
    _run(kind, layout, *shape, off=3)


@pytest.mark.parametrize("layout", sorted(LAYOUTS))
@pytest.mark.parametrize("kind", ["i8", "f16", "bf16"])
@pytest.mark.parametrize("M, N, tile", [(31, 33, (32, 32)), (33, 31, (32, 32)), (65, 1, (32, 32)), (705, 497, (64, 32)), (703, 511, (64, 32)),
                                        (1021, 1003, (64, 64)), (963, 1023, (64, 64))])
def test_small_tiles(kind, layout, M, N, tile):
    """32 x 32, 64 x 32 and 64 x 64 tiles at their edges, K around two K tiles"""
    assert _tile(M, N) == tile
    for K in (127, 129, 259):
        _run(kind, layout, M, N, K, off=0)
        _run(kind, layout, M, N, K, off=5)


def test_batches_past_one_launch_dimension():
    """More than 2^24 workgroups of 256 threads in one launch: the threads along a grid dimension are counted in 32 bits."""
    import torch
    import gpu_util
    G, N = 65281, 32769
    g = torch.Generator(device="cuda").manual_seed(5)
    a, b = (torch.randint(-9, 10, (n,), generator=g, device="cuda").to(torch.int8) for n in (G, N))
    c = torch.full((G, N), 77, dtype=torch.int8, device="cuda")
    op = ck.DeviceBatchedGemmInt8()
    arg = op.MakeArgumentPointer(a, b, c, 1, N, 1, 1, 1, N, 1, 0, N, G)
    assert op.IsSupportedArgument(arg), capi.last_error()
    op.MakeInvokerPointer().Run(arg, ck.StreamConfig(gpu_util.stream()))
    torch.cuda.synchronize()
    for i in range(0, G, 8192):
        assert torch.equal(c[i:i + 8192], a[i:i + 8192, None] * b[None, :]), f"batches from {i} on differ"


@pytest.mark.parametrize("kind", ["i8", "f16", "bf16"])
@pytest.mark.parametrize("K", [1, 7, 15, 31, 33, 63, 65])
def test_k_below_one_vector_and_half_a_k_tile(kind, K):
    """Rows of less than one vector are read element by element (int8 with another order of the slots), and a second k-step past
    K is left out, in C tiles of full, partial and single rows."""
    for M, N in ((147, 869), (64, 65), (1, 63), (130, 3), *SMALL.values()):
        _run(kind, "mk_nk", M, N, K, off=1)
        _run(kind, "km_nk", M, N, K, off=0)
        _run(kind, "mk_kn", M, N, K, off=1)


# ---- epilogues: 16 columns per lane on the 128 x 128 tile (256 of them and more) where B is K-contiguous, 8 on 64 x 64, 4 on 64 x 32 and 32 x 32
def _big(kind, M, N, K, lda, ldb, seed):
    """Small integers with leading dimensions of their own: fp16 results and int8 accumulators are exact."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    dt = torch.int8 if kind == "i8" else torch.float16
    a = torch.randint(-3, 4, (M, lda), generator=g, device="cuda").to(dt)
    b = torch.randint(-3, 4, (N, ldb), generator=g, device="cuda").to(dt)
    return a, b, a[:, :K].float() @ b[:, :K].float().T.contiguous()


def _requant(acc, sg, sr, rounded):
    """The two requantisations in fp32, operation by operation."""
    import torch
    sg, sr = torch.tensor(sg, device="cuda"), torch.tensor(sr, device="cuda")  # fp32, as the kernel's arguments
    if rounded:
        x = (acc * sg).round().clamp(-128, 127).clamp_min(0)
        return (x * sr).round().clamp(-128, 127).to(torch.int8)
    x = (acc * sg).clamp(-128, 127).clamp_min(0)
    return (x * sr).clamp(-128, 127).to(torch.int8)  # (truncating)


@pytest.mark.parametrize("epilogue", ["rounded", "literal", "per_column", "per_column_relu"])
@pytest.mark.parametrize("shape, tile", [((2047, 2049, 195, 201, 197, 2051), (128, 128)), ((2100, 2000, 65, 65, 67, 2003), (128, 128))] +
                         [((M, N, 451, 453, 455, N + 2), tile) for tile, (M, N) in sorted(SMALL.items())])
def test_int8_epilogues(epilogue, shape, tile):
    import torch
    import gpu_util
    M, N, K, lda, ldb, ldc = shape
    assert _tile(M, N) == tile
    a, b, acc = _big("i8", M, N, K, lda, ldb, 21)
    c = torch.full((M, ldc), 77, dtype=torch.int8, device="cuda")
    if epilogue.startswith("per_column"):
        scales = torch.rand((N,), device="cuda") * 0.4
        relu = epilogue == "per_column_relu"
        op = ck.DeviceGemmMultipleDInt8()
        arg = op.MakeArgumentPointer(a, b, [scales], c, M, N, K, lda, ldb, [0], ldc, None, None,
                                     ck.ActivationMul2Clamp(ck.Relu() if relu else ck.PassThrough()))
        want = (scales * (acc.clamp_min(0) if relu else acc)).clamp(-128, 127).to(torch.int8)
    else:
        op = ck.DeviceGemmInt8()
        arg = op.MakeArgumentPointer(a, b, c, M, N, K, lda, ldb, ldc, None, None, ck.RequantReluRequant(0.3, 0.7, rounded=epilogue == "rounded"))
        want = _requant(acc, 0.3, 0.7, epilogue == "rounded")
    assert op.IsSupportedArgument(arg), capi.last_error()
    op.MakeInvokerPointer().Run(arg, ck.StreamConfig(gpu_util.stream()))
    torch.cuda.synchronize()
    assert torch.equal(c[:, :N], want), f"{int((c[:, :N] != want).sum())} elements differ"
    assert bool((c[:, N:] == 77).all()), "wrote outside the C rows"


@pytest.mark.parametrize("functor", ["relu_add", "bilinear"])
@pytest.mark.parametrize("M, N, K, tile", [(2049, 2047, 131, (128, 128))] + [(M, N, 227, tile) for tile, (M, N) in sorted(SMALL.items())])
def test_d_operands_on_any_element(functor, M, N, K, tile):
    import torch
    import gpu_util
    ldd, ldc = N + 6, N + 2
    assert _tile(M, N) == tile
    a, b, acc = _big("f16", M, N, K, K + 2, K + 4, 22)
    d = [torch.randint(-50, 51, (M * ldd + 1,), device="cuda").half() for _ in range(2)]
    rows = [x[1:].reshape(M, ldd)[:, :N].float() for x in d]
    cde, nd, want = (ck.AddReluAdd(), 2, (acc + rows[0]).clamp_min(0) + rows[1]) if functor == "relu_add" else \
        (ck.Bilinear(0.5, 2.0), 1, 0.5 * acc + 2.0 * rows[0])
    e = torch.full((M, ldc), 7, dtype=torch.float16, device="cuda")
    op = ck.DeviceGemmMultipleDF16()
    arg = op.MakeArgumentPointer(a, b, [x.data_ptr() + 2 for x in d[:nd]], e, M, N, K, K + 2, K + 4, [ldd] * nd, ldc, None, None, cde)
    assert op.IsSupportedArgument(arg), capi.last_error()
    op.MakeInvokerPointer().Run(arg, ck.StreamConfig(gpu_util.stream()))
    torch.cuda.synchronize()
    assert torch.equal(e[:, :N], want.half()) and bool((e[:, N:] == 7).all())


@pytest.mark.parametrize("kind", ["i8", "f16"])
@pytest.mark.parametrize("G, M, N, K, large", [(70, 250, 255, 67, True), (70, 129, 131, 67, False), (300, 127, 121, 33, True)])
def test_batches_on_both_tiles(kind, G, M, N, K, large):
    """Batches whose tiles add up past 256 although one has a few; odd batch strides, the gaps between the C batches untouched."""
    import torch
    import gpu_util
    assert _tile(M, N, G) == ((128, 128) if large else (64, 64))
    g = torch.Generator(device="cuda").manual_seed(23)
    dt = torch.int8 if kind == "i8" else torch.float16
    bsa, bsb, bsc = M * K + 3, N * K + 5, M * N + 7
    a, b = (torch.randint(-3, 4, (G, bs), generator=g, device="cuda").to(dt) for bs in (bsa, bsb))
    c = torch.full((G, bsc), 77, dtype=dt, device="cuda")
    op = (ck.DeviceBatchedGemmInt8 if kind == "i8" else ck.DeviceBatchedGemmF16)()
    arg = op.MakeArgumentPointer(a, b, c, M, N, K, K, K, N, bsa, bsb, bsc, G)
    assert op.IsSupportedArgument(arg), capi.last_error()
    op.MakeInvokerPointer().Run(arg, ck.StreamConfig(gpu_util.stream()))
    torch.cuda.synchronize()
    for i in range(G):
        want = a[i, :M * K].reshape(M, K).float() @ b[i, :N * K].reshape(N, K).float().T.contiguous()
        want = want.to(torch.int32).to(torch.int8) if kind == "i8" else want.half()
        assert torch.equal(c[i, :M * N].reshape(M, N), want), f"batch {i}"
    assert bool((c[:, M * N:] == 77).all()), "wrote between the C batches"
