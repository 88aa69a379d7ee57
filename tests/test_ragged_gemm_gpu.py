"""GPU parity of the GEMM for operands that are no whole 16-byte vectors (csrc/gemm_ragged.hpp) where it can go wrong: both of
its tiles (128 x 128 from 256 C tiles on, 64 x 64 below), K below, at and just past one, two, three and four K tiles of 128
bytes, extents one short of and one past a C tile, fewer elements than one vector in the contiguous direction, operands that
end at their last element, all layouts. Integer operands small enough that every fp32 partial sum is exact: the result is the
rounded exact product, whatever the order of the sum, and int8 is compared bit for bit after wrapping."""
import numpy as np
import pytest

import composable_kernel_amd as ck
from composable_kernel_amd import capi

pytestmark = pytest.mark.gpu

LAYOUTS = {"mk_nk": (ck.RowMajor, ck.ColumnMajor), "km_kn": (ck.ColumnMajor, ck.RowMajor),
           "km_nk": (ck.ColumnMajor, ck.ColumnMajor), "mk_kn": (ck.RowMajor, ck.RowMajor)}


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
def test_k_around_the_k_tiles(kind, layout):
    kt = 128 if kind == "i8" else 64
    for tiles in range(0, 7):
        for d in (-1, 0, 1):
            K = tiles * kt + d
            if K > 0:
                _run(kind, layout, 67, 93, K, 1)


@pytest.mark.parametrize("layout", sorted(LAYOUTS))
@pytest.mark.parametrize("kind", ["i8", "f16", "bf16"])
@pytest.mark.parametrize("shape", [(63, 65, 131), (65, 63, 200), (1, 127, 129), (129, 1, 127), (5, 7, 300), (15, 17, 9), (2, 3, 1),
                                   (2047, 2049, 195), (2049, 2047, 321), (2000, 2001, 64)])
def test_tile_edges(kind, layout, shape):
    _run(kind, layout, *shape, off=0)
    _run(kind, layout, *shape, off=3)


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
    for M, N in ((147, 869), (64, 65), (1, 63), (130, 3)):
        _run(kind, "mk_nk", M, N, K, off=1)
        _run(kind, "km_nk", M, N, K, off=0)
        _run(kind, "mk_kn", M, N, K, off=1)
