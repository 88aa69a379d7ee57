"""GPU parity of AUTO GEMMs whose K is no whole number of 16-byte vectors and that come with a workspace: the operands are copied to whole
vectors there (csrc/gemm_pack.hip) and the instances for those take over. K one to all but one element past a vector, K tile and row tile edges,
K-major operands whose extent ends inside a 16-byte chunk, NaNs (int8: 100) between the rows, operands that start at any element. Integer operands small
enough that every fp32 partial sum is exact: the result is the rounded exact product, whatever the route."""
import pytest

import composable_kernel_amd as ck
from composable_kernel_amd import capi

pytestmark = pytest.mark.gpu
LAYOUTS = {"mk_nk": (ck.RowMajor, ck.ColumnMajor), "km_kn": (ck.ColumnMajor, ck.RowMajor),
           "km_nk": (ck.ColumnMajor, ck.ColumnMajor), "mk_kn": (ck.RowMajor, ck.RowMajor)}
KINDS = {"i8": (1, ck.DeviceGemmInt8), "f16": (2, ck.DeviceGemmF16), "bf16": (2, ck.DeviceGemmBF16)}


def _copies(es, M, N, K):
    pitch = -(-K * es // 128) * 128
    return (M + N) * pitch


def _run(kind, layout, M, N, K, gap, off, workspace, c_op=None):
    """workspace: None, or bytes beyond (or short of) the copies and the byte that they start at."""
    import torch
    import gpu_util
    g = torch.Generator(device="cuda").manual_seed(M + 10 * N + K)
    es, device_op = KINDS[kind]
    dt = {"i8": torch.int8, "f16": torch.float16, "bf16": torch.bfloat16}[kind]
    al, bl = LAYOUTS[layout]

    def operand(rows, cols):
        x = torch.randint(-3, 4, (rows, cols), generator=g, device="cuda").to(dt)
        buf = torch.full((rows * (cols + gap) + off,), 100 if kind == "i8" else float("nan"), dtype=dt, device="cuda")
        buf[off:].view(rows, cols + gap)[:, :cols] = x
        return x, buf, buf.data_ptr() + off * es

    a, buf_a, pa = operand(*((K, M) if al is ck.ColumnMajor else (M, K)))
    b, buf_b, pb = operand(*((K, N) if bl is ck.RowMajor else (N, K)))
    c = torch.full((M + 1, N), 77, dtype=dt, device="cuda")
    op = device_op(ALayout=al, BLayout=bl)
    arg = op.MakeArgumentPointer(pa, pb, c, M, N, K, a.shape[1] + gap, b.shape[1] + gap, N, *((None, None, c_op) if c_op else ()))
    assert op.IsSupportedArgument(arg), capi.last_error()
    untouched = None
    if workspace is not None:
        spare, at = workspace
        need = op.GetWorkSpaceSize(arg)
        assert need >= _copies(es, M, N, K)
        ws = torch.full((need + spare + at + 64,), 0x7F, dtype=torch.uint8, device="cuda")
        op.SetWorkSpacePointer(arg, ws.data_ptr() + at, need + spare)
        untouched = ws[at + need + max(spare, 0):]
    for _ in range(2): # (the second run finds the copies of the first)
        op.MakeInvokerPointer().Run(arg, ck.StreamConfig(gpu_util.stream()))
    torch.cuda.synchronize()
    assert bool((c[M] == 77).all()), "wrote past the last row"
    assert untouched is None or bool((untouched == 0x7F).all()), "wrote past the workspace"
    want = (a.T if al is ck.ColumnMajor else a).float().contiguous() @ (b if bl is ck.RowMajor else b.T).float().contiguous()
    return c[:M], want, (ws if workspace is not None else None)


def _check(kind, got, want):
    import torch
    want = want.to(torch.int32).to(torch.int8) if kind == "i8" else want.to(got.dtype)
    assert torch.equal(got, want), f"{int((got != want).sum())} elements differ"


@pytest.mark.parametrize("kind", sorted(KINDS))
@pytest.mark.parametrize("layout", sorted(LAYOUTS))
@pytest.mark.parametrize("M, N, d", [(2049, 2047, -1), (2047, 2053, 1), (2305, 1921, 3)])
def test_copied_operands(kind, layout, M, N, d):
    for K in (1536 + d, 2048 + 8 + d): # (whole K tiles, and whole vectors that are no K tile, in 16 bits)
        for gap, off in ((0, 0), (5, 3)):
            got, want, ws = _run(kind, layout, M, N, K, gap, off, (0, 0))
            _check(kind, got, want)
            assert int((ws[:_copies(KINDS[kind][0], M, N, K)] != 0x7F).sum()) > 0, "the operands were not copied"


@pytest.mark.parametrize("kind", ["i8", "f16"])
def test_long_k_few_rows_and_a_split(kind):
    _check(kind, *_run(kind, "mk_nk", 333, 3001, 8001, 0, 0, (0, 0))[:2])
    _check(kind, *_run(kind, "mk_nk", 1500, 901, 4001, 1, 1, (0, 16))[:2])


@pytest.mark.parametrize("workspace", [None, (-(1 << 20), 0), (0, 8)])
@pytest.mark.parametrize("kind", ["i8", "f16"])
def test_without_a_usable_workspace_the_operands_are_taken_as_they_are(kind, workspace):
    got, want, ws = _run(kind, "mk_nk", 2049, 2047, 1537, 0, 0, workspace)
    _check(kind, got, want)
    assert ws is None or bool((ws == 0x7F).all())


def test_int8_epilogue_same_bytes_on_both_routes():
    import torch
    op = ck.RequantReluRequant(0.037, 0.7, rounded=True)
    for layout in sorted(LAYOUTS):
        with_copies = _run("i8", layout, 2049, 2047, 2045, 3, 1, (0, 0), op)[0]
        assert torch.equal(with_copies, _run("i8", layout, 2049, 2047, 2045, 3, 1, None, op)[0])


@pytest.mark.parametrize("layout", ["mk_nk", "km_kn"])
def test_d_operand_epilogues(layout):
    """The same exact sums through the same functor: equal, but for the functors' own fp32 rounding (an fp16 unit in the last place)."""
    import numpy as np
    from test_cde_ops_gpu import _run as run_d
    M, N, K = 1999, 1501, 2003
    rng = np.random.default_rng(7)
    a, b, d0, d1 = (rng.integers(-2, 3, s).astype(np.float16) for s in ((M, K), (K, N), (1, N), (M, N + 3)))
    for ds, strides, functor in (([d1], [N + 3], ck.Bilinear(0.5, 2.0)), ([d0, d1], [0, N + 3], ck.AddAddFastGelu())):
        out, plain = (run_d(a, b, ds, strides, functor, layout=layout, lde=N + 1, workspace=w).astype(np.float32) for w in (True, False))
        assert np.all(np.abs(out - plain) <= 2.0 ** -10 * np.abs(plain) + 2.0 ** -14)
