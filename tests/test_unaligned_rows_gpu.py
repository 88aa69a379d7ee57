"""GPU parity of the 16-byte C stores, D loads and K-split slices at rows that start on any element: leading dimensions and
base addresses of C (and D) that are no 16-byte vectors, around the 16-column groups a lane owns. K and the operand rows
stay whole vectors, so the vectorised instances run. Bit-exact: int8 by definition, 16-bit types on small integers (every
partial sum is an integer below 2^24, the rounded exact product is the only right answer)."""
import numpy as np
import pytest

import composable_kernel_amd as ck
from composable_kernel_amd import capi
from composable_kernel_amd.host_tensor import uniform_int8
from oracle import fast, lit

pytestmark = pytest.mark.gpu

# tile instances: four-/eight-wave 256 x 256, 128 x 64, 64 x 64, 256 x 64; skinny 1-row and 64-column; -1: automatic
INSTANCES = [-1, 0, 1, 3, 4, 7, 9, 13]


def _rows(M, N, ldc, off, fill, dtype):
    """An [M, ldc] C buffer whose first element sits `off` elements behind a 256-byte boundary, and its view."""
    import torch
    buf = torch.full((M * ldc + off + 64,), fill, dtype=dtype, device="cuda")
    return buf, buf.data_ptr() + off * buf.element_size()


@pytest.mark.parametrize("N", [1, 15, 17, 63, 255, 257, 515])
@pytest.mark.parametrize("kind", ["i8", "f16", "bf16"])
@pytest.mark.parametrize("instance", INSTANCES)
def test_gemm_rows_on_any_element(kind, N, instance):
    import torch
    import gpu_util
    M, K = (13 if instance >= 9 else 150), 256
    a, b = uniform_int8((M, K), -5, 5, 31 + N), uniform_int8((N, K), -5, 5, 32 + N)
    want = a.astype(np.float32) @ b.astype(np.float32).T
    tdt = {"i8": torch.int8, "f16": torch.float16, "bf16": torch.bfloat16}[kind]
    da, db = (torch.from_numpy(x).cuda().to(tdt) for x in (a, b))
    for off, pad in ((0, 0), (1, 2), (3, 7)):
        ldc = N + pad
        buf, pc = _rows(M, N, ldc, off, 77, tdt)
        op = {"i8": ck.DeviceGemmInt8, "f16": ck.DeviceGemmF16, "bf16": ck.DeviceGemmBF16}[kind](instance)
        c_op = ck.RequantReluRequant(0.02, 0.4, rounded=True) if kind == "i8" else None
        arg = op.MakeArgumentPointer(da, db, pc, M, N, K, K, K, ldc, None, None, c_op)
        assert op.IsSupportedArgument(arg), capi.last_error()
        op.MakeInvokerPointer().Run(arg, ck.StreamConfig(gpu_util.stream()))
        torch.cuda.synchronize()
        out = buf.cpu().float().numpy()
        assert np.all(out[:off] == 77) and np.all(out[off + M * ldc:] == 77), "wrote outside C"
        rows = out[off:off + M * ldc].reshape(M, ldc)
        assert np.all(rows[:, N:] == 77), "wrote outside the C rows"
        ref = fast.gemm_i8(a, b.T, lit.EPI_REQUANT_RND, 0.02, 0.4).astype(np.float32) if kind == "i8" else \
            torch.from_numpy(want).to(tdt).float().numpy()
        np.testing.assert_array_equal(rows[:, :N], ref, err_msg=f"{kind} N{N} ldc{ldc} offset {off} instance {instance}")


@pytest.mark.parametrize("N", [17, 131, 301])
@pytest.mark.parametrize("instance", [-1, 0, 1, 4])
@pytest.mark.parametrize("functor", ["relu", "relu_add", "bilinear"])
def test_d_operands_on_any_element(functor, N, instance):
    """D rows and bases off the 16-byte grid; integer values, so every functor is exact in fp32 and rounds once."""
    import torch
    import gpu_util
    M, K = 150, 128
    a, b = uniform_int8((M, K), -3, 3, 41), uniform_int8((N, K), -3, 3, 42)
    acc = a.astype(np.float32) @ b.astype(np.float32).T
    ldd = N + 3
    d_host = [uniform_int8((M, ldd), -50, 50, 43 + i).astype(np.float16) for i in range(2)]
    d_bufs = [torch.zeros(M * ldd + 1, dtype=torch.float16, device="cuda") for _ in d_host]
    for t, h in zip(d_bufs, d_host):
        t[1:] = torch.from_numpy(h.reshape(-1)).cuda()
    ptrs = [t.data_ptr() + 2 for t in d_bufs]
    d = [h[:, :N].astype(np.float32) for h in d_host]
    cde, n_d, want = {
        "relu": (ck.AddRelu(), 1, np.maximum(acc.astype(np.float16).astype(np.float32) + d[0], 0)),
        "relu_add": (ck.AddReluAdd(), 2, np.maximum(acc + d[0], 0) + d[1]),
        "bilinear": (ck.Bilinear(0.5, 2.0), 1, 0.5 * acc + 2.0 * d[0])}[functor]
    buf, pe = _rows(M, N, N + 1, 1, 7, torch.float16)
    op = ck.DeviceGemmMultipleDF16(instance)
    da, db = (torch.from_numpy(x).cuda().half() for x in (a, b))
    arg = op.MakeArgumentPointer(da, db, ptrs[:n_d], pe, M, N, K, K, K, [ldd] * n_d, N + 1, None, None, cde)
    assert op.IsSupportedArgument(arg), capi.last_error()
    op.MakeInvokerPointer().Run(arg, ck.StreamConfig(gpu_util.stream()))
    torch.cuda.synchronize()
    rows = buf.cpu().numpy()[1:1 + M * (N + 1)].reshape(M, N + 1)
    np.testing.assert_array_equal(rows[:, :N], want.astype(np.float16))
    assert np.all(rows[:, N:] == 7)


@pytest.mark.parametrize("N", [18, 65, 131])
@pytest.mark.parametrize("kind", ["i8", "f16"])
def test_split_k_slices_of_odd_rows(kind, N):
    import torch
    import gpu_util
    M, K, runs = 70, 1024, 3
    a, b = uniform_int8((M, K), -4, 4, 51), uniform_int8((N, K), -4, 4, 52)
    tdt = torch.int8 if kind == "i8" else torch.float16
    da, db = (torch.from_numpy(x).cuda().to(tdt) for x in (a, b))
    dc = torch.full((M, N), 77, dtype=tdt, device="cuda")
    op = (ck.DeviceGemmSplitKInt8 if kind == "i8" else ck.DeviceGemmSplitKF16)()
    arg = op.MakeArgumentPointer(da, db, dc, M, N, K, K, K, N, None, None,
                                 ck.RequantReluRequant(0.02, 0.4, rounded=True) if kind == "i8" else None, KBatch=runs)
    ws = torch.full((op.GetWorkSpaceSize(arg),), 0x55, dtype=torch.uint8, device="cuda")
    op.SetWorkSpacePointer(arg, ws)
    op.MakeInvokerPointer().Run(arg, ck.StreamConfig(gpu_util.stream()))
    torch.cuda.synchronize()
    want = fast.gemm_i8(a, b.T, lit.EPI_REQUANT_RND, 0.02, 0.4) if kind == "i8" else \
        (a.astype(np.float32) @ b.astype(np.float32).T).astype(np.float16)
    np.testing.assert_array_equal(dc.cpu().numpy(), want)


@pytest.mark.parametrize("K", [64, 65])
@pytest.mark.parametrize("instance", [-1, 1, 7])
def test_streamed_int8_rows_on_any_element(K, instance):
    """int8 outputs of 64 MiB and more are stored with the non-temporal hint, also at odd addresses and next to row ends in pieces
    (K = 65: the last instance of the family, which is the automatic choice)."""
    import torch
    import gpu_util
    if K % 16 and instance >= 0:
        pytest.skip("the tile instances take whole 16-byte vectors of K")
    M, N, ldc, off = 8300, 8191, 8193, 1
    g = torch.Generator(device="cuda").manual_seed(K)
    a, b = (torch.randint(-3, 4, (n, K), generator=g, device="cuda").to(torch.int8) for n in (M, N))
    buf, pc = _rows(M, N, ldc, off, 77, torch.int8)
    op = ck.DeviceGemmInt8(instance)
    arg = op.MakeArgumentPointer(a, b, pc, M, N, K, K, K, ldc)
    assert op.IsSupportedArgument(arg), capi.last_error()
    op.MakeInvokerPointer().Run(arg, ck.StreamConfig(gpu_util.stream()))
    torch.cuda.synchronize()
    rows = buf[off:off + M * ldc].reshape(M, ldc)
    want = (a.float() @ b.float().T.contiguous()).to(torch.int32).to(torch.int8)
    assert torch.equal(rows[:, :N], want) and bool((rows[:, N:] == 77).all())
    assert bool((buf[:off] == 77).all()) and bool((buf[off + M * ldc:] == 77).all())


@pytest.mark.parametrize("C, K", [(3, 45), (16, 43)])
def test_streamed_int8_conv_outputs_on_any_element(C, K):
    """The same for convolutions: the few-channel kernel and the im2col tile kernels, an odd number of output channels."""
    import torch
    import gpu_util
    N, H = 32, 224
    g = torch.Generator(device="cuda").manual_seed(C)
    x = torch.randint(-3, 4, (N, H, H, C), generator=g, device="cuda").to(torch.int8)
    w = torch.randint(-3, 4, (K, 3, 3, C), generator=g, device="cuda").to(torch.int8)
    y = torch.full((N * H * H * K + 1,), 77, dtype=torch.int8, device="cuda")
    op = ck.DeviceConv2dFwdInt8()
    arg = op.MakeArgumentPointer(x, w, y.data_ptr() + 1, N, K, C, [H, H], [3, 3], [H, H], [1, 1], [1, 1], [1, 1], [1, 1], None, None, None)
    assert op.IsSupportedArgument(arg), capi.last_error()
    op.MakeInvokerPointer().Run(arg, ck.StreamConfig(gpu_util.stream()))
    torch.cuda.synchronize()
    assert int(y[0]) == 77
    out = y[1:].reshape(N, H, H, K)
    for i in range(N):
        pixels = torch.nn.functional.pad(x[i].float(), (0, 0, 1, 1, 1, 1))
        want = sum(pixels[r:r + H, s:s + H] @ w[:, r, s].float().T.contiguous() for r in range(3) for s in range(3))
        assert torch.equal(out[i], want.to(torch.int32).to(torch.int8)), f"image {i}"
