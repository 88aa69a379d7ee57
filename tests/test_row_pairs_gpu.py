"""GPU parity of the 128 x 64 row pairs and 64 x 128 column pairs that run behind the four-stage 64 x 64 instance (csrc/tile_pairs.hip): bit for bit what the
two-stage 64 x 64 instance gives for the same problem (each element is the same sum in the same order), at the edges of the line between one
tile and a pair, with rows that end in a pair's first half, one K tile and more than the three stages hold, K splits, every
epilogue, convolutions and batches, and the exact result (small integers) by another way."""
import ctypes

import numpy as np
import pytest

import composable_kernel_amd as ck
from composable_kernel_amd import capi
from oracle import fast

pytestmark = pytest.mark.gpu
FOUR_STAGE, TWO_STAGE = 8, 4


def _pays(M, N, runs=1):
    f = capi.lib()._ZN3ckx13row_pairs_payElll
    f.argtypes, f.restype = [ctypes.c_long] * 3, ctypes.c_bool
    return f(M, N, runs)


def _columns_pay(M, N, ksplit=1, batch=1):
    f = capi.lib()._ZN3ckx16column_pairs_payEllll
    f.argtypes, f.restype = [ctypes.c_long] * 4, ctypes.c_bool
    return not _pays(M, N, ksplit * batch) and f(M, N, ksplit, batch)


def _both(make, c):
    """make(instance) -> (operator, argument writing c); the results of both instances"""
    import torch
    import gpu_util
    out = []
    for instance in (FOUR_STAGE, TWO_STAGE):
        c.fill_(77)
        op, arg = make(instance)
        assert op.IsSupportedArgument(arg), capi.last_error()
        op.MakeInvokerPointer().Run(arg, ck.StreamConfig(gpu_util.stream()))
        torch.cuda.synchronize()
        out.append(c.clone())
    assert torch.equal(out[0], out[1]), f"{int((out[0] != out[1]).sum())} elements differ"
    return out[0]


def _operand(kind, shape, seed):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    dt = {"i8": torch.int8, "f16": torch.float16, "bf16": torch.bfloat16}[kind]
    return torch.randint(-9, 10, shape, generator=g, device="cuda").to(dt)


def test_the_line():
    assert not _pays(128, 64 * 128)                                    # one 64 x 64 workgroup per CU
    assert _pays(128, 64 * 129) and not _pays(64, 64 * 300)            # two, one row tile
    assert _pays(192, 64 * 100) and not _pays(192, 64 * 129)           # 200 pairs for 300; 258 for 387
    assert _pays(128, 4096, 4) and not _pays(128, 4096, 2)
    assert _columns_pay(64, 64 * 300) and not _columns_pay(64, 64 * 256) and not _columns_pay(128, 64 * 129)
    assert _columns_pay(64, 4096, 8) and not _columns_pay(192, 2048, 5) and _columns_pay(192, 2048, 1, 5)


@pytest.mark.parametrize("M, N, K", [(65, 8260, 128), (67, 9000, 64), (127, 8257, 1040), (128, 8256, 512), (150, 6000, 272), (700, 2500, 656), (1020, 1900, 400),
                                     (1, 64 * 257, 128), (63, 20000, 272), (64, 32705, 64), (130, 8255, 528), (190, 8256, 1040), (300, 5000, 400)])
@pytest.mark.parametrize("form", ["i8", "i8_rounded", "i8_per_column", "f16", "f16_add_relu_add", "bf16"])
def test_gemm(form, M, N, K):
    import torch
    assert _pays(M, N) or _columns_pay(M, N)
    kind = form.split("_")[0]
    a, b = _operand(kind, (M, K), 1), _operand(kind, (N, K), 2)
    c = torch.empty((M + 1, N), dtype=a.dtype, device="cuda")
    d = [_operand("f16", (N,), 3), _operand("f16", (M, N), 4)]
    scales = torch.rand((N,), device="cuda") * 0.4

    def make(instance):
        if form == "i8_per_column":
            op = ck.DeviceGemmMultipleDInt8(instance)
            return op, op.MakeArgumentPointer(a, b, [scales], c, M, N, K, K, K, [0], N, None, None, ck.ActivationMul2Clamp(ck.Relu()))
        if form == "f16_add_relu_add":
            op = ck.DeviceGemmMultipleDF16(instance)
            return op, op.MakeArgumentPointer(a, b, d, c, M, N, K, K, K, [0, N], N, None, None, ck.AddReluAdd())
        op = {"i8": ck.DeviceGemmInt8, "f16": ck.DeviceGemmF16, "bf16": ck.DeviceGemmBF16}[kind](instance)
        cop = ck.RequantReluRequant(0.02, 0.7, rounded=True) if form == "i8_rounded" else ck.PassThrough()
        return op, op.MakeArgumentPointer(a, b, c, M, N, K, K, K, N, None, None, cop)

    got = _both(make, c)
    assert bool((got[M] == 77).all()), "wrote past the last row"
    acc = a.float() @ b.float().T.contiguous()  # |sums| < 2^24: the exact product
    if kind == "i8":
        acc = acc.to(torch.int32).cpu().numpy()
        want = fast.epilogue_i8_mul2_clamp(acc, scales.cpu().numpy(), True) if form == "i8_per_column" else \
            fast.epilogue_i8(acc, fast.EPI_REQUANT_RND if form == "i8_rounded" else fast.EPI_PASSTHROUGH, 0.02, 0.7)
        np.testing.assert_array_equal(got[:M].cpu().numpy(), want)
    else:
        assert torch.equal(got[:M], ((acc + d[0].float()).clamp_min(0) + d[1].float() if form == "f16_add_relu_add" else acc).to(a.dtype))


@pytest.mark.parametrize("kind", ["i8", "f16", "bf16"])
@pytest.mark.parametrize("layout", ["km_nk", "mk_kn", "km_kn"])
@pytest.mark.parametrize("M, N, K", [(80, 8272, 128), (176, 6000, 272), (1008, 1904, 528), (704, 2512, 64)])
def test_k_major(kind, layout, M, N, K):
    import torch
    assert _pays(M, N)
    la, lb = layout.split("_")
    a, b = _operand(kind, (M, K) if la == "mk" else (K, M), 13), _operand(kind, (N, K) if lb == "nk" else (K, N), 14)
    c = torch.empty((M + 1, N), dtype=a.dtype, device="cuda")
    lay = dict(ALayout=ck.RowMajor if la == "mk" else ck.ColumnMajor, BLayout=ck.ColumnMajor if lb == "nk" else ck.RowMajor)

    def make(instance):
        op = {"i8": ck.DeviceGemmInt8, "f16": ck.DeviceGemmF16, "bf16": ck.DeviceGemmBF16}[kind](instance, **lay)
        cop = ck.RequantReluRequant(0.02, 0.7, rounded=True) if kind == "i8" else ck.PassThrough()
        return op, op.MakeArgumentPointer(a, b, c, M, N, K, a.shape[1], b.shape[1], N, None, None, cop)

    got = _both(make, c)
    assert bool((got[M] == 77).all()), "wrote past the last row"
    a_mk, b_kn = (a if la == "mk" else a.T).float().contiguous(), (b.T if lb == "nk" else b).float().contiguous()
    acc = a_mk @ b_kn  # |sums| < 2^24: the exact product
    if kind == "i8":
        np.testing.assert_array_equal(got[:M].cpu().numpy(), fast.epilogue_i8(acc.to(torch.int32).cpu().numpy(), fast.EPI_REQUANT_RND, 0.02, 0.7))
    else:
        assert torch.equal(got[:M], acc.to(a.dtype))


@pytest.fixture
def force_runs():
    L = capi.lib()
    before = L.ckx_set_forced_k_runs(0)
    yield L.ckx_set_forced_k_runs
    L.ckx_set_forced_k_runs(before)


@pytest.mark.parametrize("kind", ["i8", "f16", "bf16"])
@pytest.mark.parametrize("M, N, K, runs", [(128, 4096, 1024, 4), (500, 1104, 1600, 3), (112, 2208, 2064, 5)])
def test_k_split_with_a_k_major_b(force_runs, kind, M, N, K, runs):
    """B K-major keeps its pairs under a K split (A K-major does not)."""
    import torch
    assert _pays(M, N, runs)
    a, b = _operand(kind, (M, K), 15), _operand(kind, (K, N), 16)
    c = torch.empty((M, N), dtype=a.dtype, device="cuda")
    force_runs(runs)

    def make(instance):
        op = {"i8": ck.DeviceGemmInt8, "f16": ck.DeviceGemmF16, "bf16": ck.DeviceGemmBF16}[kind](instance, BLayout=ck.RowMajor)
        arg = op.MakeArgumentPointer(a, b, c, M, N, K, K, N, N, None, None, ck.PassThrough())
        need = op.GetWorkSpaceSize(arg)
        assert need == runs * M * N * 4
        op.SetWorkSpacePointer(arg, torch.full((need,), 0x7F, dtype=torch.uint8, device="cuda"))
        return op, arg

    got, acc = _both(make, c), a.float() @ b.float()
    assert torch.equal(got, acc.to(torch.int32).to(torch.int8) if kind == "i8" else acc.to(a.dtype))


@pytest.mark.parametrize("kind", ["i8", "f16"])
@pytest.mark.parametrize("M, N, K, runs", [(128, 4096, 1024, 4), (100, 2200, 2064, 5), (500, 1100, 1600, 3), (40, 4100, 1552, 5), (64, 2816, 1024, 8)])
def test_k_split(kind, M, N, K, runs):
    import torch
    a, b = _operand(kind, (M, K), 5), _operand(kind, (N, K), 6)
    c = torch.empty((M, N), dtype=a.dtype, device="cuda")
    ws = torch.full((runs * M * N * 4 + 16,), 0x7F, dtype=torch.uint8, device="cuda")
    assert _pays(M, N, runs) or _columns_pay(M, N, runs)

    def make(instance):
        op = (ck.DeviceGemmInt8 if kind == "i8" else ck.DeviceGemmF16)(instance)
        arg = op.MakeArgumentPointer(a, b, c, M, N, K, K, K, N, None, None, ck.PassThrough())
        op.SetWorkSpacePointer(arg, ws, runs * M * N * 4)
        return op, arg

    before = capi.lib().ckx_set_forced_k_runs(runs)
    try:
        _both(make, c)
    finally:
        capi.lib().ckx_set_forced_k_runs(before)


@pytest.mark.parametrize("G, M, N, K, columns", [(5, 120, 1900, 272, False), (7, 60, 2700, 272, True)])
def test_batches(G, M, N, K, columns):
    import torch
    assert _columns_pay(M, N, 1, G) if columns else _pays(M, N, G)
    a, b = _operand("f16", (G, M, K), 7), _operand("f16", (G, N, K), 8)
    c = torch.empty((G, M, N), dtype=torch.float16, device="cuda")

    def make(instance):
        op = ck.DeviceBatchedGemmF16(instance)
        return op, op.MakeArgumentPointer(a, b, c, M, N, K, K, K, N, M * K, N * K, M * N, G)
    _both(make, c)


@pytest.mark.parametrize("form", ["i8", "f16", "f16_bias_relu", "f16_bias_relu_add", "i8_3d", "f16_3d"])
@pytest.mark.parametrize("N, C, K, hw, f, stride, runs", [(32, 64, 256, 14, 3, 1, 1), (9, 48, 72, 41, 5, 1, 1), (5, 32, 264, 63, 3, 2, 1),
                                                          (8, 64, 256, 14, 3, 1, 3), (3, 48, 136, 29, 3, 1, 4)])
def test_conv(force_runs, form, N, C, K, hw, f, stride, runs):
    import torch
    nd = 3 if form.endswith("3d") else 2
    if nd == 3:
        N, hw, K, runs = (2, 13 * stride - (stride - 1), 264, 1) if runs == 1 else (1, 12, 264, 3)
    ho = (hw + 2 * (f // 2) - f) // stride + 1
    M = N * ho ** nd
    assert _pays(M, K, runs)
    kind = form.split("_")[0]
    x, w = _operand(kind, (N, *[hw] * nd, C), 9), _operand(kind, (K, *[f] * nd, C), 10)
    bias, r = _operand("f16", (K,), 11), _operand("f16", (N, *[ho] * nd, K), 12)
    y = torch.empty((N, *[ho] * nd, K), dtype=x.dtype, device="cuda")
    geom = (N, K, C, [hw] * nd, [f] * nd, [ho] * nd, [stride] * nd, [1] * nd, [f // 2] * nd, [f // 2] * nd)
    force_runs(runs if runs > 1 else 0)

    def make(instance):
        if "bias" in form:
            op = ck.DeviceConv2dFwdBiasActivationF16(instance)
            if form.endswith("add"):
                arg = op.MakeArgumentPointer(x, w, y, bias, r, *geom, None, None, ck.AddReluAdd())
            else:
                arg = op.MakeArgumentPointer(x, w, y, bias, *geom, None, None, ck.AddRelu())
        else:
            if nd == 3:
                op = (ck.DeviceConvNdFwdInt8 if kind == "i8" else ck.DeviceConvNdFwdF16)(3, instance)
            else:
                op = (ck.DeviceConv2dFwdInt8 if kind == "i8" else ck.DeviceConv2dFwdF16)(instance)
            cop = ck.RequantReluRequant(0.02, 0.7, rounded=True) if kind == "i8" else ck.PassThrough()
            arg = op.MakeArgumentPointer(x, w, y, *geom, None, None, cop)
        if runs > 1:
            need = op.GetWorkSpaceSize(arg)
            assert need == runs * M * K * 4
            op.SetWorkSpacePointer(arg, torch.full((need,), 0x7F, dtype=torch.uint8, device="cuda"))
        return op, arg

    got, (hx, hw_) = _both(make, y).cpu().numpy(), (t.cpu().numpy() for t in (x, w))  # |sums| < 2^24: exact
    where = ([stride] * nd, [1] * nd, [f // 2] * nd)
    if "bias" in form:
        want = fast.conv2d_fwd_bias_relu_f16(hx, hw_, bias.cpu().numpy(), r.cpu().numpy() if form.endswith("add") else None, *where)
    else:
        want = fast.convnd_fwd(hx, hw_, *where, epi=fast.EPI_REQUANT_RND if kind == "i8" else fast.EPI_PASSTHROUGH, scale_gemm=0.02, scale_relu=0.7)
    np.testing.assert_array_equal(got, want)
