"""GPU parity: batched fused GEMM-GEMM (fp16) through the C ABI against the CPU oracle
(two chained ReferenceBatchedGemm with an fp16 intermediate). The operator is absent from the
reference snapshot: parity is unpinned by reference vectors, pinned by the oracle's brute-force
and closed-form tests. Tolerance rtol = atol = 1e-2."""
import numpy as np
import pytest

import composable_kernel_amd as ck
from composable_kernel_amd import capi
from composable_kernel_amd.host_tensor import uniform_f16, uniform_int8
from oracle import fast, lit

pytestmark = pytest.mark.gpu
RTOL = ATOL = 1e-2


def _close(out, ref):
    bad, max_err = lit.check_err_f16(out, ref, RTOL, ATOL)
    assert bad == 0, f"{bad} outside tolerance, max err {max_err}"


@pytest.mark.parametrize("shape", [
    # G, M, N, K, O
    (3, 128, 128, 64, 64), (2, 200, 136, 64, 64), (2, 96, 512, 32, 64), (1, 130, 260, 128, 128),
    (2, 64, 72, 40, 24), (5, 16, 8, 8, 8), (1, 256, 256, 96, 128),
])
def test_gemm_gemm_small_shapes(shape):
    import gpu_util
    G, M, N, K, O = shape
    a = uniform_f16((G, M, K), -0.5, 0.5, 900 + M)
    b0_gnk = uniform_f16((G, N, K), -0.5, 0.5, 901 + N)
    b1 = uniform_f16((G, N, O), -0.5, 0.5, 902 + O)
    out = gpu_util.gemm_gemm_f16(a, b0_gnk, b1)
    _close(out, lit.batched_gemm_gemm_f16(a, b0_gnk.transpose(0, 2, 1), b1))


def test_gemm_gemm_closed_form():
    import gpu_util
    G, M, N, K, O = 2, 128, 64, 32, 64
    out = gpu_util.gemm_gemm_f16(np.ones((G, M, K), np.float16), np.ones((G, N, K), np.float16),
                                 np.full((G, N, O), 0.25, np.float16))
    np.testing.assert_array_equal(out, np.full((G, M, O), K * N * 0.25, np.float16))


def test_gemm_gemm_config5():
    """Benchmark configuration 5: batch 64, (512x64)(64x512)(512x64), U[-0.5, 0.5]."""
    import gpu_util
    G, M, N, K, O = 64, 512, 512, 64, 64
    a = uniform_f16((G, M, K), -0.5, 0.5, 910)
    b0_gnk = uniform_f16((G, N, K), -0.5, 0.5, 911)
    b1 = uniform_f16((G, N, O), -0.5, 0.5, 912)
    out = gpu_util.gemm_gemm_f16(a, b0_gnk, b1)
    _close(out, fast.batched_gemm_gemm_f16(a, b0_gnk.transpose(0, 2, 1), b1))
    for g in (0, 63):
        _close(out[g:g + 1], lit.batched_gemm_gemm_f16(a[g:g + 1], b0_gnk[g:g + 1].transpose(0, 2, 1), b1[g:g + 1]))
    # batches are independent: permuting the batch permutes the output
    perm = np.random.default_rng(3).permutation(G)
    out2 = gpu_util.gemm_gemm_f16(a[perm], b0_gnk[perm], b1[perm])
    np.testing.assert_array_equal(out2.view(np.uint16), out[perm].view(np.uint16))


@pytest.mark.parametrize("instance", [capi.INSTANCE_AUTO, 0, 1, 2])
def test_gemm_gemm_config5_integer_operands_bit_exact(instance):
    """Benchmark configuration 5's shape on integers in [-3, 3]: the intermediate (|sum| <= 9 * 64) is exact in fp32
    and in its fp16 rounding, the output sums (|sum| <= 576 * 3 * 512 < 2^24) are exact in fp32 in any order, so the
    fp16 output must equal the rounded exact product bit for bit."""
    import gpu_util
    G, M, N, K, O = 64, 512, 512, 64, 64
    a = uniform_int8((G, M, K), -3, 3, 920).astype(np.float32)
    b0_gnk = uniform_int8((G, N, K), -3, 3, 921).astype(np.float32)
    b1 = uniform_int8((G, N, O), -3, 3, 922).astype(np.float32)
    exact = np.matmul(np.matmul(a, b0_gnk.transpose(0, 2, 1)), b1)
    assert np.abs(exact).max() < 60000
    out = gpu_util.gemm_gemm_f16(a.astype(np.float16), b0_gnk.astype(np.float16), b1.astype(np.float16),
                                 instance=instance)
    np.testing.assert_array_equal(out, exact.astype(np.float16))


def test_gemm_gemm_unsupported():
    import torch
    d = torch.zeros(1 << 16, dtype=torch.float16, device="cuda")
    op = ck.DeviceBatchedGemmGemmF16()
    arg = op.MakeArgumentPointer(d, d, d, d, 64, 64, 256, 64, 1, 256, 256, 64, 64, 0, 0, 0, 0)
    assert not op.IsSupportedArgument(arg)          # K > 128
    with pytest.raises(RuntimeError):
        op.MakeInvokerPointer().Run(arg)


@pytest.mark.parametrize("K", [8, 32, 64, 128])
@pytest.mark.parametrize("instance", [0, 1, 2])
def test_columns_of_the_intermediate_in_order(K, instance):
    """Every column of the intermediate meets its own row of B1: B0 is a scaled selection, so that the intermediate holds one value
    of A per column, and B1's rows are all different. Small integers, exact in fp16: one misplaced fragment row shows."""
    import torch
    import gpu_util
    M, N, O = 130, 300, 64
    a = torch.randint(-2, 3, (1, M, K), device="cuda").half()
    b0 = torch.zeros((1, N, K), device="cuda", dtype=torch.float16)
    n = torch.arange(N, device="cuda")
    b0[0, n, (n * 7 + n // K) % K] = (n % 3 - 1).half()
    b1 = ((n[:, None] * 5 + torch.arange(O, device="cuda")[None, :] * 3) % 7 - 3).half()[None].contiguous()
    c = torch.full((1, M, O), float("nan"), device="cuda", dtype=torch.float16)
    op = ck.DeviceBatchedGemmGemmF16(instance)
    arg = op.MakeArgumentPointer(a, b0, b1, c, M, N, K, O, 1, K, K, O, O, M * K, N * K, N * O, M * O)
    assert op.IsSupportedArgument(arg)
    op.MakeInvokerPointer().Run(arg, ck.StreamConfig(gpu_util.stream()))
    torch.cuda.synchronize()
    want = (a[0].double() @ b0[0].double().T) @ b1[0].double()  # |sums| <= 300 * 2 * 3: exact
    assert torch.equal(c[0].double(), want)


@pytest.mark.parametrize("softmax", [False, True])
def test_batches_past_one_launch(softmax):
    """More workgroups than one launch has threads for in 32 bits (2^23 of 512 threads)."""
    import torch
    import gpu_util
    G, K = (1 << 23) + 24, 8
    n = torch.arange(G, device="cuda")
    a, b0, b1 = (((n % m)[:, None] + torch.arange(K, device="cuda")[None, :] % 3 - 3).half() for m in (5, 7, 11))
    c = torch.full((G, K), float("nan"), device="cuda", dtype=torch.float16)
    dims = (1, 1, K, K, G, K, K, K, K, K, K, K, K)
    if softmax:  # one column: its probability is 1
        op = ck.DeviceBatchedGemmSoftmaxGemmF16(MaskOutUpperTriangle=True)
        arg = op.MakeArgumentPointer(a, b0, b1, c, *dims, ck.PassThrough(), ck.PassThrough(), ck.Scale(1.0))
        want = b1
    else:
        op = ck.DeviceBatchedGemmGemmF16()
        arg = op.MakeArgumentPointer(a, b0, b1, c, *dims)
        want = ((a.float() * b0.float()).sum(1, keepdim=True) * b1.float()).half()  # (small integers: exact)
    assert op.IsSupportedArgument(arg)
    op.MakeInvokerPointer().Run(arg, ck.StreamConfig(gpu_util.stream()))
    torch.cuda.synchronize()
    assert torch.equal(c, want)


@pytest.mark.parametrize("G, M, N, K, O", [
    (4, 130, 1025, 32, 32), (3, 65, 1152, 64, 64), (1, 64, 1290, 64, 24), (2, 33, 1300, 128, 128), (1, 200, 1311, 96, 40), (2, 1, 1281, 24, 104),   # 4 shares
    (110, 129, 770, 32, 32), (129, 128, 1400, 40, 64), (100, 130, 1281, 128, 120), (98, 65, 1295, 80, 72),                                      # 2
    (2, 129, 448, 32, 32), (2, 133, 479, 8, 24), (257, 33, 289, 32, 32), (129, 1, 768, 64, 40), (257, 65, 577, 64, 64), (2, 133, 264, 128, 128),
    (2, 31, 161, 72, 128), (257, 40, 66, 128, 128), (3, 97, 327, 40, 128), (1, 260, 385, 128, 72),                                              # 1
    (2, 129, 447, 32, 32), (2, 64, 1100, 64, 64), (2, 65, 200, 128, 128), (2, 130, 1000, 128, 32)])                                             # steps of 128
def test_gemm_gemm_on_both_sides_of_the_32_row_kernels_rule(G, M, N, K, O):
    """Units, shares and rows that end anywhere, NaNs between the rows of A, B0 and B1, nothing written between those of C."""
    import torch
    import gpu_util
    pads = (8, 24, 16, 8)
    ops = [uniform_f16((G, x, y), -0.5, 0.5, 930 + i) for i, (x, y) in enumerate(((M, K), (N, K), (N, O)))]
    dev = []
    for x, pad in zip(ops, pads):
        buf = np.full(x.shape[:2] + (x.shape[2] + pad,), np.nan, np.float16)
        buf[..., :x.shape[2]] = x
        dev.append(torch.from_numpy(buf.view(np.int16)).cuda())
    c = torch.full((G, M, O + pads[3]), 0x7E00, dtype=torch.int16, device="cuda")
    sa, sb0, sb1, sc = K + pads[0], K + pads[1], O + pads[2], O + pads[3]
    op = ck.DeviceBatchedGemmGemmF16()
    arg = op.MakeArgumentPointer(*dev, c, M, N, K, O, G, sa, sb0, sb1, sc, M * sa, N * sb0, N * sb1, M * sc)
    assert op.IsSupportedArgument(arg), capi.last_error()
    op.MakeInvokerPointer().Run(arg, ck.StreamConfig(gpu_util.stream()))
    torch.cuda.synchronize()
    out = c.cpu().numpy().view(np.float16)
    assert np.all(out[..., O:].view(np.uint16) == 0x7E00), "wrote between the C rows"
    a, b0, b1 = ops
    for g in {0, G - 1}:
        _close(out[g:g + 1, :, :O], lit.batched_gemm_gemm_f16(a[g:g + 1], b0[g:g + 1].transpose(0, 2, 1), b1[g:g + 1]))
    # against float64, with the intermediate rounded to fp16 as the operator rounds it: a fp32 sum that lies next to a rounding boundary may
    # round to the neighbour, 2^-11 of itself (|.| <= K / 4), once in about 2^11 / K of them, and the result to 2^-11 of itself
    s = (a[0].astype(np.float64) @ b0[0].astype(np.float64).T).astype(np.float32).astype(np.float16)
    want = s.astype(np.float64) @ b1[0].astype(np.float64)
    assert np.linalg.norm(out[0, :, :O] - want) <= 6e-4 * np.linalg.norm(want)


@pytest.mark.parametrize("G, M, N, K", [(2, 133, 479, 32), (4, 130, 1025, 32), (1, 260, 385, 128)])
def test_gemm_gemm_nan_row_stays_in_its_row(G, M, N, K):
    import gpu_util
    a, b0, b1 = (uniform_f16((G, x, K), -0.5, 0.5, 940 + i) for i, x in enumerate((M, N, N)))
    clean = gpu_util.gemm_gemm_f16(a, b0, b1)
    for row in (0, 31, M - 1):
        x = a.copy()
        x[0, row, 3] = np.nan
        out = gpu_util.gemm_gemm_f16(x, b0, b1)
        assert np.all(np.isnan(out[0, row]))
        keep = np.arange(M) != row
        np.testing.assert_array_equal(out[:, keep].view(np.uint16), clean[:, keep].view(np.uint16))
