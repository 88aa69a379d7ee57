"""GPU parity of the few-channel conv kernel (csrc/conv_few.hpp) where it can go wrong: 1 .. 8 channels (every piece a pixel is
loaded in, both padded widths), output channels around the 16-, 32- and 64-channel blocks and more of them than one workgroup
holds, patches that end inside a row or a band, images wider than a patch, strides, dilations and one-sided padding, and an
infinite pixel, which may only reach the windows that hold it. Small integers: fp16 results are exact, so both data types
are compared bit for bit."""
import numpy as np
import pytest

import composable_kernel_amd as ck
from oracle import fast, lit

pytestmark = pytest.mark.gpu


def _ints(shape, seed, dtype):
    return np.random.default_rng(seed).integers(-3, 4, shape).astype(np.int8 if dtype == "i8" else np.float16)


@pytest.mark.parametrize("dtype", ["i8", "f16"])
@pytest.mark.parametrize("C", range(1, 9))
def test_channel_counts_and_output_blocks(dtype, C):
    import gpu_util
    if dtype == "f16" and C == 8:
        pytest.skip("a 16-byte pixel is the vectorised instances'")
    for i, (K, N, H, W, Y, X, s, d, p) in enumerate([(1, 2, 5, 7, 3, 3, (1, 1), (1, 1), (1, 1)),
                                                     (17, 1, 40, 33, 3, 5, (2, 1), (1, 1), (0, 2)),
                                                     (32, 3, 29, 131, 5, 5, (2, 2), (1, 1), (2, 2)),
                                                     (48, 1, 9, 300, 1, 1, (1, 1), (1, 1), (0, 0)),
                                                     (100, 1, 20, 17, 7, 7, (2, 2), (1, 2), (3, 6)),
                                                     (257, 1, 12, 12, 3, 3, (1, 3), (2, 1), (2, 0))]):
        inp, wei = _ints((N, H, W, C), 100 * C + i, dtype), _ints((K, Y, X, C), 200 * C + i, dtype)
        out = gpu_util.conv2d_fwd(inp, wei, s, d, p)
        want = (fast.conv2d_fwd_i8 if dtype == "i8" else fast.conv2d_fwd_f16)(inp, wei, s, d, p)
        np.testing.assert_array_equal(out, want, err_msg=f"C {C} K {K} {H} x {W} filter {Y} x {X}")


def test_more_weights_than_a_workgroup_holds():
    import gpu_util
    inp, wei = _ints((1, 20, 20, 7), 1, "f16"), _ints((600, 7, 7, 7), 2, "f16")
    np.testing.assert_array_equal(gpu_util.conv2d_fwd(inp, wei, (1, 1), (1, 1), (3, 3)),
                                  fast.conv2d_fwd_f16(inp, wei, (1, 1), (1, 1), (3, 3)))


def test_filter_beyond_the_lds():
    """A reach of 200 rows does not fit: the element-wise kernel takes the layer, as before."""
    import gpu_util
    inp, wei = _ints((1, 210, 220, 5), 3, "f16"), _ints((8, 3, 3, 5), 4, "f16")
    np.testing.assert_array_equal(gpu_util.conv2d_fwd(inp, wei, (1, 1), (100, 100), (0, 0)),
                                  fast.conv2d_fwd_f16(inp, wei, (1, 1), (100, 100), (0, 0)))


def test_int8_epilogues():
    import gpu_util
    inp, wei = _ints((2, 30, 30, 3), 5, "i8"), _ints((40, 3, 3, 3), 6, "i8")
    for op, epi in ((ck.RequantReluRequant(0.05, 0.7, rounded=True), (lit.EPI_REQUANT_RND, 0.05, 0.7)),
                    (ck.RequantReluRequant(0.05, 0.7), (lit.EPI_REQUANT_CK, 0.05, 0.7))):
        out = gpu_util.conv2d_fwd(inp, wei, (2, 2), (1, 1), (1, 1), out_op=op)
        np.testing.assert_array_equal(out, fast.conv2d_fwd_i8(inp, wei, (2, 2), (1, 1), (1, 1), epi=epi[0], scale_gemm=epi[1],
                                                              scale_relu=epi[2]))


@pytest.mark.parametrize("K", [5, 16, 24, 64, 90])
@pytest.mark.parametrize("residual", [False, True])
def test_bias_relu_and_residual(K, residual):
    import torch
    import gpu_util
    N, C, H, W = 2, 3, 19, 23
    inp, wei = _ints((N, H, W, C), 7, "f16"), _ints((K, 3, 3, C), 8, "f16")
    bias, resi = _ints((K,), 9, "f16"), _ints((N, H, W, K), 10, "f16")
    di, dw, db, dr = (gpu_util.dev(x) for x in (inp, wei, bias, resi))
    do = torch.full((N, H, W, K), float("nan"), dtype=torch.float16, device="cuda")
    op = ck.DeviceConv2dFwdBiasActivationF16()
    geom = (N, K, C, [H, W], [3, 3], [H, W], [1, 1], [1, 1], [1, 1], [1, 1], None, None)
    arg = op.MakeArgumentPointer(di, dw, do, db, dr, *geom, ck.AddReluAdd()) if residual else \
        op.MakeArgumentPointer(di, dw, do, db, *geom, ck.AddRelu())
    assert op.IsSupportedArgument(arg)
    op.MakeInvokerPointer().Run(arg, ck.StreamConfig(gpu_util.stream()))
    torch.cuda.synchronize()
    acc = fast.conv2d_fwd_f16(inp, wei, (1, 1), (1, 1), (1, 1)).astype(np.float32)  # (integers below 2048: exact)
    want = np.maximum(acc + bias.astype(np.float32), 0) + (resi.astype(np.float32) if residual else 0)
    np.testing.assert_array_equal(do.cpu().numpy(), want.astype(np.float16))


@pytest.mark.parametrize("f", [3, 5])
def test_an_infinite_pixel_stays_in_its_windows(f):
    import gpu_util
    inp, wei = np.abs(_ints((1, 21, 25, 3), 11, "f16")), np.abs(_ints((16, f, f, 3), 12, "f16")) + np.float16(1)
    clean = gpu_util.conv2d_fwd(inp, wei, (1, 1), (1, 1), (f // 2, f // 2))
    inp[0, 10, 12, 1] = np.inf
    out = gpu_util.conv2d_fwd(inp, wei, (1, 1), (1, 1), (f // 2, f // 2))
    hit = np.zeros(out.shape, bool)
    hit[0, 10 - f // 2:11 + f // 2, 12 - f // 2:13 + f // 2] = True
    assert np.all(np.isposinf(out[hit]))
    np.testing.assert_array_equal(out[~hit], clean[~hit])


@pytest.mark.parametrize("dtype", ["i8", "f16"])
@pytest.mark.parametrize("layer", [(8, 90, 50, 49, 5, 3, (1, 1), (1, 1), (1, 1)), (8, 257, 60, 60, 3, 5, (1, 1), (2, 2), (1, 1)),
                                   (6, 600, 30, 31, 7, 7, (1, 1), (1, 1), (3, 3)), (2, 1000, 10, 10, 3, 3, (8, 8), (1, 1), (0, 0))])
def test_several_channel_blocks(dtype, layer):
    """Output channels of more than one block with enough pixels for the few-channel kernel; the last layer is one of too few
    pixels, which the gather takes."""
    import gpu_util
    from conv_few_plan import takes
    N, K, H, W, C, f, s, d, p = layer
    assert takes(dtype, N, H, W, C, K, f, f, s, d, p)[0] == (K != 1000)
    inp, wei = _ints((N, H, W, C), K, dtype), _ints((K, f, f, C), K + 1, dtype)
    out = gpu_util.conv2d_fwd(inp, wei, s, d, p)
    np.testing.assert_array_equal(out, (fast.conv2d_fwd_i8 if dtype == "i8" else fast.conv2d_fwd_f16)(inp, wei, s, d, p))
