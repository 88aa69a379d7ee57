"""GPU parity of the windowed conv kernel (csrc/conv_window.hpp) where it can go wrong, each tile shape by force: edges of boxes and images,
several images in a box, depth planes, odd 16-byte units of a pixel, K tiles that end inside a chunk or past GEMM-K, several chunks, several
tiles of a workgroup, output channels around the tiles' and lanes' runs, dilations, one-sided padding, epilogues, an infinite pixel. Small
integers: fp16 results are exact, so both data types are compared bit for bit."""
import numpy as np
import pytest

import composable_kernel_amd as ck
from conv_window_plan import SHAPES, run
from oracle import fast, lit

pytestmark = pytest.mark.gpu


def _ints(shape, seed, dtype):
    return np.random.default_rng(seed).integers(-2, 3, shape).astype(np.int8 if dtype == "i8" else np.float16)


def _want(inp, wei, dil, pads, right=None, **kw):
    return fast.convnd_fwd(inp, wei, (1,) * len(dil), dil, pads, right, **kw)


# spatial, N, C, K, filter, dilation, pads, right pads
LAYERS = [
    ((14, 14), 3, 64, 40, (3, 3), (1, 1), (1, 1), None),            # a whole image, and several, in a box
    ((7, 7), 21, 48, 72, (3, 3), (1, 1), (1, 1), None),             # int8: three units a pixel
    ((1, 37), 5, 48, 8, (3, 5), (1, 1), (1, 2), None),              # one row, K tiles past GEMM-K
    ((29, 61), 2, 80, 136, (3, 3), (1, 1), (0, 0), None),           # boxes cut by both edges, no padding
    ((30, 21), 1, 16, 33, (5, 5), (1, 2), (2, 4), (2, 0)),          # int8: one unit a pixel; dilation, one-sided padding, 25 taps
    ((40, 40), 70, 64, 24, (3, 3), (1, 1), (1, 1), None),           # more tiles than CUs
    ((20, 18), 2, 432, 130, (3, 3), (1, 1), (1, 1), None),          # several chunks of one tile, output channels past 128
    ((64, 9), 1, 256, 64, (2, 5), (1, 1), (0, 2), (1, 2)),          # whole lines per chunk, an even filter
    ((8, 8, 8), 2, 64, 64, (3, 3, 3), (1, 1, 1), (1, 1, 1), None),
    ((5, 11, 13), 3, 48, 20, (3, 3, 3), (1, 1, 1), (1, 1, 1), None),
    ((6, 7, 19), 2, 80, 100, (2, 3, 2), (2, 1, 1), (1, 0, 1), (0, 2, 1)),
    ((33, 6, 6), 1, 144, 16, (3, 1, 3), (1, 1, 2), (2, 0, 2), None),
]


@pytest.mark.parametrize("dtype", ["i8", "f16"])
@pytest.mark.parametrize("shape", range(len(SHAPES)))
@pytest.mark.parametrize("at", range(len(LAYERS)))
def test_layers(dtype, shape, at):
    spatial, N, C, K, filt, dil, pads, right = LAYERS[at]
    inp, wei = _ints((N, *spatial, C), at, dtype), _ints((K, *filt, C), 50 + at, dtype)
    out = run(dtype, shape, inp, wei, dil, pads, right)
    assert out is not None
    np.testing.assert_array_equal(out, _want(inp, wei, dil, pads, right))


@pytest.mark.parametrize("shape", range(len(SHAPES)))
def test_int8_epilogues(shape):
    inp, wei = _ints((2, 25, 25, 96), 5, "i8"), _ints((70, 3, 3, 96), 6, "i8")
    for epi, code in ((1, lit.EPI_REQUANT_CK), (2, lit.EPI_REQUANT_RND)):
        out = run("i8", shape, inp, wei, (1, 1), (1, 1), epi=epi, scales=(0.37, 0.7))
        np.testing.assert_array_equal(out, _want(inp, wei, (1, 1), (1, 1), epi=code, scale_gemm=0.37, scale_relu=0.7))
    scales = np.random.default_rng(7).uniform(0.01, 0.5, 70).astype(np.float32)
    for epi, relu in ((6, False), (7, True)):
        out = run("i8", shape, inp, wei, (1, 1), (1, 1), epi=epi, d0=scales)
        np.testing.assert_array_equal(out, fast.conv2d_fwd_i8_mul2_clamp(inp, wei, scales, relu, (1, 1), (1, 1), (1, 1)))


@pytest.mark.parametrize("shape", range(len(SHAPES)))
@pytest.mark.parametrize("K", [8, 41, 130])
@pytest.mark.parametrize("residual", [False, True])
def test_bias_relu_and_residual(shape, K, residual):
    inp, wei = _ints((3, 19, 23, 32), 7, "f16"), _ints((K, 3, 3, 32), 8, "f16")
    bias, resi = _ints((K,), 9, "f16"), _ints((3, 19, 23, K), 10, "f16")
    out = run("f16", shape, inp, wei, (1, 1), (1, 1), epi=4 if residual else 3, d0=bias, d1=resi if residual else None)
    acc  = _want(inp, wei, (1, 1), (1, 1)).astype(np.float32)  # (integers below 2048: exact)
    want = np.maximum(acc + bias.astype(np.float32), 0) + (resi.astype(np.float32) if residual else 0)
    np.testing.assert_array_equal(out, want.astype(np.float16))


@pytest.mark.parametrize("shape", range(len(SHAPES)))
@pytest.mark.parametrize("C", [24, 40])
def test_an_infinite_pixel_stays_in_its_windows(shape, C):
    """Units past GEMM-K (27 and 45 units here) and the borders multiply zeros, and not an infinite pixel."""
    inp, wei = np.abs(_ints((1, 21, 25, C), 11, "f16")), np.abs(_ints((16, 3, 3, C), 12, "f16")) + np.float16(1)
    clean = run("f16", shape, inp, wei, (1, 1), (1, 1))
    for at in ((0, 0), (10, 12), (20, 24)):
        x = inp.copy()
        x[0, at[0], at[1], C - 1] = x[0, at[0], at[1], 0] = np.inf
        out = run("f16", shape, x, wei, (1, 1), (1, 1))
        hit = np.zeros(out.shape, bool)
        hit[0, max(0, at[0] - 1):at[0] + 2, max(0, at[1] - 1):at[1] + 2] = True
        assert np.all(np.isposinf(out[hit]))
        np.testing.assert_array_equal(out[~hit], clean[~hit])


# data type, form, spatial, N, C, K, filter, dilation, pads, right pads: layers that the library's rule runs on the windowed kernel
AUTO = [
    ("i8", "requant", (57, 57), 32, 176, 24, (3, 3), (1, 1), (1, 1), (1, 1)),
    ("i8", "columns", (41, 41), 64, 304, 24, (3, 3), (1, 1), (1, 1), (1, 1)),
    ("i8", "plain", (96, 96), 240, 176, 32, (3, 3), (1, 1), (1, 1), (1, 1)),     # 68 MB: stored past the L2
    ("i8", "requant", (34, 33, 35), 4, 112, 32, (3, 3, 3), (1, 1, 1), (1, 1, 1), (1, 1, 1)),
    ("f16", "plain", (93, 93), 26, 48, 32, (5, 5), (1, 1), (2, 2), (2, 2)),
    ("f16", "plain", (61, 50), 24, 208, 32, (3, 5), (1, 2), (2, 1), (0, 5)),
    ("f16", "bias", (33, 33), 64, 104, 24, (3, 3), (1, 1), (1, 1), (1, 1)),
    ("f16", "residual", (57, 57), 48, 88, 24, (3, 3), (1, 1), (1, 1), (1, 1)),
    ("f16", "plain", (34, 33, 35), 4, 112, 32, (3, 3, 3), (1, 1, 1), (1, 1, 1), (1, 1, 1)),
]


@pytest.mark.parametrize("at", range(len(AUTO)))
def test_the_automatic_choice_agrees_with_the_tile_kernel(at):
    """The operators with the automatic choice, on layers where it is the windowed kernel, against a tile instance by name."""
    import ctypes as C

    import torch

    import gpu_util
    from composable_kernel_amd import capi
    dtype, form, spatial, N, channels, K, filt, dil, pads, right = AUTO[at]
    nd, family = len(spatial), capi.OP_CONV2D_FWD_I8 if dtype == "i8" else capi.OP_CONV2D_FWD_F16
    out_len = [spatial[i] + pads[i] + right[i] - (filt[i] - 1) * dil[i] for i in range(nd)]
    geom = (N, K, channels, list(spatial), list(filt), out_len, [1] * nd, list(dil), list(pads), list(right))
    if nd == 3:
        chosen = capi.lib()._ZN3ckx18auto_conv3d_windowEiPK15ckx_convnd_desc
        chosen.restype, chosen.argtypes = C.c_int, [C.c_int, C.POINTER(capi.ConvNdDesc)]
        assert chosen(family, C.byref(capi.ConvNdDesc.make(*geom))) >= 0
    else:
        epi  = {"plain": capi.EPI_PASSTHROUGH, "requant": capi.EPI_REQUANT_RND, "columns": capi.EPI_RELU_MUL2_CLAMP, "bias": capi.EPI_ADD_RELU,
                "residual": capi.EPI_ADD_RELU_ADD}[form]
        desc = capi.Conv2dDesc(N, K, channels, *spatial, *filt, *out_len, 1, 1, *dil, *pads, *right)
        assert capi.conv2d_fwd_plan(family, desc, epi) == (capi.INSTANCE_AUTO, 1)
    g    = torch.Generator(device="cuda").manual_seed(at)
    td   = torch.int8 if dtype == "i8" else torch.float16
    ints = lambda *s: torch.randint(-2, 3, s, generator=g, device="cuda", dtype=torch.int8).to(td)
    x, w, bias, resi = ints(N, *spatial, channels), ints(K, *filt, channels), ints(K), ints(N, *out_len, K)
    scales = torch.rand(K, generator=g, device="cuda") * 0.2 + 0.01

    def result(instance):
        y = torch.full((N, *out_len, K), 77, dtype=td, device="cuda")
        if form == "columns":
            op  = ck.DeviceConv2dFwdMultipleDInt8(instance)
            arg = op.MakeArgumentPointer(x, w, y, scales, *geom, None, None, ck.ActivationMul2Clamp(ck.Relu()))
        elif form in ("bias", "residual"):
            op  = ck.DeviceConv2dFwdBiasActivationF16(instance)
            arg = op.MakeArgumentPointer(x, w, y, bias, resi, *geom, None, None, ck.AddReluAdd()) if form == "residual" else \
                op.MakeArgumentPointer(x, w, y, bias, *geom, None, None, ck.AddRelu())
        else:
            op  = (ck.DeviceConvNdFwdInt8 if dtype == "i8" else ck.DeviceConvNdFwdF16)(nd, instance)
            arg = op.MakeArgumentPointer(x, w, y, *geom, None, None, ck.RequantReluRequant(0.05, 0.7, rounded=True) if form == "requant" else None)
        assert op.IsSupportedArgument(arg), capi.last_error()
        op.MakeInvokerPointer().Run(arg, ck.StreamConfig(gpu_util.stream()))
        torch.cuda.synchronize()
        return y
    got = result(capi.INSTANCE_AUTO)
    assert torch.equal(got, result(7)) and int((got != 0).sum()) > got.numel() // 8
