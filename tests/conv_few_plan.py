"""The tiling choice of the few-channel conv kernel (csrc/conv_few.hip), host code of the library: whether a layer runs on it."""
import ctypes as C

from composable_kernel_amd import capi

_INTS = "N Hi Wi C Ho Wo K X taps sH sW dH dW pT pL R TW PC patch_pixels"


class _MagicDiv(C.Structure):
    _fields_ = [(n, C.c_uint32) for n in ("mul", "shift", "d")]


class ConvFewArgs(C.Structure):
    _fields_ = [(n, C.c_void_p) for n in ("in_", "wei", "out", "d0", "d1")] + [("ldd1", C.c_int)] + \
        [(n, C.c_int) for n in _INTS.split()] + [("div_pc", _MagicDiv), ("div_tw", _MagicDiv)] + \
        [(n, C.c_int) for n in ("row_blocks", "col_blocks", "units", "nks", "kblocks", "epi")] + \
        [("scale_gemm", C.c_float), ("scale_relu", C.c_float), ("nt_store", C.c_int)]


def takes(dtype, N, H, W, channels, K, Y, X, strides=(1, 1), dilations=(1, 1), pads=(0, 0)):
    """Whether the kernel takes the layer (symmetric padding), and its plan."""
    a = ConvFewArgs()
    a.N, a.Hi, a.Wi, a.C, a.K, a.X = N, H, W, channels, K, X
    a.Ho = (H + 2 * pads[0] - ((Y - 1) * dilations[0] + 1)) // strides[0] + 1
    a.Wo = (W + 2 * pads[1] - ((X - 1) * dilations[1] + 1)) // strides[1] + 1
    (a.sH, a.sW), (a.dH, a.dW), (a.pT, a.pL) = strides, dilations, pads
    plan = capi.lib()._ZN3ckx13plan_conv_fewEiRNS_11ConvFewArgsEi
    plan.restype, plan.argtypes = C.c_bool, [C.c_int, C.POINTER(ConvFewArgs), C.c_int]
    return plan({"i8": 0, "f16": 1}[dtype], C.byref(a), Y), a
