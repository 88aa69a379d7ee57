"""The windowed conv kernel's host code (csrc/conv_window.hip): the box and chunks of a layer on one of its shapes, and a launch of that shape
where the library would choose the tile kernel."""
import ctypes as C

from composable_kernel_amd import capi

SHAPES = ((512, 64), (256, 128), (512, 32))  # output pixels and channels of a tile


class _MagicDiv(C.Structure):
    _fields_ = [(n, C.c_uint32) for n in ("mul", "shift", "d")]


def _ints(names):
    return [(n, C.c_int) for n in names.split()]


class ConvWindowArgs(C.Structure):
    _fields_ = [(n, C.c_void_p) for n in ("in_", "wei", "out", "d0", "d1")] + [("ldd1", C.c_int)] + \
        [(n, C.c_uint32) for n in ("in_bytes", "wei_bytes")] + \
        _ints("three_d N Di Hi Wi Do Ho Wo K pix_bytes units Y X taps dD dH dW pF pT pL TO TH TW box Wh pitch win_px") + \
        [(n, _MagicDiv) for n in "div_thw div_tw div_plane div_row div_chunk div_cu div_last div_yx div_x".split()] + \
        _ints("cu chunks total nk spp wbuf issue tiles_o tiles_h tiles_w tiles_n tiles epi") + \
        [("scale_gemm", C.c_float), ("scale_relu", C.c_float), ("nt_store", C.c_int)]


def layer(dtype, spatial, N, channels, K, filt, dil, pads, right_pads=None):
    """The layer's extents in the kernel's arguments (unit strides; two or three spatial dimensions)."""
    a, three = ConvWindowArgs(), len(spatial) == 3
    right_pads = right_pads or pads
    out = [spatial[i] + pads[i] + right_pads[i] - (filt[i] - 1) * dil[i] for i in range(len(spatial))]
    lift = (lambda v: list(v)) if three else (lambda v: [1] + list(v))
    (a.Di, a.Hi, a.Wi), (a.Do, a.Ho, a.Wo), (a.dD, a.dH, a.dW) = lift(spatial), lift(out), lift(dil)
    a.pF, a.pT, a.pL = lift(pads) if three else [0] + list(pads)
    z, a.Y, a.X = lift(filt)
    a.three_d, a.N, a.K, a.taps = int(three), N, K, z * a.Y * a.X
    a.pix_bytes = channels * (1 if dtype == "i8" else 2)
    a.units = a.pix_bytes // 16
    a.in_bytes = N * a.Di * a.Hi * a.Wi * a.pix_bytes
    a.wei_bytes = K * a.taps * a.pix_bytes
    a.ldd1 = K
    return a, out


def plan(dtype, shape, a):
    f = capi.lib()._ZN3ckx16plan_conv_windowEiiRNS_14ConvWindowArgsE
    f.restype, f.argtypes = C.c_double, [C.c_int, C.c_int, C.POINTER(ConvWindowArgs)]
    return f({"i8": 0, "f16": 1}[dtype], shape, C.byref(a))


def choose(dtype, a, tile_us):
    f = capi.lib()._ZN3ckx18choose_conv_windowEiRNS_14ConvWindowArgsEd
    f.restype, f.argtypes = C.c_int, [C.c_int, C.POINTER(ConvWindowArgs), C.c_double]
    return f({"i8": 0, "f16": 1}[dtype], C.byref(a), tile_us)


def run(dtype, shape, inp, wei, dil, pads, right_pads=None, epi=0, scales=(1.0, 1.0), d0=None, d1=None):
    """The layer on `shape`, numpy in and out (None: the shape does not take it)."""
    import numpy as np
    import torch

    import gpu_util
    N, spatial, channels, K, filt = inp.shape[0], inp.shape[1:-1], inp.shape[-1], wei.shape[0], wei.shape[1:-1]
    a, out = layer(dtype, spatial, N, channels, K, filt, dil, pads, right_pads)
    if plan(dtype, shape, a) < 0:
        return None
    di, dw = gpu_util.dev(inp), gpu_util.dev(wei)
    do = torch.full((N, *out, K), 77, dtype=torch.int8 if dtype == "i8" else torch.float16, device="cuda")
    dd = [None if x is None else gpu_util.dev(x) for x in (d0, d1)]
    a.in_, a.wei, a.out = di.data_ptr(), dw.data_ptr(), do.data_ptr()
    a.d0, a.d1 = [None if x is None else x.data_ptr() for x in dd]
    a.epi, a.scale_gemm, a.scale_relu = epi, *scales
    f = capi.lib()._ZN3ckx18launch_conv_windowEiiRKNS_14ConvWindowArgsEP12ihipStream_t
    f.restype, f.argtypes = C.c_int, [C.c_int, C.c_int, C.POINTER(ConvWindowArgs), C.c_void_p]
    assert f({"i8": 0, "f16": 1}[dtype], shape, C.byref(a), gpu_util.stream()) == 0
    torch.cuda.synchronize()
    r = do.cpu().numpy()
    assert r.shape == (N, *out, K) and np.isfinite(r.astype(np.float32)).any()
    return r
