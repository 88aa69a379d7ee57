"""GPU parity of the short tiles in the last round of int8 GEMMs on 256 x 256 tiles (csrc/tile_pairs.hip, short_tail): less than a round of tiles,
tails below and beside whole tiles, every tail height, shapes around the rule, M and N that end inside a tile and a vector, all plain epilogues. Bit for bit."""
import numpy as np
import pytest

import composable_kernel_amd as ck
import gpu_util
from oracle import fast, lit

pytestmark = pytest.mark.gpu

SHAPES = [(1300, 7600, 160), (1296, 7632, 992), (5000, 5103, 144), (4096, 11008, 128), (2687, 3214, 304), (3447, 10021, 400), (257, 65800, 272),
          (8200, 2060, 1040), (6144, 4096, 256), (300, 33000, 144), (3500, 4000, 208), (2675, 9622, 272), (3810, 6671, 320)]


def _tail(M, N, K):
    """The library's rule: rows of a short tile (0: whole tiles), below the whole tiles rather than beside them."""
    import ctypes as C

    from composable_kernel_amd import capi
    rule = capi.lib()._ZN3ckx15short_tail_rowsEiiiRb
    rule.restype, rule.argtypes = C.c_int, [C.c_int] * 3 + [C.POINTER(C.c_bool)]
    below = C.c_bool()
    return rule(M, N, K, C.byref(below)), below.value


def test_the_shapes_are_what_they_are_meant_to_be():
    """Every height, below whole tiles and beside them, and less than a round of tiles; whole tiles where a tail does not pay."""
    tails = {s: _tail(*s) for s in SHAPES}
    assert {h for h, _ in tails.values()} == {0, 128, 160, 192}
    assert any(h and not below for h, below in tails.values()) and any(h and below and -(-M // 256) * -(-N // 256) > 256 for (M, N, _), (h, below) in tails.items())
    assert any(h and -(-M // 256) * -(-N // 256) < 256 for (M, N, _), (h, _) in tails.items())


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("epi", ["none", "ck", "rounded"])
def test_int8_bit_exact(shape, epi):
    M, N, K = shape
    rng = np.random.default_rng(M)
    a, b = rng.integers(-3, 4, (M, K)).astype(np.int8), rng.integers(-3, 4, (N, K)).astype(np.int8)
    op   = {"none": ck.PassThrough(), "ck": ck.RequantReluRequant(0.13, 0.7), "rounded": ck.RequantReluRequant(0.13, 0.7, rounded=True)}[epi]
    code = {"none": lit.EPI_PASSTHROUGH, "ck": lit.EPI_REQUANT_CK, "rounded": lit.EPI_REQUANT_RND}[epi]
    out  = gpu_util.gemm_i8(a, b, op, instance=0, ldc=N + 16 if epi == "ck" else None)
    np.testing.assert_array_equal(out, fast.gemm_i8(a, b.T, code, 0.13, 0.7))
