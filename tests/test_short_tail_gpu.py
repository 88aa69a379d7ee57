"""GPU parity of the short tiles in the last round of int8 GEMMs on 256 x 256 tiles (csrc/tile_pairs.hip, short_tail): less than a round of tiles,
tails below and beside whole tiles, every tail height, M and N that end inside a tile and a vector, all plain epilogues. Bit for bit."""
import numpy as np
import pytest

import composable_kernel_amd as ck
import gpu_util
from oracle import fast, lit

pytestmark = pytest.mark.gpu

# M, N, K; what the rule makes of them on 256 CUs is worked out in _tail() below
SHAPES = [(1300, 7600, 160), (1296, 7632, 992), (5000, 5103, 144), (4096, 11008, 128), (2687, 3214, 304), (3447, 10021, 400), (257, 65800, 272),
          (8200, 2060, 1040), (6144, 4096, 256), (300, 33000, 144), (3500, 4000, 208)]


def _tail(M, N, grid=256):
    """The rule restated: (whole row tiles, whole column tiles, rows of a short tile, tails beside rather than below)."""
    tm, tn = -(-M // 256), -(-N // 256)
    rounds = tm * tn // grid
    columns, rows = rounds * grid // tm, rounds * grid // tn
    for h in (64, 80, 96, 112):
        if rows * tn + -(-(M - rows * 256) // (2 * h)) * tn <= (rounds + 1) * grid:
            return rows, tn, 2 * h, False
        if columns * tm + -(-M // (2 * h)) * (tn - columns) <= (rounds + 1) * grid:
            return tm, columns, 2 * h, True
    return None


def test_the_shapes_are_what_they_are_meant_to_be():
    kinds = [_tail(M, N) for M, N, _ in SHAPES]
    assert {k[2] for k in kinds if k} == {128, 160, 192, 224}
    assert any(k and k[3] for k in kinds) and any(k and not k[3] and k[0] for k in kinds) and any(k and k[0] == 0 for k in kinds)


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
