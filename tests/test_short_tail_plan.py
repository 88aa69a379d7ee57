"""Where int8 GEMMs on 256 x 256 tiles cut their last round into short tiles (csrc/tile_pairs.hip, short_tail_rows), host logic: both sides of its
lines, each measured (us, whole tiles / short ones)."""
import ctypes as C

from composable_kernel_amd import capi


def _rows(M, N, K):
    rule = capi.lib()._ZN3ckx15short_tail_rowsEiiiRb
    rule.restype, rule.argtypes = C.c_int, [C.c_int] * 3 + [C.POINTER(C.c_bool)]
    return rule(M, N, K, C.byref(C.c_bool()))


def test_short_tiles_only_where_they_win():
    assert _rows(4852, 5968, 544) == 0      # 224 rows behind one round: 28.0 / 30.4
    assert _rows(1610, 7437, 1568) == 0     # 224 rows, less than a round: 27.2 / 27.8
    assert _rows(7430, 3687, 2176) == 0     # 192 rows behind one round: 58.9 / 61.5
    assert _rows(4100, 10272, 368) == 0     # 192 rows behind two, few K tiles: 31.5 / 32.5
    assert _rows(4096, 11008, 4096) == 192  # 192 rows behind two, 32 K tiles: 152.9 / 148.1
    assert _rows(8156, 6764, 640) == 0      # 128 rows behind three, few K tiles: 50.2 / 51.4
    assert _rows(8076, 7252, 688) == 0      # 160 rows behind three, few K tiles: 58.9 / 60.7
    assert _rows(2687, 3214, 2384) == 160   # less than a round: 35.7 / 30.6
    assert _rows(2551, 4400, 2080) == 192   # less than a round: 31.4 / 30.4
    assert _rows(6653, 2959, 2512) == 128   # behind one round: 71.6 / 63.7
    assert _rows(3447, 10022, 3600) == 128  # behind two: 146.4 / 136.0
    assert _rows(3972, 10622, 3792) == 160  # behind two: 169.3 / 159.4
    assert _rows(6298, 8870, 1968) == 128   # behind three: 124.2 / 119.8
    assert _rows(4096, 4096, 4096) == 0     # a whole number of rounds
