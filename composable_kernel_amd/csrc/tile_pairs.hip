// Two row (column) tiles of the four-stage 64 x 64 instance as one 128 x 64 (64 x 128) workgroup of eight waves: a translation unit of its own so that its
// kernels compile beside the others.
#include "tile_launch.hpp"

namespace ckx {
namespace {

template <int DT, int IM2COL, bool FUSED>
constexpr tile_launch_fn pairs = &launch_tile<DT, 128, 64, 8, 1, 128, 3, IM2COL, false, false, FUSED>;

} // namespace

int short_tail_rows(int M, int N, int K, bool& below)
{
    // Where the tiles are no whole number of rounds of the CUs, as many of them as the whole rounds hold keep 256 rows, and the columns (or rows)
    // behind them are cut into tiles of the fewest rows, 128 to 192 by 32, that still fit one round. The kernel's branches cost its whole rounds 2
    // to 7 %, so the last one has to save enough: any height up to 160 rows while there are few whole rounds, 192 rows without one or with 24 K
    // tiles and more; 224 nowhere. 210 random problems by height and whole rounds, speed against whole tiles: 128 rows 1 1.04 to 1.15, 2 1.04
    // (0.97 to 1.09), 3 1.04 from nine K tiles on (0.98 to 1.04 below); 160 rows 0 1.08 to 1.17, 1 1.03 (0.98 to 1.07), 2 1.02 (0.97 to 1.06), 3
    // 1.01 (0.97 below eight K tiles); 192 rows 0 1.05, from 24 K tiles on 1 and 2 1.005 (0.99 to 1.03), 3 1.06, below 0.96 to 1.03; 224 rows 0.92
    // to 1.02. us: int8 2687 x 3214 x 2384 35.7 -> 30.6, 4910 x 1681 x 3072 34.8 -> 30.9, 3447 x 10022 x 3600 146.4 -> 136.0, 4096 x 11008 x 4096
    // (192 rows behind two rounds) 152.9 -> 148.1, but 4852 x 5968 x 544 28.0 / 30.4, 7430 x 3687 x 2176 58.9 / 61.5. fp16 and bf16 stay on the
    // four-wave body, which is ahead by more than that (28 problems: 0.82 to 1.10, 0.95 on average), and strided fp16 convolutions on whole tiles:
    // what a short tile saves them is products, and they wait for loads (648 tiles, 2.5 rounds: 153.8 and 153.1).
    const long grid = num_cus() - num_cus() % 8, tm = (M + 255l) / 256, tn = (N + 255l) / 256, rounds = tm * tn / grid;
    if(tm * tn == rounds * grid)
        return 0;
    const long columns = rounds * grid / tm, rows = rounds * grid / tn; // column tiles and row tiles that the whole rounds hold
    const long k_tiles = (K + 127l) / 128;
    for(int h = 128; h <= 192; h += 32)
    {
        below = rows * tn + (M - rows * 256 + h - 1) / h * tn <= (rounds + 1) * grid;
        if(below || columns * tm + (M + h - 1l) / h * (tn - columns) <= (rounds + 1) * grid)
            return (h < 192 ? rounds < 3 || k_tiles >= 8 : rounds == 0 || k_tiles >= 24) ? h : 0;
    }
    return 0;
}

bool short_tail(GemmArgs& g)
{
    bool below  = false;
    const int h = g.ksplit != 1 || g.batch > 1 ? 0 : short_tail_rows(g.M, g.N, g.K, below);
    if(h == 0)
        return false;
    const int grid = num_cus() - num_cus() % 8, whole = g.tiles_m * g.tiles_n / grid * grid;
    g.tail_h       = h / 2;
    if(below)
    {
        const int rows = whole / g.tiles_n;
        g.tail_m = (g.M - rows * 256 + h - 1) / h, g.tail_n = g.tiles_n, g.tail_row0 = rows * 256;
        g.tiles_m = rows;
    }
    else
    {
        const int columns = whole / g.tiles_m;
        g.tail_m = (g.M + h - 1) / h, g.tail_n = g.tiles_n - columns, g.tail_col0 = columns;
        g.tiles_n = columns;
    }
    return true;
}

tile_launch_fn short_tail_tile() { return &launch_tile<DT_I8, 256, 256, 2, 4, 128, 2, 0, false, false, false, false, true>; }

bool row_pairs_pay(long M, long N, long runs)
{
    // What bounds two co-resident 64 x 64 workgroups is the operand bytes that their CU loads (65 to 82 bytes per ns), and both load the same
    // rows of B where they are above one another: a pair loads 192 rows per K tile where they load 256. So the line is
    // where the busiest CU loads fewer: no gain with one workgroup per CU, with a single row tile, or with an odd number of row tiles that makes
    // a second round. Random problems on this side: 9 GEMMs 0.80 to 0.97 of the time, 0.88 on average, 11 convolutions 0.83 to 0.93 (0.96 of it their
    // branch-free range checks), 12 GEMMs with K-major operands 0.79 to 1.02, 0.90 on average; on the other side single tiles as before, and pairs
    // 1.00 to 1.25 of their time. us: int8 67 x 10992 x 9024 36.4 -> 24.2, 128 x 4096 x 11008 20.9 -> 19.5, 32 x 14 x 14, C = K = 256 12.2 -> 11.0, fp16
    // 83 x 9560 x 4928 30.1 -> 25.7, 512 x 2736 x 8160 with a K-major B 71.3 -> 49.7. Eight waves of 16 rows as in the 64 x 64 kernel (four of 32
    // take 1.2 to 1.5 times as long), three LDS stages (two workgroups per CU; four stages, and one: 2 % behind).
    const long cus = num_cus(), cols = (N + 63) / 64 * runs, one = (M + 63) / 64 * cols, pair = (M + 127) / 128 * cols;
    return (pair + cus - 1) / cus * (128 + 64) < (one + cus - 1) / cus * (64 + 64);
}

bool column_pairs_pay(long M, long N, long ksplit, long batch)
{
    // Where row pairs do not pay -- a single row tile, an odd number of them -- two column tiles share their rows of A in the same way. 23
    // random GEMMs on this side 0.81 to 0.99 of the time, 0.89 on average: int8 277 x 6261 x 4928 22.6 -> 18.1 us, 146 x 10644 x 8384 35.8 -> 29.1, fp16
    // 26 x 2321 x 8736 in K runs 21.3 -> 19.2. K runs of several row tiles are level, 0.96 to 1.02 (157 x 1521 x 5696 19.1 -> 19.5), and stay.
    if(ksplit > 1 && M > 64)
        return false;
    const long runs = ksplit * batch;
    const long cus = num_cus(), rows = (M + 63) / 64 * runs, one = (N + 63) / 64 * rows, pair = (N + 127) / 128 * rows;
    return (pair + cus - 1) / cus * (64 + 128) < (one + cus - 1) / cus * (64 + 64);
}

tile_launch_fn column_pairs_tile(int dt)
{
    return dt == DT_I8     ? &launch_tile<DT_I8, 64, 128, 4, 2, 128, 3, 0>
           : dt == DT_BF16 ? &launch_tile<DT_BF16, 64, 128, 4, 2, 128, 3, 0>
                           : &launch_tile<DT_F16, 64, 128, 4, 2, 128, 3, 0>;
}

tile_launch_fn row_pairs_tile(int dt, bool im2col, bool fused)
{
    if(dt == DT_BF16)
        return im2col || fused ? nullptr : pairs<DT_BF16, 0, false>;
    if(dt == DT_I8)
        return im2col ? (fused ? pairs<DT_I8, 1, true> : pairs<DT_I8, 1, false>) : fused ? pairs<DT_I8, 0, true> : pairs<DT_I8, 0, false>;
    return im2col ? (fused ? pairs<DT_F16, 1, true> : pairs<DT_F16, 1, false>) : fused ? pairs<DT_F16, 0, true> : pairs<DT_F16, 0, false>;
}

tile_launch_fn row_pairs_conv3d_tile(int dt) { return dt == DT_I8 ? pairs<DT_I8, 2, false> : pairs<DT_F16, 2, false>; }

} // namespace ckx
