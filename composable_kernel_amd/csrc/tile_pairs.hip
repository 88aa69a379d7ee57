// Two row (column) tiles of the four-stage 64 x 64 instance as one 128 x 64 (64 x 128) workgroup of eight waves: a translation unit of its own so that its
// kernels compile beside the others.
#include "tile_launch.hpp"

namespace ckx {
namespace {

template <int DT, int IM2COL, bool FUSED>
constexpr tile_launch_fn pairs = &launch_tile<DT, 128, 64, 8, 1, 128, 3, IM2COL, false, false, FUSED>;

} // namespace

bool short_tail(GemmArgs& g)
{
    // Where the tiles are no whole number of rounds of the CUs, as many of them as the whole rounds hold keep 256 rows, and the columns (or
    // rows) behind them are cut into tiles of the fewest rows, 128 to 224 by 32, that still fit one round: 4096 x 11008, 688 tiles in three
    // rounds, as 512 tiles of 256 rows and 242 of 192. Any saving pays: 13 random problems 1.02 to 1.17 of the speed, 1.09 on average. us: int8
    // 4096 x 11008 x 4096 152.6 -> 147.7, 2687 x 3214 x 2384 35.5 -> 30.3, 4910 x 1681 x 3072 34.7 -> 30.0, 3447 x 10022 x 3600 147 -> 135. fp16
    // and bf16 stay on the four-wave body, which is ahead by more than that (28 problems: 0.82 to 1.10, 0.95 on average), and strided fp16
    // convolutions on whole tiles: what a short tile saves them is products, and they wait for loads (648 tiles, 2.5 rounds: 153.8 and 153.1).
    const long grid = num_cus() - num_cus() % 8, tm = g.tiles_m, tn = g.tiles_n, rounds = tm * tn / grid;
    if(tm * tn == rounds * grid || g.ksplit != 1 || g.batch > 1)
        return false;
    const long columns = rounds * grid / tm, rows = rounds * grid / tn; // column tiles and row tiles that the whole rounds hold
    for(int h = 64; h < 128; h += 16)
    {
        const long in_columns = (g.M + 2 * h - 1) / (2 * h), in_rows = (g.M - rows * 256 + 2 * h - 1) / (2 * h);
        if(rows * tn + in_rows * tn <= (rounds + 1) * grid)
        {
            g.tail_m = (int)in_rows, g.tail_n = (int)tn, g.tail_row0 = (int)rows * 256;
            g.tiles_m = (int)rows;
        }
        else if(columns * tm + in_columns * (tn - columns) <= (rounds + 1) * grid)
        {
            g.tail_m = (int)in_columns, g.tail_n = (int)(tn - columns), g.tail_col0 = (int)columns;
            g.tiles_n = (int)columns;
        }
        else
            continue;
        g.tail_h = h;
        return true;
    }
    return false;
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
