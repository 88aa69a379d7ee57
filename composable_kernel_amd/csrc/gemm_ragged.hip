// Launcher of the GEMM for operands that are no whole 16-byte vectors (a translation unit of its own so that its kernels
// compile beside the others).
#include "gemm_ragged.hpp"
#include "tile_launch.hpp"

namespace ckx {

// The threads of a grid dimension are counted in 32 bits, and a launch past them wraps around without an error.
constexpr long kMostBlocks = ((1l << 32) - 1) / 256;

template <int DT, int BM, int BN, bool TA, bool TB>
static hipError_t launch_one(GemmArgs a, hipStream_t s)
{
    constexpr long es = DT == DT_I8 ? 1 : 2;
    a.tiles_m = (a.M + BM - 1) / BM, a.tiles_n = (a.N + BN - 1) / BN;
    const long per_batch = (long)a.tiles_m * a.tiles_n, fit = kMostBlocks / per_batch;
    if(fit < 1)
        return hipErrorInvalidValue;
    // (more batches than fit a launch go out in launches of their own; an earlier 1 x 32769 x 1 in 65281 batches, 2^24 + 1 workgroups,
    // computed one of them. A second grid dimension instead, with a check of its last row in the kernel, cost up to 2 % everywhere)
    int left = a.batch > 1 ? a.batch : 1;
    while(left > 0)
    {
        const int n = left < fit ? left : (int)fit;
        a.batch     = n;
        hipLaunchKernelGGL((gemm_ragged_kernel<DT, BM, BN, TA, TB>), dim3((unsigned)(per_batch * n)), dim3(256), 0, s, a);
        const hipError_t e = hipGetLastError();
        if(e != hipSuccess)
            return e;
        a.a = reinterpret_cast<const uint8_t*>(a.a) + n * a.bsa * es;
        a.b = reinterpret_cast<const uint8_t*>(a.b) + n * a.bsb * es;
        a.c = reinterpret_cast<uint8_t*>(a.c) + n * a.bsc * es;
        left -= n;
    }
    return hipSuccess;
}

int ragged_tile(int M, int N, int batch)
{
    // One 128 x 128 tile per CU and more: half the operand bytes per product. 4001 x 4003 x 4095 fp16 197 us against 323 on
    // 64 x 64, int8 118 against 192; 1000 x 4001 x 513 (exactly 256 tiles) 15.5 against 16.4; 2049 x 2047 x 2047 K-major
    // (272) level at 55. Below, the smaller tile fills CUs that would idle: 2001 x 1003 x 1025 fp16 (128 tiles) 16.1 us
    // against 21.3, int8 1500 x 1501 x 1025 K-major B (144) 14.2 against 17.8, 122 x 1283 x 3001 17.4 against 43.7.
    // And only where its tiles cover at most a fifth more than the small ones do: batches of small problems reach any count of
    // tiles that are mostly padding. Batches at K = 1001 (fp16; 257): covering 9 % more (700 x 321) the large tile takes 0.94
    // (1.10) of the small one's time, 33 % more (150 x 500) 1.08 (1.31), 78 % more (129 x 131) 1.49 (1.70); 20000 x (3 x 5
    // x 7) 116 us against 45, 2000 x (33 x 35 x 37) 17.7 against 8.4.
    const long n        = batch > 1 ? batch : 1;
    const long tiles128 = (long)((M + 127) / 128) * ((N + 127) / 128) * n, tiles64 = (long)((M + 63) / 64) * ((N + 63) / 64) * n;
    // (... or where one batch of the small ones is more than a launch holds)
    return (tiles128 >= num_cus() && 10 * tiles128 <= 3 * tiles64) || tiles64 / n > kMostBlocks ? 128 : 64;
}

RaggedTile ragged_small_tile(int M, int N, int batch)
{
    // The tile with the fewest operand rows through the busiest CU, its tiles times (m + n); a smaller one for a sixteenth less. A
    // K tile takes 0.31 us of a CU for 64 + 64 rows, 0.24 for 64 + 32, 0.16 for 32 + 32, whether one workgroup or several ask for
    // them. Of 137 random problems below the 128 x 128 line 115 run on 32 x 32 tiles, in 0.50 to 1.02 of the time on 64 x 64 ones, 0.84 on
    // average, and four on 64 x 32, 0.92: 34 x 479 x 3569 20.8 -> 12.1 us, 1184 x 551 x 143 5.2 -> 4.6, 305 x 1011 x 2521 15.3 -> 12.0;
    // 2001 x 1003 x 1025 stays (15.6 against 19.9 on 64 x 32, 23.7 on 32 x 32; 15.4 on a 128 x 64 one, which gains 10 % at most
    // elsewhere and is not built).
    const long n     = batch > 1 ? batch : 1, cus = num_cus();
    const auto tiles = [&](RaggedTile t) { return (((long)M + t.m - 1) / t.m) * (((long)N + t.n - 1) / t.n) * n; };
    RaggedTile best  = {64, 64};
    long least       = (tiles(best) + cus - 1) / cus * 128;
    for(const RaggedTile t : {RaggedTile{64, 32}, RaggedTile{32, 32}})
    {
        const long rows = (tiles(t) + cus - 1) / cus * (t.m + t.n);
        if(16 * rows <= 15 * least && tiles(t) / n <= kMostBlocks)
            best = t, least = rows;
    }
    return best;
}

template <int DT, bool TA, bool TB>
static hipError_t launch_tile_size(const GemmArgs& a, hipStream_t s)
{
    if(ragged_tile(a.M, a.N, a.batch) == 128)
        return launch_one<DT, 128, 128, TA, TB>(a, s);
    const RaggedTile t = ragged_small_tile(a.M, a.N, a.batch);
    if(t.m == 32)
        return launch_one<DT, 32, 32, TA, TB>(a, s);
    return t.n == 32 ? launch_one<DT, 64, 32, TA, TB>(a, s) : launch_one<DT, 64, 64, TA, TB>(a, s);
}

template <int DT>
static hipError_t launch_layout(bool ta, bool tb, const GemmArgs& a, hipStream_t s)
{
    return ta ? (tb ? launch_tile_size<DT, true, true>(a, s) : launch_tile_size<DT, true, false>(a, s))
              : (tb ? launch_tile_size<DT, false, true>(a, s) : launch_tile_size<DT, false, false>(a, s));
}

hipError_t launch_ragged(int dt, bool ta, bool tb, GemmArgs a, hipStream_t s)
{
    if(a.batch > 65535)
        return hipErrorInvalidValue;
    return dt == DT_I8 ? launch_layout<DT_I8>(ta, tb, a, s) : dt == DT_BF16 ? launch_layout<DT_BF16>(ta, tb, a, s) : launch_layout<DT_F16>(ta, tb, a, s);
}

} // namespace ckx
