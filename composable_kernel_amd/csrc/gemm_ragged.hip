// Launcher of the GEMM for operands that are no whole 16-byte vectors (a translation unit of its own so that its kernels
// compile beside the others).
#include "gemm_ragged.hpp"

namespace ckx {

template <int DT, int B, bool TA, bool TB>
static hipError_t launch_one(GemmArgs a, hipStream_t s)
{
    a.tiles_m = (a.M + B - 1) / B, a.tiles_n = (a.N + B - 1) / B;
    const long blocks = (long)a.tiles_m * a.tiles_n * (a.batch > 1 ? a.batch : 1);
    if(blocks >= (1l << 31))
        return hipErrorInvalidValue;
    hipLaunchKernelGGL((gemm_ragged_kernel<DT, B, B, TA, TB>), linear_grid(blocks), dim3(256), 0, s, a);
    return hipGetLastError();
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
    return tiles128 >= 256 && 10 * tiles128 <= 3 * tiles64 ? 128 : 64;
}

template <int DT, bool TA, bool TB>
static hipError_t launch_tile_size(const GemmArgs& a, hipStream_t s)
{
    return ragged_tile(a.M, a.N, a.batch) == 128 ? launch_one<DT, 128, TA, TB>(a, s) : launch_one<DT, 64, TA, TB>(a, s);
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
