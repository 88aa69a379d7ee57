// Second pass of the split-K launches (gemm_tile.hpp): a translation unit of its own so that it compiles beside the others.
#include "tile_launch.hpp"

namespace ckx {
namespace {

// Second pass of a split-K launch: C = epilogue(sum over the K runs of the workspace slices).
// One thread per four consecutive columns of a row, slices added in run order (deterministic), all of them requested before the first is
// added: bound by the latency of that one round trip and, from a few MB of slices on, by their bytes. Sixteen columns per thread, slice after
// slice, left most CUs without a workgroup, and rows that are no multiple of sixteen took one load per element at their ends: whole launches, us,
// sixteen / eight / four columns: int8 78 x 1212 x 6144 20.9 / 13.1 / 10.3, 128 x 4096 x 11008 19.2 / 18.7 / 18.6, fp16 94 x 1086 x 8320 25.2 / 15.6 / 13.5,
// 662 x 578 x 7584 25.5 / 24.9 / 23.4; 45 random problems 1 / 0.82 / 0.73 of the time.
template <int DT>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const GemmArgs p)
{
    using acc_t   = typename std::conditional<DT == DT_I8, i32x4, f32x4>::type;
    constexpr int ES = DT == DT_I8 ? 1 : 2, COLS = 4, MOST = 8; // (at most eight K runs)
    const int groups_per_row = (p.N + COLS - 1) / COLS;
    const long gid = (long)blockIdx.x * 256 + threadIdx.x;
    if(gid >= (long)p.M * groups_per_row)
        return;
    const int m    = (int)(gid / groups_per_row);
    const int n0   = (int)(gid - (long)m * groups_per_row) * COLS;
    const int room = p.N - n0;
    acc_t v = acc_t{0, 0, 0, 0}, w[MOST];
#pragma unroll
    for(int sp = 0; sp < MOST; ++sp)
        if(sp < p.ksplit)
        {
            const uint8_t* wrow = reinterpret_cast<const uint8_t*>(p.ws) + (((size_t)sp * p.M + m) * p.N + n0) * 4;
            if(room >= COLS)
                w[sp] = load_vec<acc_t>(wrow);
            else
            {
#pragma unroll
                for(int e = 0; e < COLS; ++e)
                    w[sp][e] = e < room ? reinterpret_cast<const decltype(v[0] + 0)*>(wrow)[e] : 0;
            }
        }
#pragma unroll
    for(int sp = 0; sp < MOST; ++sp)
        if(sp < p.ksplit)
            v[0] += w[sp][0], v[1] += w[sp][1], v[2] += w[sp][2], v[3] += w[sp][3];
    uint8_t* const to = reinterpret_cast<uint8_t*>(p.c) + ((size_t)m * p.ldc + n0) * ES;
    if constexpr(DT == DT_I8)
    {
        float scale[COLS];
#pragma unroll
        for(int e = 0; e < COLS; ++e)
            scale[e] = epi_per_column_scale(p.epi) && e < room ? reinterpret_cast<const float*>(p.d0)[n0 + e] : 0.0f;
        int b[COLS];
        int8_results(GemmEpilogue{p.epi, p.scale_gemm, p.scale_relu}, b, [&](int e) { return v[e]; }, [&](int e) { return scale[e]; });
        const int words[1] = {pack4_low_bytes(b[0], b[1], b[2], b[3])};
        store_run<1>(to, words, room);
    }
    else
    {
        using T = typename std::conditional<DT == DT_BF16, __bf16, _Float16>::type;
        typedef T tx2 __attribute__((ext_vector_type(2)));
        float x[COLS];
#pragma unroll
        for(int e = 0; e < COLS; ++e)
            x[e] = v[e];
        if constexpr(DT == DT_F16)
        {
            if(p.epi != EPI_PASSTHROUGH)
            {
                const bool d1     = epi_has_d1(p.epi);
                const f16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
                const int bytes   = (room < COLS ? room : COLS) * 2;
                const f16x8 a = load_head16<f16x8>(reinterpret_cast<const _Float16*>(p.d0) + (size_t)m * p.ldd0 + n0, bytes);
                const f16x8 b = d1 ? load_head16<f16x8>(reinterpret_cast<const _Float16*>(p.d1) + (size_t)m * p.ldd1 + n0, bytes) : zero8;
#pragma unroll
                for(int e = 0; e < COLS; ++e)
                    x[e] = epi_f16_value(p.epi, x[e], (float)a[e], (float)b[e], p.scale_gemm, p.scale_relu);
            }
        }
        int words[COLS / 2];
#pragma unroll
        for(int e = 0; e < COLS; e += 2)
            words[e / 2] = __builtin_bit_cast(int, tx2{(T)x[e], (T)x[e + 1]});
        store_run<2>(to, words, room * 2);
    }
}

template <int DT>
hipError_t launch(const GemmArgs& a, hipStream_t s)
{
    const long groups = (long)a.M * ((a.N + 3) / 4);
    hipLaunchKernelGGL((splitk_reduce_kernel<DT>), dim3((unsigned)((groups + 255) / 256)), dim3(256), 0, s, a);
    return hipGetLastError();
}

} // namespace

hipError_t launch_splitk_reduce(int dt, const GemmArgs& a, hipStream_t s)
{
    return dt == DT_I8 ? launch<DT_I8>(a, s) : dt == DT_BF16 ? launch<DT_BF16>(a, s) : launch<DT_F16>(a, s);
}

} // namespace ckx
