// Operands that are no whole 16-byte vectors, copied to rows that are (gemm_pack.hpp): a translation unit of its own so that it compiles
// beside the others.
#include "gemm_pack.hpp"
#include "gemm_ragged.hpp"

namespace ckx {
namespace {

struct PackArgs
{
    const uint8_t* src[2]; // A, B
    uint8_t* dst[2];
    int rows[2], ld[2];    // rows of the copy (M, N); elements from one row (K-major: k row) of the operand to the next
    bool kmajor[2];
    uint32_t blocks0;      // workgroups of A
    int K;
    uint32_t pitch;        // bytes of a row of the copies
    MagicDiv chunks;       // 16-byte chunks of a row that hold elements
};

constexpr int kPackChunks = 4; // chunks of a thread, all loads in flight

// What bounds it: the bytes, read at any byte and written in whole lines, once. K-contiguous operands: thread t takes chunks t, t + 256 ... of
// the workgroup's 1024 consecutive ones. K-major operands: 64 columns x 128 bytes of K through LDS, whose rows are 4 bytes longer than the
// 64 columns so that the eight lanes of an output row read different banks.
// 2001 x 1025 + 1003 x 1025 in fp16 take a GEMM on aligned rows from 10.8 us to 14.5 ... 15.0, 3.4 of it the launch (packing_pays() has the sides of the choice).
template <int ES>
__global__ __launch_bounds__(256) void gemm_pack_kernel(const PackArgs p)
{
    using elem_t         = typename std::conditional<ES == 1, uint8_t, uint16_t>::type;
    constexpr int EPC    = 16 / ES;
    const bool second    = blockIdx.x >= p.blocks0;
    const uint32_t block = second ? blockIdx.x - p.blocks0 : blockIdx.x;
    const uint8_t* src   = second ? p.src[1] : p.src[0];
    uint8_t* dst         = second ? p.dst[1] : p.dst[0];
    const int X = second ? p.rows[1] : p.rows[0], ld = second ? p.ld[1] : p.ld[0], tid = threadIdx.x;
    // 16 bytes from element `at` of a line of `extent` elements, zeros past its end (the load ends with the line)
    auto chunk = [&](const uint8_t* line, int at, int extent) {
        const int last = extent - EPC, from = at < last ? at : last;
        return shift_down_bytes(load_vec<i32x4>(line + (int64_t)from * ES), (at - from) * ES);
    };
    if(!(second ? p.kmajor[1] : p.kmajor[0]))
    {
        const uint32_t all = (uint32_t)X * p.chunks.d, first = block * (256u * kPackChunks) + (uint32_t)tid;
        i32x4 v[kPackChunks];
        uint32_t to[kPackChunks];
#pragma unroll
        for(int i = 0; i < kPackChunks; ++i)
        {
            const uint32_t idx = first + 256u * i < all ? first + 256u * i : all - 1;
            const uint32_t r = magic_div(idx, p.chunks), c = idx - r * p.chunks.d;
            to[i] = r * p.pitch + c * 16u;
            v[i]  = chunk(src + (int64_t)r * ld * ES, (int)c * EPC, p.K);
        }
#pragma unroll
        for(int i = 0; i < kPackChunks; ++i)
            if(first + 256u * i < all)
                *reinterpret_cast<i32x4*>(dst + to[i]) = v[i];
        return;
    }
    constexpr int KE = 128 / ES, RS = 64 * ES + 4, CPR = 64 * ES / 16, NCH = KE * CPR / 256;
    __shared__ __attribute__((aligned(16))) uint8_t tile[KE * RS];
    const uint32_t across = (uint32_t)(X + 63) / 64, tk = block / across;
    const int x0 = (int)(block - tk * across) * 64, k0 = (int)tk * KE;
    i32x4 v[NCH];
#pragma unroll
    for(int i = 0; i < NCH; ++i)
    {
        const int idx = tid + 256 * i, r = idx / CPR, x = x0 + idx % CPR * EPC;
        const bool live = k0 + r < p.K && x < X;
        const i32x4 got = chunk(src + (int64_t)(live ? k0 + r : 0) * ld * ES, live ? x : 0, X);
        v[i] = live ? got : i32x4{0, 0, 0, 0};
    }
#pragma unroll
    for(int i = 0; i < NCH; ++i)
    {
        const int idx = tid + 256 * i;
        int* const at = reinterpret_cast<int*>(tile + idx / CPR * RS + idx % CPR * 16);
        at[0] = v[i][0], at[1] = v[i][1], at[2] = v[i][2], at[3] = v[i][3];
    }
    __syncthreads();
#pragma unroll
    for(int i = 0; i < 2; ++i)
    {
        const int x = tid / 8 + 32 * i, c = tid % 8;
        elem_t e[EPC];
#pragma unroll
        for(int j = 0; j < EPC; ++j)
            e[j] = *reinterpret_cast<const elem_t*>(tile + (c * EPC + j) * RS + x * ES);
        if(x0 + x < X && (uint32_t)(k0 / EPC + c) < p.chunks.d)
        {
            i32x4 out;
            __builtin_memcpy(&out, e, 16);
            *reinterpret_cast<i32x4*>(dst + (uint32_t)(x0 + x) * p.pitch + (uint32_t)(k0 * ES + c * 16)) = out;
        }
    }
}

} // namespace

hipError_t launch_gemm_pack(const GemmPack& g, hipStream_t s)
{
    PackArgs p;
    p.K = g.K, p.pitch = (uint32_t)g.pitch * g.es;
    p.chunks = make_magic((uint32_t)(((long)g.K * g.es + 15) / 16));
    uint32_t blocks[2];
    for(int i = 0; i < 2; ++i)
    {
        p.src[i] = reinterpret_cast<const uint8_t*>(i ? g.b : g.a), p.dst[i] = reinterpret_cast<uint8_t*>(i ? g.to_b : g.to_a);
        p.rows[i] = i ? g.N : g.M, p.ld[i] = i ? g.ldb : g.lda, p.kmajor[i] = i ? g.tb : g.ta;
        const long ke = 128 / g.es;
        blocks[i] = (uint32_t)(p.kmajor[i] ? (p.rows[i] + 63l) / 64 * ((g.K + ke - 1) / ke)
                                           : ((long)p.rows[i] * p.chunks.d + 256 * kPackChunks - 1) / (256 * kPackChunks));
    }
    p.blocks0  = blocks[0];
    auto* kern = g.es == 1 ? &gemm_pack_kernel<1> : &gemm_pack_kernel<2>;
    hipLaunchKernelGGL(kern, dim3(blocks[0] + blocks[1]), dim3(256), 0, s, p);
    return hipGetLastError();
}

} // namespace ckx
