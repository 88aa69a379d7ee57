// Conv2d forward for inputs of few channels -- the first layers of image networks: RGB, RGB + depth, grey -- on gfx950, NHWC /
// KYXC / NHWK, any filter, stride, dilation, padding and number of output channels. Takes the place of the reference's OddC
// conv instances (convolution_forward_specialization.hpp:13-19, device_conv2d_fwd_xdl_nhwc_kyxc_nhwk.hpp:224-301), whose
// loads are one element each because no 16-byte vector of such an input is aligned to a filter tap.
//
//   * A workgroup (four waves) computes a patch of R x TW output pixels of one image. The input pixels under it are copied into
//     LDS once, each padded to CP = 4 or 8 channels and the borders written out as zeros, so that every tap of every
//     window is one aligned LDS read of CP channels. (As an implicit GEMM each pixel is gathered Y * X times.)
//   * GEMM-K runs over (tap, channel of CP): a lane's 16 bytes of an MFMA k-step are 16 / PX whole taps, read at the
//     window's base plus the tap's offset out of a table in LDS. Taps past Y * X read zeros (not a pixel times a zero weight:
//     an infinite pixel stays out of windows that do not hold it).
//   * The weights sit in LDS in fragment order for the life of the workgroup, which walks its patches with a grid stride; the
//     output channels of a block of 16 NT are permuted so that a lane ends with 4 NT consecutive ones of its pixel.
// Bound by the vector instructions around few MFMAs (window addresses, pixel copies, epilogue) and by the stores. Against the
// element-by-element gather that served these layers, fp16: C 3 -> K 32, 3 x 3 stride 2, 224 x 224, N = 64 (70 MB) 67 -> 20 us,
// with bias + ReLU 72 -> 22; C 4 -> K 64, 7 x 7 stride 2, N = 32 134 -> 38; C 6 -> K 96, 7 x 7, 200 x 200, N = 16 510 -> 89; int8
// C 3 -> K 96, 5 x 5, 128 x 128, N = 32 199 -> 40; C 5 -> K 48, 3 x 3, 64 x 64, N = 128 67 -> 21; one 28 x 28 image 5.6 -> 5.
#pragma once

#include "gemm_tile.hpp"

namespace ckx {

struct ConvFewArgs
{
    const void* in;
    const void* wei;
    void* out;
    const void* d0; // fp16: bias row [K]; int8 with a per-column scale: fp32 [K]
    const void* d1; // fp16: residual, rows of K at stride ldd1
    int ldd1;
    int N, Hi, Wi, C, Ho, Wo, K;
    int X, taps; // filter width, taps of the filter
    int sH, sW, dH, dW, pT, pL;
    int R, TW, PC, patch_pixels; // output patch, input columns and pixels under it
    MagicDiv div_pc, div_tw;
    int row_blocks, col_blocks, units;
    int nks, kblocks; // MFMA k-steps, blocks of 16 NT output channels per workgroup (blockIdx.y: the next such group)
    int epi;
    float scale_gemm, scale_relu;
    int nt_store;
};

template <int DT, int CP, int NT>
struct ConvFew
{
    static_assert((DT == DT_F16 || DT == DT_I8) && (CP == 4 || CP == 8), "fp16 or int8, pixels padded to 4 or 8 channels");
    static constexpr int ES = DT == DT_I8 ? 1 : 2, EPC = 16 / ES;
    static constexpr int PX  = CP * ES;  // bytes of a padded pixel
    static constexpr int TPL = 16 / PX;  // taps in a lane's 16 bytes of a k-step
    static constexpr int TPS = 4 * TPL;  // taps of a k-step
    static constexpr int MT  = NT == 4 ? 2 : 4; // 16-pixel tiles a wave works on together
    static constexpr int RUN = 4 * NT;   // consecutive output channels of a lane
    static constexpr int KB  = 16 * NT;  // output channels of a block
    using acc_t  = typename std::conditional<DT == DT_I8, i32x4, f32x4>::type;
    using elem_t = typename std::conditional<DT == DT_I8, int8_t, _Float16>::type;

    __host__ __device__ static constexpr int table_bytes(int nks) { return 16 + (nks * TPS * 4 + 15) / 16 * 16; }
    __host__ __device__ static constexpr int weight_bytes(int nks, int kblocks) { return nks * kblocks * NT * 1024; }

    // RUN halves of a row that has `room` bytes left
    __device__ static __forceinline__ void load_run(const _Float16* src, int room, float (&v)[RUN])
    {
        room = room < RUN * 2 ? room : RUN * 2;
#pragma unroll
        for(int e = 0; e < RUN; e += 8)
        {
            const f16x8 x = load_head16<f16x8>(src + e, room - 2 * e);
#pragma unroll
            for(int j = 0; j < 8 && e + j < RUN; ++j)
                v[e + j] = (float)x[j];
        }
    }

    // The input pixels under a patch into LDS, PX bytes each. NB: bytes of an input pixel, loaded as one piece of 8, 4, 2 and 1
    // bytes each; the loads of four pixels of a thread are in flight together.
    template <int NB>
    __device__ static __forceinline__ void copy_patch(const ConvFewArgs& p, const uint8_t* image, int hi0, int wi0, int tid, uint8_t* patch)
    {
        static_assert(NB < 16 && NB <= PX, "pieces of 8 bytes and less");
        for(int i0 = tid; i0 < p.patch_pixels; i0 += 4 * 256)
        {
            int v[4][4];
#pragma unroll
            for(int u = 0; u < 4; ++u)
            {
                const int idx = i0 + 256 * u;
                const int pr = (int)magic_div((uint32_t)idx, p.div_pc), pc = idx - pr * p.PC;
                const int hi = hi0 + pr, wi = wi0 + pc;
                const bool ok = idx < p.patch_pixels && (uint32_t)hi < (uint32_t)p.Hi && (uint32_t)wi < (uint32_t)p.Wi;
                const uint8_t* src = image + (ok ? (hi * p.Wi + wi) * NB : 0);
                constexpr int AT4 = NB & 8, AT2 = AT4 + (NB & 4), AT1 = AT2 + (NB & 2);
                int w[4] = {0, 0, 0, 0};
                if constexpr((NB & 8) != 0)
                {
                    const i32x2 x = reinterpret_cast<const AnyAlign<i32x2>*>(src)->v;
                    w[0] = x[0], w[1] = x[1];
                }
                if constexpr((NB & 4) != 0)
                    w[AT4 / 4] = reinterpret_cast<const AnyAlign<int>*>(src + AT4)->v;
                if constexpr((NB & 2) != 0)
                    w[AT2 / 4] = reinterpret_cast<const AnyAlign<uint16_t>*>(src + AT2)->v;
                if constexpr((NB & 1) != 0)
                    w[AT2 / 4] |= (int)src[AT1] << ((NB & 2) * 8);
#pragma unroll
                for(int e = 0; e < PX / 4; ++e)
                    v[u][e] = ok ? w[e] : 0;
            }
#pragma unroll
            for(int u = 0; u < 4; ++u)
                if(i0 + 256 * u < p.patch_pixels)
                    __builtin_memcpy(__builtin_assume_aligned(patch + (i0 + 256 * u) * PX, PX), v[u], PX);
        }
    }

    __device__ static __forceinline__ void run(const ConvFewArgs& p, uint8_t* smem)
    {
        const int tid = threadIdx.x, lane = tid & 63;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const uint32_t r = lane & 15, q = lane >> 4;
        // LDS: 16 zero bytes, the taps' offsets, the weights, the padded input pixels
        int* table          = reinterpret_cast<int*>(smem + 16);
        uint8_t* weights    = smem + table_bytes(p.nks);
        uint8_t* patch      = weights + weight_bytes(p.nks, p.kblocks);
        const int kb0       = (int)blockIdx.y * p.kblocks * KB;
        const uint8_t* in   = reinterpret_cast<const uint8_t*>(p.in);
        const elem_t* wei   = reinterpret_cast<const elem_t*>(p.wei);
        const int nb        = p.C * ES; // bytes of a pixel

        if(tid < 4)
            reinterpret_cast<int*>(smem)[tid] = 0;
        for(int t = tid; t < p.nks * TPS; t += 256)
        {
            const int y = t / p.X, x = t - y * p.X;
            table[t]    = t < p.taps ? (y * p.dH * p.PC + x * p.dW) * PX : -1;
        }
        // weights: 16-byte chunk (block, k-step, tile, lane); the chunk's taps are a run of the filter's memory
#pragma unroll 2
        for(int i = tid; i < p.nks * p.kblocks * NT * 64; i += 256)
        {
            const int l = i & 63, tile = (i >> 6) % NT, rest = (i >> 6) / NT, ks = rest % p.nks, b = rest / p.nks;
            const int ch   = kb0 + b * KB + RUN * ((l & 15) >> 2) + 4 * tile + (l & 3);
            const int tap0 = ks * TPS + (l >> 4) * TPL;
            elem_t e[EPC];
#pragma unroll
            for(int j = 0; j < EPC; ++j)
            {
                const int tap = tap0 + j / CP, c = j % CP;
                const bool ok = ch < p.K && tap < p.taps && c < p.C;
                e[j]          = ok ? wei[((int64_t)ch * p.taps + tap) * p.C + c] : (elem_t)0;
            }
            __builtin_memcpy(weights + (int64_t)i * 16, e, 16);
        }

        for(int unit = (int)blockIdx.x; unit < p.units; unit += (int)gridDim.x)
        {
            const int per_image = p.row_blocks * p.col_blocks;
            const int n = unit / per_image, in_image = unit - n * per_image;
            const int ho0 = in_image / p.col_blocks * p.R, wo0 = in_image % p.col_blocks * p.TW;
            const int hi0 = ho0 * p.sH - p.pT, wi0 = wo0 * p.sW - p.pL;
            __syncthreads(); // (every wave is done with the previous patch)
            // (a pixel's bytes fixed when compiled: as run-time branches the pieces were loaded and waited for one by one)
            const uint8_t* image = in + (int64_t)n * p.Hi * p.Wi * nb;
            constexpr int NB1 = (CP - 4) * ES; // the pixel has NB1 + 1, 2, 3 or 4 elements
            switch(p.C & 3)
            {
            case 1: copy_patch<NB1 + ES>(p, image, hi0, wi0, tid, patch); break;
            case 2: copy_patch<NB1 + 2 * ES>(p, image, hi0, wi0, tid, patch); break;
            case 3: copy_patch<NB1 + 3 * ES>(p, image, hi0, wi0, tid, patch); break;
            default:
                if constexpr(NB1 + 4 * ES < 16)
                    copy_patch<NB1 + 4 * ES>(p, image, hi0, wi0, tid, patch);
                break;
            }
            __syncthreads();
            // ---- MT tiles of 16 consecutive pixels of the patch at a time, dealt to the waves
            const int pixels = p.R * p.TW;
            for(int t0 = wave * MT; t0 * 16 < pixels; t0 += 4 * MT)
            {
                int base[MT];    // LDS byte offset of the pixel's window
                int64_t orow[MT]; // output pixel, -1: none
#pragma unroll
                for(int i = 0; i < MT; ++i)
                {
                    const int pos  = (t0 + i) * 16 + (int)r;
                    const int at   = pos < pixels ? pos : 0;
                    const int hl   = (int)magic_div((uint32_t)at, p.div_tw), wl = at - hl * p.TW;
                    base[i]        = (hl * p.sH * p.PC + wl * p.sW) * PX;
                    const bool live = pos < pixels && ho0 + hl < p.Ho && wo0 + wl < p.Wo;
                    orow[i] = live ? ((int64_t)n * p.Ho + ho0 + hl) * p.Wo + wo0 + wl : -1;
                }
                for(int b = 0; b < p.kblocks; ++b)
                {
                    const int ch0 = kb0 + b * KB;
                    if(ch0 >= p.K)
                        break;
                    // the lane owns channels ch .. ch + RUN - 1 of its pixel of every tile; their bias / scale
                    const int ch   = ch0 + RUN * (int)q;
                    const int room = (p.K - ch) * ES;
                    float dcol[RUN];
#pragma unroll
                    for(int e = 0; e < RUN; ++e)
                        dcol[e] = 0.0f;
                    if(p.epi >= EPI_ADD_RELU)
                    {
                        if constexpr(DT == DT_F16)
                            load_run(reinterpret_cast<const _Float16*>(p.d0) + ch, room, dcol);
                        else
                        {
#pragma unroll
                            for(int e = 0; e < RUN; ++e)
                                if(ch + e < p.K)
                                    dcol[e] = reinterpret_cast<const float*>(p.d0)[ch + e];
                        }
                    }
                    acc_t acc[MT][NT];
#pragma unroll
                    for(int i = 0; i < MT; ++i)
#pragma unroll
                        for(int t = 0; t < NT; ++t)
                            acc[i][t] = acc_t{0, 0, 0, 0};
                    const uint8_t* wblock = weights + (int64_t)b * p.nks * NT * 1024 + lane * 16;
                    for(int ks = 0; ks < p.nks; ++ks)
                    {
                        int off[TPL];
#pragma unroll
                        for(int j = 0; j < TPL; ++j)
                            off[j] = table[ks * TPS + (int)q * TPL + j];
                        i32x4 bf[NT], af[MT];
#pragma unroll
                        for(int t = 0; t < NT; ++t)
                            bf[t] = *reinterpret_cast<const i32x4*>(wblock + (ks * NT + t) * 1024);
#pragma unroll
                        for(int i = 0; i < MT; ++i)
                        {
                            const int pbase = (int)(patch - smem) + base[i];
#pragma unroll
                            for(int j = 0; j < TPL; ++j)
                            {
                                const uint8_t* src = smem + (off[j] < 0 ? 0 : pbase + off[j]);
                                int x[PX / 4];
                                __builtin_memcpy(x, __builtin_assume_aligned(src, PX), PX);
#pragma unroll
                                for(int e = 0; e < PX / 4; ++e)
                                    af[i][j * (PX / 4) + e] = x[e];
                            }
                        }
#pragma unroll
                        for(int i = 0; i < MT; ++i)
#pragma unroll
                            for(int t = 0; t < NT; ++t)
                            {
                                if constexpr(DT == DT_I8)
                                    acc[i][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(bf[t], af[i], acc[i][t], 0, 0, 0);
                                else
                                    acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, bf[t]),
                                                                                    __builtin_bit_cast(f16x8, af[i]), acc[i][t], 0, 0, 0);
                            }
                    }
                    if(room <= 0)
                        continue;
#pragma unroll
                    for(int i = 0; i < MT; ++i)
                    {
                        if(orow[i] < 0)
                            continue;
                        elem_t* dst = reinterpret_cast<elem_t*>(p.out) + orow[i] * p.K + ch;
                        int w[RUN * ES / 4];
                        if constexpr(DT == DT_I8)
                        {
                            int o[RUN];
                            int8_results(GemmEpilogue{p.epi, p.scale_gemm, p.scale_relu}, o,
                                         [&](int e) { return acc[i][e / 4][e % 4]; }, [&](int e) { return dcol[e]; });
#pragma unroll
                            for(int e = 0; e < RUN / 4; ++e)
                                w[e] = pack4_low_bytes(o[4 * e], o[4 * e + 1], o[4 * e + 2], o[4 * e + 3]);
                        }
                        else
                        {
                            float d1v[RUN];
#pragma unroll
                            for(int e = 0; e < RUN; ++e)
                                d1v[e] = 0.0f;
                            if(p.epi == EPI_ADD_RELU_ADD)
                                load_run(reinterpret_cast<const _Float16*>(p.d1) + orow[i] * p.ldd1 + ch, room, d1v);
#pragma unroll
                            for(int e = 0; e < RUN; e += 2)
                            {
                                float v[2] = {acc[i][e / 4][e % 4], acc[i][e / 4][e % 4 + 1]};
                                if(p.epi != EPI_PASSTHROUGH) // (bias + ReLU, with or without a residual)
                                {
                                    v[0] = epi_f16_value<false>(EPI_ADD_RELU_ADD, v[0], dcol[e], d1v[e]);
                                    v[1] = epi_f16_value<false>(EPI_ADD_RELU_ADD, v[1], dcol[e + 1], d1v[e + 1]);
                                }
                                w[e / 2] = __builtin_bit_cast(int, f16x2{(_Float16)v[0], (_Float16)v[1]});
                            }
                        }
                        store_run<ES>(reinterpret_cast<uint8_t*>(dst), w, room, p.nt_store != 0);
                    }
                }
            }
        }
    }
};

template <int DT, int CP, int NT>
__global__ __launch_bounds__(256, 4) void conv_few_kernel(const ConvFewArgs p)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t ckx_smem[];
    ConvFew<DT, CP, NT>::run(p, ckx_smem);
}

// (conv_few.hip) Fills the tiling of `a`, div_pc and div_tw apart, whose problem and epilogue are set: false if it is not one of few channels
// (a pixel of less than 16 bytes, at most 8 channels), the filter or its reach does not fit the LDS, or the gather is
// rated faster on it.
bool plan_conv_few(int dt, ConvFewArgs& a, int filter_h);
hipError_t launch_conv_few(int dt, const ConvFewArgs& a, hipStream_t s);

} // namespace ckx
