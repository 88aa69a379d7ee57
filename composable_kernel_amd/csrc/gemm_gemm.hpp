// Batched fused GEMM-GEMM for gfx950, fp16:  C[g] = half( half(A[g] * B0[g]) * B1[g] ).
// A [G,M,K] row-major, B0 stored [G,N,K] (column-major K x N), B1 [G,N,O] row-major,
// C [G,M,O] row-major (layout gmk_gnk_gno_gmo of upstream's DeviceBatchedGemmGemm; batch
// offsets as in kernel_batched_gemm_xdlops_v2r3, device_batched_gemm_xdl.hpp:79-88).
//
// One workgroup owns 64 or 128 rows of one batch and walks N in steps of 128 columns; the next
// step's B0 / B1 slices are prefetched into registers while the current one is multiplied.
// The slice of the intermediate never leaves registers:
//   gemm0 is issued as S^T = B0_frag x A_frag, so lane (l%16 = m, l/16 = q) holds S[m][n]
//   for 4 values of n per MFMA tile; the B0 rows fed to a PAIR of tiles are chosen so that
//   the pair gives the lane n = 32*pair + 8q .. +7, i.e. exactly the eight K-slots that the
//   same lane must supply as the second operand of gemm1 (C^T = B1T_frag x S_frag) after a
//   round-to-nearest-even conversion to fp16. B1 is transposed while it is staged into LDS
//   so that its fragment is one 16-byte read as well.
//
// SOFTMAX variant (upstream's DeviceBatchedGemmSoftmaxGemm, "attention") on 16 rows per wave, for launches whose shorter
// chain of steps wins: about one workgroup per CU and short N or wide heads, see rows_in_16s() (gemm_softmax_gemm.hpp has the kernel for all others):
//   C[g] = half( half(softmax_n(scale * A[g] * B0[g], masked)) * B1[g] )
// with the softmax along N in one pass over N (running row maximum and running sum): a step's
// scores become p = exp(s - running max), the output accumulators and the running sum are rescaled
// whenever the maximum grows, and the division by the sum happens once at the end. A row's 128
// scores of a step sit in four lanes (l%16 = row, l/16 = q), 32 each: the row maximum crosses those
// lanes with v_permlane16_swap / v_permlane32_swap, and so does the final sum. Columns past N and, with the
// upper-triangle mask, columns n > m count as -infinity; masked-out steps are skipped altogether.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <mutex>
#include <string>

#include "gemm_tile.hpp"
#include "tile_launch.hpp"

namespace ckx {

// Order of a masked launch (slab_order()): batches go out in groups, the slabs of a group heaviest first.
struct SlabOrder
{
    MagicDiv group, in_group, in_last; // by: workgroups of a group, batches of a group, batches of the last one
    int groups;
};

struct GemmGemmArgs
{
    const _Float16* a;
    const _Float16* b0;
    const _Float16* b1;
    _Float16* c;
    int M, N, K, O, batch;
    int sa, sb0, sb1, sc;
    int64_t bsa, bsb0, bsb1, bsc;
    int slabs; // ceil(M / rows per workgroup)
    float scale;   // softmax variant: scores are scale * (A * B0)
    int mask_upper; // softmax variant: scores with n > m are masked out
    SlabOrder order; // masked launches only
};

// maximum / sum over the four lanes l, l^16, l^32, l^48 (every one of them gets the result)
typedef short s16x4_t __attribute__((__vector_size__(4 * sizeof(short))));
typedef __attribute__((address_space(3))) s16x4_t lds_s16x4;

__device__ __forceinline__ float quad_rows_sum(float x)
{
    auto a = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, x), false, false);
    const uint32_t a0 = a[0], a1 = a[1];
    x      = __builtin_bit_cast(float, a0) + __builtin_bit_cast(float, a1);
    auto b = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, x), false, false);
    const uint32_t b0 = b[0], b1 = b[1];
    return __builtin_bit_cast(float, b0) + __builtin_bit_cast(float, b1);
}
// Maximum of scores. fmaxf, an IEEE-754-2008 maxNum, has every operand that the compiler cannot prove to be a quiet number (an
// MFMA result, a lane swap) canonicalised by a v_max_f32 x, x, x of its own; the 2019 maximumNumber has not, and two of
// them are one v_max3_f32. (A NaN score makes its row of the output NaN through the exponentials whatever the maximum is.)
__device__ __forceinline__ float score_max(float a, float b) { return __builtin_elementwise_maximumnum(a, b); }
// (of two operands only maximumNumber is canonicalised after all; maximum, which a NaN wins, is one v_maximum3_f32)
__device__ __forceinline__ float quad_rows_max(float x)
{
    auto a = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, x), false, false);
    const uint32_t a0 = a[0], a1 = a[1];
    x      = __builtin_elementwise_maximum(__builtin_bit_cast(float, a0), __builtin_bit_cast(float, a1));
    auto b = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, x), false, false);
    const uint32_t b0 = b[0], b1 = b[1];
    return __builtin_elementwise_maximum(__builtin_bit_cast(float, b0), __builtin_bit_cast(float, b1));
}

// (batch, slab of rows) of workgroup `bid`. Workgroups of one batch share B0[g] and B1[g]: they are kept on one XCD (ids are
// dealt round-robin over 8 XCDs) where the batch count allows, so that those panels are fetched into one L2 only.
// With the upper-triangle mask slab i has i + 1 times the work of slab 0, and the launch lasts until its last slab is
// through: the slabs go out heaviest first, over groups of batches at once, in the order that slab_order() lays out on the host
// (three divisions of the kernel's own took 0.15 us of every launch: 2 x 55 x 55 x 32 3.6 -> 3.8).
__device__ __forceinline__ void slab_of_block_masked(int bid, int slabs, const SlabOrder& o, int& g, int& slab)
{
    const uint32_t group = magic_div((uint32_t)bid, o.group), in = (uint32_t)bid - group * o.group.d;
    const bool last      = group == (uint32_t)o.groups - 1;
    const MagicDiv here  = {last ? o.in_last.mul : o.in_group.mul, last ? o.in_last.shift : o.in_group.shift, last ? o.in_last.d : o.in_group.d};
    const uint32_t up    = magic_div(in, here);
    slab                 = slabs - 1 - (int)up;
    g                    = (int)(group * o.in_group.d + in - up * here.d);
}

template <bool SOFTMAX>
__device__ __forceinline__ void slab_of_block(int bid, const GemmGemmArgs& p, int& g, int& slab)
{
    if(SOFTMAX && p.mask_upper)
        slab_of_block_masked(bid, p.slabs, p.order, g, slab);
    else if((p.batch & 7) == 0)
    {
        const int xcd = bid & 7, local = bid >> 3;
        g    = xcd + 8 * (local / p.slabs);
        slab = local - (local / p.slabs) * p.slabs;
    }
    else
    {
        g    = bid / p.slabs;
        slab = bid - g * p.slabs;
    }
}

// KS  k-steps of gemm0 (K padded to 32*KS), OG  64-column groups of the output (O padded to 64*OG),
// MT  16-row MFMA tiles per wave, NW waves: a workgroup owns 16*MT*NW rows of one batch.
template <int KS, int OG, int MT, int NW>
struct GemmGemmCfg
{
    static constexpr int NT   = 64 * NW;
    static constexpr int BM   = 16 * MT * NW;
    static constexpr int BNC  = 128; // columns of the intermediate per step
    static constexpr int KP   = KS * 32;
    static constexpr int OP   = OG * 64;
    // LDS rows are unpadded and their 16-byte chunks XOR-swizzled with bits of the row index (ab_key / b1_key).
    // A ds_read_b128 is served in four cycles of 16 lanes each, and the lanes of a cycle are those with equal
    // (lane bit 5, parity of lane bits 2..4) -- measured with random bank-balanced address patterns, which that
    // partition predicts exactly; row padding (16 bytes) left every fragment read of this kernel with two- to
    // four-way bank conflicts under it (SQ_LDS_BANK_CONFLICT = half of SQ_LDS_IDX_ACTIVE). The keys make the 16
    // lanes of every cycle of every fragment read land on 16 different 16-byte bank groups.
    static constexpr int AST  = KP * 2; // LDS row stride of A / B0 (bytes)
    // chunk position of chunk c of staged row r of A / B0: c ^ ab_key(r)
    __device__ static __forceinline__ uint32_t ab_key(uint32_t r)
    {
        // (KP / 8 chunks per row: 4, 8 or 16 -- the key stays inside the row)
        return (((r >> 3) & 1u) << 1) | (KP >= 64 ? ((r >> 1) & 1u) << 2 : 0u) | (KP == 128 ? (r & 1u) << 3 : 0u);
    }
    // The B1 slice of a step stays as it is in memory, [n][o] (row stride B1RS bytes), and the gemm1 operand -- for
    // one o, eight consecutive n -- comes out of it through the transposing read ds_read_b64_tr_b16: within 16 lanes,
    // lane 4e + j points at four consecutive o of row n + e, and lane i receives element i of the 16 so addressed
    // in each of the four rows. (Transposing on the way in took 32 two-byte LDS writes per thread and step.)
    // b1_key(n): XOR mask on the byte offset inside row n, so that the 32 lanes of a half wave (rows n + e and
    // n + 8 + e, four 8-byte pieces each) touch 32 different 8-byte bank pairs: with 128-byte rows the parity of n
    // already selects the bank half and bits 1 and 3 of n move the piece (bits 3, 4 of the offset); 256-byte rows
    // all start at bank 0, and bit 0 of n swaps the two 128-byte halves as well.
    static constexpr int B1RS = OP * 2;
    __device__ static __forceinline__ uint32_t b1_key(uint32_t n)
    {
        return (((n >> 1) & 1u) << 3) | (((n >> 3) & 1u) << 4) | (OG == 2 ? (n & 1u) << 7 : 0u);
    }
    static constexpr int A_BYTES   = BM * AST;
    static constexpr int B0_BYTES  = BNC * AST;
    static constexpr int B1T_BYTES = BNC * B1RS;
    static constexpr int LDS       = A_BYTES + B0_BYTES + B1T_BYTES;
    static constexpr int KCH = KP / 8; // 16-byte chunks per staged row of A / B0
    static constexpr int OCH = OP / 8;
    static constexpr int NB0 = BNC * KCH / NT; // 16-byte loads per thread and step
    static constexpr int NB1 = BNC * OCH / NT;
    static_assert(NB0 >= 1 && NB1 >= 1, "too many threads for one step");
};

// Waves per SIMD that the registers are allocated for. The 8-wave softmax variant for K up to 32 is held to 128, two workgroups per
// CU. The 8-wave variants past K or O of 64 take more than 128 registers and a whole CU, two waves per SIMD, whatever they do: told
// so, the compiler spends up to 256 on reads ahead instead of saving some for a third wave that no workgroup has. Without softmax
// K 64, O 128: 16 x 20 x 1000 17.2 -> 14.9 us, 60 x 300 x 256 8.0 -> 7.3; K 128, O 32 and K 32, O 128 0.88 and 0.94 of the time; with
// softmax level.
constexpr int gemm_gemm_min_waves(int KS, int OG, int NW, bool SOFTMAX)
{
    if(NW == 8 && (KS == 4 || OG == 2))
        return 2;
    return SOFTMAX && OG == 1 && NW == 8 && KS == 1 ? 4 : 1;
}
constexpr int gemm_gemm_max_waves(int KS, int OG, int NW) { return NW == 8 && (KS == 4 || OG == 2) ? 2 : 8; }

template <int KS, int OG, int MT, int NW, bool SOFTMAX = false>
__global__ __launch_bounds__(NW * 64)
    __attribute__((amdgpu_waves_per_eu(gemm_gemm_min_waves(KS, OG, NW, SOFTMAX), gemm_gemm_max_waves(KS, OG, NW)))) void gemm_gemm_kernel(
        const GemmGemmArgs p)
{
    using Cfg = GemmGemmCfg<KS, OG, MT, NW>;
    constexpr int KCH = Cfg::KCH, OCH = Cfg::OCH, NB0 = Cfg::NB0, NB1 = Cfg::NB1, NT = Cfg::NT;
    extern __shared__ __attribute__((aligned(16))) uint8_t gg_smem[];
    uint8_t* sA   = gg_smem;
    uint8_t* sB0  = sA + Cfg::A_BYTES;
    uint8_t* sB1T = sB0 + Cfg::B0_BYTES;

    const int tid  = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int fr   = lane & 15; // MFMA row/col index supplied by this lane
    const int q    = lane >> 4; // K-slot group

    int g, slab;
    slab_of_block<SOFTMAX>((int)blockIdx.x, p, g, slab);
    const int m0       = slab * Cfg::BM;
    const _Float16* A  = p.a + (int64_t)g * p.bsa;
    const _Float16* B0 = p.b0 + (int64_t)g * p.bsb0;
    const _Float16* B1 = p.b1 + (int64_t)g * p.bsb1;
    _Float16* C        = p.c + (int64_t)g * p.bsc;
    const i32x4 zero4  = {0, 0, 0, 0};

    // ---- register prefetch of one step's B0 / B1 slices ------------------------------------
    // Buffer loads: one resource per operand over the batch's rows, and per thread and load a byte offset that is fixed
    // for the whole kernel (row inside the slice, 16-byte chunk; out of range for chunks past K / O) -- a step adds its
    // first row, one addition per load, and rows past N read as zeros through the range check.
    const __amdgpu_buffer_rsrc_t rsrc_b0 = make_rsrc(B0, p.N > 0 ? (uint32_t)(((int64_t)(p.N - 1) * p.sb0 + p.K) * 2) : 0u);
    const __amdgpu_buffer_rsrc_t rsrc_b1 = make_rsrc(B1, p.N > 0 ? (uint32_t)(((int64_t)(p.N - 1) * p.sb1 + p.O) * 2) : 0u);
    uint32_t vb0[NB0], vb1[NB1];
#pragma unroll
    for(int i = 0; i < NB0; ++i)
    {
        const int idx = tid + NT * i;
        const int row = idx / KCH, ch = idx - row * KCH;
        vb0[i]        = ch * 8 < p.K ? (uint32_t)row * (uint32_t)p.sb0 * 2u + (uint32_t)ch * 16u : kOutOfRange;
    }
#pragma unroll
    for(int i = 0; i < NB1; ++i)
    {
        const int idx = tid + NT * i;
        const int row = idx / OCH, ch = idx - row * OCH;
        vb1[i]        = ch * 8 < p.O ? (uint32_t)row * (uint32_t)p.sb1 * 2u + (uint32_t)ch * 16u : kOutOfRange;
    }
    i32x4 rb0[NB0], rb1[NB1];
    auto load_into = [&](int n0, i32x4(&r0)[NB0], i32x4(&r1)[NB1]) {
        const uint32_t step0 = (uint32_t)n0 * (uint32_t)p.sb0 * 2u, step1 = (uint32_t)n0 * (uint32_t)p.sb1 * 2u;
#pragma unroll
        for(int i = 0; i < NB0; ++i)
            r0[i] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc_b0, vb0[i] + step0, 0, 0));
#pragma unroll
        for(int i = 0; i < NB1; ++i)
            r1[i] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc_b1, vb1[i] + step1, 0, 0));
    };
    auto load_step = [&](int n0) { load_into(n0, rb0, rb1); };
    auto store_step = [&]() {
#pragma unroll
        for(int i = 0; i < NB0; ++i)
        {
            const int idx = tid + NT * i;
            const int row = idx / KCH, ch = idx - row * KCH;
            *reinterpret_cast<i32x4*>(sB0 + row * Cfg::AST + ((uint32_t)ch ^ Cfg::ab_key((uint32_t)row)) * 16) = rb0[i];
        }
#pragma unroll
        for(int i = 0; i < NB1; ++i)
        {
            const int idx = tid + NT * i;
            const int row = idx / OCH, ch = idx - row * OCH;
            // (two 8-byte halves: the key may swap them)
            uint8_t* dst = sB1T + row * Cfg::B1RS;
            const uint32_t off = (uint32_t)(ch * 16) ^ Cfg::b1_key((uint32_t)row);
            *reinterpret_cast<i32x2*>(dst + off)       = i32x2{rb1[i][0], rb1[i][1]};
            *reinterpret_cast<i32x2*>(dst + (off ^ 8)) = i32x2{rb1[i][2], rb1[i][3]};
        }
    };

    // the same for the second register set of the two-step prefetch (unused, and gone, where PF == 1)
    i32x4 rb0b[NB0], rb1b[NB1];
    auto store_from = [&](const i32x4(&r0)[NB0], const i32x4(&r1)[NB1]) {
#pragma unroll
        for(int i = 0; i < NB0; ++i)
        {
            const int idx = tid + NT * i;
            const int row = idx / KCH, ch = idx - row * KCH;
            *reinterpret_cast<i32x4*>(sB0 + row * Cfg::AST + ((uint32_t)ch ^ Cfg::ab_key((uint32_t)row)) * 16) = r0[i];
        }
#pragma unroll
        for(int i = 0; i < NB1; ++i)
        {
            const int idx = tid + NT * i;
            const int row = idx / OCH, ch = idx - row * OCH;
            uint8_t* dst = sB1T + row * Cfg::B1RS;
            const uint32_t off = (uint32_t)(ch * 16) ^ Cfg::b1_key((uint32_t)row);
            *reinterpret_cast<i32x2*>(dst + off)       = i32x2{r1[i][0], r1[i][1]};
            *reinterpret_cast<i32x2*>(dst + (off ^ 8)) = i32x2{r1[i][2], r1[i][3]};
        }
    };

    load_step(0);

    // ---- A slab -> LDS -> registers (kept for the whole kernel) -----------------------
    for(int idx = tid; idx < Cfg::BM * KCH; idx += NT)
    {
        const int row = idx / KCH, ch = idx - row * KCH;
        const int m = m0 + row, k = ch * 8;
        i32x4 v = zero4;
        if(m < p.M && k < p.K)
            v = *reinterpret_cast<const i32x4*>(A + (int64_t)m * p.sa + k);
        *reinterpret_cast<i32x4*>(sA + row * Cfg::AST + ((uint32_t)ch ^ Cfg::ab_key((uint32_t)row)) * 16) = v;
    }
    __syncthreads();
    f16x8 af[MT][KS];
#pragma unroll
    for(int mt = 0; mt < MT; ++mt)
#pragma unroll
        for(int ks = 0; ks < KS; ++ks)
        {
            const uint32_t arow = (uint32_t)(wave * 16 * MT + mt * 16 + fr);
            af[mt][ks] = *reinterpret_cast<const f16x8*>(sA + arow * Cfg::AST + ((uint32_t)(ks * 4 + q) ^ Cfg::ab_key(arow)) * 16);
        }

    // byte offset inside the B1 slice that this lane addresses in the transposing reads of gemm1
    const uint32_t b1_lane =
        (uint32_t)(8 * q + (fr >> 2)) * Cfg::B1RS + ((uint32_t)(32 * (fr & 3)) ^ Cfg::b1_key((uint32_t)(8 * q + (fr >> 2))));

    // byte offsets of this lane's B0 fragments of score tiles 0 and 1: rows 8 * (fr / 4) + fr % 4 and 4 more. Tile t is 32 * (t / 2)
    // rows on, and neither step changes ab_key (bits 0, 1 and 3 of the row): immediates of the read. Worked out tile by tile
    // they became eight address registers and, in some of the kernels, a slower order of the step: without softmax 45 x 32 x
    // 1046 x 16 9.6 -> 11.3 us, 12 x 54 x 3073 x 32 22.6 -> 28.1. (Two registers for K up to 32 in the plain 8-wave
    // kernel, where one reads fewer fragments ahead: 231 x 45 x 2741 x 16 20.8 -> 20.0, 57 x 1934 x 61 x 32 7.3 -> 7.4, 7.7 with eight.)
    uint32_t b0_lane[KS][2];
#pragma unroll
    for(int ks = 0; ks < KS; ++ks)
    {
        const uint32_t row = (uint32_t)(8 * (fr >> 2) + (fr & 3));
        b0_lane[ks][0]     = row * Cfg::AST + ((uint32_t)(ks * 4 + q) ^ Cfg::ab_key(row)) * 16;
        b0_lane[ks][1]     = b0_lane[ks][0] + 4 * Cfg::AST;
        if constexpr(KS == 1 && !SOFTMAX && NW == 8)
            asm volatile("" : "+v"(b0_lane[ks][1]));
    }

    f32x4 acc1[MT][OG * 4];
#pragma unroll
    for(int mt = 0; mt < MT; ++mt)
#pragma unroll
        for(int t = 0; t < OG * 4; ++t)
            acc1[mt][t] = f32x4{0, 0, 0, 0};

    // softmax state of the MT rows this lane holds scores of (identical in the four lanes of a row,
    // except row_sum, which is each lane's share until the end)
    constexpr float kLog2e = 1.4426950408889634f;
    const float ninf       = -__builtin_inff();
    float row_max[MT], row_sum[MT];
#pragma unroll
    for(int mt = 0; mt < MT; ++mt)
        row_max[mt] = ninf, row_sum[mt] = 0.0f;
    // (never exactly 0: a masked score is -inf, and -inf * 0 would be a NaN; with the smallest normal number
    // instead, scale 0 still turns every unmasked score into 0)
    const float c2 = __builtin_fmaxf(__builtin_fabsf(p.scale) * kLog2e, 1.17549435e-38f);
    if(SOFTMAX && p.scale < 0.0f)
    {
        // scores = scale * (A * B0) = |scale| * ((-A) * B0): flip the sign bits of the A fragments once
#pragma unroll
        for(int mt = 0; mt < MT; ++mt)
#pragma unroll
            for(int ks = 0; ks < KS; ++ks)
                af[mt][ks] = __builtin_bit_cast(f16x8, __builtin_bit_cast(i32x4, af[mt][ks]) ^ (int)0x80008000);
    }
    // with the upper-triangle mask, columns past the slab's last row are masked for every row of it
    const int n_end = (SOFTMAX && p.mask_upper && m0 + Cfg::BM < p.N) ? m0 + Cfg::BM : p.N;

    // The softmax step is compiled in three forms, chosen per step and wave (wave-uniform): without a masked column it is straight-line
    // code without compares; with masked columns in all of its four 32-column pairs it compares, in straight-line code still; past
    // the wave's last unmasked column (EDGE) the pairs that lie there are left out, behind branches. With the first and the last:
    // causal 200 x 300 x 300 x 128 27.0 -> 26.0 us. With the middle one, which most steps of a single-step problem and the last of
    // N % 128 > 96 take: 26 x 66 x 121 x 64 4.83 -> 4.62, 53 x 226 x 363 x 64 -> 128 11.3 -> 10.7; not for K and O past 64, whose
    // other forms it slows down (206 x 1803 x 1803 x 128 560 -> 582).
    // RAISE: MFMA sections at raised wave priority, so that the other wave of the SIMD does its softmax meanwhile: faster with K of
    // 33 to 64, slower with K of 72 ... 128 (32 x 2048 x 2048 x 128 93.3 -> 94.6) and 32 and without softmax (128 x 1024 x 1024 x 64
    // 38.2 -> 39.2).
    constexpr bool RAISE = SOFTMAX && KS == 2;
    // One form, with the compares behind a branch, where more forms' registers cost a co-resident workgroup: 8 waves with
    // K up to 32 and O up to 64 (122 registers, 150 with two forms: 200 x 500 x 500 x 32 24.4 -> 32.7 us) and the 64-row instances.
    constexpr bool FORMS = SOFTMAX && NW == 8 && !(KS == 1 && OG == 1);
    constexpr bool MIDDLE_FORM = FORMS && !(KS == 4 && OG == 2);
    const int wave_m0    = m0 + wave * 16 * MT;
    const int wave_n_end = (p.mask_upper && wave_m0 + 16 * MT < p.N) ? wave_m0 + 16 * MT : p.N;
    const int full_end   = (p.mask_upper && wave_m0 + 1 < p.N) ? wave_m0 + 1 : p.N;
    auto edge_step       = [&](int n0) { return n0 + Cfg::BNC > full_end; };
    auto pairs_of        = [&](int n0) { return (wave_n_end - n0 + 31) >> 5; };

    // ---- main loop over the steps ---------------------------------------------------------------------------
    // A step's MFMAs take well under a microsecond, a load out of HBM longer: with one step of register prefetch
    // every step of a short problem (N = 512: four steps) ends waiting for its successor's slices. Where the
    // registers allow, the slices of TWO steps are in flight (PF == 2: a second register set, the loop unrolled by
    // two). The softmax variants and the largest plain one have no room (they would spill) and keep one.
    constexpr int PF = ((MT == 2 && NW == 4) || (SOFTMAX && (NW != 8 || (KS == 4 && OG == 2)))) ? 1 : 2;
    if constexpr(PF == 1)
    {
        for(int n0 = 0; n0 < n_end; n0 += Cfg::BNC)
        {
            __syncthreads(); // everyone is done reading the previous step from LDS
            store_step();
            __syncthreads();
            if(n0 + Cfg::BNC < n_end)
                load_step(n0 + Cfg::BNC); // in flight while this step is multiplied
#include "gemm_gemm_forms.inc"
        }
    }
    else
    {
        // step i lives in register set i % 2 until it goes to LDS
        if(Cfg::BNC < n_end)
            load_into(Cfg::BNC, rb0b, rb1b);
        for(int nb = 0; nb < n_end; nb += 2 * Cfg::BNC)
        {
            {
                const int n0 = nb;
                __syncthreads();
                store_from(rb0, rb1);
                __syncthreads();
                if(n0 + 2 * Cfg::BNC < n_end)
                    load_into(n0 + 2 * Cfg::BNC, rb0, rb1);
#include "gemm_gemm_forms.inc"
            }
            if(nb + Cfg::BNC < n_end)
            {
                const int n0 = nb + Cfg::BNC;
                __syncthreads();
                store_from(rb0b, rb1b);
                __syncthreads();
                if(n0 + 2 * Cfg::BNC < n_end)
                    load_into(n0 + 2 * Cfg::BNC, rb0b, rb1b);
#include "gemm_gemm_forms.inc"
            }
        }
    }

    if constexpr(SOFTMAX)
    {
#pragma unroll
        for(int mt = 0; mt < MT; ++mt)
        {
            const float total = quad_rows_sum(row_sum[mt]);
            const float inv   = total > 0.0f ? 1.0f / total : 0.0f; // N == 0: an empty sum, C = 0
#pragma unroll
            for(int ot = 0; ot < OG * 4; ++ot)
                acc1[mt][ot] = acc1[mt][ot] * inv;
        }
    }
#pragma unroll
    for(int mt = 0; mt < MT; ++mt)
    {
        const int m = m0 + wave * 16 * MT + mt * 16 + fr;
        if(m >= p.M)
            continue;
#pragma unroll
        for(int og = 0; og < OG; ++og)
        {
            const int o0 = 64 * og + 16 * q;
            if(o0 >= p.O)
                continue;
            const f32x4 v[4] = {acc1[mt][og * 4], acc1[mt][og * 4 + 1], acc1[mt][og * 4 + 2],
                                acc1[mt][og * 4 + 3]};
            store_row16_f16(C + (int64_t)m * p.sc, o0, p.O, v);
        }
    }
}

// ---------------------------------------------------------------- host side
constexpr int kNumGemmGemmInstances = 3;

inline const char* gemm_gemm_instance_name(int i, bool softmax)
{
    return i == 0 && softmax ? "MI355X_Mfma32_GemmSoftmaxGemm<128 rows, 4 waves x 32, steps of 64 or 32 cols, K<=128, O<=128>"
           : i == 0 ? "MI355X_Mfma16_GemmGemm<128 rows, 4 waves x 32, 128-col steps, K<=128, O<=128>"
           : i == 1 ? "MI355X_Mfma16_GemmGemm<64 rows, 4 waves x 16, 128-col steps, K<=128, O<=128>"
                    : "MI355X_Mfma16_GemmGemm<128 rows, 8 waves x 16, 128-col steps, K<=128, O<=128>";
}

inline bool gemm_gemm_supported(int M, int N, int K, int O, int batch, int sa, int sb0, int sb1, int sc,
                                int64_t bsa, int64_t bsb0, int64_t bsb1, int64_t bsc, int instance,
                                std::string& why)
{
    (void)bsc;
    if(M < 0 || N < 0 || K < 0 || O < 0 || batch < 0)
        return why = "invalid: negative dimension", false;
    if(instance < -1 || instance >= kNumGemmGemmInstances)
        return why = "invalid: no such instance", false;
    if(K > 128 || O > 128)
        return why = "K and O above 128 are not built", false;
    if(K % 8 || O % 8 || sa % 8 || sb0 % 8 || sb1 % 8 || bsa % 8 || bsb0 % 8 || bsb1 % 8)
        return why = "K, O and the A/B0/B1 strides must be multiples of 8 elements (16 bytes)", false;
    if(sa < K || sb0 < K || sb1 < O || sc < O)
        return why = "stride smaller than the contiguous extent", false;
    if((long)((M + 63) / 64) * batch >= (1l << 31))
        return why = "grid too large", false;
    // (the slices of a batch are addressed through 32-bit buffer offsets)
    if((long)N * sb0 * 2 >= (1l << 31) || (long)N * sb1 * 2 >= (1l << 31))
        return why = "B0 / B1 of one batch must stay below 2 GiB", false;
    return true;
}

// A group is 64 to 127 batches: 8 per XCD and up keep both of a CU's places filled to the end, and more would only widen what the
// L2s hold at a time. (Batch by batch the heavy slabs of the last batch started when the rest was done: half of the CUs idle for
// the last third. Causal 64 x 4096 x 4096 x 64: 246.8 -> 202.8 us.) Groups of 32 to 63 and of 128 to 255, over 20 causal problems of
// 128 to 512 batches, N 1024 to 4096: heads of 64 1.02 and 0.97 of the time (128 x 1024: 1.10 and 1.05, 200 x 1024: 1.00 and
// 0.91), heads of 128, whose B0 and B1 take twice the L2, 0.98 and 1.01.
inline SlabOrder slab_order(int slabs, int batch)
{
    const int wanted = batch >= 128 ? batch / 64 : 1;
    int size         = (batch + wanted - 1) / wanted;
    if((batch & 7) == 0)
        size = (size + 7) & ~7; // (every group starts at XCD 0)
    const int groups = (batch + size - 1) / size;
    return SlabOrder{make_magic((uint32_t)size * (uint32_t)slabs), make_magic((uint32_t)size), make_magic((uint32_t)(batch - (groups - 1) * size)), groups};
}

template <int BM, int NT, int LDS>
inline hipError_t gemm_gemm_launch_kernel(void (*kern)(GemmGemmArgs), GemmGemmArgs a, hipStream_t s)
{
    a.slabs = (a.M + BM - 1) / BM;
    // (the threads of a grid dimension are counted in 32 bits, and a launch past them wraps around without an error: more batches
    // than fit go out in launches of their own, whole groups of eight of them for the XCD mapping)
    const long fit = ((1l << 32) - 1) / NT / a.slabs;
    if(fit < 1)
        return hipErrorInvalidValue;
    const int most = (int)(fit >= a.batch ? a.batch : fit >= 8 ? fit & ~7l : fit);
    for(int left = a.batch; left > 0; left -= most)
    {
        a.batch = left < most ? left : most;
        if(a.mask_upper)
            a.order = slab_order(a.slabs, a.batch);
        hipLaunchKernelGGL(kern, dim3(a.slabs * a.batch), dim3(NT), LDS, s, a);
        const hipError_t e = hipGetLastError();
        if(e != hipSuccess)
            return e;
        a.a += most * a.bsa, a.b0 += most * a.bsb0, a.b1 += most * a.bsb1, a.c += most * a.bsc;
    }
    return hipSuccess;
}

template <int KS, int OG, int MT, int NW, bool SOFTMAX>
inline hipError_t gemm_gemm_launch_t(const GemmGemmArgs& a, hipStream_t s)
{
    using Cfg  = GemmGemmCfg<KS, OG, MT, NW>;
    auto* kern = &gemm_gemm_kernel<KS, OG, MT, NW, SOFTMAX>;
    static std::once_flag once;
    static hipError_t attr_err = hipSuccess;
    std::call_once(once, [&] {
        attr_err = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::LDS);
    });
    if(attr_err != hipSuccess)
        return attr_err;
    return gemm_gemm_launch_kernel<Cfg::BM, Cfg::NT, Cfg::LDS>(kern, a, s);
}

template <int MT, int NW, bool SOFTMAX>
inline hipError_t gemm_gemm_launch_mt(const GemmGemmArgs& g, hipStream_t s)
{
    const int ks = g.K <= 32 ? 1 : (g.K <= 64 ? 2 : 4);
    const int og = g.O <= 64 ? 1 : 2;
    if(ks == 1)
        return og == 1 ? gemm_gemm_launch_t<1, 1, MT, NW, SOFTMAX>(g, s) : gemm_gemm_launch_t<1, 2, MT, NW, SOFTMAX>(g, s);
    if(ks == 2)
        return og == 1 ? gemm_gemm_launch_t<2, 1, MT, NW, SOFTMAX>(g, s) : gemm_gemm_launch_t<2, 2, MT, NW, SOFTMAX>(g, s);
    return og == 1 ? gemm_gemm_launch_t<4, 1, MT, NW, SOFTMAX>(g, s) : gemm_gemm_launch_t<4, 2, MT, NW, SOFTMAX>(g, s);
}

hipError_t gemm_gemm_wide_launch(const GemmGemmArgs& a, int parts, hipStream_t s); // gemm_gemm_wide.hip: the same kernel without its softmax
hipError_t gemm_softmax_gemm_launch(const GemmGemmArgs& a, int parts, hipStream_t s); // gemm_softmax_gemm.hip; parts: shares of the columns, 1, 2 or 4

// Attention on waves of 16 rows (instance 2) instead of 32 (instance 0). Up to 256 slabs of 128 rows there is one workgroup to a CU: one
// wave of 32 rows per SIMD, or two of 16, and the launch lasts as long as one wave's chain of steps. The shorter chain wins then, up to an
// N from which the 32-row kernel's faster steps do; with heads past 96 at any N, and with the mask, whose launch ends with its longest
// slabs alone on their CUs, up to 512 slabs. From there on, and with heads of 65 to 96, which the 16-row kernel pads to 128, 32 rows.
// 16 / 32 rows, us: heads of 64: 64 x 512 x 512 10.6 / 11.2, 128 x 256 x 256 7.2 / 8.0, 42 x 768 x 768 causal 13.4 / 14.4, 8 x 1024 x 1024
// causal 15.5 / 15.8, but 32 x 1024 x 1024 19.6 / 17.3, 5 x 1536 x 1536 21.8 / 21.2, 175 x 512 x 512 33.2 / 26.7, 350 x 256 x 256 21.4 / 18.2;
// heads of 128: 64 x 512 x 512 17.1 / 18.1, 21 x 1536 x 1536 causal 37.9 / 38.6, 35 x 1362 x 1362 causal 37.5 / 40.2, but 36 x 1384 x 1384
// 72.0 / 54.6, 63 x 1357 x 1357 causal 67.9 / 51.2; heads of 32: 128 x 256 x 256 5.6 / 5.8, but 64 x 512 x 512 8.3 / 8.1, 32 x 1024 x 1024
// 15.6 / 12.5; of 80: 32 x 256 x 256 8.6 / 7.9. The lines in N lie on the careful side: with one slab to a batch (M = 128) 32 rows are level with 16 at N 768 and
// 1.02 to 1.08 ahead from 832 on (heads of 64, 200 batches: 960 17.4 / 16.1, 968 17.7 / 16.8, 1024 17.6 / 16.7, 1032 18.7 / 17.6), and for heads of
// 32 1.02 to 1.14 ahead from 320 on (128 batches: 384 6.8 / 6.5, 440 8.2 / 7.5, 448 8.3 / 7.2, 480 8.1 / 7.7).
// Past 256 slabs of heads past 96 the masked 16-row kernel, of which a CU holds one workgroup, stays ahead from 896 columns up to 384 slabs (40 x 946 x 946
// 24.5 / 26.4, level at 48 x 952 x 952), and up to 512 where the launch lasts no longer than its longest chain (second_slabs_fit()) and either the
// chains are long or every XCD has whole batches, whose columns stay in its L2. us, 16 rows / 32 rows, heads of 128: 24 x 2304 x 2304 54.5 / 60.8, 16 x 3102 x
// 3102 68.5 / 75.0, 28 x 1909 x 1909 46.8 / 51.2, 32 x 1588 x 1588 38.0 / 40.9, 48 x 869 x 869 24.0 / 26.5, 64 x 611 x 611 18.5 / 20.4; where they do not
// fit: 48 x 1030 x 1030 32.2 / 29.7, 51 x 1244 x 1244 45.2 / 40.1, 54 x 815 x 815 28.8 / 25.4, 112 x 397 x 397 22.9 / 16.5, 297 x 104 x 104 15.3 / 11.9; with a
// few batches more on some XCDs: 51 x 813 x 813 29.0 / 25.9, 46 x 858 x 858 26.3 / 26.0, 37 x 1365 x 1365 39.8 / 38.5. (With columns past the last row, masked for all,
// its line is 512 slabs.) Of 195 random problems with M = N > 576 the choice is at most 4 % behind the other kernel but for four (up to 8 %), and up to 1.29 ahead;
// heads of 64, 134 x 158 x 158 9.8 / 8.2, 442 x 128 x 128 11.1 / 9.4, 112 x 353 x 353 11.2 / 10.4, but with K 32 and O 64 104 x 352 x 352 8.3 / 8.9.
//
// Masked slabs, M >= N, one workgroup to a CU, up to two rounds, longest chains first: the k-th slab past the CUs starts where the k-th slab ends
// from the back. Whether they all end before the longest one, with 80 columns' time for a slab's first loads: looked at where the first slab's
// chain becomes a longer one, as the second's only become shorter.
inline bool second_slabs_fit(int M, int N, int batch)
{
    const long per_batch = (M + 127) / 128, cus = num_cus(), slabs = batch * per_batch;
    if(slabs > 2 * cus)
        return false;
    const auto chain = [&](long rank) { const long c = 128 * (per_batch - rank / batch); return c < N ? c : (long)N; };
    for(long k = 0; cus + k < slabs; k = cus - (cus - 1 - k) / batch * batch)
        if(chain(cus + k) + chain(cus - 1 - k) + 80 > N)
            return false;
    return true;
}
inline bool rows_in_16s(int M, int N, int K, int O, int batch, bool mask_upper)
{
    const int head   = K > O ? K : O;
    const long slabs = (long)batch * ((M + 127) / 128) * 256 / num_cus(); // (as on 256 CUs, which the lines here were measured on)
    if(head > 96)
        return slabs <= (!mask_upper ? 256 : M < N ? 512 : N >= 896 ? 384 : 256) ||
               (mask_upper && M >= N && N > 576 && (N >= 1600 || batch % 8 == 0) && second_slabs_fit(M, N, batch));
    if(slabs > 256 && M >= N && N <= 352 && K > 32)
        return false;
    // (130 x 375 x 375 13.2 / 13.8 us; longer N, where the second workgroup of some CUs comes late enough: 43 x 768 x 768 13.9 / 14.9, 64 x 768 x
    // 768 13.5 / 14.7, 47 x 896 x 896 0.97 of the time, but 75 x 640 x 640 1.04, 67 x 768 x 768 1.00)
    if(mask_upper && head > 32 && head <= 64 && N < 1024)
        return slabs <= (N <= 512 ? 512 : N < 768 ? 304 + 3 * (N - 512) / 8 : 384);
    return slabs <= 256 && (head > 64 ? false : head > 32 ? N <= (slabs <= 128 ? 1024 : 960) : N < 448);
}

// Attention, the shares of the columns that a workgroup's groups of waves take side by side: 1, 2 (128 rows) or 4 (64 rows), see
// gemm_softmax_gemm.hpp. With one workgroup or fewer to a CU the launch lasts as long as a wave's chain of units, which the shares shorten;
// with more the CUs are busy anyway, and what the shares cost shows: the merge, and with 64 rows every column read twice as often. A launch
// under the triangular mask may have more of them once its chain is long: they start longest first, and the short ones fit in behind. Below
// the lines in the chain's length the first loads and the merge cost more than the shares give; heads of 65 to 96 in quarters pad to 128. Behind
// every line: S shares take (1 - 1 / S) of a chain's units away and add a merge that grows with the head, and in quarters the first
// loads of twice the workgroups; a CU with a second workgroup has the units' waits filled already.
// Up to 64 rows of heads of 33 to 64 have one share up to 1025 columns, because outputs there are held bit for bit to those of the 16-row
// kernel, and at 1025 of the 32-row one. From 736 columns on that costs time: batch x 64 x N of heads 64, one share / four, us: 16 x 736 12.1 / 10.7, 16 x
// 960 15.0 / 11.8, 96 x 1024 15.6 / 12.6, 224 x 960 16.8 / 14.9, 224 x 1024 15.5 / 15.2; below not: 16 x 640 10.3 / 10.5, 224 x 640 12.2 / 12.9.
// 1 part (16 or 32 rows as rows_in_16s() chooses) / 2 / 4, us, full: batch x M x N 3 x 3034 x 3034 of heads 32 28.5 / 24.0 / 15.5, 6 x
// 3760 x 1709 / 64 23.7 / 20.7 / 16.5, 14 x 802 x 802 / 64 14.7 / 13.4 / 12.7, 12 x 1275 x 1275 / 80 23.0 / 21.2 / 21.7, 8 x 1676 x 1676 / 128
// 39.8 / 32.5 / 27.2, 4 x 991 x 3837 / 128 81.2 / 62.1 / 45.6, but 6 x 2806 x 2806 / 64 (264 slabs of 64) 35.4 / 29.4 / 43.1, 8 x 1918 x 490 / 64 9.7 /
// 10.2 / 9.6, 125 x 70 x 931 / 128 25.2 / 21.2 / 25.7 (two slabs of 64 for one of 128). Causal: 6 x 3772 / 64 44.9 / 37.0 / 28.3 (354 slabs of
// 64), 25 x 936 / 64 16.3 / 15.0 / 19.7 (375), 15 x 591 / 64 11.0 / 11.4 / 11.8, 6 x 3707 / 128 78.7 / 60.8 / 47.9, 18 x 573 / 128 16.5 / 16.3 / 16.7.
// Of 340 random problems none that takes parts is slower than with one; 2 parts give up to 1.34, 4 up to 1.84 times.
inline int column_parts(int M, int N, int K, int O, int batch, bool mask_upper)
{
    const int head     = K > O ? K : O;
    const bool tri     = mask_upper && M <= N;
    const int chain    = mask_upper && M < N ? M : N;
    const long by64    = (long)batch * ((M + 63) / 64) * 256 / num_cus(), by128 = (long)batch * ((M + 127) / 128) * 256 / num_cus();
    const long most    = tri && chain >= 1792 ? 384 : tri && chain >= 1024 ? 320 : 256;
    const int line64   = M <= 64 ? 1026 : 640;
    const int from4    = head <= 32 ? 576 : head <= 64 ? line64 : head <= 96 ? 1536 : 640;
    const int from2    = head <= 32 ? 576 : head <= 64 ? (mask_upper && line64 < 768 ? 768 : line64) : head <= 96 ? 768 : 576;
    if(chain >= from4 && by64 <= (M > 64 && M <= 128 ? 192 : most))
        return 4;
    return chain >= from2 && by128 <= (chain < 1024 ? 224 : most) ? 2 : 1;
}

// Without softmax: shares of the columns (1, 2 or 4, as above) on the 32-row kernel, or 0 for the kernels of 128-column steps.
// The 32-row waves read B0 and B1 fragments half as often per product and keep other units' reads and conversions between their MFMAs; their
// units of 32 or 64 columns pad N less than steps of 128. The kernels of 128-column steps have more waves per row, and stay ahead on short chains
// and, with heads of 33 to 64, while few workgroups leave the CUs to one wave of 32 rows per SIMD. us, steps of 128 / 1 / 2 / 4 shares, by slabs of
// 128 rows and N: heads of 32: 351 slabs, 299 8.0 / 6.3 / 9.5 / 13.3; 408, 1087 16.3 / 11.7 / 15.2 / 27.4; 109, 975 9.6 / 8.3 / 6.9 / 8.2; 96, 1388 11.7 / 9.8 / 8.1 / 7.7;
// but 72, 402 level. Of 64: 328, 747 16.6 / 15.1 / 20.1 / 22.1; 180, 946 12.0 / 11.2 / 12.3 / 21.5; 147, 1997 19.3 / 17.5 / 16.9 / 22.9; 50, 1753 15.3 / 15.6 / 14.8 /
// 13.6, but 99, 811 9.3 / 9.8 / 10.2 / 9.9; 256, 512 7.7 / 8.4 / 9.1 / 14.9; 576, 275 13.5 / 14.5; 84, 1881 (168 slabs of 64) 16.9 and 17.4 in four shares. Of 128: 592,
// 294 36.4 / 25.4 / 34.1 / 52.8; 51, 692 16.6 / 14.0 / 14.7 / 14.6; 45, 1946 36.5 / 29.2 / 27.1 / 23.4; 45, 142 7.8 / 7.3, but 27, 235, which fills its steps,
// 7.2 / 7.6; 63, 111 6.0 / 6.9; of K 128 and O 32, 75, 738 12.4 / 12.8. 190 random problems up to 1400 slabs: 1.12 times as fast on average, up to 1.95.
inline int wide_parts(int M, int N, int K, int O, int batch)
{
    const int head   = K > O ? K : O;
    const long by64  = (long)batch * ((M + 63) / 64) * 256 / num_cus(), by128 = (long)batch * ((M + 127) / 128) * 256 / num_cus();
    const bool few   = by128 <= 256;
    if(N >= (head <= 32 ? 1024 : head <= 64 ? 1152 : 1280) && by64 <= (head > 32 && head <= 64 ? 160 : 192))
        return 4;
    if(head <= 32)
        return few && N >= 768 ? 2 : N >= (few ? 448 : 288) ? 1 : 0;
    if(head <= 64)
        return few ? (by128 <= 128 || N < 768 ? 0 : N < 1400 ? 1 : 2) : N >= 576 ? 1 : 0;
    if(few && N >= 1280)
        return 2;
    if(few && N < 1024 && (K <= 32 || O <= 32))
        return 0;
    return N >= 264 || (K > 64 && O > 64 && (!few || (N > 128 && N <= 192))) ? 1 : 0;
}

// softmax: the attention variant with scores scale * (A * B0) and the optional upper-triangle mask
inline hipError_t gemm_gemm_launch(const void* a, const void* b0, const void* b1, void* c, int M, int N, int K,
                                   int O, int batch, int sa, int sb0, int sb1, int sc, int64_t bsa,
                                   int64_t bsb0, int64_t bsb1, int64_t bsc, int instance, hipStream_t s,
                                   bool softmax = false, float scale = 1.0f, bool mask_upper = false)
{
    GemmGemmArgs g;
    g.a = (const _Float16*)a, g.b0 = (const _Float16*)b0, g.b1 = (const _Float16*)b1, g.c = (_Float16*)c;
    g.M = M, g.N = N, g.K = K, g.O = O, g.batch = batch;
    g.sa = sa, g.sb0 = sb0, g.sb1 = sb1, g.sc = sc;
    g.bsa = bsa, g.bsb0 = bsb0, g.bsb1 = bsb1, g.bsc = bsc;
    g.slabs = 0, g.order = SlabOrder{};
    g.scale = scale, g.mask_upper = mask_upper;
    if(softmax)
    {
        if(instance < 0)
        {
            const int parts = column_parts(M, N, K, O, batch, mask_upper);
            if(parts > 1)
                return gemm_softmax_gemm_launch(g, parts, s);
            instance = rows_in_16s(M, N, K, O, batch, mask_upper) ? 2 : 0;
        }
        return instance == 0   ? gemm_softmax_gemm_launch(g, 1, s)
               : instance == 1 ? gemm_gemm_launch_mt<1, 4, true>(g, s)
                               : gemm_gemm_launch_mt<1, 8, true>(g, s);
    }
    if(instance < 0)
    {
        // Many short waves (8 x 16 rows, the instance with two steps of prefetch where registers allow) are ahead on short
        // problems: G 64, 512 x 64 x 512 x 64 8.5 against 10.1 us. Up to 128 slabs of small heads the 64-row instance, which doubles
        // the workgroups, is (20.6 against 25.4 us).
        const long slabs128 = (long)batch * ((M + 127) / 128);
        const bool small_heads = K <= 64 && O <= 64;
        const int parts        = wide_parts(M, N, K, O, batch);
        if(parts > 0)
            return gemm_gemm_wide_launch(g, parts, s);
        instance = small_heads && slabs128 <= 128 ? 1 : 2;
    }
    return instance == 0 ? gemm_gemm_launch_mt<2, 4, false>(g, s)
           : instance == 1 ? gemm_gemm_launch_mt<1, 4, false>(g, s)
                           : gemm_gemm_launch_mt<1, 8, false>(g, s);
}

} // namespace ckx
