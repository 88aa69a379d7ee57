// Batched fused GEMM-softmax-GEMM ("attention") for gfx950, fp16:
//   C[g] = half( half(softmax_n(scale * A[g] * B0[g], masked)) * B1[g] )
// A [G,M,K] row-major, B0 stored [G,N,K], B1 [G,N,O] row-major, C [G,M,O] row-major (the layout of gemm_gemm.hpp), softmax along N
// in one pass: running row maximum and sum, probabilities exp(s - maximum) rounded to fp16, one division at the end. Columns past N and,
// with the upper-triangle mask, columns n > m count as -infinity; units of columns masked for all rows of a wave are left out.
//
// A wave owns 32 rows and walks N in units of 64 (or 32) columns. gemm0 is issued as S^T = B0_frag x A_frag in 32x32x16 MFMAs: lane l
// holds row l%32 and, of every 32 columns, n = 8*(i/4) + 4*(l/32) + i%4 in its 16 registers. Eight of them, rounded to fp16, are the lane's
// share of the second operand of gemm1 (C^T = B1T_frag x P^T) over 16 columns, whose first operand is read in the same order of n: the
// scores never leave their lane.
//
// What bounds it: the vector instructions of the softmax (per score a multiply-add, an exponential that takes the pipe for two, half a
// conversion, half a three-way maximum) beside the matrix core. How long a SIMD takes for a 32x32x16 MFMA with two exponentials and n
// multiply-adds, two waves doing the same (cycles): n = 2 33.6, n = 4 41.6, n = 6 50.9, the MFMA alone 32 and 2 exponentials + 4
// multiply-adds alone 33.5. So the two overlap, but an MFMA costs about 8 cycles of issue, whatever its size: 16x16x32 ones, half the
// work each, need 51.8 for the n = 4 mix. v_dot2_f32_f16, which would sum the probabilities, does not overlap (32x32x16 MFMA + 4 of them
// 61 cycles, + 4 multiply-adds 33). Hence 32x32x16 MFMAs, and the middle units written out as one MFMA, then four or five vector
// instructions of ANOTHER unit, and so on: unit u's softmax among the products of unit u + 1's scores and unit u - 1's output.
// What is left over 4096 columns of heads of 64: the running maximum of some row of the wave rises in two units of three, and raising it and
// rescaling what has been accumulated takes about 50 vector instructions (a maximum that lags behind, moved on a 2^8-fold excess only, would
// take 0.98 and 0.96 of the time of the first two figures below, but its probabilities are rounded at less favourable places: 2-norm of the
// error against float64 2.62e-4 where this one and the 16-row kernel have 2.53e-4); and the clock, which the power limit holds at 1.9 GHz (with
// operands of zeros the same launch takes 0.75 of the time).
// Counters of 64 x 4096 x 4096 x 64 (of the time that two waves share a SIMD): matrix core busy 50 %, vector instructions active 71 %, 1.21 together; with
// 16x16x32 MFMAs, sums by v_dot2 and softmax and products one after the other 34 and 64 %, 0.98. us, that kernel and this one in turn on one card:
// 394.7 -> 359.1, causal 184.6 -> 179.4 (192.4 -> 189.5 with new operands in each pass); 32 x 2048 x 2048 x 128 92.4 -> 80.9, x 80 89.8 -> 58.8; 64 x 2048
// x 2048 x 32 79.1 -> 59.2. 48 + 120 random problems 0.76 and 0.88 of the time.
// SM = false: the same kernel without the softmax, for the fused pair of GEMMs (gemm_gemm_wide.hip; wide_parts() has its figures).
#pragma once

#include "gemm_gemm.hpp"

namespace ckx {

typedef float f32x16 __attribute__((ext_vector_type(16)));

// KS  k-steps of 16 of gemm0 (K padded to 16*KS), OT  32-column tiles of the output (O padded to 32*OT),
// NW  waves: a workgroup owns 32*NW rows of one batch.
template <int KS, int OT, int NW>
struct SoftmaxGemmCfg
{
    static constexpr int NT  = 64 * NW;
    static constexpr int BM  = 32 * NW;
    static constexpr int UC  = KS <= 6 && OT <= 3 ? 64 : 32; // columns of the scores per unit
    static constexpr int NB  = UC / 32;                      // 32-column blocks of a unit
    static constexpr int NK2 = UC / 16;                      // k-steps of gemm1 in a unit
    static constexpr int KRS = KS <= 2 ? 64 : KS <= 4 ? 128 : KS <= 6 ? 192 : 256; // LDS row strides of B0 and B1 in bytes
    static constexpr int VRS = 64 * OT;
    static constexpr int KCH = KRS / 16, VCH = VRS / 16; // 16-byte chunks of a row
    static constexpr int ROWS_K = KCH == 12 ? 16 * (NT / 192) : NT / KCH, ROWS_V = VCH == 12 ? 16 * (NT / 192) : NT / VCH; // rows per load
    static constexpr int NLK = (UC + ROWS_K - 1) / ROWS_K, NLV = (UC + ROWS_V - 1) / ROWS_V;
    static_assert((UC % ROWS_K == 0 || NLK == 1) && (UC % ROWS_V == 0 || NLV == 1), "");
    static_assert((ROWS_K % 16 == 0 || NLK == 1 || (KRS == 256 && ROWS_K == 8)) && (ROWS_V % 4 == 0 || NLV == 1), "the keys repeat after 16 and 4 rows");
    // (in steps of eight rows the key of a 256-byte row flips its highest bit every time)
    static constexpr uint32_t k_flip(int i) { return ROWS_K == 8 && (i & 1) ? 128u : 0u; }
    static constexpr int KSLOT = UC * KRS, VSLOT = UC * VRS;
    static constexpr int LDS = 2 * KSLOT + 2 * VSLOT;
    // XOR on the chunk position of row r. A ds_read_b128 is served 16 lanes at a time, those with equal (lane bit 5, parity of lane
    // bits 2..4); the lanes of a B0 fragment read are 32 rows of one chunk column, and under these keys the 16 rows of every group
    // lie in 16 different 16-byte banks. A transposing read of B1 is served 32 lanes at a time, four rows of 64 bytes.
    __device__ static __forceinline__ uint32_t k_key(uint32_t r)
    {
        return KRS == 128 ? (r >> 1) & 7u : KRS == 256 ? r & 15u : (r >> 2) & 3u;
    }
    __device__ static __forceinline__ uint32_t v_key(uint32_t r) { return VRS == 128 ? ((r >> 1) & 1u) << 2 : VRS == 256 ? (r & 3u) << 2 : 0u; }
};

// NS > 1: NS groups of NW waves own the same rows and take a share of the columns each, with slices of B0 and B1 of their own; at the end
// the other groups' maxima, sums and accumulators cross over to the first through LDS. For launches of few workgroups, which last as long as a
// wave's chain of units: a part of the chain, and a second wave on every SIMD to fill the first one's waits.
// (two groups of four waves, or four of two, which halves the rows of a workgroup too). One group / two / four, us: 1 x 2995 x 2995 of heads of 128
// 65.4 / 50.4 / 38.5, 1 x 3082 x 3082 / 64 38.3 / 31.4 / 24.0; 170 random problems up to 540 slabs,
// as column_parts() chooses, 1.17 times as fast on average, up to 1.84. The merge: 2-norm of the error against float32 as with one group (2.8e-4).
template <int KS, int OT, int NW, int NS = 1>
struct SoftmaxGemmSplit
{
    using Cfg = SoftmaxGemmCfg<KS, OT, NW>;
    static constexpr int CROSS = (NS - 1) * NW * (16 * OT + 2) * 256; // bytes that cross over
    static constexpr int LDS   = NS * Cfg::LDS > CROSS ? NS * Cfg::LDS : CROSS;
};

// SM: with the softmax; without, the scores rounded to fp16 take the probabilities' place (C = half( half(A * B0) * B1 ))
template <int KS, int OT, int NW, int NS = 1, bool SM = true>
__global__ __launch_bounds__(NW * NS * 64) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_softmax_gemm_kernel(const GemmGemmArgs p)
{
    using Cfg = SoftmaxGemmCfg<KS, OT, NW>;
    constexpr int NT = Cfg::NT, UC = Cfg::UC, NB = Cfg::NB, NK2 = Cfg::NK2, KRS = Cfg::KRS, VRS = Cfg::VRS, KCH = Cfg::KCH, VCH = Cfg::VCH,
                  NLK = Cfg::NLK, NLV = Cfg::NLV, ROWS_K = Cfg::ROWS_K, ROWS_V = Cfg::ROWS_V;
    extern __shared__ __attribute__((aligned(16))) uint8_t gg_smem[];
    const int all_waves = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int part      = NS == 1 ? 0 : all_waves / NW; // which columns
    const int wave      = all_waves - part * NW;
    const int tid       = threadIdx.x - part * NT;
    const int lane      = tid & 63;
    uint8_t* const sK   = gg_smem + part * Cfg::LDS;
    uint8_t* const sV   = sK + 2 * Cfg::KSLOT;
    const int row  = lane & 31; // this lane's row of the wave's 32
    const int h    = lane >> 5; // K-slot half

    int g, slab;
    slab_of_block<true>((int)blockIdx.x, p, g, slab);
    const int m0       = slab * Cfg::BM;
    const _Float16* A  = p.a + (int64_t)g * p.bsa;
    _Float16* C        = p.c + (int64_t)g * p.bsc;

    // with the upper-triangle mask, columns past the last row are masked for every row
    const int wave_m0 = m0 + wave * 32;
    const int n_end   = p.mask_upper && m0 + Cfg::BM < p.N ? m0 + Cfg::BM : p.N;
    // units that every wave takes part in; this part's first column, and its columns (everything below counts columns from there)
    const int all_units = (n_end + UC - 1) / UC, units = (all_units + NS - 1) / NS;
    const int n_first   = part * units * UC;
    const int N         = NS == 1 ? p.N : p.N <= n_first ? 0 : part < NS - 1 && p.N - n_first > units * UC ? units * UC : p.N - n_first;
    const int wave_c0   = wave_m0 - n_first;
    const _Float16* B0  = p.b0 + (int64_t)g * p.bsb0 + (int64_t)(NS == 1 ? 0 : n_first) * p.sb0;
    const _Float16* B1  = p.b1 + (int64_t)g * p.bsb1 + (int64_t)(NS == 1 ? 0 : n_first) * p.sb1;
    const int w_end     = p.mask_upper && wave_c0 + 32 < N ? wave_c0 + 32 : N;
    const int full      = p.mask_upper && wave_c0 + 1 < N ? wave_c0 + 1 : N; // columns below are unmasked for every row of the wave
    const int w_units   = wave_m0 < p.M && (NS == 1 || w_end > 0) ? (w_end + UC - 1) / UC : 0;

    // ---- B0 / B1 on their way: global -> registers -> LDS -----------------------------------------------------------------
    const __amdgpu_buffer_rsrc_t rsrc_k = make_rsrc(B0, N > 0 ? (uint32_t)(((int64_t)(N - 1) * p.sb0 + p.K) * 2) : 0u);
    const __amdgpu_buffer_rsrc_t rsrc_v = make_rsrc(B1, N > 0 ? (uint32_t)(((int64_t)(N - 1) * p.sb1 + p.O) * 2) : 0u);
    // (thread t takes chunk t % KCH of row t / KCH and of the same row ROWS_K further on: one offset into the operand and one into a
    // slot, whose keys repeat after 16 rows)
    const uint32_t rk0 = tid / KCH, ck = tid - rk0 * KCH, rv0 = tid / VCH, cv = tid - rv0 * VCH;
    const bool live_k = (KCH != 12 && ROWS_K <= UC) || rk0 < (ROWS_K < UC ? ROWS_K : UC);
    const bool live_v = (VCH != 12 && ROWS_V <= UC) || rv0 < (ROWS_V < UC ? ROWS_V : UC);
    const uint32_t gk = live_k && (int)ck * 8 < p.K ? rk0 * (uint32_t)p.sb0 * 2u + ck * 16u : kOutOfRange;
    const uint32_t gv = live_v && (int)cv * 8 < p.O ? rv0 * (uint32_t)p.sb1 * 2u + cv * 16u : kOutOfRange;
    const uint32_t lk = rk0 * KRS + (ck ^ Cfg::k_key(rk0)) * 16, lv = rv0 * VRS + (cv ^ Cfg::v_key(rv0)) * 16;
    // Byte offset of a unit's first row in the operand; a unit that does not exist starts at row N, the first past the end. Chunks past K or O
    // begin at kOutOfRange and stay out of range with all rows up to 64 past N added, but for operands that end less than 64 rows
    // below 2 GiB: there a sum may wrap around into the operand, for rows past N only. What is read then goes nowhere: columns past N get
    // -inf for a score by a select (mask), whatever it was, output columns past O are not stored, and units that do not exist meet no
    // product. (The out-of-range bit OR-ed into the sum instead, two to four instructions a unit: 1.03 of the time with one wave per SIMD.)
    auto first = [&](int u, int stride) { return (uint32_t)(u * UC < N ? u * UC : N) * (uint32_t)stride * 2u; };
    // (rows past the last one read as zeros through the range check; CHECKED: they are found by their number, for strides whose
    // offsets of rows past the last one may wrap around)
    auto load_k = [&](int u, i32x4(&r)[NLK], auto checked) {
        const uint32_t step = first(u, p.sb0);
#pragma unroll
        for(int i = 0; i < NLK; ++i)
        {
            uint32_t off = gk + (step + (uint32_t)(i * ROWS_K) * (uint32_t)p.sb0 * 2u);
            if(decltype(checked)::value)
                off = tid < (N - u * UC - i * ROWS_K) * KCH ? off : kOutOfRange;
            r[i] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc_k, off, 0, 0));
        }
    };
    auto load_v = [&](int u, i32x4(&r)[NLV], auto checked) {
        const uint32_t step = first(u, p.sb1);
#pragma unroll
        for(int i = 0; i < NLV; ++i)
        {
            uint32_t off = gv + (step + (uint32_t)(i * ROWS_V) * (uint32_t)p.sb1 * 2u);
            if(decltype(checked)::value)
                off = tid < (N - u * UC - i * ROWS_V) * VCH ? off : kOutOfRange;
            r[i] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc_v, off, 0, 0));
        }
    };
    auto store_k = [&](int slot, const i32x4(&r)[NLK]) {
#pragma unroll
        for(int i = 0; i < NLK; ++i)
            if(live_k)
                *reinterpret_cast<i32x4*>(sK + slot * Cfg::KSLOT + (lk ^ Cfg::k_flip(i)) + i * ROWS_K * KRS) = r[i];
    };
    auto store_v = [&](int slot, const i32x4(&r)[NLV]) {
#pragma unroll
        for(int i = 0; i < NLV; ++i)
            if(live_v)
                *reinterpret_cast<i32x4*>(sV + slot * Cfg::VSLOT + lv + i * ROWS_V * VRS) = r[i];
    };

    f16x8 af[KS]; // A: this lane's row, K-slots 16*ks + 8*h .. +7

    // ---- fragments ---------------------------------------------------------------------------------------------------------
    // B0, first operand of gemm0: rows n = 32*b + lane%32, K-slots 16*ks + 8*h .. +7 = chunk 2*ks + h
    uint32_t ka[KS];
#pragma unroll
    for(int ks = 0; ks < KS; ++ks)
        ka[ks] = (uint32_t)row * KRS + ((uint32_t)(2 * ks + h) ^ Cfg::k_key((uint32_t)row)) * 16;
    auto k_frag = [&](int slot, int b, int ks) { return *reinterpret_cast<const f16x8*>(sK + slot * Cfg::KSLOT + ka[ks] + 32 * b * KRS); };
    // B1, first operand of gemm1: MFMA row r = 8g + 4h' + i holds output column 16h' + 4g + i of the tile (a lane then ends with 16
    // consecutive columns), K-slot 8h + j holds n = 16*ks2 + 8*(j/4) + 4h + j%4 (what a lane holds of the scores). Two transposing reads
    // of four rows each: lane 4e + j of 16 addresses the four columns of MFMA rows 4j .. 4j+3 of row 4h + e (8 further for the second).
    uint32_t va[OT];
#pragma unroll
    for(int t = 0; t < OT; ++t)
    {
        const uint32_t j = lane & 3, e = (lane >> 2) & 3, gg = 2 * ((lane >> 4) & 1) + (j >> 1);
        va[t] = (4 * h + e) * VRS + ((64 * t + 32 * (j & 1) + 8 * gg) ^ (Cfg::v_key(e) << 4));
    }
    auto v_frag = [&](int slot, int ks2, int t) {
        const uint8_t* src = sV + slot * Cfg::VSLOT + va[t] + 16 * ks2 * VRS;
        const i32x2 lo     = __builtin_bit_cast(i32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)src));
        const i32x2 hi     = __builtin_bit_cast(i32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(src + 8 * VRS)));
        return __builtin_bit_cast(f16x8, i32x4{lo[0], lo[1], hi[0], hi[1]});
    };
    // Row sums of exactly the fp16 values that gemm1 multiplies, on the matrix core (a v_dot2_f32_f16 keeps it as busy and costs a vector
    // instruction as well): in a 4x4x4 MFMA with ones for its first operand every lane adds up its own four values, so that nothing of
    // one row, not even a NaN, reaches another.
    typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
    const f16x4 ones = {(_Float16)1.0f, (_Float16)1.0f, (_Float16)1.0f, (_Float16)1.0f};
    auto add_up      = [&](f32x4 c, f16x8 v) {
        c = __builtin_amdgcn_mfma_f32_4x4x4f16(ones, f16x4{v[0], v[1], v[2], v[3]}, c, 0, 0, 0);
        return __builtin_amdgcn_mfma_f32_4x4x4f16(ones, f16x4{v[4], v[5], v[6], v[7]}, c, 0, 0, 0);
    };

    f32x16 acc[OT];
    f32x4 sum = {0, 0, 0, 0};

    // scores are kept as the products come; x = score * |scale| * log2(e) turns exp into one multiply-add and one v_exp_f32
    constexpr float kLog2e = 1.4426950408889634f;
    const float ninf       = -__builtin_inff();
    // (never exactly 0: a masked score is -inf, and -inf * 0 would be a NaN)
    const float c2 = __builtin_fmaxf(__builtin_fabsf(p.scale) * kLog2e, 1.17549435e-38f);
    float m_run = ninf, m_use = 0.0f; // running maximum, and the same with 0 for -inf

    auto max_of = [&](const f32x16(&s)[NB]) {
        float mxa = score_max(s[0][0], s[0][1]), mxb = score_max(s[0][2], s[0][3]);
#pragma unroll
        for(int b = 0; b < NB; ++b)
#pragma unroll
            for(int i = b == 0 ? 4 : 0; i < 16; i += 4)
            {
                mxa = score_max(score_max(mxa, s[b][i]), s[b][i + 1]);
                mxb = score_max(score_max(mxb, s[b][i + 2]), s[b][i + 3]);
            }
        return score_max(mxa, mxb);
    };
    auto exceeded = [&](float mx) { return __builtin_amdgcn_ballot_w64(mx * c2 > m_run) != 0; }; // by some row of the wave
    // moves the running maximum up to that of a row's scores, which two lanes share; the factor for what refers to the old one
    auto raise = [&](float mx) {
        auto sw = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, mx), __builtin_bit_cast(uint32_t, mx), false, false);
        const uint32_t s0 = sw[0], s1 = sw[1];
        const float m_old = m_run;
        m_run             = __builtin_fmaxf(m_old, score_max(__builtin_bit_cast(float, s0), __builtin_bit_cast(float, s1)) * c2);
        m_use             = m_run == ninf ? 0.0f : m_run;
        return __builtin_amdgcn_exp2f(m_old - m_use);
    };
    auto rescale = [&](float corr) {
#pragma unroll
        for(int t = 0; t < OT; ++t)
            acc[t] *= corr;
        sum[0] *= corr; // (the one of its four equal rows that is used)
    };
    auto scores = [&](int slot, f32x16(&s)[NB]) {
#pragma unroll
        for(int ks = 0; ks < KS; ++ks)
#pragma unroll
            for(int b = 0; b < NB; ++b)
                s[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(k_frag(slot, b, ks), af[ks], ks == 0 ? f32x16{} : s[b], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    // (blocks: 32-column blocks that hold an unmasked column of some row of the wave; the others' rows of B1 stay out, whatever they hold)
    auto accumulate = [&](int slot, const f16x8(&pr)[NK2], int blocks) {
#pragma unroll
        for(int k2 = 0; k2 < NK2; ++k2)
        {
            if(k2 / 2 >= blocks)
                break;
#pragma unroll
            for(int t = 0; t < OT; ++t)
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v_frag(slot, k2, t), pr[k2], acc[t], 0, 0, 0);
            if constexpr(SM)
                sum = add_up(sum, pr[k2]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // probabilities, two at a time, in three stages that a step runs for different pairs: s -> x - m -> exp -> fp16
    constexpr int NP = NK2 * 4; // pairs
    auto stage_fma   = [&](f32x16(&s)[NB], int q) {
        const int b = q / 8, i = 2 * (q % 8);
        s[b][i]     = __builtin_fmaf(s[b][i], c2, -m_use);
        s[b][i + 1] = __builtin_fmaf(s[b][i + 1], c2, -m_use);
    };
    auto stage_exp = [&](f32x16(&s)[NB], int q) {
        const int b = q / 8, i = 2 * (q % 8);
        s[b][i]     = __builtin_amdgcn_exp2f(s[b][i]);
        s[b][i + 1] = __builtin_amdgcn_exp2f(s[b][i + 1]);
    };
    auto stage_half = [&](const f32x16(&s)[NB], f16x8(&pr)[NK2], int q) {
        const int b = q / 8, i = 2 * (q % 8);
        pr[q / 4][2 * (q % 4)]     = (_Float16)s[b][i];
        pr[q / 4][2 * (q % 4) + 1] = (_Float16)s[b][i + 1];
    };

    // (what is computed in a unit for the next one stays there: left alone, the compiler moves it to its use)
    auto pin = [&](f16x8(&pr)[NK2]) {
#pragma unroll
        for(int k2 = 0; k2 < NK2; ++k2)
            asm volatile("" : "+v"(pr[k2]));
    };
    auto softmax = [&](f32x16(&s)[NB], f16x8(&pr)[NK2]) {
#pragma unroll
        for(int q = 0; q < NP; ++q)
        {
            if constexpr(SM)
                stage_fma(s, q), stage_exp(s, q);
            stage_half(s, pr, q);
        }
        pin(pr);
    };
    auto mask = [&](int u, f32x16(&s)[NB]) {
        const int n0 = u * UC;
        if(n0 + UC <= full)
            return;
        const int c     = wave_c0 + row;
        const int n_lim = (p.mask_upper && c + 1 < N ? c + 1 : N) - n0 - 4 * h; // columns from here on are masked
#pragma unroll
        for(int b = 0; b < NB; ++b)
#pragma unroll
            for(int i = 0; i < 16; ++i)
                s[b][i] = 32 * b + 8 * (i / 4) + i % 4 < n_lim ? s[b][i] : SM ? ninf : 0.0f;
    };

    // ---- the units ----------------------------------------------------------------------------------------------------------
    // Unit u: B0 of unit u + 1 gives the next scores, the scores of unit u become probabilities, those of unit u - 1 meet their rows of
    // B1. All of it reads the slots (u + 1) & 1; B0 of unit u + 2 and B1 of unit u go into the others meanwhile, out of registers
    // whose loads were issued a unit before. Every wave takes part in units 0 ... units, whatever it has to compute there.
    i32x4 rk[NLK], rv[NLV];
    auto stage = [&](int u, int slot, auto checked) {
        store_k(slot, rk);
        store_v(slot, rv);
        load_k(u + 3, rk, checked);
        load_v(u + 1, rv, checked);
    };
    constexpr std::true_type kChecked{};
    {
        i32x4 k0[NLK], k1[NLK];
        load_k(0, k0, kChecked);
        load_k(1, k1, kChecked);
        const int m        = wave_m0 + row;
        const _Float16* am = A + (int64_t)(m < p.M ? m : p.M - 1) * p.sa;
#pragma unroll
        for(int ks = 0; ks < KS; ++ks)
        {
            const int k = 16 * ks + 8 * h;
            i32x4 v     = {0, 0, 0, 0};
            if(p.K > 0)
                v = *reinterpret_cast<const i32x4*>(am + (k < p.K ? k : 0));
            af[ks] = __builtin_bit_cast(f16x8, v);
        }
        load_v(0, rv, kChecked);
        load_k(2, rk, kChecked);
        store_k(0, k0);
        store_k(1, k1);
#pragma unroll
        for(int ks = 0; ks < KS; ++ks)
        {
            i32x4 v = __builtin_bit_cast(i32x4, af[ks]);
            v       = 16 * ks + 8 * h < p.K ? v : i32x4{0, 0, 0, 0};
            af[ks]  = __builtin_bit_cast(f16x8, SM && p.scale < 0.0f ? v ^ (int)0x80008000 : v); // scale * (A * B0) = |scale| * ((-A) * B0)
        }
    }
    __syncthreads();

    f32x16 sa[NB], sb[NB];
    f16x8 pa[NK2], pb[NK2];
    int u = 0;
    if(w_units > 0)
    {
        scores(0, sa);
        __syncthreads();
        stage(0, 0, kChecked);
        mask(0, sa);
        if constexpr(SM)
            raise(max_of(sa)); // (nothing accumulated yet)
        softmax(sa, pa);
        if(w_units > 1)
            scores(1, sa);
        u = 1;
    }
#pragma unroll
    for(int t = 0; t < OT; ++t)
#pragma unroll
        for(int i = 0; i < 16; ++i)
            acc[t][i] = 0.0f;

    // a unit in the middle of a wave's columns, none of them masked: matrix instructions with other units' vector work between them.
    // Its end finds the maximum of the next scores (mx). Where that raises the running maximum, what has been accumulated is rescaled a
    // unit later, when the unit before has been added too and acc is idle again.
    float mx = 0.0f, corr = 1.0f;
    bool pending = false; // wave-uniform: acc still waits for corr
    auto middle = [&](int u, auto parity, f32x16(&s)[NB], f32x16(&s_next)[NB], f16x8(&pr)[NK2], f16x8(&p_prev)[NK2]) {
        constexpr int W = decltype(parity)::value, R = 1 - W; // slots written and read
        constexpr int OTS = OT + SM, G0 = NB * KS, L = G0 + NK2 * OTS, AHEAD = 4; // (OTS: the row sums have a step of their own)
        f16x8 frag[L];
        auto fetch = [&](auto ic) {
            constexpr int i = decltype(ic)::value;
            if constexpr(i < G0)
                frag[i] = k_frag(R, i % NB, i / NB);
            else if constexpr(i < L && (i - G0) % OTS < OT)
                frag[i] = v_frag(R, (i - G0) / OTS, (i - G0) % OTS);
        };
        __builtin_amdgcn_s_setprio(0);
        __syncthreads();
        static_for<AHEAD>(fetch);
        __builtin_amdgcn_sched_barrier(0);
        // (four units and more here: at least 3 * UC rows, and the offsets of 64 more stay below 2^32)
        stage(u, W, std::false_type{});
        if constexpr(SM)
        {
            if(pending)
                rescale(corr);
            pending = exceeded(mx);
            if(pending)
                corr = raise(mx);
        }
        __builtin_amdgcn_s_setprio(1); // (32 x 2048 x 2048 x 80 61.4 -> 58.8 us, x 128 86.4 -> 82.9, 64 x 4096 x 4096 x 64 346 -> 340)
        auto vector_work = [&](auto ic) {
            constexpr int i = decltype(ic)::value, steps = SM ? NP + 2 : NP, q0 = i * steps / L, q1 = (i + 1) * steps / L;
#pragma unroll
            for(int q = q0; q < q1; ++q)
            {
                if constexpr(!SM)
                {
                    stage_half(s, pr, q);
                    continue;
                }
                if(q >= 2)
                    stage_half(s, pr, q - 2);
                if(q >= 1 && q - 1 < NP)
                    stage_exp(s, q - 1);
                if(q < NP)
                    stage_fma(s, q);
            }
        };
        static_for<G0>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            fetch(std::integral_constant<int, i + AHEAD>{});
            s_next[i % NB] = __builtin_amdgcn_mfma_f32_32x32x16_f16(frag[i], af[i / NB], i < NB ? f32x16{} : s_next[i % NB], 0, 0, 0);
            vector_work(ic);
            __builtin_amdgcn_sched_barrier(0);
        });
        float mxa, mxb;
        static_for<L - G0>([&](auto jc) {
            constexpr int j = decltype(jc)::value, k2 = j / OTS, t = j % OTS;
            fetch(std::integral_constant<int, G0 + j + AHEAD>{});
            if constexpr(t < OT)
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(frag[G0 + j], p_prev[k2], acc[t], 0, 0, 0);
            else
                sum = add_up(sum, p_prev[k2]);
            vector_work(std::integral_constant<int, G0 + j>{});
            // (the next scores are complete: their maximum)
            constexpr int NM = SM ? NB * 16 / 4 : 0, r0 = j * NM / (L - G0), r1 = (j + 1) * NM / (L - G0);
#pragma unroll
            for(int r = r0; r < r1; ++r)
            {
                const f32x16& v = s_next[r / 4];
                const int e     = 4 * (r % 4);
                mxa             = r == 0 ? score_max(v[0], v[1]) : score_max(score_max(mxa, v[e]), v[e + 1]);
                mxb             = r == 0 ? score_max(v[2], v[3]) : score_max(score_max(mxb, v[e + 2]), v[e + 3]);
            }
            if constexpr(r1 > r0)
                asm volatile("" : "+v"(mxa), "+v"(mxb));
            __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr(SM)
            mx = score_max(mxa, mxb);
        pin(pr);
    };
    // (two units at a time, so that scores and probabilities change places without copies; what is left goes step after step)
    if(SM && w_units > 3)
        mx = max_of(sa);
    for(; u + 2 < w_units; u += 2)
    {
        middle(u, std::integral_constant<int, 1>{}, sa, sb, pb, pa);
        middle(u + 1, std::integral_constant<int, 0>{}, sb, sa, pa, pb);
    }
    __builtin_amdgcn_s_setprio(0);
    if(SM && pending)
        rescale(corr);
    for(; u < w_units; ++u)
    {
        __syncthreads();
        stage(u, u & 1, kChecked);
        accumulate((u + 1) & 1, pa, NB);
        mask(u, sa);
        if constexpr(SM)
        {
            const float top = max_of(sa);
            if(exceeded(top))
                rescale(raise(top));
        }
        softmax(sa, pa);
        if(u + 1 < w_units)
            scores((u + 1) & 1, sa);
    }
    if(w_units > 0)
    {
        __syncthreads();
        stage(u, u & 1, kChecked);
        accumulate((u + 1) & 1, pa, (w_end - (u - 1) * UC + 31) >> 5);
        ++u;
    }
    for(; u <= units; ++u)
    {
        __syncthreads();
        stage(u, u & 1, kChecked);
    }

    // ---- C ------------------------------------------------------------------------------------------------------------------
    const int m       = wave_m0 + row;
    auto halves       = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, sum[0]), __builtin_bit_cast(uint32_t, sum[0]), false, false);
    const uint32_t s0 = halves[0], s1 = halves[1];
    float total       = __builtin_bit_cast(float, s0) + __builtin_bit_cast(float, s1);
    if constexpr(NS > 1)
    {
        constexpr int OVER = (16 * OT + 2) * 64; // floats of a wave
        float* const over  = reinterpret_cast<float*>(gg_smem) + wave * OVER + lane;
        __syncthreads();
        if(part)
        {
            float* const to = over + (part - 1) * (NW * OVER);
#pragma unroll
            for(int t = 0; t < OT; ++t)
#pragma unroll
                for(int i = 0; i < 16; ++i)
                    to[(16 * t + i) * 64] = acc[t][i];
            if constexpr(SM)
                to[16 * OT * 64] = m_run, to[(16 * OT + 1) * 64] = total;
        }
        __syncthreads();
        if(part)
            return;
#pragma unroll
        for(int q = 0; q < NS - 1; ++q)
        {
            const float* const from = over + q * (NW * OVER);
            if constexpr(!SM)
            {
#pragma unroll
                for(int t = 0; t < OT; ++t)
#pragma unroll
                    for(int i = 0; i < 16; ++i)
                        acc[t][i] += from[(16 * t + i) * 64];
                continue;
            }
            const float m_other = from[16 * OT * 64], m_both = __builtin_fmaxf(m_run, m_other), m_to = m_both == ninf ? 0.0f : m_both;
            const float mine = __builtin_amdgcn_exp2f(m_run - m_to), other = __builtin_amdgcn_exp2f(m_other - m_to);
            m_run = m_both;
            total = total * mine + from[(16 * OT + 1) * 64] * other;
#pragma unroll
            for(int t = 0; t < OT; ++t)
#pragma unroll
                for(int i = 0; i < 16; ++i)
                    acc[t][i] = acc[t][i] * mine + from[(16 * t + i) * 64] * other;
        }
    }
    const float inv   = total > 0.0f ? 1.0f / total : 0.0f; // N == 0: an empty sum, C = 0
    if(m >= p.M)
        return;
#pragma unroll
    for(int t = 0; t < OT; ++t)
    {
        const int o0 = 32 * t + 16 * h;
        if(o0 >= p.O)
            continue;
        f32x4 v[4];
#pragma unroll
        for(int i = 0; i < 16; ++i)
            v[i / 4][i % 4] = SM ? acc[t][i] * inv : acc[t][i];
        store_row16_f16(C + (int64_t)m * p.sc, o0, p.O, v);
    }
}

// NS parts of the columns, on 4 or (NS = 4) 2 waves of rows each
template <int KS, int OT, int NS, bool SM>
hipError_t gemm_softmax_gemm_launch_one(const GemmGemmArgs& a, hipStream_t s)
{
    constexpr int NW  = NS == 4 ? 2 : 4;
    using Cfg         = SoftmaxGemmCfg<KS, OT, NW>;
    constexpr int LDS = SoftmaxGemmSplit<KS, OT, NW, NS>::LDS;
    auto* kern        = &gemm_softmax_gemm_kernel<KS, OT, NW, NS, SM>;
    if constexpr(LDS > 64 * 1024)
    {
        static std::once_flag once;
        static hipError_t attr_err = hipSuccess;
        std::call_once(once, [&] {
            attr_err = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
        });
        if(attr_err != hipSuccess)
            return attr_err;
    }
    return gemm_gemm_launch_kernel<Cfg::BM, Cfg::NT * NS, LDS>(kern, a, s);
}

} // namespace ckx
