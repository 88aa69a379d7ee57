// GEMM on operands that are no whole 16-byte vectors for gfx950: any M, N, K, leading dimension, batch stride and base
// address, all four layouts, every epilogue of the data type. Takes the place of the reference's padded GEMM instances
// (GemmSpecialization::KPadding / MNKPadding, include/ck/tensor_operation/gpu/device/gemm_specialization.hpp:10-20,
// device_gemm_xdl_cshuffle.hpp:99-184).
//
// One workgroup of 4 waves (2 x 2) computes a BM x BN tile of C; a K tile is 128 bytes of every row (two MFMA k-steps). The
// operands come in as 16-byte loads at ANY byte (the part takes them; a load that straddles a cache line costs its second
// line) into registers, two K tiles ahead of the one being multiplied, and go to one of two LDS stages: one barrier per K tile.
// Direct global -> LDS loads would deposit the elements at whatever shift the row has; through registers they land on
// chunk boundaries and the fragment reads are the tile kernel's (gemm_tile.hpp).
//
// Padding is done where it is needed and nowhere else:
//   * rows past M / N repeat the last row (their results are not stored);
//   * the K tile that reaches past K -- at most one -- is multiplied FIRST, out of loads that end at the operand's last
//     element and are shifted down in registers, zeros behind; every other K tile is loaded without a check;
//   * a K-major operand's chunk that reaches past M / N runs into the next k row (its results are not stored); the tile with
//     the last k row, which has no next one, is the checked one there, whether or not K ends in it.
// Operands with less than one vector in the contiguous direction take the checked path element by element.
//
// What bounds it: the operand bytes through a CU's L1. A row that starts anywhere costs the L1 both lines that every 128
// bytes of it touch: 35 to 49 bytes per ns and CU, 77 where rows start on a line (0.27 of the MFMA rate at 4001 x 4003 x
// 4095 fp16). Reading whole lines and moving the chunks into place in registers took more than it saved (25 vector instructions
// per 16 bytes; 2001 x 1003 x 1025 15.7 -> 19.3 us), unaligned LDS writes 50 to 120 cycles each instead of 13, and four K tiles in
// flight instead of two nothing. (Large products with a workspace: gemm_pack.hpp copies the operands to whole lines first.) Against the element-by-element gather
// that served these shapes (one load instruction per element), fp16: 2001 x 1003 x 1025 98.7 -> 15.4 us, 4001 x 4003 x 4095
// 2623 -> 197, 122 x 1283 x 3001 148 -> 17.4, 2049 x 2047 x 2047 with a K-major A 290 -> 55; int8 4001 x 4003 x 4095 3019 -> 118,
// 40 x 333 x 3999 156 -> 16; bf16 3000 x 2999 x 1001 275 -> 47; one tile (32 x 33 x 65) 5.7, as before.
//
// Four tiles, 128 x 128 to 32 x 32: the larger read fewer operand bytes per product, the smaller fewer bytes per workgroup, which
// is what a launch takes that does not fill the CUs; ragged_tile() and ragged_small_tile() say where the lines lie.
#pragma once

#include "gemm_tile.hpp"

namespace ckx {

// 16 bytes moved down by `bytes` (0 and up), zeros from above
__device__ __forceinline__ i32x4 shift_down_bytes(i32x4 v, int bytes)
{
    typedef uint64_t u64x2 __attribute__((ext_vector_type(2)));
    const u64x2 x     = __builtin_bit_cast(u64x2, v);
    const int s       = bytes * 8;
    uint64_t lo = x[0], hi = x[1];
    if(bytes >= 8)
    {
        lo = bytes < 16 ? hi >> ((s - 64) & 63) : 0;
        hi = 0;
    }
    else if(bytes > 0)
    {
        lo = (lo >> s) | (hi << (64 - s));
        hi >>= s;
    }
    return __builtin_bit_cast(i32x4, u64x2{lo, hi});
}

// One operand: BX rows of C (A) or columns of C (B) per tile, K-contiguous or K-major (KM). PERM: the LDS rows of a
// K-contiguous B tile are permuted so that a lane ends up with G / 4 consecutive columns of every G-column group.
template <int ES, int BX, bool KM, int G>
struct RaggedOperand
{
    static constexpr int BKB   = 128, KE = BKB / ES, EPC = 16 / ES;
    static constexpr int NCH   = BX * BKB / 16 / 256; // chunks per thread and K tile
    static constexpr int CPR   = KM ? BX * ES / 16 : BKB / 16;
    static constexpr int BYTES = BX * BKB;
    static constexpr int SEGSH = ES == 2 ? 5 : 4; // log2 bytes of a 16-element segment of a K-major row

    uint32_t off[NCH]; // byte offset of this thread's chunks from the K tile's first byte
    int64_t kstep;     // bytes from one K tile to the next (uniform)

    // swizzle of a K-major tile: see GemmTile::tswz
    __device__ static __forceinline__ uint32_t tswz(uint32_t r)
    {
        constexpr int P     = BX * ES;
        constexpr int LB    = P >= 256 ? 0 : (P == 128 ? 1 : (P == 64 ? 2 : 3));
        const uint32_t full = ES == 2 ? ((r & 3u) | (((r >> 3) & 1u) << 2)) : ((r & 7u) | (((r >> 4) & 1u) << 3));
        return full >> LB;
    }
    // row of C (column for B) that K-contiguous LDS row r holds
    __device__ static __forceinline__ int row_of(int r)
    {
        if constexpr(G == 0)
            return r;
        else
            return (r & ~(G - 1)) | ((r & 15) >> 2) * (G / 4) | (((r & (G - 1)) >> 4) << 2) | (r & 3);
    }

    __device__ __forceinline__ void setup(int tid, int x0, int X, int ld)
    {
        kstep = KM ? (int64_t)KE * ld * ES : (int64_t)BKB;
#pragma unroll
        for(int i = 0; i < NCH; ++i)
        {
            const int idx = tid + 256 * i, r = idx / CPR, c = idx % CPR;
            if constexpr(KM)
            {
                const int x = x0 + c * EPC;
                off[i]      = ((uint32_t)r * (uint32_t)ld + (uint32_t)(x < X ? x : x0)) * ES;
            }
            else
            {
                const int x = x0 + row_of(r);
                off[i]      = (uint32_t)(x < X ? x : X - 1) * (uint32_t)ld * ES + (uint32_t)c * 16u;
            }
        }
    }
    // K tile `kt`, all of it inside the operand
    __device__ __forceinline__ void load(const uint8_t* base, int kt, i32x4 (&v)[NCH]) const
    {
        const uint8_t* src = base + (int64_t)kt * kstep;
#pragma unroll
        for(int i = 0; i < NCH; ++i)
            v[i] = load_vec<i32x4>(src + off[i]);
    }
    // Row and chunk of slot idx of a checked K tile. across: an operand that is read element by element; int8 (16 loads a
    // chunk) then has the rows across the lanes, so that the chunks past K are whole waves', which skip them: 147 x 869 x 15 5.7
    // -> 5.0 us, 3621 x 2 x 7 4.8 -> 4.2. In 16 bits (8 loads) it costs as much as it saves: 20000 x (3 x 5 x 7) 45.0 -> 47.7.
    __device__ static __forceinline__ void slot(int idx, bool across, int& r, int& c)
    {
        across = across && !KM && ES == 1;
        r      = across ? idx % BX : idx / CPR;
        c      = across ? idx / BX : idx % CPR;
    }
    // K tile `kt` with every bound checked; vec: at least one vector in the contiguous direction
    __device__ __forceinline__ void load_checked(const uint8_t* base, int kt, int tid, int x0, int X, int K, int ld, bool vec,
                                                 i32x4 (&v)[NCH]) const
    {
        using elem_t = typename std::conditional<ES == 1, uint8_t, uint16_t>::type;
#pragma unroll
        for(int i = 0; i < NCH; ++i)
        {
            int r, c;
            slot(tid + 256 * i, !vec, r, c);
            // the chunk is elements [e0, e0 + EPC) of a contiguous line of `extent` elements
            const int line   = KM ? kt * KE + r : x0 + row_of(r);
            const int e0     = KM ? x0 + c * EPC : kt * KE + c * EPC;
            const int extent = KM ? X : K;
            const bool live  = line < (KM ? K : X) && e0 < extent;
            const uint8_t* src = base + (int64_t)(live ? line : 0) * ld * ES;
            v[i]               = i32x4{0, 0, 0, 0};
            if(vec)
            {
                const int last = extent - EPC, at = e0 < last ? e0 : last;
                const i32x4 x  = load_vec<i32x4>(src + (int64_t)at * ES);
                v[i]           = live ? shift_down_bytes(x, (e0 - at) * ES) : v[i];
            }
            else if(live)
            {
                elem_t e[EPC];
#pragma unroll
                for(int j = 0; j < EPC; ++j)
                    e[j] = e0 + j < extent ? reinterpret_cast<const elem_t*>(src)[e0 + j] : (elem_t)0;
                __builtin_memcpy(&v[i], e, 16);
            }
        }
    }
    __device__ __forceinline__ void store_lds(uint8_t* s, int tid, const i32x4 (&v)[NCH], bool across = false) const
    {
#pragma unroll
        for(int i = 0; i < NCH; ++i)
        {
            int ri, ci;
            slot(tid + 256 * i, across, ri, ci);
            const uint32_t r = (uint32_t)ri, c = (uint32_t)ci;
            uint32_t at;
            if constexpr(KM)
                at = r * (BX * ES) + ((((c * EPC) >> 4) ^ tswz(r)) << SEGSH) + (ES == 2 ? (c & 1u) << 4 : 0u);
            else
                at = r * BKB + ((c ^ (r & 7u)) << 4);
            *reinterpret_cast<i32x4*>(s + at) = v[i];
        }
    }
    // MFMA fragment `f` (16 rows from wave_x0 + 16 * f) of k-step ks
    __device__ static __forceinline__ i32x4 fragment(const uint8_t* s, int wave_x0, int f, int ks, uint32_t frow, uint32_t fq)
    {
        if constexpr(!KM)
        {
            const uint32_t r = (uint32_t)(wave_x0 + 16 * f) + frow;
            return *reinterpret_cast<const i32x4*>(s + r * BKB + ((((uint32_t)ks * 4 + fq) ^ (frow & 7u)) << 4));
        }
        else
        {
            // (transposing reads: lane 4e + j (b8: 2e + j) points at four (eight) consecutive elements of k row e)
            constexpr int P  = BX * ES, TKS = ES == 2 ? 32 : 64, THALF = ES == 2 ? 4 : 8;
            const uint32_t e = ES == 2 ? frow >> 2 : frow >> 1, j = ES == 2 ? (frow & 3u) : (frow & 1u);
            const uint32_t r = (ES == 2 ? 8u : 16u) * fq + e;
            const uint32_t a = r * P + (((((uint32_t)wave_x0 >> 4) + (uint32_t)f) ^ tswz(r)) << SEGSH) + (j << 3) + (uint32_t)ks * TKS * P;
            // (the swizzle key of row r + THALF and of row r + TKS is that of row r)
            i32x2 lo, hi;
            if constexpr(ES == 2)
            {
                typedef short s16x4 __attribute__((__vector_size__(4 * sizeof(short))));
                typedef __attribute__((address_space(3))) s16x4 lds_t;
                lo = __builtin_bit_cast(i32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_t*)(s + a)));
                hi = __builtin_bit_cast(i32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_t*)(s + a + THALF * P)));
            }
            else
            {
                typedef int s32x2 __attribute__((__vector_size__(2 * sizeof(int))));
                typedef __attribute__((address_space(3))) s32x2 lds_t;
                lo = __builtin_bit_cast(i32x2, __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_t*)(s + a)));
                hi = __builtin_bit_cast(i32x2, __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_t*)(s + a + THALF * P)));
            }
            return i32x4{lo[0], lo[1], hi[0], hi[1]};
        }
    }
};

template <int DT, int BM, int BN, bool TA, bool TB>
__global__ __launch_bounds__(256, 2) void gemm_ragged_kernel(const GemmArgs p)
{
    constexpr int ES = DT == DT_I8 ? 1 : 2, KE = 128 / ES;
    constexpr int WTM = BM / 2, WTN = BN / 2, MT = WTM / 16, NTL = WTN / 16;
    constexpr int G   = TB ? 0 : WTN;           // column group of the permuted B tile: a lane gets G / 4 columns in a row
    constexpr int RUN = TB ? 4 : WTN / 4;       // columns in a row per lane
    constexpr int TPR = RUN / 4;                // MFMA tiles per run
    using OpA   = RaggedOperand<ES, BM, TA, 0>;
    using OpB   = RaggedOperand<ES, BN, TB, G>;
    using acc_t = typename std::conditional<DT == DT_I8, i32x4, f32x4>::type;
    constexpr int STAGE = OpA::BYTES + OpB::BYTES;
    __shared__ __attribute__((aligned(16))) uint8_t smem[2 * STAGE];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const uint32_t frow = lane & 15, fq = lane >> 4;
    int g, tm, tn;
    tile_of_block((int)blockIdx.x, p.tiles_m, p.tiles_n, p.batch > 1 ? p.batch : 1, g, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;
    const uint8_t* A = reinterpret_cast<const uint8_t*>(p.a) + (int64_t)g * p.bsa * ES;
    const uint8_t* B = reinterpret_cast<const uint8_t*>(p.b) + (int64_t)g * p.bsb * ES;

    const bool vec_a = (TA ? p.M : p.K) * ES >= 16, vec_b = (TB ? p.N : p.K) * ES >= 16;
    const int nk     = (p.K + KE - 1) / KE;
    // K tiles loaded without a check (0: all are checked)
    const int nfull  = vec_a && vec_b ? ((TA || TB) ? (p.K > 0 ? (p.K - 1) / KE : 0) : p.K / KE) : 0;

    OpA opa;
    OpB opb;
    opa.setup(tid, m0, p.M, p.lda);
    opb.setup(tid, n0, p.N, p.ldb);

    acc_t acc[MT][NTL];
#pragma unroll
    for(int i = 0; i < MT; ++i)
#pragma unroll
        for(int t = 0; t < NTL; ++t)
            acc[i][t] = acc_t{0, 0, 0, 0};

    auto multiply = [&](const uint8_t* s) {
#pragma unroll
        for(int ks = 0; ks < 2; ++ks)
        {
            i32x4 af[MT], bf[NTL];
#pragma unroll
            for(int t = 0; t < NTL; ++t)
                bf[t] = OpB::fragment(s + OpA::BYTES, wn * WTN, t, ks, frow, fq);
#pragma unroll
            for(int i = 0; i < MT; ++i)
                af[i] = OpA::fragment(s, wm * WTM, i, ks, frow, fq);
#pragma unroll
            for(int i = 0; i < MT; ++i)
#pragma unroll
                for(int t = 0; t < NTL; ++t)
                {
                    if constexpr(DT == DT_I8)
                        acc[i][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(bf[t], af[i], acc[i][t], 0, 0, 0);
                    else if constexpr(DT == DT_BF16)
                        acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, bf[t]),
                                                                         __builtin_bit_cast(bf16x8, af[i]), acc[i][t], 0, 0, 0);
                    else
                        acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, bf[t]),
                                                                        __builtin_bit_cast(f16x8, af[i]), acc[i][t], 0, 0, 0);
                }
        }
    };
    i32x4 ra0[OpA::NCH], rb0[OpB::NCH], ra1[OpA::NCH], rb1[OpB::NCH];
    // registers -> stage, the next load into the freed registers, multiply. One barrier per K tile: a stage is written
    // again only after the barrier of the tile in between, which every wave passes when it is done reading.
    auto step = [&](int stage, i32x4(&ra)[OpA::NCH], i32x4(&rb)[OpB::NCH], int next, bool across_a = false, bool across_b = false) {
        uint8_t* s = smem + stage * STAGE;
        opa.store_lds(s, tid, ra, across_a);
        opb.store_lds(s + OpA::BYTES, tid, rb, across_b);
        if(next >= 0)
        {
            opa.load(A, next, ra);
            opb.load(B, next, rb);
        }
        __syncthreads();
        multiply(s);
    };

    // the checked K tiles: the last one, or all of them; the first unchecked ones are in flight meanwhile
    if(nfull > 0)
    {
        opa.load(A, 0, ra0);
        opb.load(B, 0, rb0);
        const int second = nfull > 1 ? 1 : 0;
        opa.load(A, second, ra1);
        opb.load(B, second, rb1);
    }
    for(int kt = nfull; kt < nk; ++kt)
    {
        i32x4 ra[OpA::NCH], rb[OpB::NCH];
        opa.load_checked(A, kt, tid, m0, p.M, p.K, p.lda, vec_a, ra);
        opb.load_checked(B, kt, tid, n0, p.N, p.K, p.ldb, vec_b, rb);
        step((nk - 1 - kt) & 1 ? 0 : 1, ra, rb, -1, !vec_a, !vec_b); // (stages alternate, the last checked tile in stage 1)
    }
    if(nfull > 0)
    {
        int kt = 0;
        for(; kt + 3 < nfull; kt += 2)
        {
            step(0, ra0, rb0, kt + 2);
            step(1, ra1, rb1, kt + 3);
        }
        // one to three K tiles left
        const int left = nfull - kt;
        if(left == 3)
        {
            step(0, ra0, rb0, kt + 2);
            step(1, ra1, rb1, -1);
            step(0, ra0, rb0, -1);
        }
        else
        {
            step(0, ra0, rb0, -1);
            if(left == 2)
                step(1, ra1, rb1, -1);
        }
    }

    // ---- epilogue: the lane owns row (lane % 16) of every 16-row tile, RUN columns in a row of every run
    const _Float16* d0p = reinterpret_cast<const _Float16*>(p.d0);
    const _Float16* d1p = reinterpret_cast<const _Float16*>(p.d1);
#pragma unroll
    for(int i = 0; i < MT; ++i)
    {
        const int64_t m = (int64_t)m0 + wm * WTM + 16 * i + (int)frow;
        if(m >= p.M)
            continue;
#pragma unroll
        for(int r = 0; r < NTL / TPR; ++r)
        {
            const int n     = n0 + wn * WTN + (TB ? 16 * r + 4 * (int)fq : RUN * (int)fq);
            const int room  = (p.N - n) * ES;
            uint8_t* dst    = reinterpret_cast<uint8_t*>(p.c) + ((int64_t)g * p.bsc + m * p.ldc + n) * ES;
            if(room <= 0)
                continue;
            int w[RUN * ES / 4];
            if constexpr(DT == DT_I8)
            {
                int o[RUN];
                int8_results(GemmEpilogue{p.epi, p.scale_gemm, p.scale_relu}, o,
                             [&](int e) { return acc[i][r * TPR + e / 4][e % 4]; },
                             [&](int e) { return n + e < p.N ? reinterpret_cast<const float*>(p.d0)[n + e] : 0.0f; });
#pragma unroll
                for(int e = 0; e < RUN / 4; ++e)
                    w[e] = pack4_low_bytes(o[4 * e], o[4 * e + 1], o[4 * e + 2], o[4 * e + 3]);
            }
            else
            {
                typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
#pragma unroll
                for(int e = 0; e < RUN; e += 2)
                {
                    float v[2] = {acc[i][r * TPR + e / 4][e % 4], acc[i][r * TPR + e / 4][e % 4 + 1]};
                    if constexpr(DT == DT_BF16)
                        w[e / 2] = __builtin_bit_cast(int, bf16x2{(__bf16)v[0], (__bf16)v[1]});
                    else
                    {
                        if(p.epi != EPI_PASSTHROUGH)
                        {
#pragma unroll
                            for(int h = 0; h < 2; ++h)
                            {
                                const int nn = n + e + h < p.N ? n + e + h : n; // (a column past N is not stored)
                                v[h] = epi_f16_value(p.epi, v[h], (float)d0p[m * p.ldd0 + nn],
                                                     epi_has_d1(p.epi) ? (float)d1p[m * p.ldd1 + nn] : 0.0f, p.scale_gemm,
                                                     p.scale_relu);
                            }
                        }
                        w[e / 2] = __builtin_bit_cast(int, f16x2{(_Float16)v[0], (_Float16)v[1]});
                    }
                }
            }
            store_run<ES>(dst, w, room);
        }
    }
}

// rows and columns of the C tile a problem runs on: 128, or 64 and below (ragged_small_tile)
int ragged_tile(int M, int N, int batch);
struct RaggedTile
{
    int m, n;
};
RaggedTile ragged_small_tile(int M, int N, int batch);
// ta / tb: the operand is K-major. tiles_m / tiles_n are set here.
hipError_t launch_ragged(int dt, bool ta, bool tb, GemmArgs a, hipStream_t s);

} // namespace ckx
