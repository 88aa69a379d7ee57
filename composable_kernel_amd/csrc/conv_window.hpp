// Conv forward with the input under a box of output pixels in LDS: 2-D and 3-D, NHWC / NDHWC, unit strides, filters of nine and more taps,
// fp16 and int8, gfx950.
//
// Takes the place of the same reference kernels as the tile kernel's im2col view
// (device_conv2d_fwd_xdl_nhwc_kyxc_nhwk.hpp:57-720, device_convnd_fwd_xdl_nhwc_kyxc_nhwk.hpp:76-1046). There every K tile gathers its
// rows of A anew, so each input pixel crosses a CU's load path once per tap, 27 times for a 3 x 3 x 3 filter, and with few output channels
// that path (75 bytes per ns) is what bounds the launch.
//
//   * A workgroup computes a box of TO x TH x TW output pixels (TO: depth planes, or images in two dimensions) times BN channels. The input
//     pixels under the box (its window, borders as zeros) come into LDS once per channel chunk, by direct loads, and every tap reads its
//     fragments there at the window position of the lane's pixel plus the tap's offset: one addition per fragment.
//   * A chunk is `cu` 16-byte units of a pixel. The window is kept as planes of 32 bytes of every pixel, so that the 16 consecutive pixels
//     and two units that an LDS cycle serves (lanes 0-3, 12-15, 20-23, 24-27 and so on) lie on distinct banks at any tap's offset. Two
//     window buffers: the next chunk's -- of the next tile behind the last one -- is loaded beside the products of this one.
//   * GEMM-K runs over (chunk, tap, unit), 8 units per K tile, without padding: a table in LDS has for each unit its offset in the window and
//     in a weight row. The weights come through a ring of three stages of 128 bytes per channel, as in the tile kernel.
//
// us, tile kernel and this one in turn on one card: 16 x 32^3, C 64 -> K 64 149 -> 117; 18 x 42^3, 160 -> 16 849 -> 529; 7 x 34^3, 112 -> 32 148 -> 105; int8
// 12 x 96^2, 992 -> 24, 3 x 3 148 -> 62; 115 x 32^2, 592 -> 280 with bias, ReLU and residual 603 -> 453; 23 x 110^2, 272 -> 160 399 -> 329.
// What bounds it: of the first one's time a tile's ends take a sixth (every CU stores at once) and loading the windows, which are read in pieces
// of 64 of a line's 128 bytes, a fifth; the K loop keeps the matrix cores 60 % busy, the rest being the barrier and the wait for the
// fragments around only sixteen MFMAs of a wave. With strides it loses to the tile kernel (a window of every second pixel is four times as large: 0.14 to 0.9).
#pragma once

#include "gemm_tile.hpp"

namespace ckx {

struct ConvWindowArgs
{
    const void* in;
    const void* wei;
    void* out;
    const void* d0; // fp16: bias row [K]; int8 with a per-column scale: fp32 [K]
    const void* d1; // fp16: residual, rows of K at stride ldd1
    int ldd1;
    uint32_t in_bytes, wei_bytes;
    int three_d;                       // depth is convolved: the outer extent of a box is depth planes of one image
    int N, Di, Hi, Wi, Do, Ho, Wo, K;  // (two dimensions: Di = Do = 1, and the images are the outer extent)
    int pix_bytes, units;              // bytes and 16-byte units of a pixel
    int Y, X, taps;
    int dD, dH, dW, pF, pT, pL;
    int TO, TH, TW, box;               // output pixels of a tile
    int Wh, pitch, win_px;             // window rows per outer plane, pixels of a row and of the window
    MagicDiv div_thw, div_tw, div_plane, div_row;
    MagicDiv div_chunk, div_cu, div_last, div_yx, div_x; // of the K table: units of a chunk, of a tap in a chunk and in the last one, taps
    int cu, chunks, total;             // units per chunk (even), chunks, units of GEMM-K
    int nk;                            // K tiles
    int spp, wbuf;                     // 1 KB load slots per 32-byte plane of the window, bytes of a window buffer
    int issue;                         // window loads of a wave per K tile, at most four
    int tiles_o, tiles_h, tiles_w, tiles_n, tiles;
    int epi;
    float scale_gemm, scale_relu;
    int nt_store;
};

template <int DT, int WM, int WN, int MT, int NT, int NST>
struct ConvWindow
{
    static_assert((DT == DT_F16 || DT == DT_I8) && (NT == 2 || NT == 4), "fp16 or int8, 32 or 64 columns per wave");
    static constexpr int ES = DT == DT_I8 ? 1 : 2;
    static constexpr int NW = WM * WN, THREADS = NW * 64;
    static constexpr int BM = WM * MT * 16, BN = WN * NT * 16;
    // The first half of the waves loads weights, the second half windows: a wave's loads return in order, and weights, which the next K
    // tiles wait for, would stand behind windows from HBM.
    static constexpr int NWB    = NW / 2;
    static constexpr int BROWS  = BN > NWB * 8 ? BN : NWB * 8; // rows of a B stage: whole loads of every weight wave
    static constexpr int BSTAGE = BROWS * 128;
    static constexpr int NLB    = BROWS / (NWB * 8);
    static constexpr int NLW    = 12; // most load slots of a window wave per plane
    static constexpr int LUT    = DT == DT_I8 ? 256 : 0;
    static constexpr int RUN    = 4 * NT; // consecutive output channels of a lane
    using acc_t = typename std::conditional<DT == DT_I8, i32x4, f32x4>::type;

    // LDS: B stages, two window buffers, table of the K units (whole K tiles), requantisation table
    __host__ __device__ static constexpr int table_bytes(int nk) { return (nk * 32 + 255) / 256 * 256; }
    __host__ __device__ static constexpr int lds_bytes(int nk, int wbuf) { return NST * BSTAGE + 2 * wbuf + table_bytes(nk) + LUT; }

    struct Tile
    {
        int o0, h0, w0, tn;      // first output pixel (outer: image, or depth plane of image n) and column tile
        int first, lo, extent;   // window: outer coordinate of its first plane, and the planes [lo, lo + extent) that exist for it
        int hi0, wi0;            // input row and column of its first pixel
        int n;
    };
    // The launch's arguments read anew where few of them are needed once per tile or chunk: held in scalar registers through the K loop
    // they made it spill sixty of them.
    typedef const __attribute__((address_space(4))) ConvWindowArgs* args_ptr;
    __device__ static __forceinline__ args_ptr args()
    {
        uint64_t a = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(a));
        return (args_ptr)a;
    }
    __device__ static __forceinline__ Tile tile_at(args_ptr p, int bid)
    {
        // ids of one XCD contiguous; the column tiles of a box, which read the same window, next to one another
        const int xcd = bid & 7, local = bid >> 3, q = p->tiles >> 3, r = p->tiles & 7;
        const uint32_t id = (uint32_t)(xcd * q + (xcd < r ? xcd : r) + local);
        const uint32_t tiles_n = (uint32_t)p->tiles_n, tiles_w = (uint32_t)p->tiles_w, tiles_h = (uint32_t)p->tiles_h;
        Tile t;
        const uint32_t s = id / tiles_n, a = s / tiles_w, b = a / tiles_h;
        t.tn = (int)(id - s * tiles_n);
        t.w0 = (int)(s - a * tiles_w) * p->TW;
        t.h0 = (int)(a - b * tiles_h) * p->TH;
        if(p->three_d)
        {
            const uint32_t tiles_o = (uint32_t)p->tiles_o;
            t.n      = (int)(b / tiles_o);
            t.o0     = ((int)b - t.n * (int)tiles_o) * p->TO;
            t.lo     = t.n * p->Di;
            t.first  = t.lo + t.o0 - p->pF;
            t.extent = p->Di;
        }
        else
        {
            t.n      = 0;
            t.o0     = (int)b * p->TO;
            t.lo     = 0;
            t.first  = t.o0;
            t.extent = p->N;
        }
        t.hi0 = t.h0 - p->pT;
        t.wi0 = t.w0 - p->pL;
        return t;
    }

    __device__ static __forceinline__ int lds_read_dword(uint32_t addr)
    {
        int v;
        asm volatile("ds_read_b32 %0, %1" : "=v"(v) : "v"(addr));
        return v;
    }

    __device__ static __forceinline__ void run(const ConvWindowArgs& p, uint8_t* smem)
    {
        const int tid = threadIdx.x, lane = tid & 63;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int wm = wave / WN, wn = wave % WN;
        const uint32_t frow = (uint32_t)(lane & 15), fq = (uint32_t)(lane >> 4);
        const uint32_t smem_lds  = (uint32_t)(uintptr_t)(lds_ptr_t)smem;
        constexpr int WIN0       = NST * BSTAGE;
        const int table_at       = WIN0 + 2 * p.wbuf;
        const uint32_t table_lds = smem_lds + (uint32_t)table_at;
        const int lut_at         = table_at + table_bytes(p.nk);
        const int gstride        = (int)gridDim.x, nk = p.nk;

        const __amdgpu_buffer_rsrc_t rsrc_in  = make_rsrc(p.in, p.in_bytes);
        const __amdgpu_buffer_rsrc_t rsrc_wei = make_rsrc(p.wei, p.wei_bytes);

        // ---- K units: low half offset in the window in units (bit 15: second buffer), high half unit of the weight row
        for(int i = tid; i < p.nk * 8; i += THREADS)
        {
            uint32_t e = 0;
            if(i < p.total)
            {
                const args_ptr q = args();
                auto divide      = [](int n, const __attribute__((address_space(4))) MagicDiv& d) {
                    return (int)((__umulhi((uint32_t)n, d.mul) + (uint32_t)n) >> d.shift);
                };
                int ch        = divide(i, q->div_chunk);
                ch            = ch < q->chunks ? ch : q->chunks - 1;
                const bool last = ch == q->chunks - 1;
                const int w   = last ? q->units - ch * q->cu : q->cu;
                const int r   = i - ch * q->taps * q->cu, tap = last ? divide(r, q->div_last) : divide(r, q->div_cu), c = r - tap * w;
                const int z   = divide(tap, q->div_yx), yx = tap - z * q->Y * q->X, y = divide(yx, q->div_x), x = yx - y * q->X;
                const int px  = (z * q->dD * q->Wh + y * q->dH) * q->pitch + x * q->dW;
                const uint32_t a = (uint32_t)((c >> 1) * q->spp * 64 + 2 * px + (c & 1));
                e              = a | ((uint32_t)(ch & 1) << 15) | ((uint32_t)(tap * q->units + ch * q->cu + c) << 16);
            }
            reinterpret_cast<uint32_t*>(smem + table_at)[i] = e;
        }
        if constexpr(DT == DT_I8)
            if(p.epi == EPI_REQUANT_RND)
                requant_lut_fill(smem + lut_at, p.scale_relu, tid, THREADS);

        // ---- the lane's pixels: position in the window, and (outer, row, column) in the box for the stores
        uint32_t abase[MT], pix[MT];
#pragma unroll
        for(int i = 0; i < MT; ++i)
        {
            const uint32_t m = (uint32_t)(wm * MT * 16 + i * 16) + frow;
            pix[i]           = 0xffffffffu; // (no such pixel: past every limit; its products use pixel 0)
            abase[i]         = smem_lds + (uint32_t)WIN0;
            if(m < (uint32_t)p.box)
            {
                const uint32_t o = magic_div(m, p.div_thw), r = m - o * p.div_thw.d;
                const uint32_t h = magic_div(r, p.div_tw), w = r - h * p.div_tw.d;
                pix[i]           = (o << 20) | (h << 10) | w;
                abase[i] += ((o * (uint32_t)p.Wh + h) * (uint32_t)p.pitch + w) * 32u;
            }
        }

        // ---- window loads. Load slot s of a plane covers 32 of its pixels, a lane 16 bytes of one; window wave w takes the slots w,
        // w + NWB, ... of every plane, so that the lane's offsets hold for all planes and chunks of a tile.
        const bool b_wave = wave < NWB;
        const int w_wave  = wave - NWB;
        uint32_t voffs[NLW];
        auto setup_window = [&](int t_id) {
            const args_ptr q = args();
            const Tile t     = tile_at(q, t_id);
#pragma unroll
            for(int j = 0; j < NLW; ++j)
            {
                voffs[j] = kOutOfRange;
                if(j * NWB < q->spp)
                {
                    const uint32_t px = (uint32_t)((j * NWB + w_wave) * 32 + (lane >> 1));
                    const MagicDiv dp{q->div_plane.mul, q->div_plane.shift, q->div_plane.d}, dr{q->div_row.mul, q->div_row.shift, q->div_row.d};
                    const uint32_t o = magic_div(px, dp), r = px - o * dp.d;
                    const uint32_t y = magic_div(r, dr);
                    const uint32_t x = r - y * dr.d;
                    const int gi = t.first + (int)o, yi = t.hi0 + (int)y, xi = t.wi0 + (int)x;
                    const bool ok = ((uint32_t)(gi - t.lo) < (uint32_t)t.extent) & ((uint32_t)yi < (uint32_t)q->Hi) &
                                    ((uint32_t)xi < (uint32_t)q->Wi) & (px < (uint32_t)q->win_px);
                    voffs[j] = (((uint32_t)((gi * q->Hi + yi) * q->Wi + xi) * (uint32_t)q->pix_bytes + (uint32_t)(lane & 1) * 16u) |
                                     (ok ? 0u : kOutOfRange));
                }
            }
        };
        const int spp           = p.spp;
        const int wave_slots    = b_wave ? 0 : (spp - w_wave + NWB - 1) / NWB;
        const uint32_t odd_unit = (lane & 1) ? kOutOfRange : 0u; // (the second unit of the last plane of a pixel of odd units)
        int w_tile, w_chunk, w_planes, w_buf = 0, w_j, w_pl, w_left;
        auto open_window = [&]() {
            w_planes = (w_chunk == p.chunks - 1 ? p.units - w_chunk * p.cu + 1 : p.cu) >> 1;
            w_j = w_pl = 0;
            w_left     = w_tile < p.tiles ? w_planes * wave_slots : 0;
        };
        auto next_window = [&]() {
            w_buf ^= 1;
            if(++w_chunk == p.chunks)
            {
                w_chunk = 0;
                w_tile += gstride;
                if(w_tile < p.tiles && !b_wave)
                    setup_window(w_tile);
            }
            open_window();
        };
        // (one branch per position of the offset's register: chosen by compares and selects it took fifty instructions a load, which the other
        // waves wait for at the barrier)
        auto load_window = [&]() {
            const int unit   = w_chunk * p.cu + w_pl * 2;
            uint8_t* const to = smem + WIN0 + w_buf * p.wbuf + (w_pl * spp + w_j * NWB + w_wave) * 1024;
            const uint32_t odd = unit + 1 == p.units ? odd_unit : 0u;
            switch(w_j)
            {
#define CKX_WINDOW_SLOT(J) \
    case J: __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_in, (lds_ptr_t)to, 16, voffs[J] | odd, unit * 16, 0, 0); break;
                CKX_WINDOW_SLOT(0) CKX_WINDOW_SLOT(1) CKX_WINDOW_SLOT(2) CKX_WINDOW_SLOT(3) CKX_WINDOW_SLOT(4) CKX_WINDOW_SLOT(5)
                CKX_WINDOW_SLOT(6) CKX_WINDOW_SLOT(7) CKX_WINDOW_SLOT(8) CKX_WINDOW_SLOT(9) CKX_WINDOW_SLOT(10)
            default: __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_in, (lds_ptr_t)to, 16, voffs[11] | odd, unit * 16, 0, 0);
#undef CKX_WINDOW_SLOT
            }
            --w_left;
            if(++w_pl == w_planes)
                w_pl = 0, ++w_j;
        };

        // ---- weight loads
        const uint32_t kpos = ((uint32_t)lane & 7u) ^ (((uint32_t)lane >> 3) & 7u);
        uint32_t b_off[NLB];
        auto setup_b = [&](int tile) {
            const bool live = tile < p.tiles;
            const args_ptr q = args();
            const int n0     = live ? tile_at(q, tile).tn * BN : 0;
#pragma unroll
            for(int j = 0; j < NLB; ++j)
            {
                const uint32_t r = (uint32_t)((j * NWB + wave) * 8 + lane / 8);
                const uint32_t col = NT == 4 ? b_row_to_col(r) : ((r & ~31u) | (((r & 15u) >> 2) << 3) | (((r >> 4) & 1u) << 2) | (r & 3u));
                const uint32_t gn  = (uint32_t)n0 + col;
                b_off[j] = (live && r < (uint32_t)BN && gn < (uint32_t)q->K) ? gn * (uint32_t)(q->taps * q->pix_bytes) : kOutOfRange;
            }
        };
        auto load_b = [&](int j, int stage, uint32_t entry, uint32_t past) {
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_wei, (lds_ptr_t)(smem + stage * BSTAGE + (j * NWB + wave) * 1024), 16,
                                                     (b_off[j] + ((entry >> 16) << 4)) | past, 0, 0, 0);
        };
        auto b_past = [&](int kt) { return kt * 8 + (int)kpos < p.total ? 0u : kOutOfRange; };

        // ---- accumulators and fragments
        acc_t acc[MT][NT];
#pragma unroll
        for(int i = 0; i < MT; ++i)
#pragma unroll
            for(int t = 0; t < NT; ++t)
                acc[i][t] = acc_t{0, 0, 0, 0};
        i32x4 af0[MT], bf0[NT], af1[MT], bf1[NT];
        const uint32_t fb0 = smem_lds + ((uint32_t)(wn * NT * 16) + frow) * 128u + ((fq ^ (frow & 7u)) << 4);
        const uint32_t fb1 = smem_lds + ((uint32_t)(wn * NT * 16) + frow) * 128u + (((4u + fq) ^ (frow & 7u)) << 4);

        auto window_offset = [&](uint32_t entry, int parity) {
            return ((entry & 0x7fffu) << 4) + ((((entry >> 15) ^ (uint32_t)parity) & 1u) ? (uint32_t)p.wbuf : 0u);
        };
        auto wait_frags = [&]() {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
        };
        auto barrier = [&]() {
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        };
        auto read_one = [&](auto r_c, uint32_t bbase, uint32_t aoff, i32x4(&af)[MT], i32x4(&bf)[NT]) {
            constexpr int R = decltype(r_c)::value;
            if constexpr(R < NT)
                bf[R] = lds_read_b128<R * 16 * 128>(bbase);
            else
                af[R - NT] = lds_read_b128<0>(abase[R - NT] + aoff);
        };
        auto mfma_one = [&](int m, const i32x4(&af)[MT], const i32x4(&bf)[NT]) {
            const int i = m / NT, t = (i & 1) ? NT - 1 - m % NT : m % NT;
            if constexpr(DT == DT_I8)
                acc[i][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(bf[t], af[i], acc[i][t], 0, 0, 0);
            else
                acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, bf[t]), __builtin_bit_cast(f16x8, af[i]),
                                                                acc[i][t], 0, 0, 0);
        };
        // MFMAs of one k-step with the reads of the next one between them; `extra(g)` adds the loads of group g
        auto half_step = [&](const i32x4(&caf)[MT], const i32x4(&cbf)[NT], uint32_t bbase, uint32_t aoff, i32x4(&naf)[MT], i32x4(&nbf)[NT],
                             auto extra) {
            constexpr int NGRP = 4, NR = MT + NT, NM = MT * NT, RG = 3;
            static_for<NGRP>([&](auto g_c) {
                constexpr int g = decltype(g_c)::value;
                extra(g_c);
                constexpr int r0 = g * NR / RG, r1 = g < RG ? (g + 1) * NR / RG : r0;
                static_for<(r1 > NR ? NR : r1) - (r0 > NR ? NR : r0)>([&](auto r_c) {
                    read_one(std::integral_constant<int, r0 + decltype(r_c)::value>{}, bbase, aoff, naf, nbf);
                });
#pragma unroll
                for(int m = g * NM / NGRP; m < (g + 1) * NM / NGRP; ++m)
                    mfma_one(m, caf, cbf);
                __builtin_amdgcn_sched_barrier(0);
            });
        };
        // the units past GEMM-K's end: B holds zeros there, and A whatever its entry 0 points at
        auto clear_past = [&](int kt, int ks, i32x4(&af)[MT]) {
            if((kt + 1) * 8 > p.total && kt * 8 + ks * 4 + 4 > p.total)
            {
                const bool live = kt * 8 + ks * 4 + (int)fq < p.total;
#pragma unroll
                for(int i = 0; i < MT; ++i)
#pragma unroll
                    for(int e = 0; e < 4; ++e)
                        af[i][e] = live ? af[i][e] : 0;
            }
        };

        // ---- epilogue
        auto epilogue = [&](int tile) {
            const args_ptr q = args();
            const Tile t     = tile_at(q, tile);
            const bool nt    = q->nt_store != 0;
            const int n0 = t.tn * BN + wn * NT * 16 + RUN * (int)fq;
            const int olimit = (q->three_d ? q->Do : q->N) - t.o0;
            // (D values are awaited right behind their loads, where every lane passes: a load not provably consumed makes the compiler wait for
            // all loads in every K tile)
            float bias[DT == DT_F16 ? RUN : 1];
            float scale[DT == DT_I8 ? RUN : 1];
            if constexpr(DT == DT_F16)
            {
                f16x8 b[RUN / 8];
#pragma unroll
                for(int e = 0; e < RUN / 8; ++e)
                    b[e] = f16x8{0, 0, 0, 0, 0, 0, 0, 0};
                if(q->epi != EPI_PASSTHROUGH)
                {
#pragma unroll
                    for(int e = 0; e < RUN / 8; ++e)
                        b[e] = load_head16<f16x8>(reinterpret_cast<const _Float16*>(q->d0) + n0 + 8 * e, (q->K - n0 - 8 * e) * 2);
                    __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0)
                }
#pragma unroll
                for(int e = 0; e < RUN; ++e)
                    bias[e] = (float)b[e / 8][e % 8];
            }
            else
            {
#pragma unroll
                for(int e = 0; e < RUN; ++e)
                    scale[e] = 0.0f;
                if(epi_per_column_scale(q->epi))
                {
                    const __amdgpu_buffer_rsrc_t rs = make_rsrc(q->d0, (uint32_t)q->K * 4u);
#pragma unroll
                    for(int e = 0; e < RUN; ++e)
                        scale[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, (n0 + e) * 4, 0, 0));
                    __builtin_amdgcn_s_waitcnt(0x0F70);
                }
            }
#pragma unroll
            for(int i = 0; i < MT; ++i)
            {
                const int o = (int)(pix[i] >> 20), h = (int)((pix[i] >> 10) & 1023u), w = (int)(pix[i] & 1023u);
                const bool live = (o < olimit) & (h < q->Ho - t.h0) & (w < q->Wo - t.w0) & (n0 < q->K) & (pix[i] != 0xffffffffu);
                const int row   = ((t.n * q->Do + t.o0 + o) * q->Ho + t.h0 + h) * q->Wo + t.w0 + w;
                const size_t at = (size_t)(uint32_t)row * (uint32_t)q->K + (uint32_t)n0;
                if constexpr(DT == DT_F16)
                {
                    f16x8 d1[RUN / 8];
#pragma unroll
                    for(int e = 0; e < RUN / 8; ++e)
                        d1[e] = f16x8{0, 0, 0, 0, 0, 0, 0, 0};
                    if(q->epi == EPI_ADD_RELU_ADD)
                    {
                        if(live)
                        {
#pragma unroll
                            for(int e = 0; e < RUN / 8; ++e)
                                d1[e] = load_head16<f16x8>(reinterpret_cast<const _Float16*>(q->d1) + (size_t)(uint32_t)row * q->ldd1 + n0 + 8 * e,
                                                           (q->K - n0 - 8 * e) * 2);
                        }
                        __builtin_amdgcn_s_waitcnt(0x0F70);
                    }
                    if(live)
                    {
                        int words[RUN / 2];
#pragma unroll
                        for(int e = 0; e < RUN; e += 2)
                        {
                            _Float16 two[2];
#pragma unroll
                            for(int k = 0; k < 2; ++k)
                            {
                                float v = acc[i][(e + k) / 4][(e + k) % 4];
                                if(q->epi != EPI_PASSTHROUGH)
                                    v = epi_f16_value<false>(q->epi, v, bias[e + k], (float)d1[(e + k) / 8][(e + k) % 8]);
                                two[k] = (_Float16)v;
                            }
                            words[e / 2] = __builtin_bit_cast(int, f16x2{two[0], two[1]});
                        }
                        store_run<2>(reinterpret_cast<uint8_t*>(q->out) + at * 2, words, (q->K - n0) * 2, nt);
                    }
                }
                else
                {
                    int b[RUN];
                    if(q->epi == EPI_REQUANT_RND)
                        requant_lut<NT>(acc[i], q->scale_gemm, smem_lds + (uint32_t)lut_at, b);
                    else
                    {
                        const GemmEpilogue ep{q->epi, q->scale_gemm, q->scale_relu};
                        int8_results(ep, b, [&](int e) { return acc[i][e / 4][e % 4]; }, [&](int e) { return scale[e]; });
                    }
                    if(live)
                    {
                        int words[RUN / 4];
#pragma unroll
                        for(int e = 0; e < RUN / 4; ++e)
                            words[e] = pack4_low_bytes(b[4 * e], b[4 * e + 1], b[4 * e + 2], b[4 * e + 3]);
                        store_run<1>(reinterpret_cast<uint8_t*>(q->out) + at, words, q->K - n0, nt);
                    }
                }
#pragma unroll
                for(int j = 0; j < NT; ++j)
                    acc[i][j] = acc_t{0, 0, 0, 0};
            }
        };

        // ---- prologue: the first chunk's window, then NST K tiles of weights
        int tile = (int)blockIdx.x;
        w_tile = tile, w_chunk = 0;
        if(!b_wave)
            setup_window(tile);
        open_window();
        while(w_left > 0)
            load_window();
        next_window();
        setup_b(tile);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        barrier(); // (the tables are written)
        int btile = tile, bkt = 0;
        auto advance_b = [&]() {
            if(++bkt == nk)
            {
                bkt = 0;
                btile += gstride;
                setup_b(btile);
            }
        };
#pragma unroll
        for(int st = 0; st < NST; ++st)
        {
            const uint32_t e = (uint32_t)lds_read_dword(table_lds + (uint32_t)(bkt * 8) * 4u + kpos * 4u);
            wait_frags();
            const uint32_t past = b_past(bkt);
#pragma unroll
            for(int j = 0; j < NLB; ++j)
                if(b_wave)
                    load_b(j, st, e, past);
            advance_b();
        }
        uint32_t ea = (uint32_t)lds_read_dword(table_lds + fq * 4u);
        uint32_t e1 = (uint32_t)lds_read_dword(table_lds + 16u + fq * 4u);
        if(b_wave)
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((NST - 1) * NLB) : "memory");
        else
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        barrier();
        static_for<MT + NT>([&](auto r_c) { read_one(r_c, fb0, window_offset(ea, 0), af0, bf0); });

        int kt = 0, parity = 0, stage = 0;
        int landed   = 0; // K tiles whose weights are known to have landed although stores are in flight
        const int issue = p.issue;
        // One K tile. EVENT: the next K tile reaches into another chunk's window (lands), and / or this one is the last of its chunk (ends).
        auto k_tile = [&](auto event, int kn, int parity_n, bool lands, bool ends) {
            constexpr bool EVENT = decltype(event)::value;
            const int stage_n    = stage + 1 == NST ? 0 : stage + 1;
            wait_frags();
            if constexpr(EVENT)
                clear_past(kt, 0, af0);
            uint32_t ea_n = 0, e1_n = 0, eb = 0;
            const uint32_t tn_lds = table_lds + (uint32_t)(kn * 32) + fq * 4u;
            half_step(af0, bf0, fb1 + (uint32_t)(stage * BSTAGE), window_offset(e1, parity), af1, bf1, [&](auto g_c) {
                if constexpr(decltype(g_c)::value == 0)
                {
                    ea_n = (uint32_t)lds_read_dword(tn_lds);
                    e1_n = (uint32_t)lds_read_dword(tn_lds + 16u);
                    eb   = (uint32_t)lds_read_dword(table_lds + (uint32_t)(bkt * 32) + kpos * 4u);
                }
            });
            // The next K tile's weights have landed once at most the weight wave's loads for the NST - 2 K tiles behind it are in flight. Where the next K tile reaches into another
            // chunk, that chunk's window as well.
            if constexpr(EVENT)
            {
                if(lands)
                    while(w_left > 0)
                        load_window();
            }
            if(EVENT && lands && !b_wave)
                asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
            else if(b_wave && landed == 0)
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((NST - 2) * NLB) : "memory");
            else
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
            landed -= landed > 0;
            barrier();
            // this K tile is in registers: its stage takes new weights, and a chunk that ends with it gives its window's place to the
            // chunk after the next
            if constexpr(EVENT)
            {
                clear_past(kt, 1, af1);
                if(ends)
                    next_window();
            }
            const uint32_t past = b_past(bkt);
            half_step(af1, bf1, fb0 + (uint32_t)(stage_n * BSTAGE), window_offset(ea_n, parity_n), af0, bf0, [&](auto g_c) {
                constexpr int g = decltype(g_c)::value;
                if(b_wave)
                    static_for<NLB>([&](auto j_c) {
                        if constexpr(decltype(j_c)::value * 4 / NLB == g)
                            load_b(decltype(j_c)::value, stage, eb, past);
                    });
                else if(g < issue && w_left > 0)
                    load_window();
            });
            advance_b();
            e1     = e1_n;
            stage  = stage_n;
            parity = parity_n;
            kt     = kn;
        };
        using std::false_type;
        using std::true_type;
        const int per = p.taps * p.cu, chunks = p.chunks;
        for(;;)
        {
            for(int chunk = 0, from = per; chunk < chunks; ++chunk, from += per)
            {
                const bool last   = chunk == chunks - 1;
                const int last_kt = last ? nk - 1 : (from - 1) >> 3, land = last ? nk - 1 : (from >> 3) - 1;
                while(kt < land)
                    k_tile(false_type{}, kt + 1, parity, false, false);
                // (up to two K tiles: the one before the next chunk's first and, where the chunks meet inside a K tile, that one)
                do
                {
                    const int now = kt, kn = now + 1 == nk ? 0 : now + 1;
                    k_tile(true_type{}, kn, kn == 0 ? parity ^ (chunks & 1) : parity, now == land, now == last_kt);
                    if(now == last_kt)
                        break;
                } while(true);
            }
            // (stores share the loads' counter and are in no order with them: what is on its way lands first, and the next K tiles' waits, whose
            // weights those are, pass the stores by)
            if(b_wave)
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            epilogue(tile);
            landed = NST - 1;
            tile += gstride;
            if(tile >= p.tiles)
                break;
        }
        // the trailing loads still target this workgroup's LDS, and the fragments read ahead are not used
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    }
};

template <int DT, int WM, int WN, int MT, int NT, int NST>
__global__ __launch_bounds__((WM * WN * 64), 2) void conv_window_kernel(const ConvWindowArgs p)
{
    extern __shared__ __attribute__((aligned(1024))) uint8_t ckx_window_smem[];
    ConvWindow<DT, WM, WN, MT, NT, NST>::run(p, ckx_window_smem);
}

// (conv_window.hip) Box and chunks of tile shape `shape` for the layer in `a` (operands, extents, filter, strides, epilogue), and the
// time in us that they are rated at; negative: the shape does not take the layer
constexpr int kConvWindowShapes = 3;
double plan_conv_window(int dt, int shape, ConvWindowArgs& a);
// the fastest shape where it is rated faster than the tile kernel's `tile_us`, its box in `a`; else -1
int choose_conv_window(int dt, ConvWindowArgs& a, double tile_us);
hipError_t launch_conv_window(int dt, int shape, const ConvWindowArgs& a, hipStream_t s);

} // namespace ckx
