// Boxes and launcher of the windowed conv kernel (conv_window.hpp): a translation unit of its own so that it compiles beside the others.
#include "conv_window.hpp"
#include "tile_launch.hpp"

#include <algorithm>
#include <mutex>

namespace ckx {
namespace {

constexpr int kLdsCu = 160 * 1024;

struct Shape
{
    int bm, bn, fixed_lds; // output pixels and channels of a tile, LDS without windows and table
    float k_us, tile_us, window_us; // time of a K tile, of a tile's ends, and of 1000 lines of a window
    hipError_t (*launch)(const ConvWindowArgs&, hipStream_t);
};

template <int DT, int WM, int WN, int MT, int NT, int NST>
hipError_t launch_one(const ConvWindowArgs& a, hipStream_t s)
{
    using T       = ConvWindow<DT, WM, WN, MT, NT, NST>;
    auto* kern    = &conv_window_kernel<DT, WM, WN, MT, NT, NST>;
    static std::once_flag once;
    static hipError_t attr_err = hipSuccess;
    std::call_once(once, [&] {
        attr_err = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kLdsCu);
    });
    if(attr_err != hipSuccess)
        return attr_err;
    const int cus = num_cus() - num_cus() % 8;
    hipLaunchKernelGGL(kern, dim3((unsigned)std::min(a.tiles, cus)), dim3(T::THREADS), T::lds_bytes(a.nk, a.wbuf), s, a);
    return hipGetLastError();
}

template <int DT, int WM, int WN, int MT, int NT, int NST>
constexpr Shape shape(float k_us, float tile_us, float window_us)
{
    using T = ConvWindow<DT, WM, WN, MT, NT, NST>;
    return Shape{T::BM, T::BN, T::lds_bytes(0, 0), k_us, tile_us, window_us, &launch_one<DT, WM, WN, MT, NT, NST>};
}
// 512 x 64, 256 x 128 and 512 x 32 pixels x channels. The times are fitted to 117 layers of random sizes (C 16 ... 992, K 16 ... 928, 7^2 ...
// 110^2 and 8^3 ... 45^3 pixels, both data types) timed on each of them, with an rms error of 7 %.
template <int DT>
constexpr Shape kShapes[kConvWindowShapes] = {shape<DT, 8, 1, 4, 4, 3>(0.67f, 5.0f, 1.5f), shape<DT, 4, 2, 4, 4, 3>(0.75f, 4.7f, 1.0f),
                                              shape<DT, 8, 1, 4, 2, 3>(0.50f, 3.8f, 1.55f)};
const Shape& shape_of(int dt, int i) { return dt == DT_I8 ? kShapes<DT_I8>[i] : kShapes<DT_F16>[i]; }

} // namespace

double plan_conv_window(int dt, int shape, ConvWindowArgs& a)
{
    const Shape& sh = shape_of(dt, shape);
    a.total         = a.taps * a.units;
    a.nk            = (a.total + 7) / 8;
    // (nine taps: a 3 x 3 filter is the smallest that this was measured on; entries of the K table have 16 bits for the unit of a weight row; a chunk's K tiles have to outlast the one they share with the next)
    if(a.taps < 9 || a.total >= 65536 || a.nk < 4)
        return -1.0;
    const int fz = a.taps / (a.Y * a.X), outer = a.three_d ? a.Do : a.N, planes = (a.units + 1) / 2;
    const int space = (kLdsCu - sh.fixed_lds - (a.nk * 32 + 255) / 256 * 256) / 2048; // KB of a window buffer
    a.tiles_n       = (a.K + sh.bn - 1) / sh.bn;
    double best     = -1.0;
    // columns of a box: about 8, 16, 24, 32 of them, or whole rows; rows and depth (2-D: whole images) from what is left
    int last_tw = 0;
    for(const int want : {8, 16, 24, 32, 1 << 20})
    {
        const int nw = std::max(1, (a.Wo + want / 2) / want), tw = (a.Wo + nw - 1) / nw;
        if(tw == last_tw || tw > sh.bm || tw > 1023)
            continue;
        last_tw     = tw;
        int last_th = 0;
        for(const int want_h : {4, 8, 16, 1 << 20})
        {
            int th = std::min(a.Ho, sh.bm / tw);
            if(a.three_d)
                th = std::min(th, want_h);
            else if(want_h != 4)
                break;
            const int nh = (a.Ho + th - 1) / th;
            th           = (a.Ho + nh - 1) / nh;
            if(th == last_th)
                continue;
            last_th = th;
            int to  = a.three_d || (tw == a.Wo && th == a.Ho) ? std::min(outer, sh.bm / (tw * th)) : 1;
            const int no = (outer + to - 1) / to;
            to           = (outer + no - 1) / no;
            const int wo = a.three_d ? to + (fz - 1) * a.dD : to, wh = th + (a.Y - 1) * a.dH, ww = tw + (a.X - 1) * a.dW;
            const long px = (long)wo * wh * ww;
            if(px > 32 * 4 * ConvWindow<DT_F16, 8, 1, 4, 4, 3>::NLW)
                continue;
            const int spp = (int)((px + 31) / 32), fit = std::min(space / spp, planes);
            if(fit < 1)
                continue;
            int cp           = (planes + (planes + fit - 1) / fit - 1) / ((planes + fit - 1) / fit);
            if(a.pix_bytes % 128 == 0 && cp < planes) // (whole lines, or a half or a quarter of one)
                cp = fit >= 4 ? fit / 4 * 4 : fit >= 2 ? 2 : 1;
            const int chunks = (planes + cp - 1) / cp;
            const long tiles = (long)nw * nh * no * a.tiles_n * (a.three_d ? a.N : 1);
            if((chunks > 1 && a.taps * cp * 2 < 16) || tiles >= (1l << 31) - 65536)
                continue;
            const long rounds = (tiles + num_cus() - 1) / num_cus();
            // a chunk's window: the 128-byte lines that its pixels' pieces lie in
            const int piece      = 32 * cp;
            const double lines   = a.pix_bytes % 128 == 0 && (128 % piece == 0 || piece % 128 == 0) ? std::max(1, piece / 128) : 1 + (piece - 16) / 128.0;
            const double us      = 2.5 + rounds * (a.nk * sh.k_us + sh.tile_us + chunks * px * lines * sh.window_us * 1e-3);
            if(best >= 0.0 && us >= best)
                continue;
            best = us;
            a.TO = to, a.TH = th, a.TW = tw, a.box = to * th * tw;
            a.Wh = wh, a.pitch = ww, a.win_px = (int)px;
            a.cu = 2 * cp, a.chunks = chunks, a.spp = spp, a.wbuf = cp * spp * 1024;
            a.tiles_o = no, a.tiles_h = nh, a.tiles_w = nw, a.tiles = (int)tiles;
        }
    }
    if(best < 0.0)
        return best;
    a.div_thw = make_magic((uint32_t)(a.TH * a.TW)), a.div_tw = make_magic((uint32_t)a.TW);
    a.div_plane = make_magic((uint32_t)(a.Wh * a.pitch)), a.div_row = make_magic((uint32_t)a.pitch);
    a.div_chunk = make_magic((uint32_t)(a.taps * a.cu)), a.div_cu = make_magic((uint32_t)a.cu);
    a.div_last = make_magic((uint32_t)(a.units - (a.chunks - 1) * a.cu)), a.div_yx = make_magic((uint32_t)(a.Y * a.X));
    a.div_x = make_magic((uint32_t)a.X);
    // a wave's loads of a chunk spread over the K tiles of the one before it but the last two
    const int loads = a.cu / 2 * ((a.spp + 3) / 4), room = std::max(1, std::min(a.taps * a.cu / 8, a.nk) - 2);
    a.issue         = std::min(4, std::max(2, (loads + room - 1) / room));
    return best;
}

int choose_conv_window(int dt, ConvWindowArgs& a, double tile_us)
{
    // Above this the windowed kernel won on 67 of 70 random layers (1.02 to 2.80, 1.34 on average), from 1.0 to 1.15 on half of 27 (0.83 to
    // 1.18), below on none but two (1.07, 1.10). The 14 us spare small calls the search for a box.
    // (Below twelve K tiles a tile's ends outweigh them: 15 x 27^3, C 16 -> K 16, seven of them, 25.3 -> 27.0 us though rated faster. From there to
    // fifteen that is so where a pixel is a single chunk, and the next tile's whole window has to come in behind them: C 32, 14 of them, 25 x 18^3 -> K 16
    // 24.6 -> 26.0 us rated 1.31, 4 x 33^3 -> K 32 26.2 -> 27.4 rated 1.28, 3 x 45^3 -> K 16 level rated 1.29; int8 23 x 35^3, C 64 -> K 16 130.5 -> 109.3 rated 1.39.
    // The third layer that lost: int8 8 x 102^2, C 512 -> K 72, 62.8 -> 68.3, three column tiles that load the window each.)
    constexpr double margin = 1.15, margin_short = 1.35;
    if(tile_us < 14.0 || a.taps * a.units < 12 * 8)
        return -1;
    ConvWindowArgs best = a;
    int shape           = -1;
    for(int i = 0; i < kConvWindowShapes; ++i)
    {
        ConvWindowArgs w = a;
        const double us  = plan_conv_window(dt, i, w);
        const double m  = w.chunks == 1 && w.nk < 16 ? margin_short : margin;
        if(us >= 0.0 && us * m < tile_us)
            best = w, shape = i, tile_us = us * m;
    }
    a = best;
    return shape;
}

hipError_t launch_conv_window(int dt, int shape, const ConvWindowArgs& a, hipStream_t s) { return shape_of(dt, shape).launch(a, s); }

} // namespace ckx
