// Tiling and launcher of the few-channel conv kernel (conv_few.hpp): a translation unit of its own so that it compiles beside
// the others.
#include "conv_few.hpp"
#include "tile_launch.hpp"

#include <algorithm>
#include <cmath>
#include <mutex>

namespace ckx {
namespace {

constexpr long kLdsCu = 160 * 1024;
// channel tiles of a block: the fewest that hold K, four (64 channels) from 33 on
int few_nt(int K) { return K <= 16 ? 1 : K <= 32 ? 2 : 4; }
int few_cp(int C) { return C <= 4 ? 4 : 8; }

template <int DT, int CP, int NT>
int lds_bytes(const ConvFewArgs& a)
{
    using T = ConvFew<DT, CP, NT>;
    return T::table_bytes(a.nks) + T::weight_bytes(a.nks, a.kblocks) + (a.patch_pixels * T::PX + 15) / 16 * 16;
}

template <int DT, int CP, int NT>
hipError_t launch_one(const ConvFewArgs& a, hipStream_t s)
{
    using T       = ConvFew<DT, CP, NT>;
    auto* kern    = &conv_few_kernel<DT, CP, NT>;
    const int lds = lds_bytes<DT, CP, NT>(a);
    static std::once_flag once;
    static hipError_t attr_err = hipSuccess;
    std::call_once(once, [&] {
        attr_err = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsCu);
    });
    if(attr_err != hipSuccess)
        return attr_err;
    const int groups = (a.K + T::KB * a.kblocks - 1) / (T::KB * a.kblocks);
    const long slots = std::max(1l, num_cus() * std::min(4l, kLdsCu / lds) / groups);
    hipLaunchKernelGGL(kern, dim3((unsigned)std::min((long)a.units, slots), (unsigned)groups), dim3(256), lds, s, a);
    return hipGetLastError();
}

template <int DT, int CP>
hipError_t launch_nt(const ConvFewArgs& a, hipStream_t s)
{
    const int nt = few_nt(a.K);
    return nt == 1 ? launch_one<DT, CP, 1>(a, s) : nt == 2 ? launch_one<DT, CP, 2>(a, s) : launch_one<DT, CP, 4>(a, s);
}

} // namespace

bool plan_conv_few(int dt, ConvFewArgs& a, int filter_h)
{
    const int es = dt == DT_I8 ? 1 : 2, px = few_cp(a.C) * es, tps = 4 * (16 / px), nt = few_nt(a.K);
    if(a.C < 1 || a.C > 8 || a.C * es >= 16 || a.N < 1 || a.Ho < 1 || a.Wo < 1 || a.K < 1)
        return false;
    a.taps       = filter_h * a.X;
    a.nks        = (a.taps + tps - 1) / tps;
    const long wblock = (long)a.nks * nt * 1024, table = 16 + ((long)a.nks * tps * 4 + 15) / 16 * 16;
    const int blocks  = (a.K + 16 * nt - 1) / (16 * nt);
    // the weights of as many channel blocks as half the LDS holds: the patch is copied once for all of them
    if(wblock + table > kLdsCu / 2)
        return false;
    a.kblocks       = (int)std::min((long)blocks, (kLdsCu / 2 - table) / wblock);
    const int groups = (blocks + a.kblocks - 1) / a.kblocks;
    a.kblocks        = (blocks + groups - 1) / groups;
    const long fixed = table + a.kblocks * wblock;
    // Patch: at most 128 columns and 1024 pixels; of the row counts whose LDS fits the one with the least of (rounds of
    // workgroups) x (work of a round): a copied pixel counts one, an output pixel one per channel block, and a patch 300 for
    // its barriers and the latency of its first loads.
    const int col_blocks = (a.Wo + 127) / 128;
    a.TW                 = (a.Wo + col_blocks - 1) / col_blocks;
    a.col_blocks         = col_blocks;
    a.PC                 = (a.TW - 1) * a.sW + (a.X - 1) * a.dW + 1;
    double best          = -1.0;
    for(int r = 1; r <= a.Ho && (r == 1 || r * a.TW <= 1024); ++r)
    {
        const long rows = (long)(r - 1) * a.sH + (long)(filter_h - 1) * a.dH + 1, pixels = rows * a.PC;
        const long lds  = fixed + (pixels * px + 15) / 16 * 16;
        if(lds > kLdsCu)
            break;
        const long per_cu = std::min(4l, kLdsCu / lds), units = (long)a.N * ((a.Ho + r - 1) / r) * col_blocks;
        const long slots  = std::max(1l, num_cus() * per_cu / groups), rounds = (units + slots - 1) / slots;
        const double cost = (double)rounds * per_cu * (pixels + (double)r * a.TW * a.kblocks + 300.0);
        if(best < 0.0 || cost < best)
        {
            best           = cost;
            a.R            = r;
            a.patch_pixels = (int)pixels;
            a.row_blocks   = (a.Ho + r - 1) / r;
        }
    }
    if(best < 0.0)
        return false;
    const long units = (long)a.N * a.row_blocks * a.col_blocks;
    if(units >= (1l << 31) - 65536)
        return false;
    a.units  = (int)units;
    // Refused where the element-by-element gather (gemm_generic.hpp) is rated faster: few output pixels for many weights to lay out
    // in every workgroup, or a patch of many more pixels than it multiplies (a stride or a dilation past the filter). Both times in
    // us, fitted to 1458 layers (C 1 ... 8, K 1 ... 1000, filters 1 ... 11, strides to 16, dilations to 45, with and without D
    // operands) timed on both kernels, with an rms error of 14 and 22 %. int8 2 x 10^2, C 3 -> K 1000, 3 x 3 stride 8: 27.8 us
    // here, 5.8 gathered; fp16 1 x 78^2, C 2 -> K 64, 3 x 3 dilation 20: 16.5 and 5.4; fp16 52 x 10^2, C 7 -> K 1000, 2 x 2:
    // 38.8 and 13.9. 289 of them were more than 3 % slower here than gathered, at worst 5.3 times; with this line 66 are, at worst
    // 1.6 times, and 5 that are faster here, at worst 1.27 times, are refused.
    const int mt       = nt == 4 ? 2 : 4;
    const long lds     = fixed + ((long)a.patch_pixels * px + 15) / 16 * 16, per_cu = std::min(4l, kLdsCu / lds);
    const long slots   = std::max(1l, num_cus() * per_cu / groups), per_wg = (units + slots - 1) / slots;
    const long rounds  = std::max(1l, (groups + num_cus() * per_cu - 1) / (num_cus() * per_cu));
    const double here  = std::max(1.0, std::min((double)per_cu, (double)(std::min(units, slots) * groups) / num_cus()));
    const int d_ops    = a.epi == EPI_ADD_RELU_ADD ? 2 : a.epi >= EPI_ADD_RELU ? 1 : 0;
    const double lay   = 0.045 * a.nks * a.kblocks * nt * 64 / 256 * (16 / es);
    const long turns   = ((long)a.R * a.TW + 64 * mt - 1) / (64 * mt);
    const double patch = turns * a.kblocks * (0.024 * mt * nt * a.nks + 0.83 + 0.13 * d_ops) + 0.12 * a.patch_pixels / 256;
    const double few_us = 2.5 + rounds * std::pow(here, 2.0 / 3) * (lay + per_wg * patch);
    const double waves  = (double)(((long)a.N * a.Ho * a.Wo + 63) / 64) * ((a.K + 63) / 64) / (2.0 * num_cus());
    const int ksteps    = (int)(((long)a.taps * a.C * es + 63) / 64);
    const double gather_us = 2.3 + (ksteps * (es == 1 ? 2.9 : 1.5) + 0.9 + (d_ops ? 1.2 + 0.4 * d_ops : 0.0)) *
                                       std::max(1.0, waves > 3.0 ? waves : std::ceil(waves));
    return groups <= 65535 && few_us <= 1.3 * gather_us;
}

hipError_t launch_conv_few(int dt, const ConvFewArgs& a, hipStream_t s)
{
    return dt == DT_I8 ? (few_cp(a.C) == 4 ? launch_nt<DT_I8, 4>(a, s) : launch_nt<DT_I8, 8>(a, s))
                       : (few_cp(a.C) == 4 ? launch_nt<DT_F16, 4>(a, s) : launch_nt<DT_F16, 8>(a, s));
}

} // namespace ckx
