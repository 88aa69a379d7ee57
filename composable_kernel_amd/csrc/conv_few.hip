// Tiling and launcher of the few-channel conv kernel (conv_few.hpp): a translation unit of its own so that it compiles beside
// the others.
#include "conv_few.hpp"
#include "tile_launch.hpp"

#include <algorithm>
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
    return true;
}

hipError_t launch_conv_few(int dt, const ConvFewArgs& a, hipStream_t s)
{
    return dt == DT_I8 ? (few_cp(a.C) == 4 ? launch_nt<DT_I8, 4>(a, s) : launch_nt<DT_I8, 8>(a, s))
                       : (few_cp(a.C) == 4 ? launch_nt<DT_F16, 4>(a, s) : launch_nt<DT_F16, 8>(a, s));
}

} // namespace ckx
