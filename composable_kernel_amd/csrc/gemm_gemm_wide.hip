// Launcher of the 32-row kernel (gemm_softmax_gemm.hpp) without its softmax: a translation unit of its own so that it compiles beside the others.
#include "gemm_softmax_gemm.hpp"

namespace ckx {
namespace {

template <int KS, int OT, int NS>
hipError_t launch(const GemmGemmArgs& a, hipStream_t s)
{
    return gemm_softmax_gemm_launch_one<KS, OT, NS, false>(a, s);
}

template <int NS>
hipError_t launch_any(const GemmGemmArgs& a, hipStream_t s)
{
    return a.K <= 32   ? (a.O <= 32 ? launch<2, 1, NS>(a, s) : a.O <= 64 ? launch<2, 2, NS>(a, s) : launch<2, 4, NS>(a, s))
           : a.K <= 64 ? (a.O <= 32 ? launch<4, 1, NS>(a, s) : a.O <= 64 ? launch<4, 2, NS>(a, s) : launch<4, 4, NS>(a, s))
                       : (a.O <= 32 ? launch<8, 1, NS>(a, s) : a.O <= 64 ? launch<8, 2, NS>(a, s) : launch<8, 4, NS>(a, s));
}

} // namespace

hipError_t gemm_gemm_wide_launch(const GemmGemmArgs& a, int parts, hipStream_t s)
{
    return parts == 4 ? launch_any<4>(a, s) : parts == 2 ? launch_any<2>(a, s) : launch_any<1>(a, s);
}

} // namespace ckx
