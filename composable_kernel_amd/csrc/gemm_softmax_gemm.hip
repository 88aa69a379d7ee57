// Launcher of the fused GEMM-softmax-GEMM kernels (gemm_softmax_gemm.hpp).
#include "gemm_softmax_gemm.hpp"

namespace ckx {

namespace {

template <int KS, int OT, int NS>
hipError_t launch(const GemmGemmArgs& a, hipStream_t s)
{
    return gemm_softmax_gemm_launch_one<KS, OT, NS, true>(a, s);
}

template <int KS, int NS>
hipError_t launch_ks(const GemmGemmArgs& a, hipStream_t s)
{
    return a.O <= 32 ? launch<KS, 1, NS>(a, s) : a.O <= 64 ? launch<KS, 2, NS>(a, s) : a.O <= 96 ? launch<KS, 3, NS>(a, s) : launch<KS, 4, NS>(a, s);
}

template <int NS>
hipError_t launch_any(const GemmGemmArgs& a, hipStream_t s)
{
    return a.K <= 32 ? launch_ks<2, NS>(a, s) : a.K <= 64 ? launch_ks<4, NS>(a, s) : a.K <= 80 ? launch_ks<5, NS>(a, s)
         : a.K <= 96 ? launch_ks<6, NS>(a, s) : launch_ks<8, NS>(a, s);
}

} // namespace

hipError_t gemm_softmax_gemm_launch(const GemmGemmArgs& a, int parts, hipStream_t s)
{
    if(parts == 4) // (rows of 192 bytes are not laid out for two waves)
        return a.K <= 32   ? (a.O <= 32 ? launch<2, 1, 4>(a, s) : a.O <= 64 ? launch<2, 2, 4>(a, s) : launch<2, 4, 4>(a, s))
               : a.K <= 64 ? (a.O <= 32 ? launch<4, 1, 4>(a, s) : a.O <= 64 ? launch<4, 2, 4>(a, s) : launch<4, 4, 4>(a, s))
                           : (a.O <= 32 ? launch<8, 1, 4>(a, s) : a.O <= 64 ? launch<8, 2, 4>(a, s) : launch<8, 4, 4>(a, s));
    return parts == 2 ? launch_any<2>(a, s) : launch_any<1>(a, s);
}

} // namespace ckx
