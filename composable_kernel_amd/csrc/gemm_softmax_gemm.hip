// Launcher of the fused GEMM-softmax-GEMM kernels (gemm_softmax_gemm.hpp).
#include "gemm_softmax_gemm.hpp"

namespace ckx {

namespace {

template <int KS, int OT, int NW>
hipError_t launch(const GemmGemmArgs& a, hipStream_t s)
{
    using Cfg = SoftmaxGemmCfg<KS, OT, NW>;
    return gemm_gemm_launch_kernel<Cfg::BM, Cfg::NT, Cfg::LDS>(&gemm_softmax_gemm_kernel<KS, OT, NW>, a, s);
}

template <int KS, int NW>
hipError_t launch_ks(const GemmGemmArgs& a, hipStream_t s)
{
    return a.O <= 32 ? launch<KS, 1, NW>(a, s) : a.O <= 64 ? launch<KS, 2, NW>(a, s) : a.O <= 96 ? launch<KS, 3, NW>(a, s) : launch<KS, 4, NW>(a, s);
}

} // namespace

hipError_t gemm_softmax_gemm_launch(const GemmGemmArgs& a, hipStream_t s)
{
    return a.K <= 32 ? launch_ks<2, 4>(a, s) : a.K <= 64 ? launch_ks<4, 4>(a, s) : a.K <= 80 ? launch_ks<5, 4>(a, s)
         : a.K <= 96 ? launch_ks<6, 4>(a, s) : launch_ks<8, 4>(a, s);
}

} // namespace ckx
