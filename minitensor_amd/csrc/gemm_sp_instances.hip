// gemm_sp_instances.hip -- instantiates gemm_f32_sp for one configuration
// (selected with -DMT_CFG=<n>): the 2x2 contiguous operand layouts, two alike
// also with the row sums of A (not 2, whose operands are off 16-byte alignment:
// their sums are a launch of its own), the forward convolution operands (L_IM and L_IMR:
// configurations 0, 1, 3; L_IM4: 1, 3) and the weight gradient's (L_IMW, with dY copied or
// read in NCHW; not 1 and 2).  Configuration 7: L_IM and
// L_IM4 only.
#include "gemm_configs.hpp"
#include "gemm_sp_kernel.hpp"

#ifndef MT_CFG
#error "build with -DMT_CFG=<configuration index>"
#endif

namespace mtk {
namespace {

template <int LA, int LB, bool RS = false>
hipError_t launch_sp(const GemmParams& p, unsigned nblocks, hipStream_t s) {
    using C = SpCfg<MT_CFG>;
    hipLaunchKernelGGL((gemm_f32_sp<C::BM, C::BNB, C::BN, C::WM, C::WN, LA, LB, C::WPE, RS>),
                       dim3(nblocks), dim3((C::BM / C::WM) * (C::BNB / C::WN) * 64), 0, s, p);
    return hipGetLastError();
}

#if MT_CFG == 7
GemmLaunchFn launcher(int la, int lb, bool rs) {
    if (la == L_KV && lb == L_IM && !rs) return launch_sp<L_KV, L_IM>;
    if (la == L_KV && lb == L_IM4 && !rs) return launch_sp<L_KV, L_IM4>;
    return nullptr;
}
#else
GemmLaunchFn launcher(int la, int lb, bool rs) {
    if (rs) {
#if MT_CFG == 0
        if (la == L_KV && lb == L_IMW) return launch_sp<L_KV, L_IMQ, true>;
        if (la == L_KVI && lb == L_IMW) return launch_sp<L_KVI, L_IMQ, true>;
#endif
#if MT_CFG != 2
        if (la == L_KV && lb == L_KV) return launch_sp<L_KV, L_KV, true>;
        if (la == L_MV && lb == L_MV) return launch_sp<L_MV, L_MV, true>;
#endif
        return nullptr;
    }
    if (la == L_KV && lb == L_KV) return launch_sp<L_KV, L_KV>;
    if (la == L_KV && lb == L_MV) return launch_sp<L_KV, L_MV>;
    if (la == L_MV && lb == L_KV) return launch_sp<L_MV, L_KV>;
    if (la == L_MV && lb == L_MV) return launch_sp<L_MV, L_MV>;
#if MT_CFG == 0 || MT_CFG == 1 || MT_CFG == 3
    if (la == L_KV && lb == L_IM) return launch_sp<L_KV, L_IM>;
#if MT_CFG != 0
    if (la == L_KV && lb == L_IM4) return launch_sp<L_KV, L_IM4>;
#endif
    if (la == L_KV && lb == L_IMR) return launch_sp<L_KV, L_IMR>;
#endif
#if MT_CFG == 0
    if (la == L_KV && lb == L_IMW) return launch_sp<L_KV, L_IMQ>;
    if (la == L_KVI && lb == L_IMW) return launch_sp<L_KVI, L_IMQ>;
#elif MT_CFG != 1 && MT_CFG != 2
    if (la == L_KV && lb == L_IMW) return launch_sp<L_KV, L_IMW>;
    if (la == L_KVI && lb == L_IMW) return launch_sp<L_KVI, L_IMW>;
#endif
    return nullptr;
}
#endif

}  // namespace

#define MT_CAT(a, b) a##b
#define MT_NAME(n) MT_CAT(sp_launcher_cfg, n)
GemmLaunchFn MT_NAME(MT_CFG)(int la, int lb, bool rs) { return launcher(la, lb, rs); }

}  // namespace mtk
