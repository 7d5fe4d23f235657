// gemm_dl_instances.hip -- instantiates gemm_f32_dl for configuration 2 (64x64
// tiles): the 2x2 vector operand layouts (k-contiguous / mn-contiguous for A
// and for B), the implicit-im2col convolution (A k-contiguous weights, B = L_IM
// from a channels-last input or L_IMR from an NCHW view) and its weight gradient
// (A = dY as [c_out][n*h_out*w_out] or read in NCHW, B = L_IMW; configuration
// 1 too), and the
// contiguous pairs with fused row sums of A (the Linear dW GEMM with its bias
// gradient); and the halo-patch convolution kernel gemm_f32_dlh for the tiles
// of configurations 0-3.
#include "gemm_configs.hpp"
#include "gemm_dl_kernel.hpp"
#include "gemm_dlh_kernel.hpp"

namespace mtk {
namespace {

template <int LA, int LB, bool RS = false, class C = DlCfg<2>>
hipError_t launch_dl(const GemmParams& p, unsigned nblocks, hipStream_t s) {
    hipLaunchKernelGGL((gemm_f32_dl<C::BM, C::BN, C::WM, C::WN, LA, LB, C::STAGES, RS>),
                       dim3(nblocks), dim3((C::BM / C::WM) * (C::BN / C::WN) * 64), 0, s, p);
    return hipGetLastError();
}

// The halo-patch kernel's LDS depends on the convolution's geometry.
template <int CFG>
hipError_t launch_dlh(const GemmParams& p, unsigned nblocks, hipStream_t s) {
    using C = DlhCfg<CFG>;
    const size_t bytes = sizeof(float) * dlh_lds_floats<C::BM, C::BN, C::WM, C::WN>(p.cv);
    HaloTable t;
    halo_table(p.cv, C::BN, &t);
    hipLaunchKernelGGL((gemm_f32_dlh<C::BM, C::BN, C::WM, C::WN>), dim3(nblocks),
                       dim3((C::BM / C::WM) * (C::BN / C::WN) * 64), bytes, s, p, t);
    return hipGetLastError();
}

}  // namespace

GemmLaunchFn dl_launcher_cfg2(int la, int lb) {
    static const GemmLaunchFn table[2][2] = {{launch_dl<L_KV, L_KV>, launch_dl<L_KV, L_MV>},
                                             {launch_dl<L_MV, L_KV>, launch_dl<L_MV, L_MV>}};
    return table[la][lb];
}
GemmLaunchFn dl_conv_launcher_cfg2() { return launch_dl<L_KV, L_IM>; }
GemmLaunchFn dl_convr_launcher_cfg2() { return launch_dl<L_KV, L_IMR>; }
GemmLaunchFn dl_convw_launcher_cfg2() { return launch_dl<L_KV, L_IMW>; }
GemmLaunchFn dl_convwi_launcher_cfg2() { return launch_dl<L_KVI, L_IMW>; }
GemmLaunchFn dl_convw_launcher_cfg1() { return launch_dl<L_KV, L_IMW, false, DlwCfg<1>>; }
GemmLaunchFn dl_convwi_launcher_cfg1() { return launch_dl<L_KVI, L_IMW, false, DlwCfg<1>>; }
GemmLaunchFn dl_rowsum_launcher_cfg2(bool kv) {
    return kv ? launch_dl<L_KV, L_KV, true> : launch_dl<L_MV, L_MV, true>;
}
GemmLaunchFn dlh_launcher(int cfg) {
    static const GemmLaunchFn table[4] = {launch_dlh<0>, launch_dlh<1>, launch_dlh<2>,
                                          launch_dlh<3>};
    return cfg >= 0 && cfg <= 3 ? table[cfg] : nullptr;
}

}  // namespace mtk
