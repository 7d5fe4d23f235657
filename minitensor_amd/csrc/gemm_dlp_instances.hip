// gemm_dlp_instances.hip -- instantiates gemm_f32_dlp (direct-to-LDS with
// fragment prefetch) for configuration 5, with and without a partial last
// K-chunk, for the 2x2 vector operand layouts, the row-sum forms of two
// mn-contiguous or two k-contiguous operands and the convolution weight
// gradient (A = dY k-contiguous or read in NCHW, B = L_IMW).
#include "gemm_configs.hpp"
#include "gemm_dlp_kernel.hpp"

namespace mtk {
namespace {

template <bool TAIL, int LA, int LB, bool RS = false>
hipError_t launch_dlp(const GemmParams& p, unsigned nblocks, hipStream_t s) {
    using C = DlCfg<5>;
    hipLaunchKernelGGL(
        (gemm_f32_dlp<C::BM, C::BN, C::WM, C::WN, LA, LB, C::STAGES, C::WPE, TAIL, RS>),
        dim3(nblocks), dim3((C::BM / C::WM) * (C::BN / C::WN) * 64), 0, s, p);
    return hipGetLastError();
}

#define MT_DLP_TABLE(TAIL) \
    { { launch_dlp<TAIL, L_KV, L_KV>, launch_dlp<TAIL, L_KV, L_MV> }, \
      { launch_dlp<TAIL, L_MV, L_KV>, launch_dlp<TAIL, L_MV, L_MV> } }

}  // namespace

GemmLaunchFn dlp_convw_launcher(bool tail) {
    return tail ? launch_dlp<true, L_KV, L_IMW> : launch_dlp<false, L_KV, L_IMW>;
}

GemmLaunchFn dlp_convwi_launcher() { return launch_dlp<false, L_KVI, L_IMW>; }

GemmLaunchFn dlp_rowsum_launcher(bool tail, bool kv) {
    static const GemmLaunchFn table[2][2] = {
        {launch_dlp<false, L_MV, L_MV, true>, launch_dlp<true, L_MV, L_MV, true>},
        {launch_dlp<false, L_KV, L_KV, true>, launch_dlp<true, L_KV, L_KV, true>}};
    return table[kv][tail];
}

GemmLaunchFn dlp_launcher(bool tail, int la, int lb) {
    static const GemmLaunchFn table[2][2][2] = {MT_DLP_TABLE(false), MT_DLP_TABLE(true)};
    return table[tail][la][lb];
}

}  // namespace mtk
