// gemm_configs.hpp -- the tile configurations the dispatcher chooses from and
// the launcher table each instantiation unit (gemm_instances.hip) exports.
#pragma once

#include <hip/hip_runtime.h>

#include "gemm_kernel.hpp"

namespace mtk {

// Block tile BM x BN x BK, wave tile WM x WN.  Threads = (BM/WM)*(BN/WN)*64.
template <int CFG> struct TileCfg;
// 256x128: 8 waves, 2 per SIMD.
template <> struct TileCfg<0> { static constexpr int BM = 256, BN = 128, BK = 16, WM = 64, WN = 64; };
// 128x128: 4 waves; several workgroups share a CU.
template <> struct TileCfg<1> { static constexpr int BM = 128, BN = 128, BK = 16, WM = 64, WN = 64; };
// 64x64: 4 waves of 32x32, for small and skinny problems (usually with split-K).
template <> struct TileCfg<2> { static constexpr int BM = 64, BN = 64, BK = 16, WM = 32, WN = 32; };

constexpr int kNumCfg = 3;
constexpr int kNumLayout = 4;

template <int CFG>
constexpr int cfg_threads() {
    return (TileCfg<CFG>::BM / TileCfg<CFG>::WM) * (TileCfg<CFG>::BN / TileCfg<CFG>::WN) * 64;
}

using GemmLaunchFn = hipError_t (*)(const GemmParams&, unsigned nblocks, hipStream_t);

// Launcher of configuration CFG for (layout of A, layout of B); defined in the
// instantiation unit built with MT_CFG == CFG.
GemmLaunchFn launcher_cfg0(int la, int lb);
GemmLaunchFn launcher_cfg1(int la, int lb);
GemmLaunchFn launcher_cfg2(int la, int lb);

// The bf16-unit kernel gemm_f32_sp (gemm_sp_kernel.hpp): block tile BM x BN
// (on blocks of BNB columns), wave tile WM x WN, WPE: waves per SIMD its
// registers are sized for.  It makes configurations 0, 1, 3, 4, 6 and 7 below
// (same index)
// and, for contiguous operands of any alignment, the register-staged ones (2: 64x64).
template <int CFG> struct SpCfg;
template <> struct SpCfg<0> { static constexpr int BM = 64, BN = 256, BNB = 256, WM = 64, WN = 64, WPE = 2; };
template <> struct SpCfg<1> { static constexpr int BM = 128, BN = 128, BNB = 128, WM = 64, WN = 64, WPE = 2; };
template <> struct SpCfg<2> { static constexpr int BM = 64, BN = 64, BNB = 64, WM = 32, WN = 32, WPE = 4; };
template <> struct SpCfg<3> { static constexpr int BM = 256, BN = 128, BNB = 128, WM = 64, WN = 64, WPE = 2; };
template <> struct SpCfg<4> { static constexpr int BM = 128, BN = 256, BNB = 256, WM = 64, WN = 64, WPE = 2; };
template <> struct SpCfg<6> { static constexpr int BM = 128, BN = 64, BNB = 64, WM = 64, WN = 32, WPE = 3; };
template <> struct SpCfg<7> { static constexpr int BM = 64, BN = 112, BNB = 128, WM = 32, WN = 64, WPE = 3; };
constexpr bool is_sp_cfg(int cfg) {
    return cfg == 0 || cfg == 1 || cfg == 3 || cfg == 4 || cfg == 6 || cfg == 7;
}

// Its launcher for (layout of A: L_KV, L_MV, L_KVI; of B: L_KV, L_MV, L_IM, L_IM4,
// L_IMW, L_IMR), with the row sums of A if rs (two L_KV, two L_MV, or B L_IMW);
// nullptr where the configuration has no such form.
GemmLaunchFn sp_launcher_cfg0(int la, int lb, bool rs);
GemmLaunchFn sp_launcher_cfg1(int la, int lb, bool rs);
GemmLaunchFn sp_launcher_cfg2(int la, int lb, bool rs);
GemmLaunchFn sp_launcher_cfg3(int la, int lb, bool rs);
GemmLaunchFn sp_launcher_cfg4(int la, int lb, bool rs);
GemmLaunchFn sp_launcher_cfg6(int la, int lb, bool rs);
GemmLaunchFn sp_launcher_cfg7(int la, int lb, bool rs);

// Configurations of the direct-to-LDS family, for operands whose layouts are
// both L_KV or L_MV and the implicit convolution operands.
template <int CFG> struct DlCfg;
template <> struct DlCfg<0> : SpCfg<0> {};
template <> struct DlCfg<1> : SpCfg<1> {};
// gemm_f32_dl (gemm_dl_kernel.hpp): STAGES-deep LDS ring of 16-deep K-chunks;
// 4 waves of 32x32; 2 x 8 KB ring, up to eight workgroups per CU.  (Deeper
// rings measured slower for these tiles: occupancy hides more latency.)
template <> struct DlCfg<2> { static constexpr int BM = 64, BN = 64, WM = 32, WN = 32, STAGES = 2; };
template <> struct DlCfg<3> : SpCfg<3> {};
// 4-6: not the implicit im2col operand of the forward convolution.
template <> struct DlCfg<4> : SpCfg<4> {};
// gemm_f32_dlp (gemm_dlp_kernel.hpp), with fragment prefetch: 4 waves of 32x32.
// WPE: waves per SIMD its registers are sized for.
template <> struct DlCfg<5> { static constexpr int BM = 64, BN = 64, WM = 32, WN = 32, STAGES = 2, WPE = 8; };
template <> struct DlCfg<6> : SpCfg<6> {};

// Configuration 1's weight gradient (L_IMW) runs on gemm_f32_dl, whose 16-byte
// gathers take four channels at once: 8 waves of 64x32, 2 x 16 KB ring.
template <int CFG> struct DlwCfg;
template <> struct DlwCfg<1> { static constexpr int BM = 128, BN = 128, WM = 64, WN = 32, STAGES = 2; };

// Wave tiles of the halo-patch kernel gemm_f32_dlh in the tiles of DlCfg 0-3.
template <int CFG> struct DlhCfg;
template <> struct DlhCfg<0> { static constexpr int BM = 64, BN = 256, WM = 64, WN = 64; };
template <> struct DlhCfg<1> { static constexpr int BM = 128, BN = 128, WM = 64, WN = 32; };
template <> struct DlhCfg<2> { static constexpr int BM = 64, BN = 64, WM = 32, WN = 32; };
template <> struct DlhCfg<3> { static constexpr int BM = 256, BN = 128, WM = 64, WN = 64; };

// 7: the channels-last convolution operands only (L_IM, L_IM4), tiles of 112 columns on
// blocks of 128 (4 waves of 32x64).  112 = 7*16 divides the pixel count of
// ResNet layers (multiples of 7*7*16 at even batch sizes), so that such a layer
// has no ragged tile: 28x28 with 128 channels at batch 32 is 448 tiles, two on
// most CUs, where 128 columns give 392.
template <> struct DlCfg<7> : SpCfg<7> {};
constexpr int kNumDlCfg = 8;
constexpr int kNarrowCfg = 7;

constexpr bool is_dlp_cfg(int cfg) { return cfg == 5; }                 // gemm_f32_dlp
constexpr bool is_wide_cfg(int cfg) { return cfg >= 4 && cfg <= 6; }    // no L_IM, L_IMR

// Configuration 2 (gemm_f32_dl); la, lb in {L_KV, L_MV}.
GemmLaunchFn dl_launcher_cfg2(int la, int lb);
// Configuration 5 (gemm_f32_dlp); la, lb in {L_KV, L_MV}; tail: K is not a
// multiple of 16.
GemmLaunchFn dlp_launcher(bool tail, int la, int lb);
// ... with the row sums of A (GemmParams::rowsum); A and B L_MV, or both L_KV.
GemmLaunchFn dlp_rowsum_launcher(bool tail, bool kv);
// ... for the convolution weight gradient (A L_KV, B L_IMW).
GemmLaunchFn dlp_convw_launcher(bool tail);
// ... for the weight gradient with A = dY in NCHW (L_KVI).
GemmLaunchFn dlp_convwi_launcher();
// Implicit-im2col convolution: A = weights (L_KV), B = L_IM (GemmParams::cv).
GemmLaunchFn dl_conv_launcher_cfg2();
// Implicit-im2col convolution from an NCHW view: A = OIHW weights (L_KV), B = L_IMR.
GemmLaunchFn dl_convr_launcher_cfg2();
// The same convolution with B built in LDS from a halo patch (L_IMH,
// gemm_dlh_kernel.hpp) in the tile of configuration cfg (0-3): ConvGeom::hp and
// pw set, LDS per workgroup dlh_lds_floats of the configuration's tile.
GemmLaunchFn dlh_launcher(int cfg);
// Convolution weight gradient: A = dY [c_out][n*h_out*w_out] (L_KV), B = L_IMW.
GemmLaunchFn dl_convw_launcher_cfg2();
// The same with A = dY in NCHW (L_KVI; K a multiple of 16).
GemmLaunchFn dl_convwi_launcher_cfg2();
// Both in configuration 1's tile.
GemmLaunchFn dl_convw_launcher_cfg1();
GemmLaunchFn dl_convwi_launcher_cfg1();
// Two mn-contiguous or two k-contiguous operands, with the row sums of A
// (GemmParams::rowsum).
GemmLaunchFn dl_rowsum_launcher_cfg2(bool kv);

// Wave-split kernel (gemm_ksw_kernel.hpp): tile (R*MB) x (R*NB) of R x R
// MFMA blocks (R = 32: gemm_f32_ksw, R = 16: gemm_f32_ksw16), W waves
// splitting the tile's K range, D chunks in flight per wave.  Any operand
// layout: VA / VB select 16-byte fragment loads for k-contiguous operands
// (L_KV) or scalar ones (every other layout).
template <int CFG> struct KswCfg;
template <> struct KswCfg<0> { static constexpr int R = 32, MB = 1, NB = 1, W = 4, D = 6; };
template <> struct KswCfg<1> { static constexpr int R = 32, MB = 1, NB = 1, W = 8, D = 4; };
template <> struct KswCfg<2> { static constexpr int R = 32, MB = 2, NB = 1, W = 4, D = 4; };
template <> struct KswCfg<3> { static constexpr int R = 32, MB = 1, NB = 2, W = 4, D = 4; };
template <> struct KswCfg<4> { static constexpr int R = 16, MB = 2, NB = 1, W = 4, D = 8; };
template <> struct KswCfg<5> { static constexpr int R = 16, MB = 1, NB = 2, W = 4, D = 8; };
template <> struct KswCfg<6> { static constexpr int R = 16, MB = 2, NB = 1, W = 8, D = 4; };
// 7, 8: the 64x32 and 32x64 tiles again on 16x16 blocks (eight accumulator
// chains per wave where configurations 2 and 3 have two).
template <> struct KswCfg<7> { static constexpr int R = 16, MB = 4, NB = 2, W = 4, D = 4; };
template <> struct KswCfg<8> { static constexpr int R = 16, MB = 2, NB = 4, W = 4, D = 4; };
constexpr int kNumKswCfg = 9;
template <int CFG> struct KswTile {
    static constexpr int bm = KswCfg<CFG>::R * KswCfg<CFG>::MB;
    static constexpr int bn = KswCfg<CFG>::R * KswCfg<CFG>::NB;
};

// Configuration cfg of the wave-split kernel; va / vb: A / B is L_KV.
GemmLaunchFn ksw_launcher(int cfg, bool va, bool vb);
// ... with the row sums of A (GemmParams::rowsum): scalar loads of both operands,
// no split; nullptr for the 32x32-block configurations 0-3.
GemmLaunchFn ksw_rowsum_launcher(int cfg);
void ksw_tile(int cfg, int* bm, int* bn);

// Vector-ALU kernels of the HBM-bound shapes (gemm_skinny_kernel.hpp):
// GEMV for M <= rows <= 8 (B k-contiguous when kv, else mn-contiguous;
// nullptr for more rows), rank-k for 1 <= K <= 16, and the reduction of the
// GEMV kernels' split-K partials (16-byte workspace, grid over groups of
// 16 column quads x M*batch rows).
constexpr int kGemvMaxRows = 8;    // rows of A the GEMV kernels take
constexpr int kRankKMax = 16;      // K the rank-k kernel takes
constexpr int kGemvMvCols = 256;   // columns per GEMV workgroup, B mn-contiguous
constexpr int kGemvKvCols = 16;    // columns per GEMV workgroup, B k-contiguous
constexpr int kRankKCols = 1024;   // columns per rank-k workgroup
constexpr int kRankKRows = 16;     // rows per rank-k workgroup
GemmLaunchFn gemv_launcher(bool kv, int rows);
GemmLaunchFn rankk_launcher(int K);
hipError_t launch_skinny_reduce(const GemmParams& p, hipStream_t s);

}  // namespace mtk
