// gemm_sp_kernel.hpp -- fp32 GEMM on the bf16 matrix units (gemm_split.hpp),
// staged through registers.
//
//   * K advances in chunks of 16.  Chunk kt+2 is on its way from memory into
//     registers and chunk kt+1, loaded a chunk earlier, is cut into its bf16
//     parts and written to LDS, while chunk kt is multiplied out of LDS; one
//     barrier per chunk.  Each value is cut once per workgroup (6.5 vector
//     instructions; a wave that cut what it reads itself, from an fp32 ring,
//     repeated that for every wave of its row or column and was bound by it:
//     4096^3 took 852 us against 660
//     here).
//   * Wave tiles of 64x64 (32 KB of accumulators with the small products'): per
//     chunk 24 MFMAs, and 12 16-byte fragment reads; two waves per SIMD.
//   * Loads need no alignment beyond the element's: along k a thread takes four
//     consecutive values of one row with one 16-byte load (4-byte aligned),
//     along mn one value of each of four k; the four are cut together and go to
//     LDS as 8 bytes per part.
//   * LDS: per operand and part the two 8-k groups of the chunk, each a column
//     of 16-byte entries, one per row (128 bytes more, so that the groups of a
//     row fall on different banks): a fragment read is 512 contiguous bytes per
//     half wave.
//   * A workgroup whose sums are not finite takes its tile again with fp32
//     MFMAs, from the same loaders.
// Operand forms: L_KV / L_MV (any alignment and, across, any stride), L_IM,
// L_IMW, L_IMR and L_KVI as in gemm_dl_kernel.hpp, and L_IM4 and L_IMQ.
#pragma once

#include <type_traits>

#include "gemm_dl_kernel.hpp"
#include "gemm_split.hpp"

namespace mtk {

typedef f32x4 f32x4_u __attribute__((aligned(4)));   // a 16-byte load at any element

// A global load of a selected address (a select with the zero page makes the
// pointer generic to the compiler, and a flat load waits for LDS too).
template <class T>
__device__ __forceinline__ T sp_global(const float* p) {
    return *(const T __attribute__((address_space(1)))*)p;
}

template <int L>
constexpr bool sp_kc() { return L == L_KV || L == L_KVI || L == L_IM || L == L_IM4; }

// Items of four consecutive k of one row: BMN x 4 per chunk.  k-contiguous
// forms put the four items of a row on consecutive lanes; the others put
// consecutive rows there, and the k of an item is the same across the wave.
template <int L, int BMN, int NT>
struct SpItems {
    static constexpr int NI = BMN * 4 / NT;
    static_assert(NI * NT == BMN * 4 && BMN % 64 == 0, "whole items per thread");
    __device__ __forceinline__ static int row(int i, int t) {
        const int v = i * NT + t;
        return sp_kc<L>() ? v >> 2 : v % BMN;
    }
    __device__ __forceinline__ static int kq(int i, int t) {
        const int v = i * NT + t;
        return sp_kc<L>() ? v & 3 : __builtin_amdgcn_readfirstlane(v / BMN);
    }
    // the row's entry in a group of the LDS tile
    static constexpr int kEntries = BMN + 8;
    __device__ __forceinline__ static int entry(int row) { return row; }
};

// L_IMQ: a thread's four items are the same four k of four consecutive rows.
// Their entries lie in four runs (row % 4), so that consecutive lanes write
// consecutive entries; a run is BMN/4 entries and 64 bytes more, which puts
// the rows of a fragment read on different banks.
template <int BMN, int NT>
struct SpItems<L_IMQ, BMN, NT> {
    static constexpr int NI = 4;
    static_assert(BMN == 256 && NT == 256, "one quad per thread");
    __device__ __forceinline__ static int row(int i, int t) { return (t & 63) * 4 + i; }
    __device__ __forceinline__ static int kq(int, int t) {
        return __builtin_amdgcn_readfirstlane(t >> 6);
    }
    static constexpr int kRun = BMN / 4 + 4;
    static constexpr int kEntries = 4 * kRun + 8;
    __device__ __forceinline__ static int entry(int row) { return (row & 3) * kRun + (row >> 2); }
};

// load(): the items of the next chunk in order (0, 1, 2, ... from the k0 given
// to init), then on to the chunk after it if adv (otherwise the next load
// fetches the same chunk again); PART: a chunk of `left` < 16 k, zero past it.
template <int L, int BMN, int NT> struct SpLoader;

// k-contiguous rows.  Offsets within the tile are 32-bit (the host checks
// BMN rows fit), the chunk's address is uniform.
template <int BMN, int NT>
struct SpLoader<L_KV, BMN, NT> {
    using I = SpItems<L_KV, BMN, NT>;
    const char* base;
    uint32_t off[I::NI];
    int kq;

    __device__ __forceinline__ void init(const GemmParams&, const float* X, int64_t s_mn, int64_t,
                                         int MN, int mn0, int k0, int t) {
        base = reinterpret_cast<const char*>(X + (int64_t)mn0 * s_mn + k0);
        kq = t & 3;
#pragma unroll
        for (int i = 0; i < I::NI; ++i) {
            const int r = min(I::row(i, t), MN - 1 - mn0);
            off[i] = ((uint32_t)r * (uint32_t)s_mn + 4u * kq) * 4u;
        }
    }
    template <bool PART>
    __device__ __forceinline__ void load(f32x4 (&x)[I::NI], int left, bool adv) {
        if constexpr (!PART) {
#pragma unroll
            for (int i = 0; i < I::NI; ++i)
                x[i] = *reinterpret_cast<const f32x4_u*>(base + off[i]);
        } else {
            const int n = left - 4 * kq;
#pragma unroll
            for (int i = 0; i < I::NI; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    x[i][e] = e < n ? *reinterpret_cast<const float*>(base + off[i] + 4 * e) : 0.f;
        }
        base += adv ? 64 : 0;
    }
};

// mn-contiguous: one value of each of four k, consecutive rows on consecutive
// lanes.
template <int BMN, int NT>
struct SpLoader<L_MV, BMN, NT> {
    using I = SpItems<L_MV, BMN, NT>;
    const float* base;   // (k of the chunk, mn0)
    int64_t sk;
    uint32_t off[I::NI];
    int kq[I::NI];

    __device__ __forceinline__ void init(const GemmParams&, const float* X, int64_t, int64_t s_k,
                                         int MN, int mn0, int k0, int t) {
        base = X + (int64_t)k0 * s_k + mn0;
        sk = s_k;
#pragma unroll
        for (int i = 0; i < I::NI; ++i) {
            off[i] = (uint32_t)min(I::row(i, t), MN - 1 - mn0);
            kq[i] = I::kq(i, t);
        }
    }
    template <bool PART>
    __device__ __forceinline__ void load(f32x4 (&x)[I::NI], int left, bool adv) {
        if constexpr (!PART) {
#pragma unroll
            for (int i = 0; i < I::NI; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) x[i][e] = (base + (4 * kq[i] + e) * sk)[off[i]];
        } else {
#pragma unroll
            for (int i = 0; i < I::NI; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int k = 4 * kq[i] + e;   // uniform
                    x[i][e] = k < left ? (base + k * sk)[off[i]] : 0.f;
                }
        }
        base += adv ? 16 * sk : 0;
    }
};

// dY of a convolution as [row][image, position] (GemmParams::a_img, a_hw): an
// item is four positions of one image.
template <int BMN, int NT>
struct SpLoader<L_KVI, BMN, NT> {
    using I = SpItems<L_KVI, BMN, NT>;
    const float* row[I::NI];
    int k, hw;
    double rhw;
    int64_t img;

    __device__ __forceinline__ void init(const GemmParams& p, const float* X, int64_t, int64_t,
                                         int MN, int mn0, int k0, int t) {
        k = k0 + 4 * (t & 3);
        hw = p.a_hw;
        rhw = 1.0 / (double)p.a_hw;
        img = p.a_img;
#pragma unroll
        for (int i = 0; i < I::NI; ++i)
            row[i] = X + (int64_t)min(mn0 + I::row(i, t), MN - 1) * p.a_mn;
    }
    // (K ranges of whole chunks)
    template <bool PART>
    __device__ __forceinline__ void load(f32x4 (&x)[I::NI], int, bool adv) {
        const int im = div_by(k, hw, rhw);
        const int64_t o = (int64_t)im * img + (k - im * hw);
#pragma unroll
        for (int i = 0; i < I::NI; ++i) x[i] = *reinterpret_cast<const f32x4_u*>(row[i] + o);
        k += adv ? 16 : 0;
    }
};

// Implicit im2col of a channels-last input: four channels of one tap at the
// item's output pixel; the tap is the same for the whole chunk (c % 16 == 0).
template <int BMN, int NT>
struct SpLoader<L_IM, BMN, NT> {
    using I = SpItems<L_IM, BMN, NT>;
    const float* pix[I::NI];
    int ih0[I::NI], iw0[I::NI];
    int rt, st, ci0, c, h, w, kw;

    __device__ __forceinline__ void init(const GemmParams& p, const float* X, int64_t, int64_t,
                                         int MN, int mn0, int k0, int t) {
        const ConvGeom& g = p.cv;
        c = g.c; h = g.h; w = g.w; kw = g.kw;
        const int hw = g.ho * g.wo;
#pragma unroll
        for (int i = 0; i < I::NI; ++i) {
            const int n = mn0 + I::row(i, t);
            const int img = n / hw, rem = n - img * hw;
            const int oh = rem / g.wo, ow = rem - oh * g.wo;
            ih0[i] = n < MN ? oh * g.stride - g.pad : -(1 << 30);   // past N: zeros
            iw0[i] = ow * g.stride - g.pad_w;
            pix[i] = X + (int64_t)img * g.img_stride + ((int64_t)ih0[i] * g.w + iw0[i]) * g.c +
                     4 * (t & 3);
        }
        const int tap = k0 / g.c;
        ci0 = k0 - tap * g.c;
        rt = tap / g.kw;
        st = tap - rt * g.kw;
    }
    template <bool PART>
    __device__ __forceinline__ void load(f32x4 (&x)[I::NI], int, bool adv) {
        const int64_t toff = ((int64_t)rt * w + st) * c + ci0;
#pragma unroll
        for (int i = 0; i < I::NI; ++i) {
            const bool ok = (unsigned)(ih0[i] + rt) < (unsigned)h &&
                            (unsigned)(iw0[i] + st) < (unsigned)w;
            const float* src = ok ? pix[i] + toff : dl_zero_page;
            x[i] = sp_global<f32x4>(src);
        }
        ci0 += adv ? 16 : 0;
        if (ci0 == c) {
            ci0 = 0;
            if (++st == kw) { st = 0; ++rt; }
        }
    }
};

// Implicit im2col of an NCHW view in the K order (ci, r, s): an item's lane
// keeps its output pixel, and its four k step through (ci, r, s) in scalar
// registers.
template <int BMN, int NT>
struct SpLoader<L_IMR, BMN, NT> {
    using I = SpItems<L_IMR, BMN, NT>;
    const float* pix[I::NI];
    int ih0[I::NI], iw0[I::NI];
    int kq[I::NI], r[I::NI], s[I::NI];
    int64_t off[I::NI];            // c*sc + r*sh + s*sw of the item's first k
    int kh, kw, h, w, dr, ds;
    int64_t sw, step, carry_s, carry_r;

    __device__ __forceinline__ void init(const GemmParams& p, const float* X, int64_t, int64_t,
                                         int MN, int mn0, int k0, int t) {
        const ConvGeom& g = p.cv;
        kh = g.kh; kw = g.kw; h = g.h; w = g.w;
        sw = g.sw;
        // twelve k (to the next chunk's item) in mixed radix (c, r, s)
        const int khw = kh * kw, dci = 12 / khw;
        dr = (12 - dci * khw) / kw;
        ds = 12 - dci * khw - dr * kw;
        step = dci * g.sc + dr * g.sh + ds * sw;
        carry_s = g.sh - kw * sw;
        carry_r = g.sc - kh * g.sh;
        const int hw = g.ho * g.wo;
#pragma unroll
        for (int i = 0; i < I::NI; ++i) {
            const int row = mn0 + I::row(i, t), n = min(row, MN - 1);
            const int img = n / hw, rem = n - img * hw;
            const int oh = rem / g.wo, ow = rem - oh * g.wo;
            ih0[i] = row < MN ? oh * g.stride - g.pad : -(1 << 29);
            iw0[i] = ow * g.stride - g.pad_w;
            pix[i] = X + (int64_t)img * g.img_stride +
                     (int64_t)(oh * g.stride - g.pad) * g.sh + (int64_t)iw0[i] * sw;
            kq[i] = I::kq(i, t);
            const int k = k0 + 4 * kq[i], c = k / khw, tap = k - c * khw;
            r[i] = tap / kw;
            s[i] = tap - r[i] * kw;
            off[i] = c * g.sc + r[i] * g.sh + s[i] * sw;
        }
    }
    template <bool PART>
    __device__ __forceinline__ void load(f32x4 (&x)[I::NI], int left, bool adv) {
#pragma unroll
        for (int i = 0; i < I::NI; ++i) {
            int rr = r[i], ss = s[i];
            int64_t o = off[i];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const bool ok = (!PART || 4 * kq[i] + e < left) && (unsigned)(ih0[i] + rr) < (unsigned)h &&
                                (unsigned)(iw0[i] + ss) < (unsigned)w;
                const float* src = ok ? pix[i] + o : dl_zero_page;
                x[i][e] = sp_global<float>(src);
                o += sw;
                ++ss;
                carry(rr, ss, o);
            }
            ss += ds;
            rr += dr;
            o += step;
            carry(rr, ss, o);
            r[i] = adv ? rr : r[i];
            s[i] = adv ? ss : s[i];
            off[i] = adv ? o : off[i];
        }
    }
    __device__ __forceinline__ void carry(int& rr, int& ss, int64_t& o) const {
        const bool a = ss >= kw;
        ss -= a ? kw : 0;
        rr += a;
        o += a ? carry_s : 0;
        const bool b = rr >= kh;
        rr -= b ? kh : 0;
        o += b ? carry_r : 0;
    }
};

// The window origins of consecutive output pixels (img, oh, ow) of a
// channels-last input, in scalar registers, by additions alone.
struct SpPixels {
    int st, ih0, iw0, ih1, iw1;    // first and one-past-last origins
    int dy, dq;                    // 12 pixels in mixed radix (img, oh, ow), scaled
    int64_t pix_step, row_step, img_step, step12;
    struct At {
        int y, q;                  // the origin, and its address (which may lie in
        const float* org;          // the padding)
    };

    __device__ __forceinline__ void init(const ConvGeom& g) {
        st = g.stride;
        ih0 = -g.pad; iw0 = -g.pad_w;
        ih1 = g.ho * st - g.pad; iw1 = g.wo * st - g.pad_w;
        const int64_t pitch = (int64_t)st * g.w * g.c;
        pix_step = (int64_t)st * g.c;
        row_step = pitch - g.wo * pix_step;
        img_step = g.img_stride - g.ho * pitch;
        const int hw = g.ho * g.wo, img = 12 / hw, rem = 12 - img * hw, oh = rem / g.wo;
        dy = oh * st;
        dq = (rem - oh * g.wo) * st;
        step12 = img * g.img_stride + oh * pitch + (rem - oh * g.wo) * pix_step;
    }
    __device__ __forceinline__ At at(const ConvGeom& g, const float* X, int k) const {
        const int hw = g.ho * g.wo, img = k / hw, rem = k - img * hw;
        const int oh = rem / g.wo, ow = rem - oh * g.wo;
        const int y = oh * st - g.pad, q = ow * st - g.pad_w;
        return {y, q, X + (int64_t)img * g.img_stride + ((int64_t)y * g.w + q) * g.c};
    }
    __device__ __forceinline__ void carry(At& a) const {
        const bool r = a.q >= iw1;
        a.q -= r ? iw1 - iw0 : 0;
        a.y += r ? st : 0;
        a.org += r ? row_step : 0;
        const bool i = a.y >= ih1;
        a.y -= i ? ih1 - ih0 : 0;
        a.org += i ? img_step : 0;
    }
    __device__ __forceinline__ void next(At& a) const {
        a.q += st;
        a.org += pix_step;
        carry(a);
    }
    __device__ __forceinline__ void next12(At& a) const {
        a.q += dq;
        a.y += dy;
        a.org += step12;
        carry(a);
    }
};

// Implicit im2colᵀ of a channels-last input (the weight gradient): a lane
// keeps its column (tap, channel); the output pixels of its item's four k are
// scalar.
template <int BMN, int NT>
struct SpLoader<L_IMW, BMN, NT> {
    using I = SpItems<L_IMW, BMN, NT>;
    uint32_t off[I::NI];           // (r*w + s)*c + ci of the lane's column
    int r[I::NI], s[I::NI];        // its tap (r: far out for a column past N)
    int kq[I::NI], h, w;
    SpPixels px;
    SpPixels::At at[I::NI];        // the pixel of the item's first k

    __device__ __forceinline__ void init(const GemmParams& p, const float* X, int64_t, int64_t,
                                         int MN, int mn0, int k0, int t) {
        const ConvGeom& g = p.cv;
        h = g.h; w = g.w;
        px.init(g);
#pragma unroll
        for (int i = 0; i < I::NI; ++i) {
            const int row = mn0 + I::row(i, t), n = min(row, MN - 1);
            const int tap = n / g.c, ci = n - tap * g.c;
            const int rr = tap / g.kw;
            s[i] = tap - rr * g.kw;
            r[i] = row < MN ? rr : -(1 << 29);
            off[i] = (uint32_t)((rr * g.w + s[i]) * g.c + ci);
            kq[i] = I::kq(i, t);
            at[i] = px.at(g, X, k0 + 4 * kq[i]);
        }
    }
    template <bool PART>
    __device__ __forceinline__ void load(f32x4 (&x)[I::NI], int left, bool adv) {
#pragma unroll
        for (int i = 0; i < I::NI; ++i) {
            SpPixels::At a = at[i];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const bool ok = (!PART || 4 * kq[i] + e < left) &&
                                (unsigned)(a.y + r[i]) < (unsigned)h &&
                                (unsigned)(a.q + s[i]) < (unsigned)w;
                const float* src = ok ? a.org + off[i] : dl_zero_page;
                x[i][e] = sp_global<float>(src);
                px.next(a);
            }
            px.next12(a);
            at[i].y = adv ? a.y : at[i].y;
            at[i].q = adv ? a.q : at[i].q;
            at[i].org = adv ? a.org : at[i].org;
        }
    }
};

// L_IMW with four consecutive channels of one tap per load: the four k of a
// thread's quad of columns are four 16-byte loads, and change places in
// registers.
template <int BMN, int NT>
struct SpLoader<L_IMQ, BMN, NT> {
    using I = SpItems<L_IMQ, BMN, NT>;
    uint32_t off;                  // (r*w + s)*c + ci of the quad
    int r, s;                      // its tap (r: far out for columns past N)
    int kq, h, w;
    SpPixels px;
    SpPixels::At at;               // the pixel of the first k

    __device__ __forceinline__ void init(const GemmParams& p, const float* X, int64_t, int64_t,
                                         int MN, int mn0, int k0, int t) {
        const ConvGeom& g = p.cv;
        h = g.h; w = g.w;
        px.init(g);
        const int row = mn0 + I::row(0, t), n = min(row, MN - 4);   // MN % 4 == 0
        const int tap = n / g.c, ci = n - tap * g.c, rr = tap / g.kw;
        s = tap - rr * g.kw;
        r = row < MN ? rr : -(1 << 29);
        off = (uint32_t)((rr * g.w + s) * g.c + ci);
        kq = I::kq(0, t);
        at = px.at(g, X, k0 + 4 * kq);
    }
    template <bool PART>
    __device__ __forceinline__ void load(f32x4 (&x)[I::NI], int left, bool adv) {
        SpPixels::At a = at;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const bool ok = (!PART || 4 * kq + e < left) && (unsigned)(a.y + r) < (unsigned)h &&
                            (unsigned)(a.q + s) < (unsigned)w;
            const f32x4 v = sp_global<f32x4>(ok ? a.org + off : dl_zero_page);
#pragma unroll
            for (int j = 0; j < 4; ++j) x[j][e] = v[j];
            px.next(a);
        }
        px.next12(a);
        at.y = adv ? a.y : at.y;
        at.q = adv ? a.q : at.q;
        at.org = adv ? a.org : at.org;
    }
};

// L_IM for any c % 4 == 0: the tap and channel of a thread's items are its own
// (an item of each chunk: the k of its lane's group).
template <int BMN, int NT>
struct SpLoader<L_IM4, BMN, NT> {
    using I = SpItems<L_IM4, BMN, NT>;
    const float* pix[I::NI];
    int ih0[I::NI], iw0[I::NI];
    int rt, st, ci, kq;
    int c, h, w, kw, dr, ds, dc;   // 16 k in mixed radix (r, s, ci)

    __device__ __forceinline__ void init(const GemmParams& p, const float* X, int64_t, int64_t,
                                         int MN, int mn0, int k0, int t) {
        const ConvGeom& g = p.cv;
        c = g.c; h = g.h; w = g.w; kw = g.kw;
        const int hw = g.ho * g.wo;
#pragma unroll
        for (int i = 0; i < I::NI; ++i) {
            const int n = mn0 + I::row(i, t);
            const int img = n / hw, rem = n - img * hw;
            const int oh = rem / g.wo, ow = rem - oh * g.wo;
            ih0[i] = n < MN ? oh * g.stride - g.pad : -(1 << 30);   // past N: zeros
            iw0[i] = ow * g.stride - g.pad_w;
            pix[i] = X + (int64_t)img * g.img_stride + ((int64_t)ih0[i] * g.w + iw0[i]) * g.c;
        }
        kq = t & 3;
        const int k = k0 + 4 * kq, tap = k / c, dtap = 16 / c;
        ci = k - tap * c;
        rt = tap / kw;
        st = tap - rt * kw;
        dc = 16 - dtap * c;
        dr = dtap / kw;
        ds = dtap - dr * kw;
    }
    template <bool PART>
    __device__ __forceinline__ void load(f32x4 (&x)[I::NI], int left, bool adv) {
        const int toff = (rt * w + st) * c + ci;
#pragma unroll
        for (int i = 0; i < I::NI; ++i) {
            const bool ok = (!PART || 4 * kq < left) && (unsigned)(ih0[i] + rt) < (unsigned)h &&
                            (unsigned)(iw0[i] + st) < (unsigned)w;
            const float* src = ok ? pix[i] + toff : dl_zero_page;
            x[i] = sp_global<f32x4>(src);
        }
        ci += adv ? dc : 0;
        const bool cc = ci >= c;
        ci -= cc ? c : 0;
        st += adv ? ds + cc : 0;
        const bool cs = st >= kw;
        st -= cs ? kw : 0;
        rt += adv ? dr + cs : 0;
    }
};

// LDS of one operand's chunk: three parts of two 8-k groups of 16-byte
// entries, in bytes.
template <class I>
constexpr int sp_group() { return I::kEntries * 16; }
template <class I>
constexpr int sp_plane() { return 2 * sp_group<I>(); }

template <class I>
__device__ __forceinline__ void sp_frag(const char* lds, int row, int half, SplitFrag& f) {
    const char* p = lds + half * sp_group<I>() + I::entry(row) * 16;
    f.h = *reinterpret_cast<const u32x4*>(p);
    f.m = *reinterpret_cast<const u32x4*>(p + sp_plane<I>());
    f.l = *reinterpret_cast<const u32x4*>(p + 2 * sp_plane<I>());
}

// A barrier that orders LDS alone: global loads stay in flight across it.
__device__ __forceinline__ void sp_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// BN: columns of the tile's blocks; BNT <= BN: columns of the tile.
// RS: also the row sums of A (GemmParams::rowsum).
template <int BM, int BN, int BNT, int WM, int WN, int LA, int LB, int WPE, bool RS = false>
__global__ void __launch_bounds__((BM / WM) * (BN / WN) * 64, WPE)
gemm_f32_sp(GemmParams p) {
    constexpr int WAVES_N = BN / WN;
    constexpr int NW = (BM / WM) * WAVES_N;
    constexpr int NT = NW * 64;
    constexpr int MB = WM / 32, NB = WN / 32;
    using IA = SpItems<LA, BM, NT>;
    using IB = SpItems<LB, BN, NT>;
    constexpr int BUF = 3 * (sp_plane<IA>() + sp_plane<IB>());
    __shared__ __attribute__((aligned(1024))) char smem[2 * BUF];

    const int t = threadIdx.x;
    const int lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int ra = (wave / WAVES_N) * WM, rb = (wave % WAVES_N) * WN;
    const int half = lane >> 5, lrow = lane & 31;

    const TileId id = tile_id(p);
    const int m0 = id.tm * BM, n0 = id.tn * BNT;
    const int n_end = min(p.N, n0 + BNT);
    const int k_begin = id.split * p.k_per_split;
    const int k_end = min(p.K, k_begin + p.k_per_split);
    const int klen = max(k_end - k_begin, 0);
    const int whole = klen >> 4, part = klen & 15;   // whole chunks, k of a partial one
    const int nk = whole + (part != 0);
    const float* Ab = p.A + (int64_t)id.bz * p.a_b;
    const float* Bb = p.B + (int64_t)id.bz * p.b_b;

    f32x16 acc[MB][NB];
    // Row sums: every thread adds up the items of A that it loads; those of a
    // row meet after the loop, in a fixed order.  Those of a weight gradient's dY
    // would be one chain per thread, where a launch of their own
    // (block_channel_sum) has eight: every two chunks the sum goes to rtot, and
    // what that addition rounds off (but for an early rtot below rsum) starts the
    // next sum (Kahan).  Error against 64 bits of normal values, plain / so / the
    // launch of their own: 32 x 12544 in 512 splits 1.58e-7 / 1.04e-7 / 1.16e-7,
    // 32 x 196 in 8 1.55e-7 / 0.81e-7 / 0.97e-7; 8 x 784 in 2 0.73e-7 / 0.99e-7.
    // Its three additions beside the MFMAs cost at most 1 % of a dW (Knuth's
    // two-sum between the steps had cost 1-5).
    constexpr bool kFold = RS && LB == L_IMQ;
    float rsum[IA::NI], rtot[kFold ? IA::NI : 1];
    SpLoader<LA, BM, NT> la;
    SpLoader<LB, BN, NT> lb;
    auto seek = [&](int k) {
        la.init(p, Ab, p.a_mn, p.a_k, p.M, m0, k, t);
        lb.init(p, Bb, p.b_mn, p.b_k, n_end, n0, k, t);
    };
    auto start = [&] {
        zero_blocks<MB, NB>(acc);
#pragma unroll
        for (int i = 0; i < IA::NI; ++i) rsum[i] = 0.f;
#pragma unroll
        for (float& r : rtot) r = 0.f;
    };
    auto add_rows = [&](const f32x4 (&xa)[IA::NI]) {
        if constexpr (RS)
#pragma unroll
            for (int i = 0; i < IA::NI; ++i)
                rsum[i] += (xa[i][0] + xa[i][1]) + (xa[i][2] + xa[i][3]);
    };
    auto fold_rows = [&] {
        if constexpr (kFold)
#pragma unroll
            for (int i = 0; i < IA::NI; ++i) {
                const float s = rtot[i] + rsum[i];
                rsum[i] -= s - rtot[i];
                rtot[i] = s;
            }
    };

    __shared__ int bad;
    if (t == 0) bad = 0;   // (waited for at the first barrier)
    {
        f32x16 sml[MB][NB];
        zero_blocks<MB, NB>(sml);
        start();
        auto put = [&](char* dst, auto& x, auto items) {
            using It = decltype(items);
#pragma unroll
            for (int i = 0; i < It::NI; ++i) {
                u32x2 h, m, l;
                split4(x[i], h, m, l);
                const int kq = It::kq(i, t);
                char* q = dst + (kq >> 1) * sp_group<It>() + It::entry(It::row(i, t)) * 16 +
                          (kq & 1) * 8;
                *reinterpret_cast<u32x2*>(q) = h;
                *reinterpret_cast<u32x2*>(q + sp_plane<It>()) = m;
                *reinterpret_cast<u32x2*>(q + 2 * sp_plane<It>()) = l;
            }
        };
        auto cut = [&](int chunk, f32x4 (&xa)[IA::NI], f32x4 (&xb)[IB::NI]) {
            char* const buf = smem + (chunk & 1) * BUF;
            add_rows(xa);
            put(buf, xa, IA{});
            put(buf + 3 * sp_plane<IA>(), xb, IB{});
        };
        // The last product (h·l) of a chunk is left for the next step, which
        // issues it between its barrier and the arrival of its fragments.
        SplitFrag fa[MB], fb[NB];
#pragma unroll
        for (int i = 0; i < MB; ++i) fa[i].h = u32x4{0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < NB; ++j) fb[j].l = u32x4{0, 0, 0, 0};
        auto multiply = [&](int kt) {
            const char* const buf = smem + (kt & 1) * BUF;
            SplitFrag na[MB], nb[NB];
#pragma unroll
            for (int i = 0; i < MB; ++i) sp_frag<IA>(buf, ra + 32 * i + lrow, half, na[i]);
#pragma unroll
            for (int j = 0; j < NB; ++j)
                sp_frag<IB>(buf + 3 * sp_plane<IA>(), rb + 32 * j + lrow, half, nb[j]);
            mfma_split<MB, NB, 5, 6>(acc, sml, fa, fb);
            mfma_split<MB, NB, 0, 5>(acc, sml, na, nb);
#pragma unroll
            for (int i = 0; i < MB; ++i) fa[i].h = na[i].h;
#pragma unroll
            for (int j = 0; j < NB; ++j) fb[j].l = nb[j].l;
        };
        // Chunk kt out of LDS; xa / xb hold chunk kt+1, ya / yb take chunk
        // kt+2.  The barrier: every wave's part of chunk kt is in LDS, and its
        // reads of the buffer that chunk kt+1 goes to are done.
        int ahead = whole;   // whole chunks from the loaders' position on
        auto fetch = [&](f32x4 (&xa)[IA::NI], f32x4 (&xb)[IB::NI]) {
            const bool adv = ahead > 1;
            ahead -= adv;
            la.template load<false>(xa, 16, adv);
            lb.template load<false>(xb, 16, adv);
        };
        auto step = [&](int kt, f32x4 (&xa)[IA::NI], f32x4 (&xb)[IB::NI], f32x4 (&ya)[IA::NI],
                        f32x4 (&yb)[IB::NI], auto fold) {
            sp_barrier();
            fetch(ya, yb);   // (past the last chunk: that chunk again)
            __builtin_amdgcn_sched_barrier(0);   // not behind the MFMAs
            multiply(kt);
            if constexpr (fold) fold_rows();
            cut(kt + 1, xa, xb);
            // The fragment reads under the first MFMAs (read where they are used,
            // as the compiler had it, each exposed its latency: 3-4 % of the
            // kernel), then the cutting, whose values have had that much longer
            // to arrive, spread over the other MFMAs.
            constexpr int NM = 6 * MB * NB, NR = 3 * (MB + NB), NP = MB * NB;
            constexpr int WORK = ((BM + BN) * 16 / NT * 13 / 2 + 16) / (NM - NP) + 1;
            constexpr int MOST = LB == L_IMR ? 5 : 6;   // (its addresses take registers)
            constexpr int NV = WORK < MOST ? WORK : MOST;
            __builtin_amdgcn_sched_group_barrier(0x100, MB + NB, 0);
#pragma unroll
            for (int g = 0; g < NM; ++g) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if (MB + NB + 2 * g < NR) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
                if (g >= NP) __builtin_amdgcn_sched_group_barrier(0x002, NV, 0);
            }
        };
        f32x4 xa[IA::NI], xb[IB::NI], ya[IA::NI], yb[IB::NI];
        if (nk > 0) {
            // a partial chunk goes first, so that the loop has no test for it
            if (part) {
                seek(k_begin + 16 * whole);
                la.template load<true>(xa, part, false);
                lb.template load<true>(xb, part, false);
                seek(k_begin);
            } else {
                seek(k_begin);
                fetch(xa, xb);
            }
            if (nk > 1) fetch(ya, yb);
            cut(0, xa, xb);
            int kt = 0;
            for (; kt + 2 < nk; kt += 2) {
                step(kt, ya, yb, xa, xb, std::false_type{});
                step(kt + 1, xa, xb, ya, yb, std::true_type{});
            }
            if (kt + 1 < nk) step(kt, ya, yb, xa, xb, std::false_type{});
            sp_barrier();
            multiply(nk - 1);
            mfma_split<MB, NB, 5, 6>(acc, sml, fa, fb);
        }
        if (split_finish<MB, NB>(acc, sml)) bad = 1;
    }
    __syncthreads();
    if (bad) {
        // The tile again in fp32, through the k-contiguous LDS tile of the
        // direct-to-LDS kernels ([row][16], swizzled groups of four k).
        start();
        float* const At = reinterpret_cast<float*>(smem);
        float* const Bt = At + BM * 16;
        seek(k_begin);
        for (int kt = 0; kt < nk; ++kt) {
            f32x4 xa[IA::NI], xb[IB::NI];
            if (kt < whole) {
                la.template load<false>(xa, 16, true);
                lb.template load<false>(xb, 16, true);
            } else {
                la.template load<true>(xa, part, true);
                lb.template load<true>(xb, part, true);
            }
            add_rows(xa);
            __syncthreads();
#pragma unroll
            for (int i = 0; i < IA::NI; ++i) {
                const int r = IA::row(i, t);
                *reinterpret_cast<f32x4*>(At + r * 16 + ((IA::kq(i, t) ^ kswz(r)) << 2)) = xa[i];
            }
#pragma unroll
            for (int i = 0; i < IB::NI; ++i) {
                const int r = IB::row(i, t);
                *reinterpret_cast<f32x4*>(Bt + r * 16 + ((IB::kq(i, t) ^ kswz(r)) << 2)) = xb[i];
            }
            __syncthreads();
            float fa[MB][8], fb[NB][8];
            dl_frags<L_KV, BM, MB>(At, ra, lane, fa);
            dl_frags<L_KV, BN, NB>(Bt, rb, lane, fb);
            mfma_chunk<MB, NB>(acc, fa, fb);
        }
    }

    if constexpr (RS) {
        if constexpr (kFold)
#pragma unroll
            for (int i = 0; i < IA::NI; ++i) rsum[i] += rtot[i];
        // The four items of a row: on consecutive lanes (k-contiguous A), or
        // on threads BM apart, through LDS.
        if (id.tn == 0) {
            auto write = [&](int r, float tot) {
                const int m = m0 + r;
                if (m >= p.M) return;
                if (p.splits > 1 || p.part) {   // this (split, batch entry)'s partial
                    p.rowsum[((int64_t)id.split * p.batch + id.bz) * p.M + m] = tot;
                } else {
                    float* d = p.rowsum + (int64_t)m * p.rowsum_stride;
                    *d = (p.rowsum_beta != 0.f ? p.rowsum_beta * *d : 0.f) + tot;
                }
            };
            if constexpr (sp_kc<LA>()) {
#pragma unroll
                for (int i = 0; i < IA::NI; ++i) {
                    float v = rsum[i];
                    v += __shfl_xor(v, 1);
                    v += __shfl_xor(v, 2);
                    if ((t & 3) == 0) write(IA::row(i, t), v);
                }
            } else {
                float* const red = reinterpret_cast<float*>(smem);
                __syncthreads();
#pragma unroll
                for (int i = 0; i < IA::NI; ++i)
                    red[(i * NT + t) / BM * BM + IA::row(i, t)] = rsum[i];
                __syncthreads();
                if (t < BM) write(t, (red[t] + red[BM + t]) + (red[2 * BM + t] + red[3 * BM + t]));
            }
        }
    }

    store_tile_lds<MB, NB, NW, WAVES_N, WM, WN, 2 * BUF / 4>(
        p, acc, reinterpret_cast<float*>(smem), m0, n0, wave, lane, id.split, id.bz, n_end);
}

}  // namespace mtk
