// noalloc_rule.hpp -- which calls mt_gemm_noalloc_f32 takes: those whose sizes
// need at most its scratch under the prices below.
//
// A rule of that entry point and no plan: a call that it took is taken, and one
// that it refused is refused, whatever kernels and prices the planner has by
// then.  So the tiles, the prices and the formula are written out here (they are
// those of the fp32 matrix units' tiles when the entry point appeared) and
// nothing of the planner is used.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstdint>

namespace noalloc_rule {

struct Tile {
    int bm, bn;
    double eff;
    int occ;
};
// register-staged; direct-to-LDS (the first four; all where fragments are prefetched)
constexpr Tile kStaged[3] = {{256, 256, 0.86, 1}, {128, 128, 0.75, 2}, {64, 64, 0.57, 4}};
constexpr Tile kDirect[7] = {{256, 256, 0.90, 1}, {128, 128, 0.86, 4}, {64, 64, 0.68, 8},
                             {256, 128, 0.87, 3}, {256, 256, 0.98, 1}, {64, 64, 0.72, 8},
                             {128, 128, 0.90, 3}};

struct Split {
    int64_t kps, splits, wgs, tiles_m;
    size_t bytes;
};

inline Split split_of(const Tile& t, int64_t M, int64_t N, int64_t K, int64_t batch, int64_t s) {
    const int64_t tm = (M + t.bm - 1) / t.bm, tn = (N + t.bn - 1) / t.bn;
    const int64_t kps = K > 0 ? ((K + s - 1) / s + 15) / 16 * 16 : 16;
    const int64_t splits = K > 0 ? (K + kps - 1) / kps : 1;
    return {kps, splits, tm * tn * batch * splits, tm,
            splits > 1 ? (size_t)splits * batch * M * N * sizeof(float) : 0};
}

// Modelled cycles of the partials and their sum.
inline double split_cycles(int64_t splits, int64_t M, int64_t N, int64_t batch) {
    return (double)(2 * splits + 1) * M * N * batch * 4.0 / 6400.0 + 17700.0;
}

// ... of the whole; `small`: a direct-to-LDS tile of 64 x 64, `prefetching`: the
// one of the two with fragment prefetch.
inline double cycles(const Tile& t, const Split& p, bool small, bool prefetching, int64_t M,
                     int64_t N, int64_t batch, int cus) {
    const double per_cu = std::ceil((double)p.wgs / cus);
    const double rounds = std::ceil((double)p.wgs / ((double)cus * t.occ));
    const double work = (double)t.bm * t.bn * (double)std::max<int64_t>(p.kps, 16) * 2.0 /
                        (256.0 * t.eff);
    const double epilogue = (double)t.bm * t.bn * 4.0 / 7.9;
    const double pair = prefetching && p.tiles_m == 1 && per_cu == 2 ? 0.75 : 1.0;
    const double alone = per_cu <= 1 && small && p.kps >= 1024 ? 1.3 : 1.0;
    double c = per_cu * work * pair * alone + per_cu * epilogue / t.occ + rounds * 6200.0;
    if (p.splits > 1) c += split_cycles(p.splits, M, N, batch);
    return c;
}

// Partials of a product of m <= 8 rows (k-contiguous `kv`: 4) against n columns.
inline size_t few_rows(int64_t m, int64_t n, int64_t k, int64_t batch, bool kv, int cus) {
    const int64_t tiles = (n + (kv ? 16 : 256) - 1) / (kv ? 16 : 256);
    const bool large = !kv && k * n * batch * 4 > ((int64_t)64 << 20);
    const int64_t base = tiles * batch, per_cu = large ? 6 : 4;
    int64_t want = std::max<int64_t>(1, (per_cu * cus + base - 1) / base);
    want = std::min<int64_t>({want, std::max<int64_t>(1, k / (kv ? 256 : large ? 32 : 64)),
                              large ? 128 : 64});
    const int64_t gran = kv ? 64 : 4;
    const int64_t kps = ((k + want - 1) / want + gran - 1) / gran * gran;
    const int64_t splits = (k + kps - 1) / kps;
    return splits > 1 ? (size_t)splits * batch * m * n * sizeof(float) : 0;
}

// Whether M x N x K with `batch` entries needs at most `limit` bytes of scratch on
// a GPU of `cus` compute units.
inline bool takes(int64_t M, int64_t N, int64_t K, int64_t batch, int cus, size_t limit) {
    if (K >= 16) {
        for (bool kv : {false, true}) {
            if (M <= (kv ? 4 : 8) && few_rows(M, N, K, batch, kv, cus) > limit) return false;
            if (N <= (kv ? 4 : 8) && few_rows(N, M, K, batch, kv, cus) > limit) return false;
        }
    }
    const int64_t most = std::min<int64_t>(256, std::max<int64_t>(K / 48, 1));
    if ((double)M * N * batch * 4 * most <= (double)limit) return true;   // however it is split
    for (int form = 0; form < 3; ++form) {
        const bool direct = form > 0;
        double best = 1e300;
        size_t bytes = 0;
        for (int i = 0; i < (form == 0 ? 3 : form == 1 ? 4 : 7); ++i) {
            const Tile& t = direct ? kDirect[i] : kStaged[i];
            for (int64_t s = 1; s <= 256; ++s) {
                if (s > 1 && split_cycles(s, M, N, batch) > best) break;   // nor any further split
                const Split p = split_of(t, M, N, K, batch, s);
                if (s > 1 && p.kps < 64) break;
                if (s > 16 && p.kps < 256) break;
                const int64_t k = std::min<int64_t>(p.kps, K);
                if (direct && i == 6 && k < 256) break;
                if (p.splits != s) continue;
                if (direct && i == 6 && k < 512 && p.wgs > cus) continue;
                if (p.wgs * 512 >= ((int64_t)1 << 32)) continue;
                const double c = cycles(t, p, direct && (i == 2 || i == 5), direct && i == 5, M, N,
                                        batch, cus);
                if (c < best) {
                    best = c;
                    bytes = p.bytes;
                }
            }
        }
        if (bytes > limit) return false;
    }
    return true;
}

}  // namespace noalloc_rule
