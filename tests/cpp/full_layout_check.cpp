// Host-side checks of what the FULL kernels alone use (compfinance_amd/csrc/
// cf_internal.h): the knot search by one 8-byte (FP64: 16-byte) entry a bucket
// against std::upper_bound (interp.h:40), in FP32 through the entry's offset as
// the kernels form it from the float's bits; and the shared-memory regions of
// the Black-Scholes barrier's rows and of the split Sobol table.  Prints one
// JSON object; tests/test_full_layout.py reads it.
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <limits>
#include <random>
#include <vector>

#include "../../compfinance_amd/csrc/cf_internal.h"

using namespace cfk;

static long g_probes = 0, g_wrong = 0, g_outside = 0, g_grids = 0, g_skipped = 0;

template <typename R>
static void check(const std::vector<R>& knots, std::mt19937_64& rng)
{
    const KnotTable<R> t = build_knot_table(knots.data(), int(knots.size()));
    if (t.fix > 1) {   // the LEAN layout's
        ++g_skipped;
        return;
    }
    ++g_grids;
    // the block's copy, at an offset of its own in the block's memory
    const size_t nb = t.entries.size(), at = 1040;
    std::vector<unsigned char> lds(at + nb * sizeof(BucketOne<R>), 0xff);
    for (size_t e = 0; e < nb; ++e) {
        BucketOne<R> one;
        one.k0 = t.entries[e].k0;
        one.lo = t.entries[e].lo;
        std::memcpy(&lds[at + e * sizeof one], &one, sizeof one);
    }
    const R top = R(int(nb) - 1);
    std::vector<R> xs;
    const R inf = std::numeric_limits<R>::infinity();
    for (R k : knots)
        for (R x : {k, std::nextafter(k, inf), std::nextafter(k, -inf)}) xs.push_back(x);
    std::uniform_real_distribution<double> u(double(knots.front()) - 1.0, double(knots.back()) + 1.0);
    for (int i = 0; i < 2000; ++i) xs.push_back(R(u(rng)));
    for (R x : {inf, -inf, std::numeric_limits<R>::max(), -std::numeric_limits<R>::max(), R(0)}) xs.push_back(x);
    for (R x : xs) {
        uint32_t off;
        if constexpr (sizeof(R) == 4) off = bucket_offset(x, t.invh, t.c0, top, bucket_base(at));
        else off = uint32_t(at) + uint32_t(bucket_index(x, t.invh, t.c0, top, int(nb) - 1)) * uint32_t(sizeof(BucketOne<R>));
        ++g_probes;
        if (off < at || off + sizeof(BucketOne<R>) > lds.size() || (off - at) % sizeof(BucketOne<R>)) {
            ++g_outside;
            continue;
        }
        BucketOne<R> e;
        std::memcpy(&e, &lds[off], sizeof e);
        if (count_le_one(e, x) != int(std::upper_bound(knots.begin(), knots.end(), x) - knots.begin())) ++g_wrong;
    }
}

template <typename R>
static void grids(std::mt19937_64& rng)
{
    // spots 50 + 150 i / (n - 1) as log states; FP32 relative to the spot
    for (int n : {1, 2, 20, 30, 60, 255}) {
        std::vector<R> k(static_cast<size_t>(n));
        for (int i = 0; i < n; ++i)
            k[size_t(i)] = R(std::log(50.0 + 150.0 * i / std::max(n - 1, 1)) - (sizeof(R) == 4 ? std::log(100.0) : 0.0));
        check(k, rng);
    }
    std::uniform_real_distribution<double> gap(0.001, 0.2);
    std::uniform_int_distribution<int> nm(1, 255);
    for (int g = 0; g < 300; ++g) {
        std::vector<R> k(size_t(nm(rng)));
        double x = (g % 3 - 1) * 5.0 + gap(rng);
        for (R& v : k) v = R(x += g % 2 ? gap(rng) : 0.05);
        check(k, rng);
    }
}

int main()
{
    std::mt19937_64 rng(20260101);
    grids<float>(rng);
    grids<double>(rng);

    // regions: [offset, offset + used) before the next region, inside the total
    long regions = 0, bad = 0;
    auto region = [&](size_t off, size_t used, size_t next, size_t total) {
        ++regions;
        if (off % 16 || off + used > next || next > total) ++bad;
    };
    for (int rb : {4, 8})
        for (int ad = 0; ad < 2; ++ad)
            for (int lean = 0; lean < 2; ++lean)
                for (int n : {1, 2, 3, 4, 5, 156, 260, 261})
                    for (int waves : {1, 4, 16}) {
                        // Black-Scholes barrier: a step's reals; other layouts none
                        const bool rows = bs_row_layout(false, PRD_BARRIER, lean != 0);
                        const SmemLayout L = smem_layout(n, 0, n + 1, 2, waves, rb, false, false, ad != 0, lean != 0, 0, 1,
                                                         false, rows);
                        const size_t used = rows ? size_t(n) * size_t(bs_row_reals(ad != 0)) * size_t(rb) : 0;
                        region(L.bs, used, L.samples, L.total);
                        region(L.stdv, rows ? 0 : size_t(n) * size_t(rb), L.bs, L.total);
                        if (rows == (lean != 0)) ++bad;
                        // FP64 Dupire adjoint: sixteen words a dimension, by fours, and the tail rows
                        const bool split = split_layout(rb, true, ad != 0, lean != 0);
                        const SmemLayout S = smem_layout(n, 30, n + 1, 2, waves, rb, true, false, ad != 0, lean != 0, 64, 1,
                                                         split, false);
                        if (split != (rb == 8 && ad == 1 && lean == 0)) ++bad;
                        if (split) {
                            region(S.lo, size_t((n + 3) / 4) * 64 * 4, S.mtab, S.total);
                            region(S.mtab, size_t(kMoroTailRows - kMoroLdsRow) * kMoroTailCoefs * 8, S.hi, S.total);
                        }
                    }
    std::printf("{\"probes\": %ld, \"wrong\": %ld, \"outside\": %ld, \"grids\": %ld, \"skipped\": %ld, "
                "\"regions\": %ld, \"bad\": %ld}\n",
                g_probes, g_wrong, g_outside, g_grids, g_skipped, regions, bad);
    return 0;
}
