// Places visibilities on cell, tile and w-plane boundaries twice, as the sort's
// count and scatter do (one keeps the bucket alone, the other the whole
// placement), and counts the visibilities whose buckets differ and the calls
// whose records do not fill every slot once. Built for the host with the
// contraction mode of the device code and fused multiply-adds enabled.
// Prints: calls, visibilities, differing buckets, calls without a permutation,
// planes that differ from the unfused formula, visibilities within an ulp of a
// plane boundary, grids whose tiles do not fill their rings.

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <string>
#include <vector>

#include "wg_place.h"
#include "wg_plan.h"

namespace {

// What wg_place.h reads of a call's geometry.
struct Geo {
    int nu, nv, supp, nb, wgrid;
    double pixsize_x, pixsize_y, ushift, vshift;
    long long maxiu0, maxiv0;
    double wshift, xdw, r_l, r_m, fu, fv, fw;
    int Tu, Tv, ntu, ntv;
    unsigned mTu, mTv;
};

unsigned magic(unsigned d) { return unsigned(((1ull << 32) + d - 1) / d); }

__attribute__((noinline)) void count(const Geo& g, const double* uvw, double f, int n, std::uint32_t* key) {
    for (int i = 0; i < n; ++i) {
        double c[3];
        rang::coord_of(g, uvw + 3 * i, c);
        key[i] = rang::place_at(g, c, f).key;
    }
}

__attribute__((noinline)) void place(const Geo& g, const double* uvw, double f, int n, rang::Place* out) {
    for (int i = 0; i < n; ++i) {
        double c[3];
        rang::coord_of(g, uvw + 3 * i, c);
        out[i] = rang::place_at(g, c, f);
    }
}

// The tile order's two passes: one keeps the counts alone, the other the rings.
__attribute__((noinline)) void ring_counts(const Geo& g, float scale, int* count) {
    for (int t = 0; t < g.ntu * g.ntv; ++t) ++count[rang::ring_of(g, t, scale)];
}

__attribute__((noinline)) void rings_of(const Geo& g, float scale, int* ring) {
    for (int t = 0; t < g.ntu * g.ntv; ++t) ring[t] = rang::ring_of(g, t, scale);
}

// Whether every ring's count is that of the tiles dealt to it, each the ring of
// the unfused distance.
bool rings_agree(const Geo& g) {
    const double far = 0.5 * std::sqrt(double(g.nu + g.Tu) * double(g.nu + g.Tu) + double(g.nv + g.Tv) * double(g.nv + g.Tv));
    const float scale = float(rang::kRings / far);
    std::vector<int> count(rang::kRings, 0), ring(g.ntu * g.ntv);
    ring_counts(g, scale, count.data());
    rings_of(g, scale, ring.data());
    for (int t = 0; t < g.ntu * g.ntv; ++t) {
        --count[ring[t]];
        volatile float hu = (float(t / g.ntv) + 0.5f) * float(g.Tu), hv = (float(t % g.ntv) + 0.5f) * float(g.Tv);
        volatile float cu = hu - 0.5f * float(g.nu), cv = hv - 0.5f * float(g.nv);
        volatile float uu = cu * cu, vv = cv * cv;
        volatile float d2 = uu + vv;
        if (std::min(int(std::sqrt(d2) * scale), rang::kRings - 1) != ring[t]) return false;
    }
    return std::all_of(count.begin(), count.end(), [](int c) { return c == 0; });
}

}  // namespace

int main() {
    long long calls = 0, vis = 0, differ = 0, broken = 0, off = 0, edge = 0, rings = 0;
    for (int trial = 0; trial < 4000; ++trial) {
        const int K = 2 * (8 + trial % 61);  // even: the middle w is (wmin + wmax) / 2
        const double epss[] = {1e-3, 1e-5, 1e-7, 1e-9};
        rang::Options o;
        o.nx = o.ny = 32 + 2 * (trial % 7);
        o.epsilon = epss[trial % 4];
        const double freq = 1.0e9 + 1.37e5 * trial, f = freq / rang::kCLight;
        o.pixsize_x = o.pixsize_y = 0.2 / double(o.nx) + 1e-7 * (trial % 11);
        o.center_x = trial % 3 ? 0.0 : 0.013;
        o.allow_nshift = true;
        const double d = 0.31 + 0.0173 * (trial % 97);
        std::vector<double> uvw(3 * (K + 1));
        double lo = 1e300, hi = 0;
        for (int k = 0; k <= K; ++k) {
            const double w = std::fabs(d * k * f);
            lo = std::min(lo, w);
            hi = std::max(hi, w);
        }
        rang::Geometry G;
        std::string err;
        if (!rang::make_geometry(o, false, std::size_t(K + 1), lo, hi, G, err)) {
            std::fprintf(stderr, "%s\n", err.c_str());
            return 1;
        }
        const int T = std::max(16, G.supp);
        Geo g{int(G.nu), int(G.nv), G.supp, int(std::max<std::size_t>(G.nplanes, 1)), 1, G.pixsize_x, G.pixsize_y,
              G.ushift, G.vshift, G.maxiu0, G.maxiv0, G.wshift, G.xdw, G.r_l, G.r_m, 1.0, 1.0, 1.0, T, T,
              int(G.nu + T - 1) / T, int(G.nv + T - 1) / T, magic(T), magic(T)};
        // w evenly spaced; u and v on cell edges (half cells for odd supports),
        // every T-th of them a tile's
        for (int k = 0; k <= K; ++k) {
            const double half = G.supp % 2 ? 0.5 : 0.0;
            uvw[3 * k] = (double(k % 3 * T - T) + half) / (double(G.nu) * G.pixsize_x * f);
            uvw[3 * k + 1] = (double(k) + half) / (double(G.nv) * G.pixsize_y * f);
            uvw[3 * k + 2] = (k % 2 ? -1.0 : 1.0) * d * k;
        }
        const int n = K + 1;
        std::vector<std::uint32_t> key(n);
        std::vector<rang::Place> at(n);
        count(g, uvw.data(), f, n, key.data());
        place(g, uvw.data(), f, n, at.data());
        // the counting sort: ranks from the count, slots from the placement
        const std::size_t nkeys = std::size_t(g.ntu) * g.ntv * 4 * g.nb;
        std::vector<std::uint32_t> cnt(nkeys + 1, 0), first(nkeys + 1, 0), rank(n);
        bool ok = true;
        for (int i = 0; i < n; ++i) rank[i] = cnt[key[i]]++;
        for (std::size_t k = 0; k < nkeys; ++k) first[k + 1] = first[k] + cnt[k];
        std::vector<int> used(n, 0);
        for (int i = 0; i < n; ++i) {
            const std::uint32_t slot = first[at[i].key] + rank[i];
            if (slot >= std::uint32_t(n) || used[slot]++) ok = false;
            if (at[i].key != key[i]) ++differ;
            volatile double sum = at[i].w + g.wshift;  // rounded on its own
            volatile double p = sum * g.xdw;
            const int m = p > 0.0 ? std::min(int(p), g.nb - 1) : 0;
            if (m != at[i].mp) ++off;
            if (std::floor(p * (1.0 + 4e-16)) != std::floor(p * (1.0 - 4e-16))) ++edge;
        }
        if (!ok) ++broken;
        // tile sides 8 to 64 on grids up to 6000 cells
        Geo r = g;
        r.Tu = 8 + trial % 57;
        r.Tv = 8 + (trial / 3) % 57;
        r.ntu = 3 + trial % 90;
        r.ntv = 2 + (trial / 7) % 90;
        r.nu = r.ntu * r.Tu - trial % 5;
        r.nv = r.ntv * r.Tv - trial % 3;
        if (!rings_agree(r)) ++rings;
        ++calls;
        vis += n;
    }
    std::printf("%lld %lld %lld %lld %lld %lld %lld\n", calls, vis, differ, broken, off, edge, rings);
    return 0;
}
