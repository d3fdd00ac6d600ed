// Places visibilities on cell, tile and w-plane boundaries twice, as the sort's
// count and scatter do (one keeps the bucket alone, the other the whole
// placement), and counts the visibilities whose buckets differ and the calls
// whose records do not fill every slot once. Built for the host with the
// contraction mode of the device code and fused multiply-adds enabled.
// Prints: calls, visibilities, differing buckets, calls without a permutation,
// planes that differ from the unfused formula, visibilities within an ulp of a
// plane boundary.

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

}  // namespace

int main() {
    long long calls = 0, vis = 0, differ = 0, broken = 0, off = 0, edge = 0;
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
        ++calls;
        vis += n;
    }
    std::printf("%lld %lld %lld %lld %lld %lld\n", calls, vis, differ, broken, off, edge);
    return 0;
}
