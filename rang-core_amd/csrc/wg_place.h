// Where the w-gridder places a visibility: its cells, tile and first w-plane
// (wgridder.rs:583-586, 1003-1031). Compiles for the device and for the host.
//
// The sort places each visibility twice, once to count its bucket and once to
// write its record, in two kernels that keep different parts of the result, and
// a record's slot is only right if both find the same bucket. Each function
// here therefore switches contraction off: the compiler would otherwise fuse a
// product into an addition where the product is not needed elsewhere (w + wshift
// in the counting kernel, not in the one that stores w), and a w, u or v within
// a rounding of a boundary would count in one bucket and be written to its
// neighbour's slots. Unfused IEEE operations have one result in any kernel.
#pragma once

#include <cmath>
#include <cstdint>

#include <hip/hip_runtime.h>

#define RANG_PLACE __host__ __device__ __forceinline__

namespace rang {

// Width in u and v of a tile: the matrix-core gridding's last tiles may be
// partial (every other tiling divides the grid).
template <class Geo>
RANG_PLACE int tile_wu(const Geo& g, int tu) {
    const int left = g.nu - tu * g.Tu;
    return g.Tu < left ? g.Tu : left;
}
template <class Geo>
RANG_PLACE int tile_wv(const Geo& g, int tv) {
    const int left = g.nv - tv * g.Tv;
    return g.Tv < left ? g.Tv : left;
}

// Flipped and recentred coordinates of a row.
template <class Geo>
RANG_PLACE void coord_of(const Geo& g, const double* uvw, double c[3]) {
#pragma clang fp contract(off)
    const double tu = g.fu * uvw[0], tv = g.fv * uvw[1];
    const double tw = g.fw * uvw[2];
    c[0] = tu + g.r_l * tw;
    c[1] = tv + g.r_m * tw;
    c[2] = tw;
}

// The first cell of a footprint and the position from it, along one axis of n
// cells. u + shift lies in [n - supp / 2, 2 n + 1): 32-bit cells.
RANG_PLACE void getpix(double uin, double pixsize, int n, double shift, int maxi0, double& uf, int& i0) {
#pragma clang fp contract(off)
    double u = uin * pixsize;
    u = (u - floor(u)) * double(n);
    const int i = int(u + shift) - n;
    i0 = i < maxi0 ? i : maxi0;
    uf = u - double(i0);
}

// (i0 + n / 2) mod n for i0 in [-n / 2, n + n / 2).
RANG_PLACE int shifted(int i0, int n) {
    int v = i0 + n / 2;
    if (v < 0) v += n;
    return v >= n ? v - n : v;
}

// x / d with m = ceil(2^32 / d): exact for x d < 2^32 (grid sides below 2^20
// times tiles of 8 to 64 cells).
RANG_PLACE int tile_of(int x, unsigned m) { return int((unsigned long long)unsigned(x) * m >> 32); }

template <class Geo>
RANG_PLACE int minplane(const Geo& g, double w) {
#pragma clang fp contract(off)
    if (!g.wgrid) return 0;
    const double p = (w + g.wshift) * g.xdw;
    const int m = p > 0.0 ? int(p < 2147483647.0 ? p : 2147483647.0) : 0;
    return m < g.nb - 1 ? m : g.nb - 1;
}

// A visibility's FixW-signed coordinates, the position of its footprint and its
// bucket (tile, spill class, first plane). The spill class says whether its
// footprint reaches the next tile in u (2) and in v (1).
struct Place {
    double imflip, b[3];  // the sign of w and the coordinates times it
    double w, uf, vf;
    int ou, ov, mp;
    std::uint32_t key;
};

// c: coord_of's coordinates; f: frequency / speed of light.
template <class Geo>
RANG_PLACE Place place_at(const Geo& g, const double c[3], double f) {
#pragma clang fp contract(off)
    Place r;
    r.imflip = c[2] < 0.0 ? -1.0 : 1.0;  // FixW (wgridder.rs:583-586)
    r.b[0] = c[0] * r.imflip;
    r.b[1] = c[1] * r.imflip;
    r.b[2] = c[2] * r.imflip;
    const double u = r.b[0] * f, v = r.b[1] * f;
    r.w = r.b[2] * f;
    int iu0, iv0;
    getpix(u, g.pixsize_x, g.nu, g.ushift, int(g.maxiu0), r.uf, iu0);
    getpix(v, g.pixsize_y, g.nv, g.vshift, int(g.maxiv0), r.vf, iv0);
    const int su = shifted(iu0, g.nu), sv = shifted(iv0, g.nv);
    const int tu = tile_of(su, g.mTu), tv = tile_of(sv, g.mTv);
    r.ou = su - tu * g.Tu;
    r.ov = sv - tv * g.Tv;
    const int cat = ((r.ou + g.supp > tile_wu(g, tu)) ? 2 : 0) | ((r.ov + g.supp > tile_wv(g, tv)) ? 1 : 0);
    r.mp = minplane(g, r.w);
    r.key = std::uint32_t((((long long)tu * g.ntv + tv) * 4 + cat) * g.nb + r.mp);
    return r;
}

// Ring of tile t: the distance of its centre from the grid's centre in steps of
// 1 / scale cells. Counted in one kernel and dealt out in another, as above.
constexpr int kRings = 1024;
template <class Geo>
RANG_PLACE int ring_of(const Geo& g, int t, float scale) {
#pragma clang fp contract(off)
    const int tu = t / g.ntv, tv = t - tu * g.ntv;
    const float cu = (float(tu) + 0.5f) * float(g.Tu) - 0.5f * float(g.nu);
    const float cv = (float(tv) + 0.5f) * float(g.Tv) - 0.5f * float(g.nv);
    const int ring = int(sqrtf(cu * cu + cv * cv) * scale);
    return ring < kRings - 1 ? ring : kRings - 1;
}

}  // namespace rang

#undef RANG_PLACE
