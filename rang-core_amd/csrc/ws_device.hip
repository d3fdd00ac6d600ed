// The w-stacking gridder (core/src/grid.rs, rang-core's port of WSClean 3.6's
// inversion) on the GPU: the w range and the counters, the placement of
// every sample on its w-layer's grid, then per batch of layers the gridding
// with the oversampled Kaiser-Bessel kernel, the backward 2-D transforms in
// LDS and the projection with the w-screen, added into the image in layer
// order; the normalisation, kernel correction, trim and PSF normalisation
// close. Grid and transforms in T (float or double), sums in double.
//
// Arithmetic is not contracted (no a*b+c fused unless written), as in the
// reference's Rust.
#pragma clang fp contract(off)

#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "wg_fft.h"
#include "ws_device.h"
#include "ws_fft.h"

namespace rang {
namespace ws {

namespace {

struct Fail {
    int status;
    std::string msg;
};

void chk(hipError_t e, const char* what) {
    if (e != hipSuccess) throw Fail{2, std::string(what) + ": " + hipGetErrorString(e)};
}
#define WSCHK(x) chk((x), #x)

constexpr double kC = 299792458.0;

struct Geo {
    int W, H, ks, os, nl;
    double psx, psy, min_w, max_w;  // max_w as the gridder uses it (never equal to min_w)
};

struct In {
    const double* uvw;
    const double* freq;
    const float* data;
    const float* wt;
    const float* iw;
    long long n;
    int nchan;
};

// A sample as WSClean's AddDataSample places it (grid.rs:393-448).
struct Sample {
    int x, y;
    unsigned short xk, yk;
    int layer;
    float re, im, weight;
};

// A sample as the gridding reads it: the first cell of its footprint (x, y of
// the sample less half the kernel, modulo the grid), the sub-cell kernels
// (xk | yk << 16) and the values.
struct Rec {
    int cx, cy;
    unsigned sub;
    float re, im, weight;
};

// WToLayer (grid.rs:334-347): -1 where the rounded value is negative.
__device__ __forceinline__ long long layer_of(const Geo& g, double w) {
    if (g.nl == 1) return 0;
    const double v = round((fabs(w) - g.min_w) * double(g.nl - 1) / (g.max_w - g.min_w));
    return v < 0.0 ? -1 : (long long)v;
}

// sqrt(1 - l^2 - m^2) - 1 at grid index (x, y) (grid.rs:364-391).
__device__ __forceinline__ double sqrt_lm(const Geo& g, int x, int y) {
    int ys = (g.H - y) + g.H / 2;
    if (ys >= g.H) ys -= g.H;
    const double m = (double(ys) - double(g.H / 2)) * g.psy;
    int xs = x + g.W / 2;
    if (xs >= g.W) xs -= g.W;
    const double l = (double(g.W / 2) - double(xs)) * g.psx;
    const double r = l * l + m * m;
    return r < 1.0 ? sqrt(1.0 - l * l - m * m) - 1.0 : 0.0;
}

__device__ __forceinline__ void block_reduce2(double& a, double& b, bool use_min) {
    __shared__ double sa[256], sb[256];
    sa[threadIdx.x] = a;
    sb[threadIdx.x] = b;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if (int(threadIdx.x) < h) {
            sa[threadIdx.x] = use_min ? fmin(sa[threadIdx.x], sa[threadIdx.x + h]) : sa[threadIdx.x] + sa[threadIdx.x + h];
            sb[threadIdx.x] = fmax(sb[threadIdx.x], sb[threadIdx.x + h]);
        }
        __syncthreads();
    }
    a = sa[0];
    b = sb[0];
    __syncthreads();
}

// CalculateMsLimits (grid.rs:652-693): |w| range of the samples with both
// weights nonzero whose cell lies in the image, both bounds from u as in
// WSClean 3.6. Per block: min, max.
__global__ __launch_bounds__(256) void k_limits(In in, Geo g, double* part) {
    double lo = 1e100, hi = 0.0;
    const double hw = 0.5 * double(g.W), hh = 0.5 * double(g.H);
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < in.n; i += (long long)gridDim.x * 256) {
        if (in.wt[i] == 0.0f) continue;
        const long long row = i / in.nchan;
        const int ch = int(i - row * in.nchan);
        const double lam = kC / in.freq[ch];
        const double u = in.uvw[3 * row] / lam, w = in.uvw[3 * row + 2] / lam;
        const double x = u * g.psx * double(g.W), y = u * g.psy * double(g.H);
        if (in.iw[i] != 0.0f && floor(x) > -hw && ceil(x) < hw && floor(y) > -hh && ceil(y) < hh) {
            hi = fmax(hi, fabs(w));
            lo = fmin(lo, fabs(w));
        }
    }
    block_reduce2(lo, hi, true);
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = lo;
        part[2 * blockIdx.x + 1] = hi;
    }
}

// The placement of sample i (grid.rs:763-810 and 393-448): its layer, or -1
// where it adds nothing or falls outside every layer or the grid.
__device__ __forceinline__ bool place(const In& in, const Geo& g, long long i, Sample& s, float& weight_out,
                                      float& cw_out) {
    const long long row = i / in.nchan;
    const int ch = int(i - row * in.nchan);
    const double lam = kC / in.freq[ch];
    double u = in.uvw[3 * row] / lam, v = in.uvw[3 * row + 1] / lam;
    const double w = in.uvw[3 * row + 2] / lam;
    const long long layer = layer_of(g, w);
    const bool inrange = layer >= 0 && layer < g.nl;
    const float weight = inrange ? in.wt[i] : 0.0f;
    const float cw = weight * in.iw[i];
    weight_out = weight;
    cw_out = cw;
    const float re = in.data[2 * i] * cw;
    float im = in.data[2 * i + 1] * cw;
    if ((cw == 0.0f && re == 0.0f && im == 0.0f) || !inrange) return false;
    if (w < 0.0) {
        u = -u;
        v = -v;
        im = -im;
    }
    const long long W = g.W, H = g.H, OS = g.os;
    const double xe = u * g.psx * double(g.W), ye = v * g.psy * double(g.H);
    long long x = (long long)round(xe), y = (long long)round(ye);
    long long xk = (long long)round((xe - double(x)) * double(g.os));
    long long yk = (long long)round((ye - double(y)) * double(g.os));
    xk = (xk + (OS * 3) / 2) % OS;
    yk = (yk + (OS * 3) / 2) % OS;
    if (!(x > -W / 2 && y > -H / 2 && x <= W / 2 && y <= H / 2)) return false;
    if (x < 0) x += W;
    if (y < 0) y += H;
    s.x = int(x);
    s.y = int(y);
    s.xk = (unsigned short)xk;
    s.yk = (unsigned short)yk;
    s.layer = int(layer);
    s.re = re;
    s.im = im;
    s.weight = cw;
    return true;
}

// Per sample its layer (or -1) and per block the counters' partials: image
// weight, visibility weight sum, gridded count, largest gridded weight.
__global__ __launch_bounds__(256) void k_keys(In in, Geo g, int* keys, double* part) {
    double iwsum = 0.0, vsum = 0.0, cnt = 0.0, maxw = 0.0;
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < in.n; i += (long long)gridDim.x * 256) {
        Sample s;
        float weight, cw;
        const bool ok = place(in, g, i, s, weight, cw);
        keys[i] = ok ? s.layer : -1;
        if (cw != 0.0f) {
            vsum += double(weight);
            cnt += 1.0;
        }
        maxw = fmax(maxw, double(cw));
        iwsum += double(cw);
    }
    double a = iwsum, b = maxw;
    block_reduce2(a, b, false);
    double c = vsum, d = 0.0;
    block_reduce2(c, d, false);
    double e = cnt, f = 0.0;
    block_reduce2(e, f, false);
    if (threadIdx.x == 0) {
        part[4 * blockIdx.x] = a;
        part[4 * blockIdx.x + 1] = c;
        part[4 * blockIdx.x + 2] = e;
        part[4 * blockIdx.x + 3] = b;
    }
}

// Samples per layer: a histogram in LDS per block, one atomic per block and
// layer.
__global__ __launch_bounds__(256) void k_hist(const int* keys, long long n, int L, unsigned* counts) {
    extern __shared__ unsigned hist[];
    for (int l = threadIdx.x; l < L; l += 256) hist[l] = 0;
    __syncthreads();
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256)
        if (keys[i] >= 0) atomicAdd(&hist[keys[i]], 1u);
    __syncthreads();
    for (int l = threadIdx.x; l < L; l += 256)
        if (hist[l]) atomicAdd(&counts[l], hist[l]);
}

// The tiling of a batch's grids: tiles of T x T cells (the last ones of a row
// or column as wide as what is left), bucketed per (layer of the batch, tile,
// spill class). The spill class says whether a sample's footprint reaches the
// next tile in x (2) and in y (1). No tile is narrower than ks - 1 cells, so
// none is crossed.
struct Tiling {
    int T, ntx, nty, nb;
    __host__ __device__ int tiles() const { return ntx * nty; }
};

constexpr unsigned kNoKey = 0xffffffffu;

// Runs of equal keys among consecutive lanes (channels of one row usually
// share a tile): whether this lane starts a run, the run's length, this
// lane's position in it and its first lane.
__device__ __forceinline__ void runs(unsigned key, bool& head, int& len, int& pos, int& headlane) {
    const int lane = threadIdx.x & 63;
    const unsigned prev = __shfl_up(key, 1, 64);
    head = lane == 0 || prev != key;
    const unsigned long long heads = __ballot(head);
    const unsigned long long upto = lane == 63 ? ~0ull : ((2ull << lane) - 1);
    headlane = 63 - __clzll(heads & upto);
    pos = lane - headlane;
    const unsigned long long after = heads & ~upto;
    len = (after ? __ffsll((long long)after) - 1 : 64) - lane;
}

// Bucket of each sample of the batch's layers (kNoKey otherwise) and the
// buckets' counts.
__global__ __launch_bounds__(256) void k_bucket(In in, Geo g, Tiling t, const int* layers, const int* slot,
                                                unsigned* keys, unsigned* counts) {
    const long long step = (long long)gridDim.x * 256;
    const long long top = (in.n + 255) / 256 * 256;
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < top; i += step) {
        unsigned key = kNoKey;
        if (i < in.n) {
            const int layer = layers[i];
            const int b = layer >= 0 ? slot[layer] : -1;
            if (b >= 0) {
                Sample s;
                float weight, cw;
                place(in, g, i, s, weight, cw);
                const int mid = g.ks / 2;
                const int cx = (s.x + g.W - mid) % g.W, cy = (s.y + g.H - mid) % g.H;
                const int tx = cx / t.T, ty = cy / t.T;
                const int wx = min(t.T, g.W - tx * t.T), wy = min(t.T, g.H - ty * t.T);
                const int cat = (cx - tx * t.T + g.ks > wx ? 2 : 0) | (cy - ty * t.T + g.ks > wy ? 1 : 0);
                key = unsigned(((long long)b * t.tiles() + ty * t.ntx + tx) * 4 + cat);
            }
            keys[i] = key;
        }
        bool head;
        int len, pos, headlane;
        runs(key, head, len, pos, headlane);
        if (head && key != kNoKey) atomicAdd(&counts[key], unsigned(len));
    }
}

__global__ __launch_bounds__(256) void k_bucket_scatter(In in, Geo g, const unsigned* keys, const unsigned* off,
                                                        unsigned* cursor, Rec* out) {
    const long long step = (long long)gridDim.x * 256;
    const long long top = (in.n + 255) / 256 * 256;
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < top; i += step) {
        const unsigned key = i < in.n ? keys[i] : kNoKey;
        bool head;
        int len, pos, headlane;
        runs(key, head, len, pos, headlane);
        unsigned base = 0;
        if (head && key != kNoKey) base = off[key] + atomicAdd(&cursor[key], unsigned(len));
        base = __shfl(base, headlane, 64);
        if (key == kNoKey) continue;
        Sample s;
        float weight, cw;
        place(in, g, i, s, weight, cw);
        const int mid = g.ks / 2;
        out[base + pos] = Rec{(s.x + g.W - mid) % g.W, (s.y + g.H - mid) % g.H, unsigned(s.xk) | (unsigned(s.yk) << 16),
                              s.re, s.im, s.weight};
    }
}

// Exclusive prefix sums in blocks of 4096 values; block totals to sums.
constexpr int kScan = 4096;
__global__ __launch_bounds__(1024) void k_scan_part(const unsigned* in, unsigned* out, unsigned* sums, long long n) {
    __shared__ unsigned s[1024];
    const long long base = (long long)blockIdx.x * kScan + threadIdx.x * 4;
    unsigned v[4], tot = 0;
    for (int k = 0; k < 4; ++k) {
        v[k] = base + k < n ? in[base + k] : 0u;
        tot += v[k];
    }
    s[threadIdx.x] = tot;
    __syncthreads();
    for (int d = 1; d < 1024; d <<= 1) {
        const unsigned add = threadIdx.x >= unsigned(d) ? s[threadIdx.x - d] : 0u;
        __syncthreads();
        s[threadIdx.x] += add;
        __syncthreads();
    }
    unsigned run = s[threadIdx.x] - tot;
    for (int k = 0; k < 4; ++k) {
        if (base + k < n) out[base + k] = run;
        run += v[k];
    }
    if (threadIdx.x == 1023) sums[blockIdx.x] = s[1023];
}

__global__ __launch_bounds__(256) void k_scan_add(unsigned* out, const unsigned* sums, long long n) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) out[i] += sums[i / kScan];
}

// The nine bucket ranges whose samples reach a tile: its own four spill
// classes, those of the tile before in x that spill in x, of the one before
// in y that spill in y, and of the diagonal one that spill in both.
__device__ __forceinline__ void source_of(int src, int& du, int& dv, int& cat) {
    du = (src == 4 || src == 5 || src == 8) ? 1 : 0;
    dv = src >= 6 ? 1 : 0;
    cat = src < 4 ? src : src < 6 ? src - 2 : src < 8 ? 2 * src - 11 : 3;
}

__device__ __forceinline__ void source_range(const Tiling& t, const unsigned* off, int b, int tx, int ty, int src,
                                             unsigned& a, unsigned& e) {
    int du, dv, cat;
    source_of(src, du, dv, cat);
    const int sx = du ? (tx ? tx - 1 : t.ntx - 1) : tx, sy = dv ? (ty ? ty - 1 : t.nty - 1) : ty;
    const long long k = ((long long)b * t.tiles() + sy * t.ntx + sx) * 4 + cat;
    a = off[k];
    e = off[k + 1];
}

// Items (chunks of at most kChunk samples) of each (layer, tile).
constexpr unsigned kChunk = 4096;
__global__ __launch_bounds__(256) void k_items(Tiling t, const unsigned* off, unsigned* items) {
    const long long units = (long long)t.nb * t.tiles();
    const long long u = (long long)blockIdx.x * 256 + threadIdx.x;
    if (u > units) return;
    unsigned total = 0;
    if (u < units) {
        const int b = int(u / t.tiles()), tile = int(u - (long long)b * t.tiles());
        for (int src = 0; src < 9; ++src) {
            unsigned a, e;
            source_range(t, off, b, tile % t.ntx, tile / t.ntx, src, a, e);
            total += e - a;
        }
    }
    items[u] = (total + kChunk - 1) / kChunk;
}

// Clears the cells of the tiles that no item writes whole: those without
// samples and those whose several items add into them.
template <class T>
__global__ __launch_bounds__(256) void k_clear(Tiling t, Geo g, const unsigned* item_off, cx<T>* gd, cx<T>* gp) {
    const long long u = blockIdx.x;
    if (item_off[u + 1] - item_off[u] == 1) return;
    const int b = int(u / t.tiles()), tile = int(u - (long long)b * t.tiles());
    const int ty = tile / t.ntx, tx = tile - ty * t.ntx;
    const int wx = min(t.T, g.W - tx * t.T), wy = min(t.T, g.H - ty * t.T);
    const long long base = (long long)b * g.W * g.H + (long long)ty * t.T * g.W + tx * t.T;
    const int col = threadIdx.x & 31;
    if (col >= wx) return;
    for (int r = threadIdx.x >> 5; r < wy; r += 8) {
        gd[base + (long long)r * g.W + col] = cx<T>{T(0), T(0)};
        gp[base + (long long)r * g.W + col] = cx<T>{T(0), T(0)};
    }
}

// grid_layer (grid.rs:450-495) of one item: a chunk of the samples whose
// footprints reach one tile of one layer, dirty and PSF accumulated in LDS in
// double and written once (added with global atomics into cleared cells where
// a tile has several items). One sample per wave at a time, a lane per tap
// (KS 7; any odd kernel otherwise): a wave loads 64 records, one a lane, and
// broadcasts them in turn, so the sample's position is wave-uniform. The row
// stride 7 mod 32 (in doubles) spreads a 7 x 7 footprint over the banks.
// A wave per sample adding its 147 values to the grids in memory took 67.8 ms
// for 23.8 M samples on 64 layers of 1232^2 (f64), bound by the memory-side
// atomics; the LDS adds (5.5 a clock and CU) leave 3.5e9 adds 1.0 ms of work,
// and this kernel takes 3.0 ms (with the bucket sort 4.5).
constexpr int kTile = 32;
template <class T, int KS>
__global__ __launch_bounds__(256) void k_grid_tile(const Rec* __restrict__ recs, const unsigned* __restrict__ off,
                                                   const unsigned* __restrict__ item_off, Tiling t, Geo g,
                                                   const double* __restrict__ kern, cx<T>* __restrict__ gd,
                                                   cx<T>* __restrict__ gp) {
    constexpr int STR = kTile + 7, PL = kTile * STR;
    __shared__ double acc[3 * PL];
    __shared__ unsigned s_start[9], s_pre[10];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
    const long long units = (long long)t.nb * t.tiles();
    const unsigned item = blockIdx.x;
    if (item >= item_off[units]) return;
    // the unit holding the item: a search 64 ways at a time
    long long lo = 0, hi = units;  // item_off[lo] <= item < item_off[hi]
    while (hi - lo > 1) {
        const long long step = (hi - lo + 63) / 64, probe = lo + lane * step;
        const bool le = probe < hi && item_off[probe] <= item;
        const int c = __popcll(__ballot(le));
        hi = min(hi, lo + c * step);
        lo += (c - 1) * step;
    }
    const unsigned chunk = item - item_off[lo];
    const bool whole = item_off[lo + 1] - item_off[lo] == 1;
    const int b = int(lo / t.tiles()), tile = int(lo - (long long)b * t.tiles());
    const int ty = tile / t.ntx, tx = tile - ty * t.ntx;
    const int x0 = tx * t.T, y0 = ty * t.T;
    const int wx = min(t.T, g.W - x0), wy = min(t.T, g.H - y0);
    for (int e = threadIdx.x; e < 3 * PL; e += 256) acc[e] = 0.0;
    if (threadIdx.x < 9) {
        unsigned a, e;
        source_range(t, off, b, tx, ty, int(threadIdx.x), a, e);
        s_start[threadIdx.x] = a;
        s_pre[threadIdx.x + 1] = e - a;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        s_pre[0] = 0;
        for (int k = 1; k <= 9; ++k) s_pre[k] += s_pre[k - 1];
    }
    __syncthreads();
    const int ks = KS ? KS : g.ks;
    const unsigned jbeg = chunk * kChunk, jend = min(s_pre[9], jbeg + kChunk);
    // the lane's tap, for kernels of at most 64 taps
    const int tj = lane / ks, ti = lane - tj * ks;
    const bool tap = lane < ks * ks;
    for (unsigned base = jbeg + 64u * unsigned(wave); base < jend; base += 256) {
        const int nrec = int(min(jend - base, 64u));
        Rec r{};
        if (lane < nrec) {
            const unsigned j = base + unsigned(lane);
            int src = 0;
            while (j >= s_pre[src + 1]) ++src;
            r = recs[s_start[src] + (j - s_pre[src])];
            int du, dv, cat;
            source_of(src, du, dv, cat);
            // offsets from the tile's first cell, negative from the tiles before
            r.cx -= x0 + (du && tx == 0 ? g.W : 0);
            r.cy -= y0 + (dv && ty == 0 ? g.H : 0);
        }
        for (int k = 0; k < nrec; ++k) {
            const int ox = __builtin_amdgcn_readlane(r.cx, k), oy = __builtin_amdgcn_readlane(r.cy, k);
            const unsigned sub = unsigned(__builtin_amdgcn_readlane(int(r.sub), k));
            const double re = double(__int_as_float(__builtin_amdgcn_readlane(__float_as_int(r.re), k)));
            const double im = double(__int_as_float(__builtin_amdgcn_readlane(__float_as_int(r.im), k)));
            const double wt = double(__int_as_float(__builtin_amdgcn_readlane(__float_as_int(r.weight), k)));
            const double* kx = kern + (sub & 0xffffu) * unsigned(ks);
            const double* ky = kern + (sub >> 16) * unsigned(ks);
            if constexpr (KS != 0) {
                const int cx_ = ox + ti, cy_ = oy + tj;
                if (tap && unsigned(cx_) < unsigned(wx) && unsigned(cy_) < unsigned(wy)) {
                    const double kv = ky[tj] * kx[ti];
                    double* at = acc + cy_ * STR + cx_;
                    atomicAdd(at, re * kv);
                    atomicAdd(at + PL, im * kv);
                    atomicAdd(at + 2 * PL, wt * kv);
                }
            } else {
                for (int q = lane; q < ks * ks; q += 64) {
                    const int j = q / ks, i = q - j * ks;
                    const int cx_ = ox + i, cy_ = oy + j;
                    if (unsigned(cx_) < unsigned(wx) && unsigned(cy_) < unsigned(wy)) {
                        const double kv = ky[j] * kx[i];
                        double* at = acc + cy_ * STR + cx_;
                        atomicAdd(at, re * kv);
                        atomicAdd(at + PL, im * kv);
                        atomicAdd(at + 2 * PL, wt * kv);
                    }
                }
            }
        }
    }
    __syncthreads();
    const long long base = (long long)b * g.W * g.H + (long long)y0 * g.W + x0;
    const int col = threadIdx.x & 31;
    if (col >= wx) return;
    for (int row = threadIdx.x >> 5; row < wy; row += 8) {
        const double* at = acc + row * STR + col;
        const long long c = base + (long long)row * g.W + col;
        if (whole) {
            gd[c] = cx<T>{T(at[0]), T(at[PL])};
            gp[c] = cx<T>{T(at[2 * PL]), T(0)};
        } else {
            if (at[0] != 0.0 || at[PL] != 0.0) {
                atomicAdd(&gd[c].re, T(at[0]));
                atomicAdd(&gd[c].im, T(at[PL]));
            }
            if (at[2 * PL] != 0.0) atomicAdd(&gp[c].re, T(at[2 * PL]));
        }
    }
}

// The tile side for a grid of w x h cells and kernels of ks: the largest up to
// kTile for which the last tiles are at least ks - 1 cells wide (footprints
// then reach at most one tile further), 0 where there is none (grids below
// ks cells, kernels wider than a tile) or where a batch of layers has more tiles
// than a launch holds workgroups.
bool tiles(int n, int T, int ks) { return n >= ks && (n % T == 0 || n % T >= ks - 1); }

int tile_side(int w, int h, int ks, int batch) {
    for (int T = kTile; T >= std::max(ks, 16); --T)
        if (tiles(w, T, ks) && tiles(h, T, ks))
            return (long long)batch * ((w + T - 1) / T) * ((h + T - 1) / T) < (1LL << 24) ? T : 0;
    return 0;
}

// grid_layer on grids or kernels that do not tile (tile_side 0): one wave per
// sample, a lane per tap, the weighted sample into the dirty grid and its
// weight into the PSF grid of its slot in the batch by global atomics. Taps
// in double, added in T.
template <class T>
__global__ __launch_bounds__(256) void k_grid_any(In in, Geo g, const int* layers, const int* slot,
                                                  const double* kern, cx<T>* gd, cx<T>* gp) {
    const int lane = threadIdx.x & 63;
    const long long plane = (long long)g.W * g.H;
    const int mid = g.ks / 2;
    for (long long i = (long long)blockIdx.x * 4 + (threadIdx.x >> 6); i < in.n; i += (long long)gridDim.x * 4) {
        if (layers[i] < 0 || slot[layers[i]] < 0) continue;
        Sample q;
        float weight, cw;
        place(in, g, i, q, weight, cw);
        const long long base = (long long)slot[q.layer] * plane;
        const double re = double(q.re), im = double(q.im), wt = double(q.weight);
        for (int tap = lane; tap < g.ks * g.ks; tap += 64) {
            const int j = tap / g.ks, k = tap - j * g.ks;
            // kernels wider than the grid wrap more than once
            const int cy = ((q.y + j - mid) % g.H + g.H) % g.H;
            const int cx = ((q.x + k - mid) % g.W + g.W) % g.W;
            const double kv = kern[q.yk * g.ks + j] * kern[q.xk * g.ks + k];
            const long long at = base + cx + (long long)cy * g.W;
            atomicAdd(&gd[at].re, T(re * kv));
            atomicAdd(&gd[at].im, T(im * kv));
            atomicAdd(&gp[at].re, T(wt * kv));
        }
    }
}

// Unnormalised backward transform of contiguous rows of length d.n, in place.
template <class T, int NT, int MT>
__global__ __launch_bounds__(NT) void k_rows(cx<T>* data, FftDesc d, const cx<T>* tw) {
    extern __shared__ __align__(16) unsigned char smem[];
    cx<T>* buf = reinterpret_cast<cx<T>*>(smem);
    cx<T>* row = data + (long long)blockIdx.x * d.n;
    for (int e = threadIdx.x; e < d.n; e += NT) buf[e] = row[e];
    __syncthreads();
    fft_lds<T, NT, MT, +1>(buf, d, 1, tw);
    for (int e = threadIdx.x; e < d.n; e += NT) row[e] = buf[e];
}

// A linear block index remapped so that the workgroups one XCD holds at a
// time take consecutive indices (consecutive workgroups go to the eight
// XCDs in turn, each with its own L2).
__device__ __forceinline__ int xcd_remap(int bid, int nblocks) {
    constexpr int X = 8;
    const int per = nblocks / X, rem = nblocks - per * X;
    const int x = bid % X, k = bid / X;
    return x * per + min(x, rem) + k;
}

// Backward transform of C neighbouring columns (length d.n = H, stride W) of
// one of the grids, in place.
template <class T, int NT, int MT>
__global__ __launch_bounds__(NT) void k_cols(cx<T>* data, FftDesc d, const cx<T>* tw, int W, int C, int ncb) {
    extern __shared__ __align__(16) unsigned char smem[];
    cx<T>* buf = reinterpret_cast<cx<T>*>(smem);
    const int lin = xcd_remap(blockIdx.x, gridDim.x);
    const int gi = lin / ncb, x0 = (lin - gi * ncb) * C, nc = min(C, W - x0);
    const int H = d.n;
    cx<T>* base = data + (long long)gi * W * H;
    for (int e = threadIdx.x; e < H * nc; e += NT) {
        const int y = e / nc, c = e - y * nc;
        buf[c * H + y] = base[(long long)y * W + x0 + c];
    }
    __syncthreads();
    fft_lds<T, NT, MT, +1>(buf, d, nc, tw);
    for (int e = threadIdx.x; e < H * nc; e += NT) {
        const int y = e / nc, c = e - y * nc;
        base[(long long)y * W + x0 + c] = buf[c * H + y];
    }
}

// project (grid.rs:497-529) of the batch's layers, their terms added to the
// running sums in layer order.
template <class T>
__global__ __launch_bounds__(256) void k_project(const cx<T>* gd, const cx<T>* gp, int nb, const double* wl,
                                                 Geo g, double* sd, double* sp) {
    const long long plane = (long long)g.W * g.H;
    const long long e = (long long)blockIdx.x * 256 + threadIdx.x;
    if (e >= plane) return;
    const int y = int(e / g.W), x = int(e - (long long)y * g.W);
    int ys = (g.H - y) + g.H / 2;
    if (ys >= g.H) ys -= g.H;
    int xs = x + g.W / 2;
    if (xs >= g.W) xs -= g.W;
    const long long t = xs + (long long)ys * g.W;
    const double slm = sqrt_lm(g, x, y);
    double ad = sd[t], ap = sp[t];
    for (int b = 0; b < nb; ++b) {
        const double rad = (-2.0 * M_PI * wl[b]) * slm;
        double sn, cs;
        sincos(rad, &sn, &cs);
        const cx<T> vd = gd[b * plane + e], vp = gp[b * plane + e];
        ad += double(vd.re) * cs - double(vd.im) * sn;
        ap += double(vp.re) * cs - double(vp.im) * sn;
    }
    sd[t] = ad;
    sp[t] = ap;
}

// normalise and correct_for_kernel (grid.rs:597-650), then the trim
// (grid.rs:91-107) into the output images.
__global__ __launch_bounds__(256) void k_finish(const double* sd, const double* sp, Geo g, double factor,
                                                const double* ox, const double* oy, int ow, int oh,
                                                double* od, double* op) {
    const long long e = (long long)blockIdx.x * 256 + threadIdx.x;
    if (e >= (long long)ow * oh) return;
    const int yo = int(e / ow), xo = int(e - (long long)yo * ow);
    const int x = (g.W - ow) / 2 + xo, y = (g.H - oh) / 2 + yo;
    const double yv = y >= g.H / 2 ? oy[y - g.H / 2] : oy[g.H / 2 - y];
    const double xv = x >= g.W / 2 ? ox[x - g.W / 2] : ox[g.W / 2 - x];
    const double div = xv * yv * (1.0 / (double(g.os) * double(g.os)));
    const long long s = x + (long long)y * g.W;
    od[e] = (sd[s] * factor) / div;
    op[e] = (sp[s] * factor) / div;
}

// The PSF normalisation (grid.rs:862-873).
__global__ __launch_bounds__(256) void k_normalise(double* od, double* op, double pn, long long n) {
    const long long e = (long long)blockIdx.x * 256 + threadIdx.x;
    if (e >= n) return;
    od[e] *= pn;
    op[e] *= pn;
}

// dct3_prefix (grid.rs:263-279): out[k] = in[0] + 2 sum_j in[j] cos(pi j (k + 1/2) / n),
// one block per k.
__global__ __launch_bounds__(256) void k_dct3(const double* in, int len, double n, double* out) {
    const double kk = double(blockIdx.x) + 0.5;
    double s = 0.0, unused = 0.0;
    for (int j = 1 + int(threadIdx.x); j < len; j += 256) s += 2.0 * in[j] * cos(M_PI * double(j) * kk / n);
    block_reduce2(s, unused, false);
    if (threadIdx.x == 0) out[blockIdx.x] = in[0] + s;
}

template <int V>
using ic = std::integral_constant<int, V>;

template <class T, class F>
void fft_sizes(int need, F&& f) {
    if (need <= 1024)
        f(ic<256>{}, ic<1024>{});
    else if (need <= 2048)
        f(ic<256>{}, ic<2048>{});
    else if (need <= 4096)
        f(ic<256>{}, ic<4096>{});
    else if (need <= 8192)
        f(ic<512>{}, ic<8192>{});
    else if constexpr (sizeof(T) == 4) {
        if (need <= 16384)
            f(ic<512>{}, ic<16384>{});
        else
            throw Fail{1, "padded image side above the GPU transform limit"};
    } else {
        throw Fail{1, "padded image side above the GPU transform limit"};
    }
}

template <class K>
void set_lds(K kernel, std::size_t bytes) {
    WSCHK(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, int(bytes)));
}

// Zeros in 4-byte words, by a kernel of this library.
__global__ __launch_bounds__(256) void k_zero(unsigned* p, long long words) {
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < words; i += (long long)gridDim.x * 256) p[i] = 0u;
}

void clear(void* p, std::size_t bytes, hipStream_t st) {
    const long long words = (long long)(bytes / 4);
    if (words == 0) return;
    k_zero<<<unsigned(std::min<long long>((words + 255) / 256, 16384)), 256, 0, st>>>(static_cast<unsigned*>(p), words);
    WSCHK(hipGetLastError());
}

// Exclusive prefix sum of n <= 2^26 + 1 values; sums: 2 (n / kScan + 32) words
// of scratch.
void exclusive_scan(const unsigned* in, unsigned* out, long long n, unsigned* sums, hipStream_t st) {
    const long long blocks = (n + kScan - 1) / kScan, upper = (blocks + kScan - 1) / kScan;
    unsigned* total = sums + blocks;  // scanned block totals follow
    k_scan_part<<<unsigned(blocks), 1024, 0, st>>>(in, out, sums, n);
    if (blocks > 1) {
        // block totals, then (beyond kScan blocks) the totals of those: at
        // most kScan * kScan blocks, so one more level is enough
        k_scan_part<<<unsigned(upper), 1024, 0, st>>>(sums, total, total + blocks, blocks);
        if (upper > 1) {
            k_scan_part<<<1, 1024, 0, st>>>(total + blocks, total + blocks, total + blocks + upper, upper);
            k_scan_add<<<unsigned((blocks + 255) / 256), 256, 0, st>>>(total, total + blocks, blocks);
        }
        k_scan_add<<<unsigned((n + 255) / 256), 256, 0, st>>>(out, total, n);
    }
    WSCHK(hipGetLastError());
}

// Device buffers kept per device between calls (allocating and freeing
// gigabytes per call cost more than the gridding): the k-th request of a
// call reuses the k-th slot, grown when too small. Calls on one device are
// serialised by the pool's mutex.
struct Pool {
    std::mutex mu;
    std::vector<std::pair<void*, std::size_t>> slots;
};

Pool& pool_of_current_device() {
    static std::mutex mu;
    static std::map<int, Pool*> pools;
    int dev = 0;
    WSCHK(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(mu);
    Pool*& p = pools[dev];
    if (!p) p = new Pool;  // kept until the process ends, as the buffers are
    return *p;
}

struct Bufs {
    Pool& pool;
    std::size_t next = 0;
    std::size_t bytes = 0;
    explicit Bufs(Pool& p) : pool(p) {}
    template <class P>
    P* get(std::size_t n) {
        const std::size_t need = std::max<std::size_t>(n * sizeof(P), 16);
        if (next >= pool.slots.size()) pool.slots.push_back({nullptr, 0});
        auto& s = pool.slots[next++];
        if (s.second < need) {
            if (s.first) WSCHK(hipFree(s.first));
            s.first = nullptr;
            s.second = 0;
            WSCHK(hipMalloc(&s.first, need));
            s.second = need;
        }
        bytes += n * sizeof(P);
        return static_cast<P*>(s.first);
    }
};

// Transforms of contiguous lines of any length N in place (ws_fft.h): kind
// 0 one line in LDS, 1 four steps of N = M1 M2, 2 Bluestein in LDS, 3
// Bluestein over four steps of M = M1 M2.
template <class T>
struct LineFft {
    int N = 0, kind = 0, sgn = 1;
    long long M = 0;
    int M1 = 0, M2 = 0;
    FftDesc d, d1, d2;
    cx<T>*tw = nullptr, *tw1 = nullptr, *tw2 = nullptr, *chirp = nullptr, *bhat = nullptr;
    static constexpr int kBudget = 8192;  // values per workgroup in the four-step passes

    static cx<T>* upload_tw(Bufs& b, const std::vector<double>& t, hipStream_t st, std::vector<std::vector<cx<T>>>& keep) {
        keep.emplace_back(t.size() / 2);
        auto& h = keep.back();
        for (std::size_t q = 0; q < h.size(); ++q) h[q] = {T(t[2 * q]), T(t[2 * q + 1])};
        cx<T>* dptr = b.get<cx<T>>(std::max<std::size_t>(h.size(), 1));
        if (!h.empty()) WSCHK(hipMemcpyAsync(dptr, h.data(), sizeof(cx<T>) * h.size(), hipMemcpyHostToDevice, st));
        return dptr;
    }

    void describe(int n, FftDesc& dd, cx<T>*& t, Bufs& b, hipStream_t st, std::vector<std::vector<cx<T>>>& keep) {
        std::vector<double> tt;
        if (!fft_describe(n, dd, tt)) throw Fail{1, "transform length not a product of 2, 3, 5, 7 and 11"};
        t = upload_tw(b, tt, st, keep);
    }

    void setup(int n, int sign, Bufs& b, hipStream_t st, std::vector<std::vector<cx<T>>>& keep) {
        N = n;
        sgn = sign;
        const int L = lds_values<T>();
        if (is_good(N) && N <= L) {
            kind = 0;
            describe(N, d, tw, b, st, keep);
            return;
        }
        if (is_good(N)) {
            kind = 1;
            M = N;
            if (!split_two(N, L, M1, M2)) throw Fail{1, "no two-pass split of the transform length"};
            describe(M1, d1, tw1, b, st, keep);
            describe(M2, d2, tw2, b, st, keep);
            return;
        }
        M = good_length(2LL * N - 1);
        // the chirp c_k = exp(sgn pi i k^2 / N) and the filter b_m = conj(c_m) at +-m
        std::vector<cx<T>> hc(N);
        std::vector<cx<double>> hb(std::size_t(M), cx<double>{0.0, 0.0});
        const long double pi = 3.141592653589793238462643383279502884L;
        for (long long k = 0; k < N; ++k) {
            const long long r = (k * k) % (2LL * N);
            const long double a = pi * (long double)r / (long double)N;
            const double c = double(cosl(a)), sn = double(sinl(a)) * double(sgn);
            hc[k] = {T(c), T(sn)};
            hb[k] = {c, -sn};
            if (k > 0) hb[M - k] = {c, -sn};
        }
        keep.emplace_back(hc);
        chirp = b.get<cx<T>>(N);
        WSCHK(hipMemcpyAsync(chirp, keep.back().data(), sizeof(cx<T>) * N, hipMemcpyHostToDevice, st));
        keep.emplace_back(std::size_t(M));
        auto& hbt = keep.back();
        for (long long q = 0; q < M; ++q) hbt[q] = {T(hb[q].re), T(hb[q].im)};
        bhat = b.get<cx<T>>(std::size_t(M));
        WSCHK(hipMemcpyAsync(bhat, hbt.data(), sizeof(cx<T>) * M, hipMemcpyHostToDevice, st));
        if (M <= L) {
            kind = 2;
            describe(int(M), d, tw, b, st, keep);
            forward_lds(bhat, 1, st);
        } else {
            kind = 3;
            if (!split_two(M, L, M1, M2)) throw Fail{1, "no two-pass split of the chirp transform length"};
            describe(M1, d1, tw1, b, st, keep);
            describe(M2, d2, tw2, b, st, keep);
            cols(bhat, 1, -1, true, st);
            rows(bhat, 1, -1, false, st);
        }
        k_scale<T><<<unsigned((M + 255) / 256), 256, 0, st>>>(bhat, M, 1.0 / double(M));
        WSCHK(hipGetLastError());
    }

    void forward_lds(cx<T>* data, long long lines, hipStream_t st) {
        fft_sizes<T>(d.n, [&](auto nt, auto mt) {
            constexpr int NT = decltype(nt)::value, MT = decltype(mt)::value;
            const std::size_t lds = sizeof(cx<T>) * d.n;
            set_lds(k_line_lds<T, NT, MT>, lds);
            for (long long l0 = 0; l0 < lines; l0 += (1LL << 30)) {
                const long long nl = std::min(lines - l0, 1LL << 30);
                k_line_lds<T, NT, MT><<<unsigned(nl), NT, lds, st>>>(data + l0 * d.n, d, tw, -1);
            }
        });
        WSCHK(hipGetLastError());
    }

    void cols(cx<T>* buf, long long lines, int s, bool twid, hipStream_t st) {
        const int C = std::max(1, std::min(M2, kBudget / M1));
        const long long nb = lines * ((M2 + C - 1) / C);
        if (nb >= (1LL << 31)) throw Fail{1, "transform batch too large"};
        fft_sizes<T>(M1 * C, [&](auto nt, auto mt) {
            constexpr int NT = decltype(nt)::value, MT = decltype(mt)::value;
            const std::size_t lds = sizeof(cx<T>) * M1 * C;
            set_lds(k_fs_cols<T, NT, MT>, lds);
            k_fs_cols<T, NT, MT><<<unsigned(nb), NT, lds, st>>>(buf, M1, M2, C, d1, tw1, s, twid ? 1 : 0);
        });
        WSCHK(hipGetLastError());
    }

    void rows(cx<T>* buf, long long lines, int s, bool twid, hipStream_t st) {
        const int K = std::max(1, std::min(M1, kBudget / M2));
        const long long nb = lines * ((M1 + K - 1) / K);
        if (nb >= (1LL << 31)) throw Fail{1, "transform batch too large"};
        fft_sizes<T>(M2 * K, [&](auto nt, auto mt) {
            constexpr int NT = decltype(nt)::value, MT = decltype(mt)::value;
            const std::size_t lds = sizeof(cx<T>) * M2 * K;
            set_lds(k_fs_rows<T, NT, MT>, lds);
            k_fs_rows<T, NT, MT><<<unsigned(nb), NT, lds, st>>>(buf, M1, M2, K, d2, tw2, s, twid ? 1 : 0);
        });
        WSCHK(hipGetLastError());
    }

    static void transpose(const cx<T>* in, cx<T>* out, long long lines, int A, int B, hipStream_t st) {
        for (long long l0 = 0; l0 < lines; l0 += 65535) {
            const long long nl = std::min<long long>(65535, lines - l0);
            k_transpose<T><<<dim3((B + 31) / 32, (A + 31) / 32, unsigned(nl)), 256, 0, st>>>(
                in + l0 * (long long)A * B, out + l0 * (long long)A * B, A, B);
        }
        WSCHK(hipGetLastError());
    }

    // Lines of `scratch_values` complex values of work space at least
    // N (kind 1) or M (kind 3) times one line.
    void apply(cx<T>* data, long long lines, cx<T>* scratch, long long scratch_values, hipStream_t st) {
        if (kind == 0) {
            fft_sizes<T>(N, [&](auto nt, auto mt) {
                constexpr int NT = decltype(nt)::value, MT = decltype(mt)::value;
                const std::size_t lds = sizeof(cx<T>) * N;
                set_lds(k_line_lds<T, NT, MT>, lds);
                k_line_lds<T, NT, MT><<<unsigned(lines), NT, lds, st>>>(data, d, tw, sgn);
            });
            WSCHK(hipGetLastError());
            return;
        }
        if (kind == 2) {
            fft_sizes<T>(int(M), [&](auto nt, auto mt) {
                constexpr int NT = decltype(nt)::value, MT = decltype(mt)::value;
                const std::size_t lds = sizeof(cx<T>) * M;
                set_lds(k_blue_lds<T, NT, MT>, lds);
                k_blue_lds<T, NT, MT><<<unsigned(lines), NT, lds, st>>>(data, N, d, tw, chirp, bhat);
            });
            WSCHK(hipGetLastError());
            return;
        }
        const long long per = std::max<long long>(1, scratch_values / M);
        for (long long l0 = 0; l0 < lines; l0 += per) {
            const long long nl = std::min(per, lines - l0);
            cx<T>* x = data + l0 * N;
            if (kind == 1) {
                cols(x, nl, sgn, true, st);
                rows(x, nl, sgn, false, st);
                transpose(x, scratch, nl, M1, M2, st);
                WSCHK(hipMemcpyAsync(x, scratch, sizeof(cx<T>) * nl * N, hipMemcpyDeviceToDevice, st));
            } else {
                const unsigned gb = unsigned(std::min<long long>((nl * M + 255) / 256, 65536));
                k_blue_in<T><<<gb, 256, 0, st>>>(x, N, M, nl, chirp, scratch);
                cols(scratch, nl, -1, true, st);
                rows(scratch, nl, -1, false, st);
                k_mul_spec<T><<<gb, 256, 0, st>>>(scratch, M, nl, bhat);
                rows(scratch, nl, +1, true, st);
                cols(scratch, nl, +1, false, st);
                k_blue_out<T><<<gb, 256, 0, st>>>(scratch, N, M, nl, chirp, x);
                WSCHK(hipGetLastError());
            }
        }
    }
    // work space values apply() needs for one line
    long long scratch_per_line() const { return kind == 1 ? N : kind == 3 ? M : 0; }
};

using Clock = std::chrono::steady_clock;
double since(Clock::time_point t) { return std::chrono::duration<double>(Clock::now() - t).count(); }

std::size_t pad_side(std::size_t n, double padding) {
    std::size_t p = std::size_t(std::ceil(double(n) * padding));
    return p + (4 - p % 4) % 4;
}

double bessel0(double x, double precision) {
    double d = 0.0, ds = 1.0, sum = 1.0;
    for (;;) {
        d += 2.0;
        ds *= x * x / (d * d);
        sum += ds;
        if (ds <= sum * precision) break;
    }
    return sum;
}

template <class T>
int invert(const GridInputs& i, const GridOutputs& o, double* timings, std::string& err) {
    const auto t_all = Clock::now();
    double t_prepare = 0, t_bucket = 0, t_upload = 0, t_grid = 0, t_fft = 0, t_project = 0, t_download = 0,
           t_finish = 0;
    const std::size_t nrow = i.nrow, nchan = i.nchan;
    const std::size_t n = nrow * nchan;
    const std::size_t W = pad_side(i.width, i.padding), H = pad_side(i.height, i.padding);
    Geo g{int(W), int(H), int(i.kernel_size), int(i.oversampling), int(i.n_w_layers), i.pixel_size_x,
          i.pixel_size_y, 0.0, 0.0};
    hipStream_t st = nullptr;
    WSCHK(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
    struct StreamGuard {
        hipStream_t s;
        ~StreamGuard() { (void)hipStreamDestroy(s); }
    } sg{st};
    Pool& pool = pool_of_current_device();
    std::lock_guard<std::mutex> pool_lock(pool.mu);
    Bufs b(pool);
    // upload
    auto t0 = Clock::now();
    double* d_uvw = b.get<double>(3 * nrow);
    double* d_freq = b.get<double>(nchan);
    float* d_data = b.get<float>(2 * n);
    float* d_wt = b.get<float>(n);
    float* d_iw = b.get<float>(n);
    WSCHK(hipMemcpyAsync(d_uvw, i.uvw, sizeof(double) * 3 * nrow, hipMemcpyHostToDevice, st));
    WSCHK(hipMemcpyAsync(d_freq, i.frequencies, sizeof(double) * nchan, hipMemcpyHostToDevice, st));
    WSCHK(hipMemcpyAsync(d_data, i.data, sizeof(float) * 2 * n, hipMemcpyHostToDevice, st));
    WSCHK(hipMemcpyAsync(d_wt, i.weights, sizeof(float) * n, hipMemcpyHostToDevice, st));
    WSCHK(hipMemcpyAsync(d_iw, i.imaging_weights, sizeof(float) * n, hipMemcpyHostToDevice, st));
    WSCHK(hipStreamSynchronize(st));
    t_upload = since(t0);
    In in{d_uvw, d_freq, d_data, d_wt, d_iw, (long long)n, int(nchan)};
    // w limits
    t0 = Clock::now();
    const int nblk = int(std::max<long long>(1, std::min<long long>(1024, ((long long)n + 255) / 256)));
    double* d_part = b.get<double>(4 * nblk);
    std::vector<double> part(4 * nblk);
    k_limits<<<nblk, 256, 0, st>>>(in, g, d_part);
    WSCHK(hipGetLastError());
    WSCHK(hipMemcpyAsync(part.data(), d_part, sizeof(double) * 2 * nblk, hipMemcpyDeviceToHost, st));
    WSCHK(hipStreamSynchronize(st));
    double min_w = 1e100, max_w = 0.0;
    for (int k = 0; k < nblk; ++k) {
        min_w = std::min(min_w, part[2 * k]);
        max_w = std::max(max_w, part[2 * k + 1]);
    }
    if (min_w == 1e100) min_w = max_w = 0.0;
    g.min_w = min_w;
    g.max_w = min_w == max_w ? max_w + 1.0 : max_w;
    // layers and counters
    int* d_keys = b.get<int>(n);
    k_keys<<<nblk, 256, 0, st>>>(in, g, d_keys, d_part);
    WSCHK(hipGetLastError());
    WSCHK(hipMemcpyAsync(part.data(), d_part, sizeof(double) * 4 * nblk, hipMemcpyDeviceToHost, st));
    const int L = int(i.n_w_layers);
    if (std::size_t(L) * sizeof(unsigned) > 64 * 1024) throw Fail{1, "too many w-layers for the GPU sort"};
    unsigned* d_cnt = b.get<unsigned>(L);
    clear(d_cnt, sizeof(unsigned) * L, st);
    k_hist<<<nblk, 256, sizeof(unsigned) * L, st>>>(d_keys, (long long)n, L, d_cnt);
    WSCHK(hipGetLastError());
    std::vector<unsigned> cnt(L);
    WSCHK(hipMemcpyAsync(cnt.data(), d_cnt, sizeof(unsigned) * L, hipMemcpyDeviceToHost, st));
    WSCHK(hipStreamSynchronize(st));
    double image_weight = 0, vsum = 0, gridded = 0, maxw = 0;
    for (int k = 0; k < nblk; ++k) {
        image_weight += part[4 * k];
        vsum += part[4 * k + 1];
        gridded += part[4 * k + 2];
        maxw = std::max(maxw, part[4 * k + 3]);
    }
    if (image_weight == 0.0) throw Fail{1, "no visibility carries weight"};
    t_bucket = since(t0);
    t_prepare = t_bucket;
    // kernels (grid.rs:165-202)
    const std::size_t ks = i.kernel_size, os = i.oversampling, klen = ks * os, mid = klen / 2;
    std::vector<double> k1(klen), kern(klen);
    {
        const double fr = 1.0 / double(os), norm = double(os) / bessel0(8.6, 1e-8);
        for (std::size_t q = 0; q <= mid && mid + q < klen; ++q) {
            const double x = double(q);
            const double sn = q == 0 ? fr : std::sin(M_PI * fr * x) / (M_PI * x);
            const double t = double(q) / double(mid);
            k1[mid + q] = sn * bessel0(8.6 * std::sqrt(1.0 - t * t), 1e-8) * norm;
        }
        for (std::size_t q = 0; q < mid; ++q) k1[q] = k1[klen - 1 - q];
        for (std::size_t s = 0; s < os; ++s)
            for (std::size_t x = 0; x < ks; ++x) kern[(os - s - 1) * ks + x] = k1[x * os + s];
    }
    double* d_kern = b.get<double>(klen);
    WSCHK(hipMemcpyAsync(d_kern, kern.data(), sizeof(double) * klen, hipMemcpyHostToDevice, st));
    // backward transforms along x (rows of W) and y (columns of H): in LDS
    // where the side allows, else in four steps or by Bluestein (ws_fft.h)
    std::vector<std::vector<cx<T>>> keep;
    LineFft<T> fx, fy;
    fx.setup(int(W), +1, b, st, keep);
    fy.setup(int(H), +1, b, st, keep);
    const int Cw = std::max(1, std::min(8, 8192 / int(H)));
    // columns in place in LDS blocks when H is a good size there; otherwise
    // each layer is transposed so that its columns become lines
    const bool cols_direct = fy.kind == 0 && int(H) * Cw <= lds_values<T>();
    WSCHK(hipStreamSynchronize(st));
    // batches of the layers holding samples
    std::vector<int> layers;
    for (std::size_t l = 0; l < i.n_w_layers; ++l)
        if (cnt[l]) layers.push_back(int(l));
    const long long plane = (long long)W * H;
    // a layer's dirty and PSF grids, plus a transposed copy of one grid when
    // the columns are not transformed in place
    const std::size_t per_layer = (cols_direct ? 2 : 3) * sizeof(cx<T>) * std::size_t(plane);
    const std::size_t budget = std::size_t(4) << 30;
    const int batch = int(std::max<std::size_t>(1, std::min<std::size_t>(layers.size(), budget / per_layer)));
    cx<T>* d_gd = b.get<cx<T>>(std::size_t(batch) * plane);
    cx<T>* d_gp = b.get<cx<T>>(std::size_t(batch) * plane);
    cx<T>* d_tr = cols_direct ? nullptr : b.get<cx<T>>(std::size_t(batch) * plane);
    // work space of the four-step and chirp transforms: at most 1 GiB
    const long long per_line = std::max(fx.scratch_per_line(), fy.scratch_per_line());
    const long long scratch_values =
        per_line ? std::max<long long>(per_line, std::min<long long>((1LL << 30) / sizeof(cx<T>),
                                                                     per_line * std::max<long long>(W, H) * batch))
                 : 0;
    cx<T>* d_fs = per_line ? b.get<cx<T>>(std::size_t(scratch_values)) : nullptr;
    double* d_sd = b.get<double>(plane);
    double* d_sp = b.get<double>(plane);
    clear(d_sd, sizeof(double) * plane, st);
    clear(d_sp, sizeof(double) * plane, st);
    // the tiled gridding's buckets, for the batch with the most samples
    const int tile = ks > std::size_t(kTile) ? 0 : tile_side(int(W), int(H), int(ks), batch);
    Tiling tl{tile, 0, 0, 0};
    unsigned *d_bkey = nullptr, *d_bcnt = nullptr, *d_boff = nullptr, *d_item = nullptr, *d_ioff = nullptr, *d_sum = nullptr;
    Rec* d_rec = nullptr;
    if (tile) {
        tl.ntx = (int(W) + tile - 1) / tile;
        tl.nty = (int(H) + tile - 1) / tile;
        std::size_t most = 1;
        for (std::size_t l0 = 0; l0 < layers.size(); l0 += batch) {
            std::size_t ns = 0;
            for (std::size_t q = l0; q < std::min(layers.size(), l0 + batch); ++q) ns += cnt[layers[q]];
            most = std::max(most, ns);
        }
        const std::size_t units = std::size_t(batch) * tl.tiles();
        d_bkey = b.get<unsigned>(n);
        d_bcnt = b.get<unsigned>(4 * units + 1);
        d_boff = b.get<unsigned>(4 * units + 1);
        d_item = b.get<unsigned>(units + 1);
        d_ioff = b.get<unsigned>(units + 1);
        d_sum = b.get<unsigned>(2 * (4 * units / kScan + 64));
        d_rec = b.get<Rec>(most);
    }
    int* d_slot = b.get<int>(i.n_w_layers);
    double* d_wl = b.get<double>(batch);
    std::vector<int> slot(i.n_w_layers, -1);
    std::vector<double> wl(batch);
    const int ncb = (int(W) + Cw - 1) / Cw;
    int nbatches = 0;
    for (std::size_t l0 = 0; l0 < layers.size(); l0 += batch) {
        const std::size_t l1 = std::min(layers.size(), l0 + batch);
        const int nb = int(l1 - l0);
        std::fill(slot.begin(), slot.end(), -1);
        for (std::size_t q = l0; q < l1; ++q) {
            slot[layers[q]] = int(q - l0);
            const int L = layers[q];
            // LayerToW (grid.rs:354-361)
            wl[q - l0] = i.n_w_layers == 1 ? 0.0 : double(L) * (g.max_w - g.min_w) / double(i.n_w_layers - 1) + g.min_w;
        }
        WSCHK(hipMemcpyAsync(d_slot, slot.data(), sizeof(int) * i.n_w_layers, hipMemcpyHostToDevice, st));
        WSCHK(hipMemcpyAsync(d_wl, wl.data(), sizeof(double) * nb, hipMemcpyHostToDevice, st));
        auto tg = Clock::now();
        if (tile) {
            tl.nb = nb;
            const long long units = (long long)nb * tl.tiles(), nkeys = 4 * units;
            const unsigned blocks = unsigned(std::min<long long>(((long long)n + 255) / 256, 1LL << 22));
            clear(d_bcnt, sizeof(unsigned) * (nkeys + 1), st);
            k_bucket<<<blocks, 256, 0, st>>>(in, g, tl, d_keys, d_slot, d_bkey, d_bcnt);
            exclusive_scan(d_bcnt, d_boff, nkeys + 1, d_sum, st);
            clear(d_bcnt, sizeof(unsigned) * (nkeys + 1), st);
            k_bucket_scatter<<<blocks, 256, 0, st>>>(in, g, d_bkey, d_boff, d_bcnt, d_rec);
            k_items<<<unsigned((units + 256) / 256), 256, 0, st>>>(tl, d_boff, d_item);
            exclusive_scan(d_item, d_ioff, units + 1, d_sum, st);
            k_clear<T><<<unsigned(units), 256, 0, st>>>(tl, g, d_ioff, d_gd, d_gp);
            WSCHK(hipGetLastError());
            long long ns = 0;
            for (std::size_t q = l0; q < l1; ++q) ns += cnt[layers[q]];
            // a sample reaches at most four tiles; workgroups past the last
            // item end at once
            const long long items = units + 4 * ns / kChunk;
            if (items * 256 >= (1LL << 32)) throw Fail{1, "too many samples for one gridding launch"};
            if (ks == 7)
                k_grid_tile<T, 7><<<unsigned(items), 256, 0, st>>>(d_rec, d_boff, d_ioff, tl, g, d_kern, d_gd, d_gp);
            else
                k_grid_tile<T, 0><<<unsigned(items), 256, 0, st>>>(d_rec, d_boff, d_ioff, tl, g, d_kern, d_gd, d_gp);
            WSCHK(hipGetLastError());
        } else {
            clear(d_gd, sizeof(cx<T>) * nb * plane, st);
            clear(d_gp, sizeof(cx<T>) * nb * plane, st);
            k_grid_any<T><<<unsigned(std::min<long long>(((long long)n + 3) / 4, 1LL << 22)), 256, 0, st>>>(
                in, g, d_keys, d_slot, d_kern, d_gd, d_gp);
            WSCHK(hipGetLastError());
        }
        WSCHK(hipStreamSynchronize(st));
        t_grid += since(tg);
        tg = Clock::now();
        for (cx<T>* grid : {d_gd, d_gp}) {
            fx.apply(grid, (long long)nb * H, d_fs, scratch_values, st);
            if (cols_direct) {
                fft_sizes<T>(int(H) * Cw, [&](auto nt, auto mt) {
                    constexpr int NT = decltype(nt)::value, MT = decltype(mt)::value;
                    set_lds(k_cols<T, NT, MT>, sizeof(cx<T>) * H * Cw);
                    k_cols<T, NT, MT><<<nb * ncb, NT, sizeof(cx<T>) * H * Cw, st>>>(grid, fy.d, fy.tw, int(W), Cw,
                                                                                   ncb);
                });
                WSCHK(hipGetLastError());
            } else {
                LineFft<T>::transpose(grid, d_tr, nb, int(H), int(W), st);
                fy.apply(d_tr, (long long)nb * W, d_fs, scratch_values, st);
                LineFft<T>::transpose(d_tr, grid, nb, int(W), int(H), st);
            }
        }
        WSCHK(hipStreamSynchronize(st));
        t_fft += since(tg);
        tg = Clock::now();
        k_project<T><<<(plane + 255) / 256, 256, 0, st>>>(d_gd, d_gp, nb, d_wl, g, d_sd, d_sp);
        WSCHK(hipGetLastError());
        WSCHK(hipStreamSynchronize(st));
        t_project += since(tg);
        ++nbatches;
    }
    // normalise, correct, trim (grid.rs:597-650, 837-873)
    t0 = Clock::now();
    const std::size_t half = klen / 2, rlen = klen / 2 + 1;
    double* d_k1 = b.get<double>(rlen);
    WSCHK(hipMemcpyAsync(d_k1, k1.data() + half, sizeof(double) * rlen, hipMemcpyHostToDevice, st));
    double* d_ox = b.get<double>(W / 2 + 1);
    k_dct3<<<int(W / 2 + 1), 256, 0, st>>>(d_k1, int(rlen), double(W * os / 2), d_ox);
    WSCHK(hipGetLastError());
    double* d_oy = d_ox;
    if (H != W) {
        d_oy = b.get<double>(H / 2 + 1);
        k_dct3<<<int(H / 2 + 1), 256, 0, st>>>(d_k1, int(rlen), double(H * os / 2), d_oy);
        WSCHK(hipGetLastError());
    }
    const std::size_t npix = i.width * i.height;
    double* d_od = b.get<double>(npix);
    double* d_op = b.get<double>(npix);
    k_finish<<<(npix + 255) / 256, 256, 0, st>>>(d_sd, d_sp, g, 1.0 / image_weight, d_ox, d_oy, int(i.width),
                                                 int(i.height), d_od, d_op);
    WSCHK(hipGetLastError());
    const std::size_t centre = i.width / 2 + (i.height / 2) * i.width;
    double peak = 0.0;
    WSCHK(hipMemcpyAsync(&peak, d_op + centre, sizeof(double), hipMemcpyDeviceToHost, st));
    WSCHK(hipStreamSynchronize(st));
    const double pn = peak != 0.0 ? 1.0 / peak : 0.0;
    k_normalise<<<unsigned((npix + 255) / 256), 256, 0, st>>>(d_od, d_op, pn, (long long)npix);
    WSCHK(hipGetLastError());
    t_finish = since(t0);
    t0 = Clock::now();
    WSCHK(hipMemcpyAsync(o.dirty, d_od, sizeof(double) * npix, hipMemcpyDeviceToHost, st));
    WSCHK(hipMemcpyAsync(o.psf, d_op, sizeof(double) * npix, hipMemcpyDeviceToHost, st));
    WSCHK(hipStreamSynchronize(st));
    t_download = since(t0);
    const double stats[8] = {image_weight, gridded, vsum, maxw, min_w, max_w, pn, double(i.n_w_layers)};
    std::memcpy(o.stats, stats, sizeof(stats));
    if (timings) {
        const double total = since(t_all);
        // the order of Timings::as_array (core/src/gpu/invert.rs:57-74)
        const double tm[14] = {0.0,
                               0.0,
                               t_prepare,
                               t_upload,
                               total - t_upload - t_prepare - t_download - t_finish,
                               t_download,
                               t_finish,
                               double(b.bytes),
                               double(nbatches),
                               double(batch),
                               t_grid,
                               t_fft,
                               t_project,
                               t_bucket};
        std::memcpy(timings, tm, sizeof(tm));
    }
    return 0;
}

}  // namespace

int invert_gpu(const GridInputs& i, const GridOutputs& o, bool single, double* timings, std::string& err) {
    try {
        return single ? invert<float>(i, o, timings, err) : invert<double>(i, o, timings, err);
    } catch (const Fail& f) {
        err = f.msg;
        return f.status;
    }
}

int kernel(std::size_t ks, std::size_t os, double* out) {
    const std::size_t n = ks * os, mid = n / 2;
    const double fr = 1.0 / double(os), norm = double(os) / bessel0(8.6, 1e-8);
    for (std::size_t q = 0; q <= mid && mid + q < n; ++q) {
        const double x = double(q);
        const double sn = q == 0 ? fr : std::sin(M_PI * fr * x) / (M_PI * x);
        const double t = double(q) / double(mid);
        out[mid + q] = sn * bessel0(8.6 * std::sqrt(1.0 - t * t), 1e-8) * norm;
    }
    for (std::size_t q = 0; q < mid; ++q) out[q] = out[n - 1 - q];
    return 0;
}

}  // namespace ws
}  // namespace rang
