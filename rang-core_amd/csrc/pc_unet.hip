// Kernels of the learned preconditioner: a small U-Net in BF16 with FP32
// accumulation on the matrix cores (gfx950), for inference and training, and
// the vector kernels of flexible conjugate gradients. The reference has no
// counterpart; the network's graph is assembled by the caller over the C ABI
// of include/rang_core_precond.h.
//
// Tensors are NHWC: pixel p = (n H + h) W + w, channel c at p * ld + off + c,
// so a concatenation along channels is two writers into one buffer with
// different offsets. Activations and gradients that feed the matrix cores
// are BF16 (round to nearest even); pre-activations, gradients being summed
// and the master weights are FP32.
//
// A 3 x 3 convolution is an implicit GEMM on v_mfma_f32_16x16x32_bf16 with the
// image tile and its halo in LDS (k_conv3_fwd, k_conv_wgrad below); the 1 x 1
// output convolution, which only streams its tensors, and layers too small for
// the tiles take per-wave kernels on v_mfma_f32_16x16x16_bf16 (16 pixels x 32
// output channels, operands read from memory). Channel counts are multiples of 16 (callers pad the first and
// last layers).

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <map>
#include <mutex>
#include <string>
#include <utility>

#include "../../include/rang_core_precond.h"

namespace rang {
namespace {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

thread_local std::string g_nn_err;

int nn_fail(hipError_t e) {
    if (e == hipSuccess) return 0;
    g_nn_err = hipGetErrorString(e);
    return 2;
}

__device__ __forceinline__ std::uint16_t to_bf16(float f) {
    std::uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return std::uint16_t((u >> 16) | 0x40u);  // NaN stays NaN
    u += 0x7fffu + ((u >> 16) & 1u);
    return std::uint16_t(u >> 16);
}

__device__ __forceinline__ float from_bf16(std::uint16_t b) { return __uint_as_float(std::uint32_t(b) << 16); }

// Four consecutive BF16 values (8 bytes, aligned when the channel offset and
// stride are multiples of 4) or zeros.
__device__ __forceinline__ bf16x4 load4(const std::uint16_t* p, bool ok) {
    if (!ok) return bf16x4{0, 0, 0, 0};
    const uint2 v = *reinterpret_cast<const uint2*>(p);
    bf16x4 r;
    r[0] = short(v.x & 0xffffu);
    r[1] = short(v.x >> 16);
    r[2] = short(v.y & 0xffffu);
    r[3] = short(v.y >> 16);
    return r;
}

// y = conv(x, w) over B images of H x W: w as [cout][ks * ks][cin] BF16; the
// FP32 result into y (pre-activation, may be null) and BF16 relu(y) (or y
// when relu is 0) into a (may be null). Block: 4 waves, 64 pixels x 32 output
// channels, every operand read from memory: for 1 x 1 and for small 3 x 3
// convolutions (small_fwd). A row = pixel (lane mod 16), k = 4 consecutive input
// channels per lane group (lane / 16); B column = output channel, the same k
// split; D column = output channel (lane mod 16), rows 4 (lane / 16) + t.
template <int KS>
__global__ __launch_bounds__(256) void k_conv_fwd_wave(const std::uint16_t* __restrict__ x, int ldx, int xoff,
                                                       const std::uint16_t* __restrict__ w, float* __restrict__ y,
                                                       std::uint16_t* __restrict__ a, int ldy, int yoff, int B,
                                                       int H, int W, int cin, int cout, int relu) {
    const long long npix = (long long)B * H * W;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const long long p0 = (long long)blockIdx.x * 64 + wave * 16;
    const int co0 = blockIdx.y * 32;
    const int row = lane & 15, q = lane >> 4;
    // this lane's A pixel
    const long long pa = p0 + row;
    int n = 0, h = 0, wc = 0;
    if (pa < npix) {
        n = int(pa / ((long long)H * W));
        const int r = int(pa - (long long)n * H * W);
        h = r / W;
        wc = r - h * W;
    }
    f32x4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
    constexpr int T = KS * KS;
    for (int tap = 0; tap < T; ++tap) {
        const int dy = KS == 3 ? tap / 3 - 1 : 0, dx = KS == 3 ? tap % 3 - 1 : 0;
        const int hh = h + dy, ww = wc + dx;
        const bool in = pa < npix && hh >= 0 && hh < H && ww >= 0 && ww < W;
        const long long src = ((long long)n * H + hh) * W + ww;
        const std::uint16_t* xa = x + src * ldx + xoff + 4 * q;
        const std::uint16_t* wb0 = w + ((long long)(co0 + row) * T + tap) * cin + 4 * q;
        const std::uint16_t* wb1 = w + ((long long)(co0 + 16 + row) * T + tap) * cin + 4 * q;
        for (int c0 = 0; c0 < cin; c0 += 16) {
            const bf16x4 av = load4(xa + c0, in);
            const bf16x4 b0 = load4(wb0 + c0, true);
            const bf16x4 b1 = load4(wb1 + c0, co0 + 16 < cout);
            acc0 = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av, b0, acc0, 0, 0, 0);
            acc1 = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av, b1, acc1, 0, 0, 0);
        }
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const long long p = p0 + 4 * q + t;
        if (p >= npix) continue;
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            const int co = co0 + 16 * half + row;
            if (co >= cout) continue;
            const float v = half ? acc1[t] : acc0[t];
            const long long at = p * ldy + yoff + co;
            if (y) y[at] = v;
            if (a) a[at] = to_bf16(relu ? fmaxf(v, 0.f) : v);
        }
    }
}

// dw += sum over pixels of dy (x) the shifted input, dw as [cout][ks * ks][cin]
// FP32: a GEMM over pixels (16 per MFMA) for one (16 cout, tap, 16 cin)
// tile per wave; each block sums a chunk of pixels and adds its tile. For few
// pixels (small_wgrad).
template <int KS>
__global__ __launch_bounds__(256) void k_conv_wgrad_wave(const std::uint16_t* __restrict__ x, int ldx, int xoff,
                                                         const std::uint16_t* __restrict__ dy, int lddy, int dyoff,
                                                         float* __restrict__ dw, int B, int H, int W, int cin,
                                                         int cout, long long chunk) {
    constexpr int T = KS * KS;
    const long long npix = (long long)B * H * W;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int nct = cin / 16, ncot = cout / 16;
    const int tile = blockIdx.x * 4 + wave;  // (cout tile, tap, cin tile)
    if (tile >= ncot * T * nct) return;
    const int cot = tile / (T * nct), rem = tile - cot * T * nct;
    const int tap = rem / nct, ct = rem - tap * nct;
    const int ddy = KS == 3 ? tap / 3 - 1 : 0, ddx = KS == 3 ? tap % 3 - 1 : 0;
    const int row = lane & 15, q = lane >> 4;
    const long long pbeg = (long long)blockIdx.y * chunk, pend = pbeg + chunk < npix ? pbeg + chunk : npix;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (long long pb = pbeg; pb < pend; pb += 16) {
        bf16x4 av, bv;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const long long p = pb + 4 * q + t;
            short va = 0, vb = 0;
            if (p < pend) {
                va = short(dy[p * lddy + dyoff + cot * 16 + row]);
                const int n = int(p / ((long long)H * W));
                const int r = int(p - (long long)n * H * W);
                const int hh = r / W + ddy, ww = r % W + ddx;
                if (hh >= 0 && hh < H && ww >= 0 && ww < W)
                    vb = short(x[(((long long)n * H + hh) * W + ww) * ldx + xoff + ct * 16 + row]);
            }
            av[t] = va;
            bv[t] = vb;
        }
        acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av, bv, acc, 0, 0, 0);
    }
    // D row = cout within the tile (4 q + t), column = cin within the tile (row)
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const int co = cot * 16 + 4 * q + t, ci = ct * 16 + row;
        atomicAdd(&dw[((long long)co * T + tap) * cin + ci], acc[t]);
    }
}

// Eight consecutive BF16 values in accesses of `unit` values (8, 4 or 1, uniform:
// unit_of), as the tensor's base, stride and offset allow.
__device__ __forceinline__ uint4 load8(const std::uint16_t* p, int unit) {
    if (unit == 8) return *reinterpret_cast<const uint4*>(p);
    if (unit == 4) {
        const uint2 a = *reinterpret_cast<const uint2*>(p), b = *reinterpret_cast<const uint2*>(p + 4);
        return make_uint4(a.x, a.y, b.x, b.y);
    }
    std::uint32_t r[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) r[k] = p[2 * k] | (std::uint32_t(p[2 * k + 1]) << 16);
    return make_uint4(r[0], r[1], r[2], r[3]);
}

__device__ __forceinline__ bf16x8 as_bf16x8(uint4 v) { return __builtin_bit_cast(bf16x8, v); }

// 3 x 3 convolution, zero padding: y (FP32, may be null) and a (BF16 relu(y),
// or y when relu is 0; may be null) of B images of H x W.
//
// A workgroup of four waves takes 32 columns by 16 rows and 32 output channels
// (WCO 1) or by 8 rows and 64 output channels (WCO 2). Per block of 32 (or the
// last 16) input channels the tile and its one-pixel halo and the block's
// weights are staged in LDS; a wave computes 8 rows x 16 columns x 32 output
// channels in 16 result tiles of v_mfma_f32_16x16x32_bf16 (rows: output
// channels, columns: 16 pixels along w, k: 32 input channels, or 16 of two
// neighbouring taps in a block of 16). A pixel fragment of image row r serves
// the three output rows r, r - 1, r - 2, so a step of 3 dy taps reads 10
// pixel and 6 weight fragments for 48 products (85 bytes of LDS per clock of
// the 128 a CU delivers).
// Pixels lie 80 bytes apart in LDS (64 and a pad): the 16 lanes of a 16-byte
// read then cover all 64 banks. Result rows are consecutive output channels
// of one pixel, stored 16 bytes (FP32) and 8 bytes (BF16) a lane.
// Measured (four 1024^2 images, four levels of 32 channels and up, forward
// and data gradients, 27 launches): 46.6 ms -> 7.2 ms; the per-wave kernel
// before it read each pixel nine times from memory through the caches, and
// the 32-channel layers are now bound by their tensors' bytes.
constexpr int kConvCols = 32;
constexpr int kConvPixel = 5;  // 16-byte units per staged pixel
template <int WCO>
struct Conv3Tile {
    static constexpr int rows = WCO == 1 ? 16 : 8;
    static constexpr int co = 32 * WCO;
    static constexpr int pixels = (rows + 2) * (kConvCols + 2);
    static constexpr std::size_t lds = std::size_t(16) * (pixels * kConvPixel + 36 * co);
};

// The products of one staged block of CB (32 or 16) input channels.
template <int WCO, int CB>
__device__ __forceinline__ void conv3_block(const uint4* sx, const uint4* sw, int rowbase, int colbase, int cobase,
                                            int l16, int q, f32x4 (&acc)[8][2]) {
    constexpr int CO = Conv3Tile<WCO>::co;
    constexpr int steps = CB == 32 ? 3 : 2, noct = CB / 8;
#pragma unroll
    for (int s = 0; s < steps; ++s) {
        // this lane group's tap column and channel octet
        int dx = CB == 32 ? s : 2 * s + (q >> 1);
        const int oct = CB == 32 ? q : (q & 1);
        const bool valid = dx < 3;
        dx = valid ? dx : 2;
        bf16x8 wf[3][2];
#pragma unroll
        for (int dy = 0; dy < 3; ++dy)
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                uint4 v = sw[((dy * 3 + dx) * noct + oct) * CO + cobase + 16 * c + l16];
                if (CB == 16 && !valid) v = make_uint4(0u, 0u, 0u, 0u);
                wf[dy][c] = as_bf16x8(v);
            }
        const uint4* px = sx + ((rowbase * (kConvCols + 2)) + colbase + l16 + dx) * kConvPixel + oct;
#pragma unroll
        for (int r = 0; r < 10; ++r) {
            uint4 v = px[r * (kConvCols + 2) * kConvPixel];
            if (CB == 16 && !valid) v = make_uint4(0u, 0u, 0u, 0u);
            const bf16x8 xf = as_bf16x8(v);
#pragma unroll
            for (int dy = 0; dy < 3; ++dy) {
                const int o = r - dy;
                if (o < 0 || o >= 8) continue;
#pragma unroll
                for (int c = 0; c < 2; ++c)
                    acc[o][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[dy][c], xf, acc[o][c], 0, 0, 0);
            }
        }
    }
}

template <int WCO>
__global__ __launch_bounds__(256, 2) void k_conv3_fwd(const std::uint16_t* __restrict__ x, int ldx, int xoff,
                                                      const std::uint16_t* __restrict__ w, float* __restrict__ y,
                                                      std::uint16_t* __restrict__ a, int ldy, int yoff, int H, int W,
                                                      int cin, int cout, int relu, int nth, int ntw, int unit,
                                                      int out16) {
    using Tile = Conv3Tile<WCO>;
    constexpr int CO = Tile::co, HC = kConvCols + 2;
    extern __shared__ __align__(16) unsigned char conv_smem[];
    uint4* sx = reinterpret_cast<uint4*>(conv_smem);
    uint4* sw = sx + Tile::pixels * kConvPixel;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, q = lane >> 4;
    const int tw = int(blockIdx.x) % ntw, rest = int(blockIdx.x) / ntw;
    const int th = rest % nth, n = rest / nth;
    const int h0 = th * Tile::rows, w0 = tw * kConvCols, co0 = blockIdx.y * CO;
    const std::uint16_t* xi = x + (long long)n * H * W * ldx + xoff;
    const int colbase = (wave & 1) * 16;
    const int rowbase = WCO == 1 ? (wave >> 1) * 8 : 0;
    const int cobase = WCO == 1 ? 0 : (wave >> 1) * 32;
    f32x4 acc[8][2];
#pragma unroll
    for (int o = 0; o < 8; ++o)
#pragma unroll
        for (int c = 0; c < 2; ++c) acc[o][c] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int c0 = 0; c0 < cin; c0 += 32) {
        const int noct = min(32, cin - c0) / 8;  // 4, or 2 in a last block of 16
        __syncthreads();                         // the previous block is consumed
        for (int e = tid; e < Tile::pixels * 4; e += 256) {
            const int px = e >> 2, oct = e & 3;
            const int hh = h0 - 1 + px / HC, ww = w0 - 1 + px % HC;
            uint4 v = make_uint4(0u, 0u, 0u, 0u);
            if (oct < noct && hh >= 0 && hh < H && ww >= 0 && ww < W)
                v = load8(xi + ((long long)hh * W + ww) * ldx + c0 + 8 * oct, unit);
            sx[px * kConvPixel + oct] = v;
        }
        const int per = 9 * noct;  // octets of one output channel
        for (int e = tid; e < per * CO; e += 256) {
            const int co = e / per, t = e - co * per;  // t = tap noct + octet
            const int tap = t / noct, oct = t - tap * noct;
            uint4 v = make_uint4(0u, 0u, 0u, 0u);
            if (co0 + co < cout) v = load8(w + ((long long)(co0 + co) * 9 + tap) * cin + c0 + 8 * oct, unit);
            sw[t * CO + co] = v;
        }
        __syncthreads();
        if (noct == 4)
            conv3_block<WCO, 32>(sx, sw, rowbase, colbase, cobase, l16, q, acc);
        else
            conv3_block<WCO, 16>(sx, sw, rowbase, colbase, cobase, l16, q, acc);
    }
    const int ww = w0 + colbase + l16;
    if (ww >= W) return;
#pragma unroll
    for (int o = 0; o < 8; ++o) {
        const int hh = h0 + rowbase + o;
        if (hh >= H) break;
        const long long p = ((long long)n * H + hh) * W + ww;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const int co = co0 + cobase + 16 * c + 4 * q;
            if (co >= cout) continue;  // cout is a multiple of 16: all four or none
            const f32x4 v = acc[o][c];
            const long long at = p * ldy + yoff + co;
            std::uint16_t h[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) h[t] = to_bf16(relu ? fmaxf(v[t], 0.f) : v[t]);
            if (out16) {
                if (y) *reinterpret_cast<f32x4*>(y + at) = v;
                if (a)
                    *reinterpret_cast<uint2*>(a + at) =
                        make_uint2(h[0] | (std::uint32_t(h[1]) << 16), h[2] | (std::uint32_t(h[3]) << 16));
            } else {
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    if (y) y[at + t] = v[t];
                    if (a) a[at + t] = h[t];
                }
            }
        }
    }
}

// dw[co][tap][ci] += sum over pixels of dy[p][co] x[p + tap][ci] (FP32), for
// KS 3 (zero padding) or 1: a product over pixels.
//
// A workgroup takes 32 WCO output by 32 WCI input channels and runs over its
// share of the tiles of 8 rows x 32 columns. A tile's dy and x (with the
// halo) are staged in LDS transposed, channel by channel along w: a thread
// loads 8 pixels of 8 channels and turns the 8 x 8 block with 32 byte
// permutes, so that 8 consecutive pixels of one channel are 16 contiguous
// bytes, the k operand of v_mfma_f32_16x16x32_bf16. The x operand shifted one
// pixel either way is formed from the row's registers and the two
// neighbouring words by funnel shifts, not read again. A wave holds 32 x 32
// channels of every tap (36 result tiles); where the channels do not occupy
// the eight waves, they split the tile's rows and are summed through LDS at
// the end, one atomic add per weight and workgroup. One workgroup of eight
// waves per CU, not two of four: the FP32 adds of the workgroups' sums are
// most of the error, and half of them give 0.7 of it.
// Measured (four 1024^2 images, four levels of 32 channels and up, 14
// launches): 84.8 ms -> 5.1 ms (4.4 as twice the workgroups, error against 64
// bits of a 32- or 64-channel gradient 4.1e-7 and 2.9e-7 instead of 2.9e-7
// and 2.1e-7); the kernel before it read its operands
// two bytes at a time.
constexpr int kWgRows = 8, kWgThreads = 512;
template <int KS>
struct WgradTile {
    static constexpr int halo = KS / 2;
    static constexpr int xrows = kWgRows + 2 * halo;
    static constexpr int xstride = xrows * 96 + 16;  // bytes per channel: w = 0 at byte 16 of a row
    static constexpr int ystride = kWgRows * 64 + 16;
    static constexpr std::size_t lds(int cib, int cob) {
        const std::size_t tile = std::size_t(cib) * xstride + std::size_t(cob) * ystride;
        const std::size_t sum = std::size_t(KS) * KS * 1024 * 4;  // one 32 x 32 partial sum per tap
        return tile > sum ? tile : sum;
    }
};

// 8 pixels (v[p]) of 8 channels to 8 channels of 8 pixels, 16-byte rows at
// dst + c * stride.
__device__ __forceinline__ void store_turned(const uint4 (&v)[8], unsigned char* dst, int stride) {
    const std::uint32_t* d[8];
#pragma unroll
    for (int p = 0; p < 8; ++p) d[p] = reinterpret_cast<const std::uint32_t*>(&v[p]);
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        // bytes of the low or high half of the two words
        const std::uint32_t sel = (c & 1) ? 0x07060302u : 0x05040100u;
        std::uint32_t o[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) o[k] = __builtin_amdgcn_perm(d[2 * k + 1][c >> 1], d[2 * k][c >> 1], sel);
        *reinterpret_cast<uint4*>(dst + c * stride) = make_uint4(o[0], o[1], o[2], o[3]);
    }
}

template <int KS, int WCO, int WCI>
__global__ __launch_bounds__(kWgThreads, 2) void k_conv_wgrad(const std::uint16_t* __restrict__ x, int ldx, int xoff,
                                                       const std::uint16_t* __restrict__ dy, int lddy, int dyoff,
                                                       float* __restrict__ dw, int H, int W, int cin, int cout,
                                                       int nth, int ntw, int ntiles, int nci, int xunit, int yunit) {
    using Tile = WgradTile<KS>;
    constexpr int T = KS * KS, HALO = Tile::halo, WK = kWgThreads / 64 / (WCO * WCI);
    constexpr int COB = 32 * WCO, CIB = 32 * WCI;
    extern __shared__ __align__(16) unsigned char wg_smem[];
    unsigned char* sx = wg_smem;
    unsigned char* sy = wg_smem + CIB * Tile::xstride;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, q = lane >> 4;
    const int cob = (int(blockIdx.y) / nci) * COB, cib = (int(blockIdx.y) % nci) * CIB;
    const int wco = wave % WCO, wci = (wave / WCO) % WCI, wk = wave / (WCO * WCI);
    f32x4 acc[T][2][2];
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int d = 0; d < 2; ++d) acc[t][c][d] = f32x4{0.f, 0.f, 0.f, 0.f};
    const uint4 zero = make_uint4(0u, 0u, 0u, 0u);
    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const int tw = tile % ntw, rest = tile / ntw;
        const int th = rest % nth, n = rest / nth;
        const int h0 = th * kWgRows, w0 = tw * 32;
        const std::uint16_t* xi = x + (long long)n * H * W * ldx + xoff + cib;
        const std::uint16_t* yi = dy + (long long)n * H * W * lddy + dyoff + cob;
        __syncthreads();  // the previous tile is consumed
        // blocks of 8 pixels x 8 channels: x rows with the halo, then dy rows
        constexpr int XB = Tile::xrows * 4 * (CIB / 8), YB = kWgRows * 4 * (COB / 8);
        for (int e = tid; e < XB + YB; e += kWgThreads) {
            const bool isx = e < XB;
            const int f = isx ? e : e - XB;
            const int no = isx ? CIB / 8 : COB / 8;
            const int oct = f % no, g = f / no;
            const int j = g & 3, r = g >> 2;
            const int hh = h0 + r - (isx ? HALO : 0);
            const int ld = isx ? ldx : lddy;
            const bool live = hh >= 0 && hh < H && (isx ? cib + 8 * oct < cin : cob + 8 * oct < cout);
            const std::uint16_t* src = (isx ? xi : yi) + ((long long)hh * W + w0 + 8 * j) * ld + 8 * oct;
            const int unit = isx ? xunit : yunit;
            uint4 v[8];
#pragma unroll
            for (int p = 0; p < 8; ++p)
                v[p] = live && w0 + 8 * j + p < W ? load8(src + (long long)p * ld, unit) : zero;
            if (isx)
                store_turned(v, sx + 8 * oct * Tile::xstride + r * 96 + 16 + 16 * j, Tile::xstride);
            else
                store_turned(v, sy + 8 * oct * Tile::ystride + r * 64 + 16 * j, Tile::ystride);
        }
        if constexpr (HALO == 1) {
            // the columns w0 - 1 and w0 + 32
            for (int e = tid; e < Tile::xrows * 2 * (CIB / 8); e += kWgThreads) {
                const int oct = e % (CIB / 8), g = e / (CIB / 8);
                const int side = g & 1, r = g >> 1;
                const int hh = h0 + r - 1, ww = side ? w0 + 32 : w0 - 1;
                uint4 v = zero;
                if (hh >= 0 && hh < H && ww >= 0 && ww < W && cib + 8 * oct < cin)
                    v = load8(xi + ((long long)hh * W + ww) * ldx + 8 * oct, xunit);
                const std::uint32_t d[4] = {v.x, v.y, v.z, v.w};
                unsigned char* at = sx + 8 * oct * Tile::xstride + r * 96 + (side ? 80 : 14);
#pragma unroll
                for (int c = 0; c < 8; ++c)
                    *reinterpret_cast<std::uint16_t*>(at + c * Tile::xstride) =
                        std::uint16_t(c & 1 ? d[c >> 1] >> 16 : d[c >> 1] & 0xffffu);
            }
        }
        __syncthreads();
#pragma unroll 1
        for (int hr = wk; hr < kWgRows; hr += WK) {
            bf16x8 yf[2];
#pragma unroll
            for (int c = 0; c < 2; ++c)
                yf[c] = as_bf16x8(*reinterpret_cast<const uint4*>(
                    sy + (32 * wco + 16 * c + l16) * Tile::ystride + hr * 64 + 16 * q));
#pragma unroll
            for (int ddy = 0; ddy < KS; ++ddy)
#pragma unroll
                for (int d = 0; d < 2; ++d) {
                    const unsigned char* row =
                        sx + (32 * wci + 16 * d + l16) * Tile::xstride + (hr + ddy) * 96 + 16 + 16 * q;
                    const uint4 m = *reinterpret_cast<const uint4*>(row);
                    if constexpr (KS == 1) {
                        const bf16x8 xf = as_bf16x8(m);
#pragma unroll
                        for (int c = 0; c < 2; ++c)
                            acc[0][c][d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(yf[c], xf, acc[0][c][d], 0, 0, 0);
                    } else {
                        const std::uint32_t lo = *reinterpret_cast<const std::uint32_t*>(row - 4);
                        const std::uint32_t hi = *reinterpret_cast<const std::uint32_t*>(row + 16);
                        const std::uint32_t s0 = __builtin_amdgcn_alignbit(m.x, lo, 16);
                        const std::uint32_t s1 = __builtin_amdgcn_alignbit(m.y, m.x, 16);
                        const std::uint32_t s2 = __builtin_amdgcn_alignbit(m.z, m.y, 16);
                        const std::uint32_t s3 = __builtin_amdgcn_alignbit(m.w, m.z, 16);
                        const std::uint32_t s4 = __builtin_amdgcn_alignbit(hi, m.w, 16);
                        const bf16x8 xf[3] = {as_bf16x8(make_uint4(s0, s1, s2, s3)), as_bf16x8(m),
                                              as_bf16x8(make_uint4(s1, s2, s3, s4))};
#pragma unroll
                        for (int dx = 0; dx < 3; ++dx)
#pragma unroll
                            for (int c = 0; c < 2; ++c)
                                acc[ddy * 3 + dx][c][d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                                    yf[c], xf[dx], acc[ddy * 3 + dx][c][d], 0, 0, 0);
                    }
                }
        }
    }
    // the waves that split the rows: summed in LDS, wave after wave
    if constexpr (WK > 1) {
        // one 32 x 32 sum at a time per (wco, wci): slots of T * 1024 floats
        float* sum = reinterpret_cast<float*>(wg_smem);
#pragma unroll 1
        for (int grp = 0; grp < WCO * WCI; ++grp) {
#pragma unroll 1
            for (int k = WK - 1; k > 0; --k) {
                __syncthreads();
                if (wave % (WCO * WCI) == grp && wk == k) {
#pragma unroll
                    for (int t = 0; t < T; ++t)
#pragma unroll
                        for (int c = 0; c < 2; ++c)
#pragma unroll
                            for (int d = 0; d < 2; ++d)
                                *reinterpret_cast<f32x4*>(sum + ((t * 4 + c * 2 + d) * 64 + lane) * 4) = acc[t][c][d];
                }
                __syncthreads();
                if (wave % (WCO * WCI) == grp && wk == 0) {
#pragma unroll
                    for (int t = 0; t < T; ++t)
#pragma unroll
                        for (int c = 0; c < 2; ++c)
#pragma unroll
                            for (int d = 0; d < 2; ++d)
                                acc[t][c][d] += *reinterpret_cast<const f32x4*>(
                                    sum + ((t * 4 + c * 2 + d) * 64 + lane) * 4);
                }
            }
        }
        if (wk != 0) return;
    }
    // result row 4 q + t: output channel; column l16: input channel
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int d = 0; d < 2; ++d) {
                const int ci = cib + 32 * wci + 16 * d + l16;
                if (ci >= cin) continue;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const int co = cob + 32 * wco + 16 * c + 4 * q + k;
                    if (co < cout) atomicAdd(&dw[((long long)co * T + t) * cin + ci], acc[t][c][d][k]);
                }
            }
}

// The weights of the data gradient: wt[ci][T - 1 - tap][co] = w[co][tap][ci],
// BF16 from the FP32 master weights.
__global__ __launch_bounds__(256) void k_flip(const float* __restrict__ w, std::uint16_t* __restrict__ wt,
                                              int cin, int cout, int T) {
    const long long n = (long long)cin * cout * T;
    const long long e = (long long)blockIdx.x * 256 + threadIdx.x;
    if (e >= n) return;
    const int co = int(e / ((long long)T * cin));
    const int rem = int(e - (long long)co * T * cin);
    const int tap = rem / cin, ci = rem - tap * cin;
    wt[((long long)ci * T + (T - 1 - tap)) * cout + co] = to_bf16(w[e]);
}

__global__ __launch_bounds__(256) void k_to_bf16(const float* __restrict__ s, std::uint16_t* __restrict__ d,
                                                 long long n) {
    for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < n; e += (long long)gridDim.x * 256)
        d[e] = to_bf16(s[e]);
}

// g (BF16) = d (FP32) times (pre > 0) when pre is given, for C channels at
// stride ld / offset off of each of n pixels; accumulate adds into gacc
// (FP32) first when it is given.
__global__ __launch_bounds__(256) void k_relu_bwd(const float* __restrict__ d, int ldd, int doff,
                                                  const float* __restrict__ pre, int ldp, int poff,
                                                  std::uint16_t* __restrict__ g, int ldg, int goff, long long n,
                                                  int C) {
    const long long tot = n * C;
    for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < tot; e += (long long)gridDim.x * 256) {
        const long long p = e / C;
        const int c = int(e - p * C);
        float v = d[p * ldd + doff + c];
        if (pre && !(pre[p * ldp + poff + c] > 0.f)) v = 0.f;
        g[p * ldg + goff + c] = to_bf16(v);
    }
}

// The four resampling kernels take V channels a thread: 8 (16-byte BF16, two
// 16-byte FP32 accesses) where channel counts, strides, offsets and bases
// allow, else 1. They stream their tensors; one channel a thread left them at
// 2-byte accesses with an integer division each (four 1024^2 images, four
// levels: up 1167 -> 314 us a pass, pool 313 -> 242, pool_bwd 627 -> 392,
// up_bwd 522 -> 517).
template <int V>
struct Bf16s;
template <>
struct Bf16s<1> {
    std::uint16_t v;
    __device__ __forceinline__ void load(const std::uint16_t* p) { v = *p; }
    __device__ __forceinline__ void store(std::uint16_t* p) const { *p = v; }
    __device__ __forceinline__ std::uint16_t get(int) const { return v; }
    __device__ __forceinline__ void set(int, std::uint16_t x) { v = x; }
};
template <>
struct Bf16s<8> {
    typedef std::uint16_t vec __attribute__((ext_vector_type(8)));
    vec v;
    __device__ __forceinline__ void load(const std::uint16_t* p) { v = *reinterpret_cast<const vec*>(p); }
    __device__ __forceinline__ void store(std::uint16_t* p) const { *reinterpret_cast<vec*>(p) = v; }
    __device__ __forceinline__ std::uint16_t get(int i) const { return v[i]; }
    __device__ __forceinline__ void set(int i, std::uint16_t x) { v[i] = x; }
};

template <int V>
struct F32s;
template <>
struct F32s<1> {
    float v;
    __device__ __forceinline__ void load(const float* p) { v = *p; }
    __device__ __forceinline__ void store(float* p) const { *p = v; }
    __device__ __forceinline__ float get(int) const { return v; }
    __device__ __forceinline__ void add(int, float x) { v += x; }
};
template <>
struct F32s<8> {
    f32x4 v[2];
    __device__ __forceinline__ void load(const float* p) {
        v[0] = *reinterpret_cast<const f32x4*>(p);
        v[1] = *reinterpret_cast<const f32x4*>(p + 4);
    }
    __device__ __forceinline__ void store(float* p) const {
        *reinterpret_cast<f32x4*>(p) = v[0];
        *reinterpret_cast<f32x4*>(p + 4) = v[1];
    }
    __device__ __forceinline__ float get(int i) const { return v[i >> 2][i & 3]; }
    __device__ __forceinline__ void add(int i, float x) { v[i >> 2][i & 3] += x; }
};

// 2 x 2 average pooling (H, W even) of C channels: BF16 in, BF16 out.
template <int V>
__global__ __launch_bounds__(256) void k_pool(const std::uint16_t* __restrict__ x, int ldx, int xoff,
                                              std::uint16_t* __restrict__ y, int ldy, int yoff, int B, int H,
                                              int W, int C) {
    const int Ho = H / 2, Wo = W / 2, CV = C / V;
    const long long tot = (long long)B * Ho * Wo * CV;
    for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < tot; e += (long long)gridDim.x * 256) {
        const long long po = e / CV;
        const int c = int(e - po * CV) * V;
        const int n = int(po / ((long long)Ho * Wo));
        const int r = int(po - (long long)n * Ho * Wo);
        const int ho = r / Wo, wo = r - ho * Wo;
        float s[V] = {};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const long long pi = ((long long)n * H + 2 * ho + (k >> 1)) * W + 2 * wo + (k & 1);
            Bf16s<V> t;
            t.load(x + pi * ldx + xoff + c);
#pragma unroll
            for (int i = 0; i < V; ++i) s[i] += from_bf16(t.get(i));
        }
        Bf16s<V> o;
#pragma unroll
        for (int i = 0; i < V; ++i) o.set(i, to_bf16(0.25f * s[i]));
        o.store(y + po * ldy + yoff + c);
    }
}

// The gradient of the pooling: each input pixel gets a quarter of its
// output's gradient, added to g (FP32) at full resolution.
template <int V>
__global__ __launch_bounds__(256) void k_pool_bwd(const float* __restrict__ gy, int ldy, int yoff,
                                                  float* __restrict__ gx, int ldx, int xoff, int B, int H, int W,
                                                  int C) {
    const int CV = C / V;
    const long long tot = (long long)B * H * W * CV;
    for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < tot; e += (long long)gridDim.x * 256) {
        const long long p = e / CV;
        const int c = int(e - p * CV) * V;
        const int n = int(p / ((long long)H * W));
        const int r = int(p - (long long)n * H * W);
        const int h = r / W, w = r - h * W;
        const long long po = ((long long)n * (H / 2) + h / 2) * (W / 2) + w / 2;
        F32s<V> t, o;
        t.load(gy + po * ldy + yoff + c);
        o.load(gx + p * ldx + xoff + c);
#pragma unroll
        for (int i = 0; i < V; ++i) o.add(i, 0.25f * t.get(i));
        o.store(gx + p * ldx + xoff + c);
    }
}

// Nearest 2x upsampling of C channels (BF16) from H/2 x W/2 to H x W.
template <int V>
__global__ __launch_bounds__(256) void k_up(const std::uint16_t* __restrict__ x, int ldx, int xoff,
                                            std::uint16_t* __restrict__ y, int ldy, int yoff, int B, int H, int W,
                                            int C) {
    const int CV = C / V;
    const long long tot = (long long)B * H * W * CV;
    for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < tot; e += (long long)gridDim.x * 256) {
        const long long p = e / CV;
        const int c = int(e - p * CV) * V;
        const int n = int(p / ((long long)H * W));
        const int r = int(p - (long long)n * H * W);
        const int h = r / W, w = r - h * W;
        const long long pi = ((long long)n * (H / 2) + h / 2) * (W / 2) + w / 2;
        Bf16s<V> t;
        t.load(x + pi * ldx + xoff + c);
        t.store(y + p * ldy + yoff + c);
    }
}

// The gradient of the upsampling: each coarse pixel sums its four fine
// pixels' gradients (FP32), written (not added) to gx.
template <int V>
__global__ __launch_bounds__(256) void k_up_bwd(const float* __restrict__ gy, int ldy, int yoff,
                                                float* __restrict__ gx, int ldx, int xoff, int B, int H, int W,
                                                int C) {
    const int Ho = H / 2, Wo = W / 2, CV = C / V;
    const long long tot = (long long)B * Ho * Wo * CV;
    for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < tot; e += (long long)gridDim.x * 256) {
        const long long po = e / CV;
        const int c = int(e - po * CV) * V;
        const int n = int(po / ((long long)Ho * Wo));
        const int r = int(po - (long long)n * Ho * Wo);
        const int ho = r / Wo, wo = r - ho * Wo;
        F32s<V> s{};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const long long pi = ((long long)n * H + 2 * ho + (k >> 1)) * W + 2 * wo + (k & 1);
            F32s<V> t;
            t.load(gy + pi * ldy + yoff + c);
#pragma unroll
            for (int i = 0; i < V; ++i) s.add(i, t.get(i));
        }
        s.store(gx + po * ldx + xoff + c);
    }
}

// Adam on FP32 master weights with the BF16 copy refreshed
// (Kingma and Ba 2015, bias-corrected moments).
__global__ __launch_bounds__(256) void k_adam(float* __restrict__ w, const float* __restrict__ g,
                                              float* __restrict__ m, float* __restrict__ v,
                                              std::uint16_t* __restrict__ wb, long long n, float lr, float b1,
                                              float b2, float eps, float c1, float c2) {
    for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < n; e += (long long)gridDim.x * 256) {
        const float gi = g[e];
        const float mi = b1 * m[e] + (1.f - b1) * gi;
        const float vi = b2 * v[e] + (1.f - b2) * gi * gi;
        m[e] = mi;
        v[e] = vi;
        const float wi = w[e] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
        w[e] = wi;
        if (wb) wb[e] = to_bf16(wi);
    }
}

// Images (B of H x W, FP32 or FP64) as channel `c` of a BF16 tensor scaled
// by s[n] per image, and back: out[n] = scale[n] * channel c.
template <class T>
__global__ __launch_bounds__(256) void k_pack(const T* __restrict__ img, const double* __restrict__ s,
                                              std::uint16_t* __restrict__ x, int ldx, int c, int B, long long hw) {
    const long long tot = (long long)B * hw;
    for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < tot; e += (long long)gridDim.x * 256) {
        const int n = int(e / hw);
        x[e * ldx + c] = to_bf16(float(double(img[e]) * (s ? s[n] : 1.0)));
    }
}

template <class T>
__global__ __launch_bounds__(256) void k_unpack(const float* __restrict__ y, int ldy, int c,
                                                const double* __restrict__ s, T* __restrict__ out, int B,
                                                long long hw) {
    const long long tot = (long long)B * hw;
    for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < tot; e += (long long)gridDim.x * 256) {
        const int n = int(e / hw);
        out[e] = T(double(y[e * ldy + c]) * (s ? s[n] : 1.0));
    }
}

// Per-image sums over hw values: s[n] = sum a b (b null: a a), in double.
template <class T>
__global__ __launch_bounds__(256) void k_image_dot(const T* __restrict__ a, const T* __restrict__ b,
                                                   double* __restrict__ s, long long hw) {
    __shared__ double red[256];
    const int n = blockIdx.y;
    double q = 0.0;
    for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < hw; e += (long long)gridDim.x * 256) {
        const double av = double(a[n * hw + e]);
        q += av * (b ? double(b[n * hw + e]) : av);
    }
    red[threadIdx.x] = q;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if (int(threadIdx.x) < h) red[threadIdx.x] += red[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) atomicAdd(&s[n], red[0]);
}

// The loss's gradient on the output channel: g = (y - t) * inv[n] (FP32, at
// channel c of a tensor of ld channels; the other channels zero) and the
// partial sums of inv[n] (y - t)^2 into loss[0].
__global__ __launch_bounds__(256) void k_loss(const float* __restrict__ y, int ldy, int c,
                                              const float* __restrict__ t, const double* __restrict__ inv,
                                              float* __restrict__ g, int ldg, int B, long long hw,
                                              double* __restrict__ loss) {
    __shared__ double red[256];
    double q = 0.0;
    const long long tot = (long long)B * hw;
    for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < tot; e += (long long)gridDim.x * 256) {
        const int n = int(e / hw);
        const double d = double(y[e * ldy + c]) - double(t[e]);
        for (int k = 0; k < ldg; ++k) g[e * ldg + k] = 0.f;
        g[e * ldg + c] = float(d * inv[n]);
        q += 0.5 * d * d * inv[n];
    }
    red[threadIdx.x] = q;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if (int(threadIdx.x) < h) red[threadIdx.x] += red[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) atomicAdd(loss, red[0]);
}

// Random images for training: per image K Gaussian components of random
// centre, log-uniform width in [wmin, wmax] pixels and amplitude uniform in
// [-1, 1] (or [0, 1] when positive), from a counter-based hash of (seed,
// image, component).
__device__ __forceinline__ std::uint64_t mix64(std::uint64_t z) {
    z += 0x9e3779b97f4a7c15ull;
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
}

__device__ __forceinline__ double unit(std::uint64_t seed, std::uint64_t a, std::uint64_t b, int k) {
    const std::uint64_t h = mix64(seed ^ mix64(a * 0x100000001b3ull + b * 0x2545f4914f6cdd1dull + std::uint64_t(k)));
    return double(h >> 11) * (1.0 / 9007199254740992.0);
}

template <class T>
__global__ __launch_bounds__(256) void k_sky(T* __restrict__ out, int B, int H, int W, int K, double wmin,
                                             double wmax, int positive, std::uint64_t seed) {
    const long long hw = (long long)H * W;
    const long long tot = (long long)B * hw;
    for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < tot; e += (long long)gridDim.x * 256) {
        const int n = int(e / hw);
        const int r = int(e - (long long)n * hw);
        const int h = r / W, w = r - h * W;
        double v = 0.0;
        for (int k = 0; k < K; ++k) {
            const double ch = unit(seed, n, k, 0) * H, cw = unit(seed, n, k, 1) * W;
            const double sw = wmin * exp(unit(seed, n, k, 2) * log(wmax / wmin));
            const double amp = positive ? unit(seed, n, k, 3) : 2.0 * unit(seed, n, k, 3) - 1.0;
            const double dh = h - ch, dw = w - cw;
            const double q = (dh * dh + dw * dw) / (2.0 * sw * sw);
            if (q < 40.0) v += amp * exp(-q);
        }
        out[e] = T(v);
    }
}

// An output gradient from images: g[e * ldg + c] = s[n] img[e] (FP64 to
// FP32), the other channels zero.
__global__ __launch_bounds__(256) void k_grad_images(const double* __restrict__ img, const double* __restrict__ s,
                                                     float* __restrict__ g, int ldg, int c, int B, long long hw) {
    const long long tot = (long long)B * hw;
    for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < tot; e += (long long)gridDim.x * 256) {
        for (int k = 0; k < ldg; ++k) g[e * ldg + k] = 0.f;
        g[e * ldg + c] = float(img[e] * s[e / hw]);
    }
}

// out[n] = s[n] x[n] (FP64 images to FP32).
__global__ __launch_bounds__(256) void k_scale_images(const double* __restrict__ x, const double* __restrict__ s,
                                                      float* __restrict__ out, int B, long long hw) {
    const long long tot = (long long)B * hw;
    for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < tot; e += (long long)gridDim.x * 256)
        out[e] = float(x[e] * s[e / hw]);
}

// y = a x + b y.
template <class T>
__global__ __launch_bounds__(256) void k_axpby(const T* __restrict__ x, T* __restrict__ y, double a, double b,
                                               long long n) {
    for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < n; e += (long long)gridDim.x * 256)
        y[e] = T(a * double(x[e]) + b * double(y[e]));
}

int grid1(long long n) {
    const long long b = (n + 255) / 256;
    return int(b < 1 ? 1 : b > 65536 ? 65536 : b);
}

// Values per access of load8 for a BF16 tensor: 16 or 8 bytes where its base,
// stride and offset are multiples of them, else one value.
int unit_of(const void* p, int ld, int off) {
    const std::uintptr_t at = reinterpret_cast<std::uintptr_t>(p);
    if (at % 16 == 0 && ld % 8 == 0 && off % 8 == 0) return 8;
    if (at % 8 == 0 && ld % 4 == 0 && off % 4 == 0) return 4;
    return 1;
}

// Whether 8 channels from a multiple of 8 can be read in 16-byte accesses.
template <class E>
bool vector8(const E* p, int ld, int off) {
    const int unit = 16 / int(sizeof(E));
    return reinterpret_cast<std::uintptr_t>(p) % 16 == 0 && ld % unit == 0 && off % unit == 0;
}

// Lets `kernel` take `bytes` of dynamic LDS on this device, once.
int lds_once(const void* kernel, std::size_t bytes) {
    static std::mutex mu;
    static std::map<std::pair<int, const void*>, std::size_t> done;
    int dev = 0;
    if (const int e = nn_fail(hipGetDevice(&dev))) return e;
    std::lock_guard<std::mutex> lk(mu);
    std::size_t& had = done[{dev, kernel}];
    if (had >= bytes) return 0;
    if (const int e = nn_fail(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, int(bytes))))
        return e;
    had = bytes;
    return 0;
}

// Workgroups of the tiled forward product, without the output channels.
template <int WCO>
long long conv3_tiles(int B, int H, int W) {
    const int rows = Conv3Tile<WCO>::rows;
    return (long long)B * ((H + rows - 1) / rows) * ((W + kConvCols - 1) / kConvCols);
}
long long wgrad_tiles(int B, int H, int W) {
    return (long long)B * ((H + kWgRows - 1) / kWgRows) * ((W + 31) / 32);
}

// Whether a layer goes to the per-wave kernels: few workgroups of tiles take
// several times the few microseconds of a launch, the more so where the image
// fills little of its tiles. Measured, per wave / in tiles, us. Forward: 32 -> 32
// channels of 16384 pixels 6.4 / 11.3, 96 -> 32 12.6 / 22.5, 64 -> 64 (2^26
// products a tap) equal; 512 images of 2 x 2, 256 -> 256, 40 / 171, of 4 x 4 172 /
// 176. Weight gradient: 32 x 32 channels of 4096 pixels 10 / 18, 96 x 32 18.2 /
// 18.4, 256 x 256 of 64 pixels 9.8 / 20.4, of 512 images of 2 x 2 125 / 279; 1 x 1:
// 2048 pixels 4.7 / 5.4, 4096 9.0 / 5.2.
bool small_fwd(int B, int H, int W, int cin, int cout) {
    const double npix = double(B) * H * W;
    const double tiled = cout % 64 == 0 ? 256.0 * conv3_tiles<2>(B, H, W) : 512.0 * conv3_tiles<1>(B, H, W);
    return npix * cin * cout < 67108864.0 * (1.0 + tiled / npix / 16.0);
}
bool small_wgrad(int B, int H, int W, int cin, int cout, int ks) {
    const double npix = double(B) * H * W;
    if (ks == 1) return npix <= 2048.0;
    return npix * cin * cout <= 4194304.0 * (2.0 + 256.0 * wgrad_tiles(B, H, W) / npix);
}

template <int WCO>
int32_t conv3_launch(const std::uint16_t* x, int ldx, int xoff, const std::uint16_t* w, float* y, std::uint16_t* a, int ldy,
                            int yoff, int B, int H, int W, int cin, int cout, int relu, int unit, int out16,
                            hipStream_t st) {
    using Tile = Conv3Tile<WCO>;
    const int nth = (H + Tile::rows - 1) / Tile::rows, ntw = (W + kConvCols - 1) / kConvCols;
    const long long blocks = conv3_tiles<WCO>(B, H, W);
    const auto kernel = k_conv3_fwd<WCO>;
    if (const int e = lds_once(reinterpret_cast<const void*>(kernel), Tile::lds)) return e;
    kernel<<<dim3(unsigned(blocks), unsigned((cout + Tile::co - 1) / Tile::co)), 256, Tile::lds, st>>>(
        x, ldx, xoff, w, y, a, ldy, yoff, H, W, cin, cout, relu, nth, ntw, unit, out16);
    return nn_fail(hipGetLastError());
}

template <int KS, int WCO, int WCI>
int32_t wgrad_launch(const std::uint16_t* x, int ldx, int xoff, const std::uint16_t* dy, int lddy, int dyoff, float* dw,
                            int B, int H, int W, int cin, int cout, hipStream_t st) {
    const int nth = (H + kWgRows - 1) / kWgRows, ntw = (W + 31) / 32;
    const long long ntiles = wgrad_tiles(B, H, W);
    const int nco = (cout + 32 * WCO - 1) / (32 * WCO), nci = (cin + 32 * WCI - 1) / (32 * WCI);
    // a workgroup per CU (its LDS), each with its share of the tiles
    const long long want = (256 + nco * nci - 1) / (nco * nci);
    const unsigned nwg = unsigned(ntiles < want ? ntiles : want);
    const std::size_t lds = WgradTile<KS>::lds(32 * WCI, 32 * WCO);
    const auto kernel = k_conv_wgrad<KS, WCO, WCI>;
    if (const int e = lds_once(reinterpret_cast<const void*>(kernel), lds)) return e;
    kernel<<<dim3(nwg, unsigned(nco * nci)), kWgThreads, lds, st>>>(x, ldx, xoff, dy, lddy, dyoff, dw, H, W, cin, cout, nth,
                                                            ntw, int(ntiles), nci, unit_of(x, ldx, xoff),
                                                            unit_of(dy, lddy, dyoff));
    return nn_fail(hipGetLastError());
}

}  // namespace
}  // namespace rang

using namespace rang;

extern "C" {

size_t rang_amd_nn_last_error(uint8_t* buf, size_t len) {
    const std::string& e = g_nn_err;
    if (!buf || len == 0) return e.size();
    const size_t n = e.size() < len ? e.size() : len;
    for (size_t i = 0; i < n; ++i) buf[i] = uint8_t(e[i]);
    return n;
}

static int conv_args_ok(int ldx, int xoff, int ldy, int yoff, int cin, int cout, int ks) {
    if (ks != 1 && ks != 3) return g_nn_err = "kernel size must be 1 or 3", 1;
    if (cin <= 0 || cout <= 0 || cin % 16 || cout % 16) return g_nn_err = "channel counts must be multiples of 16", 1;
    if (ldx % 4 || xoff % 4 || ldx < xoff + cin || ldy < yoff + cout)
        return g_nn_err = "channel strides must hold the channels, in multiples of 4", 1;
    return 0;
}

int32_t rang_amd_nn_conv_fwd(const uint16_t* x, int32_t ldx, int32_t xoff, const uint16_t* w, float* y,
                             uint16_t* a, int32_t ldy, int32_t yoff, int32_t B, int32_t H, int32_t W,
                             int32_t cin, int32_t cout, int32_t ks, int32_t relu, void* stream) {
    if (const int e = conv_args_ok(ldx, xoff, ldy, yoff, cin, cout, ks)) return e;
    if (!x || !w || (!y && !a) || B <= 0 || H <= 0 || W <= 0) return g_nn_err = "null array or empty image", 1;
    hipStream_t st = static_cast<hipStream_t>(stream);
    // thin images have more tiles than a launch can hold
    const bool many = (cout % 64 == 0 ? conv3_tiles<2>(B, H, W) : conv3_tiles<1>(B, H, W)) >= (1LL << 24);
    if (ks == 1 || many || small_fwd(B, H, W, cin, cout)) {
        const long long npix = (long long)B * H * W;
        const dim3 grid(unsigned((npix + 63) / 64), unsigned((cout + 31) / 32));
        if (ks == 3)
            k_conv_fwd_wave<3><<<grid, 256, 0, st>>>(x, ldx, xoff, w, y, a, ldy, yoff, B, H, W, cin, cout, relu);
        else
            k_conv_fwd_wave<1><<<grid, 256, 0, st>>>(x, ldx, xoff, w, y, a, ldy, yoff, B, H, W, cin, cout, relu);
        return nn_fail(hipGetLastError());
    }
    const int ux = unit_of(x, ldx, xoff), uw = unit_of(w, 8, 0), unit = ux < uw ? ux : uw;
    const int out16 = ldy % 4 == 0 && yoff % 4 == 0 && reinterpret_cast<uintptr_t>(y) % 16 == 0 &&
                      reinterpret_cast<uintptr_t>(a) % 8 == 0;
    // 64 output channels a workgroup where they divide evenly: half the
    // reads of the input
    if (cout % 64 == 0)
        return conv3_launch<2>(x, ldx, xoff, w, y, a, ldy, yoff, B, H, W, cin, cout, relu, unit, out16, st);
    return conv3_launch<1>(x, ldx, xoff, w, y, a, ldy, yoff, B, H, W, cin, cout, relu, unit, out16, st);
}

int32_t rang_amd_nn_conv_wgrad(const uint16_t* x, int32_t ldx, int32_t xoff, const uint16_t* dy, int32_t lddy,
                               int32_t dyoff, float* dw, int32_t B, int32_t H, int32_t W, int32_t cin,
                               int32_t cout, int32_t ks, void* stream) {
    if (const int e = conv_args_ok(ldx, xoff, lddy, dyoff, cin, cout, ks)) return e;
    if (!x || !dy || !dw || B <= 0 || H <= 0 || W <= 0) return g_nn_err = "null array or empty image", 1;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (wgrad_tiles(B, H, W) >= (1LL << 30) || small_wgrad(B, H, W, cin, cout, ks)) {
        const long long npix = (long long)B * H * W;
        const int tiles = (cout / 16) * ks * ks * (cin / 16);
        // pixel chunks: enough blocks to fill the chip, chunks a multiple of 16
        long long nchunk = (2048 + (tiles + 3) / 4 - 1) / ((tiles + 3) / 4);
        if (nchunk < 1) nchunk = 1;
        long long chunk = (npix + nchunk - 1) / nchunk;
        chunk = (chunk + 15) / 16 * 16;
        nchunk = (npix + chunk - 1) / chunk;
        const dim3 grid(unsigned((tiles + 3) / 4), unsigned(nchunk));
        if (ks == 3)
            k_conv_wgrad_wave<3><<<grid, 256, 0, st>>>(x, ldx, xoff, dy, lddy, dyoff, dw, B, H, W, cin, cout, chunk);
        else
            k_conv_wgrad_wave<1><<<grid, 256, 0, st>>>(x, ldx, xoff, dy, lddy, dyoff, dw, B, H, W, cin, cout, chunk);
        return nn_fail(hipGetLastError());
    }
    const bool wo = cout % 64 == 0, wi = cin % 64 == 0;
    if (ks == 3) {
        if (wo && wi) return wgrad_launch<3, 2, 2>(x, ldx, xoff, dy, lddy, dyoff, dw, B, H, W, cin, cout, st);
        if (wo) return wgrad_launch<3, 2, 1>(x, ldx, xoff, dy, lddy, dyoff, dw, B, H, W, cin, cout, st);
        if (wi) return wgrad_launch<3, 1, 2>(x, ldx, xoff, dy, lddy, dyoff, dw, B, H, W, cin, cout, st);
        return wgrad_launch<3, 1, 1>(x, ldx, xoff, dy, lddy, dyoff, dw, B, H, W, cin, cout, st);
    }
    return wgrad_launch<1, 1, 1>(x, ldx, xoff, dy, lddy, dyoff, dw, B, H, W, cin, cout, st);
}

int32_t rang_amd_nn_flip(const float* w, uint16_t* wt, int32_t cin, int32_t cout, int32_t ks, void* stream) {
    if (!w || !wt || cin <= 0 || cout <= 0 || (ks != 1 && ks != 3)) return g_nn_err = "bad weights", 1;
    const long long n = (long long)cin * cout * ks * ks;
    k_flip<<<unsigned((n + 255) / 256), 256, 0, static_cast<hipStream_t>(stream)>>>(w, wt, cin, cout, ks * ks);
    return nn_fail(hipGetLastError());
}

int32_t rang_amd_nn_to_bf16(const float* s, uint16_t* d, int64_t n, void* stream) {
    if (!s || !d || n < 0) return g_nn_err = "null array", 1;
    if (n == 0) return 0;
    k_to_bf16<<<grid1(n), 256, 0, static_cast<hipStream_t>(stream)>>>(s, d, n);
    return nn_fail(hipGetLastError());
}

int32_t rang_amd_nn_relu_bwd(const float* d, int32_t ldd, int32_t doff, const float* pre, int32_t ldp, int32_t poff,
                             uint16_t* g, int32_t ldg, int32_t goff, int64_t npix, int32_t C, void* stream) {
    if (!d || !g || npix < 0 || C <= 0) return g_nn_err = "null array", 1;
    if (npix == 0) return 0;
    k_relu_bwd<<<grid1(npix * C), 256, 0, static_cast<hipStream_t>(stream)>>>(d, ldd, doff, pre, ldp, poff, g, ldg,
                                                                               goff, npix, C);
    return nn_fail(hipGetLastError());
}

int32_t rang_amd_nn_pool(const uint16_t* x, int32_t ldx, int32_t xoff, uint16_t* y, int32_t ldy, int32_t yoff,
                         int32_t B, int32_t H, int32_t W, int32_t C, void* stream) {
    if (!x || !y || H % 2 || W % 2) return g_nn_err = "pooling needs even sides", 1;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (C % 8 == 0 && vector8(x, ldx, xoff) && vector8(y, ldy, yoff))
        k_pool<8><<<grid1((long long)B * H * W * C / 4 / 8), 256, 0, st>>>(x, ldx, xoff, y, ldy, yoff, B, H, W, C);
    else
        k_pool<1><<<grid1((long long)B * H * W * C / 4), 256, 0, st>>>(x, ldx, xoff, y, ldy, yoff, B, H, W, C);
    return nn_fail(hipGetLastError());
}

int32_t rang_amd_nn_pool_bwd(const float* gy, int32_t ldy, int32_t yoff, float* gx, int32_t ldx, int32_t xoff,
                             int32_t B, int32_t H, int32_t W, int32_t C, void* stream) {
    if (!gy || !gx || H % 2 || W % 2) return g_nn_err = "pooling needs even sides", 1;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (C % 8 == 0 && vector8(gy, ldy, yoff) && vector8(gx, ldx, xoff))
        k_pool_bwd<8><<<grid1((long long)B * H * W * C / 8), 256, 0, st>>>(gy, ldy, yoff, gx, ldx, xoff, B, H, W, C);
    else
        k_pool_bwd<1><<<grid1((long long)B * H * W * C), 256, 0, st>>>(gy, ldy, yoff, gx, ldx, xoff, B, H, W, C);
    return nn_fail(hipGetLastError());
}

int32_t rang_amd_nn_up(const uint16_t* x, int32_t ldx, int32_t xoff, uint16_t* y, int32_t ldy, int32_t yoff,
                       int32_t B, int32_t H, int32_t W, int32_t C, void* stream) {
    if (!x || !y || H % 2 || W % 2) return g_nn_err = "upsampling needs even sides", 1;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (C % 8 == 0 && vector8(x, ldx, xoff) && vector8(y, ldy, yoff))
        k_up<8><<<grid1((long long)B * H * W * C / 8), 256, 0, st>>>(x, ldx, xoff, y, ldy, yoff, B, H, W, C);
    else
        k_up<1><<<grid1((long long)B * H * W * C), 256, 0, st>>>(x, ldx, xoff, y, ldy, yoff, B, H, W, C);
    return nn_fail(hipGetLastError());
}

int32_t rang_amd_nn_up_bwd(const float* gy, int32_t ldy, int32_t yoff, float* gx, int32_t ldx, int32_t xoff,
                           int32_t B, int32_t H, int32_t W, int32_t C, void* stream) {
    if (!gy || !gx || H % 2 || W % 2) return g_nn_err = "upsampling needs even sides", 1;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (C % 8 == 0 && vector8(gy, ldy, yoff) && vector8(gx, ldx, xoff))
        k_up_bwd<8><<<grid1((long long)B * H * W * C / 4 / 8), 256, 0, st>>>(gy, ldy, yoff, gx, ldx, xoff, B, H, W, C);
    else
        k_up_bwd<1><<<grid1((long long)B * H * W * C / 4), 256, 0, st>>>(gy, ldy, yoff, gx, ldx, xoff, B, H, W, C);
    return nn_fail(hipGetLastError());
}

int32_t rang_amd_nn_adam(float* w, const float* g, float* m, float* v, uint16_t* wb, int64_t n, double lr, double b1,
                         double b2, double eps, int64_t step, void* stream) {
    if (!w || !g || !m || !v || n < 0 || step < 1) return g_nn_err = "bad optimiser arguments", 1;
    if (n == 0) return 0;
    const double c1 = 1.0 - std::pow(b1, double(step)), c2 = 1.0 - std::pow(b2, double(step));
    k_adam<<<grid1(n), 256, 0, static_cast<hipStream_t>(stream)>>>(w, g, m, v, wb, n, float(lr), float(b1), float(b2),
                                                                   float(eps), float(c1), float(c2));
    return nn_fail(hipGetLastError());
}

int32_t rang_amd_nn_pack_f64(const double* img, const double* s, uint16_t* x, int32_t ldx, int32_t c, int32_t B,
                             int64_t hw, void* stream) {
    if (!img || !x || c < 0 || c >= ldx) return g_nn_err = "bad pack arguments", 1;
    k_pack<double><<<grid1(B * hw), 256, 0, static_cast<hipStream_t>(stream)>>>(img, s, x, ldx, c, B, hw);
    return nn_fail(hipGetLastError());
}

int32_t rang_amd_nn_pack_f32(const float* img, const double* s, uint16_t* x, int32_t ldx, int32_t c, int32_t B,
                             int64_t hw, void* stream) {
    if (!img || !x || c < 0 || c >= ldx) return g_nn_err = "bad pack arguments", 1;
    k_pack<float><<<grid1(B * hw), 256, 0, static_cast<hipStream_t>(stream)>>>(img, s, x, ldx, c, B, hw);
    return nn_fail(hipGetLastError());
}

int32_t rang_amd_nn_unpack_f64(const float* y, int32_t ldy, int32_t c, const double* s, double* out, int32_t B,
                               int64_t hw, void* stream) {
    if (!y || !out || c < 0 || c >= ldy) return g_nn_err = "bad unpack arguments", 1;
    k_unpack<double><<<grid1(B * hw), 256, 0, static_cast<hipStream_t>(stream)>>>(y, ldy, c, s, out, B, hw);
    return nn_fail(hipGetLastError());
}

int32_t rang_amd_nn_unpack_f32(const float* y, int32_t ldy, int32_t c, const double* s, float* out, int32_t B,
                               int64_t hw, void* stream) {
    if (!y || !out || c < 0 || c >= ldy) return g_nn_err = "bad unpack arguments", 1;
    k_unpack<float><<<grid1(B * hw), 256, 0, static_cast<hipStream_t>(stream)>>>(y, ldy, c, s, out, B, hw);
    return nn_fail(hipGetLastError());
}

int32_t rang_amd_nn_image_dot_f64(const double* a, const double* b, double* s, int32_t B, int64_t hw, void* stream) {
    if (!a || !s || B <= 0) return g_nn_err = "bad dot arguments", 1;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (const int e = nn_fail(hipMemsetAsync(s, 0, sizeof(double) * B, st))) return e;
    const dim3 grid(unsigned(grid1(hw) < 256 ? grid1(hw) : 256), unsigned(B));
    k_image_dot<double><<<grid, 256, 0, st>>>(a, b, s, hw);
    return nn_fail(hipGetLastError());
}

int32_t rang_amd_nn_image_dot_f32(const float* a, const float* b, double* s, int32_t B, int64_t hw, void* stream) {
    if (!a || !s || B <= 0) return g_nn_err = "bad dot arguments", 1;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (const int e = nn_fail(hipMemsetAsync(s, 0, sizeof(double) * B, st))) return e;
    const dim3 grid(unsigned(grid1(hw) < 256 ? grid1(hw) : 256), unsigned(B));
    k_image_dot<float><<<grid, 256, 0, st>>>(a, b, s, hw);
    return nn_fail(hipGetLastError());
}

int32_t rang_amd_nn_loss(const float* y, int32_t ldy, int32_t c, const float* t, const double* inv, float* g,
                         int32_t ldg, int32_t B, int64_t hw, double* loss, void* stream) {
    if (!y || !t || !inv || !g || !loss || c < 0 || c >= ldy || c >= ldg) return g_nn_err = "bad loss arguments", 1;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (const int e = nn_fail(hipMemsetAsync(loss, 0, sizeof(double), st))) return e;
    k_loss<<<unsigned(grid1(B * hw) < 1024 ? grid1(B * hw) : 1024), 256, 0, st>>>(y, ldy, c, t, inv, g, ldg, B, hw,
                                                                                   loss);
    return nn_fail(hipGetLastError());
}

int32_t rang_amd_nn_sky_f64(double* out, int32_t B, int32_t H, int32_t W, int32_t K, double wmin, double wmax,
                            int32_t positive, uint64_t seed, void* stream) {
    if (!out || B <= 0 || H <= 0 || W <= 0 || K < 0 || !(wmin > 0.0) || !(wmax >= wmin))
        return g_nn_err = "bad sky arguments", 1;
    k_sky<double><<<grid1((long long)B * H * W), 256, 0, static_cast<hipStream_t>(stream)>>>(out, B, H, W, K, wmin,
                                                                                             wmax, positive, seed);
    return nn_fail(hipGetLastError());
}

int32_t rang_amd_nn_sky_f32(float* out, int32_t B, int32_t H, int32_t W, int32_t K, double wmin, double wmax,
                            int32_t positive, uint64_t seed, void* stream) {
    if (!out || B <= 0 || H <= 0 || W <= 0 || K < 0 || !(wmin > 0.0) || !(wmax >= wmin))
        return g_nn_err = "bad sky arguments", 1;
    k_sky<float><<<grid1((long long)B * H * W), 256, 0, static_cast<hipStream_t>(stream)>>>(out, B, H, W, K, wmin,
                                                                                            wmax, positive, seed);
    return nn_fail(hipGetLastError());
}

int32_t rang_amd_nn_scale_images(const double* x, const double* s, float* out, int32_t B, int64_t hw,
                                 void* stream) {
    if (!x || !s || !out || B <= 0 || hw < 0) return g_nn_err = "bad scale arguments", 1;
    k_scale_images<<<grid1(B * hw), 256, 0, static_cast<hipStream_t>(stream)>>>(x, s, out, B, hw);
    return nn_fail(hipGetLastError());
}

int32_t rang_amd_nn_grad_images(const double* img, const double* s, float* g, int32_t ldg, int32_t c, int32_t B,
                                int64_t hw, void* stream) {
    if (!img || !s || !g || c < 0 || c >= ldg || B <= 0 || hw < 0) return g_nn_err = "bad gradient arguments", 1;
    k_grad_images<<<grid1(B * hw), 256, 0, static_cast<hipStream_t>(stream)>>>(img, s, g, ldg, c, B, hw);
    return nn_fail(hipGetLastError());
}

int32_t rang_amd_nn_axpby_f64(const double* x, double* y, double a, double b, int64_t n, void* stream) {
    if (!x || !y || n < 0) return g_nn_err = "null array", 1;
    if (n == 0) return 0;
    k_axpby<double><<<grid1(n), 256, 0, static_cast<hipStream_t>(stream)>>>(x, y, a, b, n);
    return nn_fail(hipGetLastError());
}

int32_t rang_amd_nn_axpby_f32(const float* x, float* y, double a, double b, int64_t n, void* stream) {
    if (!x || !y || n < 0) return g_nn_err = "null array", 1;
    if (n == 0) return 0;
    k_axpby<float><<<grid1(n), 256, 0, static_cast<hipStream_t>(stream)>>>(x, y, a, b, n);
    return nn_fail(hipGetLastError());
}

}  // extern "C"
