// Batched mixed-radix FFT held in LDS, for the grid transforms of the
// gridder. Lengths are ducc0's good sizes 2^a 3^b 5^c 7^d 11^e
// (core/src/wgridder.rs:185-222); the transform is the unnormalised DFT
// X[k] = sum_j x[j] exp(sgn 2 pi i j k / n), sgn -1 forward, +1 inverse, as
// rustfft's (the reference's FFT, rustfft 6.4.1).
//
// Scheme: Stockham autosort, one pass per radix (3, 5, 7, 11, then 8, 4, 2).
// A workgroup holds `ncol` transforms of length n back to back in LDS; each
// pass reads every value into registers, synchronises and writes the pass's
// output in place, so LDS holds one copy of the data. Twiddles are a per-length
// table in global memory computed on the host in double precision.
#pragma once

#include <type_traits>
#include <hip/hip_runtime.h>

#include <vector>

#include "wg_fft_consts.h"

namespace rang {

constexpr int kFftMaxPass = 24;

// Aligned as a pair, so that a value moves through LDS in one 8- or 16-byte
// access (two 4-byte ones at a stride of 8 bytes use every other bank).
template <class T>
struct alignas(2 * sizeof(T)) cx {
    T re, im;
};

template <class T>
__device__ __forceinline__ cx<T> cmul(cx<T> a, cx<T> b) {
    return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}
template <class T>
__device__ __forceinline__ cx<T> cadd(cx<T> a, cx<T> b) {
    return {a.re + b.re, a.im + b.im};
}
template <class T>
__device__ __forceinline__ cx<T> csub(cx<T> a, cx<T> b) {
    return {a.re - b.re, a.im - b.im};
}
// (SGN i) * a
template <int SGN, class T>
__device__ __forceinline__ cx<T> cmul_si(cx<T> a) {
    return SGN > 0 ? cx<T>{-a.im, a.re} : cx<T>{a.im, -a.re};
}

// Passes of one length: radix, stride Ns before the pass and offset of the
// pass's twiddles (Ns * (R - 1) values: [k * (R - 1) + t - 1] =
// exp(-2 pi i k t / (Ns R))).
struct FftDesc {
    int n = 0;
    int npass = 0;
    int radix[kFftMaxPass] = {};
    int ns[kFftMaxPass] = {};
    int twoff[kFftMaxPass] = {};
    // Multipliers of udiv for d = n / radix and d = ns.
    unsigned mnb[kFftMaxPass] = {};
    unsigned mns[kFftMaxPass] = {};
};

// x / d as the high half of x * ceil(2^32 / d), exact for x, d < 2^16 (every
// index here is below the transform length). d = 1 has no 32-bit multiplier
// (it would be 2^32) and is taken apart.
__host__ __device__ inline unsigned fft_magic(unsigned d) {
    return d <= 1 ? 0u : unsigned(((1ull << 32) + d - 1) / d);
}

__host__ __device__ __forceinline__ unsigned udiv(unsigned x, unsigned d, unsigned m) {
    return d == 1 ? x : unsigned((unsigned long long)x * m >> 32);
}

// Host: exp(-2 pi i m / n) for m < n, computed in extended precision on an
// eighth of the circle (a quarter or half where 4 or 2 are the largest powers
// of two in n) and mirrored to the rest.
inline std::vector<double> fft_roots(int n) {
    std::vector<double> r(std::size_t(2) * n);
    const long double pi = 3.141592653589793238462643383279502884L;
    auto set = [&](int m, double c, double s) {
        r[2 * std::size_t(m)] = c;
        r[2 * std::size_t(m) + 1] = s;
    };
    const int last = n % 8 == 0 ? n / 8 : n % 4 == 0 ? n / 4 : n / 2;
    for (int m = 0; m <= last && m < n; ++m) {
        const long double a = 2.0L * pi * (long double)m / (long double)n;
        set(m, double(cosl(a)), -double(sinl(a)));
    }
    // (c, -s) at m: reflected about an eighth, a quarter and a half of the circle
    if (n % 8 == 0)
        for (int m = n / 8 + 1; m <= n / 4; ++m) {
            const std::size_t k = 2 * std::size_t(n / 4 - m);
            set(m, -r[k + 1], -r[k]);
        }
    if (n % 4 == 0)
        for (int m = n / 4 + 1; m <= n / 2; ++m) {
            const std::size_t k = 2 * std::size_t(n / 2 - m);
            set(m, -r[k], r[k + 1]);
        }
    for (int m = n / 2 + 1; m < n; ++m) {
        const std::size_t k = 2 * std::size_t(n - m);
        set(m, r[k], -r[k + 1]);
    }
    return r;
}

// Host: the passes of length n and its twiddle table (double precision).
// With fuse21, 3 and 7 together go as one radix-21 pass; such a plan is for
// the transforms run by fft_lds<..., true> only.
inline bool fft_describe(int n, FftDesc& d, std::vector<double>& tw_re_im, bool fuse21 = false) {
    d = FftDesc();
    d.n = n;
    int m = n;
    auto push = [&](int r) {
        if (d.npass >= kFftMaxPass) return false;
        d.radix[d.npass++] = r;
        m /= r;
        return true;
    };
    // Odd radices first: the first pass writes at a stride of its radix, and
    // an odd stride spreads over the LDS banks where 8 would not.
    while (fuse21 && m % 21 == 0)
        if (!push(21)) return false;
    for (int r : {3, 5, 7, 11})
        while (m % r == 0)
            if (!push(r)) return false;
    while (m % 8 == 0)
        if (!push(8)) return false;
    while (m % 4 == 0)
        if (!push(4)) return false;
    while (m % 2 == 0)
        if (!push(2)) return false;
    if (m != 1 || n >= 65536) return false;
    int ns = 1, total = 0;
    for (int s = 0; s < d.npass; ++s) {
        d.ns[s] = ns;
        d.twoff[s] = total;
        total += ns * (d.radix[s] - 1);
        d.mnb[s] = fft_magic(unsigned(n / d.radix[s]));
        d.mns[s] = fft_magic(unsigned(ns));
        ns *= d.radix[s];
    }
    tw_re_im.assign(std::size_t(2) * (total > 0 ? total : 1), 0.0);
    const std::vector<double> root = fft_roots(n);
    for (int s = 0; s < d.npass; ++s) {
        const int r = d.radix[s];
        const long long den = (long long)d.ns[s] * r;  // divides n
        for (int k = 0; k < d.ns[s]; ++k)
            for (int t = 1; t < r; ++t) {
                // reduce k t / (Ns R) to [0, 1) exactly before the angle
                const std::size_t m = 2 * std::size_t(((long long)k * t) % den * (n / den));
                const std::size_t at = std::size_t(d.twoff[s] + k * (r - 1) + (t - 1));
                tw_re_im[2 * at] = root[m];
                tw_re_im[2 * at + 1] = root[m + 1];
            }
    }
    return true;
}

// Small DFTs, out[q] = sum_t v[t] exp(SGN 2 pi i t q / R), in place; SGN (+1 or
// -1) is a template argument, so signs fold into the instructions.
template <class T>
__device__ __forceinline__ void dft2(cx<T>* v) {
    cx<T> a = v[0], b = v[1];
    v[0] = cadd(a, b);
    v[1] = csub(a, b);
}

template <int SGN, class T>
__device__ __forceinline__ void dft4(cx<T>* v) {
    cx<T> t0 = cadd(v[0], v[2]), t1 = csub(v[0], v[2]);
    cx<T> t2 = cadd(v[1], v[3]), t3 = cmul_si<SGN>(csub(v[1], v[3]));
    v[0] = cadd(t0, t2);
    v[2] = csub(t0, t2);
    v[1] = cadd(t1, t3);
    v[3] = csub(t1, t3);
}

// out[2q] = DFT4(x_t + x_{t+4}), out[2q+1] = DFT4((x_t - x_{t+4}) W8^t).
template <int SGN, class T>
__device__ __forceinline__ void dft8(cx<T>* v) {
    const T h = T(0.70710678118654752440084436210484903928);
    cx<T> a[4], b[4];
    for (int t = 0; t < 4; ++t) {
        a[t] = cadd(v[t], v[t + 4]);
        b[t] = csub(v[t], v[t + 4]);
    }
    // W8^1 = h (1 + SGN i), W8^2 = SGN i, W8^3 = h (-1 + SGN i)
    b[1] = cmul(b[1], cx<T>{h, T(SGN) * h});
    b[2] = cmul_si<SGN>(b[2]);
    b[3] = cmul(b[3], cx<T>{-h, T(SGN) * h});
    dft4<SGN>(a);
    dft4<SGN>(b);
    for (int q = 0; q < 4; ++q) {
        v[2 * q] = a[q];
        v[2 * q + 1] = b[q];
    }
}

// Odd R: pairs (t, R - t) give out[q] = v0 + sum a_t cos + SGN i sum b_t sin.
template <class T, int R, int SGN>
__device__ __forceinline__ void dft_odd(cx<T>* v) {
    constexpr int m = (R - 1) / 2;
    const double* cs = R == 3 ? kCos3 : R == 5 ? kCos5 : R == 7 ? kCos7 : kCos11;
    const double* sn = R == 3 ? kSin3 : R == 5 ? kSin5 : R == 7 ? kSin7 : kSin11;
    cx<T> a[m + 1], b[m + 1], out[R];
    cx<T> s0 = v[0];
#pragma unroll
    for (int t = 1; t <= m; ++t) {
        a[t] = cadd(v[t], v[R - t]);
        b[t] = csub(v[t], v[R - t]);
        s0 = cadd(s0, a[t]);
    }
    out[0] = s0;
#pragma unroll
    for (int q = 1; q <= m; ++q) {
        cx<T> A = v[0], B = {T(0), T(0)};
#pragma unroll
        for (int t = 1; t <= m; ++t) {
            const int at = (t * q) % R;
            const T c = T(cs[at]), s = T(sn[at]);
            A = {A.re + a[t].re * c, A.im + a[t].im * c};
            B = {B.re + b[t].re * s, B.im + b[t].im * s};
        }
        const cx<T> iB = cmul_si<SGN>(B);
        out[q] = cadd(A, iB);
        out[R - q] = csub(A, iB);
    }
#pragma unroll
    for (int q = 0; q < R; ++q) v[q] = out[q];
}

// Radix 21 as 3 x 7 in registers by the prime-factor (Good-Thomas) mapping,
// so no twiddles between its two stages: a[n1][n2] = v[(7 n1 + 3 n2) mod 21],
// DFT3 along n1, DFT7 along n2, out[(7 k1 + 15 k2) mod 21] = a[k1][k2]. One
// pass (and its two barriers) fewer wherever 3 and 7 both divide a length.
template <int SGN, class T>
__device__ __forceinline__ void dft21(cx<T>* v) {
    cx<T> a[3][7];
#pragma unroll
    for (int n1 = 0; n1 < 3; ++n1)
#pragma unroll
        for (int n2 = 0; n2 < 7; ++n2) a[n1][n2] = v[(7 * n1 + 3 * n2) % 21];
#pragma unroll
    for (int n2 = 0; n2 < 7; ++n2) {
        cx<T> c[3] = {a[0][n2], a[1][n2], a[2][n2]};
        dft_odd<T, 3, SGN>(c);
#pragma unroll
        for (int k1 = 0; k1 < 3; ++k1) a[k1][n2] = c[k1];
    }
#pragma unroll
    for (int k1 = 0; k1 < 3; ++k1) {
        dft_odd<T, 7, SGN>(a[k1]);
#pragma unroll
        for (int k2 = 0; k2 < 7; ++k2) v[(7 * k1 + 15 * k2) % 21] = a[k1][k2];
    }
}

template <class T, int R, int SGN>
__device__ __forceinline__ void dft_small(cx<T>* v) {
    if constexpr (R == 2)
        dft2(v);
    else if constexpr (R == 4)
        dft4<SGN>(v);
    else if constexpr (R == 8)
        dft8<SGN>(v);
    else if constexpr (R == 21)
        dft21<SGN>(v);
    else
        dft_odd<T, R, SGN>(v);
}

// A value's place in LDS as a 32-bit address, and the place `step` values further
// on by one addition (opaque to the optimiser, which would otherwise form each
// position anew from the first).
template <class T>
struct Lds {
    typedef T pair __attribute__((ext_vector_type(2)));
    typedef __attribute__((address_space(3))) pair* ptr;
};
template <class P>
__device__ __forceinline__ P lds_step(P p, int step) {
    p += step;
    asm("" : "+v"(p));
    return p;
}

// Where a pass takes its values from and leaves them. Plain LDS is LdsEnd; any
// other end (of a single transform) is a pair of calls per value, `fetch` (every
// load of the pass, all in flight before the first use) and then `get` or `put`:
//   P fetch(u0, du)         for value u0 + du of the transform; du is uniform
//   cx get(u0, du, P)       the value to transform
//   void put(u0, du, P, v)  the value transformed
struct LdsEnd {};

// One Stockham pass of radix R over `ncol` transforms of length n in LDS.
// BMAX bounds the butterflies per thread (ceil(ncol n / (R NT))). With ONE
// (a single transform, as every row and long-column kernel) the butterfly's
// line is 0, so no division by the butterfly count is made, and its output
// base (position q within the output stride, k within the twiddles) is formed
// once in the load phase and kept for the store: the divisions are
// multiply-high, quarter-rate on the VALU. Several transforms recompute their
// indices in the store phase instead, which keeps no index registers live
// across the barrier (their kernels hold two transforms' registers).
// The passes are bound by the VALU and the LDS latency between (VALU issuing in 46
// to 70 % of the SIMDs' cycles over the four 2048^2 transforms), so
// the direction is a template argument (no sign selects) and LDS addresses step
// by nb and ns in 32-bit additions: 16.4 -> 14.2 VALU instructions a value and
// pass at radix 8, 24.5 -> 21.3 at radix 21.
template <class T, int NT, int R, int BMAX, bool ONE, int SGN, class In, class Out>
__device__ __forceinline__ void fft_pass(cx<T>* buf, int n, int ncol, int ns, unsigned mnb, unsigned mns,
                                         const cx<T>* tw, In& in, Out& out) {
    constexpr bool SRC = !std::is_same_v<In, LdsEnd>, DST = !std::is_same_v<Out, LdsEnd>;
    const int nb = n / R;
    const int total = ONE ? nb : nb * ncol;
    static_assert(ONE || !(SRC || DST));
    // butterfly j: its transform and its number within it
    auto place = [&](int j, int& c, int& jj) {
        c = 0;
        jj = j;
        if constexpr (!ONE) {
            c = int(udiv(unsigned(j), unsigned(nb), mnb));
            jj = j - c * nb;
        }
    };
    // its first output value within the transform, and its twiddle
    auto first_of = [&](int jj, int& k) {
        const int q = int(udiv(unsigned(jj), unsigned(ns), mns));
        k = jj - q * ns;
        return q * ns * R + k;
    };
    cx<T> v[BMAX][R];
    int cb[ONE ? BMAX : 1];
    if constexpr (SRC) {
        using P = decltype(in.fetch(0, 0));
        P pre[BMAX][R];
#pragma unroll
        for (int b = 0; b < BMAX; ++b) {
            const int j = int(threadIdx.x) + b * NT;
            if (j < total) {
                int c, jj;
                place(j, c, jj);
#pragma unroll
                for (int t = 0; t < R; ++t) pre[b][t] = in.fetch(jj, t * nb);
            }
        }
#pragma unroll
        for (int b = 0; b < BMAX; ++b) {
            const int j = int(threadIdx.x) + b * NT;
            if (j < total) {
                int c, jj;
                place(j, c, jj);
#pragma unroll
                for (int t = 0; t < R; ++t) v[b][t] = in.get(jj, t * nb, pre[b][t]);
            }
        }
    }
#pragma unroll
    for (int b = 0; b < BMAX; ++b) {
        const int j = int(threadIdx.x) + b * NT;
        if (j < total) {
            int c, jj, k = 0;
            place(j, c, jj);
            if constexpr (!SRC) {
                typename Lds<T>::ptr from = (typename Lds<T>::ptr)buf + (c * n + jj);
#pragma unroll
                for (int t = 0; t < R; ++t) {
                    v[b][t] = {from->x, from->y};
                    from = lds_step(from, nb);
                }
            }
            if constexpr (ONE)
                cb[b] = first_of(jj, k);
            else if (!SRC && ns > 1)
                first_of(jj, k);
            if (!SRC && ns > 1) {  // the first pass has no twiddles
                const cx<T>* w = tw + k * (R - 1);
#pragma unroll
                for (int t = 1; t < R; ++t) {
                    cx<T> f = w[t - 1];
                    if (SGN > 0) f.im = -f.im;
                    v[b][t] = cmul(v[b][t], f);
                }
            }
            dft_small<T, R, SGN>(v[b]);
        }
    }
    if constexpr (DST) {
        using P = decltype(out.fetch(0, 0));
        P pre[BMAX][R];
#pragma unroll
        for (int b = 0; b < BMAX; ++b) {
            const int j = int(threadIdx.x) + b * NT;
            if (j < total) {
                int c, jj, k;
                place(j, c, jj);
                const int base = ONE ? cb[ONE ? b : 0] : first_of(jj, k);
#pragma unroll
                for (int t = 0; t < R; ++t) pre[b][t] = out.fetch(base, t * ns);
            }
        }
#pragma unroll
        for (int b = 0; b < BMAX; ++b) {
            const int j = int(threadIdx.x) + b * NT;
            if (j < total) {
                int c, jj, k;
                place(j, c, jj);
                const int base = ONE ? cb[ONE ? b : 0] : first_of(jj, k);
#pragma unroll
                for (int t = 0; t < R; ++t) out.put(base, t * ns, pre[b][t], v[b][t]);
            }
        }
    } else {
        if constexpr (!SRC) __syncthreads();  // every value read
#pragma unroll
        for (int b = 0; b < BMAX; ++b) {
            const int j = int(threadIdx.x) + b * NT;
            if (j < total) {
                int c, jj, k;
                place(j, c, jj);
                const int base = ONE ? cb[ONE ? b : 0] : first_of(jj, k);
                typename Lds<T>::ptr to = (typename Lds<T>::ptr)buf + (c * n + base);
#pragma unroll
                for (int t = 0; t < R; ++t) {
                    to->x = v[b][t].re;
                    to->y = v[b][t].im;
                    to = lds_step(to, ns);
                }
            }
        }
        __syncthreads();
    }
}

constexpr int cdiv(int a, int b) { return (a + b - 1) / b; }

// Pass s of `d`.
template <class T, int NT, int MAXTOT, bool ONE, bool R21, int SGN, class In, class Out>
__device__ __forceinline__ void fft_pass_of(cx<T>* buf, const FftDesc& d, int s, int ncol, const cx<T>* tw, In& in,
                                            Out& out) {
    const cx<T>* tws = tw + d.twoff[s];
    const unsigned a = d.mnb[s], b = d.mns[s];
    const int ns = d.ns[s];
#define FFT_PASS(R) \
    fft_pass<T, NT, R, cdiv(MAXTOT, R * NT), ONE, SGN>(buf, d.n, ncol, ns, a, b, tws, in, out)
    switch (d.radix[s]) {
    case 2: FFT_PASS(2); break;
    case 3: FFT_PASS(3); break;
    case 4: FFT_PASS(4); break;
    case 5: FFT_PASS(5); break;
    case 7: FFT_PASS(7); break;
    case 8: FFT_PASS(8); break;
    case 21:
        if constexpr (R21) FFT_PASS(21);
        break;
    default: FFT_PASS(11); break;
    }
#undef FFT_PASS
}

template <class T, int NT, int MAXTOT, bool ONE, bool R21, int SGN>
__device__ __forceinline__ void fft_passes(cx<T>* buf, const FftDesc& d, int ncol, const cx<T>* tw) {
    LdsEnd lds;
    for (int s = 0; s < d.npass; ++s)
        fft_pass_of<T, NT, MAXTOT, ONE, R21, SGN>(buf, d, s, ncol, tw, lds, lds);
}

// One single-precision plane transform of two passes or more, the first from
// `in` and the last to `out`; the buffer holds nothing on entry.
template <class T, int NT, int MAXTOT, int SGN, class In, class Out>
__device__ __forceinline__ void fft_ends(cx<T>* buf, const FftDesc& d, const cx<T>* tw, In in, Out out) {
    LdsEnd lds;
    fft_pass_of<T, NT, MAXTOT, true, true, SGN>(buf, d, 0, 1, tw, in, lds);
    for (int s = 1; s < d.npass - 1; ++s)
        fft_pass_of<T, NT, MAXTOT, true, true, SGN>(buf, d, s, 1, tw, lds, lds);
    fft_pass_of<T, NT, MAXTOT, true, true, SGN>(buf, d, d.npass - 1, 1, tw, lds, out);
}

// All passes of `d` over ncol * d.n <= MAXTOT values in LDS (synchronised
// on entry by the caller, on exit here). PLANE (the exact gridder's
// single-precision plane transforms): the plan may hold radix-21 passes
// (fft_describe with fuse21), and a single line takes the single-line pass.
// Other kernels keep one pass form: the extra code would take registers they
// do not have to spare (the surrogate's column kernels, two transforms each,
// spilled with it).
template <class T, int NT, int MAXTOT, int SGN, bool PLANE = false>
__device__ __forceinline__ void fft_lds(cx<T>* buf, const FftDesc& d, int ncol, const cx<T>* tw) {
    if constexpr (PLANE) {
        if (ncol == 1)
            fft_passes<T, NT, MAXTOT, true, true, SGN>(buf, d, 1, tw);
        else
            fft_passes<T, NT, MAXTOT, false, true, SGN>(buf, d, ncol, tw);
    } else {
        fft_passes<T, NT, MAXTOT, false, false, SGN>(buf, d, ncol, tw);
    }
}

// The same with the direction a launch argument.
template <class T, int NT, int MAXTOT>
__device__ __forceinline__ void fft_lds_either(cx<T>* buf, const FftDesc& d, int ncol, const cx<T>* tw, int sgn) {
    if (sgn > 0)
        fft_lds<T, NT, MAXTOT, +1>(buf, d, ncol, tw);
    else
        fft_lds<T, NT, MAXTOT, -1>(buf, d, ncol, tw);
}

// Fills LDS from memory with every load of the block in flight before the
// first LDS write (a transform's loads are otherwise serialised on their
// latency): element e < count (count <= MT) is src[at(e).first], stored at
// buf[at(e).second].
template <class T, int NT, int MT, class At>
__device__ __forceinline__ void staged_fill(cx<T>* buf, const cx<T>* src, int count, At at) {
    constexpr int PER = (MT + NT - 1) / NT;
    if constexpr (sizeof(T) == 4) {
        cx<T> r[PER];
        int dst[PER];
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const int e = threadIdx.x + k * NT;
            if (e < count) {
                const auto sd = at(e);
                r[k] = src[sd.first];
                dst[k] = sd.second;
            }
        }
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const int e = threadIdx.x + k * NT;
            if (e < count) buf[dst[k]] = r[k];
        }
    } else {
        // double: the values staged as two-lane vectors (staging arrays of the
        // complex struct are placed in scratch memory by the compiler)
        using V = __attribute__((ext_vector_type(2))) double;
        V r[PER];
        int dst[PER];
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const int e = threadIdx.x + k * NT;
            if (e < count) {
                const auto sd = at(e);
                r[k] = *reinterpret_cast<const V*>(src + sd.first);
                dst[k] = sd.second;
            }
        }
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const int e = threadIdx.x + k * NT;
            if (e < count) *reinterpret_cast<V*>(buf + dst[k]) = r[k];
        }
    }
}

// The same, or value by value for lines of 1025 to 2048 doubles: with their eight
// values a thread staged the scheduler gives the kernel up to 236 registers, one or
// two waves per SIMD (the surrogate's inverse rows of 2048, eight nodes, 174 -> 354
// us; built for three waves they spill).
template <class T, int NT, int MT, class At>
__device__ __forceinline__ void line_fill(cx<T>* buf, const cx<T>* src, int count, At at) {
    if constexpr (sizeof(T) == 8 && MT == 2048) {
        for (int e = threadIdx.x; e < count; e += NT) {
            const auto sd = at(e);
            buf[sd.second] = src[sd.first];
        }
    } else {
        staged_fill<T, NT, MT>(buf, src, count, at);
    }
}

// Single-precision sine and cosine of `turns` whole turns: the whole turns and
// the nearest quarter turn are taken off in double precision; what is left, at
// most an eighth of a turn, goes through the Taylor series (first terms left
// out: x^11 / 11! < 2e-9, x^12 / 12! < 2e-10 at pi / 4). Largest error 8.5e-8;
// the angle rounded to single precision on up to 2 pi and sincosf: 2.8e-7.
__device__ __forceinline__ void sincos_turns(double turns, float& sn, float& cs) {
    const double t = 4.0 * (turns - floor(turns)), qd = rint(t);
    const int q = int(qd);
    const float x = float((t - qd) * 1.5707963267948966), z = x * x;
    float a = fmaf(z, 1.0f / 362880, -1.0f / 5040);
    a = fmaf(z, a, 1.0f / 120);
    a = fmaf(z, a, -1.0f / 6);
    a = fmaf(z * x, a, x);
    float b = fmaf(z, -1.0f / 3628800, 1.0f / 40320);
    b = fmaf(z, b, -1.0f / 720);
    b = fmaf(z, b, 1.0f / 24);
    b = fmaf(z, b, -0.5f);
    b = fmaf(z, b, 1.0f);
    // quarter turns: (c, s), (-s, c), (-c, -s), (s, -c)
    cs = (q & 1) ? a : b;
    sn = (q & 1) ? b : a;
    if ((q + 1) & 2) cs = -cs;
    if (q & 2) sn = -sn;
}

// Plane-wise transpose of complex values, [P][R][C] -> [P][C][R], through
// LDS tiles (64 x 64 in single precision, 32 x 32 in double, a column of
// padding against bank conflicts): both sides coalesced.
template <class T>
__global__ __launch_bounds__(256) void k_tile_transpose(const cx<T>* __restrict__ in, cx<T>* __restrict__ out, int R,
                                                        int C) {
    constexpr int TS = sizeof(T) == 4 ? 64 : 32;
    __shared__ cx<T> t[TS][TS + 1];
    const int c0 = blockIdx.x * TS, r0 = blockIdx.y * TS;
    const long long base = (long long)blockIdx.z * R * C;
    for (int k = threadIdx.x; k < TS * TS; k += 256) {
        const int rr = k / TS, cc = k - rr * TS, r = r0 + rr, c = c0 + cc;
        if (r < R && c < C) t[rr][cc] = in[base + (long long)r * C + c];
    }
    __syncthreads();
    for (int k = threadIdx.x; k < TS * TS; k += 256) {
        const int cc = k / TS, rr = k - cc * TS, r = r0 + rr, c = c0 + cc;
        if (r < R && c < C) out[base + (long long)c * R + r] = t[rr][cc];
    }
}

// The same for single precision with even R and C: each lane moves two
// neighbouring values (16 bytes) per access on both sides.
template <class T>
__global__ __launch_bounds__(256) void k_tile_transpose_pairs(const cx<T>* __restrict__ in, cx<T>* __restrict__ out,
                                                              int R, int C) {
    static_assert(sizeof(T) == 4, "pairs of single-precision values");
    typedef float f4 __attribute__((ext_vector_type(4)));
    constexpr int TS = 64;
    __shared__ cx<T> t[TS][TS + 1];
    const int c0 = blockIdx.x * TS, r0 = blockIdx.y * TS;
    const long long base = (long long)blockIdx.z * R * C;
    for (int k = threadIdx.x; k < TS * TS / 2; k += 256) {
        const int rr = k / (TS / 2), cp = 2 * (k - rr * (TS / 2)), r = r0 + rr, c = c0 + cp;
        if (r < R && c < C) {
            const f4 v = *reinterpret_cast<const f4*>(in + base + (long long)r * C + c);
            t[rr][cp] = cx<T>{v.x, v.y};
            t[rr][cp + 1] = cx<T>{v.z, v.w};
        }
    }
    __syncthreads();
    for (int k = threadIdx.x; k < TS * TS / 2; k += 256) {
        const int cc = k / (TS / 2), rp = 2 * (k - cc * (TS / 2)), r = r0 + rp, c = c0 + cc;
        if (r < R && c < C) {
            const cx<T> a = t[rp][cc], b = t[rp + 1][cc];
            *reinterpret_cast<f4*>(out + base + (long long)c * R + r) = f4{a.re, a.im, b.re, b.im};
        }
    }
}

}  // namespace rang
