// Bluestein (chirp-z) form of the line FFT for lengths without a compiled
// mixed-radix plan.  With a_j = exp(-i*pi*j^2/n),
//   X_k = sum_j x_j w^(jk) = a_k * sum_j (x_j a_j) conj(a_(k-j)),
// a circular convolution of length M >= 2n-1 (a power of two with a
// compiled Stockham plan PM).  One length-n transform is then
//   chirp -> FFT_M -> (x spectrum of the wrapped chirp / M) -> IFFT_M -> chirp
// entirely in registers/LDS of one kernel; the inverse direction uses
// conj(a).  PM's forward last pass and inverse first pass have the same
// radix (and the inverse last / forward first), so consecutive stages and
// consecutive transforms chain in registers exactly as line_pair does.
//
// Tables of one length (one device allocation, built on the host in double):
//   tab[0, M/2)         a_j, zero from n on (2n - 1 <= M: n <= M/2)
//   tab[M/2, 3M/2)      FFT_M(wrap(conj a)) / M   (forward transform)
//   tab[3M/2, 5M/2)     FFT_M(wrap(a)) / M        (inverse transform)
// each in the order of the registers that read it (blue_index): the chirp by
// PM's forward first pass, the spectra by its forward last one.
// wrap(b)[m] = b_m for m < n, b_(M-m) for m > M-n, 0 otherwise.
#pragma once

#include "fft_device.hpp"

namespace imr {

struct Blue {
    int n;
    Buf tab;
};

// elements of a line at the input positions of PM's forward first pass and
// at the output positions of its inverse last pass (the same ones: both have
// radix rf[0])
template <class PM> using BlueIn = Elems<PM, -1, 0, true>;
template <class PM> using BlueOut = Elems<PM, +1, PM::np - 1, true>;

// a thread's `count` values of a table at byte `base`, in pairs
template <class PM, int count>
__device__ __forceinline__ void blue_load(cf (&x)[count], const Blue &b, int t, unsigned base)
{
    static_assert(count % 2 == 0 && PM::E % 2 == 0, "values load in pairs");
#pragma unroll
    for (int q = 0; q < count; q += 2) {
        const cf2 p = b.tab.get<cf2>(16u * t, base + 8u * blue_index(q, 0, PM::T));
        x[q] = mkc(p.x, p.y);
        x[q + 1] = mkc(p.z, p.w);
    }
}

// chirp a_(t+o) of a thread's elements below M/2: register s = b*R + r has
// value b*R/2 + r
template <class PM>
struct Chirp {
    cf a[PM::E / 2];
    __device__ __forceinline__ void load(const Blue &b, int t) { blue_load<PM, PM::E / 2>(a, b, t, 0u); }
    __device__ __forceinline__ cf at(int s) const
    {
        constexpr int R = PM::rf[0];
        return a[s / R * (R / 2) + s % R];
    }
};

// v <- chirped line (conjugated chirp for the inverse).  What lies past the
// line's end becomes 0 by the table's zeros if it is finite; CLEAR sets it to
// 0 whatever it is (the first transform's values there, which may overflow
// where the line does not)
template <class PM, int DIR, bool CLEAR = false, class El>
__device__ __forceinline__ void blue_apply_chirp(cf (&v)[PM::E], const Chirp<PM> &ch, const El &el)
{
    el.all([&](int s, int o) {
        v[s] = cmul(v[s], DIR < 0 ? ch.at(s) : mkc(ch.at(s).x, -ch.at(s).y));
        if (CLEAR && !el.inside(o)) v[s] = mkc(0.f, 0.f);
    });
}

// circular convolution with the chirp: v holds the chirped line (zero from n
// to M/2; the zeros of the upper half are implied, their registers not read)
// at PM's forward first-pass input positions on entry and the result at PM's
// inverse last-pass output positions on exit.  The chirp's spectrum is loaded
// after the forward transform's last pass; `hook` runs after the inverse's
// (loads issued before the last exchange take registers from its
// butterflies: 1373 x 1101, 10 iterations 793 us so, 923 us with them ahead).
template <class PM, int DIR, class Lds, class Hook>
__device__ __forceinline__ void blue_conv(cf (&v)[PM::E], const Buf &tw, int t, const Lds &L,
                                          const Blue &b, Hook &hook)
{
    constexpr unsigned h = 8u * (PM::n / 2 + (DIR < 0 ? 0 : PM::n));
    static_assert(PM::T * PM::E == PM::n, "every register of every thread is an element");
    cf hv[PM::E];
    auto load_h = [&] { blue_load<PM, PM::E>(hv, b, t, h); };
    compute_half<PM, -1>(v, t);
    Slots<PM> sl;
    passes_from<PM, -1, 1, false, false>(v, tw, t, L, sl, load_h);
#pragma unroll
    for (int s = 0; s < PM::E; ++s) v[s] = cmul(v[s], hv[s]);
    compute<PM, +1, 0>(v, tw, t);
    passes_from<PM, +1, 1, true, false>(v, tw, t, L, sl, hook);
}

// one length-n transform of direction DIR, callbacks as line_fft
template <class PM, int DIR, class Lds, class Src, class Pre, class Dst>
__device__ __forceinline__ void blue_fft(cf (&v)[PM::E], const Buf &tw, int t, const Lds &L,
                                         const Blue &b, Src &src, Pre &pre, Dst &dst)
{
    const BlueIn<PM> in{t, b.n};
    const BlueOut<PM> out{t, b.n};
    Chirp<PM> ch;
#pragma unroll
    for (int s = 0; s < PM::E; ++s) v[s] = mkc(0.f, 0.f);
    src(v, in);
    ch.load(b, t);
    issue_loads();
    blue_apply_chirp<PM, DIR>(v, ch, in);
    auto hook = [&] {
        ch.load(b, t);
        pre(out);
    };
    blue_conv<PM, DIR>(v, tw, t, L, b, hook);
    blue_apply_chirp<PM, DIR>(v, ch, out);
    dst(v, out);
}

// transform DA, mid on its outputs, transform DB, callbacks as line_pair.
// The output chirp of DA and the input chirp of DB cancel around the modulus
// projection, but leaving both out rounds differently, by up to 1.3e-6 of an
// image after two cycles (for 1% of the passes' time): both are applied.
template <class PM, int DA, int DB, class Lds, class Src, class Pre, class Mid, class Dst>
__device__ __forceinline__ void blue_pair(cf (&v)[PM::E], const Buf &tw, int t, const Lds &L,
                                          const Blue &b, Src &src, Pre &pre, Mid &mid, Dst &dst)
{
    static_assert(DA == -DB, "a pair runs opposite directions");
    const BlueIn<PM> in{t, b.n};
    const BlueOut<PM> out{t, b.n};
    Chirp<PM> ch;
#pragma unroll
    for (int s = 0; s < PM::E; ++s) v[s] = mkc(0.f, 0.f);
    src(v, in);
    ch.load(b, t);
    issue_loads();
    blue_apply_chirp<PM, DA>(v, ch, in);
    auto at_mid = [&] {
        ch.load(b, t);
        pre(out);
    };
    blue_conv<PM, DA>(v, tw, t, L, b, at_mid);
    blue_apply_chirp<PM, DA>(v, ch, out);
    mid(v, out);
    blue_apply_chirp<PM, DB, true>(v, ch, out);
    auto at_end = [&] { ch.load(b, t); };
    blue_conv<PM, DB>(v, tw, t, L, b, at_end);
    blue_apply_chirp<PM, DB>(v, ch, out);
    dst(v, out);
}

// direct (compiled plan of the line length) or Bluestein (BL: P is the
// convolution plan, the line length is b.n) line transforms
template <class P, int DIR, bool BL, class Lds, class Src, class Pre, class Dst>
__device__ __forceinline__ void xfft(cf (&v)[P::E], const Buf &tw, int t, const Lds &L, const Blue &b,
                                     Src &src, Pre &pre, Dst &dst)
{
    if constexpr (BL) blue_fft<P, DIR>(v, tw, t, L, b, src, pre, dst);
    else line_fft<P, DIR>(v, tw, t, L, src, pre, dst);
}

template <class P, int DA, int DB, bool BL, int WHEN, class Lds, class Src, class Pre, class Mid, class Dst>
__device__ __forceinline__ void xpair(cf (&v)[P::E], const Buf &tw, int t, const Lds &L, const Blue &b,
                                      Src &src, Pre &pre, Mid &mid, Dst &dst)
{
    if constexpr (BL) blue_pair<P, DA, DB>(v, tw, t, L, b, src, pre, mid, dst);
    else line_pair<P, DA, DB, WHEN>(v, tw, t, L, src, pre, mid, dst);
}

}  // namespace imr
