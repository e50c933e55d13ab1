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
//   tab[0, n)       a_j
//   tab[n, n+M)     FFT_M(wrap(conj a)) / M   (forward transform)
//   tab[n+M, n+2M)  FFT_M(wrap(a)) / M        (inverse transform)
// wrap(b)[m] = b_m for m < n, b_(M-m) for m > M-n, 0 otherwise.
#pragma once

#include "fft_device.hpp"

namespace imr {

struct Blue {
    int n;
    const cf *tab;
};

// elements of a line at the input positions of PM's forward first pass and
// at the output positions of its inverse last pass (the same ones: both have
// radix rf[0])
template <class PM> using BlueIn = Elems<PM, -1, 0, true>;
template <class PM> using BlueOut = Elems<PM, +1, PM::np - 1, true>;

// chirp a_(t+o) of a thread's elements
template <class PM, class El>
__device__ __forceinline__ void blue_load_chirp(cf (&ch)[PM::E], const Blue &b, const El &el)
{
    el.load([&](int s, int o, int d) { ch[s] = at32(b.tab + o, d); });
}

// v <- chirped line (conjugated chirp for the inverse), zero past its end
template <class PM, int DIR, class El>
__device__ __forceinline__ void blue_apply_chirp(cf (&v)[PM::E], const cf (&ch)[PM::E], const El &el)
{
    el.all([&](int s, int o) {
        const cf z = cmul(v[s], DIR < 0 ? ch[s] : mkc(ch[s].x, -ch[s].y));
        v[s] = el.inside(o) ? z : mkc(0.f, 0.f);
    });
}

// circular convolution with the chirp: v holds the chirped, zero-padded
// line at PM's forward first-pass input positions on entry and the result
// at PM's inverse last-pass output positions on exit.  The chirp's spectrum
// is loaded before the last exchange of the forward transform; `hook` runs
// before the last exchange of the inverse one.
template <class PM, int DIR, class Lds, class Hook>
__device__ __forceinline__ void blue_conv(cf (&v)[PM::E], const cf *tw, int t, const Lds &L,
                                          const Blue &b, Hook &hook)
{
    const cf *h = b.tab + b.n + (DIR < 0 ? 0 : PM::n);
    const Elems<PM, -1, PM::np - 1> mid{t, PM::n};
    cf hv[PM::E];
    auto load_h = [&] { mid.load([&](int s, int o, int d) { hv[s] = at32(h + o, d); }); };
    compute<PM, -1, 0>(v, tw, t);
    Slots<PM> sl;
    passes_from<PM, -1, 1, false>(v, tw, t, L, sl, load_h);
    mid.all([&](int s, int) { v[s] = cmul(v[s], hv[s]); });
    compute<PM, +1, 0>(v, tw, t);
    passes_from<PM, +1, 1, true>(v, tw, t, L, sl, hook);
}

// one length-n transform of direction DIR, callbacks as line_fft
template <class PM, int DIR, class Lds, class Src, class Pre, class Dst>
__device__ __forceinline__ void blue_fft(cf (&v)[PM::E], const cf *tw, int t, const Lds &L,
                                         const Blue &b, Src &src, Pre &pre, Dst &dst)
{
    const BlueIn<PM> in{t, b.n};
    const BlueOut<PM> out{t, b.n};
    cf ch[PM::E] = {};
    src(v, in);
    blue_load_chirp<PM>(ch, b, in);
    blue_apply_chirp<PM, DIR>(v, ch, in);
    auto hook = [&] {
        blue_load_chirp<PM>(ch, b, out);
        pre(out);
    };
    blue_conv<PM, DIR>(v, tw, t, L, b, hook);
    blue_apply_chirp<PM, DIR>(v, ch, out);
    dst(v, out);
}

// transform DA, mid on its outputs, transform DB, callbacks as line_pair
template <class PM, int DA, int DB, bool EARLY, class Lds, class Src, class Pre, class Mid, class Dst>
__device__ __forceinline__ void blue_pair(cf (&v)[PM::E], const cf *tw, int t, const Lds &L,
                                          const Blue &b, Src &src, Pre &pre, Mid &mid, Dst &dst)
{
    static_assert(DA == -DB, "a pair runs opposite directions");
    const BlueIn<PM> in{t, b.n};
    const BlueOut<PM> out{t, b.n};
    cf ch[PM::E] = {};
    src(v, in);
    blue_load_chirp<PM>(ch, b, in);
    if constexpr (EARLY) pre(out);
    blue_apply_chirp<PM, DA>(v, ch, in);
    auto at_mid = [&] {
        blue_load_chirp<PM>(ch, b, out);
        if constexpr (!EARLY) pre(out);
    };
    blue_conv<PM, DA>(v, tw, t, L, b, at_mid);
    blue_apply_chirp<PM, DA>(v, ch, out);
    mid(v, out);
    blue_apply_chirp<PM, DB>(v, ch, out);
    auto at_end = [&] { blue_load_chirp<PM>(ch, b, out); };
    blue_conv<PM, DB>(v, tw, t, L, b, at_end);
    blue_apply_chirp<PM, DB>(v, ch, out);
    dst(v, out);
}

// direct (compiled plan of the line length) or Bluestein (BL: P is the
// convolution plan, the line length is b.n) line transforms
template <class P, int DIR, bool BL, class Lds, class Src, class Pre, class Dst>
__device__ __forceinline__ void xfft(cf (&v)[P::E], const cf *tw, int t, const Lds &L, const Blue &b,
                                     Src &src, Pre &pre, Dst &dst)
{
    if constexpr (BL) blue_fft<P, DIR>(v, tw, t, L, b, src, pre, dst);
    else line_fft<P, DIR>(v, tw, t, L, src, pre, dst);
}

template <class P, int DA, int DB, bool BL, bool EARLY, class Lds, class Src, class Pre, class Mid, class Dst>
__device__ __forceinline__ void xpair(cf (&v)[P::E], const cf *tw, int t, const Lds &L, const Blue &b,
                                      Src &src, Pre &pre, Mid &mid, Dst &dst)
{
    if constexpr (BL) blue_pair<P, DA, DB, EARLY>(v, tw, t, L, b, src, pre, mid, dst);
    else line_pair<P, DA, DB, EARLY>(v, tw, t, L, src, pre, mid, dst);
}

}  // namespace imr
