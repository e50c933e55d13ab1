// Device building blocks of the LDS-staged Stockham line FFT for gfx950.
//
// A line of length n = prod(R_p) is transformed by T threads (compile-time
// plan, see plans.hpp).  Pass p (radix R, span ns = R_0*...*R_{p-1}) owns
// butterflies j = t + b*T; it reads elements j + r*(n/R), multiplies element r
// by exp(-+2*pi*i*r*(j%ns)/(ns*R)), runs a radix-R DFT in registers and
// writes element r to (j - j%ns)*R + j%ns + r*ns.  The first pass therefore
// reads and the last pass writes the line in natural order j + r*(n/R): the
// accesses are coalesced in global memory, and a fused prologue/epilogue
// (HIO constraint, modulus projection, norm, error sums) runs on registers at
// exactly those positions.  Between passes the data goes through LDS; each
// thread keeps at most E = 16 complex values in VGPRs.
//
// Forward = exp(-2*pi*i*j*k/n) (FFTW_FORWARD / CUFFT_FORWARD); both
// directions are unnormalized, as the reference's FFTs.  Forward transforms
// run the radices in plan order, inverse transforms in reverse order, so the
// last pass of one direction and the first pass of the other have the same
// radix and butterfly ownership: a forward->inverse (or inverse->forward)
// pair with an elementwise operator in between never leaves registers at the
// junction (line_pair).
#pragma once

#include <type_traits>

#include "common.hpp"
#include "plans.hpp"

namespace imr {

// native 2-wide vector: one 64-bit load / store per complex value
typedef float cf __attribute__((ext_vector_type(2)));
typedef float cf2 __attribute__((ext_vector_type(4)));   // two of them
__device__ __forceinline__ cf mkc(float x, float y)
{
    cf r;
    r.x = x;
    r.y = y;
    return r;
}

// A plane in global memory: a workgroup-uniform base and size, one 32-bit
// per-lane byte offset v and a uniform byte offset s.
//
// Loads go through a buffer descriptor: a thread's elements differ by uniform
// offsets, so they share one vector register of address (plain pointers cost a
// 64-bit vector add and a register pair per element), and the hardware range
// check stands in for edge tests: a load past the end returns 0, kOutside is
// past every end.
// Stores go through plain pointers, and the caller keeps them inside: the
// address arithmetic spaces a thread's stores.  Buffer stores, issued back to
// back, were slower wherever a tile is narrower than a cache line (columns
// of 4096^2: 2-D transform pair 258 against 227 us, 8192^2: 2164 against
// 1630 us) and no faster elsewhere.
constexpr unsigned kOutside = 0x80000000u;

struct Buf {
    __amdgpu_buffer_rsrc_t r;
    char *p;
    __device__ __forceinline__ Buf(const void *base, size_t bytes)
        : r(__builtin_amdgcn_make_buffer_rsrc((void *) base, 0, (unsigned) bytes, 0x00027000)), p((char *) base)
    {
    }
    template <class T>
    __device__ __forceinline__ T get(unsigned v, unsigned s) const
    {
        if constexpr (sizeof(T) == 16) return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b128(r, v, s, 0));
        else if constexpr (sizeof(T) == 8) return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, v, s, 0));
        else if constexpr (sizeof(T) == 4) return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, v, s, 0));
        else return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b8(r, v, s, 0));
    }
    template <class T>
    __device__ __forceinline__ void put(T x, unsigned v, unsigned s) const
    {
        *(T *) (p + s + (size_t) v) = x;
    }
};

// ------------------------------------------------------------ complex math
// Products use one fma per component; the FFT is the only place that
// contracts -- the library is compiled with -ffp-contract=off so that all
// elementwise operators round exactly as the reference's C++ code.
__device__ __forceinline__ cf cadd(cf a, cf b) { return mkc(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ cf csub(cf a, cf b) { return mkc(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ cf cmul(cf a, cf b)
{
    return mkc(__builtin_fmaf(a.x, b.x, -(a.y * b.y)), __builtin_fmaf(a.x, b.y, a.y * b.x));
}
// a * conj(b)
__device__ __forceinline__ cf cmulc(cf a, cf b)
{
    return mkc(__builtin_fmaf(a.x, b.x, a.y * b.y), __builtin_fmaf(a.y, b.x, -(a.x * b.y)));
}
// a * (DIR < 0 ? -i : +i)
template <int DIR> __device__ __forceinline__ cf rot(cf a)
{
    return DIR < 0 ? mkc(a.y, -a.x) : mkc(-a.y, a.x);
}
// twiddle multiply: forward uses the table value, inverse its conjugate
template <int DIR> __device__ __forceinline__ cf twmul(cf a, cf w)
{
    return DIR < 0 ? cmul(a, w) : cmulc(a, w);
}

// cos/sin(2*pi*k/R) for the odd radices
template <int R> struct OddConst;
template <> struct OddConst<3> {
    static constexpr float c[3] = {1.f, -0.5f, -0.5f};
    static constexpr float s[3] = {0.f, 0.866025404f, -0.866025404f};
};
template <> struct OddConst<5> {
    static constexpr float c[5] = {1.f, 0.309016994f, -0.809016994f, -0.809016994f, 0.309016994f};
    static constexpr float s[5] = {0.f, 0.951056516f, 0.587785252f, -0.587785252f, -0.951056516f};
};

// ------------------------------------------------------------ butterflies
template <int DIR>
__device__ __forceinline__ void bf2(cf *v)
{
    const cf a = v[0], b = v[1];
    v[0] = cadd(a, b);
    v[1] = csub(a, b);
}

template <int DIR>
__device__ __forceinline__ void bf4io(cf a, cf b, cf c, cf d, cf &o0, cf &o1, cf &o2, cf &o3)
{
    const cf t0 = cadd(a, c), t1 = csub(a, c), t2 = cadd(b, d), t3 = rot<DIR>(csub(b, d));
    o0 = cadd(t0, t2);
    o2 = csub(t0, t2);
    o1 = cadd(t1, t3);
    o3 = csub(t1, t3);
}

// the same for c = d = 0
template <int DIR>
__device__ __forceinline__ void bf4io_half(cf a, cf b, cf &o0, cf &o1, cf &o2, cf &o3)
{
    const cf t3 = rot<DIR>(b);
    o0 = cadd(a, b);
    o2 = csub(a, b);
    o1 = cadd(a, t3);
    o3 = csub(a, t3);
}

template <int DIR>
__device__ __forceinline__ void bf4(cf *v)
{
    cf o0, o1, o2, o3;
    bf4io<DIR>(v[0], v[1], v[2], v[3], o0, o1, o2, o3);
    v[0] = o0; v[1] = o1; v[2] = o2; v[3] = o3;
}

// HALF: the upper half of the inputs is 0 and is not read
template <int DIR, bool HALF = false>
__device__ __forceinline__ void bf8(cf *v)
{
    constexpr float c = 0.707106781f;
    cf e0, e1, e2, e3, o0, o1, o2, o3;
    if constexpr (HALF) {
        bf4io_half<DIR>(v[0], v[2], e0, e1, e2, e3);
        bf4io_half<DIR>(v[1], v[3], o0, o1, o2, o3);
    } else {
        bf4io<DIR>(v[0], v[2], v[4], v[6], e0, e1, e2, e3);
        bf4io<DIR>(v[1], v[3], v[5], v[7], o0, o1, o2, o3);
    }
    o1 = cmul(o1, mkc(c, DIR * c));
    o2 = rot<DIR>(o2);
    o3 = cmul(o3, mkc(-c, DIR * c));
    v[0] = cadd(e0, o0); v[4] = csub(e0, o0);
    v[1] = cadd(e1, o1); v[5] = csub(e1, o1);
    v[2] = cadd(e2, o2); v[6] = csub(e2, o2);
    v[3] = cadd(e3, o3); v[7] = csub(e3, o3);
}

template <int DIR, bool HALF = false>
__device__ __forceinline__ void bf16(cf *v)
{
    constexpr float c1 = 0.923879533f, s1 = 0.382683432f, c2 = 0.707106781f;
    cf y[16];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        if constexpr (HALF)
            bf4io_half<DIR>(v[q], v[q + 4], y[4 * q + 0], y[4 * q + 1], y[4 * q + 2], y[4 * q + 3]);
        else
            bf4io<DIR>(v[q], v[q + 4], v[q + 8], v[q + 12], y[4 * q + 0], y[4 * q + 1], y[4 * q + 2],
                       y[4 * q + 3]);
    }
    // y[4*q + s] *= W16^(q*s), W16^k = (cos(2 pi k/16), DIR sin(2 pi k/16))
    y[5] = cmul(y[5], mkc(c1, DIR * s1));     // k = 1
    y[6] = cmul(y[6], mkc(c2, DIR * c2));     // k = 2
    y[7] = cmul(y[7], mkc(s1, DIR * c1));     // k = 3
    y[9] = cmul(y[9], mkc(c2, DIR * c2));     // k = 2
    y[10] = rot<DIR>(y[10]);                  // k = 4
    y[11] = cmul(y[11], mkc(-c2, DIR * c2));  // k = 6
    y[13] = cmul(y[13], mkc(s1, DIR * c1));   // k = 3
    y[14] = cmul(y[14], mkc(-c2, DIR * c2));  // k = 6
    y[15] = cmul(y[15], mkc(-c1, -DIR * s1)); // k = 9
#pragma unroll
    for (int s = 0; s < 4; ++s)
        bf4io<DIR>(y[s], y[4 + s], y[8 + s], y[12 + s], v[s], v[s + 4], v[s + 8], v[s + 12]);
}

template <int R, int DIR>
__device__ __forceinline__ void bf_odd(cf *v)
{
    constexpr int H = (R - 1) / 2;
    cf t[H], u[H];
#pragma unroll
    for (int k = 1; k <= H; ++k) {
        t[k - 1] = cadd(v[k], v[R - k]);
        u[k - 1] = csub(v[k], v[R - k]);
    }
    const cf x0 = v[0];
    cf sum = x0;
#pragma unroll
    for (int k = 0; k < H; ++k) sum = cadd(sum, t[k]);
#pragma unroll
    for (int s = 1; s <= H; ++s) {
        cf a = x0, b = mkc(0.f, 0.f);
#pragma unroll
        for (int k = 1; k <= H; ++k) {
            const float cc = OddConst<R>::c[(k * s) % R];
            const float ss = OddConst<R>::s[(k * s) % R];
            a = mkc(__builtin_fmaf(t[k - 1].x, cc, a.x), __builtin_fmaf(t[k - 1].y, cc, a.y));
            b = mkc(__builtin_fmaf(u[k - 1].x, ss, b.x), __builtin_fmaf(u[k - 1].y, ss, b.y));
        }
        const cf rb = rot<DIR>(b);
        v[s] = cadd(a, rb);
        v[R - s] = csub(a, rb);
    }
    v[0] = sum;
}

template <int R, int DIR>
__device__ __forceinline__ void bfly(cf *v);

// inverse of a modulo m (a, m coprime, m small), for the index maps below
__host__ __device__ constexpr int inv_mod(int a, int m)
{
    for (int x = 1; x < m; ++x)
        if ((a * x) % m == 1) return x;
    return m == 1 ? 0 : -1;
}

// Radix N1*N2 with N1, N2 coprime (6, 10, 12, 15) by the prime-factor
// (Good-Thomas) algorithm: with input n = (N2 n1 + N1 n2) mod N and output
// k = (N2 (N2^-1 mod N1) k1 + N1 (N1^-1 mod N2) k2) mod N, the length-N DFT
// is N2 length-N1 DFTs over n1 followed by N1 length-N2 DFTs over n2, with
// no twiddle factors between them.  The index maps are compile-time
// register permutations.
template <int N1, int N2, int DIR>
__device__ __forceinline__ void bf_pfa(cf *v)
{
    constexpr int N = N1 * N2;
    constexpr int i1 = inv_mod(N2 % N1, N1), i2 = inv_mod(N1 % N2, N2);
    static_assert(i1 > 0 && i2 > 0, "prime-factor radices must be coprime");
    cf a[N1][N2];
#pragma unroll
    for (int n2 = 0; n2 < N2; ++n2) {
        cf c[N1];
#pragma unroll
        for (int n1 = 0; n1 < N1; ++n1) c[n1] = v[(N2 * n1 + N1 * n2) % N];
        bfly<N1, DIR>(c);
#pragma unroll
        for (int k1 = 0; k1 < N1; ++k1) a[k1][n2] = c[k1];
    }
#pragma unroll
    for (int k1 = 0; k1 < N1; ++k1) {
        bfly<N2, DIR>(a[k1]);
#pragma unroll
        for (int k2 = 0; k2 < N2; ++k2) v[(N2 * i1 * k1 + N1 * i2 * k2) % N] = a[k1][k2];
    }
}

template <int R, int DIR>
__device__ __forceinline__ void bfly(cf *v)
{
    if constexpr (R == 1) (void) v;   // length-1 line: identity
    else if constexpr (R == 2) bf2<DIR>(v);
    else if constexpr (R == 4) bf4<DIR>(v);
    else if constexpr (R == 8) bf8<DIR>(v);
    else if constexpr (R == 16) bf16<DIR>(v);
    else if constexpr (R == 6) bf_pfa<2, 3, DIR>(v);
    else if constexpr (R == 10) bf_pfa<2, 5, DIR>(v);
    else if constexpr (R == 12) bf_pfa<4, 3, DIR>(v);
    else if constexpr (R == 15) bf_pfa<3, 5, DIR>(v);
    else bf_odd<R, DIR>(v);
}

// ------------------------------------------------------------ LDS layout
// One padding slot every 16 values spreads the stride-R accesses of the
// passes over the LDS banks (two 4-byte banks per complex value).
__host__ __device__ constexpr int lpad(int i) { return i + (i >> 4); }
__host__ __device__ constexpr int lds_elems(int n) { return n + (n >> 4) + 1; }

// One line in LDS, slots of STRIDE lines interleaved: slot e at
// p[lpad(e*STRIDE)].  at<STEP, MUL>(e0, r) addresses slot e0 + r*STEP for an
// e0 that is a multiple of MUL: where the padding allows it, r moves the
// address by a constant, which becomes an immediate offset of the LDS
// instruction.  sync() orders a line's writes before its reads: a line whose
// threads share one wave (WAVE) needs no workgroup barrier, for the LDS
// executes a wave's instructions in order.
template <int STRIDE, bool WAVE>
struct LdsLine {
    cf *p;
    template <int STEP, int MUL>
    __device__ __forceinline__ cf &at(int e0, int r) const
    {
        constexpr int d = STEP * STRIDE;
        if constexpr (d % 16 == 0) return p[lpad(e0 * STRIDE) + r * (d / 16 * 17)];
        else if constexpr ((MUL * STRIDE) % 16 == 0) return p[lpad(e0 * STRIDE) + lpad(r * d)];
        else return p[lpad(e0 * STRIDE + r * d)];
    }
    __device__ __forceinline__ void sync() const
    {
        if constexpr (WAVE) {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        } else {
            __syncthreads();
        }
    }
};

// Keeps the loads issued above it above it: left alone, the scheduler sinks
// each load to its use to save registers, one memory round trip per element.
__device__ __forceinline__ void issue_loads() { __builtin_amdgcn_sched_barrier(0); }

// ------------------------------------------------------------ passes
// Pass I of plan P in direction DIR (forward: plan order, inverse: reversed).
template <class P, int DIR, int I>
struct PassOf {
    static constexpr bool INV = DIR > 0;
    static constexpr int R = P::rad(INV, I), NS = P::ns(INV, I), TWOFF = P::twoff(INV, I);
    static constexpr int T = P::T, nb = P::n / R, B = (nb + T - 1) / T;
    static_assert(B * R <= P::E, "plan exceeds the per-thread element budget");
    __device__ static constexpr bool full() { return nb % T == 0; }
};

// The line elements a thread owns at pass I of direction DIR, where I reads
// (a first pass) or writes (a last pass) the line in natural order: register
// s holds element t + o with o = b*T + r*n/R known at compile time.  BL: the
// line is the first len <= n/2 of the plan's n elements.
//
// The callers load every operand of a step, then compute, then store: a
// store between two loads orders them (the planes may alias) and a wait for
// the later load waits for the store too, a chain of one memory round trip
// per element.
template <class P, int DIR, int I, bool BL = false>
struct Elems {
    using Q = PassOf<P, DIR, I>;
    static_assert(I == 0 || I == P::np - 1, "natural order: the first or the last pass");
    static constexpr int span = BL ? P::n / 2 : P::n;   // len <= span
    int t, len;

    // f(s, o): every element below span
    template <class F>
    __device__ __forceinline__ void all(F &&f) const
    {
#pragma unroll
        for (int b = 0; b < Q::B; ++b) {
            if (Q::full() || t + b * Q::T < Q::nb) {
#pragma unroll
                for (int r = 0; r < Q::R; ++r)
                    if (b * Q::T + r * Q::nb < span) f(b * Q::R + r, b * Q::T + r * Q::nb);
            }
        }
    }
    // f(s, o): operand loads, without the elements that lie past the end of
    // the line for every thread
    template <class F>
    __device__ __forceinline__ void load(F &&f) const
    {
        all([&](int s, int o) {
            if (!BL || o < len) f(s, o);
        });
    }
    // f(s, o): the elements of the line, for stores
    template <class F>
    __device__ __forceinline__ void store(F &&f) const
    {
        all([&](int s, int o) {
            if (inside(o)) f(s, o);
        });
    }
    __device__ __forceinline__ bool inside(int o) const { return !BL || t + o < len; }
};

// twiddles of pass I for this thread's butterflies (none for a first pass)
template <class P, int DIR, int I>
struct TwRegs {
    using Q = PassOf<P, DIR, I>;
    static constexpr int count = Q::NS > 1 ? Q::B * (Q::R - 1) : 0;
    cf w[count > 0 ? count : 1];
};

// global (L1/L2-resident) twiddle loads of pass I; issued before the LDS
// exchange that precedes the pass so their latency overlaps the barrier
template <class P, int DIR, int I>
__device__ __forceinline__ void load_tw(TwRegs<P, DIR, I> &w, const Buf &tw, int t)
{
    using Q = PassOf<P, DIR, I>;
    if constexpr (Q::NS > 1) {
#pragma unroll
        for (int b = 0; b < Q::B; ++b) {
            const int j = t + b * Q::T;
            if (Q::full() || j < Q::nb) {
                const unsigned k = (unsigned) (j % Q::NS);
#pragma unroll
                for (int r = 1; r + 1 < Q::R; r += 2) {
                    const cf2 x = tw.get<cf2>(16u * k, 8u * (Q::TWOFF + tw_index(Q::R, Q::NS, 0, r)));
                    w.w[b * (Q::R - 1) + r - 1] = mkc(x.x, x.y);
                    w.w[b * (Q::R - 1) + r] = mkc(x.z, x.w);
                }
                if constexpr ((Q::R & 1) == 0)
                    w.w[b * (Q::R - 1) + Q::R - 2] =
                        tw.get<cf>(8u * k, 8u * (Q::TWOFF + tw_index(Q::R, Q::NS, 0, Q::R - 1)));
            }
        }
    }
}

// twiddle multiply + radix-R butterflies of pass I, in registers
template <class P, int DIR, int I>
__device__ __forceinline__ void compute_tw(cf (&v)[P::E], const TwRegs<P, DIR, I> &w, int t)
{
    using Q = PassOf<P, DIR, I>;
#pragma unroll
    for (int b = 0; b < Q::B; ++b) {
        const int j = t + b * Q::T;
        if (Q::full() || j < Q::nb) {
            if constexpr (Q::NS > 1) {
#pragma unroll
                for (int r = 1; r < Q::R; ++r)
                    v[b * Q::R + r] = twmul<DIR>(v[b * Q::R + r], w.w[b * (Q::R - 1) + r - 1]);
            }
            bfly<Q::R, DIR>(&v[b * Q::R]);
        }
    }
}

// the first pass of a line whose upper half is 0 (and whose registers there
// are not read)
template <class P, int DIR>
__device__ __forceinline__ void compute_half(cf (&v)[P::E], int t)
{
    using Q = PassOf<P, DIR, 0>;
    static_assert(Q::R == 8 || Q::R == 16, "first radix of a convolution plan");
#pragma unroll
    for (int b = 0; b < Q::B; ++b) {
        if (Q::full() || t + b * Q::T < Q::nb) {
            if constexpr (Q::R == 8) bf8<DIR, true>(&v[b * Q::R]);
            else bf16<DIR, true>(&v[b * Q::R]);
        }
    }
}

template <class P, int DIR, int I>
__device__ __forceinline__ void compute(cf (&v)[P::E], const Buf &tw, int t)
{
    TwRegs<P, DIR, I> w;
    load_tw<P, DIR, I>(w, tw, t);
    compute_tw<P, DIR, I>(v, w, t);
}

// Slots of the exchanges.  Pass I writes its outputs where it read its
// inputs (register r of butterfly j to the slot of input r), so a slot
// belongs to one thread from its read to its next write and an exchange needs
// one barrier, between its writes and its reads, where a fixed slot per
// element needs a second one before the writes.  (2048^2 projection pass:
// 24.0 us with two barriers, 19.9 us with one.)  slot<DIR, I, SECOND>(e) is the slot of
// element e (of the Stockham order: the output positions of pass I-1, the
// input positions of pass I) in the exchange before pass I:
//   I = 1         e itself for the first transform of a chain; the second
//                 transform of a pair (SECOND) starts in the slots that the
//                 last pass of the first one read;
//   I > 1         the slot of the input of pass I-1 that e replaced.
// The radices of the two transforms of a pair are mirrored, so the pair's
// last pass reads the slots its first pass wrote, and the next pair of a
// chain starts over with slot = element.  slot is linear in r along a pass's
// inputs e = j + r*n/R.
template <class P, int DIR, int I, bool SECOND>
__host__ __device__ constexpr unsigned slot(unsigned e)
{
    constexpr bool INV = DIR > 0;
    if constexpr (I == 1) {
        if constexpr (SECOND) {
            constexpr unsigned R = P::rad(INV, 0);
            return slot<P, -DIR, P::np - 1, false>(e / R + (e % R) * (P::n / R));
        } else {
            return e;
        }
    } else {
        constexpr unsigned R = P::rad(INV, I - 1), NS = P::ns(INV, I - 1);
        return slot<P, DIR, I - 1, SECOND>(e / (NS * R) * NS + e % NS + (e / NS) % R * (P::n / R));
    }
}

// slot of input 0 of the thread's butterflies in the latest exchange
template <class P> struct Slots {
    int s[P::E];
};

// inputs of pass I from their slots
template <class P, int DIR, int I, bool SECOND, class Lds>
__device__ __forceinline__ void read_slots(cf (&v)[P::E], int t, const Lds &L, Slots<P> &at)
{
    using Q = PassOf<P, DIR, I>;
    constexpr int STEP = (int) (slot<P, DIR, I, SECOND>(Q::nb) - slot<P, DIR, I, SECOND>(0));
#pragma unroll
    for (int b = 0; b < Q::B; ++b) {
        const int j = t + b * Q::T;
        if (Q::full() || j < Q::nb) {
            at.s[b] = (int) slot<P, DIR, I, SECOND>((unsigned) j);
#pragma unroll
            for (int r = 0; r < Q::R; ++r) v[b * Q::R + r] = L.template at<STEP, 1>(at.s[b], r);
        }
    }
}

// outputs of pass I to the slots its inputs came from, which pass IR of
// direction DR read (the pass itself, or the last pass of the transform
// before it); a chain's first pass has read none and writes slot = element
template <class P, int DIR, int I, int DR, int IR, bool SR, class Lds>
__device__ __forceinline__ void write_slots(const cf (&v)[P::E], int t, const Lds &L, const Slots<P> &at)
{
    using Q = PassOf<P, DIR, I>;
#pragma unroll
    for (int b = 0; b < Q::B; ++b) {
        const int j = t + b * Q::T;
        if (Q::full() || j < Q::nb) {
#pragma unroll
            for (int r = 0; r < Q::R; ++r) {
                if constexpr (IR == 0) {
                    L.template at<1, Q::R>(j * Q::R, r) = v[b * Q::R + r];
                } else {
                    constexpr int STEP = (int) (slot<P, DR, IR, SR>(Q::nb) - slot<P, DR, IR, SR>(0));
                    L.template at<STEP, 1>(at.s[b], r) = v[b * Q::R + r];
                }
            }
        }
    }
}

// passes [I, np) of direction DIR, each preceded by an LDS exchange; SECOND:
// the transform follows one of the other direction in the same registers.
// `hook` loads operands of the step that follows: after the last pass, which
// leaves the pass the registers, or (AHEAD) before its exchange, so that they
// are in flight during the exchange and the pass.
template <class P, int DIR, int I, bool SECOND, bool AHEAD, class Lds, class Hook>
__device__ __forceinline__ void passes_from(cf (&v)[P::E], const Buf &tw, int t, const Lds &L, Slots<P> &at,
                                            Hook &hook)
{
    if constexpr (I == P::np && (P::np == 1 || !AHEAD)) {
        hook();
        issue_loads();
    }
    if constexpr (I < P::np) {
        TwRegs<P, DIR, I> w;
        load_tw<P, DIR, I>(w, tw, t);
        if constexpr (I == P::np - 1 && AHEAD) hook();
        issue_loads();
        if constexpr (I > 1) write_slots<P, DIR, I - 1, DIR, I - 1, SECOND>(v, t, L, at);
        else if constexpr (SECOND) write_slots<P, DIR, 0, -DIR, P::np - 1, false>(v, t, L, at);
        else write_slots<P, DIR, 0, DIR, 0, false>(v, t, L, at);
        L.sync();
        read_slots<P, DIR, I, SECOND>(v, t, L, at);
        compute_tw<P, DIR, I>(v, w, t);
        passes_from<P, DIR, I + 1, SECOND, AHEAD>(v, tw, t, L, at, hook);
    }
}

struct NoHook {
    __device__ __forceinline__ void operator()() const {}
};

// One full transform: src(v, in) fills the registers of the first pass,
// dst(v, out) stores those of the last; pre(out) loads operands of dst.
template <class P, int DIR, class Lds, class Src, class Pre, class Dst>
__device__ __forceinline__ void line_fft(cf (&v)[P::E], const Buf &tw, int t, const Lds &L, Src &src,
                                         Pre &pre, Dst &dst)
{
    const Elems<P, DIR, 0> in{t, P::n};
    const Elems<P, DIR, P::np - 1> out{t, P::n};
    auto hook = [&] { pre(out); };
    src(v, in);
    issue_loads();
    compute<P, DIR, 0>(v, tw, t);
    Slots<P> sl;
    passes_from<P, DIR, 1, false, false>(v, tw, t, L, sl, hook);
    dst(v, out);
}

// Transform in direction DA, elementwise `mid` on its natural-order output,
// then the transform in direction DB.  A's last pass and B's first pass
// have the same radix (mirrored sequences), so the junction never leaves
// registers: B's first pass consumes exactly the positions A's last pass
// produced in the same thread.  `pre(at)` loads the operands of `mid` from
// global memory, WHEN (a variant the autotuner picks by size): at the
// junction itself, which costs no registers during the transform; ahead of
// the first transform's last exchange; or early, right after the input
// gather, in flight during the whole first transform.
enum { kAtJunction = 0, kAhead = 1, kEarly = 2 };

template <class P, int DA, int DB, int WHEN, class Lds, class Src, class Pre, class Mid, class Dst>
__device__ __forceinline__ void line_pair(cf (&v)[P::E], const Buf &tw, int t, const Lds &L, Src &src,
                                          Pre &pre, Mid &mid, Dst &dst)
{
    static_assert(DA == -DB, "a pair runs opposite directions");
    static_assert(P::rad(DA > 0, P::np - 1) == P::rad(DB > 0, 0), "mirrored junction radix");
    const Elems<P, DA, 0> in{t, P::n};
    const Elems<P, DA, P::np - 1> at{t, P::n};
    const Elems<P, DB, P::np - 1> out{t, P::n};
    auto hook = [&] { if constexpr (WHEN != kEarly) pre(at); };
    NoHook none;
    src(v, in);
    if constexpr (WHEN == kEarly) pre(at);
    issue_loads();
    compute<P, DA, 0>(v, tw, t);
    Slots<P> sl;
    passes_from<P, DA, 1, false, WHEN == kAhead>(v, tw, t, L, sl, hook);
    mid(v, at);
    compute<P, DB, 0>(v, tw, t);
    passes_from<P, DB, 1, true, false>(v, tw, t, L, sl, none);
    dst(v, out);
}

// ------------------------------------------------------------ reductions
// std::max / std::min semantics of the reference reductions
__device__ __forceinline__ float fmax_ref(float m, float x) { return (m < x) ? x : m; }
__device__ __forceinline__ float fmin_ref(float m, float x) { return (x < m) ? x : m; }

}  // namespace imr
