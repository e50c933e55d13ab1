// Row-pass kernels (one workgroup = P::L rows of length W = P::n, P::T
// threads per row).  Compiled once per plan group (-DIMR_GROUP=g).
//
//   RK_MID    inverse row FFT -> HIO constraint (mask, gPrev) -> forward row FFT
//             The steady-state half of an HIO iteration: the inverse 2-D FFT of
//             the previous iteration is finished here (its column half ran in
//             the column pass) and the forward 2-D FFT of this iteration starts
//             here, with the constraint (cudaVectorElementwise.cu:42-72)
//             applied in registers in between.
//   RK_FIRST  first iteration of a cycle: g' is already in real space; the
//             mask cut-off (cudaVectorElementwise.cu:198-219 with the device
//             threshold) is fused into the load, then constraint + forward FFT.
//   RK_INVOUT inverse row FFT closing a reconstruction step: writes g' and,
//             by its output set, gPrev = g' (cudaShrinkWrap.cu:304-309), |g'| for the
//             blur (:240) and the HIO error sums (cudaVectorReduce.cu:284-355).
//   RK_FWD / RK_INV  plain row transforms of the 2-D FFT entry point;
//            RK_FWD_NORM stores |z| of the forward one (the forward model).
#include "internal.hpp"
#include "blue_device.hpp"
#include "ops_device.hpp"
#include "plans.hpp"

#ifndef IMR_GROUP
#error "compile with -DIMR_GROUP=<plan group>"
#endif

namespace imr {

namespace {

enum RowKernel { RK_FWD, RK_INV, RK_INVOUT, RK_FIRST, RK_MID, RK_FWD_NORM };

// NL rows per workgroup; WHEN (RK_MID only): where gPrev and the mask are
// read (line_pair); BL: Bluestein kernels of row length a.len with P the
// convolution plan; FL (RK_INVOUT, RK_FIRST): the kRow* outputs / cut-off,
// fixed at compile time (a uniform runtime flag tested per element slows the
// memory phases measurably).  At least 4 waves per SIMD: with fewer, 2048
// rows of 2048 points no longer run as one generation of workgroups.
template <class P, int NL, int K, int WHEN = kAtJunction, bool BL = false, int FL = 0>
__global__ void __launch_bounds__(NL *P::T, 4) k_row(RowArgs a)
{
    // image b of a batch (grid.y): its planes start b * istride elements in,
    // its scalars at b * kScalStride / kFlagStride
    const int b = blockIdx.y;
    if (a.done != nullptr && a.done[b * kFlagStride]) return;
    extern __shared__ cf smem[];
    constexpr int T = P::T;
    const int n = BL ? a.len : P::n;
    const int l = threadIdx.x / T, t = threadIdx.x - l * T;
    // planes from the workgroup's first row to the image's last: loads of the
    // rows past the end return 0, and so do those of lanes past the end of a
    // Bluestein line (at), where the next row begins: another workgroup may be
    // rewriting it, and a value that overflowed there must not come in
    const size_t wb = (size_t) b * a.istride + (size_t) blockIdx.x * NL * n;
    const size_t left = (size_t) (a.H - (int) blockIdx.x * NL) * n;
    const unsigned e0 = (unsigned) (l * n + t);
    const bool valid = (int) blockIdx.x * NL + l < a.H;
    const Buf X(a.X + wb, 8 * left), G(a.G + wb, 8 * left), mask(a.mask + wb, left), Bn(a.Bn + wb, 4 * left);
    const Blue bl{n, Buf(a.bs, 8 * (size_t) (P::n / 2 + 2 * P::n))};
    const Buf tw(a.tw, 8 * (size_t) (2 * P::n - 1));
    const LdsLine<1, 64 % T == 0> L{smem + l * lds_elems(P::n)};
    cf v[P::E];
    auto at = [](unsigned e, const auto &el, int o) { return el.inside(o) ? e : kOutside; };
    auto ld = [&](const Buf &p) {
        return [&](auto &x, const auto &el) {
            el.load([&](int s, int o) { x[s] = p.template get<cf>(at(8 * e0, el, o), 8 * o); });
        };
    };
    auto st = [&](const Buf &p) {
        return [&](auto &x, const auto &el) {
            if (valid) el.store([&](int s, int o) { p.put(x[s], 8 * e0, 8 * o); });
        };
    };
    auto none = [](const auto &) {};
    auto stX = st(X);
    // The constraint runs over initialised operands and every element: over
    // operands that only el.load's branches set, in branches of its own, the
    // compiler kept all of it live at once (Bluestein RK_FIRST of 64- and
    // 512-point convolutions: 1849 and 1293 spilled registers; a 250^2
    // reconstruction of 4 cycles 332 us, 252 us like this)

    if constexpr (K == RK_FWD || K == RK_INV || K == RK_FWD_NORM) {
        const Buf in(a.in + wb, 8 * left);
        auto g0 = ld(in);
        if constexpr (K == RK_FWD_NORM) {
            // the last half of the forward model |FFT2(x)|
            // (diffractionIntensity.cpp:72-77): only |z| leaves the registers
            auto sl = [&](auto &x, const auto &el) {
                if (valid) el.store([&](int s, int o) { Bn.put(cnorm(x[s]), 4 * e0, 4 * o); });
            };
            xfft<P, -1, BL>(v, tw, t, L, bl, g0, none, sl);
        } else {
            const Buf out(a.out + wb, 8 * left);
            auto sl = st(out);
            xfft<P, K == RK_FWD ? -1 : +1, BL>(v, tw, t, L, bl, g0, none, sl);
        }
    } else if constexpr (K == RK_INVOUT) {
        __shared__ float red_f[NL * P::T];
        __shared__ unsigned red_u[NL * P::T];
        constexpr int fl = FL;
        float err = 0.f;
        unsigned cnt = 0;
        uint8_t m[P::E];
        auto ldX = ld(X);
        auto pre = [&](const auto &el) {
            if constexpr ((fl & kRowError) != 0)
                el.load([&](int s, int o) { m[s] = mask.get<uint8_t>(at(e0, el, o), o); });
        };
        auto sl = [&](auto &x, const auto &el) {
            if (!valid) return;
            el.store([&](int s, int o) {
                X.put(x[s], 8 * e0, 8 * o);
                if constexpr ((fl & kRowWriteG) != 0) G.put(x[s], 8 * e0, 8 * o);
                if constexpr ((fl & (kRowWriteBn | kRowError)) != 0) {
                    const float nrm = cnorm(x[s]);
                    if constexpr ((fl & kRowWriteBn) != 0) Bn.put(nrm, 4 * e0, 4 * o);
                    if constexpr ((fl & kRowError) != 0) {
                        if (m[s]) {
                            err += nrm;
                            cnt += 1;
                        }
                    }
                }
            });
        };
        xfft<P, +1, BL>(v, tw, t, L, bl, ldX, pre, sl);
        if constexpr ((fl & kRowError) != 0) {
            err = block_reduce(err, red_f, [](float x, float y) { return x + y; });
            cnt = block_reduce(cnt, red_u, [](unsigned x, unsigned y) { return x + y; });
            if (threadIdx.x == 0) {
                a.perr[b * gridDim.x + blockIdx.x] = err;
                a.pcnt[b * gridDim.x + blockIdx.x] = cnt;
            }
        }
    } else if constexpr (K == RK_FIRST) {
        constexpr bool cut = (FL & kRowCut) != 0;
        const float thr = cut ? a.thr[b * kScalStride] : 0.f;
        const Buf B2(a.B2 + wb, 4 * left);
        const float beta = a.beta;
        auto g0 = [&](auto &x, const auto &el) {
            cf g[P::E] = {};
            float bv[P::E] = {};
            uint8_t m[P::E] = {};
            el.load([&](int s, int o) {
                x[s] = X.get<cf>(at(8 * e0, el, o), 8 * o);
                g[s] = G.get<cf>(at(8 * e0, el, o), 8 * o);
                if constexpr (cut) bv[s] = B2.get<float>(at(4 * e0, el, o), 4 * o);
                else m[s] = mask.get<uint8_t>(at(e0, el, o), o);
            });
            el.all([&](int s, int) {
                if constexpr (cut) m[s] = bv[s] < thr ? 1 : 0;
                x[s] = hio_constraint(g[s], x[s], m[s] == 1, beta);
            });
            if (!valid) return;
            el.store([&](int s, int o) {
                if constexpr (cut) mask.put(m[s], e0, o);
                G.put(x[s], 8 * e0, 8 * o);
            });
        };
        xfft<P, -1, BL>(v, tw, t, L, bl, g0, none, stX);
    } else if constexpr (K == RK_MID) {
        const float beta = a.beta;
        cf g[P::E] = {};
        uint8_t m[P::E] = {};
        auto ldX = ld(X);
        auto pre = [&](const auto &el) {
            el.load([&](int s, int o) {
                g[s] = G.get<cf>(at(8 * e0, el, o), 8 * o);
                m[s] = mask.get<uint8_t>(at(e0, el, o), o);
            });
        };
        auto mid = [&](auto &x, const auto &el) {
            el.all([&](int s, int) { x[s] = hio_constraint(g[s], x[s], m[s] == 1, beta); });
            if (valid) el.store([&](int s, int o) { G.put(x[s], 8 * e0, 8 * o); });
        };
        xpair<P, +1, -1, BL, WHEN>(v, tw, t, L, bl, ldX, pre, mid, stX);
    }
}

// the output sets of the closing row pass
constexpr int kInit = kRowWriteG | kRowWriteBn;
constexpr int kLast = kRowWriteBn | kRowError;
constexpr int kInitErr = kRowWriteG | kRowWriteBn | kRowError;

// LDS bytes of an NL-row group
template <int NL>
constexpr size_t row_lds(int n) { return sizeof(cf) * (size_t) NL * lds_elems(n); }

template <class P, int NL, int WHEN = kAtJunction, bool BL = false>
int launch_variant(int mode, RowArgs a, hipStream_t s)
{
    static_assert(NL * P::T <= 1024, "row workgroup too large");
    const dim3 grid((a.H + NL - 1) / NL, a.batch > 1 ? a.batch : 1), block(NL * P::T);
    constexpr size_t lds = row_lds<NL>(P::n);
    static_assert(lds <= kLdsBudget, "row tile exceeds the LDS budget");
    constexpr int AJ = kAtJunction;
    if constexpr (lds > 64 * 1024) {
        static const hipError_t attr = [&] {
            hipError_t e = hipSuccess;
            for (const void *f : {(const void *) k_row<P, NL, RK_FWD, AJ, BL>,
                                  (const void *) k_row<P, NL, RK_FWD_NORM, AJ, BL>,
                                  (const void *) k_row<P, NL, RK_INV, AJ, BL>,
                                  (const void *) k_row<P, NL, RK_INVOUT, AJ, BL, kInit>,
                                  (const void *) k_row<P, NL, RK_INVOUT, AJ, BL, kLast>,
                                  (const void *) k_row<P, NL, RK_INVOUT, AJ, BL, 0>,
                                  (const void *) k_row<P, NL, RK_INVOUT, AJ, BL, kInitErr>,
                                  (const void *) k_row<P, NL, RK_FIRST, AJ, BL, kRowCut>,
                                  (const void *) k_row<P, NL, RK_FIRST, AJ, BL, 0>,
                                  (const void *) k_row<P, NL, RK_MID, WHEN, BL>})
                if (e == hipSuccess)
                    e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds);
            return e;
        }();
        if (attr != hipSuccess) return from_hip(attr);
    }
    switch (mode) {
    case ROW_FWD: IMR_LAUNCH((k_row<P, NL, RK_FWD, AJ, BL>), grid, block, lds, s, a); break;
    case ROW_FWD_NORM: IMR_LAUNCH((k_row<P, NL, RK_FWD_NORM, AJ, BL>), grid, block, lds, s, a); break;
    case ROW_INV: IMR_LAUNCH((k_row<P, NL, RK_INV, AJ, BL>), grid, block, lds, s, a); break;
    case ROW_INIT: IMR_LAUNCH((k_row<P, NL, RK_INVOUT, AJ, BL, kInit>), grid, block, lds, s, a); break;
    case ROW_LAST: IMR_LAUNCH((k_row<P, NL, RK_INVOUT, AJ, BL, kLast>), grid, block, lds, s, a); break;
    case ROW_LAST_PLAIN: IMR_LAUNCH((k_row<P, NL, RK_INVOUT, AJ, BL, 0>), grid, block, lds, s, a); break;
    case ROW_INIT_ERR: IMR_LAUNCH((k_row<P, NL, RK_INVOUT, AJ, BL, kInitErr>), grid, block, lds, s, a); break;
    case ROW_FIRST_CUT: IMR_LAUNCH((k_row<P, NL, RK_FIRST, AJ, BL, kRowCut>), grid, block, lds, s, a); break;
    case ROW_FIRST_MASK: IMR_LAUNCH((k_row<P, NL, RK_FIRST, AJ, BL, 0>), grid, block, lds, s, a); break;
    case ROW_MID: IMR_LAUNCH((k_row<P, NL, RK_MID, WHEN, BL>), grid, block, lds, s, a); break;
    default: return IMRESH_ERR_INVALID;
    }
    return imr::launch_status(__FILE__, __LINE__);
}

// Row variants of a length: index = when * shapes + shape.  `when` is where
// RK_MID reads gPrev and the mask (line_pair); shape 0 has ~256-thread
// groups, shape 1 fewer rows per group: half of them for 1024 and 2048
// points (fewer waves share each barrier, so the groups of a CU drift out of
// phase and overlap one's loads with another's arithmetic), a quarter for up
// to 512 points (4x the workgroups spread one small image over more CUs).
template <int N, int... Rs>
constexpr int small_group()
{
    using P = Plan<N, Rs...>;
    if (N <= 512 && P::L >= 8) return P::L / 4;
    if (N >= 1024 && (N & (N - 1)) == 0 && P::L >= 2) return P::L / 2;
    return 0;
}

template <int N, int... Rs>
constexpr int row_shape_count() { return small_group<N, Rs...>() > 0 ? 2 : 1; }

template <int N, int... Rs>
constexpr int row_variant_count() { return 3 * row_shape_count<N, Rs...>(); }

// Bluestein kernels exist for the power-of-two convolution lengths, with half
// the plan's rows per group (a mid-size image over more CUs)
template <int N>
constexpr bool blue_length() { return N >= 64 && N <= 2 * kMaxLine && (N & (N - 1)) == 0; }

template <class P>
constexpr int blue_rows() { return P::L > 1 ? P::L / 2 : 1; }

template <class P, int NL>
int launch_when(int when, int mode, RowArgs a, hipStream_t s)
{
    if (when == kEarly) return launch_variant<P, NL, kEarly>(mode, a, s);
    if (when == kAhead) return launch_variant<P, NL, kAhead>(mode, a, s);
    return launch_variant<P, NL>(mode, a, s);
}

template <int N, int... Rs>
int launch_row_variant(int var, int mode, RowArgs a, hipStream_t s)
{
    using P = Plan<N, Rs...>;
    if constexpr (blue_length<N>()) {
        if (var == kBlueVariant) return launch_variant<P, blue_rows<P>(), kAtJunction, true>(mode, a, s);
    }
    if constexpr (N > kMaxLine) {
        return IMRESH_ERR_UNSUPPORTED_SIZE;   // a convolution length only
    } else {
        constexpr int ns = row_shape_count<N, Rs...>();
        var %= row_variant_count<N, Rs...>();
        if constexpr (ns > 1) {
            if (var % ns == 1) return launch_when<P, small_group<N, Rs...>()>(var / ns, mode, a, s);
        }
        return launch_when<P, P::L>(var / ns, mode, a, s);
    }
}

// rows per workgroup of a variant (the host needs it for the partial sums;
// its buffers hold one slot per row, enough for any variant)
template <int N, int... Rs>
int row_variant_rows(int var)
{
    using P = Plan<N, Rs...>;
    if (var == kBlueVariant) return blue_rows<P>();
    constexpr int ns = row_shape_count<N, Rs...>();
    var %= row_variant_count<N, Rs...>();
    return var % ns == 1 ? small_group<N, Rs...>() : P::L;
}

template <int G, int N, int... Rs>
int try_plan(int mode, int var, int n, RowArgs a, hipStream_t s)
{
    if constexpr (G == IMR_GROUP) {
        if (n == N) return launch_row_variant<N, Rs...>(var, mode, a, s);
    }
    return -1;
}

template <int G, int N, int... Rs>
int try_count(int n)
{
    if constexpr (G == IMR_GROUP) {
        if (n == N) return row_variant_count<N, Rs...>();
    }
    return -1;
}

template <int G, int N, int... Rs>
int try_rows(int n, int var)
{
    if constexpr (G == IMR_GROUP) {
        if (n == N) return row_variant_rows<N, Rs...>(var);
    }
    return -1;
}

}  // namespace

#define IMR_CAT2(a, b) a##b
#define IMR_CAT(a, b) IMR_CAT2(a, b)
#define IMR_ROW_CASE(g, N, ...)                                                     \
    {                                                                               \
        const int r = try_plan<g, N, __VA_ARGS__>(mode, var, n, a, s);              \
        if (r >= 0) return r;                                                       \
    }
#define IMR_ROW_COUNT(g, N, ...)                                                    \
    {                                                                               \
        const int r = try_count<g, N, __VA_ARGS__>(n);                              \
        if (r >= 0) return r;                                                       \
    }

int IMR_CAT(launch_row_g, IMR_GROUP)(int mode, int var, int n, const LinePlan &lp, RowArgs a,
                                     hipStream_t s)
{
    a.tw = lp.tw;
    IMR_PLANS(IMR_ROW_CASE)
    return IMRESH_ERR_UNSUPPORTED_SIZE;
}

int IMR_CAT(row_variants_g, IMR_GROUP)(int n)
{
    IMR_PLANS(IMR_ROW_COUNT)
    return 0;
}

#define IMR_ROW_ROWS(g, N, ...)                                                     \
    {                                                                               \
        const int r = try_rows<g, N, __VA_ARGS__>(n, var);                          \
        if (r >= 0) return r;                                                       \
    }

int IMR_CAT(row_rows_g, IMR_GROUP)(int n, int var)
{
    IMR_PLANS(IMR_ROW_ROWS)
    return 1;
}

}  // namespace imr
