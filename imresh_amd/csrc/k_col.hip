// Column-pass kernels (one workgroup = P::C adjacent columns of length
// H = P::n, the tile staged in LDS as [H][C], P::T threads per column).
// Compiled once per plan group (-DIMR_GROUP=g).
//
//   CK_PROJ  forward column FFT -> modulus projection -> inverse column FFT.
//            Finishes the forward 2-D FFT of an HIO iteration, replaces |G'|
//            by the measured modulus (cudaVectorElementwise.cu:168-195) in
//            registers, and starts the inverse 2-D FFT.
//   CK_INV   inverse column transform; CK_INV_REAL reads the real modulus M
//            instead, the first half of IFFT2((M, 0)) (cudaShrinkWrap.cu:229-232).
//   CK_FWD   forward column transform of the 2-D FFT entry point;
//            CK_FWD_REAL reads a real plane instead, the first half of the
//            forward model FFT2((x, 0)) (diffractionIntensity.cpp:59-70).
#include "internal.hpp"
#include "blue_device.hpp"
#include "ops_device.hpp"
#include "plans.hpp"

#ifndef IMR_GROUP
#error "compile with -DIMR_GROUP=<plan group>"
#endif

namespace imr {

namespace {

enum ColKernel { CK_FWD, CK_INV, CK_PROJ, CK_FWD_REAL, CK_INV_REAL };

// C columns per workgroup; WHEN (CK_PROJ only): where the measured modulus
// is read (line_pair); BL: Bluestein kernels of column length a.len with P
// the convolution plan.  At least 4 waves per SIMD; 3 for 32 points, whose 132
// registers spill under the bound of 128 (64x32: 4.6 us, 4.1 so).
template <class P, int C, int K, int WHEN = kAtJunction, bool BL = false>
__global__ void __launch_bounds__(C *P::T, P::n == 32 ? 3 : 4) k_col(ColArgs a)
{
    // XCD-aware tile order: workgroups are dealt round-robin to the 8 XCDs
    // (workgroup x + y * gridDim.x to XCD (x + y * gridDim.x) mod 8), each
    // with its own L2; give every XCD a contiguous range of tiles so
    // neighbouring tiles (which share 128-byte lines of X and M) meet in the
    // same L2.  A grid whose width is a multiple of 8 keeps its images in
    // place and remaps within each row of tiles; any other grid is remapped
    // as a whole (consecutive tiles, of one image and the next, per XCD).
    int bid = blockIdx.x, by = blockIdx.y;
    if ((gridDim.x & 7) == 0) {
        bid = (bid & 7) * (gridDim.x >> 3) + (bid >> 3);
    } else {
        const int gx = gridDim.x, nt = gx * gridDim.y, lin = bid + by * gx;
        const int x8 = lin & 7, k = x8 * (nt >> 3) + min(x8, nt & 7) + (lin >> 3);
        bid = k % gx;
        by = k / gx;
    }
    // image b of a batch and, for the middle step of a four-step column
    // pass, its sub-block sb (grid.y = images x sub)
    const int sub = a.sub > 1 ? a.sub : 1;
    const int b = by / sub, sb = by - b * sub;
    if (a.done != nullptr && a.done[b * kFlagStride]) return;
    extern __shared__ cf smem[];
    const int c = threadIdx.x % C, t = threadIdx.x / C;
    const int col = bid * C + c;
    const bool valid = col < a.W;
    const int W = a.W;
    const int n = BL ? a.len : P::n;
    const size_t wb = (size_t) b * a.istride + (size_t) sb * a.sub_xstride + (size_t) bid * C;
    // planes from the tile's first element to the block's last row; lanes of
    // columns past the edge load past every end
    const size_t left = (size_t) n * W - (size_t) bid * C;
    const unsigned c0 = (unsigned) c, out_of = valid ? 0u : kOutside;
    const unsigned x0 = ((unsigned) (t * W) + c0) * 8u | out_of;
    const LdsLine<C, false> L{smem + c};
    const Buf tw(a.tw, 8 * (size_t) (2 * P::n - 1));
    const Blue bl{n, Buf(a.bs, 8 * (size_t) (P::n / 2 + 2 * P::n))};
    cf v[P::E];
    auto ld = [&](const Buf &p) {
        return [&](auto &x, const auto &el) {
            el.load([&](int s, int o) { x[s] = p.template get<cf>(x0, 8u * (unsigned) o * (unsigned) W); });
        };
    };
    auto st = [&](const Buf &p) {
        return [&](auto &x, const auto &el) {
            if (valid) el.store([&](int s, int o) { p.put(x[s], x0, 8u * (unsigned) o * (unsigned) W); });
        };
    };
    auto none = [](const auto &) {};

    if constexpr (K == CK_FWD || K == CK_INV || K == CK_FWD_REAL || K == CK_INV_REAL) {
        constexpr bool real_in = K == CK_FWD_REAL || K == CK_INV_REAL;
        constexpr int DIR = (K == CK_FWD || K == CK_FWD_REAL) ? -1 : +1;
        const Buf out(a.out + wb, 8 * left);
        auto sl = st(out);
        if constexpr (real_in) {
            const Buf M(a.M + wb, 4 * left);
            const unsigned m0 = ((unsigned) (t * W) + c0) * 4u | out_of;
            auto g0 = [&](auto &x, const auto &el) {
                el.load([&](int s, int o) {
                    x[s] = mkc(M.get<float>(m0, 4u * (unsigned) o * (unsigned) W), 0.f);
                });
            };
            xfft<P, DIR, BL>(v, tw, t, L, bl, g0, none, sl);
        } else {
            const Buf in(a.in + wb, 8 * left);
            auto g0 = ld(in);
            xfft<P, DIR, BL>(v, tw, t, L, bl, g0, none, sl);
        }
    } else if constexpr (K == CK_PROJ) {
        const int MP = a.mpitch > 0 ? a.mpitch : W;   // row pitch of M
        const size_t mb = (size_t) b * a.istride + (size_t) sb * a.sub_mstride + (size_t) bid * C;
        const Buf X(a.X + wb, 8 * left);
        const Buf M(a.M + mb, 4 * ((size_t) (n - 1) * MP + W - (size_t) bid * C));
        const unsigned m0 = ((unsigned) (t * MP) + c0) * 4u | out_of;
        float m[P::E] = {};   // 0 past the end of a line
        auto g0 = ld(X);
        auto pre = [&](const auto &el) {
            el.load([&](int s, int o) { m[s] = M.get<float>(m0, 4u * (unsigned) o * (unsigned) MP); });
        };
        auto mid = [&](auto &x, const auto &el) { modulus_project_line<P::E>(x, m, el, valid); };
        auto sl = st(X);
        xpair<P, -1, +1, BL, WHEN>(v, tw, t, L, bl, g0, pre, mid, sl);
    }
}

// LDS bytes of a C-column tile
template <class P, int C>
constexpr size_t col_lds() { return sizeof(cf) * (size_t) lds_elems(C * P::n); }

template <class P, int C, int WHEN = kAtJunction, bool BL = false>
int launch_variant(int mode, ColArgs a, hipStream_t s)
{
    static_assert(C * P::T <= 1024, "column workgroup too large");
    static_assert(col_lds<P, C>() <= kLdsBudget, "column tile exceeds the LDS budget");
    const int images = a.batch > 1 ? a.batch : 1;
    const dim3 grid((a.W + C - 1) / C, images * (a.sub > 1 ? a.sub : 1)), block(C * P::T);
    constexpr size_t lds = col_lds<P, C>();
    constexpr int AJ = kAtJunction;
    // the longest plans' projection pass is the four-step one
    constexpr bool proj = BL || P::n < kFourStepMinLine;
    if constexpr (lds > 64 * 1024) {
        static const hipError_t attr = [&] {
            hipError_t e = hipSuccess;
            for (const void *f : {(const void *) k_col<P, C, CK_FWD, AJ, BL>,
                                  (const void *) k_col<P, C, CK_INV, AJ, BL>,
                                  (const void *) k_col<P, C, CK_FWD_REAL, AJ, BL>,
                                  (const void *) k_col<P, C, CK_INV_REAL, AJ, BL>})
                if (e == hipSuccess)
                    e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds);
            if constexpr (proj)
                if (e == hipSuccess)
                    e = hipFuncSetAttribute((const void *) k_col<P, C, CK_PROJ, WHEN, BL>,
                                            hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds);
            return e;
        }();
        if (attr != hipSuccess) return from_hip(attr);
    }
    switch (mode) {
    case COL_FWD: IMR_LAUNCH((k_col<P, C, CK_FWD, AJ, BL>), grid, block, lds, s, a); break;
    case COL_REAL_FWD: IMR_LAUNCH((k_col<P, C, CK_FWD_REAL, AJ, BL>), grid, block, lds, s, a); break;
    case COL_INV: IMR_LAUNCH((k_col<P, C, CK_INV, AJ, BL>), grid, block, lds, s, a); break;
    case COL_INIT:
        a.out = a.X;
        IMR_LAUNCH((k_col<P, C, CK_INV_REAL, AJ, BL>), grid, block, lds, s, a);
        break;
    case COL_PROJ:
        if constexpr (proj) IMR_LAUNCH((k_col<P, C, CK_PROJ, WHEN, BL>), grid, block, lds, s, a);
        else return IMRESH_ERR_INVALID;
        break;
    default: return IMRESH_ERR_INVALID;
    }
    return imr::launch_status(__FILE__, __LINE__);
}

// Column variants of a length: index = when * shapes + shape.  `when` is where
// CK_PROJ reads the modulus (line_pair; one choice where that pass is the
// four-step one, whose middle step reads it at the junction); shape 0 has the plan's tile, shape 1
// (1024 and 2048 points) 4-column tiles, twice the workgroups.
template <int N, int... Rs>
constexpr int col_shape_count()
{
    return N >= 1024 && (N & (N - 1)) == 0 && Plan<N, Rs...>::C > 4 ? 2 : 1;
}

template <int N, int... Rs>
constexpr int col_variant_count() { return (N < kFourStepMinLine ? 3 : 1) * col_shape_count<N, Rs...>(); }

// Bluestein kernels exist for the power-of-two convolution lengths, with half
// as many columns per tile as the plan (measured fastest, see kBlueVariant)
template <int N>
constexpr bool blue_length() { return N >= 64 && N <= 2 * kMaxLine && (N & (N - 1)) == 0; }

template <class P, int C>
int launch_when(int when, int mode, ColArgs a, hipStream_t s)
{
    if constexpr (P::n < kFourStepMinLine) {
        if (when == kEarly) return launch_variant<P, C, kEarly>(mode, a, s);
        if (when == kAhead) return launch_variant<P, C, kAhead>(mode, a, s);
    }
    return launch_variant<P, C>(mode, a, s);
}

template <int N, int... Rs>
int launch_col_variant(int var, int mode, ColArgs a, hipStream_t s)
{
    using P = Plan<N, Rs...>;
    if constexpr (blue_length<N>()) {
        if (var == kBlueVariant)
            return launch_variant<P, (P::C >= 2 ? P::C / 2 : 1), kAtJunction, true>(mode, a, s);
    }
    if constexpr (N > kMaxLine) {
        return IMRESH_ERR_UNSUPPORTED_SIZE;   // a convolution length only
    } else {
        constexpr int ns = col_shape_count<N, Rs...>();
        var %= col_variant_count<N, Rs...>();
        if constexpr (ns > 1) {
            if (var % ns == 1) return launch_when<P, 4>(var / ns, mode, a, s);
        }
        return launch_when<P, P::C>(var / ns, mode, a, s);
    }
}

template <int G, int N, int... Rs>
int try_plan(int mode, int var, int n, ColArgs a, hipStream_t s)
{
    if constexpr (G == IMR_GROUP) {
        if (n == N) return launch_col_variant<N, Rs...>(var, mode, a, s);
    }
    return -1;
}

template <int G, int N, int... Rs>
int try_count(int n)
{
    if constexpr (G == IMR_GROUP) {
        if (n == N) return col_variant_count<N, Rs...>();
    }
    return -1;
}

}  // namespace

#define IMR_CAT2(a, b) a##b
#define IMR_CAT(a, b) IMR_CAT2(a, b)
#define IMR_COL_CASE(g, N, ...)                                                     \
    {                                                                               \
        const int r = try_plan<g, N, __VA_ARGS__>(mode, var, n, a, s);              \
        if (r >= 0) return r;                                                       \
    }
#define IMR_COL_COUNT(g, N, ...)                                                    \
    {                                                                               \
        const int r = try_count<g, N, __VA_ARGS__>(n);                              \
        if (r >= 0) return r;                                                       \
    }

int IMR_CAT(launch_col_g, IMR_GROUP)(int mode, int var, int n, const LinePlan &lp, ColArgs a,
                                     hipStream_t s)
{
    a.tw = lp.tw;
    IMR_PLANS(IMR_COL_CASE)
    return IMRESH_ERR_UNSUPPORTED_SIZE;
}

int IMR_CAT(col_variants_g, IMR_GROUP)(int n)
{
    IMR_PLANS(IMR_COL_COUNT)
    return 0;
}

}  // namespace imr
