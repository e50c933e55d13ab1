// Host check of the LDS slots of csrc/fft_device.hpp for every compiled plan:
// chains of transforms as the kernels run them (forward, inverse, forward,
// ... and the other way round) are replayed on an array of slots.  In every
// exchange a pass must write each slot once, only slots that the writing
// thread itself read last (no barrier orders the write after another thread's
// read), and the next pass must find its inputs, at a constant step.
#include <cstdio>
#include <vector>

#include "fft_device.hpp"
#include "plans.hpp"

using namespace imr;

template <class P, int DIR, int I, bool SECOND>
bool exchange(std::vector<int> &owner)
{
    constexpr bool INV = DIR > 0;
    constexpr int R = P::rad(INV, I - 1), NS = P::ns(INV, I - 1), nb = P::n / R;
    std::vector<int> at(P::n, -1);   // slot -> element written
    for (int j = 0; j < nb; ++j)
        for (int r = 0; r < R; ++r) {
            const int k = j % NS, e = (j - k) * R + k + r * NS;
            unsigned s;
            if constexpr (I > 1) s = slot<P, DIR, I - 1, SECOND>(j + r * nb);
            else if constexpr (SECOND) s = slot<P, -DIR, P::np - 1, false>(j + r * nb);
            else s = j * R + r;
            if (s >= (unsigned) P::n || at[s] >= 0) return false;
            if (owner[s] >= 0 && owner[s] != j % P::T) return false;
            at[s] = e;
        }
    constexpr int R2 = P::rad(INV, I), nb2 = P::n / R2;
    const unsigned step = slot<P, DIR, I, SECOND>(nb2) - slot<P, DIR, I, SECOND>(0);
    for (int j = 0; j < nb2; ++j)
        for (int r = 0; r < R2; ++r) {
            const unsigned s = slot<P, DIR, I, SECOND>(j + r * nb2);
            if (s >= (unsigned) P::n || s != slot<P, DIR, I, SECOND>(j) + r * step) return false;
            if (at[s] != j + r * nb2) return false;
            owner[s] = j % P::T;
        }
    if constexpr (I + 1 < P::np) return exchange<P, DIR, I + 1, SECOND>(owner);
    return true;
}

template <class P, int DIR>
bool chain()
{
    std::vector<int> owner(P::n, -1);
    for (int rep = 0; rep < 2; ++rep)
        if (!exchange<P, DIR, 1, false>(owner) || !exchange<P, -DIR, 1, true>(owner)) return false;
    return true;
}

template <int G, int N, int... Rs>
int check()
{
    using P = Plan<N, Rs...>;
    if constexpr (P::np > 1) {
        if (!chain<P, -1>() || !chain<P, +1>()) {
            std::printf("plan of length %d: wrong slots\n", N);
            return 1;
        }
    }
    return 0;
}

#define CHECK(g, N, ...) +check<g, N, __VA_ARGS__>()

int main()
{
    const int bad = 0 IMR_PLANS(CHECK);
    std::printf("%d plans with wrong slots\n", bad);
    return bad != 0;
}
