// Host check of the exact shortcuts of csrc/poisson_device.hpp: the float root
// of a count equals the double root's for every count below 2^24, and a
// division by a small integer through its two-part reciprocal equals the
// division, over random quotients and ones next to representable values.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#define __host__
#define __device__
using std::fabs;
using std::floor;
using std::frexp;
using std::ldexp;
#include "poisson_device.hpp"

using namespace imr::pois;

static uint64_t state = 88172645463325252ull;
static uint64_t next()
{
    state ^= state << 13;
    state ^= state >> 7;
    state ^= state << 17;
    return state;
}

int main()
{
    static constexpr Reciprocals r;
    long bad = 0;
    for (long k = 0; k < (1 << 24); ++k) bad += sqrt_count((double) k) != (float) sqrt_d((double) k);
    for (int k = 1; k <= Reciprocals::kCount; ++k) {
        bad += r.hi[k] != 1.0 / k || r.lo[k] != std::fma(-(double) k, r.hi[k], 1.0) / k;
        for (int i = 0; i < 400000; ++i) {
            // exponents 2^-600 ... 2^4
            const uint64_t bits = (uint64_t) (1027 - (int) (next() % 605)) << 52 | next() >> 12;
            double x;
            std::memcpy(&x, &bits, 8);
            if (i % 4 == 0) x = std::nextafter(x * k, i % 8 ? 0.0 : 1e300);
            bad += div_small(x, k, r) != x / k;
        }
    }
    std::printf("%ld wrong\n", bad);
    return bad != 0;
}
