// Host-side check of incrmt_amd/csrc/quot.hh against the division: quot gives its
// bits for the operands that quot_divisor and quot_numerator accept, and for
// other finite numerators of an accepted divisor a neighbour of its finite
// quotients at the most; over all bit patterns, every pair of exponents around
// the limits and the underflow of remainder and quotient with mantissas at
// their ends and random ones, and zeros and extremes.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <limits>
#include <random>
#include <vector>
#include "../incrmt_amd/csrc/quot.hh"
using namespace incrmt;

template <class T, class U>
struct Check {
    static constexpr int kMant = sizeof(T) == 8 ? 52 : 23, kBias = sizeof(T) == 8 ? 1023 : 127;
    std::mt19937_64 rng{11};
    long bad = 0, off = 0, used = 0;
    T make(U bits) { T v; memcpy(&v, &bits, sizeof v); return v; }
    T at(int e, int kind) {  // exponent e; mantissa: zeros, ones, one bit, random
        const U m = kind == 0 ? 0 : kind == 1 ? ~U(0) : kind == 2 ? 1 : U(rng());
        const U sign = U(rng() & 1) << (8 * sizeof(T) - 1);
        return make(sign | U(e + kBias) << kMant | (m & ((U(1) << kMant) - 1)));
    }
    template <bool POS>
    void form(T n, T d, T want, T y) {
        if (!quot_divisor<POS>(d)) return;
        const T q = quot<POS, T>(n, d, y), inf = std::numeric_limits<T>::infinity();
        if (quot_numerator(n)) {
            bad += memcmp(&want, &q, sizeof(T)) != 0;
            used++;
        } else if (std::isfinite(n) && std::isfinite(want)) {
            off += !(q >= std::nextafter(want, -inf) && q <= std::nextafter(want, inf));
        }
    }
    void one(T n, T d) {
        volatile T vn = n, vd = d;  // a division at run time
        const T want = vn / vd, y = T(1) / vd;
        form<true>(n, d, want, y);
        form<false>(n, d, want, y);
    }
    void run(long trials, const std::vector<int> &en, const std::vector<int> &ed) {
        for (long t = 0; t < trials; t++) one(make(U(rng())), make(U(rng())));
        for (long t = 0; t < trials; t++) one(at(int(rng() % 40) - 30, 3), at(int(rng() % 30) - 10, 3));
        for (int a : en)
            for (int b : ed)
                for (int k = 0; k < 16; k++)
                    for (int r = 0; r < 8; r++) one(at(a, k & 3), at(b, k >> 2));
        const T inf = std::numeric_limits<T>::infinity(), nan = std::numeric_limits<T>::quiet_NaN();
        const T odd[] = {T(0), -T(0), inf, -inf, nan, T(1), T(-3), std::numeric_limits<T>::denorm_min(),
                         std::numeric_limits<T>::min(), std::numeric_limits<T>::max()};
        for (T n : odd)
            for (T d : odd) one(n, d);
    }
};

int main(int argc, char **argv) {
    const long trials = argc > 1 ? atol(argv[1]) : 1000000;
    Check<float, uint32_t> f;
    f.run(trials, {-126, -125, -112, -110, -105, -102, -82, -81, -80, -79, -1, 0, 78, 79, 80, 81, 126, 127},
          {-126, -100, -42, -41, -40, -39, -2, 0, 2, 12, 38, 39, 40, 41, 100, 127});
    Check<double, uint64_t> d;
    d.run(trials, {-1022, -1000, -969, -402, -401, -400, -399, -1, 0, 398, 399, 400, 401, 1000, 1023},
          {-1022, -800, -402, -401, -400, -399, -2, 0, 2, 12, 398, 399, 400, 401, 800, 1023});
    printf("%ld %ld %ld %ld\n", f.bad, f.off, d.bad, d.off);
    return f.bad || f.off || d.bad || d.off || f.used < trials || d.used < trials;
}
