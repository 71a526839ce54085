// The sum of `count` equal terms added one after another in f64.
#pragma once
#include <cmath>
#include <cstdint>

namespace hbr {

// What `double s = 0.0; for (count times) s += c;` gives, bit for bit, for a
// positive normal c, without the chain of additions (10.5M of them take
// ~10 ms). While s stays in one binade its spacing u does not change, and
// every addition moves it by the same multiple of u (c rounded to u; s is a
// multiple itself) unless c lies halfway between two multiples, where the
// rounding depends on s; so all additions of a binade but the last few are
// one exact product.
inline double repeat_add(double c, uint64_t count) {
    double s = 0.0;
    while (count > 0) {
        const double next = s + c;
        count--;
        if (s > 0.0 && count > 0) {
            int e = 0;
            (void)std::frexp(next, &e);                    // next in [2^(e-1), 2^e)
            const double u = std::ldexp(1.0, e - 53), top = std::ldexp(1.0, e);
            const double inc = (next + c) - next;          // exact while the sum stays below top
            const double room = top - next;                // exact: multiples of u
            if (inc > 0.0 && next + c < top && std::fmod(c, u) * 2.0 != u) {
                // the sums stay below top, with one step's room for the rounding
                const double steps = std::floor(room / inc) - 2.0;
                if (steps >= 1.0) {
                    const uint64_t t = steps < (double)count ? (uint64_t)steps : count;
                    s = next + (double)t * inc;            // multiples of u below 2^53 u: exact
                    count -= t;
                    continue;
                }
            }
        }
        s = next;
    }
    return s;
}

}  // namespace hbr
