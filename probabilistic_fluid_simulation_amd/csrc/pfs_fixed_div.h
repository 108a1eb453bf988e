// Division by a divisor fixed per launch in two operations, and the host's
// proof that they round correctly.  Plain C++: no HIP here.
#pragma once

#include <cmath>
#include <cstdint>

namespace pfs {

// d split as hi = 1/d rounded down (strictly below) and lo = RN(1/d - hi) > 0.
// RN(x*hi + RN(x*lo)), one product and one FMA, is x/d rounded once whenever
// `ok`; lo > 0 keeps zeros' signs, infinities and NaN as IEEE division gives
// them.
struct FixedDiv {
    float hi, lo;
    int ok;
};

// The two-operation division's constants for a divisor 1 <= d <= 2^17, `ok`
// when every quotient x/d of normal floats without under- or overflow comes
// out correctly rounded.  With d = D * 2^e (D a 24-bit integer) and x's
// significand X, x/d lies |r| / (X * 2^k) (relative) from the nearest midpoint
// of two floats, r = X * 2^k - M * D != 0 an integer, M odd, k = 24 for X >= D
// and 25 below; the two operations err by less than 2^-46, so only |r| <= 8
// can round wrongly.  The few X with |r| <= 16 are found by solving
// X * 2^k = r (mod D) and tried (the method of Brisebarre and Muller,
// "Correctly rounded multiplication by arbitrary precision constants", 2008).
inline FixedDiv prove_fixed_div(float d) {
    FixedDiv f{0.0f, 0.0f, 0};
    if (!(d >= 1.0f && d <= 131072.0f)) return f;
    const double inv = 1.0 / (double)d;
    f.hi = (float)inv;
    if ((double)f.hi >= inv) f.hi = std::nextafterf(f.hi, 0.0f);
    f.lo = (float)(inv - (double)f.hi);
    int e = 0;
    const uint32_t D = (uint32_t)std::ldexp(std::frexp((double)d, &e), 24);
    int s = 0;
    while (!((D >> s) & 1u)) ++s;
    const uint32_t Dp = D >> s;  // odd
    for (int k = 24; k <= 25; ++k)
        for (int r = -16; r <= 16; ++r) {
            // Only multiples of 2^s occur; the zero r never does (M odd, k > s).
            if (r == 0 || s > 4 || (r & ((1 << s) - 1)) != 0) continue;
            long long m = (r / (1 << s)) % (long long)Dp;
            if (m < 0) m += Dp;
            uint64_t X = (uint64_t)m;  // m / 2^(k-s) mod Dp, halved k - s times
            for (int t = 0; t < k - s; ++t) X = (X & 1) ? (X + Dp) >> 1 : X >> 1;
            for (; X < (1u << 24); X += Dp) {
                if (X < (1u << 23) || (k == 24 ? X < D : X >= D)) continue;
                const float x = (float)X, t = x * f.lo;
                if (std::fmaf(x, f.hi, t) != x / d) return f;
            }
        }
    f.ok = 1;
    return f;
}

// The constants for a field's side n up to 2^24 (every such side is a float),
// from those that `fixed` (prove_fixed_div) gives up to 2^17: a larger side's are
// its 128th's, scaled exactly.  Every side up to 4,159,486 is proven.
template <typename Fixed>
inline FixedDiv side_div(float n, Fixed &&fixed) {
    if (n <= 131072.0f) return fixed(n);
    if (!(n <= 16777216.0f)) return FixedDiv{0.0f, 0.0f, 0};
    FixedDiv f = fixed(n * 0x1p-7f);
    f.hi *= 0x1p-7f;
    f.lo *= 0x1p-7f;
    return f;
}

}  // namespace pfs
