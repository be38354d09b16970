// Compares the estimator's FP64-rounded helpers (crt_math.h) with the host library over every
// sampling angle kTau * j / 2^24 and over x^5 on [0, 1].  Prints the numbers of results whose
// FP32 value differs, and the largest difference in FP32 units in the last place; then how many
// cosines fall on another side of the sun's threshold (sun_cos_in) than their angle does.
#include <cmath>
#include <cstdio>
#include <cstring>

#include "crt_math.h"

static int ulps(float a, float b)
{
    return std::abs(crt::f2ord(a) - crt::f2ord(b));
}

int main()
{
    long differ = 0, differ5 = 0;
    int  worst = 0;
    for (uint32_t j = 0; j < (1u << 24); ++j) {
        const float x = crt::kTau * crt::u01(j << 8);
        float s, c;
        crt::sincos_cr(x, s, c);
        const float rs = (float)std::sin((double)x), rc = (float)std::cos((double)x);
        differ += (s != rs) + (c != rc);
        worst = std::max(worst, std::max(ulps(s, rs), ulps(c, rc)));
        const float u = crt::u01(j << 8), p = (float)std::pow((double)u, 5.0), q = crt::pow5_cr(u);
        differ5 += p != q;
        worst = std::max(worst, ulps(p, q));
    }
    // sizes from none in reach to the whole sphere; the 2000 floats around each threshold, and
    // the ends of the range
    long sides = 0;
    for (float size : {1e-45f, 1e-8f, 3e-4f, 3.4526698e-4f, 1e-3f, 0.0654498f, 0.5f, 1.5707964f, 2.5f, 3.1415925f,
                       3.1415927f, 3.2f, 100.0f}) {
        const float t = crt::sun_cos_in(size);
        auto check = [&](float c) { sides += (c >= t) != (crt::acos_cr(c) < size); };
        const int mid = crt::f2ord(t > 1.0f ? 1.0f : t);
        for (int k = -1000; k <= 1000; ++k) {
            const float c = crt::ord2f(mid + k);
            if (c >= -1.0f && c <= 1.0f) check(c);
        }
        for (float c : {-1.0f, -0.0f, 0.0f, 1.0f}) check(c);
    }
    std::printf("%ld %ld %d %ld\n", differ, differ5, worst, sides);
    return 0;
}
