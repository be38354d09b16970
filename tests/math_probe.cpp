// Compares the estimator's FP64-rounded helpers (crt_math.h) with the host library over every
// sampling angle kTau * j / 2^24 and over x^5 on [0, 1].  Prints the numbers of results whose
// FP32 value differs, and the largest difference in FP32 units in the last place.
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
    std::printf("%ld %ld %d\n", differ, differ5, worst);
    return 0;
}
