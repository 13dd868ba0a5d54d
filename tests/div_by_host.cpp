// rdr::div_by (csrc/render_dev.h) against the division, for the gaussian's two
// constants: every significand, at exponents across the range they meet.
#include <cmath>
#include <cstdio>
#include <cstring>

#include "../blacktracer_amd/csrc/render_dev.h"

int main() {
    constexpr float sigma = 1.f / 2.5f;
    const float den[] = {sigma * sigma, sigma * BT_SQRT2PI};
    long long bad = 0;
    for (float d : den)
        for (int e : {-60, -7, -1, 0, 1, 5})
            for (unsigned s = 0; s < 1u << 23; s++) {
                const unsigned w = (unsigned)(127 + e) << 23 | s;
                float x;
                std::memcpy(&x, &w, 4);
                if (bt::rdr::div_by(x, d, 1.f / d) != x / d || bt::rdr::div_by(-x, d, 1.f / d) != -x / d) bad++;
            }
    std::printf("%lld quotients differ\n", bad);
    return bad != 0;
}
