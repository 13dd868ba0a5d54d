// Forms of csrc/render_dev.h that leave a division out, against the division:
// div_by for the gaussian's two constants (every significand, at exponents
// across the range they meet), wrap_col for small and extreme indices.
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
    long long cols = 0;
    for (int GM = 1; GM <= 260; GM++)
        for (int x = -7 * GM - 3; x <= 7 * GM + 3; x++) cols += bt::rdr::wrap_col(x, GM) != x % GM;
    for (int GM : {1, 2, 3, 4096, 65535, 0x7fffffff})
        for (int x : {-0x7fffffff, -65536, -4096, 0, 4096, 0x7ffffffe, 0x7fffffff}) cols += bt::rdr::wrap_col(x, GM) != x % GM;
    std::printf("%lld columns differ\n", cols);
    return bad != 0 || cols != 0;
}
