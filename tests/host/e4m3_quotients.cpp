// The corrected product that stands in for the division of the e4m3 quantizer's 16-bit inputs, against IEEE division: every pair of a
// maximum and an element of the type, element exponents down to where every code is zero, with the reciprocal as division rounds it
// and one unit in the last place to either side (what the hardware's reciprocal is good to). Built and run by tests/test_e4m3_quotients.py.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <initializer_list>

static uint32_t bits(float f) {
    uint32_t u;
    std::memcpy(&u, &f, 4);
    return u;
}

// Code of |q| <= 448 (1 + 2^-22), ties to even: the quantum is 2^-9 below 2^-6, 2^(e-3) for 2^e <= q.
static float e4m3_value(float q) {
    int e = int(bits(q) >> 23) - 127;
    const float quantum = std::ldexp(1.0f, (e < -6 ? -6 : e) - 3);
    return std::nearbyintf(q / quantum) * quantum;  // both exact
}

int main() {
    long long n = 0, rounded_apart = 0;
    for (int frac : {7, 10})  // bfloat16, float16
        for (int m = 1 << frac; m < 2 << frac; ++m) {
            const float amax = float(m), s = amax / 448.0f, rn = 1.0f / s;
            const float invs[3] = {std::nextafterf(rn, 0.0f), rn, std::nextafterf(rn, 2.0f * rn)};
            for (int shift = 0; shift <= 20; ++shift)  // 448 * 2^-20 is below half of the smallest code
                for (int k = 1 << frac; k < 2 << frac; ++k) {
                    const float x = std::ldexp(float(k), -shift);
                    if (x > amax) break;
                    const float want = x / s;
                    for (float inv : invs) {
                        float q = x * inv;
                        q = std::fmaf(-std::fmaf(q, s, -x), inv, q);
                        rounded_apart += q != want;
                        ++n;
                        if (e4m3_value(q) != e4m3_value(want)) return std::printf("max %d of %d bits, x %d >> %d: %a, %a\n", m, frac, k, shift, q, want), 1;
                    }
                }
        }
    std::printf("ok %lld quotients, %lld of them rounded to another float32\n", n, rounded_apart);
    return 0;
}
