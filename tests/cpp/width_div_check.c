/* CPU check of the raycast's texture coordinate (kinectfusion-cuda_amd/csrc/raycast.hip,
 * tex): x / width + 1/2 with the quotient from y = RN(1/width),
 *     q = x*y,  r = fma(-q, width, x),  fma(r, y, q)
 * must equal the correctly rounded quotient plus 1/2 for every float x of the
 * cube's half width (a seeded sample of each binade; magnitudes below 2^-30
 * included), for widths with short and long significands, the all-ones one among
 * them.  Prints the number of mismatches and exits non-zero if any. */
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

static inline uint32_t bits(float f) { uint32_t u; memcpy(&u, &f, 4); return u; }
static inline float fl(uint32_t u) { float f; memcpy(&f, &u, 4); return f; }
static uint64_t state = 0x9E3779B97F4A7C15ull;
static inline uint64_t next(void)
{
    uint64_t z = (state += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

int main(void)
{
    const float widths[] = {2.5f, 3.0f, 4.0f, 5.0f, 0.1f, 7.7f, 1e-3f, 9999.9f, fl(0x40000000u - 1u),
                            fl(0x40800000u - 1u), fl(0x40400001u), 1.0f / 3.0f};
    long bad = 0, total = 0;
    for (unsigned m = 0; m < sizeof(widths) / sizeof(widths[0]); ++m) {
        const float b = widths[m], y = 1.0f / b;
        for (int e = 1; e <= (int)(bits(b) >> 23); ++e) /* every binade up to the width's */
            for (int t = 0; t < 20000; ++t) {
                const uint64_t v = next();
                float x = fl(((uint32_t)e << 23) | (uint32_t)(v & 0x7fffff));
                if (v >> 63) x = -x;
                const float q = x * y, r = fmaf(-q, b, x), d = fmaf(r, y, q);
                ++total;
                bad += bits(d + 0.5f) != bits(x / b + 0.5f);
            }
        bad += bits(fmaf(fmaf(-0.0f, b, 0.0f), y, 0.0f) + 0.5f) != bits(0.5f);
    }
    printf("%ld of %ld coordinates differ\n", bad, total);
    return bad != 0;
}
