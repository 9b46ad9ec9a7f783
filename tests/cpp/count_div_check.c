/* CPU check of the count update's quotient (kinectfusion-cuda_amd/csrc/tsdf.hip,
 * update_voxel) for the divisors above 129, which an uploaded volume's counts of up
 * to 255 reach: with y = RN(1/b), q = RN(x*y), r = fma(-q, b, x), fma(r, y, q) must
 * equal RN(x/b).  Numerators: a seeded sample of the floats of [2^-30, 512] in both
 * signs (F * W + f with |F| <= 2, W <= 255, |f| <= 1).  Prints the number of
 * mismatches and exits non-zero if any. */
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
    long bad = 0, total = 0;
    for (int k = 130; k <= 256; ++k) {
        const float b = (float)k, y = 1.0f / b;
        for (int t = 0; t < 1000000; ++t) {
            const uint64_t v = next();
            float x = fl(bits(0x1p-30f) + (uint32_t)(v % (bits(512.0f) - bits(0x1p-30f) + 1)));
            if (v >> 63) x = -x;
            const float q = x * y, r = fmaf(-q, b, x);
            ++total;
            bad += bits(x / b) != bits(fmaf(r, y, q));
        }
    }
    printf("%ld of %ld quotients differ\n", bad, total);
    return bad != 0;
}
