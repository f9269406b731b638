// Compares csrc/exact_f32.hpp with (float)exp((double)x) and x / d on the host.
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>
#define __device__ static
#define __forceinline__ inline
#include "../../aarambh-ai_amd/csrc/exact_f32.hpp"

static float from_bits(uint32_t u) {
    float f;
    memcpy(&f, &u, 4);
    return f;
}
static bool same(float a, float b) { return memcmp(&a, &b, 4) == 0 || (a != a && b != b); }

static uint64_t state = 88172645463325252ull;
static uint32_t rnd() {
    state ^= state << 13;
    state ^= state >> 7;
    state ^= state << 17;
    return (uint32_t)(state >> 32);
}

struct Tally {
    long n = 0, wrong = 0, bad = 0;
};

static void exp_range(Tally& t, uint32_t first, uint32_t last, uint32_t step) {
    for (uint64_t u = first; u <= last; u += step) {
        const float x = from_bits((uint32_t)u);
        bool bad = false;
        const float y = expf_fast(x, bad);
        t.n++;
        t.bad += bad;
        t.wrong += !bad && !same(y, (float)exp((double)x));
    }
}

static void div_one(Tally& t, float x, float d) {
    t.n++;
    t.wrong += !same(div_fast(x, 1.0 / (double)d), x / d);
}

static uint32_t bits(float f) {
    uint32_t u;
    memcpy(&u, &f, 4);
    return u;
}

int main() {
    Tally neg, pos, sub, any, low, tie, special;
    exp_range(neg, bits(-0.0f), bits(-INFINITY), 131);  // every magnitude
    exp_range(sub, bits(-86.0f), bits(-104.5f), 7);     // subnormal results and around them
    exp_range(pos, 0, bits(88.0f), 257);
    for (long i = 0; i < 4000000; i++) {
        // any values; a probability, an exponential over a sum of at least 1, down to the smallest
        div_one(any, from_bits(rnd()), from_bits(rnd()));
        div_one(low, from_bits(rnd() % bits(1e-25f)), from_bits(bits(1.0f) + rnd() % 0x09000000u));
        // ties: odd multiples of half the smallest f32, as quotients by a divisor of few bits ...
        const uint32_t d = 1u + rnd() % 4095u, m = (rnd() % 2048u) | 1u;
        div_one(tie, ldexpf((float)(m * d), -140), ldexpf((float)d, 10));
        // ... and the quotients next to them
        div_one(tie, from_bits(bits(ldexpf((float)(m * d), -120)) + 1u - 2u * (rnd() & 1u)), ldexpf((float)d, 30));
    }
    const float v[] = {0.0f, -0.0f, 1.0f, -1.0f, INFINITY, -INFINITY, NAN, 1e-45f, 1.1754942e-38f, 1.17549435e-38f, 3.4028235e38f};
    for (float x : v)
        for (float d : v) div_one(special, x, d);
    bool inf_bad = false, nan_bad = false;
    expf_fast(INFINITY, inf_bad);
    special.n++;
    special.wrong += !inf_bad || expf_fast(NAN, nan_bad) != 0.0f || nan_bad;
    const Tally* all[] = {&neg, &sub, &pos, &any, &low, &tie, &special};
    const char* names[] = {"exp_negative", "exp_subnormal", "exp_positive", "div_any", "div_low", "div_tie", "div_special"};
    for (int i = 0; i < 7; i++) printf("%s %ld %ld %ld\n", names[i], all[i]->n, all[i]->wrong, all[i]->bad);
    return 0;
}
