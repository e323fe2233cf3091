// gh_pairf64.h's pair factor against the host's division and square root, with starting
// values as far off as v_rsq_f64's: random operands over the whole range, its ends, and
// every operand whose square root is within 2^-40 of a power of two or of sqrt(2) times one.
#include <cstdio>
#include <cstring>
#include <random>

#include "../../gravhopper_amd/csrc/gh_pairf64.h"

static uint64_t bits(double d)
{
    uint64_t b;
    memcpy(&b, &d, 8);
    return b;
}

static double value(uint64_t b)
{
    double d;
    memcpy(&d, &b, 8);
    return d;
}

static bool in_range(double d)
{
    const uint64_t b = bits(d);
    return (uint32_t)(b >> 32) - gh::kPairLoHi < gh::kPairSpan &&
           (uint32_t)b != gh::kPairLowOnes;
}

static long wrong = 0, tested = 0;

static void check(double d, double off)
{
    if (!in_range(d)) return;
    const double root = sqrt(d), inv = 1.0 / d;
    const double want = inv / root, got = gh::pair_factor(d, (1.0 / root) * (1.0 + off));
    tested++;
    if (bits(want) != bits(got) && wrong++ < 5) printf("d=%a off=%a: %a, not %a\n", d, off, got, want);
}

int main()
{
    const double most = 5e-8;  // above v_rsq_f64's 2^-24.6
    std::mt19937_64 rng(1);
    std::uniform_real_distribution<double> off(-most, most);
    for (long k = 0; k < 20000000; k++) {
        // all exponents of the range, and densely the four that all others scale from
        const uint64_t e = k & 1 ? 523 + rng() % 1001 : 1022 + rng() % 4;
        check(value(e << 52 | rng() >> 12), off(rng));
    }
    const double steps[] = {-most, -most / 7, 0.0, most / 7, most};
    for (int parity = 0; parity < 2; parity++)
        for (long k = -4096; k <= 4096; k++)
            for (int near = -4; near <= 4; near++) {
                const double s = value(bits(parity ? sqrt(2.0) : 2.0) + k);
                for (double o : steps) check(value(bits(s * s) + near), o);
            }
    for (uint64_t e : {523ull, 524ull, 1523ull})
        for (uint64_t m : {0ull, 1ull, 0xffffffffffffeull, 0xfffffffffffffull})
            for (double o : steps) check(value(e << 52 | m), o);
    // what the range leaves to the plain expressions
    const double none[] = {0.0, -1.0, 5e-324, 1e-160, 1e160, INFINITY, -INFINITY, NAN};
    for (double d : none)
        if (in_range(d)) wrong++;
    if (in_range(value(0x3fefffffffffffffull))) wrong++;
    printf("%ld tested, %ld wrong\n", tested, wrong);
    return wrong != 0;
}
