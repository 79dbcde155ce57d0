// Fixed-point accumulator words of the atomic split reductions. No HIP types: the
// functions are constexpr (host and device in HIP, plain C++ elsewhere), so the same
// header is unit-tested in a host build.
#pragma once

namespace exl3 {

// Accumulator word of the atomic split reductions for up to 2^b - 1 contributors, b = 4..8
// (fix_count_bits): the count in the upper b bits, below it the sum of the contributions, none of
// which is negative, so nothing ever borrows from or carries into the count. A finite partial sum
// is clamped to +-2^18 (fp16 ends at 65504, so a clamped total still rounds to infinity, as the
// unclamped one would), rounded to 45 - 3 b fraction bits and biased by C = 2^(63 - 3b), the clamp
// in these units: it contributes 0..2 C. A partial sum that is not finite contributes
// P = 2^(64 - 2b), more than all finite ones together ((2^b - 1) * 2 C < P), and (2^b - 1) * P
// still fits: the total is recognised and becomes NaN, so a non-finite input gives a non-finite
// output, as in the partial-row reduction.
// The fewer contributors, the more fraction bits: 33 up to 15, 30 up to 31, 27 up to 63, 24 up
// to 127, 21 up to 255. The total is rounded to fp16, whose grid is never finer than 2^-24 (below
// 2^-13): with 30 bits and 31 contributors the roundings of the partial sums have an eleventh of the rms
// error of that rounding, 0.4 % on top of it, and less above 2^-13; with 33 bits and 15, 1/128.
constexpr int fix_count_bits(int contributors) {
    const int b = 32 - __builtin_clz(contributors | 1);
    return b < 4 ? 4 : b;
}
constexpr int kFixMaxContributors = 255;

// Up to so many contributors (30 bits) the words are as good as fp32 partial rows (above).
constexpr int kFixFineContributors = 31;

constexpr float kFixClamp = 262144.f;  // 2^18
constexpr unsigned long long kFixTwo52 = 0x4330000000000000ull;  // bits of 2^52

constexpr unsigned long long fix_bias(int b) { return 1ull << (63 - 3 * b); }
constexpr unsigned long long fix_poison(int b) { return 1ull << (64 - 2 * b); }
constexpr double fix_scale(int exponent) {  // 2^exponent
    return __builtin_bit_cast(double, (unsigned long long)(1023 + exponent) << 52);
}

constexpr unsigned long long fix_word(float v, int b = 8) {
    unsigned long long fixed = fix_poison(b);
    if (v - v == 0.f) {  // finite (NaN and the infinities keep the poison value)
        v = v < -kFixClamp ? -kFixClamp : (v > kFixClamp ? kFixClamp : v);
        // in [2^52, 2^53] doubles are whole numbers: the sum's one rounding is the one to the grid
        const double biased = (double)v * fix_scale(45 - 3 * b) + __builtin_bit_cast(double, kFixTwo52 + fix_bias(b));
        fixed = __builtin_bit_cast(unsigned long long, biased) - kFixTwo52;
    }
    return (1ull << (64 - b)) + fixed;
}
constexpr int fix_count(unsigned long long w, int b = 8) { return (int)(w >> (64 - b)); }
constexpr float fix_value(unsigned long long w, int b = 8) {
    const unsigned long long sum = w & ((1ull << (64 - b)) - 1);
    if (sum >= fix_poison(b)) return __builtin_nanf("");
    const long long fixed = (long long)(sum - (unsigned long long)fix_count(w, b) * fix_bias(b));
    return (float)((double)fixed * fix_scale(3 * b - 45));
}

}  // namespace exl3
