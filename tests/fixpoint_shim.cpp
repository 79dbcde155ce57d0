// Host build of the accumulator-word helpers for tests/test_host_fixpoint.py.
#include <stddef.h>

#include "../ponyexl3_amd/csrc/exl3_fixpoint.hpp"

extern "C" {
unsigned long long shim_fix_word(float v) { return exl3::fix_word(v); }
int shim_fix_count(unsigned long long w) { return exl3::fix_count(w); }
float shim_fix_value(unsigned long long w) { return exl3::fix_value(w); }

int shim_fix_count_bits(int contributors) { return exl3::fix_count_bits(contributors); }
// totals of n accumulators that `contributors` partial sums each went into, [contributor][n]
void shim_fix_reduce(const float* partial, int contributors, int n, float* total, int* count) {
    const int bits = exl3::fix_count_bits(contributors);
    for (int i = 0; i < n; i++) {
        unsigned long long w = 0;
        for (int c = 0; c < contributors; c++) w += exl3::fix_word(partial[(size_t)c * n + i], bits);
        total[i] = exl3::fix_value(w, bits);
        count[i] = exl3::fix_count(w, bits);
    }
}
unsigned long long shim_fix_word_bits(float v, int bits) { return exl3::fix_word(v, bits); }
int shim_fix_count_of(unsigned long long w, int bits) { return exl3::fix_count(w, bits); }
}
