/*
 * Host check of the count-form draw table (gf_const_drift.hpp): for models
 * over the range of chromosome numbers, selection and dominance, every row's
 * lookup equals binom_draw of the row's mean, at random words and at each
 * threshold and its successor (where the number of partial sums passed
 * changes), and the rows in use are the leading counts whose mean is in
 * [0, 6].  Host code only.
 */
#include <cstdio>
#include <random>
#include "../../parallelpopgen_amd/csrc/gf_const_drift.hpp"

using namespace gf;

int main() {
    std::mt19937 rng(7);
    long long checked = 0, rows = 0;
    const int Ncs[] = {100, 101, 127, 500, 1999, 2000, 20000, 199999, 200000, 400000, (1 << 21) - 1, 1 << 21};
    const float ss[] = {0.0f, -5e-5f, 5e-5f, -0.002f, 0.01f, -0.1f, 0.3f, -0.5f, -1.0f};
    const float hs[] = {0.0f, 0.3f, 0.5f, 1.0f};
    for (int Nc : Ncs)
        for (float s : ss)
            for (float h : hs)
                for (float slope : {0.0f, 0.001f}) {
                    const float F = 0.1f;
                    const ConstModel C{Nc, (float)Nc, 1.0f / (float)Nc, slope, s, (F + h) - (h * F), (F + (2.0f * h)) - ((2.0f * h) * F),
                                       s == 0.0f && slope == 0.0f, mid_selection(slope, s, F, h)};
                    PoisTable table;
                    for (int id = 0; id < POIS_BUILD; id++) pois_table_entry(id, C, &table);
                    const uint4 *tab = table.v;
                    for (int row = 0; row < POIS_ROWS; row++) {
                        const float xs = const_selected((float)(row + 1) / (float)Nc, C);
                        const float mean = xs * C.N, var = (1.0f - xs) * mean;
                        if (row + 1 < table.jn && !(mean >= 0.0f && mean <= 6.0f)) { std::printf("row use\n"); return 1; }
                        if (row + 1 == table.jn && mean >= 0.0f && mean <= 6.0f) { std::printf("row unused\n"); return 1; }
                        if (row + 1 >= table.jn) continue;
                        rows++;
                        uint32_t words[2 * POIS_TERMS + 200];
                        int n = 0;
                        const uint32_t *T = (const uint32_t *)(tab + row * POIS_ROW_VECS);
                        for (int k = 0; k < POIS_TERMS; k++) { words[n++] = T[pois_word(k)]; words[n++] = T[pois_word(k)] + 1u; }
                        for (int k = 0; k < 100; k++) words[n++] = (uint32_t)rng();
                        for (int k = 0; k < 100; k++) words[n++] = 0xffffffffu - ((uint32_t)rng() >> (rng() % 31));
                        for (int k = 0; k < n; k++) {
                            int want = binom_draw(words[k], mean, var, C.N);
                            want = want < 0 ? 0 : (want > Nc ? Nc : want);
                            const int got = pois_lookup(tab, row, words[k]);
                            checked++;
                            if (got != want) {
                                std::printf("Nc %d s %g h %g count %d word %08x: %d, binom_draw %d\n", Nc, s, h, row + 1, words[k], got, want);
                                return 1;
                            }
                        }
                    }
                }
    for (int Nc : Ncs)   /* x = RN(j/N) gives j back */
        for (int k = 0; k < 200000; k++) {
            const int j = k < 1000 ? k % (Nc + 1) : (k < 2000 ? Nc - k % 100 : (int)(rng() % (unsigned)(Nc + 1)));
            if ((int)__builtin_rintf(((float)j / (float)Nc) * (float)Nc) != j) { std::printf("count %d of %d\n", j, Nc); return 1; }
        }
    std::printf("%lld rows, %lld draws: every lookup equals binom_draw\n", rows, checked);
    return 0;
}
