// The split of f32 factors into three bf16 terms (saragossa_amd/csrc/f32_terms.h): the terms add up to the
// value, each is a bf16, and the products that are kept miss at most 2^-24 (and 2^-33 for the last one left
// out) of the product. Factors: normal ones, and every second half of a bf16 cell where a term can be largest.
#include <cmath>
#include <cstdio>
#include <random>

#include "f32_terms.h"

using namespace skv;

static float term(uint32_t pair, bool second) { return word_f32(second ? pair & 0xffff0000u : pair << 16); }

int main() {
    std::mt19937 rng(1);
    std::normal_distribution<float> normal;
    double worst[3] = {0, 0, 0}, squares[3] = {0, 0, 0};
    const int n = 2000000;
    const uint32_t from[3] = {0, 0xff00u, 0x7e00u}, range[3] = {0, 0x100u, 0x400u};
    for (int kind = 0; kind < 3; ++kind) {
        for (int i = 0; i < n; ++i) {
            float x[2];
            for (float &v : x) {
                if (kind == 0) v = normal(rng) * std::exp2((float)((int)(rng() % 81) - 40));
                else v = word_f32((rng() & 0x80000000u) | 127u << 23 | (rng() % 128u) << 16 | (from[kind] + rng() % range[kind]));
                if (v == 0.0f) v = 1.0f;
            }
            uint32_t t[3];
            three_terms(x[0], x[1], t[0], t[1], t[2]);
            double sum[2] = {0, 0}, kept = 0;
            for (int k = 0; k < 3; ++k)
                for (int s = 0; s < 2; ++s) sum[s] += term(t[k], s);
            if (sum[0] != x[0] || sum[1] != x[1]) {
                std::printf("terms of %a, %a do not add up\n", x[0], x[1]);
                return 1;
            }
            for (const TermPair &p : TERMS) kept += (double)term(t[p.l], false) * term(t[p.r], true);
            const double product = (double)x[0] * x[1], off = std::fabs((kept - product) / product);
            worst[kind] = std::fmax(worst[kind], off);
            squares[kind] += off * off;
        }
        std::printf("kind %d: worst 2^%.2f, rms 2^%.2f\n", kind, std::log2(worst[kind] + 1e-99), std::log2(std::sqrt(squares[kind] / n) + 1e-99));
        if (worst[kind] > std::exp2(-24.0) + std::exp2(-33.0)) return 1;
    }
    // what is not a number, or rounds to none, must not pass for one
    const float odd[4] = {INFINITY, -INFINITY, NAN, 3.4e38f};
    for (float v : odd) {
        uint32_t t[3];
        three_terms(v, v, t[0], t[1], t[2]);
        if (std::isfinite(term(t[0], false)) || std::isfinite(term(t[1], true))) return 1;
    }
    std::printf("ok\n");
    return 0;
}
