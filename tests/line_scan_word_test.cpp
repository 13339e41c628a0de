// Host test of consume_word() (rqa_bits.hpp): with and without single_steps()
// taken first, it reports the runs of consume() word by word -- the same
// histogram, slow runs and carry -- on random and structured words.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <random>
#include <vector>

#include "rqa_bits.hpp"

using namespace rqa;

struct Out {
    std::map<uint32_t, long> hist;
    std::vector<uint32_t> slow;
    uint32_t run;
    bool operator==(const Out &o) const { return hist == o.hist && slow == o.slow && run == o.run; }
};

template <uint32_t CAP>
static Out by_consume(uint32_t nw, uint32_t run) {
    Out o;
    consume<CAP>(nw, run, CAP + 3, [&](uint32_t b) { if (b <= CAP - 2) o.hist[b + 1]++; },
                 [&](uint32_t len) { o.hist[len]++; }, [&](uint32_t f) { o.slow.push_back(f); });
    o.run = run;
    return o;
}

template <uint32_t CAP, bool DENSE>
static Out by_word(uint32_t nw, uint32_t run) {
    Out o;
    consume_word<CAP>(nw, run, [&](uint32_t len) { o.hist[len]++; },
                      [&](uint32_t &mid) {
                          if (!DENSE) return;
                          const uint32_t e = single_steps(mid);
                          if (e) o.hist[1] += __builtin_popcount(e);
                          mid ^= e;
                      },
                      [&](uint32_t len) { o.hist[len]++; }, [&](uint32_t f) { o.slow.push_back(f); });
    o.run = run;
    return o;
}

template <uint32_t CAP>
static int check(uint32_t nw, uint32_t run) {
    const Out a = by_consume<CAP>(nw, run);
    if (a == by_word<CAP, false>(nw, run) && a == by_word<CAP, true>(nw, run)) return 0;
    std::printf("differs: CAP %u nw %08x run %08x\n", CAP, nw, run);
    return 1;
}

int main() {
    std::mt19937_64 g(5);
    const uint32_t runs[] = {0u, 1u, 31u, 32u, 63u, 95u, 96u, 127u, 128u, 191u, 255u, 256u, 2047u, 1u << 29, PRE, PRE + 1,
                             PRE + 200, PRE + (1u << 29)};
    int bad = 0;
    for (int k = 0; k < 200000; k++) {
        uint32_t nw = (uint32_t)g();
        if (k % 5 == 1) nw &= (uint32_t)g() & (uint32_t)g();
        if (k % 5 == 2) nw |= (uint32_t)g() | (uint32_t)g();
        if (k % 5 == 3) nw = k & 8 ? 0xAAAAAAAAu >> (k & 1) : ~0u << (k % 32);
        if (k % 5 == 4) nw = k % 3 == 0 ? 0u : k % 3 == 1 ? ~0u : 1u << (g() % 32);
        const uint32_t run = runs[g() % (sizeof runs / sizeof runs[0])];
        bad += check<64>(nw, run) + check<128>(nw, run) + check<140>(nw, run) + check<256>(nw, run);
        if (bad > 5) break;
    }
    std::puts(bad ? "failed" : "ok");
    return bad ? 1 : 0;
}
