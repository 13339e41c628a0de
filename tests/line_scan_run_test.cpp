// Host test of the run extraction the kernels compile (rqa_bits.hpp):
//  1. consume_word(), with and without single_steps() taken first, over a
//     segment of words reports exactly the runs a direct scan finds, at the LDS
//     row lengths the kernels use: counted runs below the cap, longer ones and
//     the segment's first through the slow path, the last one as the carry;
//  2. the skip of threshold pairs: where a word is all non-recurrent and no run
//     is open at the higher of two thresholds, neither would change anything.
// Prints "ok" and exits 0 on success.
#include <cstdio>
#include <random>
#include <vector>

#include "rqa_bits.hpp"

using namespace rqa;

static int fails = 0;
#define CHECK(c, ...)                                 \
    do {                                              \
        if (!(c)) {                                   \
            if (fails < 20) std::printf(__VA_ARGS__); \
            fails++;                                  \
        }                                             \
    } while (0)

struct Result {
    std::vector<long> hist;   // runs closed on both sides, by length
    long pre, suf;
};

static Result direct(const std::vector<int> &b) {
    const long L = (long)b.size();
    Result r{std::vector<long>(L + 1, 0), 0, 0};
    long first = 0, last = L;
    while (first < L && b[first]) first++;
    if (first == L) {
        r.pre = r.suf = L;
        return r;
    }
    while (b[last - 1]) last--;
    r.pre = first;
    r.suf = L - last;
    for (long k = first, run = 0; k < last; k++) {
        if (!b[k] && run) r.hist[run]++;
        run = b[k] ? run + 1 : 0;
    }
    return r;
}

template <uint32_t CAP, bool DENSE>
static Result scanned(const std::vector<int> &b) {
    const long L = (long)b.size();
    Result r{std::vector<long>(L + 1, 0), -1, -1};
    uint32_t run = PRE;
    auto add = [&](uint32_t len, long n, uint32_t lo, uint32_t hi) {
        CHECK(len >= lo && len < hi && (long)len <= L, "run of %u steps, CAP %u\n", len, CAP);
        if ((long)len <= L) r.hist[len] += n;
    };
    for (long w0 = 0; w0 < L; w0 += 32) {
        const int nb = (int)(L - w0 < 32 ? L - w0 : 32);
        uint32_t nw = 0;
        for (int u = 0; u < nb; u++) nw |= (uint32_t)!b[w0 + u] << u;
        // steps past the end are filled as recurrent and taken back afterwards
        consume_word<CAP>(
            nw, run, [&](uint32_t len) { add(len, 1, 1, CAP); },
            [&](uint32_t &mid) {
                if (!DENSE) return;
                const uint32_t e = single_steps(mid);
                if (e) add(1, __builtin_popcount(e), 1, 2);
                mid ^= e;
            },
            [&](uint32_t len) { add(len, 1, DENSE ? 2 : 1, 31); },
            [&](uint32_t first) {
                if (first >= PRE) {
                    CHECK(r.pre < 0, "prefix written twice\n");
                    r.pre = (long)(first - PRE);
                } else {
                    add(first, 1, CAP, 1u << 29);
                }
            });
        if (nb < 32) run -= (uint32_t)(32 - nb);
    }
    const SegEnds e = seg_ends(run);
    if (e.pre_open) {
        CHECK(r.pre < 0, "open prefix but written\n");
        r.pre = e.pre;
    }
    r.suf = e.suf;
    return r;
}

template <uint32_t CAP>
static void test_runs(std::mt19937_64 &g) {
    for (int it = 0; it < 15000; it++) {
        const long L = 1 + (long)(g() % (it % 10 == 0 ? 2000 : 400));
        std::vector<int> b(L);
        const int mode = it % 7;
        const unsigned p = (unsigned)(g() % 1000);
        for (long k = 0; k < L; k++) {
            if (mode == 0) b[k] = g() % 1000 < p;
            else if (mode == 1) b[k] = 1;
            else if (mode == 2) b[k] = 0;
            else if (mode == 3) b[k] = (k / (1 + it % 37)) % 2;
            else if (mode == 4) b[k] = g() % 300 != 0;                                // runs past every cap
            else if (mode == 5) b[k] = g() % 3 == 0;                                  // mostly single steps
            else b[k] = k % (long)(CAP + 1) != (long)(CAP + 1) / 2 || g() % 9 == 0;   // runs at the cap
        }
        const Result d = direct(b);
        const Result s[2] = {scanned<CAP, false>(b), scanned<CAP, true>(b)};
        for (int f = 0; f < 2; f++) {
            CHECK(d.pre == s[f].pre && d.suf == s[f].suf, "CAP %u form %d L %ld mode %d: ends %ld %ld, %ld %ld\n", CAP, f, L,
                  mode, d.pre, d.suf, s[f].pre, s[f].suf);
            CHECK(d.hist == s[f].hist, "CAP %u form %d L %ld mode %d: histogram\n", CAP, f, L, mode);
        }
    }
}

// Runs at the segment-length limit (2^29 steps, with and without the
// open-prefix flag) close through the slow path; an all-recurrent word adds 32.
static void test_long_carry() {
    for (uint32_t flag : {PRE, 0u})
        for (uint32_t nw : {0x1u, 0x10u, 0x80000000u, 0u}) {
            uint32_t run = flag + (1u << 29) - 3u, got = 0;
            const uint32_t before = run;
            consume_word<LCAP>(
                nw, run, [&](uint32_t len) { CHECK(false, "counted %u\n", len); }, [&](uint32_t &) {},
                [&](uint32_t) { CHECK(false, "inner run in a word with one non-recurrent step\n"); },
                [&](uint32_t f) { got = f; });
            if (nw) CHECK(got == before + (uint32_t)__builtin_ctz(nw), "closing long run: %u\n", got);
            else CHECK(got == 0 && run == before + 32u, "all-recurrent word: %u %u\n", got, run);
        }
}

template <int TG>
static void test_skip(std::mt19937_64 &g) {
    constexpr int B = rank_bits<TG>();
    long skipped = 0;
    for (int it = 0; it < 4000; it++) {
        const int nt = 1 + (int)(g() % TG);
        uint32_t run[TG];
        for (int t = 0; t < TG; t++) run[t] = it % 3 == 0 ? PRE : 0u;   // what a kernel starts with; a closed prefix
        for (int w = 0; w < 6; w++) {
            uint32_t R[8] = {}, P[B];
            const int lo = (int)(g() % (nt + 1));   // no step below this rank
            for (int u = 0; u < 32; u++) R[u & 7] |= (uint32_t)(lo + g() % (nt + 1 - lo)) << (8 * (u >> 3));
            rank_planes<B>(R, P, 0xFFFFFFFFu, 0u);
            const GeTree<B> G(P);
            for (int t0 = 0; t0 < nt; t0 += 2) {
                const bool skip = (~G.ge(t0 + 2) | run[t0 + 1]) == 0u;
                for (int t = t0; t < t0 + 2 && t < nt; t++) {
                    uint32_t r = run[t];
                    int calls = 0;
                    consume_word<LCAP>(
                        G.ge(t + 1), r, [&](uint32_t) { calls++; }, [&](uint32_t &mid) { calls += mid != 0; },
                        [&](uint32_t) { calls++; }, [&](uint32_t) { calls++; });
                    if (skip) {
                        CHECK(calls == 0 && r == run[t], "TG %d t %d: a skipped threshold counts\n", TG, t);
                        skipped++;
                    } else {
                        run[t] = r;
                    }
                }
            }
        }
    }
    CHECK(skipped > 500, "TG %d: %ld skips\n", TG, skipped);
}

int main() {
    std::mt19937_64 g(99);
    test_long_carry();
    test_runs<64>(g);
    test_runs<LCAP>(g);
    test_runs<140>(g);
    test_runs<192>(g);
    test_runs<256>(g);
    test_skip<4>(g);
    test_skip<8>(g);
    test_skip<16>(g);
    test_skip<24>(g);
    test_skip<32>(g);
    std::puts(fails ? "failed" : "ok");
    return fails ? 1 : 0;
}
