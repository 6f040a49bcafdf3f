// CPU test of the balanced split's arithmetic (voltattn_amd/csrc/va_runs.hpp): built with
// g++ and run by tests/test_runs.py.
//
//   test_runs                          checks random batches, prints "runs: ok"
//   test_runs MIN NWG G TILES...       prints "runs N pieces P partials Q" of one batch: its
//                                      runs, the most pieces of any merge group and the
//                                      pieces of all merge groups that are cut
#include "va_runs.hpp"

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#define CHECK(c)                                                          \
    do {                                                                  \
        if (!(c)) {                                                       \
            std::fprintf(stderr, "%s:%d: check failed: %s\n", __FILE__, __LINE__, #c); \
            std::exit(1);                                                 \
        }                                                                 \
    } while (0)

struct Item { int w, b, g, t0, cnt, first, pieces; };

// Every item of every run, as the work-groups walk them; `later` (if given) are the
// tiles found for the sequences after a run's first one.
template <class R>
static std::vector<Item> walk(R& r, const std::vector<int>& tiles, int G, int nwg, const std::vector<int>* later = nullptr) {
    const int B = (int)tiles.size();
    int sum = 0, most = 0, least = 1 << 30;
    for (int t : tiles) { sum += t; most = std::max(most, t); least = std::min(least, t); }
    r.plan(sum, most, least, B, G, nwg);
    std::vector<Item> items;
    for (int w = 0; w < nwg; ++w) {
        if (!r.take(w)) continue;
        int b = 0, base = 0;
        while ((base + tiles[b] + r.cost) * G <= r.at) base += tiles[b++] + r.cost;
        r.enter(b, base, tiles[b] + r.cost);
        while (r.next()) {
            CHECK(r.b >= 0 && r.b < B && r.g >= 0 && r.g < G);
            r.locate();
            items.push_back({w, r.b, r.g, r.t0, r.cnt, r.first, r.pieces});
            CHECK(items.size() < 100000000u);
            if (r.pass()) r.ub = (later ? *later : tiles)[std::min(r.b, B - 1)] + r.cost;
        }
    }
    return items;
}

template <class R>
static int check_batch(const std::vector<int>& tiles, int G, int nwg) {
    R r;
    const std::vector<Item> items = walk(r, tiles, G, nwg);
    const int B = (int)tiles.size();
    CHECK(r.n >= 1 && r.n <= nwg);
    // runs cut the units evenly and in order
    int at = 0;
    for (int w = 0; w < r.n; ++w) {
        CHECK(r.start_of(w) == (int)((long long)w * r.T / r.n) || r.n > va::MAX_RUNS);
        CHECK(r.start_of(w) == at);
        at = w == r.n - 1 ? r.T : r.start_of(w + 1);
        const int len = at - r.start_of(w);
        CHECK(len == r.T / r.n || len == r.T / r.n + 1);
    }
    // every tile of every merge group once, in order; its pieces in consecutive runs
    size_t i = 0;
    int most = 0;
    for (int b = 0; b < B; ++b)
        for (int g = 0; g < G; ++g) {
            const size_t i0 = i;
            int t = 0;
            while (t < tiles[b]) {
                CHECK(i < items.size());
                const Item& x = items[i];
                CHECK(x.b == b && x.g == g && x.t0 == t && x.cnt >= 1);
                CHECK(x.first == items[i0].w && x.w == x.first + (int)(i - i0));
                t += x.cnt;
                ++i;
            }
            CHECK(t == tiles[b]);
            const int pieces = (int)(i - i0);
            CHECK(pieces <= va::MAX_PIECES);
            for (size_t k = i0; k < i; ++k) CHECK(items[k].pieces == pieces);
            most = std::max(most, pieces);
        }
    CHECK(i == items.size());
    return most;
}

// Equal sequences: every merge group in 2^shift pieces, piece s in work-group (mg << shift) + s.
static void check_even(int t, int shift, int G, int B, int nwg) {
    va::Runs<1, 1> r;
    const int P = 1 << shift;
    int to = 0;
    for (int w = 0; w < nwg; ++w) {
        r.plan_even(t, shift, w, B, G);
        if (w >= B * G * P) {
            CHECK(!r.next());
            continue;
        }
        CHECK(r.next());
        r.locate();
        CHECK(r.b * G + r.g == w / P && r.g >= 0 && r.g < G && r.first == w / P * P && r.pieces == P);
        if (w % P == 0) to = 0;
        CHECK(r.t0 == to && r.cnt >= 1 && r.cnt <= t / P + 1);
        to += r.cnt;
        if (w % P == P - 1) CHECK(to == t);
        if (r.pass()) r.ub = t;
        CHECK(!r.next());                                    // one item each
    }
}

template <int COST>
static void random_batches(unsigned seed) {
    using R = va::Runs<COST, COST>;
    std::mt19937 gen(seed);
    const auto pick = [&](int lo, int hi) { return lo + (int)(gen() % (unsigned)(hi - lo + 1)); };
    for (int k = 0; k < 1500; ++k) {
        const int nwg = k % 3 == 0 ? 256 : k % 3 == 1 ? 512 : pick(1, va::MAX_RUNS);
        const int B = pick(1, 140), G = pick(1, 8);
        int top = 1 << pick(0, 11);
        std::vector<int> tiles(B);
        const bool even = k % 5 == 0;
        for (int& t : tiles) t = even ? top : pick(1, top);
        if (k % 4 == 0) tiles[pick(0, B - 1)] = 64 * top;
        check_batch<R>(tiles, G, nwg);
        // lengths that another stream rewrites under the kernel: no item of a sequence that is not there
        std::vector<int> other(B);
        for (int& t : other) t = pick(1, top);
        R r;
        walk(r, tiles, G, nwg, &other);
    }
}

int main(int argc, char** argv) {
    if (argc > 4) {
        const int min_run = std::atoi(argv[1]), nwg = std::atoi(argv[2]), G = std::atoi(argv[3]);
        std::vector<int> tiles;
        for (int i = 4; i < argc; ++i) tiles.push_back(std::atoi(argv[i]));
        int most = 0, n = 0, cut = 0;
        const auto one = [&](auto r) {
            most = check_batch<decltype(r)>(tiles, G, nwg);
            for (const Item& x : walk(r, tiles, G, nwg)) cut += x.pieces > 1;
            n = r.n;
        };
        if (min_run == 2) one(va::Runs<2, 2>{});
        else if (min_run == 1) one(va::Runs<1, 1>{});
        else one(va::Runs<0, 0>{});
        std::printf("runs %d pieces %d partials %d\n", n, most, cut);
        return 0;
    }
    random_batches<2>(1);
    random_batches<1>(2);
    random_batches<0>(3);
    // one long sequence beside short ones, around the lengths where the shortest run grows
    int reached = 0;
    for (int t = 50; t < 400; ++t) reached = std::max(reached, check_batch<va::Runs<1, 1>>({t, 1, 1, 3}, 2, 512));
    CHECK(reached == va::MAX_PIECES || reached == va::MAX_PIECES - 1);
    for (int shift = 0; shift <= 6; ++shift)
        for (int t : {1 << shift, (1 << shift) + 1, 3 << shift, 1000, 1 << 20})
            for (int G : {1, 2, 3, 8, 12})
                if (t >= 1 << shift) check_even(t, shift, G, 512 / (G << shift), 512);
    std::printf("runs: ok\n");
    return 0;
}
