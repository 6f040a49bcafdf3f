// va_runs.hpp — the arithmetic of balanced runs (va_balance.hpp): scalars only, so that
// tests/cpp/test_runs.cpp walks the same code on the host.
//
// The units of a batch, T in all, are cut into n runs whose lengths differ by at most one;
// run w starts at unit w*q + w*r/n (q = T / n, r = T - q*n). A merge group is `cost` units
// and one per tile.
#pragma once
#include <cstdint>

#ifdef __HIPCC__
#define VA_RUNS_FN __host__ __device__ __forceinline__
#else
#define VA_RUNS_FN inline
#endif

namespace va {

constexpr int MAX_PIECES = 64;   // pieces of one merge group that one merge takes
constexpr int MAX_RUNS = 1024;

// A value every lane of the wave holds. (Float products are vector instructions: without
// this, all that follows from one would be computed, and held, in vector registers.)
VA_RUNS_FN int run_scalar(int x) {
#ifdef __HIP_DEVICE_COMPILE__
    return __builtin_amdgcn_readfirstlane(x);
#else
    return x;
#endif
}

template <int COST, int MIN_RUN>
struct Runs {
    int G, B;               // merge groups per sequence, sequences
    int cost;               // COST or 0
    int T, n, q, r;
    float rn, rt;           // 1 / n; runs per unit
    int at, end;            // units of this work-group's run still to do
    int base;               // units per merge group of the sequences before b
    int b, g, u0, ub;       // the next item: sequence, merge group in it, first unit, units of the merge group
    // the current item: its tiles, the run that holds the merge group's first tile, pieces of the merge group
    int t0, cnt, first, pieces;

    // sum, most, least: tiles of a merge group over the sequences. T below 2^30, nwg at most MAX_RUNS.
    VA_RUNS_FN void plan(int sum, int most, int least, int B_, int G_, int nwg) {
        B = B_;
        G = G_;
        cost = (int64_t)least * nwg >= (int64_t)sum * G ? 0 : COST;
        T = (sum + cost * B) * G;
        int run = (most + cost + MAX_PIECES - 3) / (MAX_PIECES - 2);   // at most MAX_PIECES pieces
        run = run > MIN_RUN ? run : MIN_RUN;
        n = T / run;
        n = n < nwg ? n : nwg;
        n = n > 1 ? n : 1;
        q = T / n;
        r = T - q * n;
        rn = 1.f / (float)n;
        rt = (float)n / (float)T;
    }
    // w*r is exact below 2^24; the product, below n, is off by less than 2^-23 of n: under the
    // half step's 2^-1 / n up to n = 1448
    VA_RUNS_FN int start_of(int w) const { return w * q + run_scalar((int)(((float)(w * r) + 0.5f) * rn)); }
    VA_RUNS_FN int run_of(int unit) const {
        int w = run_scalar((int)((float)unit * rt));
        w = w < n - 1 ? w : n - 1;
        while (w > 0 && start_of(w) > unit) --w;
        while (w < n - 1 && start_of(w + 1) <= unit) ++w;
        return w;
    }
    // Run w, and false if there is none.
    VA_RUNS_FN bool take(int w) {
        at = end = 0;
        if (w >= n) return false;
        at = start_of(w);
        end = w == n - 1 ? T : start_of(w + 1);
        return true;
    }
    // The run's first item lies in sequence b_ (units base_ before it, ub_ in it).
    VA_RUNS_FN void enter(int b_, int base_, int ub_) {
        b = b_;
        base = base_;
        ub = ub_;
        const int off = at - base * G;
        g = run_scalar((int)((float)off / (float)ub));       // at most a step off
        while (g > 0 && g * ub > off) --g;
        while ((g + 1) * ub <= off) ++g;
        u0 = off - g * ub;
    }
    // The next item of the run, or false. (b < B holds by itself while the lengths stay what
    // they were when the plan was made; without it a length rewritten under a running
    // kernel would lead past the block table and the output.)
    VA_RUNS_FN bool next() {
        const int left = u0 + end - at;
        const int u1 = ub < left ? ub : left;                // past the last unit here
        if (at >= end || b >= B || u1 <= cost) return false; // done, or the run ends before a tile
        t0 = u0 > cost ? u0 - cost : 0;
        cnt = u1 - cost - t0;
        at += u1 - u0;
        return true;
    }
    // Sequences of t >= 2^shift tiles each, every merge group in 2^shift pieces of a
    // work-group each: what plan() comes to where equal sequences fill the work-groups,
    // without its divisions. Work-groups past the last merge group have no item.
    // (Straight-line code: stores to other members on other paths would be joined through a
    // pointer, and the whole plan kept in scratch memory.)
    VA_RUNS_FN void plan_even(int t, int shift, int w, int B_, int G_) {
        const int mg = w >> shift, s = w & ((1 << shift) - 1);
        const int to = (int)(((int64_t)t * (s + 1)) >> shift);
        B = B_;
        G = G_;
        cost = 0;
        base = 0;
        n = 0;                                               // first and pieces are known: locate() leaves them
        b = (int)((uint32_t)mg / (uint32_t)G_);
        g = mg - b * G_;
        ub = t;
        u0 = (int)(((int64_t)t * s) >> shift);
        at = 0;
        end = mg < B_ * G_ ? to - u0 : 0;
        first = mg << shift;
        pieces = 1 << shift;
    }
    // Where the merge group of the current item starts, and its pieces.
    VA_RUNS_FN void locate() {
        int w = first, k = pieces;
        if (n > 0) {
            const int gs = base * G + g * ub;                // the merge group's first unit
            w = run_of(gs + cost);
            k = run_of(gs + ub - 1) - w + 1;
        }
        first = w;
        pieces = k;
    }
    // Past the current item, which ended its merge group or the run; true if it was the
    // sequence's last merge group: the caller then sets ub.
    VA_RUNS_FN bool pass() {
        u0 = 0;
        if (++g < G) return false;
        g = 0;
        base += ub;
        ++b;
        return true;
    }
};

} // namespace va
