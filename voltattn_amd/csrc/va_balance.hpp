// va_balance.hpp — the balanced work split of the paged kernels: a fixed number
// of work-groups shares the batch's tiles evenly, whatever the lengths of its
// sequences.
//
// A sequence of L positions has ceil(L / BT) tiles of BT positions (one if it is
// empty) for each of its merge groups (KV head, query sub-group). A merge group
// counts as its tiles plus COST units (what a work-group spends to begin and end
// one: lengths, page ids, query operand, first tile's latency, combine, output), unless
// every merge group fills a run, when each run begins about one item anyway. The
// units of the batch, numbered by (sequence, merge group, position), are cut into
// n <= nwg runs whose lengths differ by at most one; work-group w takes run w. A run
// covers the end of one merge group, any number of whole ones and the start of
// another: each such piece is one item. A merge group inside one run needs no merge;
// otherwise its pieces are merged by the last work-group to arrive
// (finish_counted), through partials in the caller's ws: piece w of merge group mg
// lies at slot mg + w, which no other piece shares (the next merge group starts at
// work-group w or later), so nwg + (merge groups) slots are enough.
//
// Every wave walks the plan by itself from seq_lens: one scan over the lengths
// finds the run's first item, then one length per further sequence. All of it is
// wave-uniform.
#pragma once
#include "va_device.hpp"
#include "va_fused.hpp"

namespace va {

// Positions of a tile of the plan for a kernel whose work-group tile is TB: at least 128.
constexpr int balance_tile(int TB) { return TB >= 128 ? TB : 128; }
constexpr int BIG = 1 << 30;
constexpr int MAX_PIECES = 64;   // pieces of one merge group that one merge takes

template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_rows_i(int old, int x) {
    return __builtin_amdgcn_update_dpp(old, x, CTRL, ROWS, 0xF, false);
}
// Inclusive sum over the lanes (row shifts, then the row broadcasts).
__device__ __forceinline__ int wave_scan(int x) {
    x += dpp_rows_i<0x111, 0xF>(0, x);
    x += dpp_rows_i<0x112, 0xF>(0, x);
    x += dpp_rows_i<0x114, 0xF>(0, x);
    x += dpp_rows_i<0x118, 0xF>(0, x);
    x += dpp_rows_i<0x142, 0xA>(0, x);
    x += dpp_rows_i<0x143, 0xC>(0, x);
    return x;
}
__device__ __forceinline__ int wave_scan_max(int x) {           // x >= 0; lane 63 holds the maximum
    x = max(x, dpp_rows_i<0x111, 0xF>(0, x));
    x = max(x, dpp_rows_i<0x112, 0xF>(0, x));
    x = max(x, dpp_rows_i<0x114, 0xF>(0, x));
    x = max(x, dpp_rows_i<0x118, 0xF>(0, x));
    x = max(x, dpp_rows_i<0x142, 0xA>(0, x));
    x = max(x, dpp_rows_i<0x143, 0xC>(0, x));
    return x;
}

template <int BT, int COST, int MIN_RUN>
struct Balance {
    const DecodeArgs& a;
    int G;                  // merge groups per sequence
    int cost;               // COST or 0
    int n, q, r;            // runs; run w starts at unit w*q + w*r/n
    float rn, rt;           // 1 / n; runs per unit
    int at, end;            // units of this work-group's run still to do
    int base;               // units per merge group of the sequences before b
    int b, g, u0, ub;       // the next item: sequence, merge group in it, first unit, units of the merge group
    int len;                // the sequence's recorded length
    int ahead;              // the next sequence's
    // current item: its tiles, the run that holds the merge group's first tile, pieces of the merge group
    int t0, cnt, first, pieces;

    __device__ __forceinline__ int cap() const { return min(a.L, a.max_pages << a.page_shift); }
    // An invalid length is walked as far as it may be read (its output becomes NaN).
    __device__ __forceinline__ int tiles(int x) const { return max(1, (max(0, min(x, cap())) + BT - 1) / BT); }
    // w*r < 2^22 and n < 2^11: half a step's margin is above the product's rounding
    __device__ __forceinline__ int start_of(int w) const { return w * q + (int)(((float)(w * r) + 0.5f) * rn); }
    __device__ __forceinline__ int run_of(int unit) const {
        int w = min(n - 1, (int)((float)unit * rt));
        while (w > 0 && start_of(w) > unit) --w;             // the estimate is off by the rounding of a product
        while (w < n - 1 && start_of(w + 1) <= unit) ++w;
        return w;
    }

    __device__ __forceinline__ Balance(bool on, const DecodeArgs& a_) : a(a_) {
        if (!on) return;
        const int lane = (int)(threadIdx.x & 63);
        G = a.hkv * a.nsub;
        // lengths 64 at a time; the first 64 stay for the search
        const int x0 = a.seq_lens[min(lane, a.B - 1)];
        int x = x0, t = lane < a.B ? tiles(x) : 0, p = wave_scan(t);
        int sum = __builtin_amdgcn_readlane(p, 63);
        int most = __builtin_amdgcn_readlane(wave_scan_max(t), 63);
        int least = BIG - __builtin_amdgcn_readlane(wave_scan_max(lane < a.B ? BIG - t : 0), 63);
        for (int c = 64; c < a.B; c += 64) {
            const bool in = c + lane < a.B;
            const int y = in ? tiles(a.seq_lens[min(c + lane, a.B - 1)]) : 0;
            sum += __builtin_amdgcn_readlane(wave_scan(y), 63);
            most = max(most, __builtin_amdgcn_readlane(wave_scan_max(y), 63));
            least = min(least, BIG - __builtin_amdgcn_readlane(wave_scan_max(in ? BIG - y : 0), 63));
        }
        cost = (long long)least * a.nwg >= (long long)sum * G ? 0 : COST;
        const int T = (sum + cost * a.B) * G;
        most += cost;
        t += lane < a.B ? cost : 0;
        p += min(lane + 1, a.B) * cost;
        n = min(a.nwg, max(1, T / max(MIN_RUN, (most + MAX_PIECES - 3) / (MAX_PIECES - 2))));
        at = end = 0;
        const int w = (int)blockIdx.x;
        if (w >= n) return;
        q = T / n;
        r = T - q * n;
        rn = 1.f / (float)n;
        rt = (float)n / (float)T;
        at = start_of(w);
        end = w == n - 1 ? T : start_of(w + 1);
        base = 0;
        for (int c = 0;;) {                                  // ends: at < T, the units' total
            const uint64_t hit = __builtin_amdgcn_ballot_w64((base + p) * G > at);
            if (hit) {
                const int k = (int)__builtin_ctzll(hit);
                ub = __builtin_amdgcn_readlane(t, k);
                len = __builtin_amdgcn_readlane(x, k);
                base += __builtin_amdgcn_readlane(p, k) - ub;
                b = c + k;
                break;
            }
            base += __builtin_amdgcn_readlane(p, 63);
            c += 64;
            if (c >= a.B) { at = end; return; }
            x = a.seq_lens[min(c + lane, a.B - 1)];
            t = c + lane < a.B ? tiles(x) + cost : 0;
            p = wave_scan(t);
        }
        ahead = a.seq_lens[min(b + 1, a.B - 1)];
        const int off = at - base * G;
        g = (int)((float)off * __builtin_amdgcn_rcpf((float)ub));   // at most a step off
        while (g > 0 && g * ub > off) --g;
        while ((g + 1) * ub <= off) ++g;
        g = uniform(g);
        u0 = off - g * ub;
    }

    // The next item of the run, or false.
    __device__ __forceinline__ bool next() {
        const int u1 = min(ub, u0 + end - at);               // past the last unit here
        if (at >= end || u1 <= cost) return false;           // done, or the run ends before a tile
        t0 = max(0, u0 - cost);
        cnt = u1 - cost - t0;
        at += u1 - u0;
        return true;
    }
    // Where the merge group of the current item starts, and its pieces: needed at the
    // item's end only, so the caller asks while the first loads are under way.
    __device__ __forceinline__ void locate() {
        const int gs = base * G + g * ub;                    // the merge group's first unit
        first = run_of(gs + cost);
        pieces = run_of(gs + ub - 1) - first + 1;
    }
    // Past the current item: it ended its merge group or the run.
    __device__ __forceinline__ void advance() {
        u0 = 0;
        if (++g == G) {
            g = 0;
            base += ub;
            ++b;
            len = ahead;
            ub = tiles(len) + cost;
            ahead = a.seq_lens[min(b + 1, a.B - 1)];
        }
    }
};

// End of an item of a balanced run: output if the merge group lies in one run,
// otherwise a partial and, by the last arrival, the merge.
template <int D, int NT, int QG, class Bal>
__device__ __forceinline__ void finish_item(const DecodeArgs& a, const Route& rt, const Bal& w,
                                            const float (&M)[QG], const float (&ls)[QG], const float (&acc)[QG]) {
    if (w.pieces == 1) {
        const int t = (int)threadIdx.x;
        if (t < D) {
#pragma unroll
            for (int q = 0; q < QG; ++q) {
                if (q >= rt.nq) break;
                a.out[(size_t)(rt.oh0 + q) * D + t] = f2h_rne(ls[q] == 0.f ? 0.f : acc[q] / ls[q]);
            }
        }
        return;
    }
    constexpr int PSF = D + 2;
    const PartStore ps{a.ws + (size_t)(rt.mg + w.first) * (QG * PSF), QG * PSF, PSF, w.pieces, (int)blockIdx.x - w.first};
    finish_counted<D, NT, QG>(a, rt, ps, M, ls, acc);
}

} // namespace va
