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
// Equal lengths (DecodeArgs::even): every merge group in the same power of two of
// pieces, as static splits would be, found without the plan's divisions and scans. With
// one query slot such pieces are merged by the tagged protocol in the slot's store.
// Measured on MI355X, 8 x 16384, D 128, Hq = Hkv = 8, by the plan -> so (static splits):
// q8 46.5 -> 45.9 us (44.6), f16 82.3 -> 79.0 (78.4); 32 x 4096 46.7 -> 44.5 (44.6) and
// 82.1 -> 77.1 (77.8); Hq 32 / Hkv 8, 8 x 16384: q8 51.1 -> 49.8 (51.7), q4 37.4 -> 36.1.
//
// Every wave walks the plan by itself from seq_lens: one scan over the lengths
// finds the run's first item, then one length per further sequence. All of it is
// wave-uniform (va_runs.hpp has the arithmetic).
#pragma once
#include "va_device.hpp"
#include "va_fused.hpp"
#include "va_runs.hpp"

namespace va {

// Positions of a tile of the plan for a kernel whose work-group tile is TB: at least 128.
constexpr int balance_tile(int TB) { return TB >= 128 ? TB : 128; }
constexpr int BIG = 1 << 30;

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

template <int BT, int COST, int MIN_RUN, int QG>
struct Balance : Runs<COST, MIN_RUN> {
    using R = Runs<COST, MIN_RUN>;
    using R::at, R::end, R::base, R::b, R::g, R::ub, R::cost;
    const DecodeArgs& a;
    int len;                // the next item's sequence: its recorded length
    int ahead;              // the sequence after it
    unsigned epoch;         // equal sequences, tagged protocol (QG = 1): the merge group's, read with the lengths

    __device__ __forceinline__ int cap() const { return min(a.L, a.max_pages << a.page_shift); }
    // An invalid length is walked as far as it may be read (its output becomes NaN).
    __device__ __forceinline__ int tiles(int x) const { return max(1, (max(0, min(x, cap())) + BT - 1) / BT); }

    __device__ __forceinline__ Balance(bool on, const DecodeArgs& a_) : a(a_) {
        if (!on) return;
        const int lane = (int)(threadIdx.x & 63);
        const int G = a.hkv * a.nsub;
        // lengths 64 at a time; the first 64 stay for the search
        int x = a.seq_lens[min(lane, a.B - 1)];
        epoch = 0u;
        if (a.even >= 0) {
            const int x0 = __builtin_amdgcn_readfirstlane(x), t0 = tiles(x0);
            epoch = read_epoch<QG>(a, min((int)blockIdx.x >> a.even, a.B * G - 1));
            bool even = t0 >> a.even > 0 && __builtin_amdgcn_ballot_w64(x != x0) == 0;
            for (int c = 64; c < a.B && even; c += 64)
                even = __builtin_amdgcn_ballot_w64(a.seq_lens[min(c + lane, a.B - 1)] != x0) == 0;
            if (even) {
                R::plan_even(t0, a.even, (int)blockIdx.x, a.B, G);
                len = ahead = x0;
                asm volatile("");                            // keeps the two paths' stores apart (va_runs.hpp)
                return;
            }
        }
        int t = lane < a.B ? tiles(x) : 0, p = wave_scan(t);
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
        R::plan(sum, most, least, a.B, G, a.nwg);
        if (!R::take((int)blockIdx.x)) return;
        t += lane < a.B ? cost : 0;
        p += min(lane + 1, a.B) * cost;
        int before = 0;
        for (int c = 0;;) {                                  // ends: at < T, the units' total
            const uint64_t hit = __builtin_amdgcn_ballot_w64((before + p) * G > at);
            if (hit) {
                const int k = (int)__builtin_ctzll(hit);
                const int u = __builtin_amdgcn_readlane(t, k);
                len = __builtin_amdgcn_readlane(x, k);
                R::enter(c + k, before + __builtin_amdgcn_readlane(p, k) - u, u);
                break;
            }
            before += __builtin_amdgcn_readlane(p, 63);
            c += 64;
            if (c >= a.B) { at = end; return; }
            x = a.seq_lens[min(c + lane, a.B - 1)];
            t = c + lane < a.B ? tiles(x) + cost : 0;
            p = wave_scan(t);
        }
        ahead = a.seq_lens[min(b + 1, a.B - 1)];
    }

    __device__ __forceinline__ bool even() const { return R::n == 0; }

    // Past the current item: it ended its merge group or the run.
    __device__ __forceinline__ void advance() {
        if (!R::pass()) return;
        len = ahead;
        ub = tiles(len) + cost;
        ahead = a.seq_lens[min(b + 1, a.B - 1)];
    }
};

// End of an item of a balanced run: output if the merge group lies in one run,
// otherwise a partial and, by the last arrival, the merge.
template <int D, int NT, int QG, class Bal>
__device__ __forceinline__ void finish_item(int t, const DecodeArgs& a, const Route& rt, const Bal& w,
                                            const float (&M)[QG], const float (&ls)[QG], const float (&acc)[QG],
                                            unsigned epoch) {
    if (w.pieces == 1) {
        if (t < D) {
#pragma unroll
            for (int q = 0; q < QG; ++q) {
                if (q >= rt.nq) break;
                a.out[(size_t)(rt.oh0 + q) * D + t] = f2h_rne(ls[q] == 0.f ? 0.f : acc[q] / ls[q]);
            }
        }
        return;
    }
    if constexpr (QG == 1) {
        if (w.even()) {                          // splits like any others: their protocol is the faster one
            DecodeArgs e = a;
            e.S = w.pieces;
            const Route r{rt.mg, (int)blockIdx.x - w.first, rt.nq, rt.oh0};
            finish_partial<D, NT, QG>(e, r, M, ls, acc, epoch);
            return;
        }
    }
    constexpr int PSF = D + 2;
    const PartStore ps{a.ws + (size_t)(rt.mg + w.first) * (QG * PSF), QG * PSF, PSF, w.pieces, (int)blockIdx.x - w.first};
    finish_counted<D, NT, QG>(t, a, rt, ps, M, ls, acc);
}

} // namespace va
