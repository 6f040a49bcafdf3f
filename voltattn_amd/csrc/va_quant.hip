// va_quant.hip — device-side producers of the decode path's inputs:
//   * quantize_groups / append_rows, append_span: the symmetric per-group quantizer +
//     packer (over fp32 rows, or over fp16 rows written into a paged cache at
//     given positions: the cache write path), bit-exact
//     with the reference's host quantize() (src/voltattn.cu:705-745) for
//     G in {32, 64}: amax in fp32, s = amax/lim (IEEE division), the fp16
//     scale rounded to nearest even, codes clamp(rint(x / float(scale))), with
//     a non-finite quotient giving code 0 as x86-64 lrint + int truncation does;
//   * dequantize_groups: the inverse, packed codes and fp16 scales back to
//     fp32 values, bit-exact with the reference's dq() (src/voltattn.cu:747-767);
//   * f32_to_f16: round-to-nearest-even conversion of fp32 arrays (the
//     reference's __float2half over the f16-format K/V, src/voltattn.cu:866-868);
//   * fill_normal: seeded N(0,1) bench data, Philox4x32-10 (Salmon et al.,
//     SC'11) counters through the Box-Muller transform.
#include "va_device.hpp"
#include "va_kernels.hpp"

#include <algorithm>

namespace va {

template <int BITS> struct QLim;
template <> struct QLim<8> { static constexpr int value = 127; };
template <> struct QLim<4> { static constexpr int value = 7; };
template <> struct QLim<3> { static constexpr int value = 3; };

// The quantizer, packer and unpacker give a lane E consecutive elements of a
// group (E = 4 of fp32, 8 of fp16: one 16-byte access), so a wave reads and writes
// contiguous kilobytes and the lanes of a group exchange its maximum with DPP. They
// are bound by memory; a thread per group (64 to 256 contiguous bytes each) touched
// 64 cache lines with every access. Same-box A/B on MI355X, D 128: dequantize 32 x
// 16384 rows q8 91 -> 47 us, q4 90 -> 42, q3 88 -> 41 (6.6 to 7.2 TB/s); quantize 32 x
// 32768 rows G 32 q8 122 -> 105, q4 105 -> 90, q3 102 -> 90, G 64 130 -> 90; append
// 4 x 8 x 8192 rows f16 28.4 -> 20.4, q8 29.6 -> 22.7, q4 26.9 -> 22.6, q3 24.4 -> 23.4.
constexpr int UNR = 2;               // accesses per lane in flight: 1 and 4 were 3-9% slower
constexpr int APP_U = 4;
constexpr size_t MAX_GRID = 65536;   // 16384 work-groups that stride: 2-4% slower

// Written once and not read back by the kernel: a non-temporal store (append f16
// 26.0 -> 20.4 us, quantize q8 112.7 -> 105.5 in the sizes above, dequantize q8 66.6
// -> 47.9, against plain stores).
template <class T>
__device__ __forceinline__ void stream_store(T* p, T v) { __builtin_nontemporal_store(v, p); }

// Codes of E values against the group scale sh (its fp16 value): bit-exact with
// clamp(rint(x / sh)), a non-finite quotient giving 0. x * rcp(sh) is within 2^-22 of the
// IEEE quotient, relatively. A quotient of lim + 1 or more clamps whichever side of a
// boundary it lands; below, |quotient| < 128, so the two differ by less than 2^-15:
// where no value lies within 2^-14 of a rounding boundary (twice that; and none is NaN or
// infinite), rounding it gives the same code; otherwise the wave divides.
template <int BITS, int E>
__device__ __forceinline__ void quant_codes(const float (&x)[E], float sh, int (&code)[E]) {
    constexpr int lim = QLim<BITS>::value;
    const float r = __builtin_amdgcn_rcpf(sh);
    float n[E], far = 0.f, any = 0.f;              // largest distance to the code; NaN if one is
#pragma unroll
    for (int i = 0; i < E; ++i) {
        const float y = x[i] * r;
        n[i] = __builtin_rintf(y);
        const float d = __builtin_fabsf(y - n[i]);
        far = fmaxf(far, d);
        any += d;
    }
    if (__builtin_amdgcn_ballot_w64(!(far < 0.5f - 0x1p-14f && any < (float)E)) != 0) {
        asm volatile("");                          // kept a branch: the divisions are not computed ahead of it
#pragma unroll
        for (int i = 0; i < E; ++i) {
            const float t = x[i] / sh;
            n[i] = __builtin_isfinite(t) ? __builtin_rintf(t) : 0.f;
        }
    }
#pragma unroll
    for (int i = 0; i < E; ++i) code[i] = (int)__builtin_amdgcn_fmed3f(n[i], (float)-lim, (float)lim);
}

// The fp16 scale of a group from its largest |x|.
template <int BITS>
__device__ __forceinline__ uint16_t quant_scale(float amax) {
    return f2h_rne(amax > 0.f ? amax / (float)QLim<BITS>::value : 1.f);
}

// Pack the lane's E codes and write its share of the group's bytes, the lane's
// elements starting `e` elements into the 4-byte aligned stream at dst. q3: E codes
// are 12 or 24 bits; the four 24-bit values of 32 elements make three words, word k
// from values k and k + 1.
template <int BITS, int E>
__device__ __forceinline__ void pack_store(const int (&code)[E], uint8_t* dst, size_t e, bool on) {
    if constexpr (BITS == 8) {
        uint32_t w[E / 4];
#pragma unroll
        for (int k = 0; k < E / 4; ++k)
            w[k] = ((uint32_t)code[4 * k] & 0xFFu) | ((uint32_t)code[4 * k + 1] & 0xFFu) << 8 |
                   ((uint32_t)code[4 * k + 2] & 0xFFu) << 16 | (uint32_t)code[4 * k + 3] << 24;
        if (!on) return;
        uint32_t* d = reinterpret_cast<uint32_t*>(dst + e);
#pragma unroll
        for (int k = 0; k < E / 4; ++k) stream_store(d + k, w[k]);
    } else if constexpr (BITS == 4) {             // element i: byte i/2, low nibble when i even
        uint32_t w = 0;
#pragma unroll
        for (int i = 0; i < E; ++i) w |= (uint32_t)(code[i] + 8) << (4 * i);
        if (!on) return;
        if constexpr (E == 8) stream_store(reinterpret_cast<uint32_t*>(dst + e / 2), w);
        else stream_store(reinterpret_cast<uint16_t*>(dst + e / 2), (uint16_t)w);
    } else {                                       // element i: bits [3i, 3i+3), little endian
        uint32_t w = 0;
#pragma unroll
        for (int i = 0; i < E; ++i) w |= (uint32_t)(code[i] + 4) << (3 * i);
        constexpr int SPAN = 32 / E;               // lanes of 32 elements
        const int l = (int)(threadIdx.x & (SPAN - 1));
        uint32_t next;                             // the next 24-bit value of the same 32 elements
        if constexpr (E == 4) {                    // pairs of lanes make a value, in the even lane
            w |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)w, DPP_QP_XOR1, 0xF, 0xF, true) << 12;
            next = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)w, 0x102 /* row_shl:2 */, 0xF, 0xF, true);
        } else {
            next = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)w, 0x101 /* row_shl:1 */, 0xF, 0xF, true);
        }
        const int k = E == 4 ? l >> 1 : l;
        if (!on || k == 3 || (E == 4 && (l & 1))) return;
        stream_store(reinterpret_cast<uint32_t*>(dst) + (e / 32) * 3 + k, (w & 0xFFFFFFu) >> (8 * k) | next << (24 - 8 * k));
    }
}

// 4 elements per lane; a wave's access covers 256. ne is a multiple of G.
template <int BITS, int G>
__global__ __launch_bounds__(256) void quantize_groups(const float* __restrict__ x, size_t ne,
                                                       uint8_t* __restrict__ packed,
                                                       uint16_t* __restrict__ scales) {
    constexpr size_t STEP = 256 * 4;               // elements per work-group and access
    for (size_t e0 = (size_t)blockIdx.x * (STEP * UNR); e0 < ne; e0 += (size_t)gridDim.x * (STEP * UNR)) {
        f32x4 v[UNR];
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
            const size_t e = e0 + u * STEP + threadIdx.x * 4;
            v[u] = e < ne ? __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(x + e)) : f32x4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
            const size_t e = e0 + u * STEP + threadIdx.x * 4;
            const float xv[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
            float amax = 0.f;
#pragma unroll
            for (int i = 0; i < 4; ++i) amax = fmaxf(amax, __builtin_fabsf(xv[i]));
            const uint16_t sb = quant_scale<BITS>(group_max<G / 4>(amax));
            int code[4];
            quant_codes<BITS, 4>(xv, h2f(sb), code);
            pack_store<BITS, 4>(code, packed, e, e < ne);
            if (e < ne && e % G == 0) scales[e / G] = sb;
        }
    }
}

// Inverse of the packer, 4 elements per lane: value = float(scale) * code.
// The reference's dq() forms the same product in double; an fp16 scale times a
// code of at most 7 bits is exact in fp32 (non-finite scales give the same
// inf/NaN), so the results are equal bit for bit. Code layouts as in pack_store:
// q8 int8, q4 nibble + 8 (low nibble first), q3 3-bit fields + 4. Each store
// instruction of a wave fills whole lines; the few code bytes and the scale of a
// lane come from lines that its neighbours share.
template <int BITS, int G>
__global__ __launch_bounds__(256) void dequantize_groups(const uint8_t* __restrict__ packed,
                                                         const uint16_t* __restrict__ scales,
                                                         size_t ne, float* __restrict__ out) {
    constexpr size_t STEP = 256 * 4;
    for (size_t e0 = (size_t)blockIdx.x * (STEP * UNR); e0 < ne; e0 += (size_t)gridDim.x * (STEP * UNR)) {
        uint32_t w[UNR];
        uint16_t sb[UNR];
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
            const size_t e = e0 + u * STEP + threadIdx.x * 4;
            w[u] = 0;
            sb[u] = 0;
            if (e < ne) {
                if constexpr (BITS == 8) {
                    w[u] = *reinterpret_cast<const uint32_t*>(packed + e);
                } else if constexpr (BITS == 4) {
                    w[u] = *reinterpret_cast<const uint16_t*>(packed + e / 2);
                } else {                           // 12 bits at bit 12l of the three words of 32 elements
                    const int bit = 12 * (int)(threadIdx.x & 7);
                    const uint32_t* p = reinterpret_cast<const uint32_t*>(packed) + (e / 32) * 3;
                    const int k = bit >> 5;
                    w[u] = __builtin_amdgcn_alignbit(p[k < 2 ? k + 1 : 2], p[k], bit & 31);
                }
                sb[u] = scales[e / G];
            }
        }
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
            const size_t e = e0 + u * STEP + threadIdx.x * 4;
            const float s = h2f(sb[u]);
            float f[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                int c;
                if constexpr (BITS == 8) c = (int)(w[u] << (24 - 8 * i)) >> 24;
                else if constexpr (BITS == 4) c = (int)((w[u] >> (4 * i)) & 15u) - 8;
                else c = (int)((w[u] >> (3 * i)) & 7u) - 4;
                f[i] = s * (float)c;
            }
            if (e < ne) stream_store(reinterpret_cast<f32x4*>(out + e), (f32x4{f[0], f[1], f[2], f[3]}));
        }
    }
}

// Destination row of (sequence b, KV head hk, position p) in a page pool
// [num_pages][hkv][page_rows][...], or -1 when the position lies past the
// block table or on a page id outside the pool (such rows are not written).
__device__ __forceinline__ long long paged_row(const AppendArgs& a, int b, int hk, int p) {
    if (p < 0) return -1;
    const int pi = (int)a.by_page.div((uint32_t)p);
    if (pi >= a.max_pages) return -1;
    const int page = a.block_table[(size_t)b * a.max_pages + pi];
    if (page < 0 || page >= a.num_pages) return -1;
    return ((long long)page * a.hkv + hk) * a.page_rows + (p - pi * a.page_rows);
}

// Where new row `row` = (b*hkv + hk)*n + r goes.
__device__ __forceinline__ long long append_row(const AppendArgs& a, size_t row) {
    uint32_t r, bh;
    if (a.many) {                                  // uniform: 2^31 rows or more
        bh = (uint32_t)(row / (uint32_t)a.n);
        r  = (uint32_t)(row - (size_t)bh * (uint32_t)a.n);
    } else {
        bh = a.by_n.div((uint32_t)row);
        r  = (uint32_t)row - bh * (uint32_t)a.n;
    }
    const uint32_t b = a.by_hkv.div(bh);
    return paged_row(a, (int)b, (int)(bh - b * (uint32_t)a.hkv), a.start[b] + (int)r);
}

// Quantize-and-append (f16 rows: copy) of the new rows x[b][hk][r][D] (fp16),
// written at position start[b] + r: 8 elements per lane. ne = rows * D.
template <int BITS, int G>
__device__ __forceinline__ void append_lane(const AppendArgs& a, const u32x4& w, bool on, size_t to) {
    if constexpr (BITS == 16) {
        if (on) stream_store(reinterpret_cast<u32x4*>(a.pages + to * 2), w);
    } else {
        float xv[8];
        float amax = 0.f;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            xv[2 * k]     = h2f_lo(w[k]);
            xv[2 * k + 1] = h2f_hi(w[k]);
            // max(|x0|, |x1|, amax) of converted values, so no signalling NaN
            asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(amax) : "v"(xv[2 * k]), "v"(xv[2 * k + 1]));
        }
        const uint16_t sb = quant_scale<BITS>(group_max<G / 8>(amax));
        int code[8];
        quant_codes<BITS, 8>(xv, h2f(sb), code);
        pack_store<BITS, 8>(code, a.pages, to, on);
        if (on && to % G == 0) a.scales[to / G] = sb;
    }
}

// Few rows per (sequence, KV head): lanes are dealt over all new rows.
template <int BITS, int G>
__global__ __launch_bounds__(256) void append_rows(AppendArgs a, size_t ne) {
    constexpr size_t STEP = 256 * 8;               // elements per work-group
    const int dsh = a.D == 128 ? 7 : 6;
    for (size_t e0 = (size_t)blockIdx.x * STEP; e0 < ne; e0 += (size_t)gridDim.x * STEP) {
        const size_t e = e0 + threadIdx.x * 8;
        const bool in = e < ne;
        const u32x4 w = in ? *reinterpret_cast<const u32x4*>(a.x + e) : u32x4{0u, 0u, 0u, 0u};
        const long long row = in ? append_row(a, e >> dsh) : -1;
        append_lane<BITS, G>(a, w, row >= 0, ((size_t)(row < 0 ? 0 : row) << dsh) + (e & ((1u << dsh) - 1u)));
    }
}

// A work-group takes 256 / (D/8) * U consecutive new rows of one (sequence, KV
// head), so that pair and its start are scalars and U rows per lane are in flight.
template <int BITS, int G, int D, int U>
__global__ __launch_bounds__(256) void append_span(AppendArgs a) {
    constexpr int RP = 256 * 8 / D;                // rows per access of the work-group
    const int nblk = (a.n + RP * U - 1) / (RP * U);
    for (int g = (int)blockIdx.x; g < a.B * a.hkv * nblk; g += (int)gridDim.x) {
        const int bh = g / nblk, r0 = (g - bh * nblk) * (RP * U) + (int)threadIdx.x / (D / 8);
        const int b = bh / a.hkv, hk = bh - b * a.hkv;
        const int start = a.start[b];
        const int32_t* table = a.block_table + (size_t)b * a.max_pages;
        const uint16_t* x = a.x + (size_t)bh * a.n * D + (threadIdx.x % (D / 8)) * 8;
        u32x4 w[U];
        int page[U], at[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int r = r0 + u * RP;
            w[u] = *reinterpret_cast<const u32x4*>(x + (size_t)min(r, a.n - 1) * D);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int r = r0 + u * RP, p = start + r;
            const int pi = p < 0 ? a.max_pages : (int)a.by_page.div((uint32_t)p);
            at[u] = p - pi * a.page_rows;
            page[u] = r < a.n && pi < a.max_pages ? table[pi] : -1;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool on = page[u] >= 0 && page[u] < a.num_pages;
            const size_t row = on ? ((size_t)page[u] * a.hkv + hk) * a.page_rows + at[u] : 0;
            append_lane<BITS, G>(a, w[u], on, row * D + (threadIdx.x % (D / 8)) * 8);
        }
    }
}

__global__ __launch_bounds__(256) void f32_to_f16_kernel(const float* __restrict__ x, size_t n,
                                                         uint16_t* __restrict__ out) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
        out[i] = f2h_rne(x[i]);
}

// Philox4x32-10 block: counter (c0..c3), key (k0, k1).
__device__ __forceinline__ u32x4 philox4x32_10(u32x4 c, uint32_t k0, uint32_t k1) {
    constexpr uint32_t M0 = 0xD2511F53u, M1 = 0xCD9E8D57u;
    constexpr uint32_t W0 = 0x9E3779B9u, W1 = 0xBB67AE85u;
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        const uint32_t hi0 = __umulhi(M0, c.x), lo0 = M0 * c.x;
        const uint32_t hi1 = __umulhi(M1, c.z), lo1 = M1 * c.z;
        c = u32x4{hi1 ^ c.y ^ k0, lo1, hi0 ^ c.w ^ k1, lo0};
        k0 += W0;
        k1 += W1;
    }
    return c;
}

__global__ __launch_bounds__(256) void fill_normal_kernel(float* __restrict__ x, size_t n,
                                                          uint32_t k0, uint32_t k1) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    const size_t nblk = (n + 3) / 4;
    for (size_t b = (size_t)blockIdx.x * blockDim.x + threadIdx.x; b < nblk; b += stride) {
        const u32x4 r = philox4x32_10(u32x4{(uint32_t)b, (uint32_t)(b >> 32), 0u, 0u}, k0, k1);
        float z[4];
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const uint32_t a = p ? r.z : r.x, c = p ? r.w : r.y;
            const float u1 = (float)((a >> 8) + 1u) * 5.9604644775390625e-8f;  // (0, 1]
            const float u2 = (float)(c >> 8) * 5.9604644775390625e-8f;         // [0, 1)
            const float rad = sqrtf(-2.f * logf(u1));
            float sn, cs;
            sincosf(6.28318530717958648f * u2, &sn, &cs);
            z[2 * p] = rad * cs;
            z[2 * p + 1] = rad * sn;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (4 * b + i < n) x[4 * b + i] = z[i];
    }
}

static unsigned grid_for(size_t work) {
    const size_t blocks = (work + 255) / 256;
    return (unsigned)(blocks < 16384 ? (blocks ? blocks : 1) : 16384);
}

// Work-groups of `per` elements each over ne, at most MAX_GRID (the kernels stride).
static unsigned grid_of(size_t ne, size_t per) {
    const size_t blocks = (ne + per - 1) / per;
    return (unsigned)(blocks < MAX_GRID ? (blocks ? blocks : 1) : MAX_GRID);
}

hipError_t launch_quantize(int bits, int G, const float* x, size_t rows, int D, uint8_t* packed,
                           uint16_t* scales, hipStream_t stream) {
    const size_t ne = rows * (size_t)D;
    const dim3 grid(grid_of(ne, 1024 * UNR)), block(256);
#define VA_QLAUNCH(B, GG) hipLaunchKernelGGL((quantize_groups<B, GG>), grid, block, 0, stream, x, ne, packed, scales)
    if (G == 32) {
        if (bits == 8) VA_QLAUNCH(8, 32); else if (bits == 4) VA_QLAUNCH(4, 32); else VA_QLAUNCH(3, 32);
    } else {
        if (bits == 8) VA_QLAUNCH(8, 64); else if (bits == 4) VA_QLAUNCH(4, 64); else VA_QLAUNCH(3, 64);
    }
#undef VA_QLAUNCH
    return hipGetLastError();
}

hipError_t launch_dequantize(int bits, int G, const uint8_t* packed, const uint16_t* scales, size_t rows,
                             int D, float* out, hipStream_t stream) {
    const size_t ne = rows * (size_t)D;
    const dim3 grid(grid_of(ne, 1024 * UNR)), block(256);
#define VA_DLAUNCH(B, GG) hipLaunchKernelGGL((dequantize_groups<B, GG>), grid, block, 0, stream, packed, scales, ne, out)
    if (G == 32) {
        if (bits == 8) VA_DLAUNCH(8, 32); else if (bits == 4) VA_DLAUNCH(4, 32); else VA_DLAUNCH(3, 32);
    } else {
        if (bits == 8) VA_DLAUNCH(8, 64); else if (bits == 4) VA_DLAUNCH(4, 64); else VA_DLAUNCH(3, 64);
    }
#undef VA_DLAUNCH
    return hipGetLastError();
}

hipError_t launch_append(int bits, int G, const AppendArgs& args, hipStream_t stream) {
    AppendArgs a = args;
    a.by_n    = FastDiv::of((uint32_t)a.n);
    a.by_hkv  = FastDiv::of((uint32_t)a.hkv);
    a.by_page = FastDiv::of((uint32_t)a.page_rows);
    a.many = (size_t)a.B * a.hkv * a.n >= 0x80000000ull;
    const size_t ne = (size_t)a.B * a.hkv * a.n * a.D;
    const int span = 2048 * APP_U / a.D;           // rows per work-group of append_span
    const long long spans = (long long)a.B * a.hkv * ((a.n + span - 1) / span);
    // half-filled work-groups cost more than a division per lane
    const bool wide = a.n >= span / 2 && spans < 0x40000000LL;
    const dim3 grid(wide ? (unsigned)std::min(spans, (long long)MAX_GRID) : grid_of(ne, 2048)), block(256);
#define VA_ALAUNCH(B, GG)                                                                                       \
    do {                                                                                                        \
        if (!wide) hipLaunchKernelGGL((append_rows<B, GG>), grid, block, 0, stream, a, ne);                     \
        else if (a.D == 128) hipLaunchKernelGGL((append_span<B, GG, 128, APP_U>), grid, block, 0, stream, a);   \
        else hipLaunchKernelGGL((append_span<B, GG, 64, APP_U>), grid, block, 0, stream, a);                    \
    } while (0)
    if (bits == 16) {
        VA_ALAUNCH(16, 32);
    } else if (G == 32) {
        if (bits == 8) VA_ALAUNCH(8, 32); else if (bits == 4) VA_ALAUNCH(4, 32); else VA_ALAUNCH(3, 32);
    } else {
        if (bits == 8) VA_ALAUNCH(8, 64); else if (bits == 4) VA_ALAUNCH(4, 64); else VA_ALAUNCH(3, 64);
    }
#undef VA_ALAUNCH
    return hipGetLastError();
}

hipError_t launch_f32_to_f16(const float* x, size_t n, uint16_t* out, hipStream_t stream) {
    hipLaunchKernelGGL(f32_to_f16_kernel, dim3(grid_for(n)), dim3(256), 0, stream, x, n, out);
    return hipGetLastError();
}

hipError_t launch_fill_normal(float* x, size_t n, uint64_t seed, hipStream_t stream) {
    hipLaunchKernelGGL(fill_normal_kernel, dim3(grid_for((n + 3) / 4)), dim3(256), 0, stream, x, n,
                       (uint32_t)seed, (uint32_t)(seed >> 32));
    return hipGetLastError();
}

} // namespace va
