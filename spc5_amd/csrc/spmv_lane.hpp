// spmv_lane.hpp -- one wave computes y = alpha A x + beta y over one tile of a
// beta(r,VS) matrix with one block per lane ("lane-block" tile).
//
// Per batch of up to 64 blocks (one per lane):
//   1. the batch's headers, 64 (4 + r MB) contiguous bytes loaded ahead as
//      aligned 16-byte words, go to LDS and every lane takes its own from
//      there; popcounts and a wave scan give each block's value offset;
//   2. the batch's values are loaded as aligned 16-byte words and staged in
//      LDS as they lie;
//   3. every lane loads the x window of its block (VS adjacent entries, 16
//      bytes at a time; parts no block of the batch uses are skipped);
//   4. every lane walks the bits of its block in value order with the columns
//      and rows as compile-time indices: one LDS read of the next value and
//      one fused multiply-add into the row's register sum per position;
//   5. the lanes of one block-row are neighbours: their r sums are added by a
//      segmented DPP sum inside 16-lane rows and the last lane of every run
//      adds them to the tile's row sums in LDS.
// A step costs a fixed number of instructions per block position, not per
// value, and no LDS traffic for columns, rows or products: about a third of the
// vector instructions of the value-order tile, which is what bounds float and
// bfloat16 products (27-point stencil 128^3, bfloat16 beta(2,8): 100 -> 52 us,
// float beta(2,16): 101 -> 66 us, double beta(2,8): 121 -> 108 us, 4.9 TB/s of
// algorithmic bytes).  It asks for more lines of x per request, so matrices
// with scattered blocks stay in value order (lane_block_wins in spmv.hip).
//
// Every vector memory request of a batch is issued before the first wait on
// one, x before values before the next batch's headers, so that the header
// request stays in flight across the batch.
#pragma once

#include "spc5_mat.hpp"

namespace spc5 {

// Waves per SIMD each kernel is compiled for: 8 with a 32-byte x window, 6
// with a 64-byte one or 8 rows (the most without spills).
constexpr int lane_waves_per_eu(int r, int vs, int xbytes) {
    return r == 8 || vs * xbytes > 32 ? 6 : 8;
}

// The x window of a block in registers: at most 64 bytes (not double x with
// 16-column blocks, which runs the value-order tile).
constexpr bool lane_block_fits(int vs, int xbytes) { return vs * xbytes <= 64; }

// LDS bytes of staged values per batch.  They bound the values, and so the blocks
// a batch takes; more of them cost registers and waves.  Double beta(4,8) and
// float beta(8,16), whose blocks hold up to 32 and 128 values, have more levels
// and take the lowest that holds 64 of the matrix's mean blocks, or the highest
// (lane_level in spmv.hip); past 5 KiB float leaves fewer than 5 waves a SIMD.  Stage of 4 / 5 / 6 / 8 KiB, double beta(4,8): banded 60,000 rows,
// half-width 128, 9.9 values a block 18.3 / 15.8 / 14.6 / 15.4 us, 96 banded
// matrices in one launch 621 / 571 / 588 / 611, stencil 64^3, 11.9 values a block
// 20.9 / 20.7 / 16.9 / 17.6, Laplacian 1000^2, 6.7 values a block 17.8 / 18.6 /
// 20.1 / 21.0.  3 / 4 / 6 / 8 KiB, float beta(8,16): banded 250,000 rows, 37 values
// a block 42 / 36 / 30 / 27, stencil 128^3, 24 values a block 145 / 129 / 128 / 131,
// Laplacian, 13 values a block 27.6 / 28.1 / 29.2 / 31.4.  All others lose with
// more (float beta(2,16) banded 9.7 / 10.4 / 10.6 / 11.5).
constexpr int lane_levels(int vbytes, int r, int vs) {
    return vbytes == 8 && r == 4 ? 3 : (vbytes == 4 && vs == 16 && r == 8 ? 2 : 1);
}
__host__ __device__ constexpr int lane_stage_bytes(int vbytes, int r, int vs, int level) {
    if (vbytes == 8) return r == 4 ? 4096 + 1024 * level : 4096;
    return vs == 16 && vbytes == 4 && r == 8 ? 3072 + 2048 * level : 3072;
}

// STAGE: the staged bytes at most (a tile's `stage` may be less).
template <class V, class ACC, int R, int MB, int STAGE>
struct LaneSmem {
    static constexpr int kHeader = 4 + R * MB;
    static constexpr int kHdrWords = (15 + 64 * kHeader + 15) / 16;  // 16-byte words over 64 headers
    alignas(16) unsigned char val[STAGE];
    alignas(16) unsigned hdr[4 * (kHdrWords + 1)];  // + 1: a header's last dword pair may be read past its end
    ACC acc[tile_rows(R)];
    int mark[64];
};

// The lane's header as whole dwords (first column, then the masks), from the
// staged header bytes at byte offset `o`.
template <int H>
__device__ __forceinline__ void header_from_lds(const unsigned* w, int o, unsigned* out) {
    constexpr int NO = (H + 3) / 4;
    unsigned in[NO + 1];
    const unsigned* p = w + (o >> 2);
#pragma unroll
    for (int i = 0; i <= NO; ++i) in[i] = p[i];
#pragma unroll
    for (int i = 0; i < NO; ++i) out[i] = __builtin_amdgcn_alignbyte(in[i + 1], in[i], (unsigned)o & 3u);
}

// Value of LDS byte offset `o` in the accumulation type.
template <class V, class ACC>
__device__ __forceinline__ ACC staged_value(const unsigned char* base, int o) {
    if constexpr (sizeof(V) == 2) {
        return (ACC)bf16_to_f32(*reinterpret_cast<const unsigned short*>(base + o));
    } else {
        return (ACC)*reinterpret_cast<const V*>(base + o);
    }
}

// s_waitcnt operand: no vector memory load outstanding, other counters free.
constexpr int kWaitVm0 = 0x0f70;

template <class V, class X, class ACC, int R, int VS, int MB, int STAGE>
__device__ __forceinline__ void spmv_lane_tile(LaneSmem<V, ACC, R, MB, STAGE>& sm, int stage,
                                               const int* __restrict__ bptr,
                                               const unsigned char* __restrict__ hdr, const V* __restrict__ val,
                                               const X* __restrict__ x, X* __restrict__ y, int4 first, int4 last,
                                               int64_t nrows, int64_t ncols, const Epilogue& ep) {
    constexpr int H = 4 + R * MB;
    constexpr int NMW = (R * VS + 31) / 32;                 // mask dwords
    constexpr int PER = 16 / (int)sizeof(V);                // values per 16-byte word
    constexpr int KV = STAGE / 1024;                        // 16-byte words of values per lane
    const int cap = stage / (int)sizeof(V);                 // staged values
    constexpr int KH = LaneSmem<V, ACC, R, MB, STAGE>::kHdrWords > 64 ? 2 : 1;
    constexpr int XC = 16 / (int)sizeof(X);                 // columns per 16-byte x load
    constexpr int NQ = VS / XC;                             // x loads per window
    using U4 = unsigned int __attribute__((ext_vector_type(4)));
    const int lane = lane_id();
    const int br0 = __builtin_amdgcn_readfirstlane(first.x), br1 = __builtin_amdgcn_readfirstlane(last.x);
    const int b0 = __builtin_amdgcn_readfirstlane(first.y), b1 = __builtin_amdgcn_readfirstlane(last.y);
    int v = __builtin_amdgcn_readfirstlane(first.z);
    const int vend = __builtin_amdgcn_readfirstlane(last.z);
    const int nbr = br1 - br0;  // at most 64 (tile_rows)
    const int64_t row0 = (int64_t)br0 * R;
    const int64_t rows_left = nrows - row0;
    const int nrow_t = (int)((int64_t)nbr * R < rows_left ? (int64_t)nbr * R : rows_left);

    int b = v == vend ? b1 : b0;  // no values: x is never read
    // Headers of blocks [j, j + 64) as aligned 16-byte words: one request per
    // lane instead of two unaligned ones, and a word that holds a wanted byte
    // lies in the same page as that byte.
    U4 hw[KH];
    auto load_headers = [&](int j) {
        const int n = b1 - j < 64 ? b1 - j : 64;
        const unsigned char* a = hdr + (uint64_t)(unsigned)j * H;
        const int o = (int)(reinterpret_cast<uintptr_t>(a) & 15);
        const int words = (o + n * H + 15) >> 4;
#pragma unroll
        for (int k = 0; k < KH; ++k) {
            const unsigned i = lane + 64 * k < words ? lane + 64 * k : words - 1;
            hw[k] = *reinterpret_cast<const U4*>(a - o + 16u * i);
        }
    };
    if (b < b1) load_headers(b);

    // Block-row pointers of the tile, one block-row per lane.
    const int at = bptr[br0 + (lane < nbr ? lane : nbr)], end = bptr[br0 + (lane + 1 < nbr ? lane + 1 : nbr)];
    const int s0 = at - b0;
    const bool filled = end > at;  // the block-row has blocks
    // y of the tile's rows, requested now, used at the end
    constexpr int KY = tile_rows(R) / 64;
    X yv[KY] = {};
    if (ep.beta != 0.0) {
#pragma unroll
        for (int k = 0; k < KY; ++k) {
            const int i = lane + 64 * k < nrow_t ? lane + 64 * k : nrow_t - 1;
            yv[k] = y[row0 + i];
        }
    }
    for (int i = lane; i < nbr * R; i += 64) sm.acc[i] = (ACC)0;

    int prev = 0;  // block-row of the last block so far
    const unsigned xlast = (unsigned)(ncols - XC) * (unsigned)sizeof(X);  // byte offset of x's last XC entries
    while (b < b1) {
        // the headers asked for one batch ago (and nothing else) are outstanding
        __builtin_amdgcn_s_waitcnt(kWaitVm0);
        const int n = b1 - b < 64 ? b1 - b : 64;
        const int hoff = (int)((reinterpret_cast<uintptr_t>(hdr) + (uint64_t)(unsigned)b * H) & 15);
#pragma unroll
        for (int k = 0; k < KH; ++k)
            if (lane + 64 * k < LaneSmem<V, ACC, R, MB, STAGE>::kHdrWords)
                *reinterpret_cast<U4*>(&sm.hdr[4 * (lane + 64 * k)]) = hw[k];
        sm.mark[lane] = 0;
        wave_sync();
        unsigned hd[(H + 3) / 4];
        header_from_lds<H>(sm.hdr, hoff + (lane < n ? lane : 0) * H, hd);
        unsigned m[NMW];
        int cnt = 0;
#pragma unroll
        for (int k = 0; k < NMW; ++k) {
            unsigned w = hd[1 + k];
            if constexpr (R * MB == 1) w &= 0xffu;
            if constexpr (R * MB == 2) w &= 0xffffu;
            m[k] = lane < n ? w : 0u;
            cnt += __popc(m[k]);
        }
        const int incl = wave_incl_scan(cnt);
        // 16-byte words of values from the one that holds value v
        const V* va = val + (unsigned)v;
        const int shift = (int)((reinterpret_cast<uintptr_t>(va) & 15) / sizeof(V));
        const int fit = __popcll(ballot64(incl <= cap - shift));
        const int ntake = fit < n ? fit : n;
        const int total = __builtin_amdgcn_readlane(incl, ntake - 1);
        const int words = (shift + total + PER - 1) / PER;
        const int bn = b + ntake;
        // Columns used by the lane's block and the x window from its first
        // column, one 16-byte load per XC columns the block uses.  A part that
        // would reach past x is read from x's last XC entries instead and
        // moved down afterwards.
        const bool taken = lane < ntake;
#pragma unroll
        for (int k = 0; k < NMW; ++k) m[k] = taken ? m[k] : 0u;
        unsigned cm = 0;
#pragma unroll
        for (int t = 0; t < R; ++t) cm |= (m[t * VS / 32] >> (t * VS % 32)) & ((1u << VS) - 1u);
        X xw[VS];
        int used[NQ];  // lanes that use part q
        const unsigned xoff = hd[0] * (unsigned)sizeof(X);
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const bool need = (cm & (((1u << XC) - 1u) << (q * XC))) != 0;
            used[q] = __popcll(ballot64(need));
            if (need) {
                const unsigned o = xoff + 16u * q < xlast ? xoff + 16u * q : xlast;
                __builtin_memcpy(&xw[q * XC], reinterpret_cast<const char*>(x) + o, 16);
            }
        }
        const char* vp = reinterpret_cast<const char*>(va - shift);
        U4 vw[KV];
#pragma unroll
        for (int k = 0; k < KV; ++k) {
            if (64 * k < words) {
                const unsigned i = lane + 64 * k < words ? lane + 64 * k : words - 1;
                vw[k] = __builtin_nontemporal_load(reinterpret_cast<const U4*>(vp + 16u * i));
            }
        }
        load_headers(bn < b1 ? bn : b1 - 1);  // always, so that no wait below covers it
        if (ballot64(cm != 0 && xoff + 16u * (NQ - 1) > xlast)) {
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const unsigned over = xoff + 16u * q > xlast ? (xoff + 16u * q - xlast) / (unsigned)sizeof(X) : 0u;
#pragma unroll
                for (int c = 0; c < XC; ++c) {
#pragma unroll
                    for (int e = c + 1; e < XC; ++e)
                        if (over == (unsigned)(e - c)) xw[q * XC + c] = xw[q * XC + e];
                }
            }
        }
        // block-row of every block: the filled block-rows mark their first block
        const int d = s0 - (b - b0);
        if (filled && (unsigned)d < (unsigned)ntake) sm.mark[d] = lane + 1;
        wave_sync();
        const int mk = sm.mark[lane];
        const int top = wave_incl_max(mk);
        const int br = top > 0 ? top - 1 : prev;
        const unsigned long long starts = ballot64(mk != 0) | 1ull;
        prev = __builtin_amdgcn_readlane(br, ntake - 1);
        // values to LDS
#pragma unroll
        for (int k = 0; k < KV; ++k)
            if (64 * k < words) reinterpret_cast<U4*>(sm.val)[lane + 64 * k] = vw[k];
        wave_sync();
        // products of the lane's block
        ACC s[R];
        int o = taken ? (shift + incl - cnt) * (int)sizeof(V) : 0;
#pragma unroll
        for (int t = 0; t < R; ++t) {
            s[t] = (ACC)0;
            const unsigned mt = m[t * VS / 32];
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                if (!used[q]) continue;
                unsigned on[XC];
                ACC a[XC];
#pragma unroll
                for (int c = 0; c < XC; ++c) {
                    on[c] = __builtin_amdgcn_ubfe(mt, t * VS % 32 + q * XC + c, 1);
                    a[c] = staged_value<V, ACC>(sm.val, o);
                    o += (int)(on[c] * (unsigned)sizeof(V));
                }
#pragma unroll
                for (int c = 0; c < XC; ++c) {
                    const ACC f = fma(a[c], (ACC)xw[q * XC + c], s[t]);
                    s[t] = on[c] ? f : s[t];
                }
            }
        }
        // sums of neighbouring lanes on one block-row, inside 16-lane rows
        const int lr = lane & 15;
        const unsigned rowst = (unsigned)(starts >> (lane & 48)) & 0xffffu;       // starts in this 16-lane row
        const unsigned upto = (rowst | 1u) & ((2u << lr) - 1u);
        const int dist = lr - (31 - __builtin_clz(upto));                         // lanes back to the run's first
        const bool tail = taken && (lr == 15 || lane == ntake - 1 || ((rowst >> (lr + 1)) & 1u));
#define SPC5_LANE_STEP(CTRL, N)                              \
    if (ballot64(dist >= N)) {                               \
        const bool add = dist >= N;                          \
        _Pragma("unroll") for (int t = 0; t < R; ++t) {      \
            const ACC u = dpp_val<CTRL>(s[t]);               \
            s[t] += add ? u : (ACC)0;                        \
        }                                                    \
    }
        SPC5_LANE_STEP(kDppRowShr1, 1)
        SPC5_LANE_STEP(kDppRowShr2, 2)
        SPC5_LANE_STEP(kDppRowShr4, 4)
        SPC5_LANE_STEP(kDppRowShr8, 8)
#undef SPC5_LANE_STEP
        if (tail) {
#pragma unroll
            for (int t = 0; t < R; ++t) atomicAdd(&sm.acc[br * R + t], s[t]);
        }
        v += total;
        b = bn;
        wave_sync();
    }
    wave_sync();
    // y = alpha * (A x) + beta * y; see spmv_tile.hpp for the dot partial
    const ACC alpha = (ACC)ep.alpha, beta = (ACC)ep.beta;
    const X* __restrict__ dv = reinterpret_cast<const X*>(ep.dv);
    double part = 0.0;
#pragma unroll
    for (int k = 0; k < KY; ++k) {
        const int i = lane + 64 * k;
        if (i < nrow_t) {
            const ACC ax = sm.acc[i];
            const X yn = ep.beta == 0.0 ? (X)(alpha * ax) : (X)(alpha * ax + beta * (ACC)yv[k]);
            y[row0 + i] = yn;
            if (dv) part += (double)dv[row0 + i] * (double)yn;
        }
    }
    if (ep.dot) {
        part = wave_sum_f64(part);
        if (lane == 0) ep.dot[0] = part;
    }
}

}  // namespace spc5
