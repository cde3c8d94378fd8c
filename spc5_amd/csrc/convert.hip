// convert.hip -- CSR -> beta(r,VS) on the GPU, byte-identical to the
// reference converter (src/spc5.hpp:165-228 and 455-488).
//
// The reference walks each block-row with one cursor per row: a block starts
// at the smallest unconsumed column of the block-row and takes, row by row,
// every entry with column < start+VS.  Block-rows are independent, so the
// GPU gives every 64 rows to one wave, one lane per row, the r lanes of a
// block-row walking together (see "Groups" below), in two passes:
//   count : blocks per block-row -> exclusive scan -> block-row pointers
//           (the reference's rowsSize after conversion) and the block count;
//   fill  : the same walk again, writing each block's packed header at
//           (pointer + k) * (4 + r*MB) bytes and its values at the block-row's
//           value offset, which is the CSR row pointer of its first row
//           (conversion only permutes values inside a block-row).
#include "spc5_common.hpp"

#include <mutex>

#include <climits>

namespace spc5 {

namespace {

// Groups: one wave converts kGroupRows = 64 consecutive rows, one lane per
// row; the r lanes of a block-row form a lane group.  The group's column
// indices are staged in LDS with coalesced loads, the first entry of every row
// replaced by a value larger than any column (its lane keeps the column), so
// that a window of a row always ends at the row's end.  Per block
// (walk_staged):
//   * every lane reads the next VS entries of its row; the first is its head,
//     and the block starts at the minimum of the r heads (DPP);
//   * one median per entry clamps the window to [.., start + VS) and carries
//     the clamp past the first entry outside, and one shift-or per entry
//     collects the bits modulo 32; a rotation by the start gives the row mask,
//     its popcount the lane's values in the block.
// The fill pass stores each header as it is made and leaves, at the stage
// position of the lane's first value in the block, the distance from source to
// destination; a last pass reads the values in CSR order and every lane takes
// the distance of the last such position at or before it.  (With r = 1 the
// values keep their order.)
//
// What bounds it: the chain of one LDS round trip and about 30 instructions per
// block, as long as the longest block-row of the wave, with the waves per CU
// that the staged columns leave room for; then HBM in the fill.  Clustered
// matrix of 1 M rows, double beta(4,8): count 200 -> 104 us, fill 476 -> 200 us
// (before: a chain of compares and selects per window entry, VS LDS writes of
// destinations per lane and block, and 96 registers of prefetched values).
//
// A group too large for the stage reads its columns from global memory and
// writes directly (walk_group).
//
// The stage is dynamic LDS sized at launch from the matrix's mean values per
// group (half as much again as the mean, at least 256 more): a small stage
// keeps many waves resident per CU.
constexpr int kGroupRows = 64;
constexpr int kPrefetch = 32;             // words per lane loaded at once: 2048 per group
constexpr int kMaxStageValues = 8192;     // 32 KiB of staged columns
constexpr int kStagePad = 32;             // words after the staged columns read by the walk's windows

template <int R>
constexpr int group_blockrows() { return kGroupRows / R; }

int64_t round_up64(int64_t v) { return (v + 63) / 64 * 64; }

// Staged values per group: the mean plus half of it (at least 256 more).
int stage_values(int64_t nnz, int64_t ngroups) {
    const int64_t avg = ngroups > 0 ? (nnz + ngroups - 1) / ngroups : 0;
    int64_t s = round_up64(avg + (avg / 2 > 256 ? avg / 2 : 256));
    if (s < 512) s = 512;
    return (int)(s < kMaxStageValues ? s : kMaxStageValues);
}

// Lane-group collectives over R = 1, 2, 4 or 8 consecutive lanes, as DPP
// moves inside 16-lane rows (no LDS round trip): quad_perm [1,0,3,2] and
// [2,3,0,1] exchange within pairs and quads, row_half_mirror (lane i of an
// 8-lane half-row reads lane 7 - i) joins the two quads of an 8-lane group
// once each quad holds its own result, and row_shr:n shifts for the scan.
// Every lane of a group is active whenever one of them calls these.
constexpr int kDppQuadXor1 = 0xB1;
constexpr int kDppQuadXor2 = 0x4E;
constexpr int kDppRowHalfMirror = 0x141;

template <int CTRL>
__device__ __forceinline__ int dpp_i32(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, false);
}

template <int R>
__device__ __forceinline__ int group_min(int v) {
    if constexpr (R >= 2) v = min(v, dpp_i32<kDppQuadXor1>(v));
    if constexpr (R >= 4) v = min(v, dpp_i32<kDppQuadXor2>(v));
    if constexpr (R >= 8) v = min(v, dpp_i32<kDppRowHalfMirror>(v));
    return v;
}
template <int R>
__device__ __forceinline__ unsigned group_min(unsigned v) {
    if constexpr (R >= 2) v = min(v, (unsigned)dpp_i32<kDppQuadXor1>((int)v));
    if constexpr (R >= 4) v = min(v, (unsigned)dpp_i32<kDppQuadXor2>((int)v));
    if constexpr (R >= 8) v = min(v, (unsigned)dpp_i32<kDppRowHalfMirror>((int)v));
    return v;
}
template <int R>
__device__ __forceinline__ int group_sum(int v) {
    if constexpr (R >= 2) v += dpp_i32<kDppQuadXor1>(v);
    if constexpr (R >= 4) v += dpp_i32<kDppQuadXor2>(v);
    if constexpr (R >= 8) v += dpp_i32<kDppRowHalfMirror>(v);
    return v;
}
// Exclusive prefix sum over the lanes of a group (lane t: sum over t' < t).
template <int R>
__device__ __forceinline__ int group_excl_scan(int v, int t) {
    int incl = v;
    if constexpr (R >= 2) {
        const int o = dpp_i32<kDppRowShr1>(incl);
        if (t >= 1) incl += o;
    }
    if constexpr (R >= 4) {
        const int o = dpp_i32<kDppRowShr2>(incl);
        if (t >= 2) incl += o;
    }
    if constexpr (R >= 8) {
        const int o = dpp_i32<kDppRowShr4>(incl);
        if (t >= 4) incl += o;
    }
    return incl - v;
}

// Walks the block-rows of a group over global columns; for each block of a
// lane's block-row calls on_block(k, start, t, first, n, mask, src0) on every
// lane of the group: k is the block's index in its block-row, t the lane's row
// in the block, first the value position (block order) of the lane's first
// value in the block, n its count and mask its VS-bit row mask; the lane's
// values are at source positions [src0, src0 + n).  With CHECK, returns whether
// a lane saw columns that break the format's precondition (non-negative,
// strictly increasing); without, the caller has checked them and it returns
// false.
//
// Per block a lane reads the window of its next VS + 1 columns at once (clamped
// to the row): its values in the block are the window's leading run below
// start + VS (at most VS, the columns being strictly increasing), the entry
// after them is the next head, and adjacent entries check the precondition.
template <int R, int VS, bool CHECK, class F>
__device__ __forceinline__ bool walk_group(int rb, int re, const int* __restrict__ col, F on_block) {
    const int lane = threadIdx.x;
    const int t = lane % R;
    const int end = re;
    int cur = rb;
    int head = cur < end ? col[cur] : INT_MAX;  // INT_MAX once the row is consumed
    bool bad = CHECK && head < 0;
    // the block-row's first value: the row pointer of its row 0
    int vbase = __shfl(rb, lane - t, 64);
    int k = 0;
    for (;;) {
        const int start = group_min<R>(head);
        if (!ballot64(start != INT_MAX)) break;  // every block-row of the wave is done
        if (start != INT_MAX) {
            int w[VS + 1];
            const int last = end - 1 > cur ? end - 1 : cur;
#pragma unroll
            for (int j = 0; j <= VS; ++j) w[j] = cur < end ? col[cur + j < last ? cur + j : last] : 0;
            unsigned mask = 0;
            int n = 0;
            bool alive = true;
#pragma unroll
            for (int j = 0; j < VS; ++j) {
                const unsigned d = (unsigned)w[j] - (unsigned)start;
                alive = alive && cur + j < end && d < (unsigned)VS;
                mask |= alive ? 1u << (d & 31u) : 0u;
                n += alive ? 1 : 0;
            }
            if constexpr (CHECK) {
#pragma unroll
                for (int j = 1; j <= VS; ++j) bad |= cur + j < end && w[j] <= w[j - 1];
            }
            int next = w[0];
#pragma unroll
            for (int j = 1; j <= VS; ++j) next = n == j ? w[j] : next;
            const int before = group_excl_scan<R>(n, t);
            on_block(k, start, t, vbase + before, n, mask, cur);
            vbase += group_sum<R>(n);
            cur += n;
            head = cur < end ? next : INT_MAX;
            ++k;
        }
    }
    return bad;
}

// Raw buffer loads of one word type (a read past the resource's range
// returns 0 and touches no memory).
template <class T>
struct RawWord;
template <>
struct RawWord<int> {
    __device__ __forceinline__ static int get(__amdgpu_buffer_rsrc_t r, int off) {
        return (int)__builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0);
    }
};
template <>
struct RawWord<unsigned int> {
    __device__ __forceinline__ static unsigned int get(__amdgpu_buffer_rsrc_t r, int off) {
        return __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0);
    }
};
template <>
struct RawWord<unsigned long long> {
    __device__ __forceinline__ static unsigned long long get(__amdgpu_buffer_rsrc_t r, int off) {
        return __builtin_bit_cast(unsigned long long, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
    }
};
template <>
struct RawWord<unsigned short> {
    __device__ __forceinline__ static unsigned short get(__amdgpu_buffer_rsrc_t r, int off) {
        return __builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0);
    }
};

// v[u] = src[lane + 64 u] for u < kPrefetch (0 past n), through a buffer
// resource of n words: every load unconditional and one lane offset for all,
// so all are in flight at once at little register cost.
template <class T>
__device__ __forceinline__ void prefetch_words(const T* __restrict__ src, int n, int lane, T (&v)[kPrefetch]) {
    const __amdgpu_buffer_rsrc_t r =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(src), (short)0, n * (int)sizeof(T), kRawBufferFlags);
#pragma unroll
    for (int u = 0; u < kPrefetch; ++u) v[u] = RawWord<T>::get(r, (lane + 64 * u) * (int)sizeof(T));
}

// Stage entries that are no column: the first of every row, and (from
// kMovedBase) the first value of a row's part of a block, once the walk has
// left the distance to its destination there.  Both exceed every block's end.
constexpr unsigned kRowStart = 0xffffffffu;
constexpr unsigned kMovedBase = 0xc0000000u;
constexpr int kMovedZero = 1 << 16;  // encodes distance 0

// Stages n column indices in LDS, 64 kPrefetch at a time; true where a lane
// saw a negative one.
__device__ __forceinline__ bool stage_columns(const int* __restrict__ src, unsigned* dst, int n, int lane) {
    bool bad = false;
    for (int i0 = 0; i0 < n; i0 += 64 * kPrefetch) {
        int v[kPrefetch];
        prefetch_words(src + i0, n - i0, lane, v);
#pragma unroll
        for (int u = 0; u < kPrefetch; ++u) {
            const int i = i0 + lane + 64 * u;
            if (64 * u < n - i0) {
                if (i < n) dst[i] = (unsigned)v[u];
                bad |= v[u] < 0;
            }
        }
    }
    if (lane == 0) dst[n] = kRowStart;
    wave_sync();
    return bad;
}

// The row starts marked in the stage; returns the column of the lane's first
// entry (kRowStart for an empty row).  CHECK: *bad is set where the columns of
// a row do not strictly increase.
template <bool CHECK>
__device__ __forceinline__ unsigned mark_rows(unsigned* scol, int cur, int end, int n, int lane, bool* bad) {
    const unsigned first = cur < end ? scol[cur] : kRowStart;
    if (CHECK && cur + 1 < end) *bad |= scol[cur + 1] <= first;
    wave_sync();
    if (cur < end) scol[cur] = kRowStart;
    wave_sync();
    if constexpr (CHECK) {
#pragma unroll 4
        for (int i = lane; i < n; i += 64) {
            const unsigned c0 = scol[i], c1 = scol[i + 1];
            *bad |= c0 != kRowStart && c1 <= c0;
        }
    }
    return first;
}

// Walks the block-rows of a staged group: [cur, end) are the lane's stage
// positions and `first` its first column.  Calls on_block(k, more, start, n,
// mask, src) on every lane; `more` where the block-row has a k-th block: n
// values from stage position src on, with the row mask `mask`.  MOVED: on_block leaves moved marks
// in the stage.  At most nv steps, whatever the columns.
template <int R, int VS, bool MOVED, class F>
__device__ __forceinline__ void walk_staged(const unsigned* scol, int cur, unsigned first, int nv, F on_block) {
    const int begin = cur;
    const int steps = __builtin_amdgcn_readfirstlane(nv);
    for (int k = 0; k < steps; ++k) {
        unsigned w[VS];
#pragma unroll
        for (int j = 0; j < VS; ++j) w[j] = scol[cur + j];
        // the whole window in one LDS round trip (the reads would otherwise
        // sink below the start they do not need)
#pragma unroll
        for (int j = 0; j < VS; ++j) asm volatile("" : "+v"(w[j]));
        // past the row's end: the mark at the start of the next row
        const unsigned next = MOVED && w[0] >= kMovedBase ? kRowStart : w[0];
        const unsigned head = cur == begin ? first : next;
        const unsigned start = group_min<R>(head);
        const bool more = start != kRowStart;
        if (!ballot64(more)) break;
        // entries clamped to the block's end; the first one outside and all
        // that follow it count as the end
        const unsigned lim = start + VS;
        unsigned q = head < lim ? head : lim;
        unsigned bits = 1u << (q & 31u);
#pragma unroll
        for (int j = 1; j < VS; ++j) {
            asm("v_med3_u32 %0, %1, %2, %3" : "=v"(q) : "v"(q), "v"(w[j]), "v"(lim));
            bits |= 1u << (q & 31u);
        }
        const unsigned mask = __builtin_amdgcn_alignbit(bits, bits, start & 31u) & ((1u << VS) - 1u);
        const int n = more ? __popc(mask) : 0;
        on_block(k, more, start, n, mask, cur);
        cur += n;
    }
}

// A group's rows, one per lane: [rb, re) are the lane's values (rows past the
// matrix are empty at its end), v0 the group's first value, nv its count.
struct GroupRows {
    int rb, re, v0, nv;
};
__device__ __forceinline__ GroupRows group_rows(const int* __restrict__ rowptr, int64_t row0, int64_t nrows,
                                                int lane) {
    const int64_t row = row0 + lane;
    GroupRows g;
    g.rb = rowptr[row < nrows ? row : nrows];
    g.re = rowptr[row + 1 < nrows ? row + 1 : nrows];
    g.v0 = __shfl(g.rb, 0, 64);
    g.nv = __shfl(g.re, 63, 64) - g.v0;
    return g;
}

// The next run of a group's rows, from row `lo` on, that is converted at once:
// all of them, or the largest aligned half, quarter, ... whose values fit the
// stage of sv (down to one block-row, which may not fit).  Lanes of other rows
// hold empty ones.  A group read from global memory instead takes two memory
// round trips per block, and a few such groups outlast all others: on the
// clustered matrix one group in a thousand exceeds 1.5 times the mean.
struct RowRun {
    int rows;        // rows of the run
    int rb, re;      // the lane's values
    int v0, nv;      // the run's
};
template <int R>
__device__ __forceinline__ RowRun row_run(const GroupRows& g, int lo, int sv, int lane) {
    RowRun p;
    p.rows = lo == 0 ? kGroupRows : lo & -lo;
    p.v0 = __builtin_amdgcn_readlane(g.rb, lo);
    for (;;) {
        p.nv = __builtin_amdgcn_readlane(g.re, lo + p.rows - 1) - p.v0;
        if (p.nv <= sv || p.rows == R) break;
        p.rows >>= 1;
    }
    const bool mine = lane >= lo && lane < lo + p.rows;
    p.rb = mine ? g.rb : p.v0;
    p.re = mine ? g.re : p.v0;
    return p;
}

// Blocks per block-row (the count pass); cnt_out[nbr] = 0.  A row pointer that
// does not start at 0, decreases or passes nnz sets err[0], a violation of the
// column precondition err[1]; the fill pass is then never run, and a wave whose
// row pointers fail reads no column.  Dynamic LDS: sv staged column indices and
// kStagePad words of pad.
template <int R, int VS>
__global__ __launch_bounds__(64) void k_convert_count(int64_t nrows, int64_t nbr, const int* __restrict__ rowptr,
                                                      const int* __restrict__ col, int64_t nnz,
                                                      int* __restrict__ cnt_out, int* __restrict__ err, int sv) {
    constexpr int BR = group_blockrows<R>();
    extern __shared__ __align__(16) unsigned char smem[];
    unsigned* scol = reinterpret_cast<unsigned*>(smem);
    const int lane = threadIdx.x;
    const int64_t br0 = (int64_t)blockIdx.x * BR;
    const GroupRows g = group_rows(rowptr, br0 * R, nrows, lane);
    if (br0 + BR >= nbr && lane == 0) cnt_out[nbr] = 0;
    const bool broken = g.rb < 0 || g.re < g.rb || (int64_t)g.re > nnz || (br0 == 0 && lane == 0 && g.rb != 0);
    const bool any_broken = ballot64(broken) != 0;
    if (any_broken && lane == 0) atomicOr(err, 1);
    int nb = 0;
    bool bad = false;
    for (int lo = any_broken ? kGroupRows : 0; lo < kGroupRows;) {
        const RowRun p = row_run<R>(g, lo, sv, lane);
        lo += p.rows;
        if (p.nv == 0) continue;
        if (p.nv <= sv) {
            bad |= stage_columns(col + p.v0, scol, p.nv, lane);
            const unsigned first = mark_rows<true>(scol, p.rb - p.v0, p.re - p.v0, p.nv, lane, &bad);
            if (!ballot64(bad))
                walk_staged<R, VS, false>(scol, p.rb - p.v0, first, p.nv,
                                          [&](int, bool more, unsigned, int, unsigned, int) { nb += more ? 1 : 0; });
            wave_sync();
        } else {
            bad |= walk_group<R, VS, true>(p.rb, p.re, col, [&](int, int, int, int, int, unsigned, int) { ++nb; });
        }
    }
    const int64_t br = br0 + lane / R;
    if (lane % R == 0 && br < nbr) cnt_out[br] = nb;
    if (bad) atomicOr(err + 1, 1);
}

// Header of one block, the lanes of its block-row together: lane t = 0 writes
// the first column, and the r masks are gathered into whole dwords by DPP.
template <int R, int VS, int MB>
__device__ __forceinline__ void store_header(unsigned char* h, unsigned start, unsigned mask, int t) {
    constexpr int LPD = 4 / MB;  // lanes per dword of masks
    unsigned m = mask << (8 * MB * (t % LPD));
    if constexpr (R >= 2) m |= (unsigned)dpp_i32<kDppQuadXor1>((int)m);
    if constexpr (R >= 4 && LPD == 4) m |= (unsigned)dpp_i32<kDppQuadXor2>((int)m);
    if constexpr (R * MB <= 4) {
        if (t == 0) {
            if constexpr (R * MB == 4) {
                const uint2 both = make_uint2(start, m);
                __builtin_memcpy(h, &both, 8);
            } else {
                __builtin_memcpy(h, &start, 4);
                __builtin_memcpy(h + 4, &m, R * MB);
            }
        }
    } else {
        if (t == 0) __builtin_memcpy(h, &start, 4);
        if (t % LPD == 0) __builtin_memcpy(h + 4 + t * MB, &m, 4);
    }
}

// Headers and values of the groups' blocks.  Dynamic LDS as the count pass.
template <class W, int R, int VS, int MB>
__global__ __launch_bounds__(64) void k_convert_fill(int64_t nrows, int64_t nbr, const int* __restrict__ rowptr,
                                                     const int* __restrict__ col, const W* __restrict__ vin,
                                                     const int* __restrict__ bptr, int64_t nblocks,
                                                     unsigned char* __restrict__ hdr, W* __restrict__ vout, int sv) {
    constexpr int BR = group_blockrows<R>();
    constexpr int H = 4 + R * MB;
    constexpr int U = 8;  // values per lane in flight
    extern __shared__ __align__(16) unsigned char smem[];
    unsigned* scol = reinterpret_cast<unsigned*>(smem);
    const int lane = threadIdx.x;
    const int t = lane % R;
    const int64_t br0 = (int64_t)blockIdx.x * BR;
    const int64_t br = br0 + lane / R;
    // row pointers and block-row pointers, loaded together
    const GroupRows g = group_rows(rowptr, br0 * R, nrows, lane);
    const int b_lo = bptr[br < nbr ? br : nbr];
    const int b_hi = bptr[br + 1 < nbr ? br + 1 : nbr];
    // blocks of the lane's block-row: never written past, whatever the pointers
    const int64_t b_end = b_hi < nblocks ? b_hi : nblocks;
    const int nblk = br < nbr && b_end > b_lo ? (int)(b_end - b_lo) : 0;
    unsigned char* h = hdr + (int64_t)b_lo * H;
    for (int lo = 0; lo < kGroupRows;) {
        const RowRun p = row_run<R>(g, lo, sv, lane);
        lo += p.rows;
        const int v0 = p.v0, nv = p.nv;
        if (nv == 0) continue;
        if (nv > sv) {
            // too large for the stage: global columns, direct writes
            walk_group<R, VS, false>(p.rb, p.re, col, [&](int k, int start, int tt, int first, int n, unsigned mask,
                                                          int src0) {
                if (k >= nblk) return;
                store_header<R, VS, MB>(h + (int64_t)k * H, (unsigned)start, mask, tt);
                for (int j = 0; j < n; ++j) vout[first + j] = vin[src0 + j];
            });
            continue;
        }
        (void)stage_columns(col + v0, scol, nv, lane);
        bool unused = false;
        const unsigned first = mark_rows<false>(scol, p.rb - v0, p.re - v0, nv, lane, &unused);
        W v[U];
        auto load = [&](int i0) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int i = i0 + lane + 64 * u;
                v[u] = vin[v0 + (i < nv ? i : nv - 1)];
            }
        };
        load(0);  // in flight across the walk
        int at = __shfl(p.rb, lane - t, 64) - v0;  // destination of the block-row's next value
        walk_staged<R, VS, (R > 1)>(scol, p.rb - v0, first, nv, [&](int k, bool more, unsigned start, int n,
                                                                   unsigned mask, int src) {
            if (more && k < nblk) store_header<R, VS, MB>(h + (unsigned)(k * H), start, mask, t);
            if constexpr (R > 1) {
                const int to = at + group_excl_scan<R>(n, t);
                at += group_sum<R>(n);
                if (n > 0) scol[src] = kMovedBase + (unsigned)(to - src + kMovedZero);
            }
        });
        wave_sync();
        int carry = 0;  // distance of the last part begun before the chunk
        for (int i0 = 0; i0 < nv; i0 += 64 * U) {
            if (i0 > 0) load(i0);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (i0 + 64 * u >= nv) break;
                const int i = i0 + lane + 64 * u;
                int d = 0;
                if constexpr (R > 1) {
                    const unsigned e = i < nv ? scol[i] : 0u;
                    const unsigned long long starts = ballot64(e >= kMovedBase);
                    // the last part begun at or before this lane
                    const unsigned long long upto = starts & ((2ull << lane) - 1ull);
                    const int from = upto ? 63 - __builtin_clzll(upto) : 0;
                    const int mine = __builtin_amdgcn_ds_bpermute(from << 2, (int)(e - kMovedBase)) - kMovedZero;
                    d = upto ? mine : carry;
                    carry = __builtin_amdgcn_readlane(d, 63);
                }
                if (i < nv) vout[v0 + i + d] = v[u];
            }
        }
        wave_sync();
    }
}

template <int R, int VS>
void launch_count(int64_t nrows, int64_t nbr, const int* rowptr, const int* col, int* out, int* err, int64_t nnz,
                  hipStream_t s) {
    const int64_t groups = (nbr + group_blockrows<R>() - 1) / group_blockrows<R>();
    const int sv = stage_values(nnz, groups);
    const size_t shm = (size_t)(sv + kStagePad) * 4;
    hipLaunchKernelGGL((k_convert_count<R, VS>), dim3((unsigned)groups), dim3(64), shm, s, nrows, nbr,
                       rowptr, col, nnz, out, err, sv);
}

template <class W, int VS, int MB>
int launch_fill_r(int r, int64_t nrows, int64_t nbr, const int* rowptr, const int* col, const void* vin,
                  const int* bptr, int64_t nblocks, int64_t nnz, unsigned char* hdr, void* vout, hipStream_t s) {
    const W* vi = reinterpret_cast<const W*>(vin);
    W* vo = reinterpret_cast<W*>(vout);
#define SPC5_FILL_LAUNCH(R)                                                                                    \
    do {                                                                                                       \
        const int64_t groups = (nbr + group_blockrows<R>() - 1) / group_blockrows<R>();                        \
        const int sv = stage_values(nnz, groups);                                                              \
        const size_t shm = (size_t)(sv + kStagePad) * 4;                                                       \
        hipLaunchKernelGGL((k_convert_fill<W, R, VS, MB>), dim3((unsigned)groups), dim3(64), shm, s, nrows, nbr, \
                           rowptr, col, vi, bptr, nblocks, hdr, vo, sv);                                       \
    } while (0)
    switch (r) {
    case 1: SPC5_FILL_LAUNCH(1); break;
    case 2: SPC5_FILL_LAUNCH(2); break;
    case 4: SPC5_FILL_LAUNCH(4); break;
    case 8: SPC5_FILL_LAUNCH(8); break;
    default: set_error("r must be 1, 2, 4 or 8"); return SPC5_HIP_ERR_INVALID;
    }
#undef SPC5_FILL_LAUNCH
    SPC5_HIP_TRY(hipGetLastError());
    return SPC5_HIP_OK;
}

template <class W>
int launch_fill_w(int vs, int mb, int r, int64_t nrows, int64_t nbr, const int* rowptr, const int* col,
                  const void* vin, const int* bptr, int64_t nblocks, int64_t nnz, unsigned char* hdr, void* vout,
                  hipStream_t s) {
    if (vs == 8 && mb == 1)
        return launch_fill_r<W, 8, 1>(r, nrows, nbr, rowptr, col, vin, bptr, nblocks, nnz, hdr, vout, s);
    if (vs == 16 && mb == 2)
        return launch_fill_r<W, 16, 2>(r, nrows, nbr, rowptr, col, vin, bptr, nblocks, nnz, hdr, vout, s);
    set_error("(VS, mask bytes) must be (8, 1) or (16, 2)");
    return SPC5_HIP_ERR_INVALID;
}

// Scratch of one count pass: words[0] flags a bad row pointer, words[1]
// unsorted or negative columns, words[2] receives the block total; the scan
// of the block counts uses partials[0 .. partial_cap).
struct CountScratch {
    int* words = nullptr;
    int* partials = nullptr;
    int64_t partial_cap = 0;
};

// Fixed device scratch of spc5_hip_convert_count_noalloc, one copy per GPU
// (a file-scope __device__ array): kScratchWords flag/total words, then the
// scan partials.  Host code uses the address hipGetSymbolAddress returns on
// each device, never the array's name.
constexpr int kScratchInts = 16384;  // 64 KiB
constexpr int kScratchWords = 64;    // keeps the partials 256-byte aligned
constexpr int kMaxDevices = 64;
__device__ __align__(256) int scratch[kScratchInts];

std::mutex g_scratch_mu;
int* g_scratch_ptr[kMaxDevices] = {};

// Device address of the current device's copy of `scratch` (looked up once
// per device, with that device current).
int scratch_address(int** out) {
    int dev = -1;
    SPC5_HIP_TRY(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) {
        set_error("device index out of range for the fixed scratch table");
        return SPC5_HIP_ERR_INVALID;
    }
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_ptr[dev] == nullptr) {
        void* p = nullptr;
        SPC5_HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (p == nullptr) {
            set_error("hipGetSymbolAddress returned no address for the scratch array");
            return SPC5_HIP_ERR_HIP;
        }
        g_scratch_ptr[dev] = reinterpret_cast<int*>(p);
    }
    *out = g_scratch_ptr[dev];
    return SPC5_HIP_OK;
}

// Reads n flag/total words back (synchronises the stream).
int read_words(const int* d_words, int* h, int n, hipStream_t s) {
    SPC5_HIP_TRY(hipMemcpyAsync(h, d_words, sizeof(int) * (size_t)n, hipMemcpyDeviceToHost, s));
    SPC5_HIP_TRY(hipStreamSynchronize(s));
    return SPC5_HIP_OK;
}

// Count pass of every entry point: block count per block-row, exclusive scan
// into d_rowsSize_out[0..nbr], total into *nblocks.  nnz bounds the row
// pointers and sizes the stage.  Allocates nothing and waits once.
int convert_count_impl(int vs, int r, int64_t nrows, int64_t nnz, const int* d_rowptr, const int* d_colidx,
                       int* d_rowsSize_out, int64_t* nblocks, const CountScratch& ws, hipStream_t s) {
    *nblocks = 0;
    const int64_t nbr = (nrows + r - 1) / r;
    if (scan_partials_needed(nbr + 1) > ws.partial_cap) {
        set_error("too many block-rows for the scratch space (" + std::to_string(nbr) + " > " +
                  std::to_string(ws.partial_cap * 2048 - 1) + ")");
        return SPC5_HIP_ERR_INVALID;
    }
    // A matrix without entries may come without a column array (an empty
    // tensor's storage); the count pass then reads no column.
    SPC5_CHECK_ARG(nbr == 0 || d_colidx != nullptr || nnz == 0, "colidx is null");
    // flags and total start at zero: a fill kernel, not a memset node
    hipLaunchKernelGGL(k_fill_i32, dim3(1), dim3(64), 0, s, ws.words, (int64_t)3, 0);
    SPC5_HIP_TRY(hipGetLastError());
    if (nbr == 0) {
        hipLaunchKernelGGL(k_fill_i32, dim3(1), dim3(64), 0, s, d_rowsSize_out, (int64_t)1, 0);
        SPC5_HIP_TRY(hipGetLastError());
    }
    if (nbr > 0) {
        const int key = r * 100 + vs;
        switch (key) {
        case 108: launch_count<1, 8>(nrows, nbr, d_rowptr, d_colidx, d_rowsSize_out, ws.words, nnz, s); break;
        case 208: launch_count<2, 8>(nrows, nbr, d_rowptr, d_colidx, d_rowsSize_out, ws.words, nnz, s); break;
        case 408: launch_count<4, 8>(nrows, nbr, d_rowptr, d_colidx, d_rowsSize_out, ws.words, nnz, s); break;
        case 808: launch_count<8, 8>(nrows, nbr, d_rowptr, d_colidx, d_rowsSize_out, ws.words, nnz, s); break;
        case 116: launch_count<1, 16>(nrows, nbr, d_rowptr, d_colidx, d_rowsSize_out, ws.words, nnz, s); break;
        case 216: launch_count<2, 16>(nrows, nbr, d_rowptr, d_colidx, d_rowsSize_out, ws.words, nnz, s); break;
        case 416: launch_count<4, 16>(nrows, nbr, d_rowptr, d_colidx, d_rowsSize_out, ws.words, nnz, s); break;
        case 816: launch_count<8, 16>(nrows, nbr, d_rowptr, d_colidx, d_rowsSize_out, ws.words, nnz, s); break;
        }
        SPC5_HIP_TRY(hipGetLastError());
    }
    int rc = scan_exclusive_i32_ws(d_rowsSize_out, nbr + 1, ws.words + 2, ws.partials, s);
    if (rc) return rc;
    int h[3] = {0, 0, 0};
    rc = read_words(ws.words, h, 3, s);
    if (rc) return rc;
    if (h[0]) {
        set_error("CSR row pointer must start at 0 and be non-decreasing");
        return SPC5_HIP_ERR_INVALID;
    }
    if (h[1]) {
        set_error("CSR columns must be non-negative and strictly increasing inside each row");
        return SPC5_HIP_ERR_INVALID;
    }
    *nblocks = h[2];
    return SPC5_HIP_OK;
}

// The entry count of a CSR matrix whose caller did not give it: its last row
// pointer (waits).
int read_nnz(int64_t nrows, const int* d_rowptr, int64_t* nnz, hipStream_t s) {
    int n = 0;
    const int rc = read_words(d_rowptr + nrows, &n, 1, s);
    if (rc) return rc;
    if (n < 0 || (nrows == 0 && n != 0)) {
        set_error("CSR row pointer must start at 0 and be non-decreasing");
        return SPC5_HIP_ERR_INVALID;
    }
    *nnz = n;
    return SPC5_HIP_OK;
}

int check_convert_count_args(int vs, int r, int64_t nrows, const int* d_rowptr, const int* d_rowsSize_out,
                             const int64_t* nblocks) {
    SPC5_CHECK_ARG(nblocks != nullptr, "nblocks is null");
    SPC5_CHECK_ARG(r == 1 || r == 2 || r == 4 || r == 8, "r must be 1, 2, 4 or 8");
    SPC5_CHECK_ARG(vs == 8 || vs == 16, "VS must be 8 or 16");
    SPC5_CHECK_ARG(nrows >= 0 && nrows <= INT32_MAX, "nrows out of range");
    SPC5_CHECK_ARG(d_rowptr != nullptr && d_rowsSize_out != nullptr, "null pointer");
    SPC5_CHECK_ARG((const void*)d_rowptr != (const void*)d_rowsSize_out, "rowsSize_out must not alias rowptr");
    return SPC5_HIP_OK;
}

}  // namespace

}  // namespace spc5

using namespace spc5;

extern "C" {

int spc5_hip_convert_count_sized(int vs, int r, int64_t nrows, int64_t nnz, const int* d_rowptr, const int* d_colidx,
                                 int* d_rowsSize_out, int64_t* nblocks, void* stream) {
    int rc = check_convert_count_args(vs, r, nrows, d_rowptr, d_rowsSize_out, nblocks);
    if (rc) return rc;
    *nblocks = 0;
    SPC5_CHECK_ARG(nnz >= 0 && nnz <= INT32_MAX, "nnz out of range");
    hipStream_t s = as_stream(stream);
    const int64_t nbr = (nrows + r - 1) / r;
    CountScratch ws;
    ws.partial_cap = scan_partials_needed(nbr + 1);
    DeviceBuffer buf;
    SPC5_HIP_TRY(buf.alloc(sizeof(int) * (size_t)(kScratchWords + ws.partial_cap)));
    ws.words = buf.as<int>();
    ws.partials = ws.words + kScratchWords;
    rc = convert_count_impl(vs, r, nrows, nnz, d_rowptr, d_colidx, d_rowsSize_out, nblocks, ws, s);
    // the buffer is freed on return: every launch that uses it has ended
    if (rc) SPC5_HIP_TRY(hipStreamSynchronize(s));
    return rc;
}

int spc5_hip_convert_count(int vs, int r, int64_t nrows, const int* d_rowptr, const int* d_colidx,
                           int* d_rowsSize_out, int64_t* nblocks, void* stream) {
    int rc = check_convert_count_args(vs, r, nrows, d_rowptr, d_rowsSize_out, nblocks);
    if (rc) return rc;
    *nblocks = 0;
    int64_t nnz = 0;
    rc = read_nnz(nrows, d_rowptr, &nnz, as_stream(stream));
    if (rc) return rc;
    return spc5_hip_convert_count_sized(vs, r, nrows, nnz, d_rowptr, d_colidx, d_rowsSize_out, nblocks, stream);
}

int spc5_hip_convert_count_noalloc(int vs, int r, int64_t nrows, const int* d_rowptr, const int* d_colidx,
                                   int* d_rowsSize_out, int64_t* nblocks, void* stream) {
    int rc = check_convert_count_args(vs, r, nrows, d_rowptr, d_rowsSize_out, nblocks);
    if (rc) return rc;
    *nblocks = 0;
    CountScratch ws;
    rc = scratch_address(&ws.words);
    if (rc) return rc;
    ws.partials = ws.words + kScratchWords;
    ws.partial_cap = kScratchInts - kScratchWords;
    hipStream_t s = as_stream(stream);
    const int64_t nbr = (nrows + r - 1) / r;
    if (scan_partials_needed(nbr + 1) > ws.partial_cap)  // refused before any device work
        return convert_count_impl(vs, r, nrows, 0, d_rowptr, d_colidx, d_rowsSize_out, nblocks, ws, s);
    int64_t nnz = 0;
    rc = read_nnz(nrows, d_rowptr, &nnz, s);
    if (rc) return rc;
    return convert_count_impl(vs, r, nrows, nnz, d_rowptr, d_colidx, d_rowsSize_out, nblocks, ws, s);
}

int spc5_hip_convert_fill_sized(int value_bytes, int vs, int mask_bytes, int r, int64_t nrows, int64_t nnz,
                                int64_t nblocks, const int* d_rowptr, const int* d_colidx, const void* d_values_in,
                                const int* d_rowsSize, unsigned char* d_headers_out, void* d_values_out,
                                void* stream) {
    SPC5_CHECK_ARG(value_bytes == 8 || value_bytes == 4 || value_bytes == 2, "value_bytes must be 8, 4 or 2");
    SPC5_CHECK_ARG(nrows >= 0 && nrows <= INT32_MAX, "nrows out of range");
    SPC5_CHECK_ARG(nnz >= 0 && nnz <= INT32_MAX && nblocks >= 0 && nblocks <= INT32_MAX, "sizes out of range");
    SPC5_CHECK_ARG(d_rowptr != nullptr && d_rowsSize != nullptr, "null pointer");
    hipStream_t s = as_stream(stream);
    const int64_t nbr = (nrows + r - 1) / r;
    if (nbr == 0 || nblocks == 0) return SPC5_HIP_OK;
    SPC5_CHECK_ARG(d_headers_out != nullptr && d_values_out != nullptr && d_values_in != nullptr,
                   "null output/value pointer");
    switch (value_bytes) {
    case 8:
        return launch_fill_w<unsigned long long>(vs, mask_bytes, r, nrows, nbr, d_rowptr, d_colidx, d_values_in,
                                                 d_rowsSize, nblocks, nnz, d_headers_out, d_values_out, s);
    case 4:
        return launch_fill_w<unsigned int>(vs, mask_bytes, r, nrows, nbr, d_rowptr, d_colidx, d_values_in,
                                           d_rowsSize, nblocks, nnz, d_headers_out, d_values_out, s);
    default:
        return launch_fill_w<unsigned short>(vs, mask_bytes, r, nrows, nbr, d_rowptr, d_colidx, d_values_in,
                                             d_rowsSize, nblocks, nnz, d_headers_out, d_values_out, s);
    }
}

int spc5_hip_convert_fill(int value_bytes, int vs, int mask_bytes, int r, int64_t nrows, const int* d_rowptr,
                          const int* d_colidx, const void* d_values_in, const int* d_rowsSize,
                          unsigned char* d_headers_out, void* d_values_out, void* stream) {
    SPC5_CHECK_ARG(value_bytes == 8 || value_bytes == 4 || value_bytes == 2, "value_bytes must be 8, 4 or 2");
    SPC5_CHECK_ARG(nrows >= 0 && nrows <= INT32_MAX, "nrows out of range");
    SPC5_CHECK_ARG(d_rowptr != nullptr && d_rowsSize != nullptr, "null pointer");
    hipStream_t s = as_stream(stream);
    const int64_t nbr = (nrows + r - 1) / r;
    if (nbr == 0) return SPC5_HIP_OK;
    int nb = 0, nnz = 0;
    SPC5_HIP_TRY(hipMemcpyAsync(&nb, d_rowsSize + nbr, sizeof(int), hipMemcpyDeviceToHost, s));
    SPC5_HIP_TRY(hipMemcpyAsync(&nnz, d_rowptr + nrows, sizeof(int), hipMemcpyDeviceToHost, s));
    SPC5_HIP_TRY(hipStreamSynchronize(s));
    return spc5_hip_convert_fill_sized(value_bytes, vs, mask_bytes, r, nrows, nnz, nb, d_rowptr, d_colidx, d_values_in,
                                       d_rowsSize, d_headers_out, d_values_out, stream);
}

}  // extern "C"
