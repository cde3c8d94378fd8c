// spmv.hip -- beta(r,VS) SpMV on gfx950: y += A x with A in the reference
// block layout, plus the plan builder and the handle API.
//
// Kernel design (one wave = one tile of whole block-rows):
//   * the tile's block-row pointers go to LDS; a running value offset walks
//     the value stream exactly like the reference's `values += popcount`
//     (src/spc5.hpp:2571-2617), starting from the tile's planned offset;
//   * batch step: lane i decodes block b+i (unaligned int32 column + r
//     masks), counts its values (popcount), and a DPP wave scan gives each
//     block's position in the batch; blocks are taken while the batch holds
//     at most expand_cap<V>() values;
//   * each taken lane finds its block-row by binary search in LDS and
//     expands its set bits into (column, local row) pairs in LDS -- values
//     are never zero-padded;
//   * the batch's values are then read with fully coalesced loads, one per
//     lane, multiplied by x[column] and added into per-row LDS accumulators;
//   * at the end of the tile every row does one y[row] += sum (rows of a
//     tile belong to it alone, so no global atomics and no second pass).
//
// That is the value-order tile (spmv_tile.hpp).  Matrices whose neighbouring
// blocks read neighbouring parts of x run the lane-block tile instead
// (spmv_lane.hpp); lane_block_wins() decides per handle.
#include "spc5_mat.hpp"
#include "spmv_lane.hpp"
#include "spmv_tile.hpp"

#include <mutex>
#include <vector>

namespace spc5 {

namespace {

std::mutex g_err_mu;
std::string g_err;

// Workgroups are dealt to the 8 XCDs round-robin (group g runs on XCD g % 8).
// Renumbering groups so that each XCD walks one contiguous eighth of the
// tile list keeps the x window each XCD gathers from inside its own L2.
__device__ __forceinline__ int64_t xcd_tile(int wave) {
    const int64_t g = blockIdx.x;
#if SPC5_XCD_REMAP
    const int64_t per_xcd = gridDim.x >> 3;  // the grid is a multiple of 8
    const int64_t gx = (g & 7) * per_xcd + (g >> 3);
#else
    const int64_t gx = g;
#endif
    return gx * kWavesPerGroup + wave;
}


template <class V, class X, class ACC, int R, int VS, int MB, bool SORT>
__global__ __launch_bounds__(kWavesPerGroup * 64, tile_waves_per_eu(R, SORT, sizeof(X) > sizeof(ACC))) void
k_spmv_tiles(
    const int* __restrict__ bptr, const unsigned char* __restrict__ hdr, const V* __restrict__ val,
    const X* __restrict__ x, X* __restrict__ y, const int4* __restrict__ tiles, int64_t ntiles, int64_t nrows,
    int64_t ncols, Epilogue ep) {
    __shared__ TileSmem<ACC, R, expand_cap<V>(), SORT> sm[kWavesPerGroup];
    const int w = threadIdx.x >> 6;
    const int64_t t = xcd_tile(w);
    if (t >= ntiles) return;  // whole wave leaves; no workgroup barrier is used
    Epilogue e = ep;
    if (e.dot) e.dot += t;  // one partial per tile
    spmv_tile<V, X, ACC, R, VS, MB, SORT>(sm[w], bptr, hdr, val, x, y, tiles[t], tiles[t + 1], nrows, ncols, e);
}

template <class V, class X, class ACC, int R, int VS, int MB, int STAGE>
__global__ __launch_bounds__(kWavesPerGroup * 64, lane_waves_per_eu(R, VS, sizeof(X)) - (STAGE > 5120 ? 1 : 0)) void k_spmv_lanes(
    const int* __restrict__ bptr, const unsigned char* __restrict__ hdr, const V* __restrict__ val,
    const X* __restrict__ x, X* __restrict__ y, const int4* __restrict__ tiles, int64_t ntiles, int64_t nrows,
    int64_t ncols, Epilogue ep) {
    __shared__ LaneSmem<V, ACC, R, MB, STAGE> sm[kWavesPerGroup];
    const int w = threadIdx.x >> 6;
    const int64_t t = xcd_tile(w);
    if (t >= ntiles) return;  // whole wave leaves; no workgroup barrier is used
    Epilogue e = ep;
    if (e.dot) e.dot += t;  // one partial per tile
    spmv_lane_tile<V, X, ACC, R, VS, MB, STAGE>(sm[w], STAGE, bptr, hdr, val, x, y, tiles[t], tiles[t + 1], nrows,
                                                ncols, e);
}

// ---- access probe ----------------------------------------------------------

// Memory-access probe over a double beta(1,8) matrix (a measurement aid, not
// a product): the product's tiles on the product's grid, one wave per tile,
// batches of 64 blocks (one per lane, at most 512 values).  Every block's
// header (fetched one batch ahead) and the batch's values (coalesced,
// non-temporal) are read, and then
//   MODE 0: nothing more -- the matrix stream alone;
//   MODE 1: x at every value's column, expanded through LDS in value order as
//           the product gathers it;
//   MODE 2: as 1 with each column folded into a 1024-entry window of x at the
//           tile's first column: the same gathers, all L1 hits.
// There are no row sums and no y; the sum of the products reaches memory only
// on an impossible value, which keeps every load live.
template <int MODE>
__global__ __launch_bounds__(kWavesPerGroup * 64) void k_access_probe(
    const unsigned char* __restrict__ hdr, const double* __restrict__ val, const double* __restrict__ x,
    const int4* __restrict__ tiles, int64_t ntiles, int64_t ncols,
    double* __restrict__ out) {
    constexpr int H = 5;  // int32 first column + one mask byte
    __shared__ int scol[kWavesPerGroup][512];
    const int w = threadIdx.x >> 6;
    const int64_t t = xcd_tile(w);
    if (t >= ntiles) return;
    const int lane = threadIdx.x & 63;
    int* sc = scol[w];
    const int b0 = tiles[t].y, b1 = tiles[t + 1].y;
    int64_t v = tiles[t].z;
    double acc = 0.0;
    int cs = 0;
    unsigned m = 0;
    if (b0 + lane < b1) {
        cs = load_i32_unaligned(hdr + (int64_t)(b0 + lane) * H);
        m = hdr[(int64_t)(b0 + lane) * H + 4];
    }
    // the folded window (MODE 2): 1024 columns from the tile's first column
    const int64_t wbase = ncols >= 1024 ? (__shfl(cs, 0, 64) < ncols - 1024 ? __shfl(cs, 0, 64) : ncols - 1024) : 0;
    for (int b = b0; b < b1; b += 64) {
        const int cnt = __popc(m);
        const int incl = wave_incl_scan(cnt);
        const int total = __builtin_amdgcn_readlane(incl, 63);
        double a[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int q = lane + 64 * k;
            a[k] = q < total ? __builtin_nontemporal_load(val + v + q) : 0.0;
        }
        // next batch's header
        int ncs = 0;
        unsigned nm = 0;
        if (b + 64 + lane < b1) {
            ncs = load_i32_unaligned(hdr + (int64_t)(b + 64 + lane) * H);
            nm = hdr[(int64_t)(b + 64 + lane) * H + 4];
        }
        if constexpr (MODE == 0) {
#pragma unroll
            for (int k = 0; k < 8; ++k) acc += a[k];
            acc += (double)cs;
        } else {
            int p = incl - cnt;
#pragma unroll
            for (int bit = 0; bit < 8; ++bit)
                if ((m >> bit) & 1u) sc[p++] = MODE == 1 ? cs + bit : (int)(wbase + ((cs + bit) & 1023));
            wave_sync();
            double xv[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const int q = lane + 64 * k;
                xv[k] = q < total ? x[sc[q]] : 0.0;
            }
#pragma unroll
            for (int k = 0; k < 8; ++k) acc += a[k] * xv[k];
            wave_sync();
        }
        v += total;
        cs = ncs;
        m = nm;
    }
    if (acc == 1.2345e300) out[0] = acc;
}

// ---- plan kernels --------------------------------------------------------

// Values per block-row (popcount of every mask), with a check of the block-row
// pointers (0-based, non-decreasing, ending at nblocks: err bit 0; a wave whose
// pointers fail reads no header) and of the columns (bit 1).
// One wave per 64 block-rows: the lanes read
// the group's headers in block order, coalesced, find each block's block-row
// by a binary search of the 65 group pointers in LDS and add its popcount to
// that block-row's LDS counter.  Bound by the latency of the header loads and
// the searches, so each lane takes four blocks a round, loads first
// (clustered 1 M rows, double beta(4,8): 33 -> 21 us; 96 banded matrices of 1,000
// to 200,000 rows, 24.9 -> 11.2 us at the median).
template <int R, int MB, int VS>
__global__ __launch_bounds__(256) void k_blockrow_values(const int* __restrict__ bptr,
                                                         const unsigned char* __restrict__ hdr, int64_t nbr,
                                                         int64_t nblocks, int64_t ncols, int* __restrict__ cnt_out,
                                                         int* err,
                                                         int xbytes, unsigned every) {
    constexpr int H = 4 + R * MB;
    using MW = MaskWords<R * MB>;
    __shared__ unsigned sline[4][64];
    __shared__ int sptr[4][65];
    __shared__ int scnt[4][64];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int64_t br0 = ((int64_t)blockIdx.x * 4 + w) * 64;
    if (br0 >= nbr) return;  // whole wave: nothing below synchronises across waves
    if (br0 + 64 >= nbr && lane == 0) cnt_out[nbr] = 0;  // the scan's last entry
    int* sp = sptr[w];
    int* sc = scnt[w];
    {
        const int64_t i = br0 + lane;
        sp[lane] = bptr[i < nbr ? i : nbr];
        if (lane == 0) sp[64] = bptr[br0 + 64 < nbr ? br0 + 64 : nbr];
        sc[lane] = 0;
        sline[w][lane] = 0u;
    }
    wave_sync();
    {
        const int lo = sp[lane], hi = sp[lane + 1];
        bool broken = lo < 0 || hi < lo || (int64_t)hi > nblocks;
        if (lane == 0) broken |= (br0 == 0 && lo != 0) || (br0 + 64 >= nbr && (int64_t)sp[64] != nblocks);
        if (ballot64(broken)) {
            if (br0 + lane < nbr) cnt_out[br0 + lane] = 0;
            if (lane == 0) atomicOr(err, 1);
            return;
        }
    }
    const int b0 = sp[0], bE = sp[64];
    // One group in `every` also counts the distinct 128-byte lines of x that
    // its first 64 blocks start in (a hash into 2,048 bits): err[1] sums the
    // lines, err[2] the blocks.
    const bool sample = (blockIdx.x * 4u + (unsigned)w) % every == 0;
    bool bad = false;
    constexpr int U = 4;
    for (int bb = b0 + lane; bb - lane < bE; bb += 64 * U) {
        int cs[U];
        unsigned long long mw[U][MW::kWords];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int b = bb + 64 * u < bE ? bb + 64 * u : bE - 1;
            const unsigned char* h = hdr + (int64_t)b * H;
            cs[u] = load_i32_unaligned(h);
            MW::load(h + 4, mw[u]);
        }
        if (sample && bb < b0 + 64 && bb < bE) {
            const unsigned line = (unsigned)(((uint64_t)(unsigned)cs[0] * (unsigned)xbytes) >> 7);
            const unsigned h = (line * 0x9e3779b1u) >> 21;
            atomicOr(&sline[w][h >> 5], 1u << (h & 31u));
        }
        // the blocks' block-rows: the largest i with sp[i] <= b (sp[0] <= b < sp[64])
        int lo[U];
#pragma unroll
        for (int u = 0; u < U; ++u) lo[u] = 0;
#pragma unroll
        for (int step = 32; step >= 1; step >>= 1) {
#pragma unroll
            for (int u = 0; u < U; ++u) lo[u] += sp[lo[u] + step] <= bb + 64 * u ? step : 0;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (bb + 64 * u >= bE) continue;
            int c = 0;
            unsigned rowor = 0;
            for (int k = 0; k < MW::kWords; ++k) {
                c += __popcll(mw[u][k]);
                for (int q = 0; q < 64 / VS; ++q)
                    rowor |= (unsigned)((mw[u][k] >> (q * VS)) & ((1ull << VS) - 1ull));
            }
            if (rowor != 0) {
                const int hi = 31 - __builtin_clz(rowor);
                bad |= cs[u] < 0 || (int64_t)cs[u] + hi >= ncols;
            }
            atomicAdd(&sc[lo[u]], c);
        }
    }
    wave_sync();
    if (br0 + lane < nbr) cnt_out[br0 + lane] = sc[lane];
    if (bad) atomicOr(err, 2);
    if (sample && bE > b0) {
        const int lines = wave_reduce_add(__popc(sline[w][lane]));
        if (lane == 0) {
            atomicAdd(err + 1, lines);
            atomicAdd(err + 2, bE - b0 < 64 ? bE - b0 : 64);
        }
    }
}

// Tiles never cross a multiple of maxbr <= 64 block-rows (a chunk); a chunk is
// cut into ceil(values / target) pieces of about equal values.  One wave per
// chunk, one block-row per lane; returns the lanes whose block-row starts a
// tile.
__device__ __forceinline__ unsigned long long chunk_tiles(const int* __restrict__ valptr, int64_t chunk, int64_t nbr,
                                                          int target, int maxbr, int lane, int& v) {
    const int64_t first = chunk * maxbr;
    const int n = (int)(nbr - first < maxbr ? nbr - first : maxbr);
    v = valptr[first + (lane < n ? lane : n)];
    const int v0 = __builtin_amdgcn_readfirstlane(v), all = valptr[first + n] - v0;
    int64_t piece = 0;
    if (all > target) piece = (int64_t)(v - v0) * ((all + (int64_t)target - 1) / target) / all;
    const int at = (int)piece;  // at most the chunk's values / target
    const int before = wave_prev_lane(at, -1);
    return ballot64(lane < n && at != before);
}

constexpr int kChunkWaves = 4;

// WRITE false: tiles per chunk to `at` (at[nchunks] = 0).  WRITE true: `at` is
// the scanned count; the tiles' records are written, and the results the host
// reads are gathered: out[0..2] = err, out[3] = values, out[4] = tiles.
template <bool WRITE>
__global__ __launch_bounds__(64 * kChunkWaves) void k_tiles(const int* __restrict__ valptr,
                                                           const int* __restrict__ bptr, int64_t nbr, int target,
                                                           int maxbr, int64_t nchunks, int* __restrict__ at,
                                                           int4* __restrict__ tiles, int64_t room,
                                                           const int* __restrict__ err, int* __restrict__ out) {
    const int lane = threadIdx.x & 63;
    const int64_t c = (int64_t)blockIdx.x * kChunkWaves + (threadIdx.x >> 6);
    if (c > nchunks) return;
    if (c == nchunks) {
        if (lane != 0) return;
        if constexpr (WRITE) {
            const int n = at[nchunks], nv = valptr[nbr];
            if (n >= 0 && n < room) tiles[n] = make_int4((int)nbr, bptr[nbr], nv, 0);
            out[0] = err ? err[0] : 0;
            out[1] = err ? err[1] : 0;
            out[2] = err ? err[2] : 0;
            out[3] = nv;
            out[4] = n;
        } else {
            at[nchunks] = 0;
        }
        return;
    }
    int v;
    const unsigned long long starts = chunk_tiles(valptr, c, nbr, target, maxbr, lane, v);
    if constexpr (WRITE) {
        const int64_t br = c * maxbr + lane;
        const int to = at[c] + lanes_below(starts);
        if (((starts >> lane) & 1ull) && to < room) tiles[to] = make_int4((int)br, bptr[br], v, 0);
    } else {
        if (lane == 0) at[c] = __popcll(starts);
    }
}

template <int R, int MB, int VS>
void launch_blockrow_values(const spc5_hip_mat& m, int* cnt, int* err, hipStream_t s) {
    const unsigned g = (unsigned)((m.nbr + 255) / 256);  // 4 waves of 64 block-rows per workgroup
    const unsigned every = g * 4 > 64 ? g * 4 / 64 : 1;  // 64 .. 127 sampled groups (their sums are atomics)
    hipLaunchKernelGGL((k_blockrow_values<R, MB, VS>), dim3(g), dim3(256), 0, s, m.bptr, m.hdr, m.nbr, m.nblocks, m.ncols,
                       cnt, err, m.value_type == SPC5_HIP_F64 ? 8 : 4, every);
}

template <class V, class X, class ACC, int R, int VS, int MB, bool SORT>
void launch_tiles(const spc5_hip_mat& m, const void* x, void* y, hipStream_t s, const Epilogue& ep) {
    const int64_t groups = (m.plan.ntiles + kWavesPerGroup - 1) / kWavesPerGroup;
    const unsigned grid = (unsigned)((groups + 7) / 8 * 8);
    hipLaunchKernelGGL((k_spmv_tiles<V, X, ACC, R, VS, MB, SORT>), dim3(grid), dim3(kWavesPerGroup * 64), 0, s,
                       m.bptr, m.hdr, reinterpret_cast<const V*>(m.values), reinterpret_cast<const X*>(x),
                       reinterpret_cast<X*>(y), m.plan.tiles->as<int4>(), m.plan.ntiles, m.nrows,
                       m.ncols, ep);
}

template <class V, class X, class ACC, int R, int VS, int MB, int LEVEL = 0>
void launch_lanes(const spc5_hip_mat& m, const void* x, void* y, hipStream_t s, const Epilogue& ep) {
    constexpr int kStage = lane_stage_bytes(sizeof(V), R, VS, LEVEL);
    if constexpr (LEVEL + 1 < lane_levels(sizeof(V), R, VS)) {
        if (m.lane_body > LEVEL + 1) return launch_lanes<V, X, ACC, R, VS, MB, LEVEL + 1>(m, x, y, s, ep);
    }
    const int64_t groups = (m.plan.ntiles + kWavesPerGroup - 1) / kWavesPerGroup;
    const unsigned grid = (unsigned)((groups + 7) / 8 * 8);
    hipLaunchKernelGGL((k_spmv_lanes<V, X, ACC, R, VS, MB, kStage>), dim3(grid), dim3(kWavesPerGroup * 64), 0, s, m.bptr,
                       m.hdr, reinterpret_cast<const V*>(m.values), reinterpret_cast<const X*>(x),
                       reinterpret_cast<X*>(y), m.plan.tiles->as<int4>(), m.plan.ntiles, m.nrows, m.ncols, ep);
}

template <class V, class X, class ACC, int VS, int MB>
int launch_spmv_vs(const spc5_hip_mat& m, const void* x, void* y, hipStream_t s, const Epilogue& ep) {
    const bool sort = m.row_sort != 0;
    if constexpr (lane_block_fits(VS, sizeof(X))) {
        if (m.lane_body) {
            switch (m.r) {
            case 1: launch_lanes<V, X, ACC, 1, VS, MB>(m, x, y, s, ep); break;
            case 2: launch_lanes<V, X, ACC, 2, VS, MB>(m, x, y, s, ep); break;
            case 4: launch_lanes<V, X, ACC, 4, VS, MB>(m, x, y, s, ep); break;
            default: launch_lanes<V, X, ACC, 8, VS, MB>(m, x, y, s, ep); break;
            }
            SPC5_HIP_TRY(hipGetLastError());
            return SPC5_HIP_OK;
        }
    }
    switch (m.r) {
    case 1: launch_tiles<V, X, ACC, 1, VS, MB, false>(m, x, y, s, ep); break;
    case 2:
        if (sort) launch_tiles<V, X, ACC, 2, VS, MB, true>(m, x, y, s, ep);
        else launch_tiles<V, X, ACC, 2, VS, MB, false>(m, x, y, s, ep);
        break;
    case 4:
        if (sort) launch_tiles<V, X, ACC, 4, VS, MB, true>(m, x, y, s, ep);
        else launch_tiles<V, X, ACC, 4, VS, MB, false>(m, x, y, s, ep);
        break;
    case 8: launch_tiles<V, X, ACC, 8, VS, MB, false>(m, x, y, s, ep); break;  // row sort: r = 2, 4
    default:
        set_error("invalid r");
        return SPC5_HIP_ERR_INVALID;
    }
    SPC5_HIP_TRY(hipGetLastError());
    return SPC5_HIP_OK;
}

}  // namespace

void set_error(const std::string& msg) {
    std::lock_guard<std::mutex> lk(g_err_mu);
    g_err = msg;
}

std::string hip_msg(hipError_t e, const char* what) {
    return std::string(what) + ": " + hipGetErrorName(e) + " (" + hipGetErrorString(e) + ")";
}

const char* last_error_cstr() {
    static thread_local std::string copy;
    std::lock_guard<std::mutex> lk(g_err_mu);
    copy = g_err;
    return copy.c_str();
}

int launch_spmv(const spc5_hip_mat& m, const void* x, void* y, hipStream_t s, const Epilogue& ep) {
    if (m.plan.ntiles == 0) return SPC5_HIP_OK;
    if (m.value_type == SPC5_HIP_F64) return launch_spmv_vs<double, double, double, 8, 1>(m, x, y, s, ep);
    if (m.value_type == SPC5_HIP_F32 && m.vs == 16) return launch_spmv_vs<float, float, FloatAcc, 16, 2>(m, x, y, s, ep);
    if (m.value_type == SPC5_HIP_F32 && m.vs == 8) return launch_spmv_vs<float, float, FloatAcc, 8, 1>(m, x, y, s, ep);
    if (m.value_type == SPC5_HIP_BF16) return launch_spmv_vs<unsigned short, float, FloatAcc, 8, 1>(m, x, y, s, ep);
    set_error("unsupported value type / VS");
    return SPC5_HIP_ERR_INVALID;
}

int launch_spmv_f64vec(const spc5_hip_mat& m, const double* x, double* y, hipStream_t s, const Epilogue& ep) {
    if (m.plan.ntiles == 0) return SPC5_HIP_OK;
    if (m.value_type == SPC5_HIP_F64) return launch_spmv_vs<double, double, double, 8, 1>(m, x, y, s, ep);
    if (m.value_type == SPC5_HIP_F32 && m.vs == 16) return launch_spmv_vs<float, double, FloatAcc, 16, 2>(m, x, y, s, ep);
    if (m.value_type == SPC5_HIP_F32 && m.vs == 8) return launch_spmv_vs<float, double, FloatAcc, 8, 1>(m, x, y, s, ep);
    if (m.value_type == SPC5_HIP_BF16) return launch_spmv_vs<unsigned short, double, FloatAcc, 8, 1>(m, x, y, s, ep);
    set_error("unsupported value type / VS");
    return SPC5_HIP_ERR_INVALID;
}

namespace {

// Scratch of one plan: what the host reads back, the counters of
// k_blockrow_values, scan partials and the tile count of every chunk.
struct PlanScratch {
    DeviceBuffer buf;
    int* out = nullptr;       // int[8]: see k_tiles
    int* err = nullptr;       // int[8]: flags, sampled lines, sampled blocks
    int* partials = nullptr;
    int* chunks = nullptr;    // int[nchunks + 1]
    int64_t nchunks = 0;
    int maxbr = 1;
    hipError_t alloc(const spc5_hip_mat& m, int maxrows) {
        maxbr = maxrows / m.r > 0 ? maxrows / m.r : 1;
        if (maxbr > 64) maxbr = 64;
        nchunks = (m.nbr + maxbr - 1) / maxbr;
        const int64_t np = scan_partials_needed(m.nbr + 1);
        const hipError_t e = buf.alloc(sizeof(int) * (size_t)(16 + np + nchunks + 1));
        out = buf.as<int>();
        err = out + 8;
        partials = err + 8;
        chunks = partials + np;
        return e;
    }
};

// Enqueues the tile list of p.valptr (room for every tile is known beforehand:
// a chunk has at most one piece more than its values / target).
int enqueue_tiles(const spc5_hip_mat& m, Plan& p, int target, const PlanScratch& w, const int* err, hipStream_t s) {
    p.target = target;
    const int* valptr = p.valptr->as<int>();
    p.tiles = std::make_shared<DeviceBuffer>();
    const int64_t room = m.nnz / target + w.nchunks + 1;
    SPC5_HIP_TRY(p.tiles->alloc(sizeof(int4) * (size_t)room));
    const unsigned g = (unsigned)((w.nchunks + 1 + kChunkWaves - 1) / kChunkWaves);
    hipLaunchKernelGGL(k_tiles<false>, dim3(g), dim3(64 * kChunkWaves), 0, s, valptr, m.bptr, m.nbr, target, w.maxbr,
                       w.nchunks, w.chunks, nullptr, (int64_t)0, nullptr, nullptr);
    SPC5_HIP_TRY(hipGetLastError());
    const int rc = scan_exclusive_i32_ws(w.chunks, w.nchunks + 1, nullptr, w.partials, s);
    if (rc) return rc;
    hipLaunchKernelGGL(k_tiles<true>, dim3(g), dim3(64 * kChunkWaves), 0, s, valptr, m.bptr, m.nbr, target, w.maxbr,
                       w.nchunks, w.chunks, p.tiles->as<int4>(), room, err, w.out);
    SPC5_HIP_TRY(hipGetLastError());
    return SPC5_HIP_OK;
}

}  // namespace

// Everything is enqueued at once and the host waits once, for the results (a
// wait and a read-back cost about 30 us; checking the pointers first, counting
// values, counting tiles and allocating for them took four).  Until then the
// kernels only keep inside their buffers: waves with bad pointers read no
// header, and no tile is written past the room for the handle's nnz.
int build_plan(spc5_hip_mat& m, hipStream_t s) {
    Plan& p = m.plan;
    p.ntiles = 0;
    if (m.nbr == 0) return SPC5_HIP_OK;
    PlanScratch w;
    SPC5_HIP_TRY(w.alloc(m, tile_rows(m.r)));
    SPC5_HIP_TRY(hipMemsetAsync(w.err, 0, 8 * sizeof(int), s));
    p.valptr = std::make_shared<DeviceBuffer>();
    SPC5_HIP_TRY(p.valptr->alloc(sizeof(int) * (size_t)(m.nbr + 1)));
    int* valptr = p.valptr->as<int>();
    const int key = m.r * 100 + m.mb * 10 + (m.vs == 16 ? 1 : 0);
    switch (key) {
    case 110: launch_blockrow_values<1, 1, 8>(m, valptr, w.err, s); break;
    case 210: launch_blockrow_values<2, 1, 8>(m, valptr, w.err, s); break;
    case 410: launch_blockrow_values<4, 1, 8>(m, valptr, w.err, s); break;
    case 810: launch_blockrow_values<8, 1, 8>(m, valptr, w.err, s); break;
    case 121: launch_blockrow_values<1, 2, 16>(m, valptr, w.err, s); break;
    case 221: launch_blockrow_values<2, 2, 16>(m, valptr, w.err, s); break;
    case 421: launch_blockrow_values<4, 2, 16>(m, valptr, w.err, s); break;
    case 821: launch_blockrow_values<8, 2, 16>(m, valptr, w.err, s); break;
    default: set_error("unsupported (r, VS, mask bytes)"); return SPC5_HIP_ERR_INVALID;
    }
    SPC5_HIP_TRY(hipGetLastError());
    int rc = scan_exclusive_i32_ws(valptr, m.nbr + 1, nullptr, w.partials, s);
    if (rc) return rc;
    rc = enqueue_tiles(m, p, default_tile_values(m.nnz), w, w.err, s);
    if (rc) return rc;
    int h[5];
    SPC5_HIP_TRY(hipMemcpyAsync(h, w.out, sizeof(h), hipMemcpyDeviceToHost, s));
    SPC5_HIP_TRY(hipStreamSynchronize(s));
    if (h[0] & 1) {
        set_error("rowsSize is not a 0-based non-decreasing block pointer array ending at nblocks");
        return SPC5_HIP_ERR_INVALID;
    }
    if (h[0]) {
        set_error("a block touches a column outside [0, ncols)");
        return SPC5_HIP_ERR_INVALID;
    }
    if ((int64_t)h[3] != m.nnz) {
        set_error("nnz (" + std::to_string(m.nnz) + ") differs from the mask popcount (" + std::to_string(h[3]) + ")");
        return SPC5_HIP_ERR_INVALID;
    }
    p.ntiles = h[4];
    m.scatter = h[2] > 0 ? (double)h[1] / h[2] : 0.0;
    m.lane_body = lane_block_wins(m) ? 1 + lane_level(m) : 0;
    return SPC5_HIP_OK;
}

// Which tile a product runs: lane-block (one block per lane, spmv_lane.hpp)
// or value-order (spmv_tile.hpp).  The lane-block tile costs a fixed number of
// instructions per block position and one or more 16-byte x loads per block;
// the value-order tile costs about three times as many instructions per value
// but gathers x with fewer distinct lines per request.  So the line is drawn
// on `scatter`, the distinct 128-byte lines of x per block among 64 blocks in a
// row: stencils, narrow bands and Laplacians have 0.04 .. 0.41, bands wider
// than 64 blocks 0.5 .. 0.64 (every block its own part of a line or two, read
// once), the clustered matrix from 60,000 rows on 0.68 .. 0.97 (value-order /
// lane-block, us):
//   27-point stencil 128^3, scatter 0.2: float beta(2,16) 101 / 66, bfloat16
//     beta(2,8) 95 / 53, double beta(2,8) 121 / 108
//   banded 100,000 rows, half-width 130, scatter 0.14 .. 0.27: float beta(4,16)
//     29 / 19, double beta(4,8) 28 / 21
//   banded 60,000 rows, half-width 256 and 1,000, scatter 0.50 .. 0.64: double
//     beta(4,8) 32 / 26 and 98 / 68, beta(1,8) 34 / 31 and 106 / 97, float
//     beta(4,16) at 1,000 106 / 54
//   clustered 40,000 rows, scatter 0.61 .. 0.63: 9 / 9 at every r
//   clustered 1 M rows, scatter 0.8 .. 0.97: double beta(1,8) 88 / 102, float
//     beta(2,16) 61 / 66, but bfloat16 beta(2,8) 66 / 55
//   clustered 60,000 rows (x and matrix in the L2s): double beta(2,8) 10.5 /
//     8.6, float beta(4,16) 11.5 / 10.2, double beta(4,8) 10.4 / 11.4
// Double blocks of 8 rows (64 positions of 8 bytes, mostly empty) stay in value
// order: Laplacian 1400^2 37 / 47, stencil 128^3 149 / 176.
bool lane_block_wins(const spc5_hip_mat& m) {
    if ((uint64_t)m.ncols * 8 > 0xffffffffull || m.ncols < 16) return false;  // 32-bit x offsets, a whole window
    const bool f64 = m.value_type == SPC5_HIP_F64;
    if (f64 && m.r == 8) return false;
    if (m.scatter < 0.65) return true;
    const bool small = m.nnz < (4 << 20);
    if (f64) return m.r <= 2 && small;
    if (m.value_type == SPC5_HIP_F32 && m.vs == 16) return m.r <= 4 && small;
    return m.r <= 2 || (m.r == 4 && small);
}

// The lowest stage level that holds 64 blocks of the matrix's mean size, 0 up to
// 4 KiB (see lane_stage_bytes).
int lane_level(const spc5_hip_mat& m) {
    const int vb = (int)value_bytes(m.value_type);
    const int levels = lane_levels(vb, m.r, m.vs);
    if (levels == 1 || m.nblocks == 0) return 0;
    const double need = 64.0 * vb * (double)m.nnz / (double)m.nblocks;
    int level = need > 4096.0 ? 1 : 0;
    while (level > 0 && level + 1 < levels && need > lane_stage_bytes(vb, m.r, m.vs, level)) ++level;
    return level;
}

// Values per tile aimed at when no tile size is set (a tile also ends every
// tile_rows(r) rows).  Small matrices need many waves more than long ones (at
// 128 values the 64^2 Laplacian takes 3.2 us, at 512 4.2 us, double beta(2,8));
// large ones have 8,192 tiles or more whatever the size, and 2,048 values are
// short enough to even out uneven rows (clustered 1 M rows, double beta(1,8):
// 2,048 values 84 us, 4,096 values 94 us).
int default_tile_values(int64_t nnz) {
    int64_t target = nnz / 2048;
    if (target < 128) target = 128;
    if (target > 512) target = 512;
    if (target < nnz / 8192) target = nnz / 8192;
    if (target > 2048) target = 2048;
    return (int)target;
}

// Tile cut from the block-row value offsets: a tile starts where the running
// value count crosses a multiple of `target`, and at least every
// maxrows / r block-rows.
int build_tiles(const spc5_hip_mat& m, Plan& p, int maxrows, int target, hipStream_t s) {
    p.ntiles = 0;
    p.target = target;
    if (m.nbr == 0) return SPC5_HIP_OK;
    if (!p.valptr) p.valptr = m.plan.valptr;
    PlanScratch w;
    SPC5_HIP_TRY(w.alloc(m, maxrows));
    const int rc = enqueue_tiles(m, p, target, w, nullptr, s);
    if (rc) return rc;
    int n = 0;
    SPC5_HIP_TRY(hipMemcpyAsync(&n, w.out + 4, sizeof(int), hipMemcpyDeviceToHost, s));
    SPC5_HIP_TRY(hipStreamSynchronize(s));
    p.ntiles = n;
    return SPC5_HIP_OK;
}

}  // namespace spc5

using namespace spc5;

extern "C" {

const char* spc5_hip_last_error(void) { return spc5::last_error_cstr(); }

const char* spc5_hip_version(void) { return "spc5_hip 0.1 (gfx950)"; }

int spc5_hip_mat_create(int value_type, int vs, int r, int64_t nrows, int64_t ncols, int64_t nnz, int64_t nblocks,
                        const int* d_rowsSize, const unsigned char* d_headers, const void* d_values, void* stream,
                        spc5_hip_mat_t* out) {
    SPC5_CHECK_ARG(out != nullptr, "out is null");
    *out = nullptr;
    const int mb = (vs == 16) ? 2 : 1;
    SPC5_CHECK_ARG(r == 1 || r == 2 || r == 4 || r == 8, "r must be 1, 2, 4 or 8");
    SPC5_CHECK_ARG(valid_format(value_type, vs, mb), "unsupported (value type, VS) combination");
    SPC5_CHECK_ARG(nrows >= 0 && ncols >= 0 && nnz >= 0 && nblocks >= 0, "negative size");
    SPC5_CHECK_ARG(nnz <= INT32_MAX && nblocks <= INT32_MAX && nrows <= INT32_MAX && ncols <= INT32_MAX,
                   "sizes must fit the 32-bit format");
    SPC5_CHECK_ARG(nrows == 0 || d_rowsSize != nullptr, "rowsSize is null");
    SPC5_CHECK_ARG(nblocks == 0 || d_headers != nullptr, "headers are null");
    SPC5_CHECK_ARG(nnz == 0 || d_values != nullptr, "values are null");
    std::unique_ptr<spc5_hip_mat> m(new spc5_hip_mat());
    m->value_type = value_type;
    m->vs = vs;
    m->mb = mb;
    m->r = r;
    m->nrows = nrows;
    m->ncols = ncols;
    m->nnz = nnz;
    m->nblocks = nblocks;
    m->nbr = (nrows + r - 1) / r;
    m->bptr = d_rowsSize;
    m->hdr = d_headers;
    m->values = d_values;
    const int rc = build_plan(*m, as_stream(stream));
    if (rc) return rc;
    *out = m.release();
    return SPC5_HIP_OK;
}

int spc5_hip_mat_create_values_view(spc5_hip_mat_t base, int value_type, const void* d_values, spc5_hip_mat_t* out) {
    SPC5_CHECK_ARG(base != nullptr && out != nullptr, "null handle");
    SPC5_CHECK_ARG(valid_format(value_type, base->vs, base->mb), "value type incompatible with the block format");
    SPC5_CHECK_ARG(base->nnz == 0 || d_values != nullptr, "values are null");
    std::unique_ptr<spc5_hip_mat> m(new spc5_hip_mat(*base));
    m->value_type = value_type;
    m->values = d_values;
    m->lane_body = lane_block_wins(*m) ? 1 + lane_level(*m) : 0;
    *out = m.release();
    return SPC5_HIP_OK;
}

int spc5_hip_mat_destroy(spc5_hip_mat_t h) {
    if (h) forget_spmm_plans(h);
    delete h;
    return SPC5_HIP_OK;
}

int spc5_hip_mat_info(spc5_hip_mat_t h, int64_t* ntiles, int64_t* nblockrows, int64_t* nblocks, int64_t* nnz) {
    SPC5_CHECK_ARG(h != nullptr, "null handle");
    if (ntiles) *ntiles = h->plan.ntiles;
    if (nblockrows) *nblockrows = h->nbr;
    if (nblocks) *nblocks = h->nblocks;
    if (nnz) *nnz = h->nnz;
    return SPC5_HIP_OK;
}

int spc5_hip_mat_set_option(spc5_hip_mat_t h, int option, int64_t value) {
    SPC5_CHECK_ARG(h != nullptr, "null handle");
    switch (option) {
    case SPC5_HIP_OPT_ROW_SORT:
        SPC5_CHECK_ARG(value == 0 || value == 1, "ROW_SORT must be 0 or 1");
        h->row_sort = (int)value;
        return SPC5_HIP_OK;
    case SPC5_HIP_OPT_SPMM_COLUMNS:
        SPC5_CHECK_ARG(value == 0 || value == 1, "SPMM_COLUMNS must be 0 or 1");
        h->spmm_cols = (int)value;
        return SPC5_HIP_OK;
    case SPC5_HIP_OPT_SPMM_X16:
        SPC5_CHECK_ARG(value == 0 || value == 1, "SPMM_X16 must be 0 or 1");
        h->spmm_x16 = (int)value;
        return SPC5_HIP_OK;
    case SPC5_HIP_OPT_TILE_VALUES: {
        SPC5_CHECK_ARG(value == 0 || (value >= 64 && value <= (1 << 24)), "TILE_VALUES must be 0 or in [64, 2^24]");
        const int target = value == 0 ? default_tile_values(h->nnz) : (int)value;
        if (h->nbr == 0 || target == h->plan.target) return SPC5_HIP_OK;
        Plan np;
        np.valptr = h->plan.valptr;
        const int rc = build_tiles(*h, np, tile_rows(h->r), target, nullptr);
        if (rc) return rc;
        h->plan = np;  // shared buffers of the old plan stay alive while views or batches use them
        return SPC5_HIP_OK;
    }
    default:
        set_error("unknown option");
        return SPC5_HIP_ERR_INVALID;
    }
}

int spc5_hip_access_probe(spc5_hip_mat_t h, int mode, const void* d_x, void* d_out, void* stream) {
    SPC5_CHECK_ARG(h != nullptr && d_x != nullptr && d_out != nullptr, "null argument");
    SPC5_CHECK_ARG(h->value_type == SPC5_HIP_F64 && h->r == 1 && h->vs == 8 && h->mb == 1,
                   "the access probe takes a double beta(1,8) matrix");
    SPC5_CHECK_ARG(mode >= 0 && mode <= 2, "mode must be 0, 1 or 2");
    SPC5_CHECK_ARG(mode != 2 || h->ncols >= 1024, "mode 2 needs at least 1024 columns");
    const spc5_hip_mat& m = *h;
    if (m.plan.ntiles == 0) return SPC5_HIP_OK;
    const int64_t groups = (m.plan.ntiles + kWavesPerGroup - 1) / kWavesPerGroup;
    const unsigned grid = (unsigned)((groups + 7) / 8 * 8);
    const double* xv = reinterpret_cast<const double*>(d_x);
    const double* vv = reinterpret_cast<const double*>(m.values);
    double* o = reinterpret_cast<double*>(d_out);
    const int4* tl = m.plan.tiles->as<int4>();
    hipStream_t s = as_stream(stream);
    switch (mode) {
    case 0:
        hipLaunchKernelGGL(k_access_probe<0>, dim3(grid), dim3(kWavesPerGroup * 64), 0, s, m.hdr, vv, xv, tl,
                           m.plan.ntiles, m.ncols, o);
        break;
    case 1:
        hipLaunchKernelGGL(k_access_probe<1>, dim3(grid), dim3(kWavesPerGroup * 64), 0, s, m.hdr, vv, xv, tl,
                           m.plan.ntiles, m.ncols, o);
        break;
    default:
        hipLaunchKernelGGL(k_access_probe<2>, dim3(grid), dim3(kWavesPerGroup * 64), 0, s, m.hdr, vv, xv, tl,
                           m.plan.ntiles, m.ncols, o);
        break;
    }
    SPC5_HIP_TRY(hipGetLastError());
    return SPC5_HIP_OK;
}

int spc5_hip_spmv(spc5_hip_mat_t h, const void* d_x, void* d_y, void* stream) {
    SPC5_CHECK_ARG(h != nullptr, "null handle");
    SPC5_CHECK_ARG(h->nnz == 0 || (d_x != nullptr && d_y != nullptr), "x or y is null");
    return launch_spmv(*h, d_x, d_y, as_stream(stream));
}

}  // extern "C"
