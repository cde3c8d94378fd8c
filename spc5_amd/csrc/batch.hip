// batch.hip -- many independent beta(r,VS) matrices in one
// hipGraph-captured launch (the batching form; no counterpart in the
// reference).
//
// The tiles of every matrix form one list (matrix index and tile bounds
// per entry, built once at batch creation).  A grid of
// `waves` waves walks the list with a static stride; each tile runs the
// same tile routine as the single-matrix kernel, with the matrix's own r
// (chosen per matrix, e.g. by the autotuner) selected at run time.  When
// every matrix has the same r, a kernel holding only that r's body runs
// instead (the four bodies together need far more registers than one); with
// r = 2 or 4 and row sorting switched on for every matrix, that kernel uses
// the row-sorted tile (as the single-matrix product does).
// The launch is captured once into a hipGraph; every product replays it.
#include "spc5_mat.hpp"
#include "spmv_lane.hpp"
#include "spmv_tile.hpp"

#include <algorithm>
#include <vector>

using namespace spc5;

struct BatchEntry {
    const int* bptr;
    const unsigned char* hdr;
    const void* val;
    const void* x;
    void* y;
    int64_t nrows;
    int64_t ncols;
    int r;
    int lanes;  // 1 + stage level: lane-block tile
};

// One tile of the batch: its matrix, where it starts and where it ends
// ({block-row, block, value, matrix} and the next tile's).
struct alignas(32) BatchTile {
    int4 first, last;
};

struct spc5_hip_batch {
    int value_type = SPC5_HIP_F64;
    int vs = 8;
    int nmats = 0;
    int64_t ntiles = 0;
    int waves = 0;
    int only_r = 0;         // the r shared by every matrix, 0 if they differ
    int lanes = 0;          // only_r, and every matrix runs the lane-block tile: 1 + their highest stage level
    int sorted = 0;         // only_r is 2 or 4, not all lane-block, and every matrix has row sorting on
    DeviceBuffer entries;   // BatchEntry[nmats]
    // BatchTile[ntiles], copied: a matrix's plan may be rebuilt later
    // (SPC5_HIP_OPT_TILE_VALUES).
    DeviceBuffer tiles;
    std::vector<spc5_hip_mat_t> mats;  // borrowed handles
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    hipStream_t capture_stream = nullptr;
    ~spc5_hip_batch() {
        if (exec) (void)hipGraphExecDestroy(exec);
        if (graph) (void)hipGraphDestroy(graph);
        if (capture_stream) (void)hipStreamDestroy(capture_stream);
    }
};

namespace spc5 {
namespace {

template <class V, class ACC>
union BatchSmem {
    TileSmem<ACC, 1, expand_cap<V>()> r1;
    TileSmem<ACC, 2, expand_cap<V>()> r2;
    TileSmem<ACC, 4, expand_cap<V>()> r4;
    TileSmem<ACC, 8, expand_cap<V>()> r8;
};
// The largest stage of the values (the matrices' own levels bound its use).
template <class V, int R, int MB>
constexpr int max_stage() {
    return lane_stage_bytes(sizeof(V), R, 8 * MB, lane_levels(sizeof(V), R, 8 * MB) - 1);
}

// Any r and either tile.
template <class V, class ACC, int MB>
union MixedSmem {
    BatchSmem<V, ACC> order;
    LaneSmem<V, ACC, 1, MB, max_stage<V, 1, MB>()> l1;
    LaneSmem<V, ACC, 2, MB, max_stage<V, 2, MB>()> l2;
    LaneSmem<V, ACC, 4, MB, max_stage<V, 4, MB>()> l4;
    LaneSmem<V, ACC, 8, MB, max_stage<V, 8, MB>()> l8;
};
#define SPC5_BATCH_TILE(RR, SMEM) \
    spmv_tile<V, X, ACC, RR, VS, MB>(SMEM, m.bptr, m.hdr, val, x, y, first, last, m.nrows, m.ncols, ep)

// Waves per SIMD of the batch kernel: with every r body (ONLY_R = 0) the
// most that compile without spills; with one r, the tile kernel's rule.
constexpr int batch_waves_per_eu(int only_r, bool wide_x, int value_bytes, bool sorted = false) {
    // the tile loop's own state costs one wave (two with 8-byte values)
    return only_r == 0 ? 5 : tile_waves_per_eu(only_r, sorted, wide_x) - (value_bytes == 8 ? 2 : 1);
}

#define SPC5_BATCH_LANES(RR, SMEM) \
    spmv_lane_tile<V, X, ACC, RR, VS, MB>(SMEM, lane_stage_bytes(sizeof(V), RR, VS, m.lanes - 1), m.bptr, m.hdr, val, x, y, first, last, m.nrows, m.ncols, ep)

// The batch loop over tiles: tile t of the list runs body(matrix entry,
// tile bounds) on its wave.  The record of a wave's next tile is loaded while the current one runs, so a
// tile starts with its matrix's entry (shared by its neighbours) and not with
// the chain matrix index -> matrix -> tile list -> bounds (96 banded matrices,
// double beta(4,8), tiles of 500 values: 715 -> 698 us).
template <class Body>
__device__ __forceinline__ void batch_tiles(const BatchEntry* __restrict__ mats, const BatchTile* __restrict__ tiles,
                                            int64_t ntiles, Body&& body) {
    const int w = threadIdx.x >> 6;
    const int64_t stride = (int64_t)gridDim.x * kWavesPerGroup;
    // The tile index is the same on every lane (it comes from the wave index,
    // which the compiler cannot tell is uniform): read it as a scalar, so the
    // records are loaded into scalar registers.
    const int64_t t0 = (int64_t)__builtin_amdgcn_readfirstlane((int)(blockIdx.x * kWavesPerGroup + w));
    if (t0 >= ntiles) return;
    BatchTile next = tiles[t0];
    for (int64_t t = t0; t < ntiles; t += stride) {
        const BatchTile cur = next;
        next = tiles[t + stride < ntiles ? t + stride : t];
        body(mats[cur.first.w], cur.first, cur.last);
        wave_sync();
    }
}

// Every matrix has r = R and row sorting on; those that run the lane-block
// tile keep it.
template <class V, class X, class ACC, int VS, int MB, int R>
__global__ __launch_bounds__(kWavesPerGroup * 64, batch_waves_per_eu(R, sizeof(X) > sizeof(ACC), sizeof(V), true)) void
k_spmv_batch_sorted(const BatchEntry* __restrict__ mats, const BatchTile* __restrict__ tiles, int64_t ntiles) {
    static_assert(R == 2 || R == 4, "row-sorted tiles exist for r = 2 and 4");
    __shared__ union {
        TileSmem<ACC, R, expand_cap<V>(), true> order;
        LaneSmem<V, ACC, R, MB, max_stage<V, R, MB>()> lanes;
    } sm[kWavesPerGroup];
    const int w = threadIdx.x >> 6;
    const Epilogue ep;
    batch_tiles(mats, tiles, ntiles, [&](const BatchEntry& m, int4 first, int4 last) {
        if (m.lanes)
            spmv_lane_tile<V, X, ACC, R, VS, MB>(sm[w].lanes, lane_stage_bytes(sizeof(V), R, VS, m.lanes - 1), m.bptr,
                                                 m.hdr, reinterpret_cast<const V*>(m.val),
                                                 reinterpret_cast<const X*>(m.x), reinterpret_cast<X*>(m.y), first,
                                                 last, m.nrows, m.ncols, ep);
        else
            spmv_tile<V, X, ACC, R, VS, MB, true>(sm[w].order, m.bptr, m.hdr, reinterpret_cast<const V*>(m.val),
                                              reinterpret_cast<const X*>(m.x), reinterpret_cast<X*>(m.y), first, last,
                                              m.nrows, m.ncols, ep);
    });
}

// Every matrix has r = R and runs the lane-block tile, at LEVEL or below.
template <class V, class X, class ACC, int VS, int MB, int R, int LEVEL>
__global__ __launch_bounds__(kWavesPerGroup * 64, lane_waves_per_eu(R, VS, sizeof(X)) - 1) void k_spmv_batch_lanes(
    const BatchEntry* __restrict__ mats, const BatchTile* __restrict__ tiles, int64_t ntiles) {
    __shared__ LaneSmem<V, ACC, R, MB, lane_stage_bytes(sizeof(V), R, VS, LEVEL)> sm[kWavesPerGroup];
    const int w = threadIdx.x >> 6;
    const Epilogue ep;
    batch_tiles(mats, tiles, ntiles, [&](const BatchEntry& m, int4 first, int4 last) {
        const int stage = lane_stage_bytes(sizeof(V), R, VS, LEVEL == 0 ? 0 : m.lanes - 1);
        spmv_lane_tile<V, X, ACC, R, VS, MB>(sm[w], stage, m.bptr, m.hdr, reinterpret_cast<const V*>(m.val),
                                             reinterpret_cast<const X*>(m.x), reinterpret_cast<X*>(m.y), first, last,
                                             m.nrows, m.ncols, ep);
    });
}

// Every matrix has r = R and runs the value-order tile.
template <class V, class X, class ACC, int VS, int MB, int R>
__global__ __launch_bounds__(kWavesPerGroup * 64, batch_waves_per_eu(R, sizeof(X) > sizeof(ACC), sizeof(V))) void
k_spmv_batch(const BatchEntry* __restrict__ mats, const BatchTile* __restrict__ tiles, int64_t ntiles) {
    __shared__ TileSmem<ACC, R, expand_cap<V>()> sm[kWavesPerGroup];
    const int w = threadIdx.x >> 6;
    const Epilogue ep;
    batch_tiles(mats, tiles, ntiles, [&](const BatchEntry& m, int4 first, int4 last) {
        spmv_tile<V, X, ACC, R, VS, MB>(sm[w], m.bptr, m.hdr, reinterpret_cast<const V*>(m.val),
                                        reinterpret_cast<const X*>(m.x), reinterpret_cast<X*>(m.y), first, last,
                                        m.nrows, m.ncols, ep);
    });
}

// Any r and either tile per matrix.
template <class V, class X, class ACC, int VS, int MB>
__global__ __launch_bounds__(kWavesPerGroup * 64, batch_waves_per_eu(0, sizeof(X) > sizeof(ACC), sizeof(V))) void
k_spmv_batch_mixed(const BatchEntry* __restrict__ mats, const BatchTile* __restrict__ tiles, int64_t ntiles) {
    __shared__ MixedSmem<V, ACC, MB> sm[kWavesPerGroup];
    const int w = threadIdx.x >> 6;
    const Epilogue ep;
    batch_tiles(mats, tiles, ntiles, [&](const BatchEntry& m, int4 first, int4 last) {
        const V* val = reinterpret_cast<const V*>(m.val);
        const X* x = reinterpret_cast<const X*>(m.x);
        X* y = reinterpret_cast<X*>(m.y);
        switch (m.lanes ? -m.r : m.r) {
        case 1: SPC5_BATCH_TILE(1, sm[w].order.r1); break;
        case 2: SPC5_BATCH_TILE(2, sm[w].order.r2); break;
        case 4: SPC5_BATCH_TILE(4, sm[w].order.r4); break;
        case 8: SPC5_BATCH_TILE(8, sm[w].order.r8); break;
        case -1: SPC5_BATCH_LANES(1, sm[w].l1); break;
        case -2: SPC5_BATCH_LANES(2, sm[w].l2); break;
        case -4: SPC5_BATCH_LANES(4, sm[w].l4); break;
        default: SPC5_BATCH_LANES(8, sm[w].l8); break;
        }
    });
}

// The tile records of one matrix.
__global__ __launch_bounds__(256) void k_batch_records(const int4* __restrict__ tiles, int64_t ntiles, int mat,
                                                       BatchTile* __restrict__ out) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= ntiles) return;
    const int4 a = tiles[t];
    out[t] = BatchTile{make_int4(a.x, a.y, a.z, mat), tiles[t + 1]};
}

template <class Kernel>
void launch_batch_kernel(const spc5_hip_batch& b, Kernel k, hipStream_t s) {
    const unsigned groups = (unsigned)((b.waves + kWavesPerGroup - 1) / kWavesPerGroup);
    hipLaunchKernelGGL(k, dim3(groups), dim3(kWavesPerGroup * 64), 0, s, b.entries.as<const BatchEntry>(),
                       b.tiles.as<const BatchTile>(), b.ntiles);
}

template <class V, class X, class ACC, int VS, int MB, int R, int LEVEL = 0>
void launch_batch_lanes(const spc5_hip_batch& b, hipStream_t s) {
    if constexpr (LEVEL + 1 < lane_levels(sizeof(V), R, VS)) {
        if (b.lanes > LEVEL + 1) return launch_batch_lanes<V, X, ACC, VS, MB, R, LEVEL + 1>(b, s);
    }
    launch_batch_kernel(b, k_spmv_batch_lanes<V, X, ACC, VS, MB, R, LEVEL>, s);
}

template <class V, class X, class ACC, int VS, int MB>
void launch_batch(const spc5_hip_batch& b, hipStream_t s) {
    if (b.sorted) {
        if (b.only_r == 2) launch_batch_kernel(b, k_spmv_batch_sorted<V, X, ACC, VS, MB, 2>, s);
        else launch_batch_kernel(b, k_spmv_batch_sorted<V, X, ACC, VS, MB, 4>, s);
        return;
    }
    switch (b.lanes ? -b.only_r : b.only_r) {
    case 1: launch_batch_kernel(b, k_spmv_batch<V, X, ACC, VS, MB, 1>, s); break;
    case 2: launch_batch_kernel(b, k_spmv_batch<V, X, ACC, VS, MB, 2>, s); break;
    case 4: launch_batch_kernel(b, k_spmv_batch<V, X, ACC, VS, MB, 4>, s); break;
    case 8: launch_batch_kernel(b, k_spmv_batch<V, X, ACC, VS, MB, 8>, s); break;
    case -1: launch_batch_lanes<V, X, ACC, VS, MB, 1>(b, s); break;
    case -2: launch_batch_lanes<V, X, ACC, VS, MB, 2>(b, s); break;
    case -4: launch_batch_lanes<V, X, ACC, VS, MB, 4>(b, s); break;
    case -8: launch_batch_lanes<V, X, ACC, VS, MB, 8>(b, s); break;
    default: launch_batch_kernel(b, k_spmv_batch_mixed<V, X, ACC, VS, MB>, s); break;
    }
}

// Waves launched by default for every one that is resident at once: with the
// resident ones alone the last wave to finish its share of uneven tiles sets
// the time, and none starts a tile while another waits for its first loads.
// 96 banded matrices (1,000 to 200,000 rows, half-widths 4 to 256), us at 1, 4,
// 8, 16, 32 rounds and one wave per tile: double beta(4,8) 695, 642, 615, 606,
// 606, 612; beta(8,8) 1038, 909, 860, 833, 827, 835; 4 matrices beta(4,8) 49.1,
// 42.8, 42.6, 41.9, 41.5, 41.0.
constexpr int kWaveRounds = 32;

// Waves per SIMD the batch's kernel runs at (sizes the grid).
int batch_kernel_waves(const spc5_hip_batch& b) {
    const int vb = (int)value_bytes(b.value_type);
    if (b.lanes) return lane_waves_per_eu(b.only_r, b.vs, vb == 8 ? 8 : 4) - 1;
    return batch_waves_per_eu(b.only_r, false, vb, b.sorted != 0);
}

int launch_batch_any(const spc5_hip_batch& b, hipStream_t s) {
    if (b.value_type == SPC5_HIP_F64)
        launch_batch<double, double, double, 8, 1>(b, s);
    else if (b.value_type == SPC5_HIP_F32 && b.vs == 16)
        launch_batch<float, float, FloatAcc, 16, 2>(b, s);
    else if (b.value_type == SPC5_HIP_F32)
        launch_batch<float, float, FloatAcc, 8, 1>(b, s);
    else
        launch_batch<unsigned short, float, FloatAcc, 8, 1>(b, s);
    SPC5_HIP_TRY(hipGetLastError());
    return SPC5_HIP_OK;
}

}  // namespace
}  // namespace spc5

extern "C" {

int spc5_hip_batch_create(int nmats, const spc5_hip_mat_t* mats, const void* const* d_x, void* const* d_y,
                          int waves, spc5_hip_batch_t* out) {
    SPC5_CHECK_ARG(out != nullptr && nmats > 0 && mats != nullptr && d_x != nullptr && d_y != nullptr,
                   "null argument or empty batch");
    *out = nullptr;
    std::unique_ptr<spc5_hip_batch> b(new spc5_hip_batch());
    b->value_type = mats[0]->value_type;
    b->vs = mats[0]->vs;
    b->nmats = nmats;
    std::vector<BatchEntry> ent((size_t)nmats);
    for (int i = 0; i < nmats; ++i) {
        const spc5_hip_mat* m = mats[i];
        SPC5_CHECK_ARG(m != nullptr, "null matrix handle");
        SPC5_CHECK_ARG(m->value_type == b->value_type && m->vs == b->vs, "all matrices need one value type and VS");
        SPC5_CHECK_ARG(m->nnz == 0 || (d_x[i] != nullptr && d_y[i] != nullptr), "null x or y");
        BatchEntry& e = ent[(size_t)i];
        e.bptr = m->bptr;
        e.hdr = m->hdr;
        e.val = m->values;
        e.x = d_x[i];
        e.y = d_y[i];
        e.nrows = m->nrows;
        e.ncols = m->ncols;
        e.r = m->r;
        e.lanes = m->lane_body;
        b->mats.push_back(const_cast<spc5_hip_mat*>(m));
    }
    for (const spc5_hip_mat* m : b->mats) b->ntiles += m->plan.ntiles;
    SPC5_CHECK_ARG(b->ntiles <= 0x7ffffff0, "batch: more than 2^31 - 16 tiles");
    int dev = 0, ncu = 256;
    SPC5_HIP_TRY(hipGetDevice(&dev));
    SPC5_HIP_TRY(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
    b->only_r = mats[0]->r;
    bool all_sorted = true, all_lanes = true, any_lanes = false;
    int level = 0;
    for (int i = 0; i < nmats; ++i) {
        if (mats[i]->r != mats[0]->r) b->only_r = 0;
        all_lanes = all_lanes && mats[i]->lane_body;
        any_lanes = any_lanes || mats[i]->lane_body;
        level = std::max(level, mats[i]->lane_body);
        all_sorted = all_sorted && mats[i]->row_sort != 0;
    }
    b->lanes = b->only_r && all_lanes ? level : 0;
    b->sorted = (b->only_r == 2 || b->only_r == 4) && !b->lanes && all_sorted ? 1 : 0;
    if (b->only_r && !b->lanes && !b->sorted && any_lanes) b->only_r = 0;  // both tiles: the mixed kernel
    int64_t wv = waves > 0 ? waves : (int64_t)ncu * 4 * batch_kernel_waves(*b) * kWaveRounds;
    if (wv > b->ntiles) wv = std::max<int64_t>(b->ntiles, 1);
    b->waves = (int)wv;
    SPC5_HIP_TRY(b->entries.alloc(sizeof(BatchEntry) * (size_t)nmats));
    SPC5_HIP_TRY(b->tiles.alloc(sizeof(BatchTile) * (size_t)std::max<int64_t>(b->ntiles, 1)));
    SPC5_HIP_TRY(hipMemcpy(b->entries.p, ent.data(), sizeof(BatchEntry) * (size_t)nmats, hipMemcpyHostToDevice));
    int64_t at = 0;
    for (int i = 0; i < nmats; ++i) {
        const Plan& p = mats[i]->plan;
        if (p.ntiles)
            hipLaunchKernelGGL(k_batch_records, dim3((unsigned)((p.ntiles + 255) / 256)), dim3(256), 0, nullptr,
                               p.tiles->as<const int4>(), p.ntiles, i, b->tiles.as<BatchTile>() + at);
        at += p.ntiles;
    }
    SPC5_HIP_TRY(hipGetLastError());
    SPC5_HIP_TRY(hipStreamSynchronize(nullptr));
    // Capture the launch once; products replay the graph.
    SPC5_HIP_TRY(hipStreamCreateWithFlags(&b->capture_stream, hipStreamNonBlocking));
    if (b->ntiles) {
        SPC5_HIP_TRY(hipStreamBeginCapture(b->capture_stream, hipStreamCaptureModeThreadLocal));
        const int rc = launch_batch_any(*b, b->capture_stream);
        hipGraph_t g = nullptr;
        const hipError_t e = hipStreamEndCapture(b->capture_stream, &g);
        if (rc) return rc;
        SPC5_HIP_TRY(e);
        b->graph = g;
        SPC5_HIP_TRY(hipGraphInstantiate(&b->exec, b->graph, nullptr, nullptr, 0));
    }
    *out = b.release();
    return SPC5_HIP_OK;
}

int spc5_hip_batch_spmv(spc5_hip_batch_t b, void* stream) {
    SPC5_CHECK_ARG(b != nullptr, "null batch");
    if (!b->exec) return SPC5_HIP_OK;
    SPC5_HIP_TRY(hipGraphLaunch(b->exec, as_stream(stream)));
    return SPC5_HIP_OK;
}

int spc5_hip_batch_spmv_direct(spc5_hip_batch_t b, void* stream) {
    SPC5_CHECK_ARG(b != nullptr, "null batch");
    if (!b->ntiles) return SPC5_HIP_OK;
    return launch_batch_any(*b, as_stream(stream));
}

int spc5_hip_batch_info(spc5_hip_batch_t b, int64_t* ntiles, int* waves) {
    SPC5_CHECK_ARG(b != nullptr, "null batch");
    if (ntiles) *ntiles = b->ntiles;
    if (waves) *waves = b->waves;
    return SPC5_HIP_OK;
}

int spc5_hip_batch_destroy(spc5_hip_batch_t b) {
    delete b;
    return SPC5_HIP_OK;
}

}  // extern "C"
