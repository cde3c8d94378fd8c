// scan.hip -- in-place exclusive prefix sum of int32 arrays: chunk sums, then
// every chunk scans itself from the sum of the chunks before it.  Up to
// kScanChunk chunks (4 M entries) each workgroup adds those sums itself, so a
// scan is two launches; above, one workgroup scans them in between.  Launches
// set the time at these sizes (262 K entries: three launches 14 us, two 9 us).
// Used by the plan builder and the GPU converter.
#include "spc5_common.hpp"

namespace spc5 {

namespace {

constexpr int kScanThreads = 256;
constexpr int kScanItems = 8;                            // per thread
constexpr int kScanChunk = kScanThreads * kScanItems;    // per workgroup

// Block-wide exclusive scan of one value per thread; returns the block total.
__device__ int block_excl_scan(int v, int* s_wave_tot, int& excl) {
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int incl = wave_incl_scan(v);
    if (lane == 63) s_wave_tot[wave] = incl;
    __syncthreads();
    int before = 0, total = 0;
    for (int w = 0; w < kScanThreads / 64; ++w) {
        const int t = s_wave_tot[w];
        if (w < wave) before += t;
        total += t;
    }
    __syncthreads();
    excl = before + incl - v;
    return total;
}

__global__ __launch_bounds__(kScanThreads) void k_scan_reduce(const int* __restrict__ in, int64_t n,
                                                               int* __restrict__ partial) {
    __shared__ int s_tot[kScanThreads / 64];
    const int64_t base = (int64_t)blockIdx.x * kScanChunk + (int64_t)threadIdx.x * kScanItems;
    int sum = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        const int64_t i = base + k;
        if (i < n) sum += in[i];
    }
    int excl;
    const int total = block_excl_scan(sum, s_tot, excl);
    if (threadIdx.x == 0) partial[blockIdx.x] = total;
}

// One workgroup scans all partials, chunk after chunk, carrying the total.
__global__ __launch_bounds__(kScanThreads) void k_scan_partials(int* __restrict__ partial, int64_t np,
                                                                 int* __restrict__ total_out) {
    __shared__ int s_tot[kScanThreads / 64];
    int carry = 0;
    for (int64_t c0 = 0; c0 < np; c0 += kScanChunk) {
        int v[kScanItems];
        int sum = 0;
        const int64_t base = c0 + (int64_t)threadIdx.x * kScanItems;
#pragma unroll
        for (int k = 0; k < kScanItems; ++k) {
            const int64_t i = base + k;
            v[k] = i < np ? partial[i] : 0;
            sum += v[k];
        }
        int excl;
        const int total = block_excl_scan(sum, s_tot, excl);
        int run = carry + excl;
#pragma unroll
        for (int k = 0; k < kScanItems; ++k) {
            const int64_t i = base + k;
            if (i < np) partial[i] = run;
            run += v[k];
        }
        carry += total;
        __syncthreads();
    }
    if (threadIdx.x == 0 && total_out) *total_out = carry;
}

// SCANNED: partial[b] is what comes before chunk b; otherwise the chunk sums.
template <bool SCANNED>
__global__ __launch_bounds__(kScanThreads) void k_scan_apply(int* __restrict__ data, int64_t n,
                                                              const int* __restrict__ partial,
                                                              int* __restrict__ total_out) {
    __shared__ int s_tot[kScanThreads / 64];
    int before = 0;
    if constexpr (SCANNED) {
        before = partial[blockIdx.x];
    } else {
        int mine[kScanItems];
#pragma unroll
        for (int k = 0; k < kScanItems; ++k) {
            const unsigned i = (unsigned)k * kScanThreads + threadIdx.x;
            mine[k] = i < blockIdx.x ? partial[i] : 0;
        }
#pragma unroll
        for (int k = 1; k < kScanItems; ++k) mine[0] += mine[k];
        int unused;
        before = block_excl_scan(mine[0], s_tot, unused);
    }
    const int64_t base = (int64_t)blockIdx.x * kScanChunk + (int64_t)threadIdx.x * kScanItems;
    int v[kScanItems];
    int sum = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        const int64_t i = base + k;
        v[k] = i < n ? data[i] : 0;
        sum += v[k];
    }
    int excl;
    const int total = block_excl_scan(sum, s_tot, excl);
    if (!SCANNED && total_out && blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) *total_out = before + total;
    int run = before + excl;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        const int64_t i = base + k;
        if (i < n) data[i] = run;
        run += v[k];
    }
}

}  // namespace

__global__ void k_fill_i32(int* __restrict__ p, int64_t n, int v) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

int64_t scan_partials_needed(int64_t n) { return n <= 0 ? 0 : (n + kScanChunk - 1) / kScanChunk; }

// In-place exclusive scan of d_data[0..n) with caller-provided partials
// (scan_partials_needed(n) ints); the grand total goes to *d_total (device
// pointer, may be null).  Asynchronous: the partials are in use until the
// stream reaches the end of the launches.  Totals must fit int32 (checked by
// callers).
int scan_exclusive_i32_ws(int* d_data, int64_t n, int* d_total, int* d_partial, hipStream_t s) {
    if (n <= 0) {
        if (d_total) hipLaunchKernelGGL(k_fill_i32, dim3(1), dim3(64), 0, s, d_total, (int64_t)1, 0);
        SPC5_HIP_TRY(hipGetLastError());
        return SPC5_HIP_OK;
    }
    const int64_t nblk = scan_partials_needed(n);
    hipLaunchKernelGGL(k_scan_reduce, dim3((unsigned)nblk), dim3(kScanThreads), 0, s, d_data, n, d_partial);
    SPC5_HIP_TRY(hipGetLastError());
    if (nblk <= kScanChunk) {
        hipLaunchKernelGGL(k_scan_apply<false>, dim3((unsigned)nblk), dim3(kScanThreads), 0, s, d_data, n, d_partial,
                           d_total);
    } else {
        hipLaunchKernelGGL(k_scan_partials, dim3(1), dim3(kScanThreads), 0, s, d_partial, nblk, d_total);
        SPC5_HIP_TRY(hipGetLastError());
        hipLaunchKernelGGL(k_scan_apply<true>, dim3((unsigned)nblk), dim3(kScanThreads), 0, s, d_data, n, d_partial,
                           nullptr);
    }
    SPC5_HIP_TRY(hipGetLastError());
    return SPC5_HIP_OK;
}

}  // namespace spc5
