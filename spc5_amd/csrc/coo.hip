// coo.hip -- COO -> CSR on the GPU and the MatrixMarket coordinate reader.
//
// spc5_hip_coo_to_csr does what the reference's COO_unsorted_to_CSR /
// COO_sorted_to_CSR do (src/spc5.hpp:77-114) with the GPU: entries are
// ordered by (row, column), stably.  Short rows are counted, filled and ranked
// (see "rows of few entries"); otherwise a radix sort of 64-bit keys
// (row << 32 | column; hipCUB) orders them, the row pointers come from a binary
// search of every row's first key in the sorted keys, and columns and values
// are gathered through the sort's permutation.  Duplicate (row, column) entries
// are kept, in input order, as the reference keeps them.  With `sorted` set
// the sort is skipped and the order is checked instead (the reference
// trusts it).  Every index is range-checked.
//
// spc5_hip_mm_info / spc5_hip_mm_read parse a MatrixMarket coordinate file
// (real, integer or pattern; general, symmetric or skew-symmetric) into
// 0-based COO arrays with the mirrored entries of symmetric files appended
// after each stored one, as examples/load_mm_and_compare.cpp:287-428 reads
// it (the sort that follows there is spc5_hip_coo_to_csr here).
#include "spc5_mat.hpp"

#include <hipcub/hipcub.hpp>

#include <cctype>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

using namespace spc5;

namespace {

__global__ void k_coo_keys(const int* __restrict__ ri, const int* __restrict__ cj, int64_t nnz, int64_t nrows,
                           int64_t ncols, unsigned long long* __restrict__ keys, int* __restrict__ perm,
                           int* __restrict__ err) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nnz) return;
    const int r = ri[t], c = cj[t];
    if (r < 0 || (int64_t)r >= nrows || c < 0 || (int64_t)c >= ncols) atomicOr(err, 1);
    keys[t] = ((unsigned long long)(unsigned)r << 32) | (unsigned)c;
    perm[t] = (int)t;
}

// err |= 2 where keys[t-1] > keys[t] (input said to be sorted but is not).
__global__ void k_check_sorted(const unsigned long long* __restrict__ keys, int64_t nnz, int* __restrict__ err) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x + 1;
    if (t >= nnz) return;
    if (keys[t - 1] > keys[t]) atomicOr(err, 2);
}

// rowptr[r] = number of keys below (r << 32), r = 0 .. nrows.
__global__ void k_rowptr_search(const unsigned long long* __restrict__ keys, int64_t nnz, int64_t nrows,
                                int* __restrict__ rowptr) {
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r > nrows) return;
    const unsigned long long key = (unsigned long long)r << 32;
    int64_t lo = 0, hi = nnz;
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (keys[mid] < key) lo = mid + 1;
        else hi = mid;
    }
    rowptr[r] = (int)lo;
}

template <class T>
__global__ void k_coo_gather(const unsigned long long* __restrict__ keys, const int* __restrict__ perm,
                             const T* __restrict__ v, int64_t nnz, int* __restrict__ col, T* __restrict__ val) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nnz) return;
    col[t] = (int)(keys[t] & 0xffffffffull);
    val[t] = v[perm ? perm[t] : t];
}

// ---- rows of few entries -----------------------------------------------------
//
// Most matrices have short rows, and ordering (row, column) keys of 64 bits
// with a radix sort reads and writes every entry once per 8 key bits.  Here the
// rows are the buckets: entries count themselves into their row (the count a
// counter returns is the entry's place in it), the scanned counts are the row
// pointers, every entry writes (column, input position) to its place, and then
// finds its rank among its row's keys by comparing with each of them, which
// gives the stable order whatever order the counters were reached in.  Three
// passes over the entries and one comparison per pair of entries of a row: the
// pairs bound it, so rows of more than kShortRow entries go to the radix sort
// (coo_short_rows decides on the mean; a longer row found on the way sends the
// whole matrix there).  1.25 M entries in 50 K rows: 462 us with the radix
// sort, 155 us.
constexpr int kShortRow = 1024;

// Counts per row (rowptr, cleared before) and every entry's place in its row.
// Counters in memory take an atomic per entry, 22 G/s at best and a third of it
// where neighbouring entries share a row; for matrices of many entries see
// k_coo_count_ranges.
__global__ __launch_bounds__(256) void k_coo_count(const int* __restrict__ ri, int64_t nnz, int64_t nrows,
                                                   int* __restrict__ count, int* __restrict__ place,
                                                   int* __restrict__ err) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nnz) return;
    const int r = ri[t];
    if (r < 0 || (int64_t)r >= nrows) {
        atomicOr(err, 1);
        place[t] = -1;
        return;
    }
    const int p = atomicAdd(&count[r], 1);
    if (p >= kShortRow) atomicOr(err, 4);
    place[t] = p;
}

// The counters in LDS: workgroup (c, g) takes chunk c of the entries and counts
// those whose row lies in range g of kRangeRows rows, 16 bits a counter; a place
// is then one in its chunk, and k_coo_bases turns the chunks' counts into each
// chunk's first place per row.  Every range reads all rows again and the counts
// pass through memory, so counters in memory stay for few entries (112 K: the
// same 80 us) and for more than kMaxRanges ranges (at 31 ranges, 5 M shuffled
// entries, the same 565 us).  Whole call, shuffled and in order: 260 K entries in
// 20 K rows 98 / 90 -> 91 / 84 us, 1.25 M in 50 K 184 / 186 -> 155 / 114, 9.5 M in
// 300 K 1037 / 1080 -> 916 / 513.
constexpr int kRangeRows = 32768;
constexpr int kMaxRanges = 32;
constexpr int kRangeThreads = 1024;
constexpr int64_t kChunkEntries = 16384;
constexpr int64_t kRangeEntries = 1 << 17;

struct CooChunks {
    int64_t entries = 0;  // per chunk, a multiple of 256 (0: counters in memory)
    int chunks = 0, ranges = 0;
    int64_t words = 0;    // of two counters, per chunk
    size_t bytes() const { return sizeof(unsigned) * (size_t)words * (size_t)chunks; }
};
CooChunks coo_chunks(int64_t nrows, int64_t nnz) {
    CooChunks k;
    if (nnz < kRangeEntries || nrows > (int64_t)kMaxRanges * kRangeRows) return k;
    k.ranges = (int)((nrows + kRangeRows - 1) / kRangeRows);
    const int64_t most = 512 / k.ranges;  // two workgroups per CU, and at most 32 MiB of counts
    int64_t n = (nnz + kChunkEntries - 1) / kChunkEntries;
    if (n > most) n = most;
    k.entries = ((nnz + n - 1) / n + 255) / 256 * 256;
    k.chunks = (int)((nnz + k.entries - 1) / k.entries);
    k.words = (nrows + 1) / 2;
    return k;
}

__global__ __launch_bounds__(kRangeThreads) void k_coo_count_ranges(const int* __restrict__ ri, int64_t nnz,
                                                                    int64_t nrows, int64_t entries, int64_t words,
                                                                    unsigned* __restrict__ counts,
                                                                    int* __restrict__ place, int* __restrict__ err) {
    constexpr int U = 4;
    __shared__ unsigned h[kRangeRows / 2];
    for (int i = threadIdx.x; i < kRangeRows / 2; i += kRangeThreads) h[i] = 0u;
    __syncthreads();
    const int64_t b = (int64_t)blockIdx.x * entries;
    const int64_t e = b + entries < nnz ? b + entries : nnz;
    const int64_t row0 = (int64_t)blockIdx.y * kRangeRows;
    int bad = 0;
    for (int64_t t0 = b + threadIdx.x; t0 < e; t0 += U * kRangeThreads) {
        int r[U];
#pragma unroll
        for (int u = 0; u < U; ++u) r[u] = ri[t0 + u * kRangeThreads < e ? t0 + u * kRangeThreads : e - 1];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t t = t0 + u * kRangeThreads;
            if (t >= e) continue;
            if (r[u] < 0 || (int64_t)r[u] >= nrows) {
                bad |= 1;
            } else if (r[u] >= row0 && r[u] < row0 + kRangeRows) {
                const unsigned l = (unsigned)(r[u] - row0), sh = 16u * (l & 1u);
                const int p = (int)((atomicAdd(&h[l >> 1], 1u << sh) >> sh) & 0xffffu);
                if (p >= kShortRow) bad |= 4;
                place[t] = p;
            }
        }
    }
    if (bad) atomicOr(err, bad);
    __syncthreads();
    const int64_t w0 = row0 / 2;
    unsigned* out = counts + (int64_t)blockIdx.x * words + w0;
    for (int i = threadIdx.x; i < kRangeRows / 2 && w0 + i < words; i += kRangeThreads) out[i] = h[i];
}

// Counts of the chunks -> each chunk's first place in every row (in place), and
// the rows' counts; rowptr[nrows] = 0.
__global__ __launch_bounds__(256) void k_coo_bases(unsigned* __restrict__ counts, int64_t words, int chunks,
                                                   int64_t nrows, int* __restrict__ rowptr, int* __restrict__ err) {
    constexpr int U = 8;
    const int64_t w = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (w >= words) return;
    unsigned lo = 0, hi = 0;
    for (int c0 = 0; c0 < chunks; c0 += U) {
        unsigned n[U];
#pragma unroll
        for (int u = 0; u < U; ++u) n[u] = counts[(int64_t)(c0 + u < chunks ? c0 + u : chunks - 1) * words + w];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (c0 + u >= chunks) continue;
            counts[(int64_t)(c0 + u) * words + w] = (lo & 0xffffu) | (hi << 16);
            lo += n[u] & 0xffffu;
            hi += n[u] >> 16;
        }
    }
    if (lo > (unsigned)kShortRow || hi > (unsigned)kShortRow) atomicOr(err, 4);
    rowptr[2 * w] = (int)lo;
    if (2 * w + 1 < nrows) rowptr[2 * w + 1] = (int)hi;
    if (w == 0) rowptr[nrows] = 0;
}

// keys[row pointer + place] = (column, input position).  Does nothing after an
// error (the counts may then not add up).
__global__ __launch_bounds__(256) void k_coo_place(const int* __restrict__ ri, const int* __restrict__ cj, int64_t nnz,
                                                   int64_t ncols, const int* __restrict__ rowptr,
                                                   const int* __restrict__ place, const unsigned* __restrict__ bases,
                                                   int64_t words, int64_t entries,
                                                   unsigned long long* __restrict__ keys,
                                                   const int* __restrict__ counted, int* __restrict__ err) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nnz || *counted != 0) return;
    const int r = ri[t], c = cj[t];
    int p = place[t];
    if (bases) {
        const int64_t chunk = (int64_t)blockIdx.x * 256 / entries;  // entries is a multiple of 256
        p += (int)((bases[chunk * words + (r >> 1)] >> (16 * (r & 1))) & 0xffffu);
    }
    if (c < 0 || (int64_t)c >= ncols) atomicOr(err, 1);
    keys[(int64_t)rowptr[r] + p] = ((unsigned long long)(unsigned)c << 32) | (unsigned)t;
}

// Every entry to its rank in its row.  Does nothing after an error or a long row.
template <class T>
__global__ __launch_bounds__(256) void k_coo_rank(const int* __restrict__ ri, int64_t nnz,
                                                  const int* __restrict__ rowptr,
                                                  const unsigned long long* __restrict__ keys,
                                                  const T* __restrict__ v, const int* __restrict__ err,
                                                  int* __restrict__ col, T* __restrict__ val) {
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= nnz || (err[0] | err[1]) != 0) return;
    const unsigned long long mine = keys[e];
    const unsigned t = (unsigned)mine;
    const int r = ri[t];
    const T value = v[t];
    const int b = rowptr[r], n = rowptr[r + 1] - b;
    const unsigned long long* k = keys + b;
    int rank = 0, i = 0;
    for (; i + 4 <= n; i += 4) {
        const unsigned long long k0 = k[i], k1 = k[i + 1], k2 = k[i + 2], k3 = k[i + 3];
        rank += (k0 < mine ? 1 : 0) + (k1 < mine ? 1 : 0) + (k2 < mine ? 1 : 0) + (k3 < mine ? 1 : 0);
    }
    for (; i < n; ++i) rank += k[i] < mine ? 1 : 0;
    col[(int64_t)b + rank] = (int)(mine >> 32);
    val[(int64_t)b + rank] = value;
}

// Whether the rows are short on average.
bool coo_short_rows(int64_t nrows, int64_t nnz) { return nnz > 0 && nnz / 96 <= nrows; }

size_t align256(size_t b) { return (b + 255) / 256 * 256; }

// Workspace of the short-row path: flags (of the counts, of the columns), scan
// partials, places, the chunks' counts, keys.
size_t coo_short_bytes(int64_t nrows, int64_t nnz) {
    return 256 + align256(sizeof(int) * (size_t)scan_partials_needed(nrows + 1)) + align256(sizeof(int) * (size_t)nnz) +
           sizeof(unsigned long long) * (size_t)nnz + align256(coo_chunks(nrows, nnz).bytes());
}

unsigned grid_of(int64_t n) { return (unsigned)((n + 255) / 256); }

// The short-row path in a workspace of coo_short_bytes; *flags: as `err` of the
// kernels (4: a long row was found and nothing was written but the row
// pointers).
int coo_short(int value_bytes, int64_t nrows, int64_t ncols, int64_t nnz, const int* d_i, const int* d_j,
              const void* d_v, int* d_rowptr, int* d_col, void* d_val, void* ws, int* flags, hipStream_t s) {
    unsigned char* w = reinterpret_cast<unsigned char*>(ws);
    int* err = reinterpret_cast<int*>(w);
    int* partials = reinterpret_cast<int*>(w + 256);
    w += 256 + align256(sizeof(int) * (size_t)scan_partials_needed(nrows + 1));
    int* place = reinterpret_cast<int*>(w);
    w += align256(sizeof(int) * (size_t)nnz);
    const CooChunks k = coo_chunks(nrows, nnz);
    unsigned* counts = k.entries ? reinterpret_cast<unsigned*>(w) : nullptr;
    unsigned long long* keys = reinterpret_cast<unsigned long long*>(w + align256(k.bytes()));
    hipLaunchKernelGGL(k_fill_i32, dim3(1), dim3(256), 0, s, err, (int64_t)2, 0);
    if (k.entries) {
        hipLaunchKernelGGL(k_coo_count_ranges, dim3((unsigned)k.chunks, (unsigned)k.ranges), dim3(kRangeThreads), 0, s,
                           d_i, nnz, nrows, k.entries, k.words, counts, place, err);
        hipLaunchKernelGGL(k_coo_bases, dim3(grid_of(k.words)), dim3(256), 0, s, counts, k.words, k.chunks, nrows,
                           d_rowptr, err);
    } else {
        hipLaunchKernelGGL(k_fill_i32, dim3(grid_of(nrows + 1)), dim3(256), 0, s, d_rowptr, nrows + 1, 0);
        hipLaunchKernelGGL(k_coo_count, dim3(grid_of(nnz)), dim3(256), 0, s, d_i, nnz, nrows, d_rowptr, place, err);
    }
    SPC5_HIP_TRY(hipGetLastError());
    const int rc = scan_exclusive_i32_ws(d_rowptr, nrows + 1, nullptr, partials, s);
    if (rc) return rc;
    hipLaunchKernelGGL(k_coo_place, dim3(grid_of(nnz)), dim3(256), 0, s, d_i, d_j, nnz, ncols, d_rowptr, place,
                       (const unsigned*)counts, k.words, k.entries, keys, (const int*)err, err + 1);
    if (value_bytes == 8)
        hipLaunchKernelGGL(k_coo_rank<double>, dim3(grid_of(nnz)), dim3(256), 0, s, d_i, nnz, d_rowptr, keys,
                           reinterpret_cast<const double*>(d_v), err, d_col, reinterpret_cast<double*>(d_val));
    else
        hipLaunchKernelGGL(k_coo_rank<float>, dim3(grid_of(nnz)), dim3(256), 0, s, d_i, nnz, d_rowptr, keys,
                           reinterpret_cast<const float*>(d_v), err, d_col, reinterpret_cast<float*>(d_val));
    SPC5_HIP_TRY(hipGetLastError());
    int h[2] = {0, 0};
    SPC5_HIP_TRY(hipMemcpyAsync(h, err, sizeof(h), hipMemcpyDeviceToHost, s));
    SPC5_HIP_TRY(hipStreamSynchronize(s));
    *flags = h[0] | h[1];
    return SPC5_HIP_OK;
}

bool overlap(const void* a, size_t na, const void* b, size_t nb) {
    const uintptr_t x = (uintptr_t)a, y = (uintptr_t)b;
    return na > 0 && nb > 0 && x < y + nb && y < x + na;
}

int coo_range_error() {
    set_error("COO index out of range (row not in [0, nrows) or column not in [0, ncols))");
    return SPC5_HIP_ERR_INVALID;
}

int coo_to_csr(int value_bytes, int64_t nrows, int64_t ncols, int64_t nnz, bool sorted, const int* d_i,
               const int* d_j, const void* d_v, int* d_rowptr, int* d_col, void* d_val, void* ws, hipStream_t s) {
    // The short-row path reads the rows to the end, so outputs over inputs take
    // the radix sort, which reads rows and columns first.
    const size_t in = sizeof(int) * (size_t)nnz, vb = (size_t)value_bytes * (size_t)nnz;
    const size_t rb = sizeof(int) * (size_t)(nrows + 1);
    const bool apart = !overlap(d_rowptr, rb, d_i, in) && !overlap(d_rowptr, rb, d_j, in) &&
                       !overlap(d_rowptr, rb, d_v, vb) && !overlap(d_col, in, d_i, in) &&
                       !overlap(d_col, in, d_v, vb) && !overlap(d_val, vb, d_i, in) && !overlap(d_val, vb, d_v, vb);
    if (!sorted && apart && coo_short_rows(nrows, nnz)) {
        DeviceBuffer own;
        if (!ws) {
            SPC5_HIP_TRY(own.alloc(coo_short_bytes(nrows, nnz)));
            ws = own.p;
        }
        int flags = 0;
        const int rc = coo_short(value_bytes, nrows, ncols, nnz, d_i, d_j, d_v, d_rowptr, d_col, d_val, ws, &flags, s);
        if (rc) return rc;
        if (flags & 1) return coo_range_error();
        if (!(flags & 4)) return SPC5_HIP_OK;
    }
    DeviceBuffer err;
    SPC5_HIP_TRY(err.alloc(sizeof(int)));
    SPC5_HIP_TRY(hipMemsetAsync(err.p, 0, sizeof(int), s));
    const size_t n = (size_t)std::max<int64_t>(nnz, 1);
    DeviceBuffer keys_a, keys_b, perm_a, perm_b;
    SPC5_HIP_TRY(keys_a.alloc(sizeof(unsigned long long) * n));
    SPC5_HIP_TRY(perm_a.alloc(sizeof(int) * n));
    unsigned long long* keys = keys_a.as<unsigned long long>();
    int* perm = perm_a.as<int>();
    if (nnz > 0) {
        hipLaunchKernelGGL(k_coo_keys, dim3(grid_of(nnz)), dim3(256), 0, s, d_i, d_j, nnz, nrows, ncols, keys, perm,
                           err.as<int>());
        SPC5_HIP_TRY(hipGetLastError());
    }
    if (sorted) {
        if (nnz > 1) {
            hipLaunchKernelGGL(k_check_sorted, dim3(grid_of(nnz - 1)), dim3(256), 0, s, keys, nnz, err.as<int>());
            SPC5_HIP_TRY(hipGetLastError());
        }
        perm = nullptr;
    } else if (nnz > 1) {
        SPC5_HIP_TRY(keys_b.alloc(sizeof(unsigned long long) * n));
        SPC5_HIP_TRY(perm_b.alloc(sizeof(int) * n));
        int end_bit = 32;
        while (end_bit < 64 && ((unsigned long long)nrows >> (end_bit - 32)) != 0) ++end_bit;
        size_t tmp_bytes = 0;
        SPC5_HIP_TRY(hipcub::DeviceRadixSort::SortPairs(nullptr, tmp_bytes, keys, keys_b.as<unsigned long long>(),
                                                        perm, perm_b.as<int>(), (int)nnz, 0, end_bit, s));
        DeviceBuffer tmp;
        SPC5_HIP_TRY(tmp.alloc(std::max<size_t>(tmp_bytes, 1)));
        SPC5_HIP_TRY(hipcub::DeviceRadixSort::SortPairs(tmp.p, tmp_bytes, keys, keys_b.as<unsigned long long>(), perm,
                                                        perm_b.as<int>(), (int)nnz, 0, end_bit, s));
        keys = keys_b.as<unsigned long long>();
        perm = perm_b.as<int>();
        SPC5_HIP_TRY(hipStreamSynchronize(s));  // the sort's scratch is freed on return
    }
    hipLaunchKernelGGL(k_rowptr_search, dim3(grid_of(nrows + 1)), dim3(256), 0, s, keys, nnz, nrows, d_rowptr);
    SPC5_HIP_TRY(hipGetLastError());
    if (nnz > 0) {
        if (value_bytes == 8)
            hipLaunchKernelGGL(k_coo_gather<double>, dim3(grid_of(nnz)), dim3(256), 0, s, keys, perm,
                               reinterpret_cast<const double*>(d_v), nnz, d_col, reinterpret_cast<double*>(d_val));
        else
            hipLaunchKernelGGL(k_coo_gather<float>, dim3(grid_of(nnz)), dim3(256), 0, s, keys, perm,
                               reinterpret_cast<const float*>(d_v), nnz, d_col, reinterpret_cast<float*>(d_val));
        SPC5_HIP_TRY(hipGetLastError());
    }
    int herr = 0;
    SPC5_HIP_TRY(hipMemcpyAsync(&herr, err.p, sizeof(int), hipMemcpyDeviceToHost, s));
    SPC5_HIP_TRY(hipStreamSynchronize(s));
    if (herr & 1) return coo_range_error();
    if (herr & 2) {
        set_error("COO entries not sorted by (row, column)");
        return SPC5_HIP_ERR_INVALID;
    }
    return SPC5_HIP_OK;
}

// ---- MatrixMarket ----------------------------------------------------------

struct MMFile {
    std::string text;
    size_t pos = 0;
    int64_t nrows = 0, ncols = 0, nstored = 0;
    bool symmetric = false, skew = false, pattern = false, integer = false;
};

bool read_file(const char* path, std::string& out) {
    FILE* f = std::fopen(path, "rb");
    if (!f) return false;
    std::fseek(f, 0, SEEK_END);
    const long sz = std::ftell(f);
    std::fseek(f, 0, SEEK_SET);
    out.resize(sz > 0 ? (size_t)sz : 0);
    const size_t got = sz > 0 ? std::fread(&out[0], 1, (size_t)sz, f) : 0;
    std::fclose(f);
    return got == out.size();
}

std::string lower(std::string s) {
    for (char& c : s) c = (char)std::tolower((unsigned char)c);
    return s;
}

int mm_open(const char* path, MMFile& mm) {
    SPC5_CHECK_ARG(path != nullptr, "null path");
    if (!read_file(path, mm.text)) {
        set_error(std::string("cannot read ") + path);
        return SPC5_HIP_ERR_INVALID;
    }
    const std::string& t = mm.text;
    size_t eol = t.find('\n');
    const std::string head = lower(t.substr(0, eol));
    char w[5][64] = {};
    if (std::sscanf(head.c_str(), "%63s %63s %63s %63s %63s", w[0], w[1], w[2], w[3], w[4]) != 5 ||
        std::strcmp(w[0], "%%matrixmarket") != 0 || std::strcmp(w[1], "matrix") != 0 ||
        std::strcmp(w[2], "coordinate") != 0) {
        set_error("not a MatrixMarket coordinate matrix header");
        return SPC5_HIP_ERR_INVALID;
    }
    const std::string field = w[3], sym = w[4];
    if (field != "real" && field != "integer" && field != "pattern") {
        set_error("only real, integer and pattern MatrixMarket matrices are supported (" + field + " given)");
        return SPC5_HIP_ERR_INVALID;
    }
    if (sym != "general" && sym != "symmetric" && sym != "skew-symmetric") {
        set_error("unsupported MatrixMarket symmetry " + sym);
        return SPC5_HIP_ERR_INVALID;
    }
    mm.pattern = field == "pattern";
    mm.integer = field == "integer";
    mm.symmetric = sym == "symmetric";
    mm.skew = sym == "skew-symmetric";
    size_t p = eol == std::string::npos ? t.size() : eol + 1;
    while (p < t.size() && t[p] == '%') {  // comment lines
        const size_t e = t.find('\n', p);
        p = e == std::string::npos ? t.size() : e + 1;
    }
    char* end = nullptr;
    const char* c = t.c_str() + p;
    mm.nrows = std::strtoll(c, &end, 10);
    mm.ncols = std::strtoll(end, &end, 10);
    mm.nstored = std::strtoll(end, &end, 10);
    if (end == c || mm.nrows < 0 || mm.ncols < 0 || mm.nstored < 0) {
        set_error("bad MatrixMarket size line");
        return SPC5_HIP_ERR_INVALID;
    }
    mm.pos = (size_t)(end - t.c_str());
    return SPC5_HIP_OK;
}

// Walks the stored entries; emit(i, j, v) for each entry of the matrix
// (mirrored entries right after their stored one).  Returns the count, or -1
// on a malformed or out-of-range entry.
template <class Emit>
int64_t mm_walk(const MMFile& mm, Emit&& emit) {
    const char* c = mm.text.c_str() + mm.pos;
    int64_t count = 0;
    for (int64_t k = 0; k < mm.nstored; ++k) {
        char* end = nullptr;
        const long long row = std::strtoll(c, &end, 10);
        if (end == c) return -1;
        c = end;
        const long long col = std::strtoll(c, &end, 10);
        if (end == c) return -1;
        c = end;
        double v = 1.0;
        if (!mm.pattern) {
            v = mm.integer ? (double)std::strtoll(c, &end, 10) : std::strtod(c, &end);
            if (end == c) return -1;
            c = end;
        }
        if (row < 1 || row > mm.nrows || col < 1 || col > mm.ncols) return -1;
        const int i = (int)(row - 1), j = (int)(col - 1);
        emit(count++, i, j, v);
        if ((mm.symmetric || mm.skew) && i != j) emit(count++, j, i, mm.skew ? -v : v);
    }
    return count;
}

}  // namespace

extern "C" {

int64_t spc5_hip_coo_workspace_bytes(int64_t nrows, int64_t nnz, int sorted) {
    return !sorted && nrows >= 0 && coo_short_rows(nrows, nnz) ? (int64_t)coo_short_bytes(nrows, nnz) : 0;
}

int spc5_hip_coo_to_csr_ws(int value_bytes, int64_t nrows, int64_t ncols, int64_t nnz, int sorted, const int* d_i,
                           const int* d_j, const void* d_v, int* d_rowptr, int* d_col, void* d_val, void* d_workspace,
                           int64_t workspace_bytes, void* stream) {
    SPC5_CHECK_ARG(value_bytes == 8 || value_bytes == 4, "value_bytes must be 8 or 4");
    SPC5_CHECK_ARG(nrows >= 0 && ncols >= 0 && nnz >= 0, "negative size");
    SPC5_CHECK_ARG(nrows < ((int64_t)1 << 31) && ncols < ((int64_t)1 << 31) && nnz < ((int64_t)1 << 31),
                   "sizes must fit the 32-bit CSR arrays");
    SPC5_CHECK_ARG(d_rowptr != nullptr, "null rowptr");
    SPC5_CHECK_ARG(nnz == 0 || (d_i && d_j && d_v && d_col && d_val), "null COO or CSR array");
    SPC5_CHECK_ARG(d_workspace == nullptr || ((uintptr_t)d_workspace % 256 == 0 &&
                                              workspace_bytes >= spc5_hip_coo_workspace_bytes(nrows, nnz, sorted)),
                   "workspace misaligned or too small");
    return coo_to_csr(value_bytes, nrows, ncols, nnz, sorted != 0, d_i, d_j, d_v, d_rowptr, d_col, d_val, d_workspace,
                      as_stream(stream));
}

int spc5_hip_coo_to_csr(int value_bytes, int64_t nrows, int64_t ncols, int64_t nnz, int sorted, const int* d_i,
                        const int* d_j, const void* d_v, int* d_rowptr, int* d_col, void* d_val, void* stream) {
    return spc5_hip_coo_to_csr_ws(value_bytes, nrows, ncols, nnz, sorted, d_i, d_j, d_v, d_rowptr, d_col, d_val, nullptr,
                                  0, stream);
}

int spc5_hip_mm_info(const char* path, int64_t* nrows, int64_t* ncols, int64_t* nentries) {
    MMFile mm;
    const int rc = mm_open(path, mm);
    if (rc) return rc;
    const int64_t n = mm_walk(mm, [](int64_t, int, int, double) {});
    if (n < 0) {
        set_error("malformed or out-of-range MatrixMarket entry");
        return SPC5_HIP_ERR_INVALID;
    }
    if (nrows) *nrows = mm.nrows;
    if (ncols) *ncols = mm.ncols;
    if (nentries) *nentries = n;
    return SPC5_HIP_OK;
}

int spc5_hip_mm_read(const char* path, int64_t capacity, int* ri, int* cj, double* v, int64_t* nread) {
    SPC5_CHECK_ARG(capacity == 0 || (ri && cj && v), "null output array");
    MMFile mm;
    const int rc = mm_open(path, mm);
    if (rc) return rc;
    bool overflow = false;
    const int64_t n = mm_walk(mm, [&](int64_t k, int i, int j, double x) {
        if (k >= capacity) {
            overflow = true;
            return;
        }
        ri[k] = i;
        cj[k] = j;
        v[k] = x;
    });
    if (n < 0) {
        set_error("malformed or out-of-range MatrixMarket entry");
        return SPC5_HIP_ERR_INVALID;
    }
    if (overflow) {
        set_error("capacity below the number of entries (see spc5_hip_mm_info)");
        return SPC5_HIP_ERR_INVALID;
    }
    if (nread) *nread = n;
    return SPC5_HIP_OK;
}

}  // extern "C"
