// One-time integer graph preparation on the device: edge list -> canonical CSR,
// and the transposed (by-source) view of a CSR with the edge permutation that
// links the two orders. The backward kernels use the latter to turn
// scatter-adds into gathers.
//
// Both are bound by their radix sort, whose passes (8 bits each) move every key once more:
// the keys carry no bits but those of the ids (3.4 M edges over 200,000 ids: five passes of
// 33 us instead of eight). What stands around the sorts makes one streaming pass each.
#include <hip/hip_runtime.h>

#include <cstring>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

#include "../../include/yitu_hip.h"
#include "spmm_rows.hpp"

namespace yitu {

// last row whose edges begin at or before e (0 when there is none)
__device__ __forceinline__ int32_t row_of_edge(const int32_t *__restrict__ indptr, int32_t lo, int32_t hi,
                                               int32_t e) {
    while (hi - lo > 1) {  // indptr[lo] <= e < indptr[hi]
        const int32_t mid = lo + ((hi - lo) >> 1);
        if (indptr[mid] <= e) lo = mid; else hi = mid;
    }
    return lo;
}

// Sort operands (column, edge) and the row of every edge: the rows of a workgroup's 1,024
// edges are a short range of indptr, found by two searches, so that each edge's own search is
// a few steps in cache.
__global__ __launch_bounds__(kBlock) void transpose_keys_kernel(
    const int32_t *__restrict__ indptr, const int32_t *__restrict__ indices,
    int32_t *__restrict__ keys, int32_t *__restrict__ vals, int32_t *__restrict__ edge_row, int64_t nnz,
    int32_t n_rows, int col_mask) {
    constexpr int kEdges = 1024;
    __shared__ int32_t ends[2];
    const int64_t base = (int64_t)blockIdx.x * kEdges;
    const int64_t end = min(base + kEdges, nnz);
    if (threadIdx.x % kWave == 0 && threadIdx.x < 2 * kWave)
        ends[threadIdx.x / kWave] =
            row_of_edge(indptr, 0, n_rows, (int32_t)(threadIdx.x ? end - 1 : base));
    __syncthreads();
    const int32_t lo = ends[0], hi = ends[1] + 1;
    for (int64_t i = base + threadIdx.x; i < end; i += kBlock) {
        keys[i] = indices[i] & col_mask;
        vals[i] = (int32_t)i;
        edge_row[i] = row_of_edge(indptr, lo, hi, (int32_t)i);
    }
}

// starts[c] = at for c in (lo, hi], every lane with bounds of its own. Ranges are mostly one
// or two long; the long ones (ids without edges) are shared out over the wave.
__device__ __forceinline__ void fill_starts(int32_t *__restrict__ starts, int lo, int hi, int32_t at) {
    constexpr int kOwn = 4;
    for (int c = lo + 1; c <= min(hi, lo + kOwn); c++) starts[c] = at;
    unsigned long long left = __ballot(hi > lo + kOwn);
    while (left) {
        const int src = __ffsll(left) - 1;
        left &= left - 1;
        const int l = __shfl(lo, src, kWave) + kOwn, h = __shfl(hi, src, kWave);
        const int32_t v = __shfl(at, src, kWave);
        for (int64_t c = (int64_t)l + 1 + lane_id(); c <= h; c += kWave) starts[c] = v;
    }
}

// Sorted keys -> indptr of the transposed matrix (position j closes every column in
// (keys[j-1], keys[j]], empty columns included), and the row of every edge in that order.
// (A binary search in indptr for each of those rows took 104 us for 3 M edges, this pass 28.)
__global__ __launch_bounds__(kBlock) void transpose_finish_kernel(
    const int32_t *__restrict__ keys_sorted, const int32_t *__restrict__ t_perm,
    const int32_t *__restrict__ edge_row, int32_t *__restrict__ t_indptr,
    int32_t *__restrict__ t_rows, int64_t nnz, int32_t n_cols) {
    const int64_t j = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    int lo = 0, hi = 0;  // nothing to fill
    if (j <= nnz) {
        lo = j == 0 ? -1 : keys_sorted[j - 1];
        hi = j == nnz ? n_cols : min(keys_sorted[j], n_cols);
    }
    if (j < nnz) t_rows[j] = edge_row[t_perm[j]];
    fill_starts(t_indptr, lo, hi, (int32_t)j);
}

// ---- edge list -> canonical CSR ---------------------------------------------------
// Key of an edge: row << col_bits | col. An edge with an id outside the matrix gets the key of
// (n_rows, 0), behind every other.
template <typename Id, typename Key>
__global__ __launch_bounds__(kBlock) void coo_keys_kernel(const Id *__restrict__ rows,
                                                          const Id *__restrict__ cols,
                                                          Key *__restrict__ keys, int64_t n_edges,
                                                          int32_t n_rows, int32_t n_cols, int col_bits) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n_edges) return;
    const Id r = rows[i], c = cols[i];
    const bool good = r >= 0 && r < n_rows && c >= 0 && c < n_cols;
    keys[i] = good ? (Key)r << col_bits | (Key)c : (Key)n_rows << col_bits;
}

// The distinct keys of a sorted list, counted per chunk of 4,096 (of them the ones that stand
// for an edge), numbered by a prefix sum over the chunks, and written: three short passes
// (31 us for 3.4 M keys; a library's select and a search of indptr behind it: 63).
constexpr int kChunk = 4096, kPerThread = kChunk / kBlock;

template <typename Key>
__device__ __forceinline__ bool is_first(const Key *__restrict__ keys, int64_t i, Key limit) {
    const Key k = keys[i];
    return k < limit && (i == 0 || keys[i - 1] != k);
}

template <typename Key>
__global__ __launch_bounds__(kBlock) void coo_count_kernel(const Key *__restrict__ keys, Key limit,
                                                           int64_t n_edges, int32_t *__restrict__ counts) {
    __shared__ int sums[kWavesPerBlock];
    const int64_t base = (int64_t)blockIdx.x * kChunk;
    int n = 0;
#pragma unroll
    for (int k = 0; k < kPerThread; k++) {
        const int64_t i = base + k * kBlock + threadIdx.x;
        const bool first = i < n_edges && is_first(keys, i, limit);
        n += __popcll(__ballot(first));
    }
    if (lane_id() == 0) sums[threadIdx.x / kWave] = n;
    __syncthreads();
    if (threadIdx.x == 0) counts[blockIdx.x] = sums[0] + sums[1] + sums[2] + sums[3];
}

// Exclusive prefix sum of the chunk counts in place, by one workgroup; info = {distinct edges,
// or -1 when an id was outside, 0}.
template <typename Key>
__global__ __launch_bounds__(1024) void coo_starts_kernel(const Key *__restrict__ keys, Key limit,
                                                          int64_t n_edges, int32_t *__restrict__ counts,
                                                          int n_chunks, long long *__restrict__ info,
                                                          int32_t *__restrict__ total_out) {
    __shared__ int sums[16];
    const int lane = lane_id(), wave = threadIdx.x / kWave;
    int carry = 0;
    for (int base = 0; base < n_chunks; base += 1024) {
        const int i = base + threadIdx.x;
        const int v = i < n_chunks ? counts[i] : 0;
        int pre = v;
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) {
            const int x = __shfl_up(pre, o, kWave);
            if (lane >= o) pre += x;
        }
        if (lane == kWave - 1) sums[wave] = pre;
        __syncthreads();
        int before = carry, all = 0;
        for (int w = 0; w < 16; w++) {
            before += w < wave ? sums[w] : 0;
            all += sums[w];
        }
        if (i < n_chunks) counts[i] = before + pre - v;
        carry += all;
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const bool bad = n_edges > 0 && keys[n_edges - 1] >= limit;
        info[0] = bad ? -1 : carry;
        info[1] = 0;
        *total_out = carry;
    }
}

template <typename Key>
__global__ __launch_bounds__(kBlock) void coo_write_kernel(const Key *__restrict__ keys, Key limit,
                                                           int64_t n_edges,
                                                           const int32_t *__restrict__ starts,
                                                           const int32_t *__restrict__ total,
                                                           int col_bits, int32_t n_rows,
                                                           int32_t *__restrict__ indptr,
                                                           int32_t *__restrict__ indices) {
    __shared__ int sums[kPerThread][kWavesPerBlock];
    const int64_t base = (int64_t)blockIdx.x * kChunk;
    const int lane = lane_id(), wave = threadIdx.x / kWave;
    unsigned long long ballots[kPerThread];
#pragma unroll
    for (int k = 0; k < kPerThread; k++) {
        const int64_t i = base + k * kBlock + threadIdx.x;
        ballots[k] = __ballot(i < n_edges && is_first(keys, i, limit));
        if (lane == 0) sums[k][wave] = __popcll(ballots[k]);
    }
    __syncthreads();
    int at = starts[blockIdx.x];
#pragma unroll
    for (int k = 0; k < kPerThread; k++) {
        const int64_t i = base + k * kBlock + threadIdx.x;
        int own = at;
#pragma unroll
        for (int w = 0; w < kWavesPerBlock; w++) {
            own += w < wave ? sums[k][w] : 0;
            at += sums[k][w];
        }
        const bool first = ballots[k] >> lane & 1;
        own += __popcll(ballots[k] & ((1ull << lane) - 1));
        int lo = 0, hi = 0;
        if (first) {
            const Key key = keys[i];
            indices[own] = (int32_t)(key & (((Key)1 << col_bits) - 1));
            hi = (int32_t)(key >> col_bits);
            lo = i == 0 ? -1 : (int32_t)(keys[i - 1] >> col_bits);
        }
        fill_starts(indptr, lo, hi, own);
    }
    // the rows behind the last edge's: the last edge's thread would see them, but the edges
    // behind it may be copies or bad ones
    if (blockIdx.x == gridDim.x - 1) {
        const int64_t n = *total;
        int64_t last = -1;  // row of the last good key
        int64_t a = 0, b = n_edges;
        while (a < b) {  // first key that is no edge
            const int64_t mid = (a + b) >> 1;
            if (keys[mid] < limit) a = mid + 1; else b = mid;
        }
        if (a > 0) last = (int64_t)(keys[a - 1] >> col_bits);
        for (int64_t r = last + 1 + threadIdx.x; r <= n_rows; r += kBlock) indptr[r] = (int32_t)n;
    }
}

// info[1] = the longest row
__global__ __launch_bounds__(kBlock) void longest_row_kernel(const int32_t *__restrict__ indptr,
                                                             int64_t n_rows,
                                                             long long *__restrict__ longest) {
    __shared__ int most[kWavesPerBlock];
    int m = 0;
    for (int64_t r = (int64_t)blockIdx.x * kBlock + threadIdx.x; r < n_rows;
         r += (int64_t)gridDim.x * kBlock)
        m = max(m, indptr[r + 1] - indptr[r]);
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) m = max(m, __shfl_xor(m, o, kWave));
    if (lane_id() == 0) most[threadIdx.x / kWave] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        m = max(max(most[0], most[1]), max(most[2], most[3]));
        if (m > 0) atomicMax(longest, (long long)m);
    }
}

static int longest_row(const int32_t *indptr, int64_t n_rows, long long *longest, hipStream_t stream) {
    // few workgroups: each ends in an atomic on the same word
    const int grid = (int)std::min<int64_t>(std::max<int64_t>(ceil_div(n_rows, kBlock), 1), 256);
    longest_row_kernel<<<grid, kBlock, 0, stream>>>(indptr, n_rows, longest);
    YITU_LAUNCH_CHECK();
    return 0;
}

__global__ void set_word_kernel(long long *word, long long value) { *word = value; }

static int key_bits(int64_t n_cols) {
    int b = 1;
    while (((int64_t)1 << b) < n_cols) b++;
    return b;
}

// bits of the column and of the whole key, (n_rows, 0) among the keys
static int coo_col_bits(int64_t n_cols) { return key_bits(std::max<int64_t>(n_cols, 1)); }
static int coo_key_bits(int64_t n_rows, int64_t n_cols) {
    return key_bits(n_rows + 1) + coo_col_bits(n_cols);
}

template <typename Key>
static size_t coo_sort_bytes(int64_t n_edges, int bits) {
    size_t bytes = 0;
    Key *k = nullptr;
    (void)rocprim::radix_sort_keys(nullptr, bytes, k, k, (size_t)n_edges, 0, bits);
    return bytes;
}

// of either key width, the columns' share of the bits not being known when room is made
static size_t coo_temp_bytes(int64_t n_edges) {
    if (n_edges <= 0) return 0;
    return std::max(coo_sort_bytes<uint32_t>(n_edges, 32), coo_sort_bytes<uint64_t>(n_edges, 64));
}

static size_t sort_temp_bytes(int64_t nnz, int bits) {
    size_t bytes = 0;
    int32_t *k = nullptr;
    (void)rocprim::radix_sort_pairs(nullptr, bytes, k, k, k, k, (size_t)nnz, 0, bits);
    return bytes;
}

template <typename Id, typename Key>
static int coo_build(int32_t *indptr, int32_t *indices, long long *info, const Id *rows,
                     const Id *cols, int64_t n_edges, int64_t n_rows, int64_t n_cols, char *w,
                     size_t temp_bytes, hipStream_t stream) {
    const int col_bits = coo_col_bits(n_cols), bits = coo_key_bits(n_rows, n_cols);
    const Key limit = (Key)n_rows << col_bits;
    const int n_chunks = (int)std::max<int64_t>(ceil_div(n_edges, kChunk), 1);
    int32_t *total = reinterpret_cast<int32_t *>(w);
    int32_t *counts = reinterpret_cast<int32_t *>(w + 256);
    w += 256 + align_up(sizeof(int32_t) * (size_t)n_chunks, 256);
    const size_t arr = align_up(sizeof(Key) * (size_t)n_edges, 256);
    Key *keys = reinterpret_cast<Key *>(w), *sorted = reinterpret_cast<Key *>(w + arr);
    if (n_edges > 0) {
        coo_keys_kernel<<<(int)ceil_div(n_edges, kBlock), kBlock, 0, stream>>>(
            rows, cols, keys, n_edges, (int32_t)n_rows, (int32_t)n_cols, col_bits);
        YITU_LAUNCH_CHECK();
        size_t bytes = coo_sort_bytes<Key>(n_edges, bits);
        YITU_REQUIRE(bytes <= temp_bytes, "sort scratch too small: need %zu bytes", bytes);
        YITU_HIP(rocprim::radix_sort_keys(w + 2 * arr, bytes, keys, sorted, (size_t)n_edges, 0, bits,
                                          stream));
    }
    coo_count_kernel<<<n_chunks, kBlock, 0, stream>>>(sorted, limit, n_edges, counts);
    YITU_LAUNCH_CHECK();
    coo_starts_kernel<<<1, 1024, 0, stream>>>(sorted, limit, n_edges, counts, n_chunks, info, total);
    YITU_LAUNCH_CHECK();
    coo_write_kernel<<<n_chunks, kBlock, 0, stream>>>(sorted, limit, n_edges, counts, total, col_bits,
                                                      (int32_t)n_rows, indptr, indices);
    YITU_LAUNCH_CHECK();
    return longest_row(indptr, n_rows, info + 1, stream);
}

}  // namespace yitu

namespace yitu {
namespace {

// groups of row r = ceil(deg / part_size)
__global__ __launch_bounds__(kBlock) void part_count_kernel(int32_t *__restrict__ count,
                                                            const int32_t *__restrict__ indptr,
                                                            int n_rows, int part_size) {
    const int r = blockIdx.x * kBlock + threadIdx.x;
    if (r < n_rows) count[r] = (indptr[r + 1] - indptr[r] + part_size - 1) / part_size;
}

// One wave per row: group g of row r starts at edge indptr[r] + g part_size. The entry
// behind the last group is the number of edges when the last row has edges and 0
// otherwise, as the reference leaves it (YiTu_GNN.cpp:240-241).
__global__ __launch_bounds__(kBlock) void part_fill_kernel(
    int32_t *__restrict__ part_ptr, int32_t *__restrict__ part2node, long long *__restrict__ n_parts,
    const int32_t *__restrict__ first, const int32_t *__restrict__ count,
    const int32_t *__restrict__ indptr, int n_rows, int part_size, long long capacity) {
    const int lane = threadIdx.x & (kWave - 1);
    const int r = blockIdx.x * kWavesPerBlock + threadIdx.x / kWave;
    if (r >= n_rows) return;
    const int base = first[r], n = count[r], beg = indptr[r];
    for (int g = lane; g < n; g += kWave) {
        if (base + g < capacity) {
            part_ptr[base + g] = beg + g * part_size;
            part2node[base + g] = r;
        }
    }
    if (r == n_rows - 1 && lane == 0) {
        const long long total = (long long)base + n;
        *n_parts = total;
        if (total < capacity + 1) part_ptr[total] = n > 0 ? indptr[n_rows] : 0;
    }
}

size_t part_scan_bytes(int64_t n_rows) {
    size_t bytes = 0;
    int32_t *p = nullptr;
    (void)rocprim::exclusive_scan(nullptr, bytes, p, p, 0, (size_t)std::max<int64_t>(n_rows, 1),
                                  rocprim::plus<int32_t>());
    return bytes;
}

}  // namespace
}  // namespace yitu

using namespace yitu;
#define YITU_API extern "C" __attribute__((visibility("default")))

YITU_API size_t yitu_csr_transpose_workspace_bytes(int64_t nnz, int64_t n_cols) {
    if (nnz <= 0) return 256;
    return align_up(sort_temp_bytes(nnz, key_bits(n_cols)), 256) +
           4 * align_up(sizeof(int32_t) * (size_t)nnz, 256);
}

YITU_API int yitu_csr_transpose(int32_t *t_indptr, int32_t *t_rows, int32_t *t_perm,
                                const int32_t *indptr, const int32_t *indices, int64_t n_rows,
                                int64_t n_cols, int64_t nnz, int32_t col_mask, void *workspace,
                                size_t workspace_bytes, void *stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    YITU_REQUIRE(n_rows >= 0 && n_cols >= 0 && nnz >= 0, "negative size");
    YITU_REQUIRE(t_indptr && indptr, "null indptr");
    YITU_REQUIRE(n_rows < INT32_MAX && n_cols < INT32_MAX && nnz < INT32_MAX, "size out of range");
    const int grid_c = (int)ceil_div(nnz + 1, kBlock);
    if (nnz == 0) {
        // all columns empty
        transpose_finish_kernel<<<1, kBlock, 0, stream>>>(
            nullptr, nullptr, nullptr, t_indptr, nullptr, 0, (int32_t)n_cols);
        YITU_LAUNCH_CHECK();
        return 0;
    }
    YITU_REQUIRE(t_rows && t_perm && indices, "null edge array");
    YITU_REQUIRE(workspace && workspace_bytes >= yitu_csr_transpose_workspace_bytes(nnz, n_cols),
                 "workspace too small: need %zu bytes",
                 yitu_csr_transpose_workspace_bytes(nnz, n_cols));
    const int bits = key_bits(n_cols);
    char *w = static_cast<char *>(workspace);
    const size_t arr = align_up(sizeof(int32_t) * (size_t)nnz, 256);
    int32_t *keys = reinterpret_cast<int32_t *>(w);
    int32_t *keys_sorted = reinterpret_cast<int32_t *>(w + arr);
    int32_t *vals = reinterpret_cast<int32_t *>(w + 2 * arr);
    int32_t *edge_row = reinterpret_cast<int32_t *>(w + 3 * arr);
    void *temp = w + 4 * arr;
    size_t temp_bytes = sort_temp_bytes(nnz, bits);

    transpose_keys_kernel<<<(int)ceil_div(nnz, 1024), kBlock, 0, stream>>>(
        indptr, indices, keys, vals, edge_row, nnz, (int32_t)n_rows, col_mask);
    YITU_LAUNCH_CHECK();
    // stable: inside one source column the edges keep CSR order, i.e. ascending row
    YITU_HIP(rocprim::radix_sort_pairs(temp, temp_bytes, keys, keys_sorted, vals, t_perm,
                                       (size_t)nnz, 0, bits, stream));
    transpose_finish_kernel<<<grid_c, kBlock, 0, stream>>>(
        keys_sorted, t_perm, edge_row, t_indptr, t_rows, nnz, (int32_t)n_cols);
    YITU_LAUNCH_CHECK();
    return 0;
}

YITU_API int yitu_longest_row(long long *longest, const int32_t *indptr, int64_t n_rows, void *stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    YITU_REQUIRE(n_rows >= 0 && n_rows < INT32_MAX && longest && indptr, "bad argument");
    set_word_kernel<<<1, 1, 0, stream>>>(longest, 0);
    YITU_LAUNCH_CHECK();
    return longest_row(indptr, n_rows, longest, stream);
}

YITU_API size_t yitu_coo_to_csr_workspace_bytes(int64_t n_edges, int64_t n_rows) {
    (void)n_rows;
    const int64_t n = std::max<int64_t>(n_edges, 0);
    return 512 + align_up(coo_temp_bytes(n), 256) + align_up(sizeof(int32_t) * (size_t)std::max<int64_t>(ceil_div(n, kChunk), 1), 256) +
           2 * align_up(sizeof(uint64_t) * (size_t)n, 256);
}

// The narrow keys where the ids' bits allow it (half the bytes of every pass).
YITU_API int yitu_coo_to_csr_ids(int32_t *indptr, int32_t *indices, long long *info, const void *rows,
                                 const void *cols, int id_bytes, int64_t n_edges, int64_t n_rows,
                                 int64_t n_cols, void *workspace, size_t workspace_bytes,
                                 void *stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    YITU_REQUIRE(n_edges >= 0 && n_rows >= 0 && n_cols >= 0, "negative size");
    YITU_REQUIRE(n_rows < INT32_MAX && n_cols < INT32_MAX && n_edges < INT32_MAX,
                 "size out of range");
    YITU_REQUIRE(id_bytes == 4 || id_bytes == 8, "ids are of 4 or 8 bytes");
    YITU_REQUIRE(indptr && info, "null output");
    YITU_REQUIRE(n_edges == 0 || (indices && rows && cols), "null edge array");
    YITU_REQUIRE(workspace && workspace_bytes >= yitu_coo_to_csr_workspace_bytes(n_edges, n_rows) &&
                     (reinterpret_cast<uintptr_t>(workspace) & 255u) == 0,
                 "workspace too small or not 256-byte aligned: need %zu bytes",
                 yitu_coo_to_csr_workspace_bytes(n_edges, n_rows));
    char *w = static_cast<char *>(workspace);
    const bool narrow = coo_key_bits(n_rows, n_cols) <= 32;
    const size_t temp = coo_temp_bytes(n_edges);
    const auto r4 = static_cast<const int32_t *>(rows), c4 = static_cast<const int32_t *>(cols);
    const auto r8 = static_cast<const int64_t *>(rows), c8 = static_cast<const int64_t *>(cols);
    if (id_bytes == 4)
        return narrow ? coo_build<int32_t, uint32_t>(indptr, indices, info, r4, c4, n_edges, n_rows,
                                                     n_cols, w, temp, stream)
                      : coo_build<int32_t, uint64_t>(indptr, indices, info, r4, c4, n_edges, n_rows,
                                                     n_cols, w, temp, stream);
    return narrow ? coo_build<int64_t, uint32_t>(indptr, indices, info, r8, c8, n_edges, n_rows, n_cols,
                                                 w, temp, stream)
                  : coo_build<int64_t, uint64_t>(indptr, indices, info, r8, c8, n_edges, n_rows, n_cols,
                                                 w, temp, stream);
}

namespace yitu {
__global__ void copy_word_kernel(long long *out, const long long *in) { *out = *in; }
}  // namespace yitu

YITU_API int yitu_coo_to_csr(int32_t *indptr, int32_t *indices, long long *nnz_out,
                             const int32_t *rows, const int32_t *cols, int64_t n_edges,
                             int64_t n_rows, int64_t n_cols, void *workspace,
                             size_t workspace_bytes, void *stream_) {
    YITU_REQUIRE(nnz_out, "null output");
    YITU_REQUIRE(workspace && workspace_bytes >= yitu_coo_to_csr_workspace_bytes(n_edges, n_rows) &&
                     (reinterpret_cast<uintptr_t>(workspace) & 255u) == 0,
                 "workspace too small or not 256-byte aligned: need %zu bytes",
                 yitu_coo_to_csr_workspace_bytes(n_edges, n_rows));
    // the last 256 bytes take {edges, longest row}
    const size_t used = yitu_coo_to_csr_workspace_bytes(n_edges, n_rows);
    long long *info = reinterpret_cast<long long *>(static_cast<char *>(workspace) + used - 256);
    const int rc = yitu_coo_to_csr_ids(indptr, indices, info, rows, cols, 4, n_edges, n_rows, n_cols,
                                       workspace, workspace_bytes, stream_);
    if (rc) return rc;
    copy_word_kernel<<<1, 1, 0, static_cast<hipStream_t>(stream_)>>>(nnz_out, info);
    YITU_LAUNCH_CHECK();
    return 0;
}

YITU_API size_t yitu_build_part_workspace_bytes(int64_t n_rows) {
    return 2 * align_up(sizeof(int32_t) * (size_t)std::max<int64_t>(n_rows, 1), 256) +
           align_up(part_scan_bytes(n_rows), 256);
}

namespace yitu {
__global__ void part_empty_kernel(int32_t *part_ptr, long long *n_parts_out) {
    *n_parts_out = 0;
    part_ptr[0] = 0;
}
}  // namespace yitu

YITU_API int yitu_build_part(int32_t *part_ptr, int32_t *part2node, long long *n_parts_out,
                             const int32_t *indptr, int64_t n_rows, int64_t part_size,
                             int64_t capacity, void *workspace, size_t workspace_bytes,
                             void *stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    YITU_REQUIRE(n_rows >= 0 && n_rows < INT32_MAX, "row count out of range");
    YITU_REQUIRE(part_size > 0 && part_size < INT32_MAX, "partSize must be positive");
    YITU_REQUIRE(capacity >= 0 && part_ptr && n_parts_out && (capacity == 0 || part2node),
                 "null output");
    YITU_REQUIRE(indptr, "null indptr");
    YITU_REQUIRE(workspace && workspace_bytes >= yitu_build_part_workspace_bytes(n_rows) &&
                     (reinterpret_cast<uintptr_t>(workspace) & 255u) == 0,
                 "workspace too small or misaligned: need %zu bytes, 256-byte aligned",
                 yitu_build_part_workspace_bytes(n_rows));
    if (n_rows == 0) {
        // one thread writes the two words: no memset node, so the call may be captured
        part_empty_kernel<<<1, 1, 0, stream>>>(part_ptr, n_parts_out);
        YITU_LAUNCH_CHECK();
        return 0;
    }
    char *w = static_cast<char *>(workspace);
    const size_t arr = align_up(sizeof(int32_t) * (size_t)n_rows, 256);
    int32_t *count = reinterpret_cast<int32_t *>(w);
    int32_t *first = reinterpret_cast<int32_t *>(w + arr);
    void *temp = w + 2 * arr;
    size_t temp_bytes = part_scan_bytes(n_rows);
    part_count_kernel<<<(int)ceil_div(n_rows, kBlock), kBlock, 0, stream>>>(count, indptr,
                                                                           (int)n_rows, (int)part_size);
    YITU_LAUNCH_CHECK();
    YITU_HIP(rocprim::exclusive_scan(temp, temp_bytes, count, first, 0, (size_t)n_rows,
                                     rocprim::plus<int32_t>(), stream));
    part_fill_kernel<<<(int)ceil_div(n_rows, kWavesPerBlock), kBlock, 0, stream>>>(
        part_ptr, part2node, n_parts_out, first, count, indptr, (int)n_rows, (int)part_size,
        (long long)capacity);
    YITU_LAUNCH_CHECK();
    return 0;
}
