// Builds the row plan on the device: queue the long rows, cut every long row where its
// sorted columns cross the boundaries of its source bands and into items of at most 64
// edges, and deal the items into 2^16 bins by their middle source id. An item draws its rank
// in its bin when it is made, so a prefix sum of the bins gives its place; the order inside
// a bin does not matter to the kernels.
// Bound by atomics on one address, which the memory side takes one at a time (about 8 ns
// each): so the workgroups are of 1,024 threads and claim rows and items for all of them
// with one add. 200,000 rows, 3 M edges: 55 us in five launches, where a radix sort of the
// items (all slots, used or not) and narrower workgroups took 175.
#include <hip/hip_runtime.h>

#include <cstring>

#include "../../include/yitu_hip.h"
#include "plan.hpp"

namespace yitu {

namespace {

constexpr int kBins = 1 << 16;      // of items, by middle source id
constexpr int kPlanBlock = 1024;    // threads of the building kernels
constexpr int kPlanWaves = kPlanBlock / kWave;

struct BuildBuffers {
    PlanCounters *counters;
    int4 *rows;
    int4 *records;
    int *band_info;   // the header words (plan.hpp)
    int4 *items;      // {first edge, end edge, index into rows[], row} in queue order
    int2 *place;      // {bin, rank in it} of every item, in queue order
    int *bin_start;   // items of every bin, then its first place
    int key_shift;    // bin = middle source id >> key_shift
    int band_shift;   // band of a source = id >> band_shift
    int n_bands;      // 1 = no cuts
    int max_rows, max_items;
};

__global__ __launch_bounds__(kPlanBlock) void plan_init_kernel(BuildBuffers b) {
    const int i = blockIdx.x * kPlanBlock + threadIdx.x;
    if (i == 0) {
        b.counters->n_items = 0;
        b.counters->n_rows = 0;
        b.counters->overflow = 0;
        b.counters->pad = 0;
        b.band_info[0] = b.band_shift;
        b.band_info[1] = b.n_bands;
        b.band_info[kPlanInfoLocal] = 0;
        b.band_info[kPlanInfoSampled] = 0;
        b.band_info[kPlanInfoLocalEdges] = 0;
        b.band_info[kPlanInfoEdges] = 0;
    }
    if (b.bin_start && i < kBins) b.bin_start[i] = 0;
}

// Every lane owns one row; the long rows of a workgroup are numbered with a
// block-level prefix sum and ONE atomic (hundreds of thousands of same-address
// atomics serialise in L2).
__device__ __forceinline__ int block_rank(bool flag, int *wave_sums, int *block_base, int *counter) {
    const int lane = lane_id();
    const int wave = threadIdx.x / kWave;
    int pre = flag ? 1 : 0;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const int x = __shfl_up(pre, o, kWave);
        if (lane >= o) pre += x;
    }
    if (lane == kWave - 1) wave_sums[wave] = pre;
    pre -= flag ? 1 : 0;
    __syncthreads();
    if (threadIdx.x == 0) {
        int br = 0;
        for (int w = 0; w < kPlanWaves; w++) br += wave_sums[w];
        *block_base = br > 0 ? atomicAdd(counter, br) : 0;
    }
    __syncthreads();
    int slot = *block_base + pre;
    for (int w = 0; w < wave; w++) slot += wave_sums[w];
    __syncthreads();  // the shared words are reused by the next call
    return slot;
}

// The same pass measures whether the graph is local, on the rows that the row
// kernels walk (fewer than 64 edges): up to 4 edges of every such row, evenly
// spaced, are sampled, and an edge counts as local when its source lies within
// 1/64 of the id space (at least 1,024 ids) of the row's own relative position.
// One add per workgroup and counter.
__global__ __launch_bounds__(kPlanBlock) void plan_queue_kernel(BuildBuffers b,
                                                            const int32_t *__restrict__ indptr,
                                                            const int32_t *__restrict__ indices,
                                                            int n_rows, int n_src, int col_mask) {
    __shared__ int wave_sums[kPlanWaves];
    __shared__ int block_base;
    const int row = blockIdx.x * kPlanBlock + threadIdx.x;
    int deg = 0, beg = 0;
    if (row < n_rows) {
        beg = indptr[row];
        deg = indptr[row + 1] - beg;
    }
    int sampled = 0, local = 0;
    if (deg < kPlanThreshold) {
        sampled = min(deg, 4);
        const long long own = (long long)row * n_src / n_rows;
        const long long reach = max((long long)n_src >> 6, 1024ll);
        for (int k = 0; k < sampled; k++) {
            const long long c = indices[beg + deg * k / sampled] & col_mask;
            local += c - own <= reach && own - c <= reach;
        }
    }
    int weight = sampled ? deg * local / sampled : 0;  // local edges of the row
    if (row == n_rows - 1) b.band_info[kPlanInfoEdges] = beg + deg;
    __shared__ int seen[3];  // sampled edges, local ones, local edges
    if (threadIdx.x == 0) seen[0] = seen[1] = seen[2] = 0;
    __syncthreads();
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) {
        sampled += __shfl_xor(sampled, o, kWave);
        local += __shfl_xor(local, o, kWave);
        weight += __shfl_xor(weight, o, kWave);
    }
    if (lane_id() == 0 && sampled) {
        atomicAdd(&seen[0], sampled);
        atomicAdd(&seen[1], local);
        atomicAdd(&seen[2], weight);
    }
    __syncthreads();
    if (threadIdx.x == 0 && seen[0]) {
        atomicAdd(&b.band_info[kPlanInfoSampled], seen[0]);
        if (seen[1]) atomicAdd(&b.band_info[kPlanInfoLocal], seen[1]);
        if (seen[2]) atomicAdd(&b.band_info[kPlanInfoLocalEdges], seen[2]);
    }
    const bool longrow = deg >= kPlanThreshold;
    const int slot = block_rank(longrow, wave_sums, &block_base, &b.counters->n_rows);
    if (longrow) {
        if (slot >= b.max_rows)
            atomicExch(&b.counters->overflow, 1);
        else
            b.rows[slot] = make_int4(row, 0, 0, 0);
    }
}

// One wave per long row. A row of deg edges may be cut into P = the largest
// power of two <= deg / 16 pieces (at most the number of bands), so its cut points
// are the boundaries of groups of ceil(n_bands / P) consecutive bands: the lanes
// find where the row's columns cross them (binary search), lane 0 turns the
// crossings into segments (none shorter than kPlanMinSegment), the wave then
// writes the items of every segment: ceil(len / 64) pieces of equal size. Item
// ids of a row are consecutive; a workgroup takes its ids with one atomic.
__global__ __launch_bounds__(kPlanBlock) void plan_items_kernel(BuildBuffers b,
                                                            const int32_t *__restrict__ indptr,
                                                            const int32_t *__restrict__ indices,
                                                            int col_mask) {
    __shared__ int cut[kPlanWaves][kPlanMaxBands + 1];
    __shared__ int seg_beg[kPlanWaves][kPlanMaxBands + 1];    // [n_seg] = end of the row
    __shared__ int seg_first[kPlanWaves][kPlanMaxBands + 1];  // first item of the segment, [n_seg] = total
    __shared__ int n_seg[kPlanWaves];
    __shared__ int wave_first[kPlanWaves];
    const int lane = lane_id();
    const int wave = threadIdx.x / kWave;
    const int slot = blockIdx.x * kPlanWaves + wave;
    const int n_rows = b.counters->overflow ? 0 : min(b.counters->n_rows, b.max_rows);
    const bool active = slot < n_rows;
    int row = 0, beg = 0, end = 0;
    if (active) {
        row = b.rows[slot].x;
        beg = indptr[row];
        end = indptr[row + 1];
    }
    const int deg = end - beg;
    // pieces allowed, bands per group, groups
    int allowed = 1;
    while (allowed * 2 * kPlanMinSegment <= deg && allowed * 2 <= b.n_bands) allowed *= 2;
    if (b.n_bands > 1 && allowed * 2 * kPlanMinSegment <= deg) allowed = b.n_bands;
    const int per_group = (b.n_bands + allowed - 1) / allowed;
    const int n_groups = active ? (b.n_bands + per_group - 1) / per_group : 0;
    for (int k = lane; k <= n_groups; k += kWave) {
        int c = k == 0 ? beg : end;
        if (k > 0 && k < n_groups) {
            const long long bound = ((long long)k * per_group) << b.band_shift;
            int lo = beg, hi = end;  // first edge whose column is >= bound
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if ((long long)(indices[mid] & col_mask) < bound) lo = mid + 1; else hi = mid;
            }
            c = lo;
        }
        cut[wave][k] = c;
    }
    __syncthreads();
    if (active && lane == 0) {
        // columns that are not sorted inside the row give crossings out of order;
        // a running maximum keeps the pieces a partition of the row
        int n = 0, cur = beg, total = 0, reach = beg;
        for (int k = 1; k <= n_groups; k++) {
            reach = min(end, max(reach, cut[wave][k]));
            const bool last = k == n_groups;
            const int len = reach - cur;
            if (last ? len > 0
                     : (len >= kPlanMinSegment && end - reach >= kPlanMinSegment &&
                        n < allowed - 1)) {
                seg_beg[wave][n] = cur;
                seg_first[wave][n] = total;
                total += (len + kPlanChunk - 1) / kPlanChunk;
                cur = reach;
                n++;
            }
        }
        seg_beg[wave][n] = end;
        seg_first[wave][n] = total;
        n_seg[wave] = n;
    }
    if (!active && lane == 0) {
        n_seg[wave] = 0;
        seg_first[wave][0] = 0;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int sum = 0;
        for (int w = 0; w < kPlanWaves; w++) {
            wave_first[w] = sum;
            sum += seg_first[w][n_seg[w]];
        }
        const int base = sum > 0 ? atomicAdd(&b.counters->n_items, sum) : 0;
        for (int w = 0; w < kPlanWaves; w++) wave_first[w] += base;
    }
    __syncthreads();
    if (!active) return;
    const int n = n_seg[wave];
    const int total = seg_first[wave][n];
    const int first_item = wave_first[wave];
    if (first_item + total > b.max_items) {
        if (lane == 0) atomicExch(&b.counters->overflow, 1);
        return;
    }
    if (lane == 0) b.rows[slot] = make_int4(row, first_item, total, 0);
    int s = 0;  // items of a lane come in ascending order: the segment search resumes
    for (int i = lane; i < total; i += kWave) {
        while (s + 1 < n && seg_first[wave][s + 1] <= i) s++;
        const int sb = seg_beg[wave][s], se = seg_beg[wave][s + 1];
        const int pieces = seg_first[wave][s + 1] - seg_first[wave][s];
        const int size = (se - sb + pieces - 1) / pieces;
        const int ib = sb + (i - seg_first[wave][s]) * size;
        const int ie = min(se, ib + size);
        const int mid_col = indices[(ib + ie) >> 1] & col_mask;
        b.items[first_item + i] = make_int4(ib, ie, slot, row);
        const int bin = min(mid_col >> b.key_shift, kBins - 1);
        b.place[first_item + i] = make_int2(bin, atomicAdd(&b.bin_start[bin], 1));
    }
}

// Exclusive prefix sum of the bins, by one workgroup: 64 bins per thread, four at a time.
__global__ __launch_bounds__(kPlanBlock) void plan_bin_starts_kernel(BuildBuffers b) {
    __shared__ int wave_sums[kPlanWaves];
    constexpr int kEach = kBins / kPlanBlock / 4;
    int4 *bins = reinterpret_cast<int4 *>(b.bin_start) + threadIdx.x * kEach;
    int4 v[kEach];
    int sum = 0;
#pragma unroll
    for (int k = 0; k < kEach; k++) v[k] = bins[k];
#pragma unroll
    for (int k = 0; k < kEach; k++) sum += v[k].x + v[k].y + v[k].z + v[k].w;
    const int lane = lane_id(), wave = threadIdx.x / kWave;
    int pre = sum;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const int x = __shfl_up(pre, o, kWave);
        if (lane >= o) pre += x;
    }
    if (lane == kWave - 1) wave_sums[wave] = pre;
    __syncthreads();
    pre -= sum;
    for (int w = 0; w < wave; w++) pre += wave_sums[w];
#pragma unroll
    for (int k = 0; k < kEach; k++) {
        int4 o;
        o.x = pre;
        o.y = o.x + v[k].x;
        o.z = o.y + v[k].y;
        o.w = o.z + v[k].z;
        pre = o.w + v[k].w;
        bins[k] = o;
    }
}

__global__ __launch_bounds__(kBlock) void plan_records_kernel(BuildBuffers b) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= b.max_items) return;
    const int n_items = b.counters->overflow ? 0 : min(b.counters->n_items, b.max_items);
    if (i >= n_items) {  // slots behind the last item
        b.records[i] = make_int4(0, 0, 0, 0);
        return;
    }
    const int2 at = b.place[i];
    const int4 it = b.items[i];
    // a row that is a single item is finished by the item kernel itself
    const int single = b.rows[it.z].z == 1 ? (int)0x80000000 : 0;
    const int place = b.bin_start[at.x] + at.y;
    if (place < n_items) b.records[place] = make_int4(it.x, it.y, i, it.w | single);
}

}  // namespace

size_t plan_bytes(int64_t nnz) {
    return kPlanHeaderBytes + align_up(sizeof(int4) * (size_t)plan_max_rows(nnz), 256) +
           align_up(sizeof(int4) * (size_t)plan_max_items(nnz), 256);
}

size_t plan_build_workspace_bytes(int64_t nnz) {
    const size_t items = (size_t)plan_max_items(nnz);
    return align_up(sizeof(int4) * items, 256) + align_up(sizeof(int2) * items, 256) +
           sizeof(int) * kBins;
}

size_t plan_temp_bytes(int64_t nnz) { return plan_bytes(nnz) + plan_build_workspace_bytes(nnz); }

PlanView plan_view(const void *plan, int64_t nnz) {
    PlanView v{};
    const char *w = static_cast<const char *>(plan);
    v.counters = reinterpret_cast<const PlanCounters *>(w);
    w += kPlanHeaderBytes;
    v.max_rows = (int)plan_max_rows(nnz);
    v.max_items = (int)plan_max_items(nnz);
    v.rows = reinterpret_cast<const int4 *>(w);
    w += align_up(sizeof(int4) * (size_t)v.max_rows, 256);
    v.records = reinterpret_cast<const int4 *>(w);
    v.threshold = kPlanThreshold;
    v.info = reinterpret_cast<const int *>(static_cast<const char *>(plan) + 256);
    return v;
}

static void set_bands(BuildBuffers &b, int64_t n_src, bool with_bands) {
    const int64_t span = std::max<int64_t>(n_src, 1) - 1;  // largest source id
    b.key_shift = 0;
    while ((span >> b.key_shift) >= kBins) b.key_shift++;
    b.band_shift = kPlanBandShift;
    while ((span >> b.band_shift) + 1 > kPlanMaxBands) b.band_shift++;
    b.n_bands = with_bands ? (int)((span >> b.band_shift) + 1) : 1;
}

int plan_build_header(void *plan, const int32_t *indptr, const int32_t *indices, int64_t n_rows,
                      int64_t n_src, int64_t nnz, int32_t col_mask, hipStream_t stream) {
    YITU_REQUIRE(plan && (reinterpret_cast<uintptr_t>(plan) & 255u) == 0,
                 "plan must be 256-byte aligned");
    YITU_REQUIRE(n_rows < INT32_MAX && n_src < INT32_MAX && nnz < INT32_MAX, "size out of range");
    BuildBuffers b{};  // (no room for rows or items: a long row would be an overflow)
    b.counters = static_cast<PlanCounters *>(plan);
    b.band_info = reinterpret_cast<int *>(static_cast<char *>(plan) + 256);
    set_bands(b, n_src, true);
    plan_init_kernel<<<1, kPlanBlock, 0, stream>>>(b);
    YITU_LAUNCH_CHECK();
    if (n_rows == 0) return 0;
    plan_queue_kernel<<<(int)ceil_div(n_rows, kPlanBlock), kPlanBlock, 0, stream>>>(
        b, indptr, indices, (int)n_rows, (int)n_src, col_mask);
    YITU_LAUNCH_CHECK();
    return 0;
}

int plan_build(void *plan, size_t plan_size, const int32_t *indptr, const int32_t *indices,
               int64_t n_rows, int64_t n_src, int64_t nnz, int32_t col_mask, bool with_bands,
               void *workspace, size_t workspace_bytes, hipStream_t stream) {
    YITU_REQUIRE(plan && plan_size >= plan_bytes(nnz), "plan buffer too small: need %zu bytes",
                 plan_bytes(nnz));
    YITU_REQUIRE(workspace && workspace_bytes >= plan_build_workspace_bytes(nnz),
                 "workspace too small: need %zu bytes", plan_build_workspace_bytes(nnz));
    YITU_REQUIRE((reinterpret_cast<uintptr_t>(plan) & 255u) == 0 &&
                     (reinterpret_cast<uintptr_t>(workspace) & 255u) == 0,
                 "plan and workspace must be 256-byte aligned");
    YITU_REQUIRE(n_rows < INT32_MAX && n_src < INT32_MAX && nnz < INT32_MAX, "size out of range");
    const PlanView v = plan_view(plan, nnz);
    BuildBuffers b{};
    b.counters = const_cast<PlanCounters *>(v.counters);
    b.band_info = reinterpret_cast<int *>(static_cast<char *>(plan) + 256);
    b.rows = const_cast<int4 *>(v.rows);
    b.records = const_cast<int4 *>(v.records);
    b.max_rows = v.max_rows;
    b.max_items = v.max_items;
    char *w = static_cast<char *>(workspace);
    b.items = reinterpret_cast<int4 *>(w);
    w += align_up(sizeof(int4) * (size_t)b.max_items, 256);
    b.place = reinterpret_cast<int2 *>(w);
    b.bin_start = reinterpret_cast<int *>(w + align_up(sizeof(int2) * (size_t)b.max_items, 256));
    set_bands(b, n_src, with_bands);

    plan_init_kernel<<<kBins / kPlanBlock, kPlanBlock, 0, stream>>>(b);
    YITU_LAUNCH_CHECK();
    if (n_rows > 0) {
        plan_queue_kernel<<<(int)ceil_div(n_rows, kPlanBlock), kPlanBlock, 0, stream>>>(
            b, indptr, indices, (int)n_rows, (int)n_src, col_mask);
        YITU_LAUNCH_CHECK();
    }
    plan_items_kernel<<<(int)ceil_div(b.max_rows, kPlanWaves), kPlanBlock, 0, stream>>>(
        b, indptr, indices, col_mask);
    YITU_LAUNCH_CHECK();
    plan_bin_starts_kernel<<<1, kPlanBlock, 0, stream>>>(b);
    YITU_LAUNCH_CHECK();
    plan_records_kernel<<<(int)ceil_div(b.max_items, kBlock), kBlock, 0, stream>>>(b);
    YITU_LAUNCH_CHECK();
    return 0;
}

int plan_resolve(PlanView &view, bool &has_items, const void *plan, const int32_t *indptr,
                 const int32_t *indices, int64_t n_rows, int64_t n_src, int64_t nnz,
                 int32_t col_mask, int64_t max_degree_hint, void *workspace,
                 size_t workspace_bytes, void **rest, size_t *rest_bytes, hipStream_t stream) {
    *rest = workspace;
    *rest_bytes = workspace_bytes;
    has_items = nnz >= kPlanThreshold && !(max_degree_hint >= 0 && max_degree_hint < kPlanThreshold);
    if (plan) {  // also without long rows: the header says whether the graph is local
        view = plan_view(plan, nnz);
        return 0;
    }
    if (!has_items) {
        view = plan_none();
        return 0;
    }
    const size_t pb = plan_bytes(nnz), bw = plan_build_workspace_bytes(nnz);
    YITU_REQUIRE(workspace && workspace_bytes >= pb + bw,
                 "workspace too small for a temporary row plan: need %zu bytes, got %zu", pb + bw,
                 workspace_bytes);
    char *w = static_cast<char *>(workspace);
    int rc = plan_build(w, pb, indptr, indices, n_rows, n_src, nnz, col_mask, false, w + pb, bw,
                        stream);
    if (rc) return rc;
    view = plan_view(w, nnz);
    // the build scratch is dead once the records are written: hand it back
    *rest = w + pb;
    *rest_bytes = workspace_bytes - pb;
    return 0;
}

}  // namespace yitu

using namespace yitu;
#define YITU_API extern "C" __attribute__((visibility("default")))

YITU_API size_t yitu_plan_bytes(int64_t nnz) { return plan_bytes(nnz); }
YITU_API size_t yitu_plan_workspace_bytes(int64_t nnz) { return plan_build_workspace_bytes(nnz); }

YITU_API int yitu_plan_build(void *plan, size_t plan_size, const int32_t *indptr,
                             const int32_t *indices, int64_t n_rows, int64_t n_src, int64_t nnz,
                             int32_t col_mask, void *workspace, size_t workspace_bytes,
                             void *stream) {
    YITU_REQUIRE(n_rows >= 0 && n_src >= 0 && nnz >= 0, "negative size");
    YITU_REQUIRE(indptr && (nnz == 0 || indices), "null CSR");
    return plan_build(plan, plan_size, indptr, indices, n_rows, n_src, nnz, col_mask, true,
                      workspace, workspace_bytes, static_cast<hipStream_t>(stream));
}

YITU_API size_t yitu_plan_header_bytes(void) { return kPlanHeaderBytes; }
YITU_API int yitu_plan_build_header(void *plan, const int32_t *indptr, const int32_t *indices,
                                    int64_t n_rows, int64_t n_src, int64_t nnz, int32_t col_mask,
                                    void *stream) {
    YITU_REQUIRE(n_rows >= 0 && n_src >= 0 && nnz >= 0, "negative size");
    YITU_REQUIRE(indptr && (nnz == 0 || indices), "null CSR");
    return plan_build_header(plan, indptr, indices, n_rows, n_src, nnz, col_mask,
                             static_cast<hipStream_t>(stream));
}
