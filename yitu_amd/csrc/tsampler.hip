// Temporal neighbour sampler on the device: YiTu_GNN/YiTu_T/sampler_core.cpp
// (ParallelSampler, :43-359) with the T-CSR resident in HBM, so that a training step
// needs no host sampling and no host-to-device copy of the block. yitu_tsample_recent
// is the `recent = True`, single-snapshot mode in one call; yitu_tsample_advance and
// yitu_tsample_window are the pieces of every mode (cursors or binary search, most
// recent or uniformly drawn neighbours, snapshots of a sliding window), which the
// caller strings together per layer and snapshot as the reference's sample() does.
//
// Semantics are those of the host library (csrc/host/sampler.cpp), which is
// bit-exact against the reference: per node a monotone cursor = the running
// maximum over all queries (n, t) seen so far of "last edge of n with
// ts <= t - 1e-7" (update_ts_ptr, :103-127; a running maximum is order
// independent, so an atomic max per root reproduces the sequential loop); then
// every root emits the edges k = cursor, cursor - 1, ... while
// k > max(first edge of n, cursor - fan) and ts[k] < t - 1e-7 (:295-305), in
// root order (count, exclusive scan, fill: the reference's thread-count
// independent order). Output is the COO block of combine_coo (:153-199).
#include <hip/hip_runtime.h>

#include <cstring>

#include <rocprim/device/device_scan.hpp>

#include "../../include/yitu_hip.h"
#include "spmm_rows.hpp"

namespace yitu {

namespace {

__device__ __forceinline__ float query_threshold(float t) { return (t + 0.0f) - 1e-7f; }

__global__ __launch_bounds__(kBlock) void ts_reset_kernel(int32_t *__restrict__ cursor,
                                                          const int32_t *__restrict__ indptr,
                                                          int64_t n_nodes) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i < n_nodes) cursor[i] = indptr[i];
}

// G lanes per root in each of these: two thousand roots one per thread were 32 waves, each
// walking a chain of dependent loads (count, scan and fill of 2,048 roots x 20: 6 + 8 + 17 us,
// now 2.6 + 3.6 + 3.1). As many lanes as a root has neighbours to look at (rounded up to a power
// of two): a whole wave for each of 131,072 roots x 5 took 21 us to count and 29 to fill, with
// eight lanes 4.7 and 8.6.
template <int G>
struct RootLanes {
    int64_t root;
    int lane;
    __device__ __forceinline__ RootLanes()
        : root(((int64_t)blockIdx.x * kBlock + threadIdx.x) / G), lane(lane_id() % G) {}
    // of this root's lanes (which are active together)
    __device__ __forceinline__ unsigned long long ballot(bool p) const {
        const unsigned long long all = __ballot(p);
        return G == 64 ? all : (all >> (lane_id() / G * G)) & ((1ull << (G & 63)) - 1);
    }
};

// The last edge with ts <= thr by a search of G probes a step: lane l looks at the last edge of
// the l-th of G equal parts. A cursor that is there already is not written: the roots of a batch
// that share a busy node would wait for each other's atomics (131,072 roots of a Zipf stream:
// 734 us; 157 the first time and 20 once the cursors are there; a value read early is at most
// too small, and the maximum decides).
template <int G>
__global__ __launch_bounds__(kBlock) void ts_advance_kernel(
    int32_t *__restrict__ cursor, const int32_t *__restrict__ indptr, const float *__restrict__ ts,
    const int32_t *__restrict__ roots, const float *__restrict__ root_ts, int64_t n_roots,
    int32_t n_nodes) {
    const RootLanes<G> me;
    const int64_t i = me.root;
    if (i >= n_roots) return;
    const int32_t n = roots[i];
    if (n < 0 || n >= n_nodes) return;  // (the count below reports it)
    const float thr = query_threshold(root_ts[i]);
    const int32_t first = indptr[n];
    int32_t lo = first, hi = indptr[n + 1];  // the first edge with ts > thr is in [lo, hi]
    while (lo < hi) {
        const int32_t step = (hi - lo + G - 1) / G;
        const int64_t at = (int64_t)lo + (int64_t)(me.lane + 1) * step - 1;
        const unsigned long long beyond = me.ballot(at >= hi || !(ts[at] <= thr));
        if (!beyond) {  // (G parts cover [lo, hi): the last lane's probe was not beyond it)
            lo = hi;
            break;
        }
        const int part = __ffsll(beyond) - 1;
        const int64_t end = (int64_t)lo + (int64_t)(part + 1) * step - 1;
        lo += part * step;
        hi = (int32_t)min((int64_t)hi, end);
    }
    if (me.lane == 0 && lo - 1 >= first &&
        __hip_atomic_load(&cursor[n], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < lo - 1)
        atomicMax(&cursor[n], lo - 1);
}

// Edges a root keeps, of the `fan` before its cursor; -1 for a root that is no node.
template <int G>
__global__ __launch_bounds__(kBlock) void ts_count_kernel(
    int32_t *__restrict__ counts, const int32_t *__restrict__ cursor,
    const int32_t *__restrict__ indptr, const float *__restrict__ ts,
    const int32_t *__restrict__ roots, const float *__restrict__ root_ts, int64_t n_roots,
    int32_t n_nodes, int fan) {
    const RootLanes<G> me;
    const int64_t i = me.root;
    if (i >= n_roots) return;
    const int32_t n = roots[i];
    int32_t cnt = -1;
    if (n >= 0 && n < n_nodes) {
        const float thr = query_threshold(root_ts[i]);
        const int32_t e = cursor[n], stop = max(indptr[n], e - fan);
        cnt = 0;
        for (int32_t k = e; k > stop; k -= G) {
            const int32_t mine = k - me.lane;
            cnt += __popcll(me.ballot(mine > stop && ts[max(mine, stop)] < thr));
        }
    }
    if (me.lane == 0) counts[i] = cnt;
}

// block_indptr = exclusive prefix sums of the counts, a workgroup per chunk of 16,384; *n_edges_out
// = their total, or -1 with a root that is no node. Up to one chunk is one launch (2,048 roots
// 3.6 us, 16,384 5.2); beyond, the chunks' sums are made first and every workgroup adds up those
// before it (131,072 roots 4.2 + 6.9 us).
constexpr int kStartsEach = 16, kStartsChunk = 1024 * kStartsEach;
struct ChunkSum {
    int32_t sum, bad;
};

// Sum over the workgroup's 1,024 threads (every thread gets it); red is theirs alone.
__device__ __forceinline__ int block_sum(int v, int (&red)[16]) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, kWave);
    __syncthreads();  // red may still be read
    if (lane_id() == 0) red[wave_id()] = v;
    __syncthreads();
    int all = 0;
    for (int w = 0; w < 16; w++) all += red[w];
    return all;
}

__global__ __launch_bounds__(1024) void ts_chunk_sums_kernel(ChunkSum *__restrict__ chunks,
                                                             const int32_t *__restrict__ counts,
                                                             int64_t n_roots) {
    __shared__ int red[16];
    const int64_t base = (int64_t)blockIdx.x * kStartsChunk;
    int sum = 0, bad = 0;
    for (int k = 0; k < kStartsEach; k++) {
        const int64_t i = base + k * 1024 + threadIdx.x;
        const int v = i < n_roots ? counts[i] : 0;
        sum += max(v, 0);
        bad |= v < 0;
    }
    sum = block_sum(sum, red);
    bad = block_sum(bad, red);
    if (threadIdx.x == 0) chunks[blockIdx.x] = {sum, bad};
}

__global__ __launch_bounds__(1024) void ts_starts_kernel(int32_t *__restrict__ block_indptr,
                                                         long long *__restrict__ n_edges_out,
                                                         const int32_t *__restrict__ counts,
                                                         const ChunkSum *__restrict__ chunks,
                                                         int64_t n_roots) {
    __shared__ int red[16], sums[16];
    const int lane = lane_id(), wave = wave_id(), n_chunks = gridDim.x;
    int carry = 0, bad = 0;
    if (n_chunks > 1) {
        for (int w = threadIdx.x; w < n_chunks; w += 1024) {
            carry += w < (int)blockIdx.x ? chunks[w].sum : 0;
            bad |= chunks[w].bad;
        }
        carry = block_sum(carry, red);
    }
    const int64_t base = (int64_t)blockIdx.x * kStartsChunk;
    const int64_t mine = base + (int64_t)threadIdx.x * kStartsEach;
    const bool whole = mine + kStartsEach <= n_roots;
    int v[kStartsEach], own = 0;
    if (whole) {  // (counts is the workspace's first array, 256-byte aligned)
#pragma unroll
        for (int k = 0; k < kStartsEach; k += 4)
            *reinterpret_cast<int4 *>(v + k) = *reinterpret_cast<const int4 *>(counts + mine + k);
    } else {
#pragma unroll
        for (int k = 0; k < kStartsEach; k++) v[k] = mine + k < n_roots ? counts[mine + k] : 0;
    }
#pragma unroll
    for (int k = 0; k < kStartsEach; k++) {
        bad |= v[k] < 0;
        v[k] = max(v[k], 0);
        own += v[k];
    }
    int pre = own;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const int x = __shfl_up(pre, o, kWave);
        if (lane >= o) pre += x;
    }
    if (lane == kWave - 1) sums[wave] = pre;
    bad = block_sum(bad, red);  // (its barriers order the waves' sums too)
    int at = carry + pre - own, all = 0;
    for (int w = 0; w < 16; w++) {
        at += w < wave ? sums[w] : 0;
        all += sums[w];
    }
#pragma unroll
    for (int k = 0; k < kStartsEach; k++) {
        const int next = at + v[k];
        v[k] = at;
        at = next;
    }
    if (whole && reinterpret_cast<uintptr_t>(block_indptr) % 16 == 0) {
#pragma unroll
        for (int k = 0; k < kStartsEach; k += 4)
            *reinterpret_cast<int4 *>(block_indptr + mine + k) = *reinterpret_cast<const int4 *>(v + k);
    } else {
#pragma unroll
        for (int k = 0; k < kStartsEach; k++)
            if (mine + k < n_roots) block_indptr[mine + k] = v[k];
    }
    if ((int)blockIdx.x == n_chunks - 1 && threadIdx.x == 0) {
        block_indptr[n_roots] = carry + all;
        *n_edges_out = bad ? -1 : carry + all;
    }
}

struct FillArgs {
    int32_t *row, *col, *eid_out, *nodes_out;
    float *ts_out, *dts_out;
    const int32_t *offsets, *cursor, *indptr, *indices, *eid, *roots;
    const float *ts, *root_ts;
    int64_t n_roots;
    int32_t n_nodes;
    int fan, prop_time;
};

template <int G>
__global__ __launch_bounds__(kBlock) void ts_fill_kernel(FillArgs a) {
    const RootLanes<G> me;
    const int64_t i = me.root;
    if (i >= a.n_roots) return;
    const int lane = me.lane;
    const int32_t n = a.roots[i];
    const float t = a.root_ts[i];
    if (lane == 0) {
        a.nodes_out[i] = n;
        a.ts_out[i] = t;
        a.dts_out[i] = 0.0f;
    }
    if (n < 0 || n >= a.n_nodes) return;
    const float thr = query_threshold(t);
    const int32_t e = a.cursor[n], stop = max(a.indptr[n], e - a.fan);
    int64_t base = a.offsets[i];
    for (int32_t k = e; k > stop; k -= G) {
        const int32_t mine = k - lane;
        const float when = a.ts[max(mine, stop)];
        const bool keep = mine > stop && when < thr;
        const unsigned long long kept = me.ballot(keep);
        if (keep) {
            const int64_t w = base + __popcll(kept & ((1ull << lane) - 1));
            a.row[w] = (int32_t)i;
            a.col[w] = (int32_t)(a.n_roots + w);
            a.eid_out[w] = a.eid[mine];
            a.ts_out[a.n_roots + w] = a.prop_time ? t : when;
            a.dts_out[a.n_roots + w] = t - when;
            a.nodes_out[a.n_roots + w] = a.indices[mine];
        }
        base += __popcll(kept);
    }
}

// ---- every mode: windows, draws ---------------------------------------------------

// rand_r of the C library the reference is linked against (glibc stdlib/rand_r.c):
// three steps of x -> 1103515245 x + 12345, of which 11 + 10 + 10 bits are taken.
__device__ __forceinline__ int c_rand_r(unsigned int &seed) {
    unsigned int next = seed;
    next = next * 1103515245u + 12345u;
    int result = (int)((next / 65536u) % 2048u);
    next = next * 1103515245u + 12345u;
    result <<= 10;
    result ^= (int)((next / 65536u) % 1024u);
    next = next * 1103515245u + 12345u;
    result <<= 10;
    result ^= (int)((next / 65536u) % 1024u);
    seed = next;
    return result;
}

// The generator state after `steps` steps from x (powers of one affine map commute, so
// the map is squared along the bits of `steps`).
__device__ __forceinline__ unsigned int lcg_skip(unsigned int x, unsigned long long steps) {
    unsigned int a = 1103515245u, c = 12345u;  // the map of 2^k steps
    unsigned int ra = 1u, rc = 0u;             // the map of the bits seen so far
    while (steps) {
        if (steps & 1ull) {
            ra = a * ra;
            rc = a * rc + c;
        }
        c = a * c + c;
        a = a * a;
        steps >>= 1;
    }
    return ra * x + rc;
}

__global__ __launch_bounds__(kBlock) void ts_advance_offset_kernel(
    int32_t *__restrict__ cursor, const int32_t *__restrict__ indptr, const float *__restrict__ ts,
    const int32_t *__restrict__ roots, const float *__restrict__ root_ts, int64_t n_roots,
    int32_t n_nodes, float offset) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n_roots) return;
    const int32_t n = roots[i];
    if (n < 0 || n >= n_nodes) return;  // reported by the sampling call
    const float thr = (root_ts[i] + offset) - 1e-7f;
    int32_t lo = indptr[n], hi = indptr[n + 1];  // first edge with ts > thr
    const int32_t first = lo;
    while (lo < hi) {
        const int32_t mid = lo + ((hi - lo) >> 1);
        if (ts[mid] <= thr) lo = mid + 1; else hi = mid;
    }
    if (lo - 1 >= first) atomicMax(&cursor[n], lo - 1);
}

struct WindowArgs {
    int32_t *row, *col, *eid_out, *nodes_out;
    float *ts_out, *dts_out;
    long long *n_edges_out;
    int32_t *win_lo, *win_hi, *draws, *counts;          // per root
    const int32_t *draw_prefix, *offsets;               // exclusive scans of draws / counts
    const int32_t *lo_cursor, *hi_cursor;               // null: binary search
    const int32_t *indptr, *indices, *eid, *roots;
    const float *ts, *root_ts;
    int *bad;
    int64_t n_roots, chunk;
    int32_t n_nodes;
    int fan, prop_time, recent, windowed;
    float offset, window;
};

// last edge of [b, e) with ts <= t, as an index (b - 1 when none)
__device__ __forceinline__ int32_t last_not_after(const float *ts, int32_t b, int32_t e, float t) {
    while (b < e) {
        const int32_t mid = b + ((e - b) >> 1);
        if (ts[mid] <= t) b = mid + 1; else e = mid;
    }
    return b - 1;
}

// The window [lo, hi] of every root (sampler_core.cpp:224-226 with cursors, :262-279 by
// binary search) and whether the root draws (uniform mode and at least `fan` edges).
__global__ __launch_bounds__(kBlock) void ts_window_kernel(WindowArgs a) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= a.n_roots) return;
    const int32_t n = a.roots[i];
    int32_t lo = 0, hi = 0, draws = 0;
    if (n < 0 || n >= a.n_nodes) {
        atomicExch(a.bad, 1);
    } else {
        const float t = a.root_ts[i];
        const int32_t b = a.indptr[n], e = a.indptr[n + 1];
        if (a.lo_cursor) {
            lo = a.lo_cursor[n];
            hi = a.hi_cursor[n];
        } else if (!a.windowed) {
            lo = b;
            hi = max(last_not_after(a.ts, b, e, t), lo);
        } else {
            lo = max(last_not_after(a.ts, b, e, (t + a.offset) - a.window), b);
            hi = max(last_not_after(a.ts, b, e, t + a.offset), lo);
        }
        draws = (!a.recent && hi - lo >= a.fan) ? 1 : 0;
    }
    a.win_lo[i] = lo;
    a.win_hi[i] = hi;
    a.draws[i] = draws;
}

// The edges root i keeps, in the reference's order (:295-318): emit(k) per edge.
template <typename Emit>
__device__ __forceinline__ int walk_root(const WindowArgs &a, int64_t i, Emit emit) {
    const int32_t n = a.roots[i];
    if (n < 0 || n >= a.n_nodes) return 0;
    const float thr = (a.root_ts[i] + a.offset) - 1e-7f;
    const int32_t lo = a.win_lo[i], hi = a.win_hi[i];
    int kept = 0;
    if (!a.draws[i]) {
        for (int32_t k = hi; k > max(lo, hi - a.fan); k--)
            if (a.ts[k] < thr) {
                emit(k);
                kept++;
            }
    } else {
        // thread c of the reference owns roots [c chunk, (c + 1) chunk) and the generator
        // seeded with c; every drawing root before this one in the chunk took 3 fan steps
        const int64_t c = i / a.chunk;
        const unsigned long long before = (unsigned long long)(a.draw_prefix[i] - a.draw_prefix[c * a.chunk]);
        unsigned int seed = lcg_skip((unsigned int)c, before * 3ull * (unsigned long long)a.fan);
        for (int j = 0; j < a.fan; j++) {
            const int32_t k = lo + c_rand_r(seed) % (hi - lo + 1);
            if (a.ts[k] < thr) {
                emit(k);
                kept++;
            }
        }
    }
    return kept;
}

__global__ __launch_bounds__(kBlock) void ts_window_count_kernel(WindowArgs a) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= a.n_roots) return;
    a.counts[i] = walk_root(a, i, [](int32_t) {});
}

__global__ __launch_bounds__(kBlock) void ts_window_fill_kernel(WindowArgs a) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= a.n_roots) return;
    if (i == a.n_roots - 1)
        *a.n_edges_out = *a.bad ? -1 : (long long)a.offsets[i] + a.counts[i];
    const float t = a.root_ts[i];
    a.nodes_out[i] = a.roots[i];
    a.ts_out[i] = t;
    a.dts_out[i] = 0.0f;
    int64_t w = a.offsets[i];
    walk_root(a, i, [&](int32_t k) {
        a.row[w] = (int32_t)i;
        a.col[w] = (int32_t)(a.n_roots + w);
        a.eid_out[w] = a.eid[k];
        a.ts_out[a.n_roots + w] = a.prop_time ? t : a.ts[k];
        a.dts_out[a.n_roots + w] = t - a.ts[k];
        a.nodes_out[a.n_roots + w] = a.indices[k];
        w++;
    });
}

size_t scan_bytes(int64_t n) {
    size_t bytes = 0;
    int32_t *p = nullptr;
    (void)rocprim::exclusive_scan(nullptr, bytes, p, p, 0, (size_t)n, rocprim::plus<int32_t>());
    return bytes;
}

}  // namespace

}  // namespace yitu

using namespace yitu;
#define YITU_API extern "C" __attribute__((visibility("default")))

YITU_API int yitu_tsample_reset(int32_t *cursor, const int32_t *indptr, int64_t n_nodes,
                                void *stream) {
    YITU_REQUIRE(n_nodes >= 0 && n_nodes < INT32_MAX, "size out of range");
    if (n_nodes == 0) return 0;
    YITU_REQUIRE(cursor && indptr, "null pointer");
    ts_reset_kernel<<<(int)ceil_div(n_nodes, kBlock), kBlock, 0, static_cast<hipStream_t>(stream)>>>(
        cursor, indptr, n_nodes);
    YITU_LAUNCH_CHECK();
    return 0;
}

namespace {
// Roots up to which the search takes a wave each (the chip holds 8,192 at once).
constexpr int64_t kWaveRoots = 16384;

// f(lanes per root): the power of two from 8 to 64 that covers `neighbours`.
template <typename F>
void with_lanes(int neighbours, F f) {
    if (neighbours <= 8) f(std::integral_constant<int, 8>());
    else if (neighbours <= 16) f(std::integral_constant<int, 16>());
    else if (neighbours <= 32) f(std::integral_constant<int, 32>());
    else f(std::integral_constant<int, 64>());
}

size_t root_array_bytes(int64_t n_roots) {
    return align_up(sizeof(int32_t) * (size_t)(std::max<int64_t>(n_roots, 1) + 1), 256);
}
}  // namespace

// counts, the block's indptr (yitu_tsample_recent), the chunks' sums
YITU_API size_t yitu_tsample_workspace_bytes(int64_t n_roots) {
    return 2 * root_array_bytes(n_roots) +
           align_up(sizeof(ChunkSum) * (size_t)ceil_div(n_roots, kStartsChunk), 256);
}

YITU_API int yitu_tsample_recent_block(int32_t *block_indptr, int32_t *row, int32_t *col,
                                       int32_t *eid_out, float *ts_out, float *dts_out,
                                       int32_t *nodes_out, long long *n_edges_out, int32_t *cursor,
                                       const int32_t *indptr, const int32_t *indices,
                                       const int32_t *eid, const float *ts, int64_t n_nodes,
                                       const int32_t *roots, const float *root_ts, int64_t n_roots,
                                       int fan, int prop_time, void *workspace,
                                       size_t workspace_bytes, void *stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    YITU_REQUIRE(n_nodes >= 0 && n_roots >= 0 && fan >= 0, "negative size");
    YITU_REQUIRE(n_nodes < INT32_MAX && n_roots * (int64_t)(fan + 1) < INT32_MAX,
                 "size out of range");
    YITU_REQUIRE(n_edges_out && block_indptr, "null output");
    YITU_REQUIRE(workspace && workspace_bytes >= yitu_tsample_workspace_bytes(n_roots) &&
                     (reinterpret_cast<uintptr_t>(workspace) & 255u) == 0,
                 "workspace too small or not 256-byte aligned: need %zu bytes",
                 yitu_tsample_workspace_bytes(n_roots));
    int32_t *counts = static_cast<int32_t *>(workspace);
    if (n_roots > 0) {
        YITU_REQUIRE(row && col && eid_out && ts_out && dts_out && nodes_out && cursor && indptr &&
                         roots && root_ts,
                     "null pointer");
        // a whole wave searches while the chip has room for one per root
        with_lanes(n_roots <= kWaveRoots ? kWave : 8, [&](auto lanes) {
            constexpr int G = decltype(lanes)::value;
            ts_advance_kernel<G><<<(int)ceil_div(n_roots, kBlock / G), kBlock, 0, stream>>>(
                cursor, indptr, ts, roots, root_ts, n_roots, (int32_t)n_nodes);
        });
        YITU_LAUNCH_CHECK();
        with_lanes(fan, [&](auto lanes) {
            constexpr int G = decltype(lanes)::value;
            ts_count_kernel<G><<<(int)ceil_div(n_roots, kBlock / G), kBlock, 0, stream>>>(
                counts, cursor, indptr, ts, roots, root_ts, n_roots, (int32_t)n_nodes, fan);
        });
        YITU_LAUNCH_CHECK();
    }
    const int n_chunks = (int)std::max<int64_t>(1, ceil_div(n_roots, kStartsChunk));
    ChunkSum *chunks = reinterpret_cast<ChunkSum *>(static_cast<char *>(workspace) +
                                                    2 * root_array_bytes(n_roots));
    if (n_chunks > 1) {
        ts_chunk_sums_kernel<<<n_chunks, 1024, 0, stream>>>(chunks, counts, n_roots);
        YITU_LAUNCH_CHECK();
    }
    ts_starts_kernel<<<n_chunks, 1024, 0, stream>>>(block_indptr, n_edges_out, counts, chunks, n_roots);
    YITU_LAUNCH_CHECK();
    if (n_roots == 0) return 0;
    const FillArgs a{row, col, eid_out, nodes_out, ts_out, dts_out, block_indptr, cursor, indptr,
                     indices, eid, roots, ts, root_ts, n_roots, (int32_t)n_nodes, fan, prop_time};
    with_lanes(fan, [&](auto lanes) {
        constexpr int G = decltype(lanes)::value;
        ts_fill_kernel<G><<<(int)ceil_div(n_roots, kBlock / G), kBlock, 0, stream>>>(a);
    });
    YITU_LAUNCH_CHECK();
    return 0;
}

YITU_API int yitu_tsample_recent(int32_t *row, int32_t *col, int32_t *eid_out, float *ts_out,
                                 float *dts_out, int32_t *nodes_out, long long *n_edges_out,
                                 int32_t *cursor, const int32_t *indptr, const int32_t *indices,
                                 const int32_t *eid, const float *ts, int64_t n_nodes,
                                 const int32_t *roots, const float *root_ts, int64_t n_roots,
                                 int fan, int prop_time, void *workspace, size_t workspace_bytes,
                                 void *stream) {
    YITU_REQUIRE(n_roots >= 0 && workspace &&
                     workspace_bytes >= yitu_tsample_workspace_bytes(n_roots),
                 "workspace too small: need %zu bytes", yitu_tsample_workspace_bytes(n_roots));
    int32_t *block_indptr = reinterpret_cast<int32_t *>(static_cast<char *>(workspace) +
                                                        root_array_bytes(n_roots));
    return yitu_tsample_recent_block(block_indptr, row, col, eid_out, ts_out, dts_out, nodes_out,
                                     n_edges_out, cursor, indptr, indices, eid, ts, n_nodes, roots,
                                     root_ts, n_roots, fan, prop_time, workspace, workspace_bytes,
                                     stream);
}

YITU_API int yitu_tsample_advance(int32_t *cursor, const int32_t *indptr, const float *ts,
                                  int64_t n_nodes, const int32_t *roots, const float *root_ts,
                                  int64_t n_roots, float offset, void *stream) {
    YITU_REQUIRE(n_nodes >= 0 && n_roots >= 0, "negative size");
    YITU_REQUIRE(n_nodes < INT32_MAX && n_roots < INT32_MAX, "size out of range");
    if (n_roots == 0) return 0;
    YITU_REQUIRE(cursor && indptr && roots && root_ts, "null pointer");
    ts_advance_offset_kernel<<<(int)ceil_div(n_roots, kBlock), kBlock, 0,
                               static_cast<hipStream_t>(stream)>>>(
        cursor, indptr, ts, roots, root_ts, n_roots, (int32_t)n_nodes, offset);
    YITU_LAUNCH_CHECK();
    return 0;
}

YITU_API size_t yitu_tsample_window_workspace_bytes(int64_t n_roots) {
    const int64_t n = std::max<int64_t>(n_roots, 1);
    return 256 + 6 * align_up(sizeof(int32_t) * (size_t)n, 256) + align_up(scan_bytes(n), 256);
}

YITU_API int yitu_tsample_window(int32_t *row, int32_t *col, int32_t *eid_out, float *ts_out,
                                 float *dts_out, int32_t *nodes_out, long long *n_edges_out,
                                 const int32_t *lo_cursor, const int32_t *hi_cursor,
                                 const int32_t *indptr, const int32_t *indices, const int32_t *eid,
                                 const float *ts, int64_t n_nodes, const int32_t *roots,
                                 const float *root_ts, int64_t n_roots, int fan, int prop_time,
                                 int recent, int windowed, float offset, float window,
                                 int64_t chunk, void *workspace, size_t workspace_bytes,
                                 void *stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    YITU_REQUIRE(n_nodes >= 0 && n_roots >= 0 && fan >= 0, "negative size");
    YITU_REQUIRE(n_nodes < INT32_MAX && n_roots * (int64_t)(fan + 1) < INT32_MAX,
                 "size out of range");
    YITU_REQUIRE(n_edges_out, "null output");
    YITU_REQUIRE((lo_cursor == nullptr) == (hi_cursor == nullptr),
                 "give both window cursors or neither");
    YITU_REQUIRE(recent || chunk > 0, "uniform draws need the roots per nominal thread");
    YITU_REQUIRE(workspace && workspace_bytes >= yitu_tsample_window_workspace_bytes(n_roots) &&
                     (reinterpret_cast<uintptr_t>(workspace) & 255u) == 0,
                 "workspace too small or not 256-byte aligned: need %zu bytes",
                 yitu_tsample_window_workspace_bytes(n_roots));
    int rc = fill_zero(static_cast<float *>(workspace), 64, stream);  // flag, and the count below
    if (rc) return rc;
    if (n_roots == 0) {
        YITU_HIP(hipMemcpyAsync(n_edges_out, workspace, sizeof(long long), hipMemcpyDeviceToDevice,
                                stream));
        return 0;
    }
    YITU_REQUIRE(row && col && eid_out && ts_out && dts_out && nodes_out && indptr && roots &&
                     root_ts,
                 "null pointer");
    char *w = static_cast<char *>(workspace);
    WindowArgs a{};
    a.bad = reinterpret_cast<int *>(w);
    w += 256;
    const size_t arr = align_up(sizeof(int32_t) * (size_t)n_roots, 256);
    a.win_lo = reinterpret_cast<int32_t *>(w);
    a.win_hi = reinterpret_cast<int32_t *>(w + arr);
    a.draws = reinterpret_cast<int32_t *>(w + 2 * arr);
    int32_t *draw_prefix = reinterpret_cast<int32_t *>(w + 3 * arr);
    a.counts = reinterpret_cast<int32_t *>(w + 4 * arr);
    int32_t *offsets = reinterpret_cast<int32_t *>(w + 5 * arr);
    void *temp = w + 6 * arr;
    a.draw_prefix = draw_prefix;
    a.offsets = offsets;
    a.row = row;
    a.col = col;
    a.eid_out = eid_out;
    a.nodes_out = nodes_out;
    a.ts_out = ts_out;
    a.dts_out = dts_out;
    a.n_edges_out = n_edges_out;
    a.lo_cursor = lo_cursor;
    a.hi_cursor = hi_cursor;
    a.indptr = indptr;
    a.indices = indices;
    a.eid = eid;
    a.roots = roots;
    a.ts = ts;
    a.root_ts = root_ts;
    a.n_roots = n_roots;
    a.chunk = std::max<int64_t>(chunk, 1);
    a.n_nodes = (int32_t)n_nodes;
    a.fan = fan;
    a.prop_time = prop_time;
    a.recent = recent;
    a.windowed = windowed;
    a.offset = offset;
    a.window = window;
    const int grid = (int)ceil_div(n_roots, kBlock);
    ts_window_kernel<<<grid, kBlock, 0, stream>>>(a);
    YITU_LAUNCH_CHECK();
    size_t bytes = scan_bytes(n_roots);
    if (!recent) {
        YITU_HIP(rocprim::exclusive_scan(temp, bytes, a.draws, draw_prefix, 0, (size_t)n_roots,
                                         rocprim::plus<int32_t>(), stream));
    }
    ts_window_count_kernel<<<grid, kBlock, 0, stream>>>(a);
    YITU_LAUNCH_CHECK();
    bytes = scan_bytes(n_roots);
    YITU_HIP(rocprim::exclusive_scan(temp, bytes, a.counts, offsets, 0, (size_t)n_roots,
                                     rocprim::plus<int32_t>(), stream));
    ts_window_fill_kernel<<<grid, kBlock, 0, stream>>>(a);
    YITU_LAUNCH_CHECK();
    return 0;
}
