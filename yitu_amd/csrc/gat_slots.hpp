// The attention backward when the layer's output was the mean over heads: its gradient
// g [n_dst, F] stands for grad_out[r,h,:] = g[r,:] / H, so the by-source pass gathers F floats
// per edge instead of H * F. Included by gat.hip (GatSrcParams).
//
// With F * 4 bytes per edge the pass is bound by loads in flight and by what it does around
// them, not by bandwidth, so one load instruction fetches SLOTS = 64 / LPF different edges:
// lane (s, sub) holds floats [4 sub, +4) of the gradient row of the s-th edge of a group
// (LPF = F / 4 rounded up to a power of two), and the source's own row as H slices
// x[c, h, 4 sub .. +4). Per group: H dots (one per head, reduced over the slot's lanes), H x 4
// multiply-adds into acc[h], and the softmax backward of an edge's heads on the slot's first
// lanes (or HPL heads per lane where the heads outnumber them). Head widths that do not fill
// the LPF lanes leave the last ones without a share of x: what they load reaches nothing.
#pragma once

namespace yitu {

inline bool gat_slots_shape(int64_t n_heads, int64_t n_features) {
    return (n_heads == 1 || n_heads == 2 || n_heads == 4 || n_heads == 8) && n_features >= 4 &&
           n_features <= 256 && n_features % 4 == 0;
}

template <int LPF, int H>
struct SlotRow {
    static constexpr int SLOTS = kWave / LPF;
    static constexpr int HPL = H > LPF ? H / LPF : 1;  // heads of a lane in the epilogue
    float xh[H][4], acc[H][4];
    // of the lane's own heads: key[c, .] and this slot's share of grad_key[c, .]
    float kc[HPL], gk[HPL];
    static __device__ __forceinline__ bool owner() { return lane_id() % LPF * HPL < H; }
    static __device__ __forceinline__ int head(int i) { return lane_id() % LPF * HPL + i; }
};

template <int LPF, int H>
__device__ __forceinline__ void slot_begin(SlotRow<LPF, H> &row, const GatSrcParams &p, int c,
                                           bool load) {
    using Row = SlotRow<LPF, H>;
    const int sub = lane_id() % LPF, F = p.sp.F;
#pragma unroll
    for (int i = 0; i < Row::HPL; i++) {
        row.kc[i] = row.gk[i] = 0.0f;
        if (load && Row::owner()) row.kc[i] = p.key[(size_t)c * H + Row::head(i)];
    }
#pragma unroll
    for (int h = 0; h < H; h++) {
#pragma unroll
        for (int i = 0; i < 4; i++) row.acc[h][i] = row.xh[h][i] = 0.0f;
        if (load && 4 * sub < F)
            RowLoad<4, float>::ld(p.x + (size_t)c * p.sp.L + h * F + sub * 4, row.xh[h]);
    }
}

template <int LPF, int H>
__device__ __forceinline__ void slot_window(SlotRow<LPF, H> &row, const GatSrcParams &p,
                                            const EdgeWindow &win, int first, int n) {
    using Row = SlotRow<LPF, H>;
    // U load groups in flight: 2 measured a little better than 4 (fewer registers)
    constexpr int SLOTS = Row::SLOTS, HPL = Row::HPL, U = 2;
    constexpr float scale = 1.0f / H;
    const int lane = lane_id();
    const int s = lane / LPF, sub = lane % LPF;
    const int F = p.sp.F, at = min(4 * sub, F - 4);
    const float *__restrict__ g = static_cast<const float *>(p.sp.feat);
    for (int k0 = 0; k0 < n; k0 += SLOTS * U) {
        float v[U][4], own[U][HPL];
        float2 sq[U][HPL];
        int vr[U];
        bool valid[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (k0 + u * SLOTS < n) {  // wave-uniform
                const int k = k0 + u * SLOTS + s;
                valid[u] = k < n;
                const int src = first + min(k, n - 1);
                const int r = __shfl(win.col, src, kWave);
                vr[u] = __shfl(win.vrow, src, kWave);
                RowLoad<4, float>::ld(g + (size_t)r * F + at, v[u]);
#pragma unroll
                for (int i = 0; i < HPL; i++) {
                    // the probability of (edge, own head): made from the destination's line, or
                    // read through the edge permutation
                    own[u][i] = 0.0f;
                    sq[u][i] = make_float2(0.0f, 0.0f);
                    if (Row::owner()) {
                        const float4 t4 = p.row_sq[(size_t)r * H + Row::head(i)];
                        sq[u][i] = make_float2(t4.x, t4.y);
                        own[u][i] = p.recompute ? expf(leaky(t4.y + row.kc[i]) - t4.z) * t4.w
                                                : p.sp.values[(size_t)vr[u] * H + Row::head(i)];
                    }
                }
            }
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (k0 + u * SLOTS >= n) break;  // wave-uniform
            // a slot without an edge has loaded the last edge's row again, and lanes past a head's
            // width its last floats: dropped here, where they are added up (0 x inf is not 0)
            const bool live = valid[u] && 4 * sub < F;
#pragma unroll
            for (int i = 0; i < 4; i++) v[u][i] = live ? v[u][i] : 0.0f;
            float mine[HPL];  // d_attn of (this slot's edge, own head)
#pragma unroll
            for (int i = 0; i < HPL; i++) mine[i] = 0.0f;
#pragma unroll
            for (int h = 0; h < H; h++) {
                float d = row.xh[h][0] * v[u][0] + row.xh[h][1] * v[u][1] + row.xh[h][2] * v[u][2] +
                          row.xh[h][3] * v[u][3];
                d = group_sum<LPF>(d);
                if (sub == h / HPL) mine[h % HPL] = d;
                const float a = __shfl(own[u][h % HPL], (lane - sub) + h / HPL, kWave);
                const float w = valid[u] ? a * scale : 0.0f;
#pragma unroll
                for (int i = 0; i < 4; i++) row.acc[h][i] += w * v[u][i];
            }
            if (valid[u] && Row::owner()) {
                float gl[HPL];
#pragma unroll
                for (int i = 0; i < HPL; i++) {
                    gl[i] = own[u][i] * (mine[i] * scale - sq[u][i].x) *
                            (sq[u][i].y + row.kc[i] < 0.0f ? kSlope : 1.0f);
                    row.gk[i] += gl[i];
                }
                float *dst = p.grad_a + (size_t)vr[u] * H + Row::head(0);
                if (HPL == 1 || p.grad_a_vec) {
                    store_row<HPL>(dst, gl);
                } else {
#pragma unroll
                    for (int i = 0; i < HPL; i++) dst[i] = gl[i];
                }
            }
        }
    }
}

// Adds the slots up (a fixed order) and writes the row: halves and quarters of the wave swap
// through the vector ALU and keep a part of the values each, the slots inside 16 lanes are
// added by lane rotations.
template <int LPF, int H>
__device__ __forceinline__ void slot_end(SlotRow<LPF, H> &row, int F, float *x_dst, float *k_dst) {
    using Row = SlotRow<LPF, H>;
    constexpr int PARTS = LPF == 64 ? 1 : LPF == 32 ? 2 : 4;  // of the 4 H values, one per lane group
    constexpr int N = 4 * H / PARTS;
    const int lane = lane_id(), sub = lane % LPF;
    const int part = LPF == 64 ? 0 : LPF == 32 ? lane / 32 : lane / 16;
    float v[4 * H];
#pragma unroll
    for (int i = 0; i < 4 * H; i++) v[i] = row.acc[i / 4][i % 4];
    if constexpr (LPF <= 32) {
#pragma unroll
        for (int i = 0; i < 2 * H; i++) v[i] = pair_sum32(v[i], v[i + 2 * H]);
#pragma unroll
        for (int i = 0; i < Row::HPL; i++) row.gk[i] = pair_sum32(row.gk[i], row.gk[i]);
    }
    if constexpr (LPF <= 16) {
#pragma unroll
        for (int i = 0; i < H; i++) v[i] = pair_sum16(v[i], v[i + H]);
#pragma unroll
        for (int i = 0; i < Row::HPL; i++) row.gk[i] = pair_sum16(row.gk[i], row.gk[i]);
    }
    const auto rotate = [&](auto ctrl) {
#pragma unroll
        for (int i = 0; i < N; i++) v[i] += dpp_permute<decltype(ctrl)::value>(v[i]);
#pragma unroll
        for (int i = 0; i < Row::HPL; i++) row.gk[i] += dpp_permute<decltype(ctrl)::value>(row.gk[i]);
    };
    if constexpr (LPF <= 8) rotate(std::integral_constant<int, 0x128>());  // row_ror 8
    if constexpr (LPF <= 4) rotate(std::integral_constant<int, 0x124>());  // row_ror 4
    if constexpr (LPF <= 2) rotate(std::integral_constant<int, 0x122>());  // row_ror 2
    if constexpr (LPF <= 1) rotate(std::integral_constant<int, 0x121>());  // row_ror 1
    // this lane's values are [part N, +N) of the H x 4 at columns 4 sub
    constexpr int W = N < 4 ? N : 4;
    if (4 * sub < F && (LPF >= 16 || lane % 16 < LPF)) {
#pragma unroll
        for (int i = 0; i < N; i += W) {
            float t[W];
#pragma unroll
            for (int j = 0; j < W; j++) t[j] = v[i + j];
            const int at = part * N + i;
            store_row_streaming<W>(x_dst + at / 4 * F + 4 * sub + at % 4, t);
        }
    }
    if (lane < LPF && Row::owner())
#pragma unroll
        for (int i = 0; i < Row::HPL; i++) k_dst[Row::head(i)] = row.gk[i];
}

template <int LPF, int H>
__global__ __launch_bounds__(kBlock) void gat_slot_rows_kernel(GatSrcParams p) {
    const int lane = lane_id();
    const int rpw = rows_per_wave(p.sp.n_rows);
    const int r0 = (row_block(p.sp, blockIdx.x, gridDim.x) * kWavesPerBlock + wave_id()) * rpw;
    if (r0 >= p.sp.n_rows) return;
    const int n_here = min(rpw, p.sp.n_rows - r0);
    const int my_ptr = p.sp.indptr[r0 + min(lane, n_here)];
    const int limit = __builtin_amdgcn_readlane(my_ptr, n_here);
    EdgeWindow win;
    win.base = -1;
    win.col = 0;
    win.w = 0.0f;
    win.vrow = 0;
    for (int i = 0; i < n_here; i++) {
        const int row = r0 + i;
        const int beg = __builtin_amdgcn_readlane(my_ptr, i), end = __builtin_amdgcn_readlane(my_ptr, i + 1);
        if (end - beg >= p.sp.plan.threshold) continue;  // a planned row: the item kernel
        SlotRow<LPF, H> acc;
        slot_begin<LPF, H>(acc, p, row, end > beg);
        for (int b = beg; b < end; b += kWave) {
            const int n = min(kWave, end - b);
            if (win.base < 0 || b < win.base || b + n > win.base + kWave)
                load_window<W_EDGEHEAD>(win, p.sp, b, limit);
            slot_window<LPF, H>(acc, p, win, b - win.base, n);
        }
        slot_end<LPF, H>(acc, p.sp.F, p.sp.out + (size_t)row * p.sp.L, p.grad_k + (size_t)row * H);
    }
}

template <int LPF, int H>
__global__ __launch_bounds__(kBlock) void gat_slot_items_kernel(GatSrcParams p) {
    const int lane = lane_id();
    if (p.sp.plan.counters->overflow) return;
    const int n_items = min(p.sp.plan.counters->n_items, p.sp.plan.max_items);
    const int n_waves = gridDim.x * kWavesPerBlock;
    const int L = p.sp.L;
    for (int pos0 = (blockIdx.x * kWavesPerBlock + wave_id()) * kSrcItems;
         pos0 < n_items; pos0 += n_waves * kSrcItems) {
        const int n_here = min(kSrcItems, n_items - pos0);
        const int4 my_rec = p.sp.plan.records[pos0 + min(lane, n_here - 1)];
        EdgeWindow win[kSrcItems];
        int n_edges[kSrcItems], tag[kSrcItems], item[kSrcItems];
#pragma unroll
        for (int j = 0; j < kSrcItems; j++) {
            const int beg = __builtin_amdgcn_readlane(my_rec.x, j);
            const int end = __builtin_amdgcn_readlane(my_rec.y, j);
            item[j] = __builtin_amdgcn_readlane(my_rec.z, j);
            tag[j] = __builtin_amdgcn_readlane(my_rec.w, j);
            n_edges[j] = j < n_here ? end - beg : 0;
            if (n_edges[j] > 0) load_window<W_EDGEHEAD>(win[j], p.sp, beg, end);
        }
#pragma unroll
        for (int j = 0; j < kSrcItems; j++) {
            if (n_edges[j] <= 0) continue;
            const int row = tag[j] & 0x7fffffff;
            SlotRow<LPF, H> acc;
            slot_begin<LPF, H>(acc, p, row, true);
            slot_window<LPF, H>(acc, p, win[j], 0, n_edges[j]);
            const bool single = tag[j] < 0;
            slot_end<LPF, H>(acc, p.sp.F,
                             single ? p.sp.out + (size_t)row * L : p.sp.partial + (size_t)item[j] * L,
                             single ? p.grad_k + (size_t)row * H : p.partial_k + (size_t)item[j] * H);
        }
    }
}

// The row of a lane's slot when every wave takes U * SLOTS consecutive rows. Counted in rows:
// threads (a row is LPF of them) pass 32 bits from 2^26 rows of 256 floats on.
template <int LPF>
constexpr int slot_row(unsigned wave, int u_per_wave, int lane) {
    return (int)(wave * (unsigned)(u_per_wave * (kWave / LPF)) + (unsigned)(lane / LPF));
}
static_assert(slot_row<64>(1u << 25, 2, 63) == 1 << 26 && slot_row<16>(1u << 26, 2, 17) == (1 << 29) + 1 &&
                  slot_row<2>(3, 2, 5) == 3 * 64 + 2,
              "rows beyond a 32-bit thread count");

// (S, query, max, 1 / sum) of every destination and head, S[r,h] = <g[r,:], out[r,h,:]> / H:
// a row per slot, read front to back once.
template <int LPF, int H>
__global__ __launch_bounds__(kBlock) void gat_slot_dot_kernel(float4 *__restrict__ row_sq,
                                                              const float *__restrict__ g,
                                                              const float *__restrict__ out,
                                                              const float *__restrict__ query,
                                                              const float *__restrict__ stats,
                                                              int n_rows, int F) {
    using Row = SlotRow<LPF, H>;
    typedef float f4 __attribute__((ext_vector_type(4)));
    constexpr int U = 2;
    const int lane = lane_id(), sub = lane % LPF;
    const int r0 = slot_row<LPF>(blockIdx.x * kWavesPerBlock + wave_id(), U, lane);
    f4 gv[U], ov[U][H];
#pragma unroll
    for (int u = 0; u < U; u++) {
        const size_t r = min(r0 + u * Row::SLOTS, n_rows - 1);
        const int at = min(4 * sub, F - 4);
        gv[u] = *reinterpret_cast<const f4 *>(g + r * F + at);
#pragma unroll
        for (int h = 0; h < H; h++)
            ov[u][h] = __builtin_nontemporal_load(
                reinterpret_cast<const f4 *>(out + (r * H + h) * F + at));
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
        const int r = r0 + u * Row::SLOTS;
        float mine[Row::HPL];
#pragma unroll
        for (int i = 0; i < Row::HPL; i++) mine[i] = 0.0f;
#pragma unroll
        for (int h = 0; h < H; h++) {
            float d = 0.0f;
#pragma unroll
            for (int i = 0; i < 4; i++) d += gv[u][i] * ov[u][h][i];
            d = group_sum<LPF>(4 * sub < F ? d : 0.0f);
            if (sub == h / Row::HPL) mine[h % Row::HPL] = d;
        }
        if (r < n_rows && Row::owner())
#pragma unroll
            for (int i = 0; i < Row::HPL; i++) {
                const size_t at = (size_t)r * H + Row::head(i);
                row_sq[at] = make_float4(mine[i] * (1.0f / H), query[at], stats ? stats[at * 2] : 0.0f,
                                         stats ? stats[at * 2 + 1] : 0.0f);
            }
    }
}

template <int LPF, int H>
static int gat_slots_launch(const GatSrcParams &p, bool has_items, const float *g, const float *out,
                            const float *query, int n_dst, hipStream_t stream) {
    gat_slot_dot_kernel<LPF, H>
        <<<(int)ceil_div(n_dst, kWavesPerBlock * 2 * (kWave / LPF)), kBlock, 0, stream>>>(
            const_cast<float4 *>(p.row_sq), g, out, query, p.stats, n_dst, p.sp.F);
    YITU_LAUNCH_CHECK();
    gat_slot_rows_kernel<LPF, H><<<row_grid(p.sp.n_rows), kBlock, 0, stream>>>(p);
    YITU_LAUNCH_CHECK();
    if (!has_items) return 0;
    // enough workgroups to walk the item list once (a second turn would mix source bands)
    const int item_grid = (int)std::min<int64_t>(
        ceil_div(p.sp.plan.max_items, kWavesPerBlock * kSrcItems), 1 << 20);
    gat_slot_items_kernel<LPF, H><<<item_grid, kBlock, 0, stream>>>(p);
    YITU_LAUNCH_CHECK();
    const int red_grid = (int)std::min<int64_t>(p.sp.plan.max_rows, 1 << 16);
    spmm_reduce_kernel<W_NONE, 4><<<red_grid, kBlock, 0, stream>>>(p.sp);
    YITU_LAUNCH_CHECK();
    SpmmParams k = p.sp;  // the item partials of grad_key, rows of H floats
    k.L = k.F = H;
    k.H = 1;
    k.out = p.grad_k;
    k.partial = p.partial_k;
    spmm_reduce_kernel<W_NONE, (H % 4 == 0 ? 4 : H)><<<red_grid, kBlock, 0, stream>>>(k);
    YITU_LAUNCH_CHECK();
    return 0;
}

template <int H>
static int gat_slots_launch_heads(const GatSrcParams &p, bool has_items, const float *g,
                                  const float *out, const float *query, int n_dst,
                                  hipStream_t stream) {
    const int lanes = p.sp.F / 4;
    if (lanes <= 2) return gat_slots_launch<2, H>(p, has_items, g, out, query, n_dst, stream);
    if (lanes <= 4) return gat_slots_launch<4, H>(p, has_items, g, out, query, n_dst, stream);
    if (lanes <= 8) return gat_slots_launch<8, H>(p, has_items, g, out, query, n_dst, stream);
    if (lanes <= 16) return gat_slots_launch<16, H>(p, has_items, g, out, query, n_dst, stream);
    if (lanes <= 32) return gat_slots_launch<32, H>(p, has_items, g, out, query, n_dst, stream);
    return gat_slots_launch<64, H>(p, has_items, g, out, query, n_dst, stream);
}

static int gat_slots_run(const GatSrcParams &p, bool has_items, const float *g, const float *out,
                         const float *query, int n_dst, hipStream_t stream) {
    switch (p.sp.H) {
        case 1: return gat_slots_launch_heads<1>(p, has_items, g, out, query, n_dst, stream);
        case 2: return gat_slots_launch_heads<2>(p, has_items, g, out, query, n_dst, stream);
        case 4: return gat_slots_launch_heads<4>(p, has_items, g, out, query, n_dst, stream);
        default: return gat_slots_launch_heads<8>(p, has_items, g, out, query, n_dst, stream);
    }
}

}  // namespace yitu
