// fp32 products of many rows with a small weight, any inner dimension and width:
//   C_q[M_q, N] (+)= A_q[M_q, K] . B_q (+ bias_q),  M_q in the thousands and more.
// Included by gemm.hip (GemmParams, kMaxGroup).
//
// The weight panel of a workgroup (32 * NCW columns x the whole K) sits in LDS, zero-padded;
// every wave walks 32-row tiles of A on its own, KC columns at a time through an LDS area of
// its own: no barrier in the loop, and nothing that one wave waits for holds up another. The
// next chunk (or the next tile's first) is requested before the products of this one. MFMA
// step s takes columns 2 s and 2 s + 1 of the chunk, one per half of the wave: the order of the
// tiled kernel, so a product keeps its bits when its row count moves it from one to the
// other. Both areas hold every eight columns as four even ones, then four odd ones, so the operands
// of four steps are one 16-byte LDS read of either side; rows of both areas are padded by 16 bytes
// (an odd number of 16-byte pieces: reads without bank conflicts; the writes of a chunk, two
// of 8 bytes a lane, have some, 2 % of the kernel's cycles, and neighbouring lanes that swap
// values to write 16 bytes each measured no better). The weight is the first MFMA operand: a lane
// holds four consecutive columns of a row, and rows leave through the wave's LDS area as
// 128-byte segments. A workgroup takes a run of consecutive tiles of the list of all
// problems, one workgroup per CU.
//
// Bound: HBM (A once, C once) up to about 40 flop/byte, the matrix pipes beyond (2^21 x 128 x
// 128: matrix pipes busy 78 % of the kernel's cycles, at the 1.8 GHz it settles at).
#pragma once

namespace yitu {

constexpr int kPanelLds = 160 * 1024;
constexpr int kPanelWaves = 8;

struct PanelParams {
    const float *A[kMaxGroup];
    const float *B[kMaxGroup];
    float *C[kMaxGroup];
    const float *bias[kMaxGroup];  // [N] added to every row of the problem, or null
    int M[kMaxGroup];
    int tile_start[kMaxGroup + 1];
    int n_problems, N, K;
    int k_pad, ldw;  // K rounded up to 8; floats per weight row in LDS
    int b_kcont;     // the weight is stored [N, K] (else [K, N])
    int accumulate, c_vec4;
    int64_t lda, ldb, ldc;
};

// Orders a wave's own LDS writes and reads (other lanes read what a lane wrote).
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Place of a column in its row: 0 2 4 6 1 3 5 7 of every eight.
constexpr __device__ __forceinline__ int panel_column(int k) {
    return (k & ~7) | ((k & 1) << 2) | ((k >> 1) & 3);
}

template <int KC>
constexpr int panel_chunk_floats() {
    return 32 * (KC + 4);
}

template <int NCW, int KC, bool VEC>
__global__ __launch_bounds__(64 * kPanelWaves, 1) void sgemm_panel_kernel(PanelParams p) {
    typedef float f4 __attribute__((ext_vector_type(4)));
    typedef float f2 __attribute__((ext_vector_type(2)));
    constexpr int A_LD = KC + 4;
    constexpr int LPR = VEC ? KC / 4 : KC;  // lanes that cover a row of a chunk (at most 64)
    constexpr int RPI = 64 / LPR;           // rows per load instruction
    constexpr int LI = 32 / RPI;            // load instructions per chunk
    constexpr int C_LD = 36;                // staged output row: 32 columns + 16 bytes
    extern __shared__ __attribute__((aligned(16))) float lds[];
    float *Wl = lds;                                    // [32 NCW][ldw]
    float *bias_l = Wl + (size_t)32 * NCW * p.ldw;      // [32 NCW]
    const int lane = threadIdx.x & 63, wave = wave_id(), n_waves = blockDim.x >> 6;
    float *At = bias_l + 32 * NCW + (size_t)wave * panel_chunk_floats<KC>();
    const int l32 = lane & 31, lk = lane >> 5;
    const int n0 = blockIdx.y * 32 * NCW;
    const int lrow = lane / LPR, lcol = (lane % LPR) * (VEC ? 4 : 1);
    const int n_chunks = (p.k_pad + KC - 1) / KC;

    const int n_all = p.tile_start[p.n_problems];
    const int per_wg = (n_all + (int)gridDim.x - 1) / (int)gridDim.x;
    const int my_lo = blockIdx.x * per_wg, my_hi = min(my_lo + per_wg, n_all);

    for (int q = 0; q < p.n_problems; q++) {
        const int lo = p.tile_start[q];
        const int tile0 = max(lo, my_lo), hi = min(p.tile_start[q + 1], my_hi);
        if (tile0 >= hi) continue;  // same for the whole workgroup
        const float *__restrict__ a_q = p.A[q];
        const float *__restrict__ b_q = p.B[q];
        float *__restrict__ c_q = p.C[q];
        const int m_q = p.M[q];
        f4 r4[VEC ? LI : 1];
        float r1[VEC ? 1 : LI];
        const auto gload = [&](int tile, int c) {
            const int row0 = (tile - lo) * 32;
            const float *src = a_q + (int64_t)row0 * p.lda;  // (offsets inside a tile fit 32 bits)
            const int col = min(c * KC + lcol, p.K - (VEC ? 4 : 1));  // past K: dropped below
            const int lda = (int)p.lda, step = RPI * lda;
            const int last = min(m_q - 1 - row0, 31) * lda + col;  // rows past the end: the last one
            int at = lrow * lda + col;
#pragma unroll
            for (int i = 0; i < LI; i++, at += step) {
                asm volatile("" : "+v"(at));  // made as it is needed: hoisted, LI registers
                if constexpr (VEC)
                    r4[i] = *reinterpret_cast<const f4 *>(src + (unsigned)min(at, last));
                else
                    r1[i] = src[(unsigned)min(at, last)];
            }
        };
        int tile = tile0 + wave;
        if (tile < hi) gload(tile, 0);  // (in flight while the weight comes in)
        __syncthreads();  // the previous problem's weight is no longer read
        // The weight, in memory order: eight elements of a thread in flight at a time (row by
        // row, every row waited for its own load: 8 us on 64 rows of 100)
        const int minor = p.b_kcont ? p.k_pad : 32 * NCW, total = 32 * NCW * p.k_pad;
        const int step = blockDim.x, major_step = step / minor, minor_step = step % minor;
        int major = (int)threadIdx.x / minor, at = (int)threadIdx.x % minor;
        for (int i0 = threadIdx.x; i0 < total; i0 += 8 * step) {
            float w[8];
            int to[8];
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const int n = p.b_kcont ? major : at, k = p.b_kcont ? at : major;
                const bool in = k < p.K && n0 + n < p.N && i0 + i * step < total;
                const int64_t from = p.b_kcont ? (int64_t)(n0 + n) * p.ldb + k
                                               : (int64_t)k * p.ldb + n0 + n;
                w[i] = in ? b_q[from] : 0.0f;
                to[i] = n * p.ldw + panel_column(k);
                major += major_step;
                at += minor_step;
                if (at >= minor) at -= minor, major++;
            }
#pragma unroll
            for (int i = 0; i < 8; i++)
                if (i0 + i * step < total) Wl[to[i]] = w[i];
        }
        const bool has_bias = p.bias[q] != nullptr;
        if (has_bias)
            for (int n = threadIdx.x; n < 32 * NCW; n += blockDim.x)
                bias_l[n] = n0 + n < p.N ? p.bias[q][n0 + n] : 0.0f;
        __syncthreads();
        for (; tile < hi; tile += n_waves) {
            float16v acc[NCW];
#pragma unroll
            for (int j = 0; j < NCW; j++)
#pragma unroll
                for (int e = 0; e < 16; e++) acc[j][e] = 0.0f;
            for (int c = 0; c < n_chunks; c++) {
                const bool tail = (c + 1) * KC > p.K;  // the chunk holds columns past K
#pragma unroll
                for (int i = 0; i < LI; i++) {
                    float *dst = At + (lrow + RPI * i) * A_LD + panel_column(lcol);
                    if constexpr (VEC) {
                        f4 v = r4[i];
                        if (tail && c * KC + lcol >= p.K) v = f4{0.0f, 0.0f, 0.0f, 0.0f};
                        *reinterpret_cast<f2 *>(dst) = f2{v[0], v[2]};
                        *reinterpret_cast<f2 *>(dst + 4) = f2{v[1], v[3]};
                    } else {
                        *dst = tail && c * KC + lcol >= p.K ? 0.0f : r1[i];
                    }
                }
                if (c + 1 < n_chunks) gload(tile, c + 1);
                else if (tile + n_waves < hi) gload(tile + n_waves, 0);
                wave_lds_fence();
                // the halves of the wave take the even and the odd columns
                const int half = min(KC, p.k_pad - c * KC) / 2;
                const float *arow = At + l32 * A_LD + 4 * lk;
                const float *wrow = Wl + (size_t)l32 * p.ldw + c * KC + 4 * lk;
                const auto step4 = [&](int s) {
                    const f4 a = *reinterpret_cast<const f4 *>(arow + 2 * s);
                    f4 w[NCW];
#pragma unroll
                    for (int j = 0; j < NCW; j++)
                        w[j] = *reinterpret_cast<const f4 *>(wrow + (size_t)32 * j * p.ldw + 2 * s);
#pragma unroll
                    for (int e = 0; e < 4; e++)
#pragma unroll
                        for (int j = 0; j < NCW; j++)
                            acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(w[j][e], a[e], acc[j], 0,
                                                                          0, 0);
                };
                if (half == KC / 2) {
#pragma unroll
                    for (int s = 0; s < KC / 2; s += 4) {
                        step4(s);
                        // operand reads stay a few steps ahead of their products: all of them
                        // hoisted would not fit the registers
                        if (s % 8 == 4) __builtin_amdgcn_sched_barrier(0);
                    }
                } else {
                    for (int s = 0; s < half; s += 4) step4(s);
                }
                wave_lds_fence();  // the next chunk goes to the same place
            }
            // element 4 jj + ii of acc[j] is C[32 tile + lane % 32][n0 + 32 j + 8 jj + 4 (lane / 32) + ii]
            const int row0 = (tile - lo) * 32;
#pragma unroll
            for (int j = 0; j < NCW; j++) {
                const int col0 = n0 + 32 * j;
                if (col0 >= p.N) break;  // same for the whole wave
#pragma unroll
                for (int jj = 0; jj < 4; jj++) {
                    f4 w = {acc[j][4 * jj], acc[j][4 * jj + 1], acc[j][4 * jj + 2],
                            acc[j][4 * jj + 3]};
                    if (has_bias)
                        w += *reinterpret_cast<const f4 *>(bias_l + 32 * j + 8 * jj + 4 * lk);
                    *reinterpret_cast<f4 *>(At + l32 * C_LD + 8 * jj + 4 * lk) = w;
                }
                wave_lds_fence();
                // (offsets inside a tile fit 32 bits)
                float *dst0 = c_q + (int64_t)row0 * p.ldc + col0;
                const int ldc = (int)p.ldc, rows = m_q - row0, cols = p.N - col0;
                if (p.c_vec4) {
                    const int col = 4 * (lane & 7);
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const int row = 8 * r + (lane >> 3);
                        f4 w = *reinterpret_cast<const f4 *>(At + row * C_LD + col);
                        if (row < rows && col < cols) {
                            f4 *dst = reinterpret_cast<f4 *>(dst0 + (unsigned)(row * ldc + col));
                            if (p.accumulate) w += *dst;
                            *dst = w;
                        }
                    }
                } else {
#pragma unroll 4
                    for (int r = 0; r < 16; r++) {
                        const int row = 2 * r + lk;
                        float w = At[row * C_LD + l32];
                        if (row < rows && l32 < cols) {
                            float *dst = dst0 + (unsigned)(row * ldc + l32);
                            if (p.accumulate) w += *dst;
                            *dst = w;
                        }
                    }
                }
                wave_lds_fence();
            }
        }
    }
}

// More dynamic LDS than the default limit has to be asked for, once per device and kernel.
static int allow_lds(const void *kernel, size_t bytes, bool (&prepared_on)[64]) {
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 64) device = 0;
    if (bytes <= 65536 || prepared_on[device]) return 0;
    hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                       kPanelLds);
    if (e != hipSuccess) {
        set_error("hipFuncSetAttribute(dynamic LDS): %s", hipGetErrorString(e));
        return -1;
    }
    prepared_on[device] = true;
    return 0;
}

template <int NCW, int KC, bool VEC>
static int sgemm_panel_launch_k(const PanelParams &r, int waves, size_t lds, hipStream_t stream) {
    static bool prepared_on[64] = {};
    const void *kernel = reinterpret_cast<const void *>(&sgemm_panel_kernel<NCW, KC, VEC>);
    if (int rc = allow_lds(kernel, lds, prepared_on)) return rc;
    const int n_tiles = r.tile_start[r.n_problems];
    const dim3 grid((unsigned)std::min<int64_t>(ceil_div(n_tiles, 1), 256),
                    (unsigned)ceil_div(r.N, 32 * NCW));
    sgemm_panel_kernel<NCW, KC, VEC><<<grid, 64 * waves, lds, stream>>>(r);
    YITU_LAUNCH_CHECK();
    return 0;
}

template <int NCW>
static int sgemm_panel_launch(const PanelParams &r, int kc, int waves, size_t lds, bool vec,
                              hipStream_t stream) {
    if (kc == 64)
        return vec ? sgemm_panel_launch_k<NCW, 64, true>(r, waves, lds, stream)
                   : sgemm_panel_launch_k<NCW, 64, false>(r, waves, lds, stream);
    return vec ? sgemm_panel_launch_k<NCW, 32, true>(r, waves, lds, stream)
               : sgemm_panel_launch_k<NCW, 32, false>(r, waves, lds, stream);
}

// The panel's geometry: as many column blocks side by side as leave LDS for at least six
// waves' chunks (64 columns of A each where eight of them fit, else 32).
struct PanelShape {
    int ncw = 0, kc = 0, waves = 0;
    size_t lds = 0;
};
static PanelShape panel_shape(int64_t n, int64_t k) {
    const int64_t k_pad = ceil_div(k, 8) * 8, blocks = ceil_div(n, 32);
    for (int64_t panels = ceil_div(blocks, 4); panels <= blocks; panels++) {
        const int ncw = (int)ceil_div(blocks, panels);
        const size_t weight = (size_t)32 * ncw * (size_t)(k_pad + 5) * sizeof(float);
        for (int kc : {64, 32}) {
            if (kc == 64 && k_pad <= 32) continue;
            const size_t chunk = (size_t)32 * (kc + 4) * sizeof(float);
            if (weight >= (size_t)kPanelLds) continue;
            const int waves =
                (int)std::min<size_t>(kPanelWaves, ((size_t)kPanelLds - weight) / chunk);
            if (waves >= (kc == 64 ? kPanelWaves : 6))
                return {ncw, kc, waves, weight + (size_t)waves * chunk};
        }
    }
    return {};
}

constexpr int64_t kPanelMinRows = 16384;

// Takes the group when it is one of the kernel's shapes; *taken says whether it did.
static int sgemm_panel_try(const GemmParams &p, bool trans_a, bool trans_b, int lda, int ldb,
                           hipStream_t stream, bool *taken) {
    *taken = false;
    if (trans_a || p.n_prob < 1 || p.N < 1) return 0;
    const int k = p.prob[0].K;
    if (k < 1) return 0;
    PanelParams r{};
    bool vec = k % 4 == 0 && lda % 4 == 0, c_vec = p.ldc % 4 == 0 && p.N % 4 == 0;
    int64_t total = 0;
    for (int i = 0; i < p.n_prob; i++) {
        const GemmProblem &pr = p.prob[i];
        if (pr.K != k || pr.M < 0) return 0;
        vec = vec && aligned16(pr.A);
        c_vec = c_vec && aligned16(pr.C);
        r.A[i] = pr.A;
        r.B[i] = pr.B;
        r.C[i] = pr.C;
        r.bias[i] = pr.bias;
        r.M[i] = pr.M;
        r.tile_start[i + 1] = r.tile_start[i] + (int)ceil_div(pr.M, 32);
        total += pr.M;
    }
    // (offsets inside a 32-row tile are 32-bit)
    if (total < kPanelMinRows || lda > (1 << 20) || p.ldc > (1 << 20)) return 0;
    const PanelShape s = panel_shape(p.N, k);
    if (s.ncw == 0) return 0;
    // Against the tiled kernel, measured over M = 20,000 .. 2^21: fewer row tiles than waves
    // (65,536 rows) leave a wave one tile to hide its loads behind, which pays where the tiled
    // kernel is at its worst: inner dimensions that are not whole 16-byte pieces (50,000 x 333
    // x 77: 82 -> 60 us) and outputs that fill less than half of its 64 columns (40,000 x 500 x
    // 16: 40 -> 28 us). With more rows everything gains (2^21 x 128 x 128: 750 -> 665 us,
    // 800,000 x 100 x 47: 173 -> 150 us) but outputs of exactly its tile (400,000 x 64 x 64: 46
    // against 54 us); a second panel reads A twice, paid back by the columns the 128-wide tile
    // would waste (400,000 x 136 x 136: 291 -> 229 us).
    const int64_t panels = ceil_div(p.N, 32 * s.ncw);
    const bool many = total >= 65536;
    if (panels > 2 || (panels == 2 && (!many || p.N % 128 == 0)) ||
        (panels == 1 && (many ? p.N == 64 && vec : vec && p.N > 32)))
        return 0;
    r.n_problems = p.n_prob;
    r.N = p.N;
    r.K = k;
    r.k_pad = (int)(ceil_div(k, 8) * 8);
    r.ldw = r.k_pad + 4;
    r.b_kcont = trans_b;
    r.accumulate = p.accumulate;
    r.c_vec4 = c_vec;
    r.lda = lda;
    r.ldb = ldb;
    r.ldc = p.ldc;
    *taken = true;
    switch (s.ncw) {
        case 1: return sgemm_panel_launch<1>(r, s.kc, s.waves, s.lds, vec, stream);
        case 2: return sgemm_panel_launch<2>(r, s.kc, s.waves, s.lds, vec, stream);
        case 3: return sgemm_panel_launch<3>(r, s.kc, s.waves, s.lds, vec, stream);
        default: return sgemm_panel_launch<4>(r, s.kc, s.waves, s.lds, vec, stream);
    }
}

}  // namespace yitu
