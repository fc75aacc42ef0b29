// fp32 weight gradients over many rows, C_q[KI, NO] = A_q^T . B_q with A_q [rows, KI] and
// B_q [rows, NO], any widths and strides; and with it, when asked for, the column sums of A_q
// (the bias gradient of a Linear, whose output gradient is A).
// Included by gemm.hip (GemmParams, kMaxGroup).
//
// Both MFMA operands of this product are columns of row-major matrices: lane = column, the
// two halves of the wave take the two rows of a step, so an operand is one coalesced 4-byte
// load per lane straight from memory: no LDS stage, no barrier, no alignment to ask for. A
// wave keeps TX x TY MFMA tiles (at most 8) of the output in registers and walks rows with
// the loads of the next U steps in flight. Outputs of more tiles are split over the waves of
// a workgroup ("roles"), which walk the same rows at about the same time and find each
// other's operands in the vector cache; the row groups of a workgroup (as many as make about
// eight waves) are added through LDS in a fixed order, and the workgroups' products go to
// slabs in the workspace that tn_reduce_kernel adds. Column sums cost one add per A operand.
//
// Bound: HBM (both operands once) while KI * NO / (KI + NO) stays below about 60, the matrix
// pipes beyond.
#pragma once

namespace yitu {

constexpr int kTnMaxKi = 512, kTnMaxNo = 512;

struct TnRowsParams {
    const float *A[kMaxGroup];
    const float *B[kMaxGroup];
    float *C[kMaxGroup];
    float *sums[kMaxGroup];  // [KI] column sums of A_q, or null
    int rows[kMaxGroup], z0[kMaxGroup + 1], chunk[kMaxGroup];  // workgroups [z0[q], z0[q+1])
    int n_problems, KI, NO;
    int roles, roles_j, groups;  // output blocks, blocks along NO, row groups of a workgroup
    int accumulate, want_sums;
    int64_t lda, ldb, ldc;
    float *partial;  // [workgroup][KI * NO + KI]
};

template <int TX, int TY>
__global__ __launch_bounds__(512, 2) void sgemm_tn_rows_kernel(TnRowsParams p) {
    constexpr int U = TX + TY <= 4 ? 8 : 6;  // steps (of 2 rows) in flight
    extern __shared__ __attribute__((aligned(16))) float red[];
    const int KI = p.KI, NO = p.NO;
    const int lane = threadIdx.x & 63, wave = wave_id();
    const int l32 = lane & 31, lk = lane >> 5;
    int q = 0;
    while (q + 1 < p.n_problems && (int)blockIdx.x >= p.z0[q + 1]) q++;
    const int per_wg = p.roles < 8 ? p.roles : 8;  // roles of this workgroup
    const int role = blockIdx.y * 8 + wave % per_wg, group = wave / per_wg;
    const int i0 = role / p.roles_j * 32 * TX, j0 = role % p.roles_j * 32 * TY;
    const bool active = role < p.roles;
    // the workgroup's run of rows, its groups taking blocks of 2 U of them in turn
    const int wg_beg = ((int)blockIdx.x - p.z0[q]) * p.chunk[q];
    const int rows = max(0, min(p.rows[q] - wg_beg, p.chunk[q]));
    const int n_blocks = max(0, (rows / (2 * U) - group + p.groups - 1) / p.groups);  // whole ones
    const auto row_of = [&](int s) { return (group + s * p.groups) * 2 * U; };
    const float *__restrict__ A = p.A[q] + (int64_t)wg_beg * p.lda;
    const float *__restrict__ B = p.B[q] + (int64_t)wg_beg * p.ldb;

    // A lane's operands of the TX (TY) tiles are TX (TY) neighbouring columns, one load: tile x
    // holds every TX-th column. The address path takes as long for 4 bytes a lane as for 16.
    // Lanes at the end of a ragged width take its last columns once more.
    typedef float VecA __attribute__((ext_vector_type(TX), aligned(4)));
    typedef float VecB __attribute__((ext_vector_type(TY), aligned(4)));
    const auto col_a = [&](int i) { return min(i0 + TX * i, KI - TX); };
    const auto col_b = [&](int j) { return min(j0 + TY * j, NO - TY); };
    const unsigned offa = (unsigned)(col_a(l32) + lk * (int)p.lda);
    const unsigned offb = (unsigned)(col_b(l32) + lk * (int)p.ldb);
    float16v acc[TX][TY];
    float sums[TX];
#pragma unroll
    for (int x = 0; x < TX; x++) {
        sums[x] = 0.0f;
#pragma unroll
        for (int y = 0; y < TY; y++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[x][y][e] = 0.0f;
    }
    const auto multiply = [&](const VecA &a, const VecB &b) {
#pragma unroll
        for (int x = 0; x < TX; x++) {
            sums[x] += a[x];
#pragma unroll
            for (int y = 0; y < TY; y++)
                acc[x][y] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[x], b[y], acc[x][y], 0, 0, 0);
        }
    };
    VecA a[2][U];
    VecB b[2][U];
    const auto load = [&](int set, int row) {
        const float *pa = A + (int64_t)row * p.lda, *pb = B + (int64_t)row * p.ldb;
#pragma unroll
        for (int u = 0; u < U; u++) {
            a[set][u] = *reinterpret_cast<const VecA *>(pa + offa);
            b[set][u] = *reinterpret_cast<const VecB *>(pb + offb);
            pa += 2 * p.lda;
            pb += 2 * p.ldb;
        }
    };
    if (active) {
        if (n_blocks > 0) load(0, row_of(0));
        for (int s0 = 0; s0 < n_blocks; s0 += 2) {
#pragma unroll
            for (int v = 0; v < 2; v++) {
                const int s = s0 + v;
                if (s >= n_blocks) break;
                if (s + 1 < n_blocks) load(1 - v, row_of(s + 1));
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int u = 0; u < U; u++) multiply(a[v][u], b[v][u]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // the rows behind the last whole block: its owner's; a row past the end adds nothing
        for (int row = row_of(n_blocks); row < min(rows, row_of(n_blocks) + 2 * U); row += 2) {
            VecA ta;
            VecB tb;
#pragma unroll
            for (int x = 0; x < TX; x++) ta[x] = 0.0f;
#pragma unroll
            for (int y = 0; y < TY; y++) tb[y] = 0.0f;
            if (row + lk < rows) {
                ta = *reinterpret_cast<const VecA *>(A + (int64_t)row * p.lda + offa);
                tb = *reinterpret_cast<const VecB *>(B + (int64_t)row * p.ldb + offb);
            }
            multiply(ta, tb);
        }
    }
    // the row groups, halved until one is left: the upper half hands its registers over
    constexpr int kRegs = 16 * TX * TY + TX;
    for (int n = p.groups; n > 1;) {
        const int half = (n + 1) / 2;
        if (group >= half && group < n) {
            float *to = red + (size_t)((group - half) * per_wg + wave % per_wg) * kRegs * 64 + lane;
#pragma unroll
            for (int x = 0; x < TX; x++) {
#pragma unroll
                for (int y = 0; y < TY; y++)
#pragma unroll
                    for (int e = 0; e < 16; e++) to[(16 * (x * TY + y) + e) * 64] = acc[x][y][e];
                to[(16 * TX * TY + x) * 64] = sums[x];
            }
        }
        __syncthreads();
        if (group + half < n) {
            const float *from = red + (size_t)(group * per_wg + wave % per_wg) * kRegs * 64 + lane;
#pragma unroll
            for (int x = 0; x < TX; x++) {
#pragma unroll
                for (int y = 0; y < TY; y++)
#pragma unroll
                    for (int e = 0; e < 16; e++) acc[x][y][e] += from[(16 * (x * TY + y) + e) * 64];
                sums[x] += from[(16 * TX * TY + x) * 64];
            }
        }
        __syncthreads();
        n = half;
    }
    if (group != 0 || !active) return;
    // accumulator element e of tile (x, y) is row col_a(8 (e / 4) + 4 (lane / 32) + e % 4) + x,
    // column col_b(lane % 32) + y of this workgroup's slab
    float *dst = p.partial + (size_t)blockIdx.x * ((size_t)KI * NO + KI);
    if (j0 + TY * l32 < NO)
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const int i = 8 * (e / 4) + 4 * lk + e % 4;
            if (i0 + TX * i >= KI) continue;
#pragma unroll
            for (int x = 0; x < TX; x++) {
                VecB v;
#pragma unroll
                for (int y = 0; y < TY; y++) v[y] = acc[x][y][e];
                *reinterpret_cast<VecB *>(dst + (unsigned)((col_a(i) + x) * NO + col_b(l32))) = v;
            }
        }
    if (p.want_sums && j0 == 0) {
#pragma unroll
        for (int x = 0; x < TX; x++) {
            const float both = sums[x] + __shfl_xor(sums[x], 32, kWave);
            if (lk == 0 && i0 + TX * l32 < KI) dst[(size_t)KI * NO + col_a(l32) + x] = both;
        }
    }
}

// Products of 128 and 128 or 256 and 256 columns with whole, aligned rows: the roles of the
// kernel above each read their own share of every row through the vector cache (256 columns:
// six times the operands' size, 394 us for 2^18 rows); here the rows are read once, whole, two
// 16-row stages ahead through a ring of registers into a double-buffered LDS stage, one
// barrier per stage (305 us; 128 columns, 2^21 rows: 737 -> 690 us). Eight waves, WJ of them
// side by side, of TX x TY tiles. Stage rows are padded by 128 bytes, so that the two rows of a
// step fall into different banks.
constexpr int TR_STAGE = 16;  // rows per stage

template <int TX, int TY, int WJ>
__global__ __launch_bounds__(512, TX *TY <= 2 ? 4 : 2) void sgemm_tn_square_kernel(TnRowsParams p) {
    constexpr int W = 32 * TY * WJ, LD = W + 32, P = TR_STAGE * W / 4 / 512;
    static_assert(W == 32 * TX * (8 / WJ), "a square output over eight waves");
    extern __shared__ __attribute__((aligned(16))) float stage_mem[];  // [2][A stage, B stage]
    typedef float f4 __attribute__((ext_vector_type(4)));
    const int t = threadIdx.x, lane = t & 63, wave = wave_id();
    const int l32 = lane & 31, lk = lane >> 5;
    const int i0 = wave / WJ * 32 * TX, j0 = wave % WJ * 32 * TY;
    int q = 0;
    while (q + 1 < p.n_problems && (int)blockIdx.x >= p.z0[q + 1]) q++;
    const int m_beg = ((int)blockIdx.x - p.z0[q]) * p.chunk[q];
    const int m_end = min(p.rows[q], m_beg + p.chunk[q]);
    const int n_stages = (m_end - m_beg + TR_STAGE - 1) / TR_STAGE;
    float16v acc[TX][TY];
    float sums[TX] = {};
#pragma unroll
    for (int x = 0; x < TX; x++)
#pragma unroll
        for (int y = 0; y < TY; y++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[x][y][e] = 0.0f;
    // loader: thread t takes the 16-byte pieces t and t + 512 of a stage of A and of B
    f4 ra[2][P], rb[2][P];
    const auto gload = [&](int slot, int st) {
#pragma unroll
        for (int h = 0; h < P; h++) {
            const int piece = t + 512 * h, row = m_beg + st * TR_STAGE + piece / (W / 4);
            ra[slot][h] = rb[slot][h] = f4{0.0f, 0.0f, 0.0f, 0.0f};  // past the chunk
            if (row < m_end) {
                ra[slot][h] = __builtin_nontemporal_load(reinterpret_cast<const f4 *>(
                    p.A[q] + (int64_t)row * p.lda + piece % (W / 4) * 4));
                rb[slot][h] = __builtin_nontemporal_load(reinterpret_cast<const f4 *>(
                    p.B[q] + (int64_t)row * p.ldb + piece % (W / 4) * 4));
            }
        }
    };
    gload(0, 0);
    __builtin_amdgcn_sched_barrier(0);  // oldest first
    gload(1, 1);
    for (int s0 = 0; s0 < n_stages; s0 += 2) {
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int st = s0 + u;
            if (st >= n_stages) break;  // same for the whole workgroup
            float *As = stage_mem + (size_t)(st & 1) * TR_STAGE * 2 * LD;
            float *Bs = As + TR_STAGE * LD;
            // this buffer was last read two stages ago, before the previous barrier
#pragma unroll
            for (int h = 0; h < P; h++) {
                const int piece = t + 512 * h, at = piece / (W / 4) * LD + piece % (W / 4) * 4;
                *reinterpret_cast<f4 *>(As + at) = ra[u][h];
                *reinterpret_cast<f4 *>(Bs + at) = rb[u][h];
            }
            __syncthreads();
            gload(u, st + 2);
#pragma unroll
            for (int k2 = 0; k2 < TR_STAGE; k2 += 2) {
                float a[TX], b[TY];
#pragma unroll
                for (int x = 0; x < TX; x++) a[x] = As[(k2 + lk) * LD + i0 + 32 * x + l32];
#pragma unroll
                for (int y = 0; y < TY; y++) b[y] = Bs[(k2 + lk) * LD + j0 + 32 * y + l32];
#pragma unroll
                for (int x = 0; x < TX; x++) {
                    sums[x] += a[x];
#pragma unroll
                    for (int y = 0; y < TY; y++)
                        acc[x][y] =
                            __builtin_amdgcn_mfma_f32_32x32x2f32(a[x], b[y], acc[x][y], 0, 0, 0);
                }
            }
        }
    }
    float *dst = p.partial + (size_t)blockIdx.x * (W * W + W);
#pragma unroll
    for (int x = 0; x < TX; x++)
#pragma unroll
        for (int y = 0; y < TY; y++)
#pragma unroll
            for (int e = 0; e < 16; e++)
                __builtin_nontemporal_store(
                    acc[x][y][e], dst + (i0 + 32 * x + 8 * (e / 4) + 4 * lk + e % 4) * W + j0 +
                                      32 * y + l32);
    if (j0 == 0)
#pragma unroll
        for (int x = 0; x < TX; x++) {
            const float both = sums[x] + __shfl_xor(sums[x], 32, kWave);
            if (lk == 0) dst[W * W + i0 + 32 * x + l32] = both;
        }
}

// C (+)= the sum of a problem's slabs, and the column sums behind them, in a fixed order: a
// workgroup takes 32 consecutive outputs of one problem (blockIdx.y); each of its sixteen
// 32-thread groups adds a sixteenth of the slabs, eight loads at a time, and the parts are
// combined through LDS. (Four groups with four loads at a time: 12 us for 256 slabs of
// 128 x 128, all of it waiting.)
constexpr int kTnSumGroups = 16;
__global__ __launch_bounds__(32 * kTnSumGroups) void tn_reduce_kernel(TnRowsParams p) {
    __shared__ float red[kTnSumGroups][32];
    const int q = blockIdx.y, lane_e = threadIdx.x & 31, zg = threadIdx.x >> 5;
    const int64_t out = (int64_t)p.KI * p.NO, slab = out + p.KI;
    const int64_t total = p.want_sums && p.sums[q] ? slab : out;
    const int n_split = p.z0[q + 1] - p.z0[q];
    const int64_t e = (int64_t)blockIdx.x * 32 + lane_e;
    float s = 0.0f;
    if (e < total) {
        const float *src = p.partial + (size_t)p.z0[q] * slab + e;
#pragma unroll 8
        for (int z = zg; z < n_split; z += kTnSumGroups) s += src[(size_t)z * slab];
    }
    red[zg][lane_e] = s;
    __syncthreads();
    if (zg == 0 && e < total) {
#pragma unroll
        for (int g = 1; g < kTnSumGroups; g++) s += red[g][lane_e];
        if (e < out) {
            float *c = p.C[q] + (e / p.NO) * p.ldc + e % p.NO;
            *c = p.accumulate ? *c + s : s;
        } else {
            p.sums[q][e - out] = s;
        }
    }
}

// The output's split into roles of at most 8 tiles: the fewest MFMAs per step over all roles
// (tiles that stick out of the output are computed for nothing), then the fewest operand
// loads. Roles beyond eight go to further workgroups (blockIdx.y).
struct TnGeometry {
    int tx = 0, ty = 0, roles_i = 0, roles_j = 0;
    int roles() const { return roles_i * roles_j; }
    // row groups that make up a workgroup of about eight waves
    int groups() const { return roles() >= 8 ? 1 : 8 / roles(); }
};
static TnGeometry tn_rows_geometry(int64_t ki, int64_t no) {
    TnGeometry g;
    if (ki < 1 || no < 1 || ki > kTnMaxKi || no > kTnMaxNo) return g;
    const int ib = (int)ceil_div(ki, 32), jb = (int)ceil_div(no, 32);
    int64_t best = INT64_MAX;
    for (int tx = 1; tx <= 4; tx++)
        for (int ty = 1; ty <= 4 && tx * ty <= 8; ty++) {
            if (tx > ki || ty > no) continue;
            const int ri = (int)ceil_div(ib, tx), rj = (int)ceil_div(jb, ty);
            // (two loads of 16 cycles a CU per step against 64 cycles a SIMD for each product)
            const int64_t cost = (int64_t)ri * rj * (tx * ty + 2);
            if (cost < best) {
                best = cost;
                g.tx = tx;
                g.ty = ty;
                g.roles_i = ri;
                g.roles_j = rj;
            }
        }
    return g;
}

// Workgroups along the rows: one per CU (two where a wave's registers are few); a row group
// has at least 16 rows.
static int64_t tn_rows_chunks(const TnGeometry &g, int64_t total_rows) {
    const int64_t most = std::max<int64_t>(1, (g.tx * g.ty <= 2 ? 512 : 256) / ceil_div(g.roles(), 8));
    return std::max<int64_t>(1, std::min<int64_t>(most, total_rows / (16 * g.groups())));
}

static size_t tn_rows_workspace_bytes(int64_t ki, int64_t no, int64_t rows, int64_t n_problems) {
    const TnGeometry g = tn_rows_geometry(ki, no);
    if (g.tx == 0) return 0;
    const int64_t np = std::min<int64_t>(std::max<int64_t>(n_problems, 1), kMaxGroup);
    return (size_t)(std::max<int64_t>(tn_rows_chunks(g, rows * np), ki == no && ki == 128 ? 512 : 0) +
                    2 * np) * (size_t)(ki * no + ki) * sizeof(float);
}

static int tn_reduce_launch(const TnRowsParams &r, hipStream_t stream) {
    const int64_t total = (int64_t)r.KI * r.NO + (r.want_sums ? r.KI : 0);
    const dim3 rg((unsigned)ceil_div(total, 32), (unsigned)r.n_problems);
    tn_reduce_kernel<<<rg, 32 * kTnSumGroups, 0, stream>>>(r);
    YITU_LAUNCH_CHECK();
    return 0;
}

template <int TX, int TY, int WJ>
static int sgemm_tn_square_launch(const TnRowsParams &r, hipStream_t stream) {
    constexpr size_t lds = (size_t)2 * TR_STAGE * 2 * (32 * TY * WJ + 32) * sizeof(float);
    static bool prepared_on[64] = {};
    if (int rc = allow_lds(reinterpret_cast<const void *>(&sgemm_tn_square_kernel<TX, TY, WJ>), lds,
                           prepared_on))
        return rc;
    sgemm_tn_square_kernel<TX, TY, WJ><<<r.z0[r.n_problems], 512, lds, stream>>>(r);
    YITU_LAUNCH_CHECK();
    return tn_reduce_launch(r, stream);
}

template <int TX, int TY>
static int sgemm_tn_rows_launch(const TnRowsParams &r, hipStream_t stream) {
    static bool prepared_on[64] = {};
    const int per_wg = std::min(r.roles, 8);
    const size_t lds = (size_t)(r.groups / 2) * per_wg * (16 * TX * TY + TX) * 64 * sizeof(float);
    if (int rc = allow_lds(reinterpret_cast<const void *>(&sgemm_tn_rows_kernel<TX, TY>), lds,
                           prepared_on))
        return rc;
    const dim3 grid((unsigned)r.z0[r.n_problems], (unsigned)ceil_div(r.roles, 8));
    sgemm_tn_rows_kernel<TX, TY><<<grid, 64 * per_wg * r.groups, lds, stream>>>(r);
    YITU_LAUNCH_CHECK();
    return tn_reduce_launch(r, stream);
}

// Takes a group of weight-gradient products [rows, KI]^T . [rows, NO] (`sums`: column sums of
// the A operands wanted, entries may be null); *taken says whether it did.
static int sgemm_tn_rows_try(const GemmParams &p, float *const *sums, int lda, int ldb,
                             void *workspace, size_t workspace_bytes, hipStream_t stream,
                             bool *taken) {
    *taken = false;
    if (p.n_prob < 1 || !workspace || lda > (1 << 24) || ldb > (1 << 24)) return 0;
    const int ki = p.prob[0].M, no = p.N;
    const TnGeometry g = tn_rows_geometry(ki, no);
    if (g.tx == 0) return 0;
    TnRowsParams r{};
    int64_t total = 0;
    for (int i = 0; i < p.n_prob; i++) {
        const GemmProblem &pr = p.prob[i];
        if (pr.M != ki || pr.K < 1) return 0;
        total += pr.K;
    }
    if (total < std::max<int64_t>(512, 256 * p.n_prob)) return 0;  // nothing to split
    bool square = ki == no && (ki == 128 || ki == 256) && lda % 4 == 0 && ldb % 4 == 0;
    for (int i = 0; i < p.n_prob; i++)
        square = square && aligned16(p.prob[i].A) && aligned16(p.prob[i].B);
    const int64_t chunks = square && ki == 128 && total > (1 << 16) ? 512 : tn_rows_chunks(g, total);
    // Few rows for the output's size: writing the slabs and adding them up would take longer
    // than the products (3,000 rows of 64 and 500: 18 us against 13 us for the tiled kernel
    // with its K split; at 0.4 times the operands' size the two break even).
    if (5 * chunks * ki * no > 2 * total * (ki + no)) return 0;
    for (int i = 0; i < p.n_prob; i++) {
        const GemmProblem &pr = p.prob[i];
        const int64_t want = std::max<int64_t>(1, (chunks * (int64_t)pr.K + total / 2) / total);
        r.A[i] = pr.A;
        r.B[i] = pr.B;
        r.C[i] = pr.C;
        r.sums[i] = sums ? sums[i] : nullptr;
        r.want_sums = r.want_sums || r.sums[i];
        r.rows[i] = pr.K;
        r.chunk[i] = (int)ceil_div(pr.K, want);
        r.z0[i + 1] = r.z0[i] + (int)ceil_div(pr.K, r.chunk[i]);
    }
    if ((size_t)r.z0[p.n_prob] * ((size_t)ki * no + ki) * sizeof(float) > workspace_bytes) return 0;
    *taken = true;
    r.n_problems = p.n_prob;
    r.KI = ki;
    r.NO = no;
    r.roles = g.roles();
    r.roles_j = g.roles_j;
    r.groups = g.groups();
    r.accumulate = p.accumulate;
    r.lda = lda;
    r.ldb = ldb;
    r.ldc = p.ldc;
    r.partial = static_cast<float *>(workspace);
    if (square) return ki == 256 ? sgemm_tn_square_launch<2, 4, 2>(r, stream)
                                 : sgemm_tn_square_launch<2, 1, 4>(r, stream);
    switch (10 * g.tx + g.ty) {
        case 11: return sgemm_tn_rows_launch<1, 1>(r, stream);
        case 12: return sgemm_tn_rows_launch<1, 2>(r, stream);
        case 13: return sgemm_tn_rows_launch<1, 3>(r, stream);
        case 14: return sgemm_tn_rows_launch<1, 4>(r, stream);
        case 21: return sgemm_tn_rows_launch<2, 1>(r, stream);
        case 22: return sgemm_tn_rows_launch<2, 2>(r, stream);
        case 23: return sgemm_tn_rows_launch<2, 3>(r, stream);
        case 24: return sgemm_tn_rows_launch<2, 4>(r, stream);
        case 31: return sgemm_tn_rows_launch<3, 1>(r, stream);
        case 32: return sgemm_tn_rows_launch<3, 2>(r, stream);
        case 41: return sgemm_tn_rows_launch<4, 1>(r, stream);
        default: return sgemm_tn_rows_launch<4, 2>(r, stream);
    }
}

}  // namespace yitu
