// Products of many small matrices in one launch, and the routing of a mixture of experts around them.
//
// `grouped_gemm`: out_g[r, n] = act(sum_k a_g[r, k] * w_g[n, k]) for every group g, w_g = w + g * w_group being
// [N, K] row-major.  Two ways of saying which rows a group has:
//   offsets == null: every group takes the rows 0 .. M - 1, group g reading a + g * a_group and writing
//     out + g * out_group with row strides lda / ldo: one projection per head on slices of wider rows;
//   offsets != null: group g takes the rows offsets[g] .. offsets[g + 1] - 1 of a list sorted by group (rows of
//     out; a's row is gather[row] when gather != null): the experts of a routed feed-forward.
// act: none, relu(x)^2, the exact gelu, or one of the gated forms.  Every output element is one sum over k in
// ascending order whatever rows lie beside it, so a row's result does not depend on the batch.  Accumulation is 32-bit; the bfloat16 engine multiplies on
// the matrix cores (v_mfma_f32_16x16x32_bf16, operands staged through LDS), the float engine with plain FMAs.
//
// Routing (32-bit): `router_topk_kernel` (sigmoid or softmax of a token's router logits, the best groups of neighbouring
// experts, the best experts within them), `route_sort_kernel` (the chosen (token, expert) pairs
// sorted by expert: offsets, the token of every sorted row, the sorted row of every pair),
// `route_combine_kernel` (a token's output: the weighted sum of its experts' rows, in the order of its choices, and what
// a shared expert gave).
#include "common.h"
#include <type_traits>

#define ACT_NONE 0
#define ACT_RELU2 1
// (bfloat16 kernels) gated forms: the weight holds a gate's and its up projection's rows in turn, 16 of the one and the
// matching 16 of the other ([gate 0..15 | up 0..15 | gate 16..31 | ...]); out[m, f] = act(gate_f) * up_f, N / 2 columns
#define ACT_GATED_SILU 2
#define ACT_GATED_GELU_TANH 3
// the clamped gate: g = min(gate, limit), u = clamp(up, -limit, limit), out = g sigmoid(slope g) (u + 1)
#define ACT_GATED_CLAMPED 4
#define ACT_GELU_ERF 5

struct GroupedArgs {
    const elem_t* a; long lda; long a_group;
    const elem_t* w; long w_group;
    void* out; long ldo; long out_group;
    const int32_t* offsets; const int32_t* gather;
    int M, N, K, groups, act, out_float;
    float limit, slope;                        // of the clamped gate
};
__host__ __device__ inline bool gated_form(int act) { return act >= ACT_GATED_SILU && act <= ACT_GATED_CLAMPED; }

#define GBM 64              // rows and columns of the small workgroup tile (the float engine's only one)
#define GBN 64

// Which group and which rows this workgroup serves: (group, first row, one beyond the group's last row), or
// group < 0 when the launch has more workgroups than the groups have tiles.
__device__ __forceinline__ void tile_of(const GroupedArgs& g, int& group, int& row0, int& row_end, const int tile_rows = GBM) {
    if (g.offsets == nullptr) {
        group = blockIdx.z;
        row0 = blockIdx.y * tile_rows;
        row_end = g.M;
        return;
    }
    int tile = blockIdx.y;
    group = -1;
    for (int e = 0; e < g.groups; ++e) {
        const int first = g.offsets[e], count = g.offsets[e + 1] - first;
        const int tiles = (count + tile_rows - 1) / tile_rows;
        if (tile < tiles) {
            group = e;
            row0 = first + tile * tile_rows;
            row_end = first + count;
            return;
        }
        tile -= tiles;
    }
}

__device__ __forceinline__ float activate(float x, int act) {
    if (act == ACT_RELU2) {
        const float r = fmaxf(x, 0.f);
        return r * r;
    }
    if (act == ACT_GELU_ERF) return 0.5f * x * (1.0f + erff(x * 0.70710678118654752440f));
    return x;
}

__device__ __forceinline__ float gated(float g, float u, const GroupedArgs& a) {
    if (a.act == ACT_GATED_SILU) return g / (1.0f + expf(-g)) * u;
    if (a.act == ACT_GATED_CLAMPED) {
        g = fminf(g, a.limit);
        u = fminf(fmaxf(u, -a.limit), a.limit);
        return g / (1.0f + expf(-a.slope * g)) * (u + 1.0f);
    }
    return u * 0.5f * g * (1.0f + tanhf(0.79788456080286535588f * (g + 0.044715f * g * g * g)));
}

#if !MLR_BF16
#define GBK 16
__global__ __launch_bounds__(256) void grouped_gemm_kernel(GroupedArgs g) {
    __shared__ float as[GBK][GBM + 4];
    __shared__ float ws[GBK][GBN + 4];
    int group, m0, m_end;
    tile_of(g, group, m0, m_end);
    if (group < 0 || m0 >= m_end) return;
    const int t = threadIdx.x, n0 = blockIdx.x * GBN;
    const int tx = t % 16, ty = t / 16;
    const int lrow = t / 4, lk = (t % 4) * 4;
    const float* a = g.a + (g.offsets ? 0 : (size_t)group * g.a_group);
    const float* w = g.w + (size_t)group * g.w_group;
    float* out = (float*)g.out + (g.offsets ? 0 : (size_t)group * g.out_group);
    long arow = -1;                            // the row of a that this thread stages
    if (m0 + lrow < m_end) arow = g.gather ? g.gather[m0 + lrow] : m0 + lrow;
    float acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;
    for (int k0 = 0; k0 < g.K; k0 += GBK) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int k = k0 + lk + e, wn = n0 + lrow;
            as[lk + e][lrow] = (arow >= 0 && k < g.K) ? a[arow * g.lda + k] : 0.f;
            ws[lk + e][lrow] = (wn < g.N && k < g.K) ? w[(size_t)wn * g.K + k] : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < GBK; ++k) {
            float av[4], wv[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) av[i] = as[k][ty * 4 + i];
#pragma unroll
            for (int j = 0; j < 4; ++j) wv[j] = ws[k][tx * 4 + j];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(av[i], wv[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int m = m0 + ty * 4 + i;
        if (m >= m_end) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int n = n0 + tx * 4 + j;
            if (n < g.N) out[(size_t)m * g.ldo + n] = activate(acc[i][j], g.act);
        }
    }
}
#else
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;
__device__ __forceinline__ bf16x8 load_k8(const __bf16* p, int k, int K, bool vector_ok) {
    bf16x8 v = {0, 0, 0, 0, 0, 0, 0, 0};
    if (vector_ok && k + 8 <= K) {
        v = *reinterpret_cast<const bf16x8*>(p + k);
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
            if (k + e < K) v[e] = p[k + e];
    }
    return v;
}

// A workgroup of 2 x 2 wavefronts, each T x T tiles of 16 x 16: T = 2 owns 64 x 64 outputs and takes k in blocks of
// 128, T = 4 owns 128 x 128 (half the operand traffic an output: for many rows) in blocks of 64.  A block is staged
// through LDS, the next block on its way from memory into registers meanwhile (a block's loads are all asked for
// before anything waits).  Rows of a staged block lie 16 bytes further apart than their data, so that the 16-byte
// reads of 16 rows meet no bank twice.
template <int T>
__global__ __launch_bounds__(256) void grouped_gemm_kernel(GroupedArgs g) {
    constexpr int BM = 32 * T, BN = 32 * T, BK = T == 2 ? 128 : 64, PITCH = BK + 8;
    constexpr int RT = 256 / BM;                     // threads that share a row of a staged operand
    constexpr int CH = BK / 8 / RT;                  // 16-byte chunks of it that one thread stages
    __shared__ __attribute__((aligned(16))) __bf16 as[BM * PITCH];
    __shared__ __attribute__((aligned(16))) __bf16 ws[BN * PITCH];
    int group, m0, m_end;
    tile_of(g, group, m0, m_end, BM);
    if (group < 0 || m0 >= m_end) return;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, n0 = blockIdx.x * BN;
    const int wm = wave >> 1, wn = wave & 1;
    const __bf16* a = g.a + (g.offsets ? 0 : (size_t)group * g.a_group);
    const __bf16* w = g.w + (size_t)group * g.w_group;
    const size_t out_base = g.offsets ? 0 : (size_t)group * g.out_group;
    // 16-byte loads where every row starts at a multiple of 16 bytes
    const bool a_vec = (g.K % 8) == 0 && (g.lda % 8) == 0 && (g.a_group % 8) == 0 &&
                       (reinterpret_cast<uintptr_t>(g.a) % 16) == 0;
    const bool w_vec = (g.K % 8) == 0 && (g.w_group % 8) == 0 && (reinterpret_cast<uintptr_t>(g.w) % 16) == 0;
    const int srow = t / RT, sk = (t % RT) * 8;      // this thread stages row srow of both operands: chunks sk + 8 RT c
    long arow = -1;
    if (m0 + srow < m_end) arow = g.gather ? g.gather[m0 + srow] : m0 + srow;
    const bool wrow_ok = n0 + srow < g.N;
    const __bf16* ap = a + (arow >= 0 ? arow : 0) * g.lda;
    const __bf16* wp = w + (size_t)(wrow_ok ? n0 + srow : 0) * g.K;
    floatx4 acc[T][T];
#pragma unroll
    for (int i = 0; i < T; ++i)
#pragma unroll
        for (int j = 0; j < T; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    const bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
    bf16x8 ar[CH], wr[CH];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            const int k = k0 + sk + 8 * RT * c;
            ar[c] = load_k8(ap, k, g.K, a_vec);
            wr[c] = load_k8(wp, k, g.K, w_vec);
        }
    };
    fetch(0);
    for (int k0 = 0; k0 < g.K; k0 += BK) {
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            *reinterpret_cast<bf16x8*>(&as[srow * PITCH + sk + 8 * RT * c]) = arow >= 0 ? ar[c] : zero;
            *reinterpret_cast<bf16x8*>(&ws[srow * PITCH + sk + 8 * RT * c]) = wrow_ok ? wr[c] : zero;
        }
        __syncthreads();
        if (k0 + BK < g.K) fetch(k0 + BK);
        const int frag_row = lane & 15, frag_k = (lane >> 4) * 8;
#pragma unroll
        for (int kk = 0; kk < BK; kk += 32) {
            bf16x8 af[T], wf[T];
#pragma unroll
            for (int i = 0; i < T; ++i)
                af[i] = *reinterpret_cast<const bf16x8*>(&as[((wm * T + i) * 16 + frag_row) * PITCH + kk + frag_k]);
#pragma unroll
            for (int j = 0; j < T; ++j)
                wf[j] = *reinterpret_cast<const bf16x8*>(&ws[((wn * T + j) * 16 + frag_row) * PITCH + kk + frag_k]);
#pragma unroll
            for (int i = 0; i < T; ++i)
#pragma unroll
                for (int j = 0; j < T; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i], wf[j], acc[i][j], 0, 0, 0);
        }
        __syncthreads();
    }
    // accumulator element r of a lane: row (lane / 16) * 4 + r, column lane % 16
    if (gated_form(g.act)) {
        // a wavefront's neighbouring column tiles hold a gate block and its up block: half as many columns leave
#pragma unroll
        for (int i = 0; i < T; ++i) {
#pragma unroll
            for (int j = 0; j < T; j += 2) {
                if (n0 + (wn * T + j) * 16 + (lane & 15) >= g.N) continue;
                const int n = (n0 >> 1) + ((wn * T + j) >> 1) * 16 + (lane & 15);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int m = m0 + (wm * T + i) * 16 + (lane >> 4) * 4 + r;
                    if (m >= m_end) continue;
                    const float y = gated(acc[i][j][r], acc[i][j + 1][r], g);
                    const size_t at = out_base + (size_t)m * g.ldo + n;
                    if (g.out_float) ((float*)g.out)[at] = y;
                    else ((__bf16*)g.out)[at] = (__bf16)y;
                }
            }
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < T; ++i) {
#pragma unroll
        for (int j = 0; j < T; ++j) {
            const int n = n0 + (wn * T + j) * 16 + (lane & 15);
            if (n >= g.N) continue;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int m = m0 + (wm * T + i) * 16 + (lane >> 4) * 4 + r;
                if (m >= m_end) continue;
                const float y = activate(acc[i][j][r], g.act);
                const size_t at = out_base + (size_t)m * g.ldo + n;
                if (g.out_float) ((float*)g.out)[at] = y;
                else ((__bf16*)g.out)[at] = (__bf16)y;
            }
        }
    }
}

// Experts (inner sizes in multiples of 64): 32 x 32 tiles of v_mfma_f32_32x32x16_bf16 out of LDS blocks
// of 64 k, NS of them, brought by loads that do not pass through registers (`buffer_load_dwordx4 .. lds`).  A workgroup of
// WM x WN wavefronts, each TM x TN tiles, owns 32 WM TM sorted rows of one expert and 32 WN TN of its weight's rows.  The weight
// is the instruction's first operand, so a lane ends up with four consecutive columns of one row (lane = 32 h + i: row i of
// either operand, k slots 8 h .. 8 h + 7; result column i, rows 8 q + 4 h + r in register 4 q + r); with gate and up rows in
// turn, 16 and 16, a gate and its up projection lie in one lane, eight registers apart.
// A row of a block is eight pieces of 16 bytes; a load writes eight rows side by side, so rows cannot be padded apart: piece p
// of row r lies at place p ^ (r & 7), and the eight lanes that the LDS serves together read eight different banks.
// The workgroups' tiles are counted expert by expert, within one a strip of the weight for all of the expert's rows first;
// every XCD takes a contiguous range of those there are, so a strip is fetched into one L2.
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float floatx16;
#define EB_K 64

template <int WM, int WN, int TM, int TN, int NS>
__global__ __launch_bounds__(64 * WM * WN, 2) void experts_wide_kernel(GroupedArgs g) {
    constexpr int BM = 32 * WM * TM, BN = 32 * WN * TN, ROWS = BM + BN, LOADS = ROWS / 8 / (WM * WN), STAGE = ROWS * EB_K;
    static_assert(ROWS % (8 * WM * WN) == 0, "a block's rows must divide among the wavefronts");
    extern __shared__ __attribute__((aligned(16))) __bf16 eb_lds[];
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int li = lane & 31, h = lane >> 5, wm = wave / WN, wn = wave % WN;
    // which tile: every wavefront counts the experts' tiles, a lane an expert, 64 experts at a time
    const int cols = (g.N + BN - 1) / BN;
    int total = 0;
    for (int e0 = 0; e0 < g.groups; e0 += 64) {
        const int e = e0 + lane;
        int n = e < g.groups ? (g.offsets[e + 1] - g.offsets[e] + BM - 1) / BM : 0;
        for (int d = 1; d < 64; d <<= 1) n += __shfl_xor(n, d, MLR_WAVE);
        total += n * cols;
    }
    const int share = (total + 7) / 8;
    const int tile = (int)(blockIdx.x % 8) * share + (int)(blockIdx.x / 8);
    if ((int)(blockIdx.x / 8) >= share || tile >= total) return;
    int group = -1, row0 = 0, row_end = 0, col = 0;
    for (int e0 = 0, before = 0; e0 < g.groups && group < 0; e0 += 64) {
        const int e = e0 + lane;
        const int first = e < g.groups ? g.offsets[e] : 0, count = e < g.groups ? g.offsets[e + 1] - first : 0;
        const int tiles = (count + BM - 1) / BM * cols;
        int upto = tiles;                                                     // tiles of the experts up to this lane's
        for (int d = 1; d < 64; d <<= 1) {
            const int o = __shfl_up(upto, d, MLR_WAVE);
            if (lane >= d) upto += o;
        }
        const int mine = tile - before - (upto - tiles);
        const unsigned long long here = __ballot(mine >= 0 && mine < tiles);
        if (here) {
            const int src = __ffsll((long long)here) - 1;
            group = e0 + src;
            const int at = __shfl(mine, src, MLR_WAVE), f = __shfl(first, src, MLR_WAVE), n = __shfl(count, src, MLR_WAVE);
            const int row_tiles = (n + BM - 1) / BM;
            col = at / row_tiles;
            row0 = f + (at % row_tiles) * BM;
            row_end = f + n;
        }
        before += __shfl(upto, 63, MLR_WAVE);
    }
    group = __builtin_amdgcn_readfirstlane(group);
    if (group < 0) return;
    const int n0 = col * BN, K = g.K, blocks = K / EB_K;
    // Load i of a wavefront brings rows 8 (wave LOADS + i) .. of the block (weight rows first, then the expert's rows; rows beyond
    // either are its last one again), at 32-bit byte offsets from the bases
    uint32_t src[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const int row = (wave * LOADS + i) * 8 + (lane >> 3), piece = ((lane & 7) ^ (row & 7)) * 8;
        if (row < BN) {
            src[i] = ((uint32_t)min(n0 + row, g.N - 1) * (uint32_t)K + piece) * 2u;
        } else {
            const int m = min(row0 + row - BN, row_end - 1);
            src[i] = ((uint32_t)(g.gather ? g.gather[m] : m) * (uint32_t)g.lda + piece) * 2u;
        }
    }
    const auto w_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)(g.w + (size_t)group * g.w_group), 0, (int)((uint32_t)g.N * (uint32_t)K * 2u), 0x00027000);
    const auto a_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)g.a, 0, -1, 0x00027000);        // (the gathered rows are the caller's)
    auto load = [&](int i, int kb, int stage) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds((wave * LOADS + i) * 8 < BN ? w_rsrc : a_rsrc,
                                                 (__attribute__((address_space(3))) void*)(eb_lds + stage * STAGE + (wave * LOADS + i) * 512),
                                                 16, (int)src[i], kb * (EB_K * 2), 0, 0);
    };
    floatx16 acc[TN][TM];
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[j][i][e] = 0.f;
    bf16x8 wf[2][TN], af[2][TM];                                              // the next k step's operands are asked for first
    auto read = [&](int r, int ks, int stage) {
        const __bf16* base = eb_lds + stage * STAGE + li * EB_K + ((2 * ks + h) ^ (li & 7)) * 8;
        if (r < TN) wf[ks & 1][r] = *reinterpret_cast<const bf16x8*>(base + (wn * TN + r) * 32 * EB_K);
        else af[ks & 1][r - TN] = *reinterpret_cast<const bf16x8*>(base + (BN + (wm * TM + r - TN) * 32) * EB_K);
    };
    // The products of k step ks; between them, when READ, the reads of the next step out of block `from` and, when LOAD, the loads
    // of block kb into `into`.  The scheduling barriers keep it so.
    auto products = [&](int ks, bool do_read, int from, bool do_load, int kb, int into) {
        constexpr int OPERANDS = TM + TN, STEPS = TN * TM, PER = STEPS == 1 ? OPERANDS : (OPERANDS + STEPS - 2) / (STEPS > 1 ? STEPS - 1 : 1), PER_L = (LOADS + STEPS - 1) / STEPS;
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            if (do_read) {
#pragma unroll
                for (int r = s * PER; r < (s + 1) * PER && r < OPERANDS; ++r) read(r, (ks + 1) % (EB_K / 16), from);
            }
            if (do_load) {
#pragma unroll
                for (int l = s * PER_L; l < (s + 1) * PER_L && l < LOADS; ++l) load(l, kb, into);
            }
            __builtin_amdgcn_sched_barrier(0);
            acc[s / TM][s % TM] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[ks & 1][s / TM], af[ks & 1][s % TM], acc[s / TM][s % TM], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_s_setprio(0);
    };
    auto read_first = [&](int stage) {
#pragma unroll
        for (int r = 0; r < TM + TN; ++r) read(r, 0, stage);
    };
    if (blocks >= NS) {
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int i = 0; i < LOADS; ++i) load(i, s, s);
        wide_arrive<LOADS * (NS - 1)>();
        read_first(0);
        int stage = 0;
        // A turn: three k steps' products, each beside the next one's reads; the block is read out then and, once everyone is there,
        // is filled again with block kb + NS beside the last step's products, while the next block's first operands arrive.
#pragma unroll 1
        for (int kb = 0; kb < blocks - NS; ++kb) {
            const int next = stage + 1 == NS ? 0 : stage + 1;
            products(0, true, stage, false, 0, 0);
            products(1, true, stage, false, 0, 0);
            products(2, true, stage, false, 0, 0);
            wide_arrive<LOADS * (NS - 2)>();
            products(3, true, next, true, kb + NS, stage);
            stage = next;
        }
        auto tail = [&](auto self, auto left_) {                              // the last NS blocks: nothing more to ask for
            constexpr int LEFT = decltype(left_)::value;
            if constexpr (LEFT > 0) {
                const int next = stage + 1 == NS ? 0 : stage + 1;
                products(0, true, stage, false, 0, 0);
                products(1, true, stage, false, 0, 0);
                products(2, true, stage, false, 0, 0);
                if constexpr (LEFT > 1) wide_arrive<LOADS * (LEFT > 1 ? LEFT - 2 : 0)>();
                products(3, LEFT > 1, next, false, 0, 0);
                stage = next;
                self(self, std::integral_constant<int, LEFT - 1>{});
            }
        };
        tail(tail, std::integral_constant<int, NS>{});
    } else {                                                                  // fewer blocks than the LDS holds: all at once
        for (int s = 0; s < blocks; ++s)
#pragma unroll
            for (int i = 0; i < LOADS; ++i) load(i, s, s);
        wide_arrive<0>();
        for (int s = 0; s < blocks; ++s) {
            read_first(s);
            products(0, true, s, false, 0, 0);
            products(1, true, s, false, 0, 0);
            products(2, true, s, false, 0, 0);
            products(3, false, 0, false, 0, 0);
        }
    }
    // results leave through a piece of LDS of the wavefront's own, as rows of 16-byte pieces
    const bool halves = gated_form(g.act);
    constexpr int OPITCH = TN * 32 + 8, ROWS_W = TM * 32;
    static_assert((size_t)WM * WN * ROWS_W * OPITCH <= (size_t)NS * STAGE, "the output tiles must fit the LDS");
    wide_arrive<0>();                                                         // every wavefront has read its last operands
    __bf16* mine = eb_lds + (size_t)wave * ROWS_W * OPITCH;
    typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float y[4];
                if (halves) {
                    if (q >= 2) continue;
#pragma unroll
                    for (int r = 0; r < 4; ++r) y[r] = gated(acc[j][i][4 * q + r], acc[j][i][4 * q + 8 + r], g);
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r) y[r] = activate(acc[j][i][4 * q + r], g.act);
                }
                *reinterpret_cast<bf16x4*>(mine + (i * 32 + li) * OPITCH + j * (halves ? 16 : 32) + 8 * q + 4 * h) =
                    bf16x4{(__bf16)y[0], (__bf16)y[1], (__bf16)y[2], (__bf16)y[3]};
            }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int width = halves ? TN * 16 : TN * 32, pieces = width / 8, n_out = halves ? g.N / 2 : g.N;
    const int out_n0 = (halves ? n0 / 2 : n0) + wn * width, out_m0 = row0 + wm * TM * 32;
    for (int c = lane; c < ROWS_W * pieces; c += 64) {
        const int row = c / pieces, piece = c % pieces, m = out_m0 + row, n = out_n0 + 8 * piece;
        if (m >= row_end || n >= n_out) continue;
        const bf16x8 v = *reinterpret_cast<const bf16x8*>(mine + row * OPITCH + 8 * piece);
        __bf16* o = (__bf16*)g.out + (size_t)m * g.ldo + n;
        if (n + 8 <= n_out && g.ldo % 8 == 0) {
            *reinterpret_cast<bf16x8*>(o) = v;
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (n + e < n_out) o[e] = v[e];
        }
    }
}

template <int WM, int WN, int TM, int TN, int NS>
static int launch_experts_wide(const GroupedArgs& g, hipStream_t stream) {
    constexpr int BM = 32 * WM * TM, BN = 32 * WN * TN;
    constexpr size_t lds = (size_t)NS * (BM + BN) * EB_K * sizeof(__bf16);
    static const hipError_t allowed = hipFuncSetAttribute(reinterpret_cast<const void*>(&experts_wide_kernel<WM, WN, TM, TN, NS>),
                                                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (allowed != hipSuccess) return (int)allowed;
    const long tiles = ((long)(g.M + BM - 1) / BM + g.groups) * ((g.N + BN - 1) / BN) + 8;      // (at most, and a multiple of 8)
    if (tiles > 0x7ffffff0L) return -2;
    experts_wide_kernel<WM, WN, TM, TN, NS><<<(unsigned)((tiles + 7) / 8 * 8), 64 * WM * WN, lds, stream>>>(g);
    return (int)hipGetLastError();
}

// The kernel's shapes: rows and columns of a workgroup's tile (one on a compute unit at a time), and what a round of tiles takes
// in microseconds: `round` for its first operands and its results, `all` for each 1024 k.  Fitted to 56 products of 4 to 32
// experts with uneven numbers of rows (1088 to 17000 together, 704 to 4096 k, weights out of memory; rms 7 % a shape).
// The shape with the least predicted time took 13 % less than this kernel's predecessor (128 x 128, two blocks staged through
// registers), geometric mean, 0.65 to 1.02 of it, and so would the best of the four.  What bounds it is how evenly the tiles come
// out over the compute units: full rounds of 128 x 256 run at 1.1 PFLOP/s.  Two smaller tiles beside each other on a unit hide less
// of the weight's way from memory (1462 x 2048 x 1408: 29 us, one tile with five blocks under way 22).  In all: 3554 x 2112 x 2048
// of 8 experts 71 -> 54 us, 3554 x 2048 x 2112 52 -> 41, 1462 x 2816 x 2048 with a clamped gate 48 -> 37, 4096 x 12288 x 4096
// gated 542 -> 470.
struct ExpertsCost { int bm, bn; float round, all; };
static const ExpertsCost EXPERTS_COSTS[] = {{128, 128, 5.32f, 9.03f}, {128, 192, 6.74f, 12.02f}, {128, 256, 7.25f, 14.68f}, {192, 256, 9.80f, 21.20f}};

// Fewer rows an expert than fill such tiles half: what counts is the weight's way from memory, so narrow tiles, two workgroups on a
// compute unit, and five or six blocks on their way: 32 x 64 while an expert's rows fit 32, 64 x 64 while they fit 64, or up to 128
// rows while such tiles are no more than compute units (2 experts, 176 x 1088 x 256: 5.7 us, in a tile of 128 x 128 7.9; 4 of 392 x
// 4096 x 1152 15.5, 18.6).  Measured on 126 products of 8 to 64 experts with 1 to 127 rows each (uneven; 704 to 6144 k, 768 to 12288
// rows of weight out of memory) against the kernel that stages through registers, which took all of them before: up to 20 rows 0.83
// of its time, to 55 0.81, beyond, in the tiles above, 0.60 (the bits are the same).  16 experts, 192 rows: 1408 x 2048 gated 27.4 ->
// 23.4 us, 2048 x 704 15.8 -> 12.0 (the weights alone 19 and 10); 8 experts of 64 rows, 2816 x 2048 gated 44.7 -> 28.0.
// Of up to 32 experts the products with a short k are that kernel's (-1): it asks for 128 k at a time and has four workgroups on a
// compute unit, so its whole k is under way at once, while a workgroup here sets out a pipeline of five blocks first, and 512 to 1024
// tiles are one round there and two here.  On 1100 products of 2 to 256 experts (64 to 1152 k, weights out of memory) these tiles took
// below 448 k 0.65 to 1.41 of its time, 0.97 in the mean (32 experts, 79 rows, 4064 x 256 gated: 19.0 us, here 26.7), below 704 with
// more than two tiles a unit 0.69 to 1.17 and 0.93 (16 experts, 39 rows, 3744 x 640 gated: 16.8, 19.6), beyond either line 0.52 to 1.15
// and 0.79.  Of more experts they took 0.11 to 1.08 whatever k: that kernel looks for its expert one after the other.
static int experts_shape_for(int M, int N, int K, int groups) {
    const int units = compute_units() > 0 ? compute_units() : 256;
    if ((long)M < 128L * groups) {
        const long tiles = (long)groups * ((N + 63) / 64);
        const bool one_round = (long)M >= 56L * groups && tiles <= units;
        if (groups <= 32 && !one_round && K < (tiles <= 2 * units ? 448 : 704)) return -1;
        if ((long)M < 56L * groups) return (long)M <= 20L * groups ? 4 : 5;
        if (one_round) return 5;
    }
    int best = 0;
    float least = 0.f;
    for (int s = 0; s < 4; ++s) {
        const ExpertsCost& c = EXPERTS_COSTS[s];
        const float rows = (float)groups * fmaxf((float)M / (float)groups / (float)c.bm + 0.5f, 1.f);      // an expert's last tile is half full
        const float us = ceilf(rows * (float)((N + c.bn - 1) / c.bn) / (float)units) * (c.round + c.all * (float)K * (1.0f / 1024.0f));
        if (s == 0 || us < least) {
            best = s;
            least = us;
        }
    }
    return best;
}

// Whether the kernel takes these operands at all: rows by expert, whole blocks of k, 32-bit byte offsets, rows that start on 16
// bytes.
static bool experts_wide_takes(const GroupedArgs& g, long a_rows) {
    return g.offsets != nullptr && g.N >= 128 && g.K % EB_K == 0 && g.lda % 8 == 0 && g.w_group % 8 == 0 && !g.out_float &&
           ((reinterpret_cast<uintptr_t>(g.a) | reinterpret_cast<uintptr_t>(g.w) | reinterpret_cast<uintptr_t>(g.out)) & 15) == 0 &&
           (unsigned long long)a_rows * g.lda < (1ull << 31) && (unsigned long long)g.N * g.K < (1ull << 31);
}

static int run_experts_wide(int shape, const GroupedArgs& g, hipStream_t stream) {
    switch (shape) {
        case 0: return launch_experts_wide<4, 2, 1, 2, 5>(g, stream);
        case 1: return launch_experts_wide<4, 2, 1, 3, 3>(g, stream);
        case 2: return launch_experts_wide<2, 4, 2, 2, 3>(g, stream);
        case 3: return launch_experts_wide<2, 4, 3, 2, 2>(g, stream);
        case 4: return launch_experts_wide<1, 2, 1, 1, 6>(g, stream);
        case 5: return launch_experts_wide<2, 2, 1, 1, 5>(g, stream);
        default: return -1;
    }
}
#endif

// ---------------------------------------------------------------------------------------------------------
#define MAX_EXPERTS 256         // 64 lanes x EXPERT_REGS
#define EXPERT_REGS 4

struct Routing {
    int experts, top, group_count, group_keep, renorm, softmax, group_best;
    const float* correction;
    float out_scale;
};

// A token a workgroup, an expert a thread.  s = sigmoid(z), or softmax(z) over all experts (`softmax`), z[m * ld ..] the token's router
// logits (float: a product of the framework's own, 32-bit sums).  The experts form `group_count`
// equal groups of neighbours; a group's score is the sum of its two largest s (of its only one, when a group is
// one expert), or its largest (`group_best`); only experts of the `group_keep` best groups stand; of
// those the `top` largest s are chosen (ties: the lower index), ids[m][i] in descending order of s with weights[m][i] = s itself.
// With `correction` [experts] the choice (of groups and of experts) goes by s + correction while the weights stay
// the plain s; with `renorm` the chosen weights are divided by their sum (+ 1e-20); `out_scale` multiplies them.
//
// Bound by its chain of dependent steps, not by work: so a place in the order is counted, by every thread for its own expert against
// all others, where one choice after the other took six exchanges between lanes each, and one group for all needs no rounds.
// 48 tokens, 4 of 20 experts: 7.8 -> 3.4 us; 8 of 64 in 4 of 8 groups 11.6 -> 4.6, of 256 14.7 -> 10.4; 1777 tokens, 4 of 16: 8.7 -> 3.6.
// (The choice and the sort below in one launch of one workgroup, three tokens a wavefront: 10.7 us for 3.4 and 2.0.)
// zr: the token's logits; one wavefront (WAVES 1) needs no other one of its workgroup, of which up to SLOTS choose beside each other,
// each in a slot of its own.
template <int WAVES, int SLOTS = 1>
__device__ __forceinline__ void choose_experts(const float* zr, const Routing& r, int32_t* __restrict__ ids, float* __restrict__ weights, size_t token,
                                               int slot = 0) {
    static_assert(WAVES == 1 || SLOTS == 1, "several wavefronts a token: one token a workgroup");
    auto sync = []() {
        if (WAVES > 1) {
            __syncthreads();
        } else {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
    };
    __shared__ __attribute__((aligned(16))) int keys_lds[SLOTS][64 * WAVES];
    __shared__ float by_lds[SLOTS][64 * WAVES];
    __shared__ float plain_lds[SLOTS][64 * WAVES];
    __shared__ float group_lds[SLOTS][64 * WAVES];
    __shared__ int choice_lds[SLOTS][64 * WAVES];
    int* keys = keys_lds[slot];
    float* by = by_lds[slot];                                              // what the choice goes by
    float* plain = plain_lds[slot];                                        // the plain scores
    float* group = group_lds[slot];
    int* choice = choice_lds[slot];
    const int lane = threadIdx.x % 64, e = WAVES == 1 ? lane : (int)threadIdx.x, experts = r.experts;
    const bool expert = e < experts;
    const float logit = expert ? zr[e] : 0.f;
    float z_max = 0.f, z_sum = 1.f, cand = -INFINITY;
    if (r.softmax) {                                                       // (each wavefront by itself)
        z_max = -INFINITY;
        for (int o = lane; o < experts; o += 64) z_max = fmaxf(z_max, zr[o]);
        z_max = wave_max(z_max);
        z_sum = 0.f;
        for (int o = lane; o < experts; o += 64) z_sum += expf(zr[o] - z_max);
        z_sum = wave_sum(z_sum);
    }
    if (expert) {
        const float sc = r.softmax ? expf(logit - z_max) / z_sum : 1.0f / (1.0f + expf(-logit));
        plain[e] = sc;
        cand = r.correction != nullptr ? sc + r.correction[e] : sc;
    }
    if (e < r.top) choice[e] = 0;                                          // (fewer candidates than `top`: refused on the host)
    const int per = experts / r.group_count;
    if (r.group_count == 1) {
        // the group stands if its score is more than -inf: two of its values (or one) are
        const int there = WAVES == 1 ? __popcll(__ballot(cand > -INFINITY)) : __syncthreads_count(cand > -INFINITY);
        if (there < (per >= 2 && !r.group_best ? 2 : 1)) cand = -INFINITY;
    } else {
        by[e] = cand;
        sync();
        if (e < r.group_count) {
            float first = -INFINITY, second = -INFINITY;
            for (int i = 0; i < per; ++i) {
                const float v = by[e * per + i];
                if (v > first) {
                    second = first;
                    first = v;
                } else if (v > second) {
                    second = v;
                }
            }
            group[e] = per >= 2 && !r.group_best ? first + second : first;
        }
        sync();
        if (expert) {
            const int mine = e / per;
            const float score = group[mine];
            int before = 0;
            for (int g = 0; g < r.group_count; ++g) {
                const float v = group[g];
                before += v > score || (v == score && g < mine) ? 1 : 0;
            }
            if (!(score > -INFINITY && before < r.group_keep)) cand = -INFINITY;
        }
    }
    // As whole numbers in the order of the floats (no candidate: the lowest), so that among equals the lower index is the larger by one
    // subtraction: four operations a pair, none of them on masks.
    constexpr int NONE = -0x7fffffff - 1;
    const int bits = __float_as_int(cand + 0.0f);                          // (0 for -0)
    const int key = cand > -INFINITY ? bits ^ ((bits >> 31) & 0x7fffffff) : NONE;
    keys[e] = key;
    sync();
    int before = 0;
    for (int j = 0; j < experts; j += 16) {                                // (16 at once: their reads are under way together)
        int4 v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = *reinterpret_cast<const int4*>(&keys[j + 4 * q]);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int at = j + 4 * q;
            before += v[q].x > key - (at < e ? 1 : 0) ? 1 : 0;
            before += v[q].y > key - (at + 1 < e ? 1 : 0) ? 1 : 0;
            before += v[q].z > key - (at + 2 < e ? 1 : 0) ? 1 : 0;
            before += v[q].w > key - (at + 3 < e ? 1 : 0) ? 1 : 0;
        }
    }
    if (key != NONE && before < r.top) choice[before] = e;
    sync();
    if (e >= r.top) return;
    const int which = choice[e];
    float w = plain[which];
    if (r.renorm) {
        float sum = 0.f;
        for (int c = 0; c < r.top; ++c) sum += plain[choice[c]];           // (in the order of the choices)
        w = w / (sum + 1e-20f);
    }
    ids[token * r.top + e] = which;
    weights[token * r.top + e] = r.renorm || r.out_scale != 1.0f ? w * r.out_scale : w;
}

template <int WAVES>
__global__ __launch_bounds__(64 * WAVES) void router_topk_kernel(const float* __restrict__ z, long ld, Routing r,
                                                                 int32_t* __restrict__ ids, float* __restrict__ weights) {
    choose_experts<WAVES>(z + (size_t)blockIdx.x * ld, r, ids, weights, blockIdx.x);
}

#if MLR_BF16
// The router's product with the choice behind it: TOKENS tokens a workgroup, z[e] = x . w[e] for all `outputs` rows of w (the experts,
// and beyond them a shared expert's gate) in 32-bit, written to z and chosen from.  Eight wavefronts take every eighth row, a lane eight
// neighbouring channels of every 512, in the order of the channels, and the lanes' sums by halves (`wave_sum`): a token's logits depend
// neither on the others nor on how many they are.
// Few tokens, one a workgroup: bound by its chain of trips -- row and weights, the lanes' sums, the choice -- where the product alone was
// a launch of two or three workgroups.  48 tokens, 20 outputs of 2048 channels 7.4 -> 5.0 us, 732 tokens, 8 outputs 8.9 -> 5.1.
// Many, four a workgroup from ROUTER_MANY on: bound by what the workgroups read out of the L2, the whole weight each.  One and four
// tokens a workgroup, us: 768 x 20 outputs of 2048 channels 7.5, 7.4; 1024 x 8 5.6, 5.2; 2048 x 8 7.7, 6.7; 2048 x 20 12.6, 10.0;
// 8192 x 20 39.6, 24.0.  (The product by matrix instructions, 16 tokens a workgroup, is slower up to 2048 tokens: 48 x 20 7.9.)
#define ROUTER_OUTPUTS 128
#define ROUTER_WAVES 8
#define ROUTER_MANY 768
template <int TOKENS, int AT_ONCE, int AHEAD>          // AT_ONCE: rows of w a wavefront takes side by side; AHEAD: times 512 channels
__global__ __launch_bounds__(64 * ROUTER_WAVES) void router_kernel(const __bf16* __restrict__ x, const __bf16* __restrict__ w,
                                                                   float* __restrict__ z, long ld, int rows, int width, int outputs, Routing r,
                                                                   int32_t* __restrict__ ids, float* __restrict__ weights) {
    typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2;
    struct eight { bf16x2 pair[4]; };
    static_assert(TOKENS <= ROUTER_WAVES, "a wavefront chooses for one token");
    __shared__ float z_lds[TOKENS][ROUTER_OUTPUTS];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int first = blockIdx.x * TOKENS;
    for (int e0 = wave; e0 < outputs; e0 += ROUTER_WAVES * AT_ONCE) {
        float sum[TOKENS][AT_ONCE] = {};
        for (int c0 = 0; c0 < width; c0 += 512 * AHEAD) {
            vec16 v[TOKENS][AHEAD], u[AT_ONCE][AHEAD];
#pragma unroll
            for (int q = 0; q < AHEAD; ++q) {                              // (clamped: no branch around a load)
                const int at = min(c0 + 512 * q + 8 * lane, width - 8);
#pragma unroll
                for (int i = 0; i < TOKENS; ++i) v[i][q] = *reinterpret_cast<const vec16*>(x + (size_t)min(first + i, rows - 1) * width + at);
#pragma unroll
                for (int j = 0; j < AT_ONCE; ++j)
                    u[j][q] = *reinterpret_cast<const vec16*>(w + (size_t)min(e0 + ROUTER_WAVES * j, outputs - 1) * width + at);
            }
#pragma unroll
            for (int q = 0; q < AHEAD; ++q) {
                const bool beyond = c0 + 512 * q + 8 * lane >= width;
#pragma unroll
                for (int i = 0; i < TOKENS; ++i)
                    if (beyond) v[i][q] = vec16{{0, 0, 0, 0}};
#pragma unroll
                for (int j = 0; j < AT_ONCE; ++j) {
                    // (an expert that is not finite does not reach a token through channels that are not there)
                    if (beyond) u[j][q] = vec16{{0, 0, 0, 0}};
                    const eight b = __builtin_bit_cast(eight, u[j][q]);
#pragma unroll
                    for (int i = 0; i < TOKENS; ++i) {
                        const eight a = __builtin_bit_cast(eight, v[i][q]);
#pragma unroll
                        for (int e = 0; e < 4; ++e) sum[i][j] = __builtin_amdgcn_fdot2_f32_bf16(a.pair[e], b.pair[e], sum[i][j], false);
                    }
                }
            }
        }
#pragma unroll
        for (int i = 0; i < TOKENS; ++i)
#pragma unroll
            for (int j = 0; j < AT_ONCE; ++j) {
                const float total = wave_sum(sum[i][j]);
                if (lane == 0 && e0 + ROUTER_WAVES * j < outputs) z_lds[i][e0 + ROUTER_WAVES * j] = total;
            }
    }
    __syncthreads();
    const int token = first + wave;
    if (wave >= TOKENS || token >= rows) return;
    for (int e = lane; e < outputs; e += 64) z[(size_t)token * ld + e] = z_lds[wave][e];
    choose_experts<1, TOKENS>(z_lds[wave], r, ids, weights, token, wave);
}
#endif

// The same, one choice after the other, a wavefront a token: a round is six exchanges between the lanes' best.
// The largest value among the lanes' candidates and, among equals, the lowest index; every lane gets both.
__device__ __forceinline__ void wave_best(float& value, int& index) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const float ov = __shfl_xor(value, off, MLR_WAVE);
        const int oi = __shfl_xor(index, off, MLR_WAVE);
        if (ov > value || (ov == value && oi < index)) {
            value = ov;
            index = oi;
        }
    }
}

__global__ __launch_bounds__(64) void router_rounds_kernel(const float* __restrict__ z, long ld, Routing r,
                                                           int32_t* __restrict__ ids, float* __restrict__ weights) {
    __shared__ float s_lds[MAX_EXPERTS];      // what the choice goes by
    __shared__ float w_lds[MAX_EXPERTS];      // the plain scores
    __shared__ float g_lds[MAX_EXPERTS];
    const int m = blockIdx.x, lane = threadIdx.x, experts = r.experts, top = r.top, group_count = r.group_count;
    const float* zr = z + (size_t)m * ld;
    float z_max = 0.f, z_sum = 1.f;
    if (r.softmax) {
        z_max = -INFINITY;
        for (int e = lane; e < experts; e += 64) z_max = fmaxf(z_max, zr[e]);
        z_max = wave_max(z_max);
        z_sum = 0.f;
        for (int e = lane; e < experts; e += 64) z_sum += expf(zr[e] - z_max);
        z_sum = wave_sum(z_sum);
    }
    for (int e = lane; e < experts; e += 64) {
        const float sc = r.softmax ? expf(zr[e] - z_max) / z_sum : 1.0f / (1.0f + expf(-zr[e]));
        w_lds[e] = sc;
        s_lds[e] = r.correction != nullptr ? sc + r.correction[e] : sc;
    }
    __syncthreads();
    const int per = experts / group_count;
    for (int gidx = lane; gidx < group_count; gidx += 64) {
        float first = -INFINITY, second = -INFINITY;
        for (int i = 0; i < per; ++i) {
            const float v = s_lds[gidx * per + i];
            if (v > first) {
                second = first;
                first = v;
            } else if (v > second) {
                second = v;
            }
        }
        g_lds[gidx] = per >= 2 && !r.group_best ? first + second : first;
    }
    __syncthreads();
    // the groups that stand: r.group_keep times the best of those left; their experts become candidates
    float cand[EXPERT_REGS];
#pragma unroll
    for (int i = 0; i < EXPERT_REGS; ++i) cand[i] = -INFINITY;
    for (int round = 0; round < r.group_keep; ++round) {
        float best = -INFINITY;
        int which = 0x7fffffff;
        for (int gidx = lane; gidx < group_count; gidx += 64) {
            const float v = g_lds[gidx];
            if (v > best) {                    // (ascending indices: the lowest among equals stays)
                best = v;
                which = gidx;
            }
        }
        wave_best(best, which);
        if (which == 0x7fffffff) break;
        __syncthreads();
        if (lane == 0) g_lds[which] = -INFINITY;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < EXPERT_REGS; ++i) {
            const int e = lane + 64 * i;
            if (e < experts && e / per == which) cand[i] = s_lds[e];
        }
    }
    float chosen_sum = 0.f;
    for (int round = 0; round < top; ++round) {
        float best = -INFINITY;
        int which = 0x7fffffff;
#pragma unroll
        for (int i = 0; i < EXPERT_REGS; ++i) {
            const int e = lane + 64 * i;
            if (e < experts && cand[i] > best) {
                best = cand[i];
                which = e;
            }
        }
        wave_best(best, which);
        if (which == 0x7fffffff) which = 0, best = 0.f;      // (fewer candidates than `top`: refused on the host)
#pragma unroll
        for (int i = 0; i < EXPERT_REGS; ++i)
            if (lane + 64 * i == which) cand[i] = -INFINITY;
        chosen_sum += w_lds[which];                           // (the same on every lane, in the order of the choices)
        if (lane == 0) {
            ids[(size_t)m * top + round] = which;
            weights[(size_t)m * top + round] = w_lds[which];
        }
    }
    if (r.renorm || r.out_scale != 1.0f) {
        __syncthreads();
        for (int c = lane; c < top; c += 64) {
            float w = weights[(size_t)m * top + c];
            if (r.renorm) w = w / (chosen_sum + 1e-20f);
            weights[(size_t)m * top + c] = w * r.out_scale;
        }
    }
}

// Which of the two a step takes, by their predicted times (us).  Counting is a comparison of every expert with every other in four
// wavefronts, so it is bound by that work once the tokens are many; the rounds' time is their number, and one lane's walk over the
// scores of a group.  Up to 64 experts counting is the faster one always (0.23 to 0.97 of the rounds' time).  Measured, rounds and
// counting: 8 of 256 in 4 of 8 groups 13.0 and 9.3 for one token, 15.6 and 21.9 for 2048; 6 of 160 16.7 and 5.7, 2048 tokens 21.3 and
// 13.5, 4096 20.9 and 23.0; 1 of 256 in 1 of 8 groups 6.3 and 9.2.  (By this line 72 to 256 experts, 1 to 4096 tokens, 1 to 12 chosen
// took 0.27 to 1.01 of the rounds' time.)
static bool choose_in_rounds(const Routing& r, int rows) {
    if (r.experts <= 64) return false;
    const float per = (float)(r.experts / r.group_count), m = (float)rows, e = (float)r.experts;
    const float rounds = 2.6f + 0.06f * per + 0.67f * (float)(r.group_keep + r.top) + 0.0007f * m;
    const float counting = 2.4f + 0.018f * e + (r.group_count > 1 ? 0.5f + 0.055f * per : 0.f) + m * (0.0008f + 2.26e-5f * e);
    return rounds < counting;
}

// Where the experts' rows of the sorted list start: start[e] the sum of count[0 .. e - 1], offsets[experts] of all; one wavefront
// (one thread from expert to expert: 256 of them, 4.6 us of the sort below for 3.0).
__device__ __forceinline__ void expert_starts(const int* count, int experts, int* start, int32_t* __restrict__ offsets) {
    const int lane = threadIdx.x % 64;
    int before = 0;
    for (int e0 = 0; e0 < experts; e0 += 64) {
        const int own = e0 + lane < experts ? count[e0 + lane] : 0;
        int sum = own;
#pragma unroll
        for (int off = 1; off < 64; off *= 2) {
            const int other = __shfl_up(sum, off, MLR_WAVE);
            if (lane >= off) sum += other;
        }
        if (e0 + lane < experts) offsets[e0 + lane] = start[e0 + lane] = before + sum - own;
        before += __shfl(sum, 63, MLR_WAVE);
    }
    if (lane == 0) offsets[experts] = before;
}

// The `pairs` chosen (token, expert) pairs sorted by expert, by ONE workgroup: offsets[e] .. offsets[e + 1] are
// expert e's rows of the sorted list, token_of[row] the pair's token, row_of[pair] where the pair went.  The
// order of an expert's rows among themselves is whatever the atomics give; no result depends on it.
__global__ __launch_bounds__(1024) void route_sort_kernel(const int32_t* __restrict__ ids, int pairs, int top,
                                                          int experts, int32_t* __restrict__ offsets,
                                                          int32_t* __restrict__ token_of, int32_t* __restrict__ row_of) {
    __shared__ int count[MAX_EXPERTS];
    __shared__ int cursor[MAX_EXPERTS];
    const int t = threadIdx.x;
    for (int e = t; e < experts; e += blockDim.x) count[e] = 0;
    __syncthreads();
    for (int i = t; i < pairs; i += blockDim.x) atomicAdd(&count[ids[i]], 1);
    __syncthreads();
    if (t < 64) expert_starts(count, experts, cursor, offsets);
    __syncthreads();
    for (int i = t; i < pairs; i += blockDim.x) {
        const int row = atomicAdd(&cursor[ids[i]], 1);
        token_of[row] = i / top;
        row_of[i] = row;
    }
}

// out[m, :] = sum_i weights[m][i] * y[row_of[m * top + i], :], the sum in 32-bit in the order of the choices; with
// `shared` [rows, width] plus shared[m, :], times sigmoid(shared_gate[m * gate_stride]) when that is given.  With `ids`
// [rows, top] a choice ids[m * top + i] >= experts stands for an expert that gives its input back: x[m, :] takes its row's
// place (no row of y was computed for it).
// VEC: MLR_VEC values in one access, or 1.
template <int VEC>
__global__ void route_combine_kernel(const elem_t* __restrict__ y, const int32_t* __restrict__ row_of,
                                     const float* __restrict__ weights, elem_t* __restrict__ out, int width, int top,
                                     const elem_t* __restrict__ shared, const float* __restrict__ shared_gate, long gate_stride,
                                     const int32_t* __restrict__ ids, int experts, const elem_t* __restrict__ x) {
    const int m = blockIdx.x;
    auto source = [&](int i) {
        if (ids != nullptr && ids[(size_t)m * top + i] >= experts) return x + (size_t)m * width;
        return y + (size_t)row_of[(size_t)m * top + i] * width;
    };
    const float f = shared_gate != nullptr ? 1.0f / (1.0f + expf(-shared_gate[(size_t)m * gate_stride])) : 1.0f;
    if (VEC > 1) {
        for (int c = threadIdx.x * VEC; c < width; c += blockDim.x * VEC) {
            float sum[MLR_VEC], v[MLR_VEC];
#pragma unroll
            for (int e = 0; e < MLR_VEC; ++e) sum[e] = 0.f;
            for (int i = 0; i < top; ++i) {
                const float w = weights[(size_t)m * top + i];
                load_vec(source(i) + c, v);
#pragma unroll
                for (int e = 0; e < MLR_VEC; ++e) sum[e] = fmaf(w, v[e], sum[e]);
            }
            if (shared != nullptr) {
                load_vec(shared + (size_t)m * width + c, v);
#pragma unroll
                for (int e = 0; e < MLR_VEC; ++e) sum[e] = fmaf(f, v[e], sum[e]);
            }
            store_vec(out + (size_t)m * width + c, sum);
        }
        return;
    }
    for (int c = threadIdx.x; c < width; c += blockDim.x) {
        float sum = 0.f;
        for (int i = 0; i < top; ++i)
            sum = fmaf(weights[(size_t)m * top + i], to_float(source(i)[c]), sum);
        if (shared != nullptr) sum = fmaf(f, to_float(shared[(size_t)m * width + c]), sum);
        out[(size_t)m * width + c] = from_float<elem_t>(sum);
    }
}

extern "C" {

int mlr_grouped_gemm(const void* a, long lda, long a_group, const void* w, long w_group, void* out, long ldo,
                     long out_group, const int32_t* offsets, const int32_t* gather, int M, int N, int K, int groups,
                     int act, int out_float, float limit, float slope, long a_rows, hipStream_t stream) {
    if (M <= 0 || N <= 0 || groups <= 0) return 0;
    if (K <= 0 || act < ACT_NONE || act > ACT_GELU_ERF || (act == ACT_GATED_CLAMPED && !(limit > 0.f))) return -1;
#if !MLR_BF16
    if (gated_form(act)) return -3;            // (the gated forms are the matrix-core kernels')
    out_float = 1;
#else
    if (gated_form(act) && N % 32 != 0) return -3;
#endif
    GroupedArgs g{(const elem_t*)a, lda, a_group, (const elem_t*)w, w_group, out, ldo, out_group, offsets, gather,
                  M, N, K, groups, act, out_float, limit, slope};
#if MLR_BF16
    // rows by expert (the products a head, with inner sizes of 128 to 512, are faster on the small tile below)
    const int shape = experts_wide_takes(g, a_rows) ? experts_shape_for(M, N, K, groups) : -1;
    if (shape >= 0) return run_experts_wide(shape, g, stream);
    if (offsets != nullptr && (long)M >= 256L * groups && N >= 128) {
        const int row_tiles = (M + 127) / 128 + (offsets ? groups : 0);
        if (row_tiles > 65535 || groups > 65535) return -2;
        grouped_gemm_kernel<4><<<dim3((N + 127) / 128, row_tiles, offsets ? 1 : groups), 256, 0, stream>>>(g);
        return (int)hipGetLastError();
    }
#endif
    const int row_tiles = (M + GBM - 1) / GBM + (offsets ? groups : 0);
    if (row_tiles > 65535 || groups > 65535) return -2;
    dim3 grid((N + GBN - 1) / GBN, row_tiles, offsets ? 1 : groups);
#if MLR_BF16
    grouped_gemm_kernel<2><<<grid, 256, 0, stream>>>(g);
#else
    grouped_gemm_kernel<<<grid, 256, 0, stream>>>(g);
#endif
    return (int)hipGetLastError();
}

// For tests: the shape that the products of experts take, -1 for the kernel that stages through registers.
int mlr_experts_shape(int M, int N, int K, int groups) {
#if MLR_BF16
    return N >= 128 && K % EB_K == 0 ? experts_shape_for(M, N, K, groups) : -1;
#else
    return -1;
#endif
}

// For tests and measurements: the products of experts in a given shape (0 .. 5).
int mlr_experts_wide(const void* a, const void* w, void* out, const int32_t* offsets, const int32_t* gather, int M, int N, int K,
                     int groups, int act, int shape, long a_rows, hipStream_t stream) {
#if MLR_BF16
    if (M <= 0 || N <= 0 || groups <= 0 || K <= 0 || act < ACT_NONE || act > ACT_GELU_ERF || act == ACT_GATED_CLAMPED) return -1;
    GroupedArgs g{(const elem_t*)a, K, 0, (const elem_t*)w, (long)N * K, out, gated_form(act) ? N / 2 : N, 0, offsets, gather,
                  M, N, K, groups, act, 0, 0.f, 0.f};
    if ((gated_form(act) && N % 32 != 0) || !experts_wide_takes(g, a_rows)) return -1;
    return run_experts_wide(shape, g, stream);
#else
    return -3;
#endif
}

int mlr_router_topk(const float* z, long ld, int32_t* ids, float* weights, int rows, int experts, int top, int group_count,
                    int group_keep, const float* correction, int renorm, float out_scale, int softmax, int group_best,
                    hipStream_t stream) {
    if (rows <= 0) return 0;
    if (ld < experts || experts < 1 || experts > MAX_EXPERTS || group_count < 1 || experts % group_count != 0 || group_keep < 1 ||
        group_keep > group_count || top < 1 || top > group_keep * (experts / group_count))
        return -1;
    const Routing r{experts, top, group_count, group_keep, renorm, softmax, group_best, correction, out_scale};
    if (choose_in_rounds(r, rows)) router_rounds_kernel<<<rows, 64, 0, stream>>>(z, ld, r, ids, weights);
    else if (experts <= 64) router_topk_kernel<1><<<rows, 64, 0, stream>>>(z, ld, r, ids, weights);
    else router_topk_kernel<4><<<rows, 256, 0, stream>>>(z, ld, r, ids, weights);
    return (int)hipGetLastError();
}

// z = x . w^T (bfloat16, `outputs` rows of w, float sums) and the choice of `mlr_router_topk` from its first `experts` columns, in one
// launch; 1 where it does not take the sizes (more than 64 experts, rows that do not come in 16 bytes): nothing was launched.
int mlr_router(const void* x, const void* w, float* z, long ld, int32_t* ids, float* weights, int rows, int width, int outputs, int experts,
               int top, int group_count, int group_keep, const float* correction, int renorm, float out_scale, int softmax, int group_best,
               hipStream_t stream) {
#if MLR_BF16
    if (rows <= 0) return 0;
    if (outputs < experts || ld < outputs || experts < 1 || group_count < 1 || experts % group_count != 0 || group_keep < 1 ||
        group_keep > group_count || top < 1 || top > group_keep * (experts / group_count))
        return -1;
    if (experts > 64 || outputs > ROUTER_OUTPUTS || width < 8 || width % 8 != 0 ||
        ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) & 15) != 0)
        return 1;
    const Routing r{experts, top, group_count, group_keep, renorm, softmax, group_best, correction, out_scale};
    const int step = rows >= ROUTER_MANY ? 4 : 1;
    auto* kernel = step > 1 ? (outputs <= ROUTER_WAVES ? router_kernel<4, 1, 2> : outputs <= 2 * ROUTER_WAVES ? router_kernel<4, 2, 2> : router_kernel<4, 3, 2>)
                            : (outputs <= ROUTER_WAVES ? router_kernel<1, 1, 4> : outputs <= 2 * ROUTER_WAVES ? router_kernel<1, 2, 4> : router_kernel<1, 3, 4>);
    kernel<<<(rows + step - 1) / step, 64 * ROUTER_WAVES, 0, stream>>>((const __bf16*)x, (const __bf16*)w, z, ld, rows, width, outputs, r, ids, weights);
    return (int)hipGetLastError();
#else
    return 1;
#endif
}

int mlr_route_sort(const int32_t* ids, int pairs, int top, int experts, int32_t* offsets, int32_t* token_of,
                   int32_t* row_of, hipStream_t stream) {
    if (pairs <= 0) return 0;
    if (experts < 1 || experts > MAX_EXPERTS || top < 1) return -1;
    route_sort_kernel<<<1, 1024, 0, stream>>>(ids, pairs, top, experts, offsets, token_of, row_of);
    return (int)hipGetLastError();
}

int mlr_route_combine(const void* y, const int32_t* row_of, const float* weights, void* out, int rows, int width,
                      int top, const void* shared, const float* shared_gate, long gate_stride, const int32_t* ids, int experts,
                      const void* x, hipStream_t stream) {
    if (rows <= 0) return 0;
    if ((ids == nullptr) != (x == nullptr)) return -1;
    const bool vec = width % MLR_VEC == 0 && ((reinterpret_cast<uintptr_t>(y) | reinterpret_cast<uintptr_t>(out) |
                                              reinterpret_cast<uintptr_t>(shared) | reinterpret_cast<uintptr_t>(x)) & 15) == 0;
    if (vec)
        route_combine_kernel<MLR_VEC><<<rows, 256, 0, stream>>>((const elem_t*)y, row_of, weights, (elem_t*)out, width, top,
                                                                (const elem_t*)shared, shared_gate, gate_stride, ids, experts,
                                                                (const elem_t*)x);
    else
        route_combine_kernel<1><<<rows, 256, 0, stream>>>((const elem_t*)y, row_of, weights, (elem_t*)out, width, top,
                                                          (const elem_t*)shared, shared_gate, gate_stride, ids, experts,
                                                          (const elem_t*)x);
    return (int)hipGetLastError();
}

}  // extern "C"
