// out[M, N] = a[M, K] . w[N, K]^T  (both operands row-major with K contiguous, the layout of
// an activation and of a projection's weight), accumulated in 32-bit.
//
// Float engine: 32-bit matrix instructions, a wavefront a strip of columns for few rows and tiles for many; every element is
// one chain of fmaf over k from 0 up, so a row's result does not depend on the other rows of the batch.
// Bfloat16 engine, three families, each with a fixed k order for every output element (so a row's result
// does not depend on the rows beside it): up to 16 rows, and to 64 where `few_wins` does not say otherwise, the weight is
// streamed once straight into v_mfma_f32_16x16x32_bf16 (`gemm_skinny_kernel`, optionally with the residual add and RMSNorm in
// front or silu(gate) * up behind); more rows with k a multiple of 64 go to `gemm_wide_kernel` (tiles out of
// blocks of LDS that loads fill without passing through registers), and so do the rows that `few_wins` names, in a form with the
// first kernel's order; any other k to the plain 16x16-tile kernel `gemm_bf16_kernel`.
#include "common.h"
#include <type_traits>

#if !MLR_BF16
// ------------------------------------------------------------------------------ float
// v_mfma_f32_16x16x4_f32 rounds as four fmaf one behind the other in the order of its k-slots, so an element is ONE chain of
// fmaf over k from 0 up, whatever kernel and tile serve it: its bits hang neither on the rows beside it nor on how a step was
// cut, and a plain loop over k gives the same.  A matrix instruction wants k-slot b from lanes 16 b ..; a 16-byte load gives a
// lane four neighbouring k of one row, so four lane blocks exchange (`turned`): product i of a group of 16 takes k = 4 i + b.
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;

// Four consecutive k of a row from k on, zeros from K on (VEC: rows start on 16 bytes and K is a multiple of four).
template <bool VEC>
__device__ __forceinline__ floatx4 load_k4(const float* __restrict__ row, int k, int K) {
    floatx4 v = {0.f, 0.f, 0.f, 0.f};
    if (VEC) {
        if (k < K) v = *reinterpret_cast<const floatx4*>(row + k);
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (k + e < K) v[e] = row[k + e];
    }
    return v;
}

// Few tiles of 16 x 16: a wavefront owns 16 rows and NT strips of 16 columns and walks all of k alone.  The chain of products is
// the bound (measured alone 13.6 ns, 32.5 clocks, for every four k), so nothing else may stand in its way.  A wavefront cannot
// wait for memory inside it, so it has up to STAGES - 1 stages of 64 k under way, 448 k or 1.5 us of products: loads that go to
// LDS without passing registers (`buffer_load_dwordx4 .. lds`, a lane's 16 bytes at 16 bytes of its own), for which the registers
// would not do -- with blocks of 128 k in registers, one under way, every block waited for memory and four k took 20 ns.  The
// exchange between lane blocks is left to LDS (4-byte reads of what a lane needs, free of bank conflicts; no other wavefront
// takes part); a group of 16 k is read one ahead, a share of it behind each product.
// 8 rows of 4096 x 1024, 1024 x 2048, 6144 x 1024, 1024 x 3072, weights cold: 7.6, 11.5, 10.2 and 15.6 us (9.6, 14.2, 11.9,
// 19.5 with blocks in registers).
template <int LEFT> __device__ __forceinline__ void strip_wait() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LEFT) : "memory"); }

// The products of one wavefront: `a` and `w` start at its first row of each, of which there are a_rows and w_rows (more than that
// are the last one again); lds: [STAGES][G][1 + NT][256] floats of its own.
constexpr int STRIP_K = 1 << 25;                           // k must be below: a strip's 32 rows then lie within 32 bits of bytes
template <int NT, int STAGES> constexpr int strip_lds_floats() { return STAGES * 4 * (1 + NT) * 256; }
template <int NT, int STAGES>
__device__ __forceinline__ void f32_strip(const float* __restrict__ a, const float* __restrict__ w, int a_rows, int w_rows, int K,
                                          float* lds, floatx4 (&acc)[NT]) {
    constexpr int P = 1 + NT, G = 4, LOADS = G * P, STAGE = LOADS * 256;
    static_assert(STAGES >= 3 && STAGES <= 8 && P <= 4 && LOADS * (STAGES - 1) <= 63, "the counter of loads in flight has six bits");
    const int lane = threadIdx.x & 63, r = lane & 15, b = lane >> 4;
    uint32_t row[P];                                       // the lane's row of a and of every strip, in bytes from the first
    row[0] = (uint32_t)min(r, a_rows - 1) * (uint32_t)K * 4u;
#pragma unroll
    for (int j = 0; j < NT; ++j) row[1 + j] = (uint32_t)min(j * 16 + r, w_rows - 1) * (uint32_t)K * 4u;
    const auto ar = __builtin_amdgcn_make_buffer_rsrc((void*)a, 0, (int)((uint32_t)K * 64u), 0x00027000);
    const auto wr = __builtin_amdgcn_make_buffer_rsrc((void*)w, 0, (int)((uint32_t)K * (64u * NT)), 0x00027000);
    const int stages = (K + 16 * G - 1) / (16 * G), full = K / (16 * G);
    constexpr std::true_type yes{};
    constexpr std::false_type no{};
    // (whole: every place lies before K; otherwise places behind it are the row's last ones again, and what is read there counts as zero)
    auto load = [&](int t, int u, int j, int slot, bool whole) {
        const int k0 = (t * G + u) * 16;
        uint32_t at = row[j];
        if (!whole) at += (uint32_t)min(k0 + b * 4, K - 4) * 4u;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(j == 0 ? ar : wr, (__attribute__((address_space(3))) void*)(lds + slot * STAGE + (u * P + j) * 256), 16,
                                                 (int)at, whole ? k0 * 4 : 0, 0, 0);
    };
    auto wait_for = [&](int behind) {                      // all but the last `behind` stages that were asked for are there
        if (behind >= STAGES - 2) strip_wait<LOADS * (STAGES - 2)>();
        else if (behind == 1) strip_wait<LOADS>();
        else if (behind == 2) strip_wait<2 * LOADS>();
        else if (behind == 3) strip_wait<3 * LOADS>();
        else if (behind == 4) strip_wait<4 * LOADS>();
        else if (behind == 5) strip_wait<5 * LOADS>();
        else strip_wait<0>();
    };
    floatx4 now[P], next[P];
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[j] = floatx4{0.f, 0.f, 0.f, 0.f};
    const float* mine = lds + r * 4 + b;
    auto read = [&](int t, int u, int i, int slot, floatx4 (&v)[P], bool whole) {      // element i: k = 4 i + b of the group
#pragma unroll
        for (int j = 0; j < P; ++j) {
            v[j][i] = mine[slot * STAGE + (u * P + j) * 256 + i * 64];
            if (!whole && (t * G + u) * 16 + 4 * i + b >= K) v[j][i] = 0.f;
        }
    };
    for (int t = 0; t < STAGES - 1 && t < stages; ++t)
#pragma unroll
        for (int c = 0; c < LOADS; ++c) load(t, c / P, c % P, t, false);
#pragma unroll
    for (int j = 0; j < P; ++j) row[j] += (uint32_t)b * 16u;                  // (from here on: whole loads, and those of the last stage)
    wait_for(min(STAGES - 1, stages) - 1);
#pragma unroll
    for (int i = 0; i < 4; ++i) read(0, 0, i, 0, now, false);
    int slot = 0;
    // more: a further stage is asked for, into the place of the last one read; whole: it lies before K; clean: what is read does
    auto turn = [&](int t, auto more, bool whole, bool clean) {
        const int ahead = slot + 1 == STAGES ? 0 : slot + 1, behind = slot == 0 ? STAGES - 1 : slot - 1;
#pragma unroll
        for (int u = 0; u < G; ++u) {
            if (u == G - 1) {                              // the next stage is read from here on
                if constexpr (decltype(more)::value) strip_wait<LOADS * (STAGES - 3) + (G - 1) * P>();
                else wait_for(stages - 2 - t);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
#pragma unroll
                for (int j = 0; j < NT; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(now[0][i], now[1 + j][i], acc[j], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);         // (left alone, the compiler moves a load to where its value is used)
                if (u + 1 < G) read(t, u + 1, i, slot, next, clean);
                else read(t + 1, 0, i, ahead, next, clean);
                if (decltype(more)::value && i < P) load(t + STAGES - 1, u, i, behind, whole);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int j = 0; j < P; ++j) now[j] = next[j];
        }
        slot = ahead;
    };
    int t = 0;
    for (; t + STAGES - 1 < full; ++t) turn(t, yes, true, true);
    if (stages == full) {
        for (; t < stages; ++t) turn(t, no, true, true);     // (behind the last stage nothing is made of what is read)
    } else {
#pragma unroll
        for (int j = 0; j < P; ++j) row[j] -= (uint32_t)b * 16u;
        if (t + STAGES - 1 < stages) turn(t, yes, false, true), ++t;
        for (; t < stages; ++t) turn(t, no, false, false);
    }
}

template <int NT, int STAGES>
__global__ __launch_bounds__(64) void gemm_f32_strip_kernel(const float* __restrict__ a, const float* __restrict__ w,
                                                            float* __restrict__ out, int M, int N, int K) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int r = threadIdx.x & 15, b = threadIdx.x >> 4, m0 = blockIdx.y * 16, n0 = blockIdx.x * (NT * 16);
    floatx4 acc[NT];
    f32_strip<NT, STAGES>(a + (size_t)m0 * K, w + (size_t)n0 * K, M - m0, N - n0, K, lds, acc);
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int m = m0 + b * 4 + e, n = n0 + j * 16 + r;
            if (m < M && n < N) out[(size_t)m * N + n] = acc[j][e];
        }
}

// out = silu(a . w[0:N]^T) * (a . w[N:2N]^T) for the same sizes: one wavefront the gate's strip, one the up's, which meet in LDS;
// the bits of the product and the activation's own launch (8 rows of 2 * 3072 x 1024 in a decoding step: 9.6 us for 10.2 and 4.8).
template <int STAGES>
__global__ __launch_bounds__(128) void gemm_f32_gated_strip_kernel(const float* __restrict__ a, const float* __restrict__ w,
                                                                   float* __restrict__ out, int M, int N, int K) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, b = lane >> 4, m0 = blockIdx.y * 16, n0 = blockIdx.x * 16;
    floatx4 acc[1];
    f32_strip<1, STAGES>(a + (size_t)m0 * K, w + (size_t)(wave * N + n0) * K, M - m0, N - n0, K, lds + wave * strip_lds_floats<1, STAGES>(), acc);
    float* meet = lds + strip_lds_floats<1, STAGES>();     // (the second wavefront's own, which it has read out)
    if (wave == 1) *reinterpret_cast<floatx4*>(meet + lane * 4) = acc[0];
    __syncthreads();
    if (wave == 1) return;
    const floatx4 up = *reinterpret_cast<const floatx4*>(meet + lane * 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int m = m0 + b * 4 + e, n = n0 + r;
        if (m < M && n < N) out[(size_t)m * N + n] = gate_act<0>(acc[0][e]) * up[e];
    }
}

// More rows: bound by the matrix cores.  Four wavefronts of T x T tiles of 16 x 16; blocks of G groups of 16 k go through LDS as
// the products want them (rows of a group 80 bytes apart: 16 lanes' 16-byte accesses meet every bank once), the next block's
// loads under way while one is multiplied -- so small tiles, whose products take no time, take long blocks.
template <int T, int G, bool VEC>
__global__ __launch_bounds__(256) void gemm_f32_tile_kernel(const float* __restrict__ a, const float* __restrict__ w,
                                                            float* __restrict__ out, int M, int N, int K) {
    constexpr int B = 2 * T * 16, STRIDE = 20, ROWS = 2 * B, UNITS = ROWS / 16, EACH = UNITS * G / 4;     // units: 16 rows x 16 k
    static_assert(UNITS * G % 4 == 0, "as many units for every wavefront");
    extern __shared__ __attribute__((aligned(16))) float lds[];               // [buffer][group][row][STRIDE]
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, q = (lane >> 4) * 4;
    const int wm = wave / 2, wn = wave % 2;
    // neighbouring tiles of a weight strip to the same XCD (workgroups are dealt out to the eight in turn)
    const int tiles_m = (M + B - 1) / B, tiles = tiles_m * ((N + B - 1) / B), each = (tiles + 7) / 8;
    const int tile = (blockIdx.x % 8) * each + blockIdx.x / 8;
    if (blockIdx.x / 8 >= each || tile >= tiles) return;
    const int m0 = (tile % tiles_m) * B, n0 = (tile / tiles_m) * B;
    const int turns = (K + 16 * G - 1) / (16 * G);

    floatx4 stage[EACH];
    auto load = [&](int k0) {
#pragma unroll
        for (int c = 0; c < EACH; ++c) {
            const int unit = wave + 4 * c, row = unit % UNITS * 16 + r;
            const float* p = row < B ? a + (size_t)min(m0 + row, M - 1) * K : w + (size_t)min(n0 + row - B, N - 1) * K;
            stage[c] = load_k4<VEC>(p, k0 + unit / UNITS * 16 + q, K);
        }
    };
    floatx4 acc[T][T];
#pragma unroll
    for (int i = 0; i < T; ++i)
#pragma unroll
        for (int j = 0; j < T; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    load(0);
    for (int turn = 0; turn < turns; ++turn) {
        float* block = lds + (turn & 1) * (G * ROWS * STRIDE);
#pragma unroll
        for (int c = 0; c < EACH; ++c) {
            const int unit = wave + 4 * c;
            *reinterpret_cast<floatx4*>(block + (unit / UNITS * ROWS + unit % UNITS * 16 + r) * STRIDE + q) = turned(stage[c]);
        }
        // (one barrier a turn: a buffer is written again behind the barrier that follows every wavefront's reads of it)
        __syncthreads();
        if (turn + 1 < turns) load((turn + 1) * 16 * G);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const float* rows = block + g * ROWS * STRIDE;
            floatx4 av[T], wv[T];
#pragma unroll
            for (int i = 0; i < T; ++i) av[i] = *reinterpret_cast<const floatx4*>(rows + ((wm * T + i) * 16 + r) * STRIDE + q);
#pragma unroll
            for (int j = 0; j < T; ++j) wv[j] = *reinterpret_cast<const floatx4*>(rows + (B + (wn * T + j) * 16 + r) * STRIDE + q);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < T; ++i)
#pragma unroll
                    for (int j = 0; j < T; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[i][e], wv[j][e], acc[i][j], 0, 0, 0);
        }
    }
#pragma unroll
    for (int i = 0; i < T; ++i)
#pragma unroll
        for (int j = 0; j < T; ++j) {
            const int n = n0 + (wn * T + j) * 16 + r;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int m = m0 + (wm * T + i) * 16 + q + e;
                if (m < M && n < N) out[(size_t)m * N + n] = acc[i][j][e];
            }
        }
}

template <int NT, int STAGES>
static int launch_f32_strip(const float* a, const float* w, float* out, int M, int N, int K, hipStream_t stream) {
    constexpr size_t lds = strip_lds_floats<NT, STAGES>() * sizeof(float);
    static const hipError_t allowed = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_f32_strip_kernel<NT, STAGES>),
                                                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (allowed != hipSuccess) return (int)allowed;
    gemm_f32_strip_kernel<NT, STAGES><<<dim3((N + NT * 16 - 1) / (NT * 16), (M + 15) / 16), 64, lds, stream>>>(a, w, out, M, N, K);
    return (int)hipGetLastError();
}

template <int STAGES>
static int launch_f32_gated_strip(const float* a, const float* w, float* out, int M, int N, int K, hipStream_t stream) {
    constexpr size_t lds = 2 * strip_lds_floats<1, STAGES>() * sizeof(float);
    static const hipError_t allowed = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_f32_gated_strip_kernel<STAGES>),
                                                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (allowed != hipSuccess) return (int)allowed;
    gemm_f32_gated_strip_kernel<STAGES><<<dim3((N + 15) / 16, (M + 15) / 16), 128, lds, stream>>>(a, w, out, M, N, K);
    return (int)hipGetLastError();
}

template <int T, int G, bool VEC>
static int launch_f32_tile(const float* a, const float* w, float* out, int M, int N, int K, hipStream_t stream) {
    constexpr int B = 2 * T * 16;
    const long long tiles = (long long)((M + B - 1) / B) * ((N + B - 1) / B);
    if (tiles > 0x7ffffff0LL) return -2;
    static const hipError_t allowed = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_f32_tile_kernel<T, G, VEC>),
                                                          hipFuncAttributeMaxDynamicSharedMemorySize, 2 * G * 2 * B * 20 * sizeof(float));
    if (allowed != hipSuccess) return (int)allowed;
    gemm_f32_tile_kernel<T, G, VEC><<<(unsigned)((tiles + 7) / 8 * 8), 256, 2 * G * 2 * B * 20 * sizeof(float), stream>>>(a, w, out, M, N, K);
    return (int)hipGetLastError();
}

template <bool VEC>
static int launch_gemm_f32(const float* a, const float* w, float* out, int M, int N, int K, hipStream_t stream) {
    // A wavefront a tile of 16 x 16 while those are few: 8 rows of 4096 x 1024, 1024 x 2048, 6144 x 1024 and 1024 x 3072 take 7.6,
    // 11.5, 10.2 and 15.6 us (tiles of 32 14.3, 23.7, 15.8 and 34.3), 64 rows of 1024 x 3072 16.1 (40); up to 512 tiles, two a
    // compute unit, with eight stages of LDS, up to 768 with five (three a unit; 40 rows of 6144 x 1024, 1152 tiles, do not come
    // here).  Two strips a wavefront beyond that, while the rows are few or up to 1024 tiles: 64 rows of 4096 x 1024 14.1 (tiles
    // of 32 16.7), 8 of 151936 x 1024 144 (the weight alone takes 130); 64 rows of 6144 x 1024 (1536 tiles) in tiles of 32 21.3.
    const long long units = (long long)((M + 15) / 16) * ((N + 15) / 16);
    if (VEC && (M + 15) / 16 <= 65535 && K < STRIP_K) {
        if (units <= 768) return units <= 512 ? launch_f32_strip<1, 8>(a, w, out, M, N, K, stream) : launch_f32_strip<1, 5>(a, w, out, M, N, K, stream);
        if (M <= 16 || units <= 1024) return launch_f32_strip<2, 4>(a, w, out, M, N, K, stream);
    }
    // The square tile whose workgroups, one a compute unit at a time, are done first: a tile of 64 takes 1 / 3.7 of the time
    // of one of 128, a tile of 32 0.35 of one of 64 (at 2048 rows of 4096 x 4096; tiles of 128 reach 120 TFLOP/s there).  1500
    // rows of 6144 x 1024 take 198 us in tiles of 64 and 230 in those of 128, 2048 rows 257 and 231, 400 rows of 1024 x 3072 57
    // in those of 32 and 96 in those of 64.
    auto cost = [&](int b, double one) {
        return one * (double)(((long long)((M + b - 1) / b) * ((N + b - 1) / b) + 255) / 256);
    };
    const double c32 = cost(32, 0.35), c64 = cost(64, 1.0), c128 = cost(128, 3.7);
    if (c32 <= c64 && c32 <= c128)
        // (blocks of 8 groups leave room for one workgroup a compute unit, of 4 for three: 128 rows of 4096 x 1024, 512 tiles, 24.3
        // and 26.0 us, of 6144 x 1024, 768 tiles, 36.7 and 30.0)
        return c32 <= 0.7 ? launch_f32_tile<1, 8, VEC>(a, w, out, M, N, K, stream) : launch_f32_tile<1, 4, VEC>(a, w, out, M, N, K, stream);
    return c64 <= c128 ? launch_f32_tile<2, 2, VEC>(a, w, out, M, N, K, stream)
                       : launch_f32_tile<4, 1, VEC>(a, w, out, M, N, K, stream);
}

extern "C" int mlr_gemm(const void* a, const void* w, void* out, int M, int N, int K, int out_float,
                        hipStream_t stream) {
    (void)out_float;                                   // the float engine's outputs are float
    if (M <= 0 || N <= 0) return 0;
    if (K <= 0) return -1;
    if ((M + 63) / 64 > 65535) return -2;
    const bool aligned = K % 4 == 0 && ((uintptr_t)a | (uintptr_t)w) % 16 == 0;
    return aligned ? launch_gemm_f32<true>((const float*)a, (const float*)w, (float*)out, M, N, K, stream)
                   : launch_gemm_f32<false>((const float*)a, (const float*)w, (float*)out, M, N, K, stream);
}

// out[M, N] = silu(a . w[0:N]^T) * (a . w[N:2N]^T) where a workgroup's two strips find room beside another's: up to 256 tiles of
// gates with eight stages, 512 with four; returns 1 for other sizes (the caller then runs the product and the activation).
extern "C" int mlr_gemm_gated_silu(const void* a, const void* w, void* out, int M, int N, int K, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (K <= 0) return -1;
    const long long units = (long long)((M + 15) / 16) * ((N + 15) / 16);
    if (K % 4 != 0 || K >= STRIP_K || ((uintptr_t)a | (uintptr_t)w) % 16 != 0 || units > 512) return 1;
    if (units <= 256) return launch_f32_gated_strip<8>((const float*)a, (const float*)w, (float*)out, M, N, K, stream);
    return launch_f32_gated_strip<4>((const float*)a, (const float*)w, (float*)out, M, N, K, stream);
}

#else
// ------------------------------------------------------------------------------ bfloat16
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;

#define BK 32
#define LDS_STRIDE (BK + 8)      // in elements: rows 80 bytes apart

// Eight consecutive k of one row as a 16-byte vector; zero beyond the matrix.
__device__ __forceinline__ bf16x8 load_k8(const __bf16* base, int row, int rows, int k, int K,
                                          bool vector_ok) {
    bf16x8 v = {0, 0, 0, 0, 0, 0, 0, 0};
    if (row < rows) {
        const __bf16* p = base + (size_t)row * K + k;
        if (vector_ok && k + 8 <= K) {
            v = *reinterpret_cast<const bf16x8*>(p);
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (k + e < K) v[e] = p[e];
        }
    }
    return v;
}

// Workgroup tile (WM * TM * 16) x (WN * TN * 16); WM x WN wavefronts, each TM x TN MFMA tiles.
template <int WM, int WN, int TM, int TN, bool OUT_FLOAT>
__global__ __launch_bounds__(WM * WN * 64) void gemm_bf16_kernel(
    const __bf16* __restrict__ a, const __bf16* __restrict__ w, void* __restrict__ out_raw,
    int M, int N, int K) {
    constexpr int BM = WM * TM * 16, BN = WN * TN * 16, THREADS = WM * WN * 64;
    __shared__ __bf16 as[BM * LDS_STRIDE];
    __shared__ __bf16 ws[BN * LDS_STRIDE];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int wm = wave / WN, wn = wave % WN;
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    const bool vector_ok = (K % 8) == 0;

    floatx4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

    for (int k0 = 0; k0 < K; k0 += BK) {
        for (int c = t; c < BM * 4; c += THREADS) {           // 4 chunks of 8 per row
            const int r = c >> 2, kc = (c & 3) * 8;
            *reinterpret_cast<bf16x8*>(&as[r * LDS_STRIDE + kc]) =
                load_k8(a, m0 + r, M, k0 + kc, K, vector_ok);
        }
        for (int c = t; c < BN * 4; c += THREADS) {
            const int r = c >> 2, kc = (c & 3) * 8;
            *reinterpret_cast<bf16x8*>(&ws[r * LDS_STRIDE + kc]) =
                load_k8(w, n0 + r, N, k0 + kc, K, vector_ok);
        }
        __syncthreads();
        bf16x8 af[TM], wf[TN];
        const int frag_row = lane & 15, frag_k = (lane >> 4) * 8;
#pragma unroll
        for (int i = 0; i < TM; ++i)
            af[i] = *reinterpret_cast<const bf16x8*>(
                &as[((wm * TM + i) * 16 + frag_row) * LDS_STRIDE + frag_k]);
#pragma unroll
        for (int j = 0; j < TN; ++j)
            wf[j] = *reinterpret_cast<const bf16x8*>(
                &ws[((wn * TN + j) * 16 + frag_row) * LDS_STRIDE + frag_k]);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i], wf[j], acc[i][j], 0, 0, 0);
        __syncthreads();
    }

    // accumulator element r of a lane: row (lane / 16) * 4 + r, column lane % 16
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int n = n0 + (wn * TN + j) * 16 + (lane & 15);
            if (n >= N) continue;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int m = m0 + (wm * TM + i) * 16 + (lane >> 4) * 4 + r;
                if (m >= M) continue;
                if (OUT_FLOAT) ((float*)out_raw)[(size_t)m * N + n] = acc[i][j][r];
                else ((__bf16*)out_raw)[(size_t)m * N + n] = (__bf16)acc[i][j][r];
            }
        }
    }
}

// Few rows (M <= 64): the weight is streamed once, straight from memory into the matrix cores.  A
// workgroup owns 16 output columns (16 rows of w); its eight wavefronts each take an eighth of k, and
// their partial sums are added in the order 0..7, so the result does not depend on M.  The weight
// is the A operand (rows n), the activation the B operand (columns m): a lane ends up with four
// consecutive n of one m.
// GATED: w holds two stacked matrices [gate; up] of N rows each; the workgroup computes the same 16
// columns of both and writes silu(gate) * up (the feed-forward's activation fused into the projection).
// STAGE (M <= 16, K a multiple of 64): a wavefront reads its part of the activation as M rows of
// consecutive bytes, puts them into a piece of LDS of its own and takes its operand from there.  Read
// straight into the operand layout, the activation costs as many requests to the cache as the weight
// does to memory, and the weight's rate drops by a tenth to a third (measured; more with more rows).
#define SKINNY_WAVES 8
#define SKINNY_STAGE_PITCH(U) ((U) * 128 + 16)        // bytes a row of the staged activation takes
#define SKINNY_STAGE_LDS (66 * 1024)                  // the most dynamic LDS a workgroup asks for

// What a skinny product of up to 16 rows may do with its sums before it stores them: the two halves of an
// RMSNorm that is handed from the projection before it to the projection after it.
//   EPI_SCALE (the projection after the norm): its input is x * norm_w, rounded, WITHOUT the row's scale
//     rsqrt(mean(x^2) + eps), because whoever produced x knew only partial sums of squares; the scale is a
//     factor per row, so it is applied here, in 32-bit, to the finished sums: out[m] *= rsqrt(sum_p ss[m][p] *
//     inv_size + eps).  The partial sums are added in a fixed order (see the kernel).
//   EPI_RESIDUAL (the projection before the norm, which ends a mixer or a feed-forward): its sums are added
//     to the residual stream, h[m][n] += out[m][n], in 32-bit and in place (every element belongs to one
//     lane); when a norm follows (next_w != null) it also writes x_out = bf16(h * next_w) and, per row and
//     workgroup (16 columns), the sum of squares of its 16 new values of h: ss_out[m][workgroup].
#define EPI_NONE 0
#define EPI_SCALE 1
#define EPI_RESIDUAL 2
struct SkinnyEpilogue {
    const float* ss;          // EPI_SCALE: [M][ss_parts] partial sums of squares of the rows
    int ss_parts;
    int ss_vec;               // ss_parts is a multiple of 4 and ss 16-byte aligned: four sums a load
    float eps, inv_size;
    float* h;                 // EPI_RESIDUAL: [M][N] the residual stream
    const float* next_w;      // [N] weights of the norm that follows, or null
    __bf16* x_out;            // [M][N]
    float* ss_out;            // [M][gridDim.x]
    int cols;                 // PAIR: the output columns of a workgroup, 17..32 (otherwise 16, whatever this says)
    int ss_stride;            // floats between the rows of ss_out (its capacity: a strip of 16 a part)
    float glu_limit;          // GATED: > 0: the clamped gate g = min(gate, limit), u = clamp(up, +-limit),
    float glu_slope;          //        y = g sigmoid(slope g) (u + 1); 0: y = silu(gate) up; -1: gelu_tanh(gate) up; -2: relu(gate) up
    int plain_act;            // a plain product's activation: 0 none, 1 relu(x)^2, 2 the exact gelu x Phi(x)
};
// PAIR: a workgroup owns `cols` (17..32) output columns, two strips side by side, the second one partly
// used: for a number of columns that deals strips of 16 unevenly to the compute units (384 strips on 256
// units take as long as 512), 24 columns a workgroup give every unit the same work.  The second strip
// rides where GATED keeps its second matrix.
template <int MT, bool OUT_FLOAT, bool GATED, int UMAX = 4, bool STAGE = false, int EPI = EPI_NONE, bool PAIR = false>   // UMAX: the most groups of k a turn takes
__global__ __launch_bounds__(SKINNY_WAVES * 64) void gemm_skinny_kernel(const __bf16* __restrict__ a,
                                                               const __bf16* __restrict__ w,
                                                               void* __restrict__ out_raw, int M, int N, int K,
                                                               SkinnyEpilogue epi) {
    constexpr int NW = (GATED || PAIR) ? 2 : 1;
    static_assert(!PAIR || (MT == 1 && !GATED && !STAGE), "two strips: a plain product of few rows");
    static_assert(!STAGE || MT == 1, "the activation is staged for at most 16 rows");
    static_assert(EPI == EPI_NONE || MT == 1, "the norm is handed over for at most 16 rows");
    static_assert(EPI != EPI_RESIDUAL || (!GATED && !OUT_FLOAT), "the residual sum follows a plain projection");
    __shared__ float part[SKINNY_WAVES - 1][NW][MT][64][4];
    __shared__ float ss_lds[SKINNY_WAVES][16];
    extern __shared__ __attribute__((aligned(16))) char staged[];   // [SKINNY_WAVES][M][pitch] when STAGE
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, b = lane >> 4;
    const int cols = PAIR ? epi.cols : 16;
    const int n0 = blockIdx.x * cols;
    const int last_row = PAIR ? min(N - 1, n0 + cols - 1) : N - 1;     // (PAIR: rows beyond the workgroup's columns read its last one)
    // this lane's weight row for g = 0 and for g = 1 (GATED: the same row of the second matrix; PAIR: 16 rows on)
    const int wrow_of[2] = {min(n0 + r16, N - 1), GATED ? N + min(n0 + r16, N - 1) : min(n0 + 16 + r16, last_row)};
    const bool vector_ok = (K % 8) == 0;
    const int steps = (K + 31) / 32;
    const int per_wave = (steps + SKINNY_WAVES - 1) / SKINNY_WAVES;
    const int s_begin = wave * per_wave, s_end = min(steps, s_begin + per_wave);
    // What the epilogue needs from memory is asked for here, before the weight, by every wavefront alike
    // (no branch around a load); only wavefront 0 uses it.
    float ss_mine = 0.f;                                   // EPI_SCALE: this lane's share of the row's partial sums
    float4 ss4 = make_float4(0.f, 0.f, 0.f, 0.f);          // ... which are added when the weight is multiplied, where this holds them all
    const int ss_quads = epi.ss_parts >> 2, ss_run = (ss_quads + 4 * SKINNY_WAVES - 1) / (4 * SKINNY_WAVES);
    const bool ss_later = EPI == EPI_SCALE && UMAX <= 2 && epi.ss_vec && ss_run <= 1;
    float4 h4 = make_float4(0.f, 0.f, 0.f, 0.f), nw4 = h4;  // EPI_RESIDUAL: h and the next norm's weights at (row r16, columns n0 + 4 b ..)
    float4 h4b = h4, nw4b = h4;                            // ... and, PAIR, at the second strip's columns n0 + 16 + 4 b ..
    if constexpr (EPI == EPI_SCALE) {
        // the row's partial sums are dealt out to the 32 (wavefront, lane block) pairs in runs of q; a run is
        // added in ascending order (four sums that lie side by side as (0 + 1) + (2 + 3) first, when their number
        // allows 16-byte loads), the four runs of a wavefront as (0 + 1) + (2 + 3), the wavefronts in the order
        // 0..7: an order that depends on nothing but the number of partial sums.  Up to 128 of them (a short k) a lane's one load is
        // asked for here and used behind the products: used here, it costs a trip to the cache before the workgroup has asked for any of
        // its weight (0.6B sizes, one token: 1046 us a step, so 1034; eight 1623, 1606).  Of more, four are asked for before the first is
        // used: kept as well, their registers are what another workgroup on a compute unit needs (10 x 2 * 25600 x 5120 104.7 us, 115.9
        // with them; 10 x 2 * 12288 x 1024 with four 13.2 and 15.8).
        const float* row = epi.ss + (size_t)min(r16, M - 1) * epi.ss_parts;
        const int pair = wave * 4 + b;
        if (ss_later) {
            ss4 = reinterpret_cast<const float4*>(row)[min(pair, ss_quads - 1)];
        } else if (epi.ss_vec) {
            const int quads = ss_quads, q = ss_run;
            const float4* row4 = reinterpret_cast<const float4*>(row);
            for (int j0 = 0; j0 < q; j0 += 4) {
                float4 v[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) v[j] = row4[min(pair * q + j0 + j, quads - 1)];
                asm volatile("" : "+v"(v[0].x), "+v"(v[1].x), "+v"(v[2].x), "+v"(v[3].x));   // (all four are loaded, none behind a branch)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const bool mine = j0 + j < q && pair * q + j0 + j < quads;
                    ss_mine += mine ? (v[j].x + v[j].y) + (v[j].z + v[j].w) : 0.f;
                }
            }
        } else {
            const int q = (epi.ss_parts + 4 * SKINNY_WAVES - 1) / (4 * SKINNY_WAVES);
            for (int j0 = 0; j0 < q; j0 += 4) {
                float v[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) v[j] = row[min(pair * q + j0 + j, epi.ss_parts - 1)];
                asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]));
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const bool mine = j0 + j < q && pair * q + j0 + j < epi.ss_parts;
                    ss_mine += mine ? v[j] : 0.f;
                }
            }
        }
    }
    if constexpr (EPI == EPI_RESIDUAL) {
        const int n = min(n0 + 4 * b, max(N - 4, 0));      // (clamped: a narrow last strip is handled element by element below)
        const size_t at = (size_t)min(r16, M - 1) * N + n;
        if ((N & 3) == 0) {
            h4 = *reinterpret_cast<const float4*>(epi.h + at);
            if (epi.next_w) nw4 = *reinterpret_cast<const float4*>(epi.next_w + n);
            if constexpr (PAIR) {                         // (PAIR is only launched for N and cols that are multiples of 4)
                const int n2 = min(n0 + 16 + 4 * b, N - 4);
                h4b = *reinterpret_cast<const float4*>(epi.h + (size_t)min(r16, M - 1) * N + n2);
                if (epi.next_w) nw4b = *reinterpret_cast<const float4*>(epi.next_w + n2);
            }
        }
    }
    floatx4 acc[NW][MT];
#pragma unroll
    for (int g = 0; g < NW; ++g)
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[g][i] = floatx4{0.f, 0.f, 0.f, 0.f};
    if ((K & 63) == 0) {
        // The usual case, K a multiple of 64: no branch anywhere near a load (a load behind a branch makes
        // the compiler wait for every load in flight).  Rows beyond N or M read the last valid row; what
        // they produce is never stored.  Two k steps are taken together: a lane reads 32 consecutive bytes
        // of its weight row (four lanes a whole 128-byte line), each 16 of them feed one product; the
        // activation is read the same way, so the k slots of both operands agree.  (Measured: 64 bytes a
        // lane is slower again.)
        constexpr int W = 2;                              // 16-byte chunks per lane and group
        const int groups = steps / W;
        const int per_wave_g = (groups + SKINNY_WAVES - 1) / SKINNY_WAVES;
        const int g_begin = wave * per_wave_g, g_end = min(groups, g_begin + per_wave_g);
        const __bf16* wrow[NW];
#pragma unroll
        for (int g = 0; g < NW; ++g) wrow[g] = w + (size_t)wrow_of[g] * K + b * (8 * W);
        const __bf16* xrow[MT];
#pragma unroll
        for (int i = 0; i < MT; ++i) xrow[i] = a + (size_t)min(16 * i + r16, M - 1) * K + b * (8 * W);
        // Full turns of U groups first: every load of a turn (the activation, which comes from the cache,
        // before the weight that follows it in the queue) is asked for before the first product, with no
        // branch in between.  What is left (fewer than U groups) makes one shorter turn.
        constexpr int U = (MT * NW <= 2 && UMAX >= 4) ? 4 : 2;
        constexpr int PITCH = SKINNY_STAGE_PITCH(U);
        char* mine = staged + (size_t)wave * M * PITCH;
        auto turn = [&](int g0, auto count) {
            constexpr int C = decltype(count)::value;
            constexpr int PPR = C * 8;                        // 16-byte pieces in a row of this turn's chunk
            bf16x8 xf[MT][C][W], wf[NW][C][W], xg[STAGE ? C * W : 1];
            if constexpr (STAGE) {
                // piece p of the chunk: row p / PPR, bytes 16 * (p % PPR); a lane takes pieces lane, lane + 64, ...
#pragma unroll
                for (int i = 0; i < C * W; ++i) {
                    const int p = min(i * 64 + lane, M * PPR - 1);
                    xg[i] = *reinterpret_cast<const bf16x8*>(a + (size_t)(p / PPR) * K + (g0 * (32 * W) + (p % PPR) * 8));
                }
            } else {
#pragma unroll
                for (int u = 0; u < C; ++u)
#pragma unroll
                    for (int i = 0; i < MT; ++i)
#pragma unroll
                        for (int c = 0; c < W; ++c)
                            xf[i][u][c] = *reinterpret_cast<const bf16x8*>(xrow[i] + (g0 + u) * (32 * W) + 8 * c);
            }
#pragma unroll
            for (int u = 0; u < C; ++u)
#pragma unroll
                for (int g = 0; g < NW; ++g)
#pragma unroll
                    for (int c = 0; c < W; ++c)
                        wf[g][u][c] = *reinterpret_cast<const bf16x8*>(wrow[g] + (g0 + u) * (32 * W) + 8 * c);
            __builtin_amdgcn_sched_barrier(0);            // or the compiler spreads the loads among the products
            if constexpr (STAGE) {
                // LDS serves a wavefront's accesses in their order: the reads below see these writes, and
                // the next turn's writes come after these reads.  Rows from M on read row M - 1.
#pragma unroll
                for (int i = 0; i < C * W; ++i) {
                    const int p = i * 64 + lane;
                    if (p < M * PPR) *reinterpret_cast<bf16x8*>(mine + (p / PPR) * PITCH + (p % PPR) * 16) = xg[i];
                }
                const char* row = mine + min(r16, M - 1) * PITCH + b * (16 * W);
#pragma unroll
                for (int u = 0; u < C; ++u)
#pragma unroll
                    for (int c = 0; c < W; ++c)
                        xf[0][u][c] = *reinterpret_cast<const bf16x8*>(row + u * (64 * W) + 16 * c);
            }
#pragma unroll
            for (int u = 0; u < C; ++u)
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int c = 0; c < W; ++c)
#pragma unroll
                        for (int g = 0; g < NW; ++g)
                            acc[g][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[g][u][c], xf[i][u][c], acc[g][i], 0, 0, 0);
        };
        int g0 = g_begin;
        for (; g0 + U <= g_end; g0 += U) turn(g0, std::integral_constant<int, U>{});
        const int rest = g_end - g0;                      // the same in every lane of a wavefront
        if (U > 2 && rest == 3) turn(g0, std::integral_constant<int, 3>{});
        else if (U > 2 && rest == 2) turn(g0, std::integral_constant<int, 2>{});
        else if (rest == 1) turn(g0, std::integral_constant<int, 1>{});
    } else {
#pragma unroll 4
        for (int s = s_begin; s < s_end; ++s) {
            const int k = s * 32 + b * 8;
            bf16x8 wf[NW];
#pragma unroll
            for (int g = 0; g < NW; ++g) wf[g] = load_k8(w, wrow_of[g], GATED ? 2 * N : N, k, K, vector_ok);
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                const bf16x8 xf = load_k8(a, 16 * i + r16, M, k, K, vector_ok);
#pragma unroll
                for (int g = 0; g < NW; ++g)
                    acc[g][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[g], xf, acc[g][i], 0, 0, 0);
            }
        }
    }
    if (wave > 0) {
#pragma unroll
        for (int g = 0; g < NW; ++g)
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) part[wave - 1][g][i][lane][r] = acc[g][i][r];
    }
    if constexpr (EPI == EPI_SCALE) {
        if (ss_later && wave * 4 + b < ss_quads) ss_mine += (ss4.x + ss4.y) + (ss4.z + ss4.w);
        ss_mine = xor_sum<16>(ss_mine);
        ss_mine = xor_sum<32>(ss_mine);
        if (b == 0) ss_lds[wave][r16] = ss_mine;
    }
    __syncthreads();
    if (wave != 0) return;
    float row_scale = 1.f;
    if constexpr (EPI == EPI_SCALE) {
        float total = 0.f;
#pragma unroll
        for (int i = 0; i < SKINNY_WAVES; ++i) total += ss_lds[i][r16];
        row_scale = 1.0f / sqrtf(total * epi.inv_size + epi.eps);
    }
    float y4[MT][4];
    float y4b[4] = {0.f, 0.f, 0.f, 0.f};                   // PAIR: the second strip's sums of this lane
#pragma unroll
    for (int i = 0; i < MT; ++i) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            float v[NW];
#pragma unroll
            for (int g = 0; g < NW; ++g) {
                v[g] = acc[g][i][r];
                for (int p = 0; p < SKINNY_WAVES - 1; ++p) v[g] += part[p][g][i][lane][r];
                if constexpr (EPI == EPI_SCALE) v[g] *= row_scale;
            }
            float y = v[0];
            if (GATED) {
                if (epi.glu_limit > 0.f) y = clamped_glu(v[0], v[NW - 1], epi.glu_limit, epi.glu_slope);
                else y = (epi.glu_limit < -1.5f ? gate_act<2>(v[0]) : epi.glu_limit < 0.f ? gate_act<1>(v[0]) : gate_act<0>(v[0])) * v[NW - 1];
            }
            if constexpr (!GATED && !OUT_FLOAT && EPI == EPI_NONE) {
                if (epi.plain_act) {
                    y = epi.plain_act == 1 ? plain_act<0>(y) : plain_act<1>(y);
                    if constexpr (PAIR) v[1] = epi.plain_act == 1 ? plain_act<0>(v[1]) : plain_act<1>(v[1]);
                }
            }
            y4[i][r] = y;
            if constexpr (PAIR) y4b[r] = v[1];
            if constexpr (PAIR && EPI != EPI_RESIDUAL) {  // the second strip's sum of this lane: column n0 + 16 + 4 b + r
                const int n = n0 + 16 + 4 * b + r;
                if (r16 < M && n <= last_row) {
                    if (OUT_FLOAT) ((float*)out_raw)[(size_t)r16 * N + n] = v[1];
                    else ((__bf16*)out_raw)[(size_t)r16 * N + n] = (__bf16)v[1];
                }
            }
        }
    }
    if constexpr (EPI == EPI_RESIDUAL) {
        // this lane: row r16, columns n0 + 4 b .. + 3 of h
        const int n = n0 + 4 * b;
        const bool row_ok = r16 < M;
        float x[4];
        float sq = 0.f;
        if ((N & 3) == 0) {
            const bool ok = row_ok && n < N;
            const float hv[4] = {h4.x, h4.y, h4.z, h4.w}, wv[4] = {nw4.x, nw4.y, nw4.z, nw4.w};
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                x[r] = ok ? hv[r] + y4[0][r] : 0.f;
                sq += x[r] * x[r];
            }
            if (ok) {
                *reinterpret_cast<float4*>(epi.h + (size_t)r16 * N + n) = make_float4(x[0], x[1], x[2], x[3]);
                if (epi.next_w) {
                    typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
                    *reinterpret_cast<bf16x4*>(epi.x_out + (size_t)r16 * N + n) =
                        bf16x4{(__bf16)(x[0] * wv[0]), (__bf16)(x[1] * wv[1]), (__bf16)(x[2] * wv[2]), (__bf16)(x[3] * wv[3])};
                }
            }
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const bool ok = row_ok && n + r < N;
                const size_t at = (size_t)min(r16, M - 1) * N + min(n + r, N - 1);
                x[r] = ok ? epi.h[at] + y4[0][r] : 0.f;
                sq += x[r] * x[r];
                if (ok) {
                    epi.h[at] = x[r];
                    if (epi.next_w) epi.x_out[at] = (__bf16)(x[r] * epi.next_w[n + r]);
                }
            }
        }
        if constexpr (PAIR) {
            // the second strip, whole groups of four columns: first its squares on their own, (0 + 1) + (2 + 3)
            // like the first strip's, then added to them
            const int n2 = n0 + 16 + 4 * b;
            const bool ok = row_ok && n2 + 3 <= last_row;
            const float hv[4] = {h4b.x, h4b.y, h4b.z, h4b.w}, wv[4] = {nw4b.x, nw4b.y, nw4b.z, nw4b.w};
            float x2[4], sq2 = 0.f;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                x2[r] = ok ? hv[r] + y4b[r] : 0.f;
                sq2 += x2[r] * x2[r];
            }
            if (ok) {
                *reinterpret_cast<float4*>(epi.h + (size_t)r16 * N + n2) = make_float4(x2[0], x2[1], x2[2], x2[3]);
                if (epi.next_w) {
                    typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
                    *reinterpret_cast<bf16x4*>(epi.x_out + (size_t)r16 * N + n2) =
                        bf16x4{(__bf16)(x2[0] * wv[0]), (__bf16)(x2[1] * wv[1]), (__bf16)(x2[2] * wv[2]), (__bf16)(x2[3] * wv[3])};
                }
            }
            if (epi.next_w) {
                sq = xor_sum<16>(sq);
                sq = xor_sum<32>(sq);
                sq2 = xor_sum<16>(sq2);
                sq2 = xor_sum<32>(sq2);
                if (b == 0 && row_ok) {
                    // a workgroup a part; the parts beyond the workgroups, up to the buffer's capacity, are zero
                    float* parts = epi.ss_out + (size_t)r16 * epi.ss_stride;
                    parts[blockIdx.x] = sq + sq2;
                    if ((int)(gridDim.x + blockIdx.x) < epi.ss_stride) parts[gridDim.x + blockIdx.x] = 0.f;
                }
            }
            return;
        }
        if (epi.next_w) {
            sq = xor_sum<16>(sq);            // (0 + 1) + (2 + 3) over the lane blocks: the strip's 16 columns
            sq = xor_sum<32>(sq);
            if (b == 0 && row_ok) epi.ss_out[(size_t)r16 * gridDim.x + blockIdx.x] = sq;
        }
        return;
    }
    // (whole groups of four columns on 8 or 16 bytes: one store a lane)
    const bool whole = (N & 3) == 0 && (reinterpret_cast<size_t>(out_raw) & (OUT_FLOAT ? 15 : 7)) == 0;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int m = 16 * i + r16;
        if (whole) {
            const size_t at = (size_t)m * N + n0 + 4 * b;
            typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4_t;
            if (m >= M || n0 + 4 * b >= N) continue;
            if (OUT_FLOAT) *reinterpret_cast<float4*>((float*)out_raw + at) = make_float4(y4[i][0], y4[i][1], y4[i][2], y4[i][3]);
            else *reinterpret_cast<bf16x4_t*>((__bf16*)out_raw + at) = bf16x4_t{(__bf16)y4[i][0], (__bf16)y4[i][1], (__bf16)y4[i][2], (__bf16)y4[i][3]};
            continue;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int n = n0 + 4 * b + r;
            if (m < M && n < N) {
                if (OUT_FLOAT) ((float*)out_raw)[(size_t)m * N + n] = y4[i][r];
                else ((__bf16*)out_raw)[(size_t)m * N + n] = (__bf16)y4[i][r];
            }
        }
    }
}

// Columns of a workgroup when two strips side by side deal the work out more evenly than strips of 16 do, else 0.
// Only where the weight is long enough for the memory's rate to count (k from 2048).
static int skinny_pair_columns(int N, int K) {
    const int units = compute_units();
    if (units < 0 || K < 2048 || N % 4 != 0) return 0;
    const int strips = (N + 15) / 16;
    const int turns = (strips + units - 1) / units;       // strips of 16: the busiest unit's share, in strips
    for (int j = 1; j <= 4; ++j) {
        const int cols = (((N + units * j - 1) / (units * j)) + 3) / 4 * 4;
        if (cols > 32) continue;
        if (cols <= 16) break;
        return (double)(j * cols) < 0.9 * 16.0 * turns ? cols : 0;
    }
    return 0;
}

template <int MT, bool OUT_FLOAT, bool GATED, int UMAX, bool STAGE, int EPI>
static int launch_skinny_kernel(const void* a, const void* w, void* out, int M, int N, int K, size_t lds,
                                const SkinnyEpilogue& epi, hipStream_t stream) {
    if constexpr (MT == 1 && !GATED && !STAGE && UMAX == 4) {
        const int cols = skinny_pair_columns(N, K);
        if (cols > 0) {
            SkinnyEpilogue e = epi;
            e.cols = cols;
            e.ss_stride = (N + 15) / 16;
            // (the parts beyond the workgroups are zeroed by the workgroups themselves: there are at most as many)
            gemm_skinny_kernel<MT, OUT_FLOAT, false, 4, false, EPI, true>
                <<<dim3((N + cols - 1) / cols), SKINNY_WAVES * 64, 0, stream>>>((const __bf16*)a, (const __bf16*)w, out, M, N, K, e);
            return (int)hipGetLastError();
        }
    }
    auto* kernel = gemm_skinny_kernel<MT, OUT_FLOAT, GATED, UMAX, STAGE, EPI>;
    if (STAGE) {                                          // static and dynamic LDS together may pass 64 KB
        static const hipError_t allowed = hipFuncSetAttribute(
            reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, SKINNY_STAGE_LDS);
        if (allowed != hipSuccess) return (int)allowed;
    }
    kernel<<<dim3((N + 15) / 16), SKINNY_WAVES * 64, lds, stream>>>((const __bf16*)a, (const __bf16*)w, out, M, N, K, epi);
    return (int)hipGetLastError();
}

template <int MT, bool GATED, int UMAX, bool STAGE, int EPI>
static int launch_skinny_as(const void* a, const void* w, void* out, int M, int N, int K, int out_float,
                            size_t lds, const SkinnyEpilogue& epi, hipStream_t stream) {
    if constexpr (EPI == EPI_NONE) {
        if (out_float) return launch_skinny_kernel<MT, true, GATED, UMAX, STAGE, EPI>(a, w, out, M, N, K, lds, epi, stream);
    }
    return launch_skinny_kernel<MT, false, GATED, UMAX, STAGE, EPI>(a, w, out, M, N, K, lds, epi, stream);
}

template <int MT, bool GATED, int EPI = EPI_NONE>
static int launch_skinny(const void* a, const void* w, void* out, int M, int N, int K, int out_float,
                         hipStream_t stream, const SkinnyEpilogue& epi = SkinnyEpilogue{}) {
    // A short k (at most two groups of 64 a wavefront) takes the variant whose turns hold two groups: it
    // needs fewer registers, so more of its short-lived workgroups fit a compute unit.
    const bool short_k = MT * (GATED ? 2 : 1) <= 2 && K <= 64 * 2 * SKINNY_WAVES;
    if constexpr (MT == 1 && !GATED) {
        // Two rows or more and a long k: the activation goes through LDS.  (Measured: with a short k the
        // extra step costs what it saves, and the gated variant, whose turns would have to shrink to stay
        // within the registers of two workgroups a compute unit, gains nothing.  At k = 2048 it pays where the
        // strips leave half of the compute units idle -- a workgroup's requests go through its unit's cache
        // one after the other, and there the activation's are half of them: 4.9 us for 5.4 on 1024 columns and
        // 8 rows, 5.2 for 6.1 with 16 -- and costs 3-6 % with a strip for every unit.)
        const size_t lds = (size_t)SKINNY_WAVES * M * SKINNY_STAGE_PITCH(4);
        const bool pair = skinny_pair_columns(N, K) > 0;     // (two strips: without the stage)
        const int units = compute_units();
        const bool long_k = K > 2048 || (K == 2048 && units > 0 && 2 * ((N + 15) / 16) <= units);
        if (!pair && M >= 2 && K % 64 == 0 && long_k && lds <= SKINNY_STAGE_LDS)
            return launch_skinny_as<MT, GATED, 4, true, EPI>(a, w, out, M, N, K, out_float, lds, epi, stream);
    }
    if (short_k) return launch_skinny_as<MT, GATED, 2, false, EPI>(a, w, out, M, N, K, out_float, 0, epi, stream);
    return launch_skinny_as<MT, GATED, 4, false, EPI>(a, w, out, M, N, K, out_float, 0, epi, stream);
}

// Many rows (prompt portions, mixed steps), K a multiple of 64: 16x16 tiles of v_mfma_f32_16x16x32_bf16, the operands brought
// to LDS in blocks of 64 k by loads that do not pass through registers (`buffer_load_dwordx4 .. lds`).  A workgroup has
// WM x WN wavefronts of TM x TN tiles each: BM = 16 WM TM rows and BN = 16 WN TN columns of the output, and STAGES blocks of LDS:
// while one block is multiplied the others are on their way.  The weight is the A operand of the instruction (its rows are
// output columns), the activation the B operand, so a lane ends up with four consecutive columns n of one row m
// (lane = 16 g + i: A holds row i, k slots 8 g .. 8 g + 7, B column i, the same k slots, C column i, rows 4 g + r in register r).
//
// What bounds it: at 2048 x 1024 x 2048 and the like a compute unit has one tile, and what counts is how many bytes of operands
// it has under way (a block staged through registers, as this kernel's predecessor did it, gave two); on large products it is
// the matrix cores at the clock that the card's power leaves them (counters on 2048 x 24576 x 4096: 69 % of the cycles' matrix
// work at 1.73 GHz, bank conflicts 3 % of the LDS cycles).  Measured inside a graph, weights cold, against the predecessor (32x32
// tiles, two blocks through registers) and the vendor library: 2048 x 1024 x 2048 12.2 us (library 16.3), 2048 x 1024 x 3072
// 17.0 (21.1), 2048 x 4096 x 1024 19.6 (21.3), with gate and activation 2048 x 2 * 3072 x 1024 25.8 (predecessor 37.6),
// 732 x 2048 x 2048 10.5 (13.1), 1533 x 4096 x 4096 47.9 (51.5), 2048 x 24576 x 4096 309-331 (278-352).
//
// A row of a block is 128 bytes, eight pieces of 16; a load writes 64 lanes' pieces side by side (eight rows), so rows cannot be
// padded apart.  Instead piece p of row r lies at place p ^ (r & 7) -- the lane that fetches it is chosen accordingly --, and
// the eight lanes that the LDS serves together read eight different banks.  (FEW: a row's even pieces first, then its odd ones.)
// Every output element is one sum over k in ascending order, 32 k an instruction, whatever M and the shape are (the forms for 17 to
// 64 rows: eight sums, see FEW).
// GATED: w = [gate; up] of N rows each; a wavefront's weight tiles alternate between the two.
#define WIDE_BK 64

template <int WM, int WN, int TM, int TN, int NS>
struct WideShape {
    static constexpr int BM = 16 * WM * TM, BN = 16 * WN * TN, WAVES = WM * WN;
    static constexpr int ROWS = BM + BN;                          // staged rows per block: weight, then activation
    static constexpr int LOADS = ROWS / 8 / WAVES;                // loads of a wavefront per block, eight rows each
    static constexpr int STAGE = ROWS * WIDE_BK;                  // elements of a block
    static constexpr size_t lds_bytes = (size_t)NS * STAGE * sizeof(__bf16);
    static_assert(ROWS % (8 * WAVES) == 0, "a block's rows must divide among the wavefronts");
    static_assert(lds_bytes <= 160 * 1024, "the blocks must fit the LDS");
    static_assert(LOADS * (NS - 1) <= 63, "the counter of loads in flight has six bits");
};

// What the epilogue does with the finished sums.  The activations after WIDE_SILU are those of the separate kernels, taken of the
// products as those read them, rounded to bfloat16: the same bits as the two launches one after the other.
enum { WIDE_PLAIN = 0, WIDE_SILU = 1, WIDE_SILU_ROUNDED = 2, WIDE_GELU_TANH = 3, WIDE_RELU = 4, WIDE_CLAMPED = 5,
       WIDE_RELU_SQUARED = 6, WIDE_GELU_ERF = 7,
       WIDE_CLAMPED_SUMS = 8 };            // (FEW) the clamped gate of the finished sums, as `gemm_skinny_kernel` takes it

struct WideArgs {
    const __bf16* a;
    const __bf16* w;
    void* out;
    int M, N, K, tiles_m, tiles_n;
    int act;              // WIDE_*
    float limit, slope;   // of WIDE_CLAMPED
    int vector_out;       // rows of the output start on 16 bytes
    int lda, ldo, a_head, out_head;       // of the form with a product a head: row pitches of activation and output, and from head to head
    float* partial;                       // SPLIT: the parts' sums, 8 - 8 / SPLIT + 1 tiles of floats a tile of the output
    int32_t* arrivals;                    // SPLIT: [tiles] workgroups that have left theirs; zero before and after a launch
};

#define QKV_HEAD 128              // channels of a head

// The LDS of that form: the finished tile in the blocks' place, head by head, then every row's position, page and place in it, and
// which eights of rows lie side by side in a page.
template <class S>
struct QkvTile {
    static constexpr int PITCH = QKV_HEAD + 8, VPITCH = S::BM + 8;                 // of a row of a head; of a channel of a head of values
    static constexpr int HEADS = S::BN / QKV_HEAD, PASSES = S::BM * HEADS * 8 / (64 * S::WAVES);
    static constexpr int HEAD = S::BM * PITCH;                                      // elements of a head
    static constexpr size_t tile_bytes = (size_t)HEADS * HEAD * sizeof(__bf16);
    static constexpr size_t rows_at = tile_bytes > S::lds_bytes ? tile_bytes : S::lds_bytes;
    static constexpr size_t lds_bytes = rows_at + (S::BM * 3 + S::BM / 8) * sizeof(int32_t);
};

// What the form with the heads' epilogue needs besides (QKV): w = [q heads; k heads; v heads] of 128 rows each.
struct QkvArgs : WideArgs {
    __bf16* q_out;                // [M, q_heads, 128]
    __bf16* k_pages;              // [pages][kv_heads][page_size][128]
    __bf16* v_pages;              // [pages][kv_heads][128][page_size]
    const int32_t* block_table; const int32_t* slots; const int32_t* positions;
    const float* q_norm_w; const float* k_norm_w; const float* rope;      // rope [positions][128]: cosines, sines; the others null: no norm
    float eps;
    int max_blocks, q_heads, kv_heads, page_size, write_cache;
};

// HEADS: head h multiplies its columns of wider rows by a weight of its own, out[m][h] = a[m][h] . w[h]^T; the tiles are counted
// head by head.
// QKV: the product of attention's q, k and v with what `qk_norm_rope_kv_vec_kernel` (rope_kv.hip) makes of it, the same bits: a tile
// holds whole heads, so once it lies in LDS, rounded to bfloat16, eight lanes take a row of a head, norm and turn it and write the
// queries to their matrix and the keys to their page; heads of values go to LDS transposed, so that eight rows of a channel are one
// read and one store into their page.
// The q/k/v matrix itself is never written: 2048 x 4096 x 1024 22.2 us for the 28.0 of the two launches, 19.1 of them the product.
// FEW (up to 64 rows): the sums of `gemm_skinny_kernel`, bit by bit, so that a row's results do not turn on whether 16 rows or 64
// are computed with it: eight parts of k, of whole blocks, each one sum and added in ascending order, and 16 consecutive bytes of
// every 32 of a row an instruction.  (The parts are also the more exact sum: worked out with normal operands, a
// rounding an instruction, its rms error is 0.63, 0.54 and 0.45 of one chain's at k = 1024, 2048 and 4096.)
// Beside one chain and a gate of hardware approximations it takes 6 % more of a product's time (108 products, geometric mean; 0.2 us
// for closing the parts, 0.4 for a gate), and 0.69 of the time of the kernels that took these rows before.
// PAIRED: a turn is two blocks, and its operands are in registers before it begins: a small tile has few products a block, and
// what its turns cost is the wait for the LDS and for the other wavefronts.
// SPLIT (FEW): SPLIT workgroups a tile, each with 8 / SPLIT of the parts; the one that arrives last adds all parts up in their order,
// the same bits (3 us of a launch: its reads of them).  What a product of few rows is bound by is what its compute units read out of the L2 (12 TB/s of all of them): strips
// narrow enough for every unit to have one each read the rows again, so wide tiles that share them, and the units that those leave
// idle given parts of k.
template <int WM, int WN, int TM, int TN, int NS, bool OUT_FLOAT, bool GATED, bool HEADS = false, bool FEW = false, bool PAIRED = false, bool QKV = false, int SPLIT = 1>
__global__ __launch_bounds__(64 * WM * WN, 2) void gemm_wide_kernel(const std::conditional_t<QKV, QkvArgs, WideArgs> args) {
    using S = WideShape<WM, WN, TM, TN, NS>;
    using Q = QkvTile<S>;
    static_assert(!QKV || (!OUT_FLOAT && !GATED && !HEADS && !FEW && S::BN % QKV_HEAD == 0), "whole heads");
    constexpr int BM = S::BM, BN = S::BN, LOADS = S::LOADS;
    static_assert(!GATED || TN % 2 == 0, "gate and up tiles come in pairs");
    static_assert((!PAIRED || FEW) && (!FEW || !HEADS) && (SPLIT == 1 || (FEW && SKINNY_WAVES % SPLIT == 0)), "forms for up to 64 rows");
    extern __shared__ __attribute__((aligned(16))) __bf16 wide_lds[];
    const int M = args.M, N = args.N, K = args.K;
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int li = lane & 15, g = lane >> 4;
    const int wm = wave / WN, wn = wave % WN;
    // Workgroups go to the 8 XCDs in turn; each XCD gets a contiguous range of tiles, and in it eight tiles of rows beside
    // each other for every tile of columns, so that an L2 holds what its tiles share.
    constexpr int GROUP = 8;
    int tm, tn, head = 0, share = 0;                              // share: of the parts of k (SPLIT)
    {
        const int one = args.tiles_m * args.tiles_n, total = HEADS || SPLIT > 1 ? (int)gridDim.x : one, xcd = blockIdx.x % 8;
        int tile = xcd * (total / 8) + min(xcd, total % 8) + blockIdx.x / 8;
        if (SPLIT > 1) {                                          // (a tile's workgroups side by side, on one XCD but for the last of them)
            share = tile % SPLIT;
            tile /= SPLIT;
        }
        if (HEADS) {
            head = tile / one;
            tile -= head * one;
        }
        const int per = GROUP * args.tiles_n, first = tile / per * GROUP, rows = min(GROUP, args.tiles_m - first);
        tm = first + tile % per % rows;
        tn = tile % per / rows;
    }
    constexpr int NOUT = GATED ? BN / 2 : BN;                     // output columns of the workgroup
    const int m0 = tm * BM, n0 = tn * NOUT;

    // Load i of a wavefront brings rows 8 (wave LOADS + i) .. of the block (weight rows first, then rows of the activation; rows
    // beyond a matrix are its last one again).  Places are 32-bit byte offsets from the matrices' bases (the host refuses
    // matrices of 2^31 elements and more).
    uint32_t src[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const int row = (wave * LOADS + i) * 8 + (lane >> 3), at = (lane & 7) ^ (row & 7), piece = (FEW ? (at & 3) * 2 + (at >> 2) : at) * 8;
        int r;
        if (row < BN) {
            if (GATED) {
                // staged weight row -> (wavefront column, tile j, row in tile); tile pairs (2 p, 2 p + 1) are gate and up
                // of output columns n0 + wn_ * (TN / 2) * 16 + p * 16 ..
                const int wn_ = row / (16 * TN), j = (row / 16) % TN;
                r = min(n0 + (wn_ * (TN / 2) + j / 2) * 16 + row % 16, N - 1) + (j & 1) * N;
            } else {
                r = min(n0 + row, N - 1);
            }
        } else {
            r = min(m0 + row - BN, M - 1);
        }
        src[i] = ((uint32_t)r * (uint32_t)(HEADS && row >= BN ? args.lda : K) + piece) * 2u;
    }
    const auto w_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)(args.w + (HEADS ? (size_t)head * N * K : 0)), 0,
                                                          (int)((uint32_t)N * (GATED ? 2u : 1u) * (uint32_t)K * 2u), 0x00027000);
    const auto a_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)(args.a + (HEADS ? (size_t)head * args.a_head : 0)), 0,
                                                          (int)((HEADS ? (uint32_t)(M - 1) * (uint32_t)args.lda + (uint32_t)K : (uint32_t)M * (uint32_t)K) * 2u), 0x00027000);
    constexpr int PER = SKINNY_WAVES / SPLIT;                     // parts of k that a workgroup has
    const int all_blocks = K / WIDE_BK, part_blocks = (all_blocks + SKINNY_WAVES - 1) / SKINNY_WAVES;
    const int first_block = SPLIT > 1 ? share * PER * part_blocks : 0;
    auto load = [&](int i, int kb, int stage) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds((wave * LOADS + i) * 8 < BN ? w_rsrc : a_rsrc,
                                                 (__attribute__((address_space(3))) void*)(wide_lds + stage * S::STAGE + (wave * LOADS + i) * 512),
                                                 16, (int)src[i], (first_block + kb) * (WIDE_BK * 2), 0, 0);
    };

    floatx4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    const int blocks = SPLIT > 1 ? min(all_blocks - first_block, PER * part_blocks) : all_blocks;
    floatx4 sum[FEW ? TM : 1][FEW ? TN : 1];                      // FEW: the parts of k that are done
    floatx4 part[SPLIT > 1 ? PER : 1][FEW ? TM : 1][FEW ? TN : 1];           // SPLIT: each by itself, but the first share's (in `sum`)
    int part_left = part_blocks, closed = 0;
    if constexpr (FEW) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                sum[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int q = 0; q < (SPLIT > 1 ? PER : 1); ++q) part[q][i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
            }
    }
    auto close_part = [&]() {
        if (SPLIT > 1 && share > 0) {
#pragma unroll
            for (int q = 0; q < (SPLIT > 1 ? PER : 1); ++q)
                if (closed == q) {                                // (the same in every lane)
#pragma unroll
                    for (int i = 0; i < TM; ++i)
#pragma unroll
                        for (int j = 0; j < TN; ++j) {
                            part[q][i][j] = acc[i][j];
                            acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
                        }
                }
            ++closed;
        } else if constexpr (FEW) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    sum[i][j] += acc[i][j];
                    acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
                }
        }
    };
    auto block_done = [&]() {
        if (FEW && --part_left == 0) {                            // (eight times a product, the same in every lane)
            asm volatile("");                                     // (a branch: as selects, every block's products would be waited for)
            close_part();
            part_left = part_blocks;
        }
    };
    // The operands of one half of a block (32 k); the other half's are read while these are multiplied.
    bf16x8 wf[2][TN], af[2][TM];
    const int place[2] = {(g ^ (li & 7)) * 8, ((4 + g) ^ (li & 7)) * 8};
    auto read = [&](int r, auto set_, int stage) {                // operand r of the half `set`
        constexpr int set = decltype(set_)::value;
        const __bf16* base = wide_lds + stage * S::STAGE + li * WIDE_BK + place[set];
        if (r < TN) wf[set][r] = *reinterpret_cast<const bf16x8*>(base + (wn * TN + r) * 16 * WIDE_BK);
        else af[set][r - TN] = *reinterpret_cast<const bf16x8*>(base + (BN + (wm * TM + r - TN) * 16) * WIDE_BK);
    };
    constexpr std::integral_constant<int, 0> H0{};
    constexpr std::integral_constant<int, 1> H1{};
    auto read_all = [&](auto set_, int stage) {
#pragma unroll
        for (int r = 0; r < TM + TN; ++r) read(r, set_, stage);
    };
    // The products of half `set`; between them, when READ, the reads of the other half out of `from` (all but the last row of
    // tiles are behind them, so that they are there when their turn comes) and, when LOAD, the loads of block kb into `into`.
    // The scheduling barriers keep it so: on its own the compiler asks for everything first and multiplies then.
    auto products = [&](auto set_, auto read_, int from, auto load_, int kb, int into) {
        constexpr int set = decltype(set_)::value;
        constexpr int OPERANDS = TM + TN, ROWS = TM > 1 ? TM - 1 : 1, PER_ROW = (OPERANDS + ROWS - 1) / ROWS;
        constexpr int LOADS_ROW = (LOADS + TM - 1) / TM;
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            if constexpr (decltype(read_)::value) {
#pragma unroll
                for (int r = i * PER_ROW; r < (i + 1) * PER_ROW && r < OPERANDS; ++r) read(r, std::integral_constant<int, set ^ 1>{}, from);
            }
            if constexpr (decltype(load_)::value) {
#pragma unroll
                for (int l = i * LOADS_ROW; l < (i + 1) * LOADS_ROW && l < LOADS; ++l) load(l, kb, into);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < TN; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[set][j], af[set][i], acc[i][j], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_s_setprio(0);
    };

    // QKV: thread t looks up where row m0 + t of the tile lies in the cache, behind the first loads of operands
    int row_pos = 0, row_slot = 0, row_page = -1;
    if constexpr (QKV) {
        const int m = min(m0 + t, M - 1);
        row_pos = args.positions[m];
        row_slot = args.slots[m];
    }
    int32_t* row_lds = reinterpret_cast<int32_t*>(reinterpret_cast<unsigned char*>(wide_lds) + (QKV ? Q::rows_at : 0));   // [BM] positions, pages, places
    auto find_page = [&]() {
        if constexpr (QKV) {
            if (t < BM) row_lds[t] = row_pos;                     // (the loop's barriers lie before its readers)
            const int block = row_pos / args.page_size;
            const int id = args.block_table[(size_t)row_slot * args.max_blocks + min(args.write_cache ? block : 0, args.max_blocks - 1)];
            row_page = args.write_cache && block < args.max_blocks && m0 + t < M ? id : -1;
        }
    };

    if constexpr (PAIRED) {
        constexpr int PAIRS = NS / 2, LOADS_PAIR = 2 * LOADS;
        static_assert(NS % 2 == 0 && PAIRS >= 2, "whole pairs of blocks");
        bf16x8 pw[2][4][TN], pa[2][4][TM];                        // two sets of a pair's four halves
        // (an odd count's last pair holds its last block twice and multiplies it once)
        auto load_pair = [&](int turn, int pair) {
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int i = 0; i < LOADS; ++i) load(i, min(2 * turn + h, blocks - 1), 2 * pair + h);
        };
        auto read_pair = [&](auto set_, int pair) {
            constexpr int set = decltype(set_)::value;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const __bf16* base = wide_lds + (2 * pair + q / 2) * S::STAGE + li * WIDE_BK + place[q & 1];
#pragma unroll
                for (int j = 0; j < TN; ++j) pw[set][q][j] = *reinterpret_cast<const bf16x8*>(base + (wn * TN + j) * 16 * WIDE_BK);
#pragma unroll
                for (int i = 0; i < TM; ++i) pa[set][q][i] = *reinterpret_cast<const bf16x8*>(base + (BN + (wm * TM + i) * 16) * WIDE_BK);
            }
        };
        auto multiply = [&](auto set_, int halves) {
            constexpr int set = decltype(set_)::value;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (q == 2 && halves == 2) break;
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pw[set][q][j], pa[set][q][i], acc[i][j], 0, 0, 0);
                if (q % 2 == 1) block_done();
            }
        };
        const int turns = (blocks + 1) / 2, last = blocks % 2 ? 2 : 4;
        if (turns >= PAIRS) {
#pragma unroll
            for (int t = 0; t < PAIRS; ++t) load_pair(t, t);
            wide_arrive<LOADS_PAIR * (PAIRS - 1)>();
            read_pair(H0, 0);
            int pair = 0;
            // A turn: behind the barrier everyone has read its pair, which is filled again, and the next one is there: it is
            // read into the other set while this one is multiplied.
            auto turn = [&](auto set_, int t) {
                constexpr int set = decltype(set_)::value;
                const int next = pair + 1 == PAIRS ? 0 : pair + 1;
                wide_arrive<LOADS_PAIR * (PAIRS - 2)>();
                read_pair(std::integral_constant<int, set ^ 1>{}, next);
                load_pair(t + PAIRS, pair);
                __builtin_amdgcn_sched_barrier(0);
                multiply(set_, 4);
                pair = next;
            };
            auto tail = [&](auto self, auto set_, auto left_) {   // the last PAIRS turns: nothing more to ask for
                constexpr int set = decltype(set_)::value, LEFT = decltype(left_)::value;
                if constexpr (LEFT > 1) {
                    const int next = pair + 1 == PAIRS ? 0 : pair + 1;
                    wide_arrive<LOADS_PAIR * (LEFT > 1 ? LEFT - 2 : 0)>();
                    read_pair(std::integral_constant<int, set ^ 1>{}, next);
                    __builtin_amdgcn_sched_barrier(0);
                    multiply(set_, 4);
                    pair = next;
                    self(self, std::integral_constant<int, set ^ 1>{}, std::integral_constant<int, LEFT - 1>{});
                } else {
                    multiply(set_, last);
                }
            };
            int t = 0;
#pragma unroll 1
            for (; t + 1 < turns - PAIRS; t += 2) {
                turn(H0, t);
                turn(H1, t + 1);
            }
            constexpr std::integral_constant<int, PAIRS> ALL{};
            if (t < turns - PAIRS) {
                turn(H0, t);
                tail(tail, H1, ALL);
            } else {
                tail(tail, H0, ALL);
            }
        } else {                                                  // fewer pairs than the LDS holds: all at once
            for (int t = 0; t < turns; ++t) load_pair(t, t);
            wide_arrive<0>();
            for (int t = 0; t < turns; ++t) {
                read_pair(H0, t);
                multiply(H0, t + 1 < turns ? 4 : last);
            }
        }
    } else if (blocks >= NS) {
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int i = 0; i < LOADS; ++i) load(i, s, s);
        find_page();
        wide_arrive<LOADS * (NS - 1)>();
        read_all(H0, 0);
        int stage = 0;
        // A turn: the first half's products beside the second half's reads; the block is read out then and, once everyone is
        // there, is filled again with block kb + NS beside the second half's products, while the next block's operands arrive.
#pragma unroll 1
        for (int kb = 0; kb < blocks - NS; ++kb) {
            const int next = stage + 1 == NS ? 0 : stage + 1;
            products(H0, std::true_type{}, stage, std::false_type{}, 0, 0);
            wide_arrive<LOADS * (NS - 2)>();
            products(H1, std::true_type{}, next, std::true_type{}, kb + NS, stage);
            block_done();
            stage = next;
        }
        auto tail = [&](auto self, auto left_) {                  // the last NS blocks: nothing more to ask for
            constexpr int LEFT = decltype(left_)::value;
            if constexpr (LEFT > 0) {
                const int next = stage + 1 == NS ? 0 : stage + 1;
                products(H0, std::true_type{}, stage, std::false_type{}, 0, 0);
                if constexpr (LEFT > 1) {
                    wide_arrive<LOADS * (LEFT > 1 ? LEFT - 2 : 0)>();
                    products(H1, std::true_type{}, next, std::false_type{}, 0, 0);
                } else {
                    products(H1, std::false_type{}, 0, std::false_type{}, 0, 0);
                }
                block_done();
                stage = next;
                self(self, std::integral_constant<int, LEFT - 1>{});
            }
        };
        tail(tail, std::integral_constant<int, NS>{});
    } else {                                                      // fewer blocks than the LDS holds: all at once
        for (int s = 0; s < blocks; ++s)
#pragma unroll
            for (int i = 0; i < LOADS; ++i) load(i, s, s);
        find_page();
        wide_arrive<0>();
        for (int s = 0; s < blocks; ++s) {
            read_all(H0, s);
            read_all(H1, s);
            products(H0, std::false_type{}, 0, std::false_type{}, 0, 0);
            products(H1, std::false_type{}, 0, std::false_type{}, 0, 0);
            block_done();
        }
    }
    if constexpr (FEW) close_part();                              // (the last part, where it is a shorter one)
    if constexpr (SPLIT > 1) {
        // The shares' sums pass the L2s (coherent at the device), whatever XCD the last workgroup runs on: they are there once the
        // stores are through, and only then is the arrival counted.
        constexpr int VALUES = SKINNY_WAVES - PER + 1, LANE = 4 * 64 * WM * WN, AROUND = 0x10;     // (AROUND: sc1)
        const int tile = tm * args.tiles_n + tn;
        const auto rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)(args.partial + (size_t)tile * VALUES * TM * TN * LANE), 0, VALUES * TM * TN * LANE * 4, 0x00027000);
        auto at = [&](int v, int i, int j) { return ((v * TM + i) * TN + j) * LANE * 4; };
        typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t u32x4_t;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                if (share == 0) {
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, sum[i][j]), rsrc, t * 16, at(0, i, j), AROUND);
                } else {
#pragma unroll
                    for (int q = 0; q < PER; ++q)
                        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, part[q][i][j]), rsrc, t * 16, at(1 + (share - 1) * PER + q, i, j), AROUND);
                }
            }
        wide_arrive<0>();
        int32_t* meet = reinterpret_cast<int32_t*>(wide_lds);
        if (t == 0) *meet = __hip_atomic_fetch_add(args.arrivals + tile, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (*meet != SPLIT - 1) return;
        if (t == 0) __hip_atomic_store(args.arrivals + tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("" ::: "memory");
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                u32x4_t got[VALUES];
#pragma unroll
                for (int v = 0; v < VALUES; ++v) got[v] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, t * 16, at(v, i, j), AROUND);
                acc[i][j] = __builtin_bit_cast(floatx4, got[0]);
#pragma unroll
                for (int v = 1; v < VALUES; ++v) acc[i][j] += __builtin_bit_cast(floatx4, got[v]);
            }
    } else if constexpr (FEW) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = sum[i][j];
    }

    if constexpr (OUT_FLOAT) {
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int m = m0 + (wm * TM + i) * 16 + li;
            if (m >= M) continue;
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int n = n0 + (wn * TN + j) * 16 + 4 * g;
                float* o = (float*)args.out + (size_t)m * N + n;
                if (args.vector_out && n + 3 < N) *reinterpret_cast<floatx4*>(o) = acc[i][j];
                else
#pragma unroll
                    for (int r = 0; r < 4; ++r) if (n + r < N) o[r] = acc[i][j][r];
            }
        }
        return;
    }
    if constexpr (QKV) {
        // What counts here is the path for requests (16 bytes a lane take it 16 cycles a wavefront) and the instructions: the norm's
        // weights are asked for once a thread, which stays with one head of the tile, and the rotation of its rows before the tile is
        // put into LDS.
        constexpr int LANES = 8, THREADS = 64 * S::WAVES, AHEAD = Q::PASSES < 4 ? Q::PASSES : 4;
        constexpr int ROWS = THREADS / LANES / Q::HEADS;          // of a pass
        static_assert(THREADS / LANES % Q::HEADS == 0 && Q::PASSES % AHEAD == 0, "a thread stays with one head");
        typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4_t;
        const int head0 = n0 / QKV_HEAD, all_heads = args.q_heads + 2 * args.kv_heads, turned = args.q_heads + args.kv_heads;
        const int P = args.page_size, c = t % LANES, at = t / LANES % Q::HEADS, my_row = t / LANES / Q::HEADS, head = head0 + at;
        const bool is_q = head < args.q_heads;
        floatx4 co[AHEAD][2], si[AHEAD][2], wl[2], wh[2];
        auto ask = [&](int pass0) {
#pragma unroll
            for (int p = 0; p < AHEAD; ++p) {
                const float* cs = args.rope + (size_t)row_lds[my_row + (pass0 + p) * ROWS] * QKV_HEAD + 8 * c;
#pragma unroll
                for (int x = 0; x < 2; ++x) {
                    co[p][x] = *reinterpret_cast<const floatx4*>(cs + 4 * x);
                    si[p][x] = *reinterpret_cast<const floatx4*>(cs + 64 + 4 * x);
                }
            }
        };
        const float* w = is_q ? args.q_norm_w : args.k_norm_w;
        const bool normed = w != nullptr;
        if (head0 < turned) {
            ask(0);
            if (normed) {
#pragma unroll
                for (int x = 0; x < 2; ++x) {
                    wl[x] = *reinterpret_cast<const floatx4*>(w + 8 * c + 4 * x);
                    wh[x] = *reinterpret_cast<const floatx4*>(w + 64 + 8 * c + 4 * x);
                }
            }
        }
        // (the last operands are there since the last turn but one: behind the barrier everyone has read them)
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (t < BM) {                                             // (whole wavefronts)
            const int place = row_pos % P;
            row_lds[BM + t] = row_page;
            row_lds[2 * BM + t] = place;
            const int page_before = __shfl_up(row_page, 1, MLR_WAVE), place_before = __shfl_up(place, 1, MLR_WAVE);       // (by all lanes)
            const bool follows = lane % 8 == 0 ? place % 8 == 0 && row_page >= 0 : page_before == row_page && place_before + 1 == place;
            const uint64_t all = __builtin_amdgcn_ballot_w64(follows);
            if (lane % 8 == 0) row_lds[3 * BM + t / 8] = (all >> lane & 0xff) == 0xff;
        }
        const int wave_head = wn * TN * 16 / QKV_HEAD, in_head = wn * TN * 16 % QKV_HEAD;         // a wavefront's columns are of one head
        static_assert(QKV_HEAD % (TN * 16) == 0 && QKV_HEAD * Q::VPITCH <= Q::HEAD, "a wavefront's columns are of one head, whose values take its place");
        __bf16* tile = wide_lds + wave_head * Q::HEAD;
        typedef __attribute__((__vector_size__(2 * sizeof(uint32_t)))) uint32_t uint2_t;
        const bool of_values = head0 + wave_head >= turned;
        const uint32_t pick = lane & 1 ? 0x03020706u : 0x05040100u;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const bf16x4_t four = {(__bf16)acc[i][j][0], (__bf16)acc[i][j][1], (__bf16)acc[i][j][2], (__bf16)acc[i][j][3]};
                if (!of_values) {
                    *reinterpret_cast<bf16x4_t*>(tile + ((wm * TM + i) * 16 + li) * Q::PITCH + in_head + j * 16 + 4 * g) = four;
                    continue;
                }
                // four channels of one row a lane become four rows of one channel, between the four lanes of a quad: halves with the
                // lane two places away, then quarters with its neighbour
                const uint2_t own = __builtin_bit_cast(uint2_t, four);
                const uint32_t other = __builtin_amdgcn_mov_dpp(lane & 2 ? own[0] : own[1], 0x4e, 0xf, 0xf, true);
                const uint32_t lo = lane & 2 ? other : own[0], hi = lane & 2 ? own[1] : other;
                const uint2_t rows = {__builtin_amdgcn_perm(__builtin_amdgcn_mov_dpp(lo, 0xb1, 0xf, 0xf, true), lo, pick),
                                      __builtin_amdgcn_perm(__builtin_amdgcn_mov_dpp(hi, 0xb1, 0xf, 0xf, true), hi, pick)};
                *reinterpret_cast<uint2_t*>(tile + (in_head + j * 16 + 4 * g + (lane & 3)) * Q::VPITCH + (wm * TM + i) * 16 + (li & ~3)) = rows;
            }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (head0 < turned) {                                     // queries and keys: eight lanes a row of a head
#pragma unroll
            for (int pass0 = 0; pass0 < Q::PASSES; pass0 += AHEAD) {
                if (pass0 > 0) ask(pass0);
#pragma unroll
                for (int p = 0; p < AHEAD; ++p) {
                    const int row = my_row + (pass0 + p) * ROWS;
                    const __bf16* from = wide_lds + at * Q::HEAD + row * Q::PITCH + 8 * c;
                    const bf16x8 lo = *reinterpret_cast<const bf16x8*>(from), hi = *reinterpret_cast<const bf16x8*>(from + 64);
                    const int page = row_lds[BM + row], place = row_lds[2 * BM + row];
                    float a[8], b[8], sum = 0.f;
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        a[e] = (float)lo[e];
                        b[e] = (float)hi[e];
                        sum += squares(a[e], b[e]);
                    }
                    sum = group_sum(sum, LANES);
                    if (normed) {
                        const float scale = 1.0f / sqrtf(sum / (float)QKV_HEAD + args.eps);
#pragma unroll
                        for (int e = 0; e < 8; ++e) {
                            a[e] = (a[e] * scale) * wl[e / 4][e % 4];
                            b[e] = (b[e] * scale) * wh[e / 4][e % 4];
                        }
                    }
                    bf16x8 x8, y8;
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        x8[e] = (__bf16)turn_x(a[e], b[e], co[p][e / 4][e % 4], si[p][e / 4][e % 4]);
                        y8[e] = (__bf16)turn_y(a[e], b[e], co[p][e / 4][e % 4], si[p][e / 4][e % 4]);
                    }
                    if (m0 + row >= M || head >= turned || (!is_q && page < 0)) continue;
                    __bf16* dst = is_q ? args.q_out + ((size_t)(m0 + row) * args.q_heads + head) * QKV_HEAD
                                       : args.k_pages + (((size_t)page * args.kv_heads + head - args.q_heads) * P + place) * QKV_HEAD;
                    *reinterpret_cast<bf16x8*>(dst + 8 * c) = x8;
                    *reinterpret_cast<bf16x8*>(dst + 64 + 8 * c) = y8;
                }
            }
        }
        // values: a thread takes eight rows of a channel, one store where they are eight neighbouring places of a page (two eights of
        // a channel side by side: with pages of sixteen, lanes that follow each other write bytes that do)
        for (int v = max(turned - head0, 0); v < Q::HEADS && head0 + v < all_heads; ++v) {
            __bf16* pages = args.v_pages + (size_t)(head0 + v - turned) * QKV_HEAD * P;
            const size_t page_elems = (size_t)args.kv_heads * QKV_HEAD * P;
#pragma unroll 2
            for (int item = t; item < BM / 8 * QKV_HEAD; item += THREADS) {
                const int d = (item >> 1) % QKV_HEAD, r0 = (item / (2 * QKV_HEAD) * 2 + (item & 1)) * 8;
                const bf16x8 rows = *reinterpret_cast<const bf16x8*>(wide_lds + v * Q::HEAD + d * Q::VPITCH + r0);
                const int page = row_lds[BM + r0], place = row_lds[2 * BM + r0];
                if (row_lds[3 * BM + r0 / 8]) {
                    *reinterpret_cast<bf16x8*>(pages + page * page_elems + (size_t)d * P + place) = rows;
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (row_lds[BM + r0 + e] >= 0) pages[row_lds[BM + r0 + e] * page_elems + (size_t)d * P + row_lds[2 * BM + r0 + e]] = rows[e];
                }
            }
        }
        return;
    }
    // bfloat16 results leave through LDS: a lane holds four columns of one row, which would be stores of 8 bytes to 64 different
    // rows; a piece of LDS of the wavefront's own turns them into rows of 16-byte pieces (measured on 2048 x 4096 x 1024 with
    // this kernel's predecessor: the stores took 8 of 28 us).  A wavefront's tiles take the LDS one half after the other
    // where all of them do not fit.
    constexpr int TNO = GATED ? TN / 2 : TN, COLS = TNO * 16, PITCH = TN * 16 + 8, PIECES = COLS / 8;
    constexpr int TC = (size_t)S::WAVES * TM * 16 * PITCH * sizeof(__bf16) <= S::lds_bytes ? TM : TM / 2, HALF = TC * 16;
    static_assert(TM % TC == 0 && (size_t)S::WAVES * HALF * PITCH * sizeof(__bf16) <= S::lds_bytes, "the output tiles must fit the LDS");
    wide_arrive<0>();                                             // every wavefront has read its last operands
    __bf16* mine = wide_lds + wave * HALF * PITCH;
    const bool fused = GATED && (args.act == WIDE_SILU || (FEW && args.act == WIDE_CLAMPED_SUMS));      // (its gate never leaves the registers)
#pragma unroll
    for (int i0 = 0; i0 < TM; i0 += TC) {
        auto put = [&](int i, int j, float y0, float y1, float y2, float y3) {
            typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4_t;
            *reinterpret_cast<bf16x4_t*>(mine + (i * 16 + li) * PITCH + j * 16 + 4 * g) = bf16x4_t{(__bf16)y0, (__bf16)y1, (__bf16)y2, (__bf16)y3};
        };
        if (fused) {
#pragma unroll
            for (int i = 0; i < TC; ++i)
#pragma unroll
                for (int j = 0; j < TN / 2; ++j) {
                    float y[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        // silu(g) = g / (1 + 2^(-g log2 e)).  Many rows: with the hardware's exponential and reciprocal (both good
                        // to an ulp or so of 32 bits; the result is rounded to bfloat16): a full division costs ten instructions,
                        // and a lane has 2 TM TN of these.  Few rows have few, and what `gemm_skinny_kernel` makes of them.
                        const float gate = acc[i0 + i][2 * j][r], up = acc[i0 + i][(2 * j + 1) % TN][r];
                        y[r] = FEW ? args.act == WIDE_CLAMPED_SUMS ? clamped_glu(gate, up, args.limit, args.slope) : gate_act<0>(gate) * up
                                   : gate * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.44269504088896340736f * gate)) * up;
                    }
                    put(i, j, y[0], y[1], y[2], y[3]);
                }
        } else {
#pragma unroll
            for (int i = 0; i < TC; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) put(i, j, acc[i0 + i][j][0], acc[i0 + i][j][1], acc[i0 + i][j][2], acc[i0 + i][j][3]);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll 2
        for (int c = lane; c < HALF * PIECES; c += 64) {
            const int row = c / PIECES, piece = c % PIECES;
            const int m = m0 + (wm * TM + i0) * 16 + row, n = n0 + wn * COLS + 8 * piece;
            if (m >= M || n >= N) continue;
            const __bf16* from = mine + row * PITCH;
            bf16x8 v;
            if (!GATED || fused) {
                v = *reinterpret_cast<const bf16x8*>(from + 8 * piece);
                if (!GATED && args.act != WIDE_PLAIN) {
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        v[e] = (__bf16)(args.act == WIDE_RELU_SQUARED ? plain_act<0>((float)v[e]) : plain_act<1>((float)v[e]));
                }
            } else {                                              // gate and up lie in neighbouring tiles
                from += (piece >> 1) * 32 + (piece & 1) * 8;
                const bf16x8 gate = *reinterpret_cast<const bf16x8*>(from), up = *reinterpret_cast<const bf16x8*>(from + 16);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float x = (float)gate[e], u = (float)up[e];
                    v[e] = (__bf16)(args.act == WIDE_CLAMPED ? clamped_glu(x, u, args.limit, args.slope)
                                    : (args.act == WIDE_GELU_TANH ? gate_act<1>(x) : args.act == WIDE_RELU ? gate_act<2>(x) : gate_act<0>(x)) * u);
                }
            }
            __bf16* o = (__bf16*)args.out + (HEADS ? (size_t)m * args.ldo + (size_t)head * args.out_head : (size_t)m * N) + n;
            if (args.vector_out && n + 8 <= N) {
                *reinterpret_cast<bf16x8*>(o) = v;
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) if (n + e < N) o[e] = v[e];
            }
        }
        if (TC < TM) {                                            // the second half's tiles overwrite what was just read
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
    }
}

template <int WM, int WN, int TM, int TN, int NS, bool OUT_FLOAT, bool GATED, bool FEW = false, bool PAIRED = false>
static int launch_wide_as(WideArgs& args, hipStream_t stream) {
    using S = WideShape<WM, WN, TM, TN, NS>;
    constexpr int NOUT = GATED ? S::BN / 2 : S::BN;
    args.tiles_m = (args.M + S::BM - 1) / S::BM;
    args.tiles_n = (args.N + NOUT - 1) / NOUT;
    if ((long long)args.tiles_m * args.tiles_n > 0x7fffffffLL / 8) return -2;
    auto* kernel = gemm_wide_kernel<WM, WN, TM, TN, NS, OUT_FLOAT, GATED, false, FEW, PAIRED>;
    static const hipError_t allowed = hipFuncSetAttribute(
        reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)S::lds_bytes);
    if (allowed != hipSuccess) return (int)allowed;
    kernel<<<dim3(args.tiles_m * args.tiles_n), 64 * S::WAVES, S::lds_bytes, stream>>>(args);
    return (int)hipGetLastError();
}
// (the gated form where its tiles must come in pairs and the plain one's do not: the same workgroup tile, other wavefronts)
template <int WM, int WN, int TM, int TN, int NS, int GWM = WM, int GWN = WN, int GTM = TM, int GTN = TN>
static int launch_wide(WideArgs& args, bool out_float, bool gated, hipStream_t stream) {
    static_assert(WM * TM == GWM * GTM && WN * TN == GWN * GTN, "one tile for both forms");
    if constexpr (GTN % 2 == 0) {
        if (gated) return launch_wide_as<GWM, GWN, GTM, GTN, NS, false, true>(args, stream);
    }
    if (gated) return -1;
    if (out_float) return launch_wide_as<WM, WN, TM, TN, NS, true, false>(args, stream);
    return launch_wide_as<WM, WN, TM, TN, NS, false, false>(args, stream);
}

// The kernel's shapes: rows and columns of a workgroup's tile (gated: half as many output columns), workgroups that a compute
// unit holds at once, and what 1024 k of a tile cost in microseconds, alone on its compute unit or beside a second one, with
// what a launch costs besides: fitted to 168 products of 33 to 2048 rows and fourteen inner and outer sizes between 1024 and
// 25600 (rms 9 to 13 % a shape; the shape with the least predicted time is then within 1 % of the best one on average).
struct WideCost { int bm, bn, per_unit; float fixed, one, all; };
#define WIDE_SHAPES 10
static const WideCost WIDE_COSTS[WIDE_SHAPES] = {
    {64, 32, 2, 1.2f, 2.9f, 4.9f},     {64, 64, 2, 1.0f, 3.9f, 6.9f},     {96, 64, 2, 0.6f, 4.6f, 8.8f},    {128, 64, 1, 0.3f, 0.f, 5.7f},
    {128, 128, 1, -0.1f, 0.f, 8.1f},   {192, 128, 1, 1.2f, 0.f, 9.8f},    {128, 192, 1, 0.6f, 0.f, 10.4f},  {256, 128, 1, 1.9f, 0.f, 11.9f},
    {256, 192, 1, -2.2f, 0.f, 19.4f},  {256, 256, 1, -1.1f, 0.f, 21.8f}};


// The same for 17 to 64 rows, where a workgroup reads its weight once and what counts is the bytes of weight under way and what a
// turn waits: narrow tiles with up to 19 blocks on their way, two of them a turn.  `turn`: what a round takes whatever k is (its
// first blocks' way, closing the parts of k, the epilogue); `row`: what 16 more rows add to 1024 k of one.  Fitted to 768 products of
// 17 to 64 rows, inner sizes drawn from 512 to 9000 and 256 to 36000 rows of weight, weights cold (the predicted tile is 0.5 % behind
// the best one, geometric mean).  Strips of 16 columns have no gated form.  32 x 4096 x 1024 5.0 us, 32 x 2112 x 4096 9.5,
// 17 x 2 * 704 x 2048 6.1; tiles of 64 x 32 and 64 x 64, which two workgroups of a compute unit share, gain nothing by two blocks a turn.
struct FewCost { int shape, bm, bn, per_unit; float fixed, turn, one, all, row; };
static const FewCost FEW_COSTS[] = {
    {10, 64, 16, 1, 0.47f, 1.99f, 0.f, 1.42f, 0.253f}, {11, 64, 96, 1, -3.38f, 6.82f, 0.f, 3.83f, 0.461f}, {12, 32, 16, 1, 0.25f, 2.28f, 0.f, 1.51f, 0.f},
    {13, 32, 32, 1, -0.86f, 3.48f, 0.f, 2.12f, 0.f},   {14, 32, 64, 1, -3.54f, 6.09f, 0.f, 3.32f, 0.f},    {15, 64, 32, 2, 1.83f, 1.25f, 2.05f, 5.37f, 0.465f},
    {16, 64, 64, 2, 2.20f, 0.93f, 2.60f, 9.16f, 0.711f}};

static int few_shape_for(int M, int N, int K, bool gated) {
    const int units = compute_units() > 0 ? compute_units() : 256, row_tiles = (M + 15) / 16;
    int best = -1;
    float time = 0.f;
    for (const FewCost& c : FEW_COSTS) {
        if (M > c.bm || (gated && c.bn == 16)) continue;
        const int bn = gated ? c.bn / 2 : c.bn, tiles = (N + bn - 1) / bn, slots = units * c.per_unit, left = tiles % slots;
        const bool alone = c.per_unit == 2 && left > 0 && left <= units;
        const float rounds = (float)(tiles / slots + (left > 0 && !alone ? 1 : 0)), more = c.row * (float)row_tiles;
        const float us = c.fixed + (rounds + (alone ? 0.6f : 0.f)) * c.turn +
                         (rounds * (c.all + more) + (alone ? c.one + 0.6f * more : 0.f)) * (float)K * (1.0f / 1024.0f);
        if (best < 0 || us < time) {
            best = c.shape;
            time = us;
        }
    }
    return best;
}

// The tiles for up to 64 rows (never with 32-bit results: those are the library's).
template <bool PAIRED, int WM, int WN, int TM, int TN, int NS, int GWM = WM, int GWN = WN, int GTM = TM, int GTN = TN>
static int launch_few(WideArgs& args, bool out_float, bool gated, hipStream_t stream) {
    static_assert(WM * TM == GWM * GTM && WN * TN == GWN * GTN, "one tile for both forms");
    if (out_float) return -1;
    if (!gated) return launch_wide_as<WM, WN, TM, TN, NS, false, false, true, PAIRED>(args, stream);
    if constexpr (GTN % 2 == 0) return launch_wide_as<GWM, GWN, GTM, GTN, NS, false, true, true, PAIRED>(args, stream);
    return -1;
}

// The forms with several workgroups a tile (SPLIT), and what they cost: as above, a round's time by 1024 k of a share, `row` by 16 rows;
// `half`: the same of a last round whose workgroups have a compute unit each.  Fitted to 560 products of 17 to 64 rows (200 of up to 32),
// inner sizes drawn from 1500 to 26000 and 512 to 16384 rows of weight, weights cold (rms 6 to 14 %; the predicted form is 0.7 %
// behind the best one, geometric mean).
struct SplitCost { int shape, splits, bm, bn, per_unit; float fixed, turn, all, row, half_turn, half_all, half_row; };
static const SplitCost SPLIT_COSTS[] = {
    {0, 2, 32, 64, 1, -2.16f, 6.78f, 0.76f, 1.53f, 0.f, 0.f, 0.f},  {1, 2, 64, 64, 2, 5.14f, 4.57f, 7.40f, 0.94f, 0.56f, 3.02f, 0.43f},
    {2, 4, 32, 32, 1, 1.61f, 3.19f, 0.48f, 0.97f, 0.f, 0.f, 0.f},   {3, 4, 32, 64, 1, 0.03f, 4.88f, 0.80f, 1.61f, 0.f, 0.f, 0.f},
    {4, 4, 64, 64, 2, 1.00f, 7.20f, 9.18f, 0.65f, 4.71f, 3.03f, 0.48f}, {5, 4, 64, 128, 1, -2.00f, 9.44f, 5.99f, 0.52f, 0.f, 0.f, 0.f},
    {6, 4, 64, 32, 2, 2.07f, 3.93f, 3.92f, 0.90f, 2.80f, 2.45f, 0.24f},
    // up to 16 rows: fitted to 250 products of them, inner sizes from 2000 to 26000 (rms 6, 11 and 14 %; 1.3 % behind the best form)
    {7, 4, 16, 32, 2, 2.11f, 2.73f, 4.85f, 0.f, 2.39f, 2.45f, 0.f}, {8, 4, 16, 64, 2, 0.52f, 4.32f, 9.20f, 0.f, 3.92f, 3.47f, 0.f},
    {9, 2, 16, 64, 1, -4.12f, 8.15f, 3.26f, 0.f, 0.f, 0.f, 0.f}};

static int split_shape_for(int M, int N, int K) {
    const int units = compute_units() > 0 ? compute_units() : 256;
    const float row_tiles = (float)((M + 15) / 16);
    int best = -1;
    float time = 0.f;
    for (const SplitCost& c : SPLIT_COSTS) {
        if (M > c.bm || (M <= 16) != (c.bm == 16)) continue;
        const int workgroups = (N + c.bn - 1) / c.bn * c.splits, slots = units * c.per_unit, left = workgroups % slots;
        const bool half = c.per_unit == 2 && left > 0 && left <= units;
        const float rounds = (float)(workgroups / slots + (left > 0 && !half ? 1 : 0)), k = (float)(K / c.splits) * (1.0f / 1024.0f);
        const float us = c.fixed + rounds * (c.turn + (c.all + c.row * row_tiles) * k) + (half ? c.half_turn + (c.half_all + c.half_row * row_tiles) * k : 0.f);
        if (best < 0 || us < time) {
            best = c.shape;
            time = us;
        }
    }
    return best;
}

template <int SPLIT, bool PAIRED, int WM, int WN, int TM, int TN, int NS>
static int launch_split(WideArgs& args, long floats, int counters, hipStream_t stream) {
    using S = WideShape<WM, WN, TM, TN, NS>;
    constexpr int PER = SKINNY_WAVES / SPLIT;
    args.tiles_m = (args.M + S::BM - 1) / S::BM;
    args.tiles_n = (args.N + S::BN - 1) / S::BN;
    const long tiles = (long)args.tiles_m * args.tiles_n, blocks = args.K / WIDE_BK, part_blocks = (blocks + SKINNY_WAVES - 1) / SKINNY_WAVES;
    // (every workgroup has something to multiply; the last one's blocks are those that are left)
    if (args.tiles_m != 1 || tiles > counters || tiles * (SKINNY_WAVES - PER + 1) * S::BM * S::BN > floats || blocks <= (SPLIT - 1) * PER * part_blocks) return -1;
    auto* kernel = gemm_wide_kernel<WM, WN, TM, TN, NS, false, false, false, true, PAIRED, false, SPLIT>;
    static const hipError_t allowed = hipFuncSetAttribute(
        reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)S::lds_bytes);
    if (allowed != hipSuccess) return (int)allowed;
    kernel<<<dim3((unsigned)(tiles * SPLIT)), 64 * S::WAVES, S::lds_bytes, stream>>>(args);
    return (int)hipGetLastError();
}

static int launch_split_shape(int shape, WideArgs& args, long floats, int counters, hipStream_t stream) {
    switch (shape) {
        case 0: return launch_split<2, true, 2, 2, 1, 2, 12>(args, floats, counters, stream);
        case 1: return launch_split<2, false, 2, 2, 2, 2, 5>(args, floats, counters, stream);
        case 2: return launch_split<4, true, 2, 1, 1, 2, 14>(args, floats, counters, stream);
        case 3: return launch_split<4, true, 2, 2, 1, 2, 12>(args, floats, counters, stream);
        case 4: return launch_split<4, false, 2, 2, 2, 2, 5>(args, floats, counters, stream);
        case 5: return launch_split<4, false, 2, 2, 2, 4, 6>(args, floats, counters, stream);
        case 6: return launch_split<4, false, 2, 2, 2, 1, 6>(args, floats, counters, stream);
        case 7: return launch_split<4, false, 1, 2, 1, 1, 12>(args, floats, counters, stream);
        case 8: return launch_split<4, false, 1, 2, 1, 2, 8>(args, floats, counters, stream);
        case 9: return launch_split<2, true, 1, 2, 1, 2, 12>(args, floats, counters, stream);
        default: return -1;
    }
}

static int launch_wide_shape(int shape, WideArgs& args, bool out_float, bool gated, hipStream_t stream) {
    switch (shape) {
        case 0: return launch_wide<2, 2, 2, 1, 6, 4, 1, 1, 2>(args, out_float, gated, stream);
        case 1: return launch_wide<2, 2, 2, 2, 5>(args, out_float, gated, stream);
        case 2: return launch_wide<2, 2, 3, 2, 4>(args, out_float, gated, stream);
        case 3: return launch_wide<4, 2, 2, 2, 6>(args, out_float, gated, stream);
        case 4: return launch_wide<2, 4, 4, 2, 4>(args, out_float, gated, stream);
        case 5: return launch_wide<4, 2, 3, 4, 3>(args, out_float, gated, stream);
        case 6: return launch_wide<2, 4, 4, 3, 3, 4, 2, 2, 6>(args, out_float, gated, stream);
        case 7: return launch_wide<4, 2, 4, 4, 3>(args, out_float, gated, stream);
        case 8: return launch_wide<4, 2, 4, 6, 2>(args, out_float, gated, stream);
        case 9: return launch_wide<2, 4, 8, 4, 2>(args, out_float, gated, stream);
        case 10: return launch_few<true, 2, 1, 2, 1, 12>(args, out_float, gated, stream);
        case 11: return launch_few<false, 2, 2, 2, 3, 7, 4, 1, 1, 6>(args, out_float, gated, stream);
        case 12: return launch_few<true, 2, 1, 1, 1, 20>(args, out_float, gated, stream);
        case 13: return launch_few<true, 2, 1, 1, 2, 14>(args, out_float, gated, stream);
        case 14: return launch_few<true, 2, 2, 1, 2, 12>(args, out_float, gated, stream);
        case 15: return launch_few<false, 2, 2, 2, 1, 6, 4, 1, 1, 2>(args, out_float, gated, stream);
        case 16: return launch_few<false, 2, 2, 2, 2, 5>(args, out_float, gated, stream);
        default: return -1;
    }
}

// The predicted time of a shape in microseconds.
static float wide_time(int shape, int M, int N, int K, bool gated) {
    const int units = compute_units() > 0 ? compute_units() : 256;
    const WideCost& c = WIDE_COSTS[shape];
    const int bn = gated ? c.bn / 2 : c.bn;
    const long long tiles = (long long)((M + c.bm - 1) / c.bm) * ((N + bn - 1) / bn), slots = (long long)units * c.per_unit;
    const long long left = tiles % slots;
    const bool alone = c.per_unit == 2 && left > 0 && left <= units;          // the last tiles have a compute unit each
    const float rounds = (float)(tiles / slots + (left > 0 && !alone ? 1 : 0));
    return c.fixed + (rounds * c.all + (alone ? c.one : 0.f)) * (float)K * (1.0f / 1024.0f);
}

// The shape with the least predicted time, and that time.
static int wide_shape_for(int M, int N, int K, bool gated, float* time) {
    int best = 0;
    for (int s = 0; s < WIDE_SHAPES; ++s) {
        const float us = wide_time(s, M, N, K, gated);
        if (s == 0 || us < *time) {
            best = s;
            *time = us;
        }
    }
    return best;
}

// Whether 17 to 64 rows are the many-row kernel's, instead of the skinny kernels' (which take 64 rows up to k = 1024, 32 up to 2048)
// and of the vendor library's beyond.  It loses where few workgroups walk a long k -- a turn of 128 k waits for a barrier, 0.14 us
// and more -- and where the activation's rows, which every strip of columns reads again, outweigh its weight.  Measured on 768
// products (the sizes of the tiles' fit above), time against those, geometric mean: up to 32 rows 0.4 to 0.85 up to k = 3072, with more than
// 1024 columns 0.5 to 0.8 up to 4096 and, of up to 8192 rows of weight, 0.61 to 0.79 up to 8192; beyond 32 rows 0.42 to 0.84 up to 2048 and,
// gated or of more than 1024 columns, 0.5 to 0.79 up to 3072, and up to 4096 0.64 to 0.93 with a gate and 0.8 to 0.9 without where there are 4096
// columns.  Not beyond: few columns at long k take up to 1.6 of the library's time (48 x 2 * 464 x 4224 10 us for 7), and weights of
// more than 32768 rows 1.03 to 1.16, from 24576 on 1.03 to 1.06 without a gate at k above 2048 (64 x 2 * 25600 x 5120: 106, 121).  All that this takes:
// 0.69 (550 products, 0.37 to 1.24); 24 x 6144 x 1024 8.0 -> 5.8 us, 64 x 6144 x 2048 13.2 -> 10.2, with gate and silu 64 x 2 * 3072 x 1024
// 11.5 -> 7.0, 64 x 2 * 12288 x 4096 46.5 -> 46.2 (the library's product and its activation's launch before).  With the clamped gate, which
// `gemm_skinny_kernel` took up to 64 rows: 17, 32 and 64 x 2 * 5632 x 2048 18.3, 21.0, 31.1 -> 13.3, 13.9, 17.1, 2 * 704 x 2048 9.6, 10.9, 16.2 ->
// 6.5, 6.6, 8.4, 2 * 12288 x 4096 49.8, 58.8, 80.9 -> 52.1, 47.7, 49.3.
static bool few_wins(int M, int N, int K, bool gated) {
    const long long weight = (long long)N * (gated ? 2 : 1);
    if (M <= 16 || M > 64 || weight > (gated || K <= 2048 ? 32768 : 24576)) return false;
    if (M <= 32) return K <= 3072 || (N > 1024 && (K <= 4096 || (K <= 8192 && weight <= 8192)));
    if (K <= 3072) return K <= 2048 || gated || N > 1024;
    return K <= 4096 && (gated ? N > 1024 : N >= 4096);
}

// Whether up to 16 rows are these tiles' as well, instead of `gemm_skinny_kernel` (the same bits), whose wavefronts make a trip to memory
// for every 256 k of their part, one behind the other.  Measured at 1 to 16 rows, weights cold, against it: 220 drawn sizes, geometric
// mean gated from k = 1024 on 0.85 (0.71 to 1.07; 0.99 to 1.08 below), plain from 1408 on, of more than 4352 columns from 1024 on, 0.90
// (0.68 to 1.09; 0.97 to 1.12 below); and 240 of many columns and whole 256s of k, which have the limits further in.  A gate
// of more than 6656 columns: up to k = 1536 1.03 to 1.17, where k is a multiple of 2048 (a tile's rows then share channels of memory,
// it seems) 1.02 to 1.45, of more than 10240 columns below 8 rows 1.03 to 1.07; the others 0.81 to 1.03.  Plain, of more than 8192
// columns, up to 8 rows: 0.97 to 1.19 up to 12288, with such k 1.03 to 1.20; the others 0.81 to 1.05.
// us: 8 x 2 * 5632 x 2048 15.5 -> 13.9, 8 x 2 * 704 x 2048 7.5 -> 6.4, 8 x 6144 x 2048 8.9 -> 7.8, 8 x 2048 x 2048 5.5 -> 5.0; left out:
// 8 x 2 * 16384 x 2048 30.9, 44.0, 1 x 2 * 12288 x 1024 11.5, 13.5, 1 x 16384 x 4096 26.6, 32.0, 4 x 8448 x 1024 6.9, 7.8.
static bool narrow_wins(int M, int N, int K, bool gated) {
    if (M <= 0 || M > 16 || N < 384 || N > 16384 || K > 6144) return false;
    if (gated)
        return K >= 1024 && (N <= 6656 || (K >= 1792 && K % 2048 != 0 && N <= (K > 3072 ? 8192 : M < 8 ? 10240 : 16384)));
    return (K >= 1408 || (K >= 1024 && N > 4352)) && (N <= 8192 || M > 8 || (N > 12800 && K % 2048 != 0));
}

// Whether the kernel takes these operands at all: whole blocks of k, 32-bit offsets, rows that start on 16 bytes.
static bool wide_takes(const void* a, const void* w, int M, int N, int K, bool gated) {
    return K % WIDE_BK == 0 && (unsigned long long)M * K < (1ull << 31) && (unsigned long long)N * (gated ? 2 : 1) * K < (1ull << 31) &&
           ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(w)) & 15) == 0;
}

extern "C" int mlr_gemm_narrow_wins(int M, int N, int K, int gated) {
    return N > 0 && K > 0 && wide_takes(nullptr, nullptr, M, N, K, gated != 0) && narrow_wins(M, N, K, gated != 0) ? 1 : 0;
}

enum { WIDE_MANY = -1, WIDE_FEW = -2 };      // the tile with the least predicted time, of one sum over k or of the forms for up to 64 rows
static int run_wide(int shape, const void* a, const void* w, void* out, int M, int N, int K, bool out_float, int act, float limit,
                    float slope, hipStream_t stream) {
    const bool gated = (act >= WIDE_SILU && act <= WIDE_CLAMPED) || act == WIDE_CLAMPED_SUMS;
    WideArgs args{(const __bf16*)a, (const __bf16*)w, out, M, N, K, 0, 0, act, limit, slope, 0, 0, 0, 0, 0, nullptr, nullptr};
    const uintptr_t row_bytes = (uintptr_t)N * (out_float ? 4 : 2);
    args.vector_out = ((reinterpret_cast<uintptr_t>(out) | row_bytes) & 15) == 0 ? 1 : 0;
    float time = 0.f;
    if (shape == WIDE_FEW) shape = few_shape_for(M, N, K, gated);             // (-1, refused below, beyond 64 rows)
    else if (shape == WIDE_MANY) shape = wide_shape_for(M, N, K, gated, &time);
    return launch_wide_shape(shape, args, out_float, gated, stream);
}

// The kernel in a given shape (0 .. 16, for tests and measurements) or in the one with the least predicted time (-1: of one sum over
// k; -2: of the forms for up to 64 rows, whose sums are those of `gemm_skinny_kernel`), plain or with gate and silu.
extern "C" int mlr_gemm_wide(const void* a, const void* w, void* out, int M, int N, int K, int out_float,
                             int shape, int gated, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (K <= 0 || (gated && out_float) || !wide_takes(a, w, M, N, K, gated != 0)) return -1;
    return run_wide(shape, a, w, out, M, N, K, out_float != 0, gated ? WIDE_SILU : WIDE_PLAIN, 0.f, 0.f, stream);
}

// Whether up to 64 rows are the forms' with several workgroups a tile, instead of the kernels above and the vendor library.  Measured,
// weights cold, against what takes them otherwise: drawn products (250 of up to 16 rows, 560 of more; the library is at its
// worst with such sizes) and 2300 of mostly round ones, whose losses the exceptions leave out.  us, otherwise and so:
// Up to 16 rows, against `gemm_skinny_kernel`: 8 x 2048 x 5632 10.4 -> 8.7, 1 x 2048 x 8448 14.6 -> 10.4, 16 x 4096 x 12288 26.0 -> 21.5, 8 x 3000
// x 8960 17.3 -> 13.3; round sizes geometric mean 0.80 (0.48 to 1.04).  Left out: below these inner sizes and where a strip of 16 columns a
// compute unit comes out even (up to 1.15); k of 8192 and 24576 over many columns (1 x 4096 x 8192 14.8, 18.4), 12288 and 20480 over more
// than 4096 (8 x 7168 x 12288 35.4, 43.4): as with the narrow tiles; up to 4 rows of more than 3072 columns (1.00 to 1.06).
// From 17 rows on: 64 x 4096 x 12288 33.1 -> 27.0, 48 x 5120 x 25600 89.8 -> 71.4, 32 x 2048 x 5632 12.4 -> 9.2, 64 x 4096 x 4096 13.9 -> 12.3,
// 20 x 3000 x 8960 19.4 -> 15.1; round sizes 0.79 (0.45 to 1.07), of 8208 to 16384 rows of weight 0.94 (0.79 to 1.09).  Left out: below these
// inner sizes and beyond these rows of weight (up to 1.4), of more than 8192 whole 512s of k (64 x 12288 x 16384 86.0, 106.8; 48 x 16384 x 16384
// 101.2, 122.4), k in whole 8192s as above (20 x 4096 x 8192 16.2, 19.1; 32 x 6144 x 24576 68.8, 77.7), up to 24 rows of short k (20 x 4096
// x 5120 11.4, 12.8), few rows of weight that the library cuts k for (48 x 1024 x 5120 8.1, 8.8).
static bool split_wins(int M, int N, int K) {
    if (M <= 0 || M > 64) return false;
    if (M <= 16) {
        const int units = compute_units() > 0 ? compute_units() : 256, strips = (N + 15) / 16;
        if (N > 2560 && K % 8192 == 0 && K % 16384 != 0) return false;
        if (N > 4096 && K > 8192 && K % 4096 == 0 && K % 16384 != 0) return false;
        if (N > 3072 && M <= 4 && K > 6144 && K < 14336) return false;
        return N <= 8192 && (K >= 5120 || (K >= 3584 && !(4 * strips > 3 * units && strips <= units)));
    }
    if (K >= 14336) {
        if (N > 16384 || (M > 32 && N > 11264 && N <= 12800)) return false;
        if (N > 8192 && K >= 15360 && (N > 11264 || K % 512 == 0)) return false;
        return K % 8192 != 0 || (N <= 6144 && (M > 32 || N <= 4096 || K % 16384 == 0));
    }
    if (K >= 9216) return N <= (M <= 32 && K % 4096 == 0 ? 6144 : 8192);
    if (K % 8192 == 0 && N > (M <= 32 ? 3072 : 4096)) return false;
    if (M <= 24 && (N > 3072 ? K <= 7168 : N > 2048 && K < 5120)) return false;
    if (M > 32 && N <= 1024 && K <= 6144 && K % 512 == 0) return false;
    if (K >= 6144) return N <= 6144;
    if (K >= 4224) return N <= 4096;
    if (K >= 3136) return N <= (M > 32 ? 4096 : 2048);
    return K >= 2560 && M > 32 && N > 1024 && N <= 2048;
}
extern "C" int mlr_gemm_split_wins(int M, int N, int K) {
    return N > 0 && K > 0 && wide_takes(nullptr, nullptr, M, N, K, false) && split_wins(M, N, K) ? 1 : 0;
}

// The product of up to 64 rows with several workgroups a tile, the bits of the other kernels of few rows; `partial`: `floats` floats on 16
// bytes, `arrivals`: `counters` zeros, which are zero again behind it; one launch at a time may use them.  shape: 0 .. 9, or -1 for
// the form with the least predicted time.  -1: sizes or room that it does not take, nothing was launched.
extern "C" int mlr_gemm_split(const void* a, const void* w, void* out, int M, int N, int K, float* partial, long floats, int32_t* arrivals,
                              int counters, int shape, hipStream_t stream) {
    if (M <= 0 || M > 64 || N <= 0 || K <= 0 || partial == nullptr || arrivals == nullptr || (reinterpret_cast<uintptr_t>(partial) & 15) != 0 ||
        !wide_takes(a, w, M, N, K, false)) return -1;
    WideArgs args{(const __bf16*)a, (const __bf16*)w, out, M, N, K, 0, 0, WIDE_PLAIN, 0.f, 0.f, 0, 0, 0, 0, 0, partial, arrivals};
    args.vector_out = ((reinterpret_cast<uintptr_t>(out) | (uintptr_t)N * 2) & 15) == 0 ? 1 : 0;
    return launch_split_shape(shape < 0 ? split_shape_for(M, N, K) : shape, args, floats, counters, stream);
}

// out[m][h] = a[m][h] . w[h]^T of many rows: out and a with rows of `ldo` and `lda` elements, heads `out_head` and `a_head` apart,
// w [heads, N, K].  128 x 64 tiles of two blocks of LDS, three workgroups on a compute unit: the inner sizes are 128 to 512, two to
// eight blocks, and what a tile waits for another one hides.  Against tiles of 64 x 64 staged through registers (`mlr_grouped_gemm`,
// same sums, same bits): 1777 rows of 16 heads, 512 x 128 21.6 -> 11.9 us, 128 x 512 17.1 -> 9.0 (36 MB each: 8 us as a copy);
// 2048 of 32, 51.8 -> 29.4 and 39.8 -> 26.2; 333 of 16, 8.3 -> 7.9 and 9.1 -> 7.6.  Other tiles, at 1777 rows: 64 x 64 12.7 and 9.4,
// 128 x 128 11.2 and 9.5, with four blocks of LDS, one on a unit, 15.9 and 8.8, 256 x 128 12.5 and 11.5.
// -3: not this kernel's (up to 64 rows, operands that it does not take), nothing was launched.
extern "C" int mlr_gemm_heads(const void* a, long lda, long a_head, const void* w, void* out, long ldo, long out_head, int M, int N,
                              int K, int heads, hipStream_t stream) {
    using S = WideShape<4, 2, 2, 2, 2>;
    if (M <= 64 || N <= 0 || heads <= 0 || K <= 0 || lda < 0 || a_head < 0 || ldo < 0 || out_head < 0 || lda % 8 != 0 || a_head % 8 != 0 ||
        !wide_takes(a, w, M, N, K, false) || (unsigned long long)M * lda >= (1ull << 31) ||
        (unsigned long long)(a_head | ldo | out_head) >= (1ull << 31))
        return -3;
    const int tiles_m = (M + S::BM - 1) / S::BM, tiles_n = (N + S::BN - 1) / S::BN;
    if ((long long)tiles_m * tiles_n * heads > 0x7fffffffLL / 8) return -3;
    const int vector_out = (reinterpret_cast<uintptr_t>(out) & 15) == 0 && ldo % 8 == 0 && out_head % 8 == 0 ? 1 : 0;
    const WideArgs args{(const __bf16*)a, (const __bf16*)w, out, M, N, K, tiles_m, tiles_n, WIDE_PLAIN, 0.f, 0.f, vector_out,
                        (int)lda, (int)ldo, (int)a_head, (int)out_head, nullptr, nullptr};
    auto* kernel = gemm_wide_kernel<4, 2, 2, 2, 2, false, false, true>;
    static const hipError_t allowed = hipFuncSetAttribute(
        reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)S::lds_bytes);
    if (allowed != hipSuccess) return (int)allowed;
    kernel<<<dim3(tiles_m * tiles_n * heads), 64 * S::WAVES, S::lds_bytes, stream>>>(args);
    return (int)hipGetLastError();
}

// Whether 17 rows and more are this kernel's beside the vendor library (act: WIDE_*): up to 64 rows as `few_wins` says.  Beyond, the
// library has the faster way
//   - on large products: of row counts whose plan it times (multiples of 64: the fastest of up to 32) from 40 GFLOP on -- up to 30 this
//     kernel takes 0.88 of its time, to 60 1.00, to 120 1.06, beyond 1.11 --, of others from 60 on where this kernel's tiles do not come out
//     evenly, below a predicted 1.3 PFLOP/s (it is 0.84, 0.94, 0.99 and 1.02 of the library's there; 1533 x 5120 x 25600 355 us for 518);
//   - on few outputs of a long k, which it cuts (128 x 792 x 11776: 21 us for 38);
//   - on weights of more than 45000 rows while the rows are few (97 x 48000 x 3000: 0.9 of this kernel's time).
// An activation makes no difference: in the epilogue it takes what its own launch does (1.4 us and 1.0 us a million outputs beside 2.3
// and 0.88: an exponential and a division an output; 2048 x 2 * 12288 x 4096: 26 and 24 us).
// Measured on 1840 products of 65 to 2048 rows (inner sizes drawn from 512 to 12000 and 512 to 60000 rows of weight, and the Qwen3
// layers at 20 row counts), against the library and the activation's launch, geometric mean: drawn sizes 0.82 plain and 0.84 gated,
// where the better of both would be 0.81 and 0.82; the Qwen3 layers 0.91 and 1.00 (0.89 and 0.98); of all that this takes 0.38 to 1.32.
// (A prediction of the library's time from its bytes, flops and k, within 16 %, chose no better.)
// one_order: the sums must not turn on which plan the library's timing picks: timed row counts are judged as the others; and up to 64
// rows the question is the tiles of one sum over k, as the library adds, up to 16384 rows of weight: 0.39 to 0.95 of the library's time and the
// activation's launch at the sizes below it (105 products from 5632 rows of weight and k from 1024 to 4096 on, weights cold, but 1.00 for
// 64 x 9216 x 3072: 48 x 8192 x 2048 13.8 -> 9.8 us, 48 x 5632 x 2048 13.2 -> 9.3, 24 x 12288 x 4096 26.1 -> 21.8), 0.82 to 1.16 beyond.
extern "C" int mlr_gemm_wide_wins(int M, int N, int K, int act, int one_order) {
    const bool gated = act >= WIDE_SILU && act <= WIDE_CLAMPED;
    if (M <= 16 || N <= 0 || K <= 0 || !wide_takes(nullptr, nullptr, M, N, K, gated)) return 0;
    const long long weight = (long long)N * (gated ? 2 : 1);
    if (M <= 64) return (one_order ? weight <= 16384 : few_wins(M, N, K, gated)) ? 1 : 0;
    if ((K > 8192 && M * weight < (1 << 17)) || (M <= 128 && weight > 45000)) return 0;
    const float gflop = 2e-9f * (float)M * (float)weight * (float)K;
    if (M % 64 == 0 && !one_order) return gflop < 40.f ? 1 : 0;
    float time = 0.f;
    wide_shape_for(M, N, K, gated, &time);
    return gflop < 60.f || time <= gflop / 1.3f ? 1 : 0;
}

template <int WM, int WN, int TM, int TN, int NS>
static int launch_qkv(QkvArgs& args, hipStream_t stream) {
    using S = WideShape<WM, WN, TM, TN, NS>;
    using Q = QkvTile<S>;
    static_assert(Q::lds_bytes <= 160 * 1024, "the tile and its rows' places must fit the LDS");
    static_assert(S::BM <= 64 * S::WAVES && S::BM * Q::HEADS * 8 % (64 * S::WAVES) == 0, "a thread a row, whole passes");
    args.tiles_m = (args.M + S::BM - 1) / S::BM;
    args.tiles_n = (args.N + S::BN - 1) / S::BN;
    if ((long long)args.tiles_m * args.tiles_n > 0x7fffffffLL / 8) return -2;
    auto* kernel = gemm_wide_kernel<WM, WN, TM, TN, NS, false, false, false, false, false, true>;
    static const hipError_t allowed = hipFuncSetAttribute(
        reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)Q::lds_bytes);
    if (allowed != hipSuccess) return (int)allowed;
    kernel<<<dim3(args.tiles_m * args.tiles_n), 64 * S::WAVES, Q::lds_bytes, stream>>>(args);
    return (int)hipGetLastError();
}

// The tiles that hold whole heads: the one with the least predicted time, the heads' epilogue with it (3 us a tile of 256 x 128).
static int qkv_shape_for(int M, int N, int K, float* time) {
    const int units = compute_units() > 0 ? compute_units() : 256;
    int best = -1;
    for (const int s : {4, 5, 7, 9}) {
        const WideCost& c = WIDE_COSTS[s];
        const long long tiles = (long long)((M + c.bm - 1) / c.bm) * ((N + c.bn - 1) / c.bn);
        const float us = wide_time(s, M, N, K, false) + 3.f / (256 * 128) * (float)((tiles + units - 1) / units * c.bm * c.bn);
        if (best < 0 || us < *time) {
            best = s;
            *time = us;
        }
    }
    return best;
}

// Whether `mlr_gemm_qkv` is the way for a product of these sizes that is this kernel's anyway: the tile of whole heads with its
// epilogue takes no longer than the best tile and the other launch, 3 us and 0.6 a million outputs.  Measured (product + launch, one
// launch): 2048 x 4096 x 1024 28.0, 22.2 us; 1024 x 4096 x 1024 19.7, 13.4; 333 x 6144 x 4096 38.9, 36.2; 700 x 6144 x 4096 50.4, 45.8;
// 333 x 10240 x 5120 56.8, 52.5.  Not where narrower tiles win by more: 256 x 6144 x 4096 32.8, 39.7; 160 x 4096 x 1024 11, 11.
extern "C" int mlr_gemm_qkv_wins(int M, int q_heads, int kv_heads, int K) {
    const int N = (q_heads + 2 * kv_heads) * QKV_HEAD;
    if (M <= 64 || q_heads <= 0 || kv_heads <= 0 || K <= 0 || !wide_takes(nullptr, nullptr, M, N, K, false)) return 0;
    float time = 0.f, any = 0.f;
    qkv_shape_for(M, N, K, &time);
    wide_shape_for(M, N, K, false, &any);
    return time <= any + 3.f + 0.6e-6f * (float)M * (float)N ? 1 : 0;
}

// attention's q, k and v = a . w^T, w [(q_heads + 2 kv_heads) * 128, K], of more than 64 rows, with the heads' norms (weights null: none),
// the rotation of whole heads in split-half pairs by `rope` [positions][128] and the writes of keys and values into their pages:
// the bits of `mlr_gemm_wide` followed by `mlr_qk_norm_rope_kv`.  shape: 4, 5, 7, 9, or -1 for the one with the least predicted time.
// Returns -1 for sizes and operands that it does not take.
extern "C" int mlr_gemm_qkv(const void* a, const void* w, int M, int K, void* q_out, void* k_pages, void* v_pages,
                            const int32_t* block_table, int max_blocks, const int32_t* slots, const int32_t* positions,
                            const float* q_norm_w, const float* k_norm_w, float eps, const float* rope, int q_heads, int kv_heads,
                            int page_size, int write_cache, int shape, hipStream_t stream) {
    if (M <= 0) return 0;
    const uintptr_t starts = reinterpret_cast<uintptr_t>(q_out) | reinterpret_cast<uintptr_t>(k_pages) | reinterpret_cast<uintptr_t>(v_pages) |
                             reinterpret_cast<uintptr_t>(q_norm_w) | reinterpret_cast<uintptr_t>(k_norm_w) | reinterpret_cast<uintptr_t>(rope);
    if (q_heads <= 0 || kv_heads <= 0 || page_size <= 0 || max_blocks <= 0 || rope == nullptr || (q_norm_w == nullptr) != (k_norm_w == nullptr) ||
        (starts & 15) != 0 || (page_size % 8 != 0) || K <= 0)
        return -1;
    const int N = (q_heads + 2 * kv_heads) * QKV_HEAD;
    if (!wide_takes(a, w, M, N, K, false)) return -1;
    QkvArgs args{};
    args.a = (const __bf16*)a;
    args.w = (const __bf16*)w;
    args.M = M;
    args.N = N;
    args.K = K;
    args.q_out = (__bf16*)q_out;
    args.k_pages = (__bf16*)k_pages;
    args.v_pages = (__bf16*)v_pages;
    args.block_table = block_table;
    args.slots = slots;
    args.positions = positions;
    args.q_norm_w = q_norm_w;
    args.k_norm_w = k_norm_w;
    args.rope = rope;
    args.eps = eps;
    args.max_blocks = max_blocks;
    args.q_heads = q_heads;
    args.kv_heads = kv_heads;
    args.page_size = page_size;
    args.write_cache = write_cache;
    float time = 0.f;
    switch (shape < 0 ? qkv_shape_for(M, N, K, &time) : shape) {
        case 4: return launch_qkv<2, 4, 4, 2, 4>(args, stream);
        case 5: return launch_qkv<4, 2, 3, 4, 3>(args, stream);
        case 7: return launch_qkv<4, 2, 4, 4, 3>(args, stream);
        case 9: return launch_qkv<2, 4, 8, 4, 2>(args, stream);
        default: return -1;
    }
}

// out[M, N] = act of the products, act one of WIDE_SILU_ROUNDED .. (gated: w is [2N, K] = [gate; up]; limit and slope are
// WIDE_CLAMPED's): the bits of the product followed by the activation's own kernel.  one_order: up to 64 rows, too, one sum over k.
extern "C" int mlr_gemm_activated(const void* a, const void* w, void* out, int M, int N, int K, int act, float limit, float slope,
                                  int one_order, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (K <= 0 || act < WIDE_SILU_ROUNDED || act > WIDE_GELU_ERF || (act == WIDE_CLAMPED && !(limit > 0.f))) return -1;
    if (!wide_takes(a, w, M, N, K, act <= WIDE_CLAMPED)) return -2;
    return run_wide(M <= 64 && !one_order ? WIDE_FEW : WIDE_MANY, a, w, out, M, N, K, false, act, limit, slope, stream);
}

template <int WM, int WN, int TM, int TN>
static int launch(const void* a, const void* w, void* out, int M, int N, int K, int out_float,
                  hipStream_t stream) {
    constexpr int BM = WM * TM * 16, BN = WN * TN * 16;
    dim3 grid((N + BN - 1) / BN, (M + BM - 1) / BM);
    if (grid.y > 65535) return -2;
    if (out_float)
        gemm_bf16_kernel<WM, WN, TM, TN, true><<<grid, WM * WN * 64, 0, stream>>>(
            (const __bf16*)a, (const __bf16*)w, out, M, N, K);
    else
        gemm_bf16_kernel<WM, WN, TM, TN, false><<<grid, WM * WN * 64, 0, stream>>>(
            (const __bf16*)a, (const __bf16*)w, out, M, N, K);
    return (int)hipGetLastError();
}

extern "C" int mlr_gemm(const void* a, const void* w, void* out, int M, int N, int K, int out_float,
                        hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (K <= 0) return -1;
    if (M <= 16) return launch_skinny<1, false>(a, w, out, M, N, K, out_float, stream);
    // 17..64 rows against many columns (the output projection): tiles through LDS re-read the rows less often
    if (M <= 64 && N >= 16384) return launch<2, 2, 2, 2>(a, w, out, M, N, K, out_float, stream);
    if (M <= 32) return launch_skinny<2, false>(a, w, out, M, N, K, out_float, stream);
    if (M <= 64) return launch_skinny<4, false>(a, w, out, M, N, K, out_float, stream);
    if (wide_takes(a, w, M, N, K, false)) return run_wide(WIDE_MANY, a, w, out, M, N, K, out_float != 0, WIDE_PLAIN, 0.f, 0.f, stream);
    if (M <= 128) return launch<2, 2, 2, 2>(a, w, out, M, N, K, out_float, stream);  // 64 x 64
    return launch<2, 2, 4, 4>(a, w, out, M, N, K, out_float, stream);                // 128 x 128
}

// out[M, N] = silu(a . w[0:N]^T) * (a . w[N:2N]^T) (w is [2N, K]: gate rows, then up rows): up to 64 rows on
// the weight-streaming kernels, more on the wide kernel when K is a multiple of 64.  Returns 1 when no kernel
// here takes the sizes: the caller then runs the projection and the activation separately.
extern "C" int mlr_gemm_gated_silu(const void* a, const void* w, void* out, int M, int N, int K,
                                   hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (K <= 0) return -1;
    if (M <= 16) return launch_skinny<1, true>(a, w, out, M, N, K, 0, stream);
    if (M <= 32) return launch_skinny<2, true>(a, w, out, M, N, K, 0, stream);
    if (M <= 64) return launch_skinny<4, true>(a, w, out, M, N, K, 0, stream);
    if (wide_takes(a, w, M, N, K, true)) return run_wide(WIDE_MANY, a, w, out, M, N, K, false, WIDE_SILU, 0.f, 0.f, stream);
    return 1;
}

// out[M, N] = g sigmoid(slope g) (u + 1) with g = min(a . w[0:N]^T, limit), u = clamp(a . w[N:2N]^T, -limit, limit):
// the clamped gate as the epilogue of the weight-streaming kernels, up to 64 rows.  Returns 1 for more rows.
extern "C" int mlr_gemm_gated_clamped(const void* a, const void* w, void* out, int M, int N, int K, float limit,
                                      float slope, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (K <= 0 || !(limit > 0.f)) return -1;
    // (8 x 2 * 5632 x 2048 14.8 -> 11.7 us; a Taletar decoding step of 8 requests 617 -> 607)
    if (M <= 64 && wide_takes(a, w, M, N, K, true) && (M <= 16 ? narrow_wins(M, N, K, true) : few_wins(M, N, K, true)))
        return run_wide(WIDE_FEW, a, w, out, M, N, K, false, WIDE_CLAMPED_SUMS, limit, slope, stream);
    SkinnyEpilogue epi{};
    epi.glu_limit = limit;
    epi.glu_slope = slope;
    if (M <= 16) return launch_skinny<1, true>(a, w, out, M, N, K, 0, stream, epi);
    if (M <= 32) return launch_skinny<2, true>(a, w, out, M, N, K, 0, stream, epi);
    if (M <= 64) return launch_skinny<4, true>(a, w, out, M, N, K, 0, stream, epi);
    return 1;
}

// out[M, N] = act(a . w[0:N]^T) * (a . w[N:2N]^T), act 1 the tanh form of gelu, 0.5 g (1 + tanh(sqrt(2 / pi) (g + 0.044715
// g^3))), or 2 relu: the gate as the epilogue of the weight-streaming kernels, up to 64 rows.  Returns 1 for more rows.
extern "C" int mlr_gemm_gated_act(const void* a, const void* w, void* out, int M, int N, int K, int act, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (K <= 0 || act < 1 || act > 2) return -1;
    SkinnyEpilogue epi{};
    epi.glu_limit = -(float)act;
    if (M <= 16) return launch_skinny<1, true>(a, w, out, M, N, K, 0, stream, epi);
    if (M <= 32) return launch_skinny<2, true>(a, w, out, M, N, K, 0, stream, epi);
    if (M <= 64) return launch_skinny<4, true>(a, w, out, M, N, K, 0, stream, epi);
    return 1;
}

// out[M, N] = act(a . w^T), act 1 relu(x)^2 or 2 the exact gelu, as the epilogue of the weight-streaming kernels, up to
// 64 rows.  Returns 1 for more rows.
extern "C" int mlr_gemm_act(const void* a, const void* w, void* out, int M, int N, int K, int act, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (K <= 0 || act < 1 || act > 2) return -1;
    SkinnyEpilogue epi{};
    epi.plain_act = act;
    if (M <= 16) return launch_skinny<1, false>(a, w, out, M, N, K, 0, stream, epi);
    if (M <= 32) return launch_skinny<2, false>(a, w, out, M, N, K, 0, stream, epi);
    if (M <= 64) return launch_skinny<4, false>(a, w, out, M, N, K, 0, stream, epi);
    return 1;
}

// The two halves of an RMSNorm handed from one projection to the next, for M <= 16 (see SkinnyEpilogue).
// out = rsqrt(sum_p ss[m][p] / norm_size + eps) * (x . w^T); gated != 0: w is [2N, K] = [gate; up] and
// out = silu(scale * gate) * (scale * up).  x is bf16(h * norm_w) as `mlr_gemm_residual` or the row kernel
// `mlr_rows_prenorm` left it.
extern "C" int mlr_gemm_prenormed(const void* x, const float* ss, int ss_parts, float eps, int norm_size, const void* w,
                                  void* out, int M, int N, int K, int gated, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (M > 16 || K <= 0 || ss_parts <= 0 || norm_size <= 0 || ss == nullptr) return -1;
    SkinnyEpilogue epi{};
    epi.ss = ss;
    epi.ss_parts = ss_parts;
    epi.ss_vec = (ss_parts % 4 == 0 && reinterpret_cast<uintptr_t>(ss) % 16 == 0) ? 1 : 0;
    epi.eps = eps;
    epi.inv_size = 1.0f / (float)norm_size;
    if (gated) return launch_skinny<1, true, EPI_SCALE>(x, w, out, M, N, K, 0, stream, epi);
    return launch_skinny<1, false, EPI_SCALE>(x, w, out, M, N, K, 0, stream, epi);
}

// h[M, N] += a[M, K] . w[N, K]^T in 32-bit, in place.  With next_w != null also x_out[M, N] = bf16(h * next_w)
// and ss_out[M, ceil(N / 16)]: per row and strip of 16 columns the sum of squares of the new h.
extern "C" int mlr_gemm_residual(const void* a, const void* w, float* h, const float* next_w, void* x_out,
                                 float* ss_out, int M, int N, int K, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (M > 16 || K <= 0 || h == nullptr) return -1;
    if (next_w != nullptr && (x_out == nullptr || ss_out == nullptr)) return -2;
    SkinnyEpilogue epi{};
    epi.h = h;
    epi.next_w = next_w;
    epi.x_out = (__bf16*)x_out;
    epi.ss_out = ss_out;
    return launch_skinny<1, false, EPI_RESIDUAL>(a, w, nullptr, M, N, K, 0, stream, epi);
}
#endif
