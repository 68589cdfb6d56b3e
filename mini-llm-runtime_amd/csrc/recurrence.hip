// Mixers with a state of fixed size per request: a short causal convolution over channels, the decays of
// gated linear attention and of Mamba-2, and the linear recurrence both share,
//     S_t = diag(a_t) S_(t-1) + k_t v_t^T,   o_t = S_t^T q_t        (S: N key channels x V value channels),
// run token by token in 32-bit from the state that earlier steps left.  A step brings any mix of prompt
// portions and single tokens; a request's tokens are consecutive rows of the batch (`seg_first`, `seg_count`,
// one entry a request of the step).  The live state of a request is read from `live + slot * stride`, the
// state that the step leads to is written to `stage + slot * stride` (the engine makes it live when every
// layer has run).  Where both are one slab, its rows come in pairs: `slots` names the live row of a pair and the other one, slot ^ 1,
// is written, so that making it live is a matter of which row the next step names (a copy of every state otherwise: 48 requests of
// eight layers of 1 MB, 133 us of a step of 1730).  Every sum is taken in an order that depends on the token's own data only, so a token's
// result does not depend on how its request was cut into steps or on what else the batch holds.
//
// The delta rule (`delta_rule_kernel`) is the same walk with a write that first takes back what the state already
// holds for the token's key:  S <- diag(g_t) S;  u = beta_t (v_t - S^T k_t);  S <- S + k_t u^T;  o_t = S^T q_t.
//
// Long portions (the bfloat16 engine) run the recurrence over pieces of a request side by side, in three passes:
// every piece from a zero state, leaving its last state L_c and the product A_c of its decays; then, piece after
// piece, the state each piece starts from, S_(c+1) = diag(A_c) S_c + L_c (element by element, from the live
// state); then every piece again from its S_c, writing the outputs.  Twice the arithmetic, as many workgroups as
// pieces; the result differs from the token-by-token order by 32-bit rounding only.
#include "common.h"

__device__ __forceinline__ float softplus_f(float x) { return fmaxf(x, 0.f) + log1pf(expf(-fabsf(x))); }
__device__ __forceinline__ float silu_f(float x) { return x / (1.0f + expf(-x)); }
__device__ __forceinline__ float sigmoid_f(float x) { return 1.0f / (1.0f + expf(-x)); }

// ---- short causal convolution -----------------------------------------------------------------------
// out[r, c] = act(b[c] + sum_j w[c, j] * in(r, taps - 1 - j)) with in(r, d) the channel's input d tokens before
// row r: a row of this step when the request brought it, else the request's state, which holds its last
// taps - 1 inputs, oldest first, as [taps - 1][C] floats (zeros at a sequence's start).  The last row of a
// request in the step writes the state that follows.  One thread per (row, channel).
struct ConvArgs {
    const elem_t* x; long x_stride;
    const float* w; const float* b;
    elem_t* out; long out_stride;
    const float* live; float* stage; long state_stride;
    const int32_t* slots; const int32_t* positions;
    int rows, channels, taps, silu, write_state;
    int pair;                                  // a slot's written row is slot ^ pair
};

#define CONV_MAX_TAPS 8

__global__ __launch_bounds__(256) void causal_conv_kernel(ConvArgs a) {
    const int r = blockIdx.x;
    const int c = blockIdx.y * 256 + threadIdx.x;
    const int slot = a.slots[r], pos = a.positions[r];
    const int before = a.taps - 1;
    int have = 0;                              // rows right before r that are this request's previous tokens
    while (have < before && r - have - 1 >= 0 && a.slots[r - have - 1] == slot && a.positions[r - have - 1] == pos - have - 1) ++have;
    const bool last = r + 1 >= a.rows || a.slots[r + 1] != slot || a.positions[r + 1] != pos + 1;
    if (c >= a.channels) return;
    float in[CONV_MAX_TAPS];                   // in[d]: the input d tokens back
#pragma unroll
    for (int d = 0; d < CONV_MAX_TAPS; ++d) {
        if (d > before) { in[d] = 0.f; continue; }
        if (d <= have) in[d] = to_float(a.x[(size_t)(r - d) * a.x_stride + c]);
        else in[d] = a.live[(size_t)slot * a.state_stride + (size_t)(before - d + have) * a.channels + c];
    }
    float acc = a.b ? a.b[c] : 0.f;
#pragma unroll
    for (int d = CONV_MAX_TAPS - 1; d >= 0; --d) {         // oldest input first; tap j = taps - 1 - d
        if (d <= before) acc += a.w[(size_t)c * a.taps + (before - d)] * in[d];
    }
    if (a.silu) acc = acc / (1.0f + expf(-acc));
    a.out[(size_t)r * a.out_stride + c] = from_float<elem_t>(acc);
    if (last && a.write_state) {
#pragma unroll
        for (int d = 0; d < CONV_MAX_TAPS - 1; ++d) {
            if (d < before) a.stage[(size_t)(slot ^ a.pair) * a.state_stride + (size_t)(before - 1 - d) * a.channels + c] = in[d];
        }
    }
}

#if MLR_BF16
// Many values: eight channels a thread (16-byte accesses) and CONV_ROWS rows, for which its weights stay in registers.  Bound by
// memory; one value a thread took 62 us for 2048 rows of 4096 channels, this 22.
#define CONV_ROWS 4
template <int TAPS>
__global__ __launch_bounds__(256) void causal_conv_rows_kernel(ConvArgs a) {
    const int c = (blockIdx.y * 256 + threadIdx.x) * 8;
    if (c >= a.channels) return;
    float w[8 * TAPS], b[8];
#pragma unroll
    for (int e = 0; e < 8 * TAPS; e += 4) *reinterpret_cast<float4*>(w + e) = *reinterpret_cast<const float4*>(a.w + (size_t)c * TAPS + e);
#pragma unroll
    for (int e = 0; e < 8; ++e) b[e] = a.b ? a.b[c + e] : 0.f;
    constexpr int before = TAPS - 1;
    for (int r = blockIdx.x * CONV_ROWS; r < min(a.rows, ((int)blockIdx.x + 1) * CONV_ROWS); ++r) {
        const int slot = a.slots[r], pos = a.positions[r];
        int have = 0;
        while (have < before && r - have - 1 >= 0 && a.slots[r - have - 1] == slot && a.positions[r - have - 1] == pos - have - 1) ++have;
        const bool last = r + 1 >= a.rows || a.slots[r + 1] != slot || a.positions[r + 1] != pos + 1;
        float in[TAPS][8];
#pragma unroll
        for (int d = 0; d < TAPS; ++d) {
            if (d <= have) {
                load_vec(a.x + (size_t)(r - d) * a.x_stride + c, in[d]);
            } else {
                const float* from = a.live + (size_t)slot * a.state_stride + (size_t)(before - d + have) * a.channels + c;
#pragma unroll
                for (int e = 0; e < 8; ++e) in[d][e] = from[e];
            }
        }
        float acc[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            acc[e] = b[e];
#pragma unroll
            for (int d = before; d >= 0; --d) acc[e] += w[e * TAPS + before - d] * in[d][e];
            if (a.silu) acc[e] = acc[e] / (1.0f + expf(-acc[e]));
        }
        store_vec(a.out + (size_t)r * a.out_stride + c, acc);
        if (last && a.write_state) {
#pragma unroll
            for (int d = 0; d < before; ++d)
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    a.stage[(size_t)(slot ^ a.pair) * a.state_stride + (size_t)(before - 1 - d) * a.channels + c + e] = in[d][e];
        }
    }
}
#endif

// ---- decays ---------------------------------------------------------------------------------------------
// Gated linear attention: the logarithm of alpha = sigmoid(z + b)^(1 / tau), that is -softplus(-(z + b)) / tau.
__global__ void gla_log_decay_kernel(const elem_t* __restrict__ z, const float* __restrict__ bias, float* __restrict__ out,
                                     size_t rows, int width, float inv_tau) {
    const size_t total = rows * width;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
        const float x = to_float(z[i]) + (bias ? bias[i % width] : 0.f);
        out[i] = -softplus_f(-x) * inv_tau;
    }
}

// Mamba-2: the step size dt = softplus(raw + dt_bias[h]) (no clamp) and the log decay -exp(A_log[h]) * dt.
__global__ void mamba_step_kernel(const elem_t* __restrict__ raw, long raw_stride, const float* __restrict__ dt_bias,
                                  const float* __restrict__ a_log, float* __restrict__ dt, float* __restrict__ log_decay,
                                  size_t rows, int heads) {
    const size_t total = rows * heads;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
        const size_t r = i / heads;
        const int h = (int)(i % heads);
        const float step = softplus_f(to_float(raw[r * raw_stride + h]) + dt_bias[h]);
        dt[i] = step;
        log_decay[i] = -expf(a_log[h]) * step;
    }
}

// ---- the recurrence --------------------------------------------------------------------------------------
struct ScanArgs {
    const elem_t* q; long q_stride;            // q[r * q_stride + (head / heads_per_group) * N + i]
    const elem_t* k; long k_stride;
    const elem_t* v; long v_stride;            // v[r * v_stride + head * V + j]
    const float* log_decay; long decay_stride; // per channel: [r * stride + head * N + i]; else [r * stride + head]
    const float* v_scale; long v_scale_stride; // factor on v, [r * stride + head], or null
    const float* skip;                         // out += skip[head] * v (unscaled), or null
    float* out;                                // [rows, heads * V]
    const float* live; float* stage; long state_stride;     // a request's S as [heads][N][V]
    const int32_t* seg_first; const int32_t* seg_count; const int32_t* slots;
    int heads, heads_per_group, N, V, decay_per_channel, write_state;
    float q_scale;
    int silu;                                  // q, k and v pass silu as they are read (before the factors)
    // q and k are turned as they are read (null: not): the first rot_dim channels of a head by the token's position, in
    // pairs (i, i + rot_dim / 2), rope [positions][rot_dim] holding cosines, then sines; 32-bit
    const float* rope; const int32_t* positions; int rot_dim;
    float* piece_state;                        // [pieces][heads][N][V]: L_c after the first pass, S_c after the second
    float* piece_decay;                        // [pieces][heads][N]: A_c
    int pair;                                  // a slot's written row is slot ^ pair
};

#define SCAN_COLS 64
#define SCAN_PARTS 4

// One workgroup per (request of the step, head, 64 value channels): wavefront p holds rows [p NR, (p + 1) NR)
// of S for its 64 columns in registers, a lane a column.  Tokens are staged TILE at a time through LDS
// (decays exponentiated, q scaled, v scaled); after a tile the four partial sums of o are added in the order
// of the parts.
// MODE 0: a request's rows of the step from its live state to the staged one.  MODE 1: a piece from a zero state,
// no outputs; leaves L_c and A_c.  MODE 2: a piece from S_c, outputs only.  (In modes 1 and 2 `seg_first` and
// `seg_count` name the pieces.)
template <int NR, int TILE, int MODE>
__global__ __launch_bounds__(256) void linear_recurrence_kernel(ScanArgs a) {
    constexpr int NPAD = NR * SCAN_PARTS;
    extern __shared__ __attribute__((aligned(16))) float lds[];
    float* a_lds = lds;                                   // [TILE][NPAD]
    float* k_lds = a_lds + TILE * NPAD;
    float* q_lds = k_lds + TILE * NPAD;
    float* v_lds = q_lds + TILE * NPAD;                   // [TILE][COLS]
    float* o_lds = v_lds + TILE * SCAN_COLS;              // [PARTS][TILE][COLS]
    const int seg = blockIdx.x, head = blockIdx.y, col0 = blockIdx.z * SCAN_COLS;
    const int r0 = a.seg_first[seg], n = a.seg_count[seg];
    const int slot = a.slots[r0];
    const int j = threadIdx.x & 63, part = threadIdx.x >> 6;
    const int col = col0 + j;
    const int N = a.N, V = a.V;
    const int qk_head = head / a.heads_per_group;
    const size_t state_at = (size_t)slot * a.state_stride + (size_t)head * N * V, stage_at = (size_t)(slot ^ a.pair) * a.state_stride + (size_t)head * N * V;
    const size_t piece_at = ((size_t)seg * a.heads + head) * N * V;
    float S[NR], A[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        const int i = part * NR + r;
        const bool in = i < N && col < V;
        S[r] = MODE == 1 || !in ? 0.f : MODE == 0 ? a.live[state_at + (size_t)i * V + col] : a.piece_state[piece_at + (size_t)i * V + col];
        A[r] = 1.f;
    }
    for (int t0 = 0; t0 < n; t0 += TILE) {
        const int nt = min(TILE, n - t0);
        __syncthreads();                                  // the tile before is read and written out
        for (int idx = threadIdx.x; idx < nt * NPAD; idx += 256) {
            const int t = idx / NPAD, i = idx % NPAD;
            const size_t row = (size_t)(r0 + t0 + t);
            float da = 0.f, dk = 0.f, dq = 0.f;
            if (i < N) {
                da = expf(a.log_decay[row * a.decay_stride + (a.decay_per_channel ? head * N + i : head)]);
                dk = to_float(a.k[row * a.k_stride + qk_head * N + i]);
                dq = to_float(a.q[row * a.q_stride + qk_head * N + i]);
                if (a.silu) { dk = silu_f(dk); dq = silu_f(dq); }
                if (i < a.rot_dim) {
                    const int half = a.rot_dim >> 1, j = i < half ? i : i - half, other = i < half ? i + half : i - half;
                    const float* cs = a.rope + (size_t)a.positions[row] * a.rot_dim;
                    float ok = to_float(a.k[row * a.k_stride + qk_head * N + other]);
                    float oq = to_float(a.q[row * a.q_stride + qk_head * N + other]);
                    if (a.silu) { ok = silu_f(ok); oq = silu_f(oq); }
                    const float c = cs[j], s = cs[half + j];
                    dk = i < half ? turn_x(dk, ok, c, s) : turn_y(ok, dk, c, s);
                    dq = i < half ? turn_x(dq, oq, c, s) : turn_y(oq, dq, c, s);
                }
                dq *= a.q_scale;
            }
            a_lds[idx] = da; k_lds[idx] = dk; q_lds[idx] = dq;
        }
        for (int idx = threadIdx.x; idx < nt * SCAN_COLS; idx += 256) {
            const int t = idx / SCAN_COLS, c = col0 + idx % SCAN_COLS;
            const size_t row = (size_t)(r0 + t0 + t);
            float x = 0.f;
            if (c < V) {
                x = to_float(a.v[row * a.v_stride + head * V + c]);
                if (a.silu) x = silu_f(x);
                if (a.v_scale) x *= a.v_scale[row * a.v_scale_stride + head];
            }
            v_lds[idx] = x;
        }
        __syncthreads();
        for (int t = 0; t < nt; ++t) {
            const float x = v_lds[t * SCAN_COLS + j];
            const float* at = a_lds + t * NPAD + part * NR;
            const float* kt = k_lds + t * NPAD + part * NR;
            const float* qt = q_lds + t * NPAD + part * NR;
            float o = 0.f;
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                S[r] = at[r] * S[r] + kt[r] * x;
                if (MODE == 1) A[r] *= at[r];
                else o += qt[r] * S[r];
            }
            if (MODE != 1) o_lds[(part * TILE + t) * SCAN_COLS + j] = o;
        }
        if (MODE == 1) continue;
        __syncthreads();
        for (int idx = threadIdx.x; idx < nt * SCAN_COLS; idx += 256) {
            const int t = idx / SCAN_COLS, c = col0 + idx % SCAN_COLS;
            if (c >= V) continue;
            const size_t row = (size_t)(r0 + t0 + t);
            float o = o_lds[idx];
#pragma unroll
            for (int p = 1; p < SCAN_PARTS; ++p) o += o_lds[p * TILE * SCAN_COLS + idx];
            if (a.skip) {
                const float x = to_float(a.v[row * a.v_stride + head * V + c]);
                o += a.skip[head] * (a.silu ? silu_f(x) : x);
            }
            a.out[row * ((size_t)a.heads * V) + head * V + c] = o;
        }
    }
    if (MODE == 0 && a.write_state && col < V) {
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            const int i = part * NR + r;
            if (i < N) a.stage[stage_at + (size_t)i * V + col] = S[r];
        }
    }
    if (MODE == 1) {
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            const int i = part * NR + r;
            if (i < N && col < V) a.piece_state[piece_at + (size_t)i * V + col] = S[r];
            if (i < N && col == 0) a.piece_decay[((size_t)seg * a.heads + head) * N + i] = A[r];
        }
    }
}

// The second pass: one thread per element (head, i, j) of the state walks the pieces in their order.  A piece
// whose request differs from the piece before starts from that request's live state; where a request's pieces
// end its state is staged.  piece_state[c] holds L_c on entry and S_c, the state piece c starts from, on exit.
__global__ void piece_states_kernel(ScanArgs a, int pieces) {
    const size_t per = (size_t)a.heads * a.N * a.V;
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= per) return;
    const size_t hi = e / a.V;                 // head * N + i
    float S = 0.f;
    for (int c = 0; c < pieces; ++c) {
        const int slot = a.slots[a.seg_first[c]];
        if (c == 0 || a.slots[a.seg_first[c - 1]] != slot) S = a.live[(size_t)slot * a.state_stride + e];
        const float last = a.piece_state[(size_t)c * per + e];
        a.piece_state[(size_t)c * per + e] = S;
        S = a.piece_decay[(size_t)c * a.heads * a.N + hi] * S + last;
        if (a.write_state && (c + 1 == pieces || a.slots[a.seg_first[c + 1]] != slot)) a.stage[(size_t)(slot ^ a.pair) * a.state_stride + e] = S;
    }
}

// ---- the delta rule ----------------------------------------------------------------------------------------
// Decays of the key channels from a step size per channel: log g = -exp(A_log[head]) * softplus(z + bias), z the
// 32-bit output of a low-rank pair of projections laid out [heads][N].
// A thread stays in its column and takes the rate and the bias once (`stride` is a multiple of the width): 19 us for 2048 rows of
// 2048 channels, 23 where every element divides its place and takes its own rate.  The logarithms bound it.
__global__ __launch_bounds__(256) void channel_log_decay_kernel(const float* __restrict__ z, const float* __restrict__ bias,
                                                                const float* __restrict__ a_log, float* __restrict__ out, size_t total,
                                                                size_t stride, int width, int per_head) {
    const size_t first = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (first >= stride) return;
    const int c = (int)(first % width);
    const float rate = -expf(a_log[c / per_head]), add = bias ? bias[c] : 0.f;
    for (size_t i = first; i < total; i += stride) out[i] = rate * softplus_f(z[i] + add);
}

struct DeltaArgs {
    const elem_t* q; long q_stride;            // q[r * q_stride + (head / heads_per_group) * N + i], as projected
    const elem_t* k; long k_stride;
    const elem_t* v; long v_stride;            // v[r * v_stride + head * V + j]
    const float* log_decay;                    // [rows][heads * N], or with decay_per_head [rows][heads]
    const float* beta_raw; long beta_stride;   // beta = sigmoid(beta_raw[r * stride + head])
    float* out;                                // [rows, heads * V]
    const float* live; float* stage; long state_stride;     // a request's S as [heads][N][V]
    const int32_t* seg_first; const int32_t* seg_count; const int32_t* slots;
    int heads, heads_per_group, N, V, write_state, unit_norm;
    float q_scale, unit_eps;
    int decay_per_head;                        // one decay for all key channels of a head
    int pair;                                  // a slot's written row is slot ^ pair
};

// Where the log decay of (row, head, key channel i) lies.
__device__ __forceinline__ size_t decay_at(const DeltaArgs& a, size_t row, int head, int i) {
    return a.decay_per_head ? row * (size_t)a.heads + head : row * ((size_t)a.heads * a.N) + (size_t)head * a.N + i;
}

#define DELTA_TILE 16

// One wavefront per (request of the step, head, COLS value channels), COLS = 64 / PARTS: lane (part, column) holds
// rows [part NR, (part + 1) NR) of its column of S in registers.  Tokens are staged DELTA_TILE at a time through LDS:
// q and k made unit vectors over the head's N channels (x / sqrt(sum x^2 + unit_eps); q times q_scale), the decays
// exponentiated, beta = sigmoid(raw), k . q of every token.  A token then costs one pass over the lane's rows for
// (g S)^T k and (g S)^T q, an exchange between the parts, and one pass for the write; the read-out after the write is
// o = (g S)^T q + (k . q) u.  Every sum's order follows from the head's sizes alone.
template <int NR, int PARTS, int TILE>
__global__ __launch_bounds__(64) void delta_rule_kernel(DeltaArgs a) {
    constexpr int COLS = 64 / PARTS;
    constexpr int NPAD = NR * PARTS;
    __shared__ __attribute__((aligned(16))) float g_lds[TILE * NPAD];
    __shared__ __attribute__((aligned(16))) float k_lds[TILE * NPAD];
    __shared__ __attribute__((aligned(16))) float q_lds[TILE * NPAD];
    __shared__ float v_lds[TILE * COLS];
    __shared__ float beta_lds[TILE], kq_lds[TILE];
    const int seg = blockIdx.x, head = blockIdx.y, col0 = blockIdx.z * COLS;
    const int r0 = a.seg_first[seg], n = a.seg_count[seg];
    const int slot = a.slots[r0];
    const int lane = threadIdx.x, j = lane % COLS, part = lane / COLS;
    const int col = col0 + j;
    const int N = a.N, V = a.V;
    const int qk_head = head / a.heads_per_group;
    const size_t state_at = (size_t)slot * a.state_stride + (size_t)head * N * V, stage_at = (size_t)(slot ^ a.pair) * a.state_stride + (size_t)head * N * V;
    float S[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        const int i = part * NR + r;
        S[r] = i < N && col < V ? a.live[state_at + (size_t)i * V + col] : 0.f;
    }
    for (int t0 = 0; t0 < n; t0 += TILE) {
        const int nt = min(TILE, n - t0);
        __syncthreads();                                  // the tile before has been read
        for (int t = 0; t < nt; ++t) {
            const size_t row = (size_t)(r0 + t0 + t);
            float qq = 0.f, kk = 0.f;
            for (int i = lane; i < NPAD; i += 64) {
                float dq = 0.f, dk = 0.f, dg = 0.f;
                if (i < N) {
                    dq = to_float(a.q[row * a.q_stride + qk_head * N + i]);
                    dk = to_float(a.k[row * a.k_stride + qk_head * N + i]);
                    dg = expf(a.log_decay[decay_at(a, row, head, i)]);
                }
                qq += dq * dq;
                kk += dk * dk;
                q_lds[t * NPAD + i] = dq; k_lds[t * NPAD + i] = dk; g_lds[t * NPAD + i] = dg;
            }
            float fq = a.q_scale, fk = 1.0f;
            if (a.unit_norm) {
                fq = a.q_scale / sqrtf(wave_sum(qq) + a.unit_eps);
                fk = 1.0f / sqrtf(wave_sum(kk) + a.unit_eps);
            }
            float dot = 0.f;
            for (int i = lane; i < NPAD; i += 64) {      // (each lane returns to the channels it wrote)
                const float dq = q_lds[t * NPAD + i] * fq, dk = k_lds[t * NPAD + i] * fk;
                q_lds[t * NPAD + i] = dq; k_lds[t * NPAD + i] = dk;
                dot += dq * dk;
            }
            dot = wave_sum(dot);
            if (lane == 0) {
                kq_lds[t] = dot;
                beta_lds[t] = sigmoid_f(a.beta_raw[row * a.beta_stride + head]);
            }
        }
        for (int idx = lane; idx < nt * COLS; idx += 64) {
            const int t = idx / COLS, c = col0 + idx % COLS;
            v_lds[idx] = c < V ? to_float(a.v[(size_t)(r0 + t0 + t) * a.v_stride + head * V + c]) : 0.f;
        }
        __syncthreads();
        for (int t = 0; t < nt; ++t) {
            const float* gt = g_lds + t * NPAD + part * NR;
            const float* kt = k_lds + t * NPAD + part * NR;
            const float* qt = q_lds + t * NPAD + part * NR;
            float sk = 0.f, sq = 0.f;
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                S[r] *= gt[r];
                sk += kt[r] * S[r];
                sq += qt[r] * S[r];
            }
            sk = far_sum<COLS>(sk);                       // the parts of a column lie COLS lanes apart
            sq = far_sum<COLS>(sq);
            const float u = beta_lds[t] * (v_lds[t * COLS + j] - sk);
#pragma unroll
            for (int r = 0; r < NR; ++r) S[r] += kt[r] * u;
            if (part == 0 && col < V) a.out[(size_t)(r0 + t0 + t) * ((size_t)a.heads * V) + head * V + col] = sq + kq_lds[t] * u;
        }
    }
    if (a.write_state && col < V) {
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            const int i = part * NR + r;
            if (i < N) a.stage[stage_at + (size_t)i * V + col] = S[r];
        }
    }
}


// ---- the delta rule over chunks of tokens --------------------------------------------------------------------
// A request's rows are cut into chunks of at most DC tokens.  With c_t[i] the sum of a chunk's log decays of key
// channel i up to and including token t, and S0 the state the chunk starts from, the rule's writes u_t obey
//     u_t = beta_t (v_t - S0^T (k_t e^{c_t}) - sum_{s<t} (sum_i k_t[i] k_s[i] e^{c_t[i] - c_s[i]}) u_s),
// a unit lower-triangular system (I + A) U = beta (V - Khat S0) whose inverse T depends on the chunk's keys, decays
// and beta alone.  The first kernel (one workgroup per chunk and head, all side by side) leaves in scratch memory
//     W = T (beta Khat) [DC, N],  Y = T (beta V) [DC, V],  B[t, s] = sum_i q_t[i] k_s[i] e^{c_t[i] - c_s[i]} (s <= t),
//     Qhat[t] = q_t e^{c_t},  Kbar[s] = k_s e^{c_last - c_s},  G = e^{c_last};
// the second (one workgroup per request, head and 16 value channels) walks a request's chunks in
// their order with the state in registers:  U = Y - W S0;  O = Qhat S0 + B U;  S <- diag(G) S0 + Kbar^T U.
// Every exponent is a difference c_t - c_s with s <= t or c_t itself, so nothing overflows however strong a decay
// is.  The result differs from the token-by-token kernel's by 32-bit rounding.
//
// Both kernels multiply with v_mfma_f32_16x16x4_f32 (32-bit products and sums; lane = 16 b + c: A row c, B column c, k-slot
// b; C column c, rows 4 b + i).  Product i of four takes the k {i, 4 + i, 8 + i, 12 + i}: A is four neighbouring k of a row,
// and what a product leaves in C is the next one's B as it lies -- the state, 16 key channels a tile, and U never leave the
// registers but to be added across wavefronts.
#define DELTA_CHUNK 32
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;

struct DeltaChunkArgs {
    DeltaArgs d;
    const int32_t* chunk_first; const int32_t* chunk_count;     // the chunks, a request's one after the other
    float* scratch;                                              // [chunks][heads][delta_chunk_floats(N, V)]
};

// W, Qhat, Kbar [DC x Np], Y [DC x Vp], B [DC x DC], G [Np]; Np, Vp: N and V up to a multiple of 16, zeros there.  All but G lie as
// the scan's wavefronts read them, 16 x 16 elements in one run of 1 KB: block (column / 16, row / 16), in it lane, element as a
// product takes them -- W, Qhat and B: lane = 16 (column % 16 / 4) + row % 16, element = column % 4; Kbar (rows are tokens) and Y:
// lane = 16 (row % 16 / 4) + column % 16, element = row % 4.  (As rows, a load of the scan touched 16 lines of which it used a half.)
__host__ __device__ inline int delta_padded(int N) { return (N + 15) / 16 * 16; }
__host__ __device__ inline size_t delta_chunk_floats(int N, int V) {
    return (size_t)DELTA_CHUNK * (3 * delta_padded(N) + delta_padded(V) + DELTA_CHUNK) + delta_padded(N);
}

__device__ __forceinline__ floatx4 mma4(const floatx4& a, const floatx4& b, floatx4 c) {
#pragma unroll
    for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[i], c, 0, 0, 0);
    return c;
}

// The same for a lower triangular A (zeros above): row t takes B's rows 0 .. t.  A zero does not keep a later row out that is
// not finite -- a token must not see what comes after it --, so then every row is taken by itself with the later ones cleared.
__device__ __forceinline__ floatx4 mma4_lower(const floatx4& a, const floatx4& b, const floatx4& c) {
    bool odd = false;
#pragma unroll
    for (int i = 0; i < 4; ++i) odd |= !(fabsf(b[i]) <= 3.402823466e38f);
    if (__builtin_expect(!__any(odd), 1)) return mma4(a, b, c);
    const int first = ((threadIdx.x & 63) >> 4) * 4;
    floatx4 out = c;
#pragma unroll 1
    for (int t = 0; t < 16; ++t) {
        floatx4 seen;
#pragma unroll
        for (int i = 0; i < 4; ++i) seen[i] = first + i <= t ? b[i] : 0.f;
        const floatx4 row = mma4(a, seen, c);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (first + i == t) out[i] = row[i];
    }
    return out;
}

// One workgroup a chunk and head.  The pairs (t, s) of one half of the chunk need an exponential a key channel each, so a
// thread takes one pair (120 a half); between the halves e^{c_t - c_s} = e^{c_t - c_15} e^{c_15 - c_s}, neither above 1, and
// the sums are a matrix product.  T = (I + A)^-1 by halves too: two triangles of 16 a lane column by column, and
// -T22 A21 T11 between them.  A thread for each of 1024 pairs, half of them idle, T row by row over 32 rows, and the two
// products with T one element a thread took 199 us for 2048 tokens of 16 heads of 128 x 128 channels; this one 104 while a
// thread waited for its elements of q, k and the decays one after the other, 87 until the loops that leave the results stopped
// dividing for their places and taking e^{c_t} twice, now 75, of which the exponentials are the most.
__global__ __launch_bounds__(256) void delta_chunk_prepare_kernel(DeltaChunkArgs g) {
    constexpr int C = DELTA_CHUNK, CS = DELTA_CHUNK + 4;
    const DeltaArgs& a = g.d;
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int N = a.N, V = a.V, Np = delta_padded(N), NS = Np + 4;
    float* q_l = lds;                    // [C][NS]
    float* k_l = q_l + C * NS;
    float* c_l = k_l + C * NS;
    float* A_l = c_l + C * NS;           // [C][CS]
    float* B_l = A_l + C * CS;
    float* T_l = B_l + C * CS;
    float* part_l = T_l + C * CS;        // [4][2][256]: the wavefronts' shares of the block between the halves
    float* beta_l = part_l + 4 * 2 * 256;        // [C]
    const int chunk = blockIdx.x, head = blockIdx.y;
    const int r0 = g.chunk_first[chunk], n = g.chunk_count[chunk];
    const int qk_head = head / a.heads_per_group;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane & 15, b4 = (lane >> 4) * 4;
    float* base = g.scratch + ((size_t)chunk * a.heads + head) * delta_chunk_floats(N, V);
    float* W = base;
    float* Qh = W + (size_t)C * Np;
    float* Kt = Qh + (size_t)C * Np;
    float* Y = Kt + (size_t)C * Np;
    float* B = Y + (size_t)C * delta_padded(V);
    float* G = B + C * C;
    // (eight elements of each asked for at once, clamped and without a branch: one after the other a thread waited for memory
    // sixteen times, and once more for every beta)
    const float beta_raw = a.beta_raw[(size_t)(r0 + min(tid, n - 1)) * a.beta_stride + head];
    constexpr int EACH = 8;
    for (int at = tid; at < C * Np; at += 256 * EACH) {
        elem_t dq[EACH], dk[EACH];
        float dc[EACH];
        int t[EACH], i[EACH];
#pragma unroll
        for (int e = 0; e < EACH; ++e) {
            t[e] = (at + 256 * e) / Np;
            i[e] = (at + 256 * e) % Np;
            const size_t row = (size_t)(r0 + min(t[e], n - 1));
            const int ch = min(i[e], N - 1);
            dq[e] = a.q[row * a.q_stride + qk_head * N + ch];
            dk[e] = a.k[row * a.k_stride + qk_head * N + ch];
            dc[e] = a.log_decay[decay_at(a, row, head, ch)];
        }
#pragma unroll
        for (int e = 0; e < EACH; ++e) {
            if (at + 256 * e >= C * Np) break;
            const bool there = t[e] < n && i[e] < N;
            q_l[t[e] * NS + i[e]] = there ? to_float(dq[e]) : 0.f;
            k_l[t[e] * NS + i[e]] = there ? to_float(dk[e]) : 0.f;
            c_l[t[e] * NS + i[e]] = there ? dc[e] : 0.f;
        }
    }
    if (tid < C) beta_l[tid] = tid < n ? sigmoid_f(beta_raw) : 0.f;
    for (int p = tid; p < C * CS; p += 256) A_l[p] = B_l[p] = T_l[p] = 0.f;
    __syncthreads();
    for (int t = wave; t < C; t += 4) {                     // unit vectors, q scaled
        float qq = 0.f, kk = 0.f;
        for (int i = lane; i < N; i += 64) {
            const float dq = q_l[t * NS + i], dk = k_l[t * NS + i];
            qq += dq * dq;
            kk += dk * dk;
        }
        float fq = a.q_scale, fk = 1.0f;
        if (a.unit_norm) {
            fq = a.q_scale / sqrtf(wave_sum(qq) + a.unit_eps);
            fk = 1.0f / sqrtf(wave_sum(kk) + a.unit_eps);
        }
        for (int i = lane; i < N; i += 64) { q_l[t * NS + i] *= fq; k_l[t * NS + i] *= fk; }
    }
    for (int i = tid; i < Np; i += 256) {                   // c_t: the running sum of the log decays (rows past n add 0)
        float sum = 0.f;
#pragma unroll
        for (int t = 0; t < C; ++t) { sum += c_l[t * NS + i]; c_l[t * NS + i] = sum; }
    }
    __syncthreads();
    auto four = [](const float* p) { return *reinterpret_cast<const floatx4*>(p); };
    if (tid < 240) {                                        // the pairs s < t of both halves
        const int p = tid % 120, h0 = tid / 120 * 16;
        int t = (int)((1.0f + sqrtf(1.0f + 8.0f * (float)p)) * 0.5f);
        t -= t * (t - 1) / 2 > p ? 1 : 0;
        t += t * (t + 1) / 2 <= p ? 1 : 0;
        const int s = p - t * (t - 1) / 2;
        const float* ct = c_l + (h0 + t) * NS; const float* cs = c_l + (h0 + s) * NS;
        const float* kt = k_l + (h0 + t) * NS; const float* ks = k_l + (h0 + s) * NS; const float* qt = q_l + (h0 + t) * NS;
        floatx4 sa = {0.f, 0.f, 0.f, 0.f}, sb = {0.f, 0.f, 0.f, 0.f};
        for (int i = 0; i < Np; i += 4) {
            const floatx4 d = four(ct + i) - four(cs + i), k4 = four(ks + i), kt4 = four(kt + i), qt4 = four(qt + i);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float x = k4[e] * expf(d[e]);
                sa[e] += kt4[e] * x;
                sb[e] += qt4[e] * x;
            }
        }
        A_l[(h0 + t) * CS + h0 + s] = beta_l[h0 + t] * ((sa[0] + sa[1]) + (sa[2] + sa[3]));
        B_l[(h0 + t) * CS + h0 + s] = (sb[0] + sb[1]) + (sb[2] + sb[3]);
    } else {                                                // the pairs s = t, of B
        for (int t = tid - 240; t < C; t += 16) {
            floatx4 sb = {0.f, 0.f, 0.f, 0.f};
            for (int i = 0; i < Np; i += 4) sb += four(q_l + t * NS + i) * four(k_l + t * NS + i);
            B_l[t * CS + t] = (sb[0] + sb[1]) + (sb[2] + sb[3]);
        }
    }
    {                                                       // rows 16 .. 31 against columns 0 .. 15: a share of the channels a wavefront
        floatx4 sa = {0.f, 0.f, 0.f, 0.f}, sb = {0.f, 0.f, 0.f, 0.f};
        for (int i0 = wave * 16; i0 < Np; i0 += 64) {
            const int i = i0 + b4;
            const floatx4 mid = four(c_l + 15 * NS + i), dt = four(c_l + (16 + c) * NS + i) - mid, ds = mid - four(c_l + c * NS + i);
            floatx4 kt = four(k_l + (16 + c) * NS + i), qt = four(q_l + (16 + c) * NS + i), ks = four(k_l + c * NS + i);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float f = expf(dt[e]);
                kt[e] *= f;
                qt[e] *= f;
                ks[e] *= expf(ds[e]);
            }
            sa = mma4(kt, ks, sa);
            sb = mma4(qt, ks, sb);
        }
        *reinterpret_cast<floatx4*>(part_l + (wave * 2) * 256 + lane * 4) = sa;
        *reinterpret_cast<floatx4*>(part_l + (wave * 2 + 1) * 256 + lane * 4) = sb;
    }
    floatx4 e_c[4];                                         // e^{c_t}, of the elements that this thread leaves in Qhat
    {                                                       // Qhat, Kbar and G (they read what the loops above read)
        const int rt = wave & 1, t = 16 * rt + c;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int i0 = 16 * ((wave >> 1) + 2 * u), i = i0 + b4;
            if (i0 >= Np) break;
            const floatx4 ct = four(c_l + t * NS + i);
            floatx4 x = four(q_l + t * NS + i);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                e_c[u][e] = expf(ct[e]);
                x[e] *= e_c[u][e];
            }
            *reinterpret_cast<floatx4*>(Qh + (size_t)(i0 / 16 * 2 + rt) * 256 + lane * 4) = x;
            const float last = c_l[(C - 1) * NS + i0 + c];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int at = (16 * rt + b4 + e) * NS + i0 + c;
                x[e] = k_l[at] * expf(last - c_l[at]);
            }
            *reinterpret_cast<floatx4*>(Kt + (size_t)(i0 / 16 * 2 + rt) * 256 + lane * 4) = x;
        }
        if (tid < Np) G[tid] = expf(c_l[(C - 1) * NS + tid]);
    }
    __syncthreads();
    {
        const int e = tid & 3, l = tid >> 2, t = 16 + (l >> 4) * 4 + e, s = l & 15;      // element e of lane l
        float sa = 0.f, sb = 0.f;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            sa += part_l[(w * 2) * 256 + tid];
            sb += part_l[(w * 2 + 1) * 256 + tid];
        }
        A_l[t * CS + s] = beta_l[t] * sa;
        B_l[t * CS + s] = sb;
    }
    {                                                       // beta Khat in q's place
        const int t = 16 * (wave & 1) + c;
        const float beta = beta_l[t];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int i0 = 16 * ((wave >> 1) + 2 * u), i = i0 + b4;
            if (i0 >= Np) break;
            floatx4 x = four(k_l + t * NS + i);
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = beta * x[e] * e_c[u][e];
            *reinterpret_cast<floatx4*>(q_l + t * NS + i) = x;
        }
    }
    if (tid < 32) {                                         // the inverses of the two triangles, a column a lane, row after row
        const int j = tid & 15, h0 = tid & 16;
        float x[16];
#pragma unroll
        for (int t = 0; t < 16; ++t) {
            x[t] = t == j ? 1.f : 0.f;
#pragma unroll
            for (int s = 0; s < t; ++s) x[t] -= A_l[(h0 + t) * CS + h0 + s] * x[s];
        }
#pragma unroll
        for (int t = 0; t < 16; ++t) T_l[(h0 + t) * CS + h0 + j] = x[t];
    }
    __syncthreads();
    if (wave == 0) {                                        // T21 = -T22 (A21 T11)
        floatx4 t11, p = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 4; ++i) t11[i] = T_l[(b4 + i) * CS + c];
        p = mma4(four(A_l + (16 + c) * CS + b4), t11, p);
        p = mma4_lower(four(T_l + (16 + c) * CS + 16 + b4), p, floatx4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
        for (int i = 0; i < 4; ++i) T_l[(16 + b4 + i) * CS + c] = -p[i];
    }
    {
        const int rt = wave & 1, st = wave >> 1;
        *reinterpret_cast<floatx4*>(B + wave * 256 + lane * 4) = four(B_l + (16 * rt + c) * CS + 16 * st + b4);
    }
    __syncthreads();
    floatx4 tf[2][2];                                       // T's rows 16 rt + c, columns 16 st + b4 ..
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
        for (int st = 0; st < 2; ++st) tf[rt][st] = four(T_l + (16 * rt + c) * CS + 16 * st + b4);
    auto product = [&](const floatx4 (&x)[2], floatx4& top, floatx4& low) {                   // T x, 16 columns
        top = mma4_lower(tf[0][0], x[0], floatx4{0.f, 0.f, 0.f, 0.f});
        low = mma4_lower(tf[1][1], x[1], mma4(tf[1][0], x[0], floatx4{0.f, 0.f, 0.f, 0.f}));
    };
    for (int i0 = wave * 16; i0 < Np; i0 += 64) {
        floatx4 x[2];
#pragma unroll
        for (int st = 0; st < 2; ++st)
#pragma unroll
            for (int i = 0; i < 4; ++i) x[st][i] = q_l[(16 * st + b4 + i) * NS + i0 + c];
        floatx4 top, low;
        product(x, top, low);
        float* dst = W + (size_t)(i0 / 16 * 2) * 256 + (c >> 2) * 64 + (c & 3);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            dst[(b4 + i) * 4] = top[i];
            dst[256 + (b4 + i) * 4] = low[i];
        }
    }
    for (int j0 = wave * 16; j0 < V; j0 += 64) {
        const int j = j0 + c;
        floatx4 x[2];
#pragma unroll
        for (int st = 0; st < 2; ++st)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int t = 16 * st + b4 + i;
                x[st][i] = t < n && j < V ? beta_l[t] * to_float(a.v[(size_t)(r0 + t) * a.v_stride + head * V + j]) : 0.f;
            }
        floatx4 top, low;
        product(x, top, low);
        float* dst = Y + (size_t)(j0 / 16 * 2) * 256 + lane * 4;
        *reinterpret_cast<floatx4*>(dst) = top;
        *reinterpret_cast<floatx4*>(dst + 256) = low;
    }
}

// One workgroup per request, head and 16 value channels; a wavefront owns the key channels of the tiles wave, wave + 4 (of 16)
// and keeps their part of the state in registers.  A chunk: every wavefront's share of W S0 goes through LDS (the one barrier
// a chunk), all add them up to U, and update their part of the state; the shares of O meet in LDS likewise and are added a
// chunk later.  A chunk's operands are on their way while the chunk before is worked on.  Scalar sums out of tiles staged in
// LDS took 598 us for 2048 tokens of 16 heads of 128 x 128 channels (64 chunks, 128 workgroups); this one 102, 1.6 us a
// chunk, of which 0.7 are its 52 matrix instructions a wavefront and the rest the chain between them: it is bound by the
// walk's length, not by memory.  (149 us with the operands as rows, a load's 64 lanes in 16 lines of which it used a half; 111 with
// a loop that waited for every load in its head and with Qhat S0 wholly before the barrier.)  Without AHEAD, for more workgroups
// than compute units, a chunk's operands are asked for as it begins, and three workgroups share a unit.
template <int NT, bool AHEAD>
__global__ __launch_bounds__(256, AHEAD ? 1 : 3) void delta_chunk_scan_kernel(DeltaChunkArgs g) {
    constexpr int C = DELTA_CHUNK;
    const DeltaArgs& a = g.d;
    __shared__ __attribute__((aligned(16))) float u_l[2][4][2][256], o_l[2][4][2][256];      // [buffer][wavefront][row tile][lane, element]
    const int N = a.N, V = a.V, Np = delta_padded(N);
    const int seg = blockIdx.x, head = blockIdx.y;
    const int r0 = a.seg_first[seg], n = a.seg_count[seg];
    const int slot = a.slots[r0];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), c = lane & 15, b4 = (lane >> 4) * 4;
    const int col = blockIdx.z * 16 + c;
    const bool col_ok = col < V;
    int chunk0 = 0;
    for (int s = 0; s < seg; ++s) chunk0 += (a.seg_count[s] + C - 1) / C;
    const size_t step = (size_t)a.heads * delta_chunk_floats(N, V);
    const size_t state_at = (size_t)slot * a.state_stride + (size_t)head * N * V, stage_at = (size_t)(slot ^ a.pair) * a.state_stride + (size_t)head * N * V;
    const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
    floatx4 S[NT];
    bool mine[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const int n0 = (wave + 4 * j) * 16;
        mine[j] = n0 < Np;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int ch = n0 + b4 + i;
            S[j][i] = ch < N && col_ok ? a.live[state_at + (size_t)ch * V + col] : 0.f;
        }
    }
    struct Chunk {
        floatx4 w[2][NT], q[2][NT], k[NT][2], gate[NT], b, y[2];
    };
    const int b_row = wave & 1, b_col = wave >> 1;          // this wavefront's quarter of B (the one above the diagonal is zero)
    auto fetch = [&](const float* from, Chunk& x) {
        const float* Qh = from + (size_t)C * Np;
        const float* Kt = Qh + (size_t)C * Np;
        const float* Y = Kt + (size_t)C * Np;
        const float* B = Y + (size_t)C * delta_padded(V);
        const float* G = B + C * C;
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const int tile = mine[j] ? wave + 4 * j : 0;                       // (for a tile that is not there: its state stays zero)
#pragma unroll
            for (int rt = 0; rt < 2; ++rt) {
                const int at = (tile * 2 + rt) * 256 + lane * 4;
                x.w[rt][j] = *reinterpret_cast<const floatx4*>(from + at);
                x.q[rt][j] = *reinterpret_cast<const floatx4*>(Qh + at);
                x.k[j][rt] = *reinterpret_cast<const floatx4*>(Kt + at);
            }
            x.gate[j] = *reinterpret_cast<const floatx4*>(G + tile * 16 + b4);
        }
        x.b = *reinterpret_cast<const floatx4*>(B + wave * 256 + lane * 4);
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) x.y[rt] = *reinterpret_cast<const floatx4*>(Y + ((int)blockIdx.z * 2 + rt) * 256 + lane * 4);
    };
    auto put_out = [&](int buf, int c0) {                   // the shares of a chunk's O, added up: two of a lane's elements a thread
        const int rt = wave >> 1, e0 = (wave & 1) * 2, t = 16 * rt + b4 + e0;
        float2 o = *reinterpret_cast<const float2*>(&o_l[buf][0][rt][lane * 4 + e0]);
#pragma unroll
        for (int w = 1; w < 4; ++w) {
            const float2 more = *reinterpret_cast<const float2*>(&o_l[buf][w][rt][lane * 4 + e0]);
            o.x += more.x;
            o.y += more.y;
        }
        float* dst = a.out + (size_t)(r0 + c0 + t) * ((size_t)a.heads * V) + head * V + col;
        if (c0 + t < n && col_ok) dst[0] = o.x;
        if (c0 + t + 1 < n && col_ok) dst[(size_t)a.heads * V] = o.y;
    };
    const float* base = g.scratch + (size_t)chunk0 * step + (size_t)head * delta_chunk_floats(N, V);
    auto work = [&](const Chunk& now, int c0, int buf) {
        floatx4 part[2] = {zero, zero}, o[2] = {zero, zero};
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int rt = 0; rt < 2; ++rt) part[rt] = __builtin_amdgcn_mfma_f32_16x16x4f32(now.w[rt][j][i], S[j][i], part[rt], 0, 0, 0);
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) *reinterpret_cast<floatx4*>(&u_l[buf][wave][rt][lane * 4]) = part[rt];
        // (Qhat S0, not on the way to U: half of it while the shares go into LDS, half while they come out)
        auto start_out = [&](int from, int to) {
#pragma unroll
            for (int e = from; e < to; ++e)
#pragma unroll
                for (int rt = 0; rt < 2; ++rt) o[rt] = __builtin_amdgcn_mfma_f32_16x16x4f32(now.q[rt][e >> 2][e & 3], S[e >> 2][e & 3], o[rt], 0, 0, 0);
        };
        start_out(0, 2 * NT);
        __syncthreads();
        floatx4 u[2], share[2][4];
#pragma unroll
        for (int rt = 0; rt < 2; ++rt)
#pragma unroll
            for (int w = 0; w < 4; ++w) share[rt][w] = *reinterpret_cast<const floatx4*>(&u_l[buf][w][rt][lane * 4]);
        __builtin_amdgcn_sched_barrier(0);
        start_out(2 * NT, 4 * NT);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
            floatx4 sum = share[rt][0];
#pragma unroll
            for (int w = 1; w < 4; ++w) sum += share[rt][w];
            u[rt] = now.y[rt] - sum;
        }
#pragma unroll
        for (int j = 0; j < NT; ++j) S[j] *= now.gate[j];
#pragma unroll
        for (int st = 0; st < 2; ++st)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) S[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(now.k[j][st][i], u[st][i], S[j], 0, 0, 0);
#pragma unroll
        for (int j = 0; j < NT; ++j)
            if (!mine[j]) S[j] = zero;                      // (the same in every lane)
        if (b_row >= b_col) {
            if (b_row == 0) o[0] = mma4_lower(now.b, u[0], o[0]);
            else o[1] = b_col == 0 ? mma4(now.b, u[0], o[1]) : mma4_lower(now.b, u[1], o[1]);
        }
        if (c0 > 0) put_out(buf ^ 1, c0 - C);               // (written before the barrier above)
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) *reinterpret_cast<floatx4*>(&o_l[buf][wave][rt][lane * 4]) = o[rt];
    };
    int buf = 0;
    if (AHEAD) {
        Chunk ring[3];                                      // the chunk at work and the two behind it
        const float* last = base + (size_t)((n - 1) / C) * step;
        fetch(base, ring[0]);
        __builtin_amdgcn_sched_barrier(0);                  // (in this order, as in the loop: its waits count on it)
        fetch(base + step <= last ? base + step : last, ring[1]);
        __builtin_amdgcn_sched_barrier(0);
        auto turn = [&](const Chunk& now, Chunk& ahead, int c0) {
            fetch(base + 2 * step <= last ? base + 2 * step : last, ahead);    // (never behind a branch)
            base += step;
            work(now, c0, buf);
            buf ^= 1;
        };
        // (no way out of the loop's middle: where such paths meet, its head waits for every load that is under way)
        int c0 = 0;
        for (; c0 + 2 * C < n; c0 += 3 * C) {
            turn(ring[0], ring[2], c0);
            turn(ring[1], ring[0], c0 + C);
            turn(ring[2], ring[1], c0 + 2 * C);
        }
        if (c0 < n) {
            work(ring[0], c0, buf);
            buf ^= 1;
        }
        if (c0 + C < n) {
            work(ring[1], c0 + C, buf);
            buf ^= 1;
        }
    } else {
        for (int c0 = 0; c0 < n; c0 += C) {
            Chunk now;
            fetch(base, now);
            base += step;
            work(now, c0, buf);
            buf ^= 1;
        }
    }
    __syncthreads();
    put_out(buf ^ 1, (n - 1) / C * C);
    if (a.write_state && col_ok)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int ch = (wave + 4 * j) * 16 + b4 + i;
                if (ch < N) a.stage[stage_at + (size_t)ch * V + col] = S[j][i];
            }
}

// (requests of one token each: room for one in LDS, as in launch_scan; 48 requests of 32 heads of 128 x 128 69.8 us, now 54.6)
template <int NR, int PARTS>
static int launch_delta(const DeltaArgs& a, int segments, bool singles, hipStream_t stream) {
    constexpr int COLS = 64 / PARTS;
    const dim3 grid(segments, a.heads, (a.V + COLS - 1) / COLS);
    if (singles) delta_rule_kernel<NR, PARTS, 1><<<grid, 64, 0, stream>>>(a);
    else delta_rule_kernel<NR, PARTS, DELTA_TILE><<<grid, 64, 0, stream>>>(a);
    return (int)hipGetLastError();
}

// Requests of one token each (`singles`) stage one at a time: the step is bound by reading and writing the states, and with
// the LDS of 16 tokens only three workgroups fit a compute unit (48 requests of 16 heads of 128 x 128: 25.2 us, with room
// for one token 20.3; one request 8.6 and 5.9).
template <int NR, int TILE>
static int launch_scan(const ScanArgs& a, int segments, bool singles, hipStream_t stream) {
    const size_t lds_token = sizeof(float) * ((size_t)3 * NR * SCAN_PARTS + (size_t)SCAN_COLS * (1 + SCAN_PARTS)), lds = TILE * lds_token;
    dim3 grid(segments, a.heads, (a.V + SCAN_COLS - 1) / SCAN_COLS);
    if (a.piece_state == nullptr) {
        if (singles) linear_recurrence_kernel<NR, 1, 0><<<grid, 256, lds_token, stream>>>(a);
        else linear_recurrence_kernel<NR, TILE, 0><<<grid, 256, lds, stream>>>(a);
        return (int)hipGetLastError();
    }
    linear_recurrence_kernel<NR, TILE, 1><<<grid, 256, lds, stream>>>(a);
    int err = (int)hipGetLastError();
    if (err != 0) return err;
    const size_t per = (size_t)a.heads * a.N * a.V;
    piece_states_kernel<<<(unsigned)((per + 255) / 256), 256, 0, stream>>>(a, segments);
    err = (int)hipGetLastError();
    if (err != 0) return err;
    linear_recurrence_kernel<NR, TILE, 2><<<grid, 256, lds, stream>>>(a);
    return (int)hipGetLastError();
}

static int grid_for(size_t count, int block) {
    size_t g = (count + block - 1) / block;
    return (int)(g > 65535 ? 65535 : (g == 0 ? 1 : g));
}

extern "C" {

int mlr_causal_conv(const void* x, long x_stride, const float* w, const float* b, void* out, long out_stride,
                    const float* live, float* stage, long state_stride, const int32_t* slots, const int32_t* positions,
                    int rows, int channels, int taps, int silu, int write_state, hipStream_t stream) {
    if (rows <= 0 || channels <= 0) return 0;
    if (taps < 1 || taps > CONV_MAX_TAPS) return -1;
    ConvArgs a{(const elem_t*)x, x_stride, w, b, (elem_t*)out, out_stride, live, stage, state_stride, slots, positions,
               rows, channels, taps, silu, write_state, live == stage};
#if MLR_BF16
    const auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    // A walk of CONV_ROWS rows takes 11 us however few they are.  The line lies where one value a thread takes as long: 256
    // rows of 6144 channels 12.2 us and 11.3 here, 384 of 4352 12.5 and 12.0; but 512 of 2048 9.2 and 11.0, 128 of 4352 6.7 and 10.9.
    const bool many = (long)rows * channels >= 3L << 19;
    if (many && taps == 4 && channels % 8 == 0 && x_stride % 8 == 0 && out_stride % 8 == 0 && aligned(x) && aligned(out) && aligned(w)) {
        causal_conv_rows_kernel<4><<<dim3((rows + CONV_ROWS - 1) / CONV_ROWS, (channels / 8 + 255) / 256), 256, 0, stream>>>(a);
        return (int)hipGetLastError();
    }
#endif
    causal_conv_kernel<<<dim3(rows, (channels + 255) / 256), 256, 0, stream>>>(a);
    return (int)hipGetLastError();
}

int mlr_gla_log_decay(const void* z, const float* bias, float* out, int rows, int width, float inv_tau, hipStream_t stream) {
    if (rows <= 0) return 0;
    gla_log_decay_kernel<<<grid_for((size_t)rows * width, 256), 256, 0, stream>>>((const elem_t*)z, bias, out, (size_t)rows,
                                                                                 width, inv_tau);
    return (int)hipGetLastError();
}

int mlr_mamba_step(const void* raw, long raw_stride, const float* dt_bias, const float* a_log, float* dt, float* log_decay,
                   int rows, int heads, hipStream_t stream) {
    if (rows <= 0) return 0;
    mamba_step_kernel<<<grid_for((size_t)rows * heads, 256), 256, 0, stream>>>((const elem_t*)raw, raw_stride, dt_bias, a_log,
                                                                              dt, log_decay, (size_t)rows, heads);
    return (int)hipGetLastError();
}

int mlr_linear_recurrence(const void* q, long q_stride, const void* k, long k_stride, const void* v, long v_stride,
                          const float* log_decay, long decay_stride, int decay_per_channel, const float* v_scale,
                          long v_scale_stride, const float* skip, float q_scale, float* out, const float* live, float* stage,
                          long state_stride, const int32_t* seg_first, const int32_t* seg_count, const int32_t* slots,
                          int rows, int segments, int heads, int heads_per_group, int n_keys, int n_values, int write_state,
                          float* piece_state, float* piece_decay, int silu, const float* rope, const int32_t* positions,
                          int rot_dim, hipStream_t stream) {
    // piece_state, piece_decay given: `seg_first`/`seg_count` name pieces of requests (a request's pieces one after
    // the other), run side by side in three passes; [segments][heads][n_keys][n_values] and [segments][heads][n_keys]
    if (segments <= 0) return 0;
    if (n_keys < 1 || n_keys > 256 || n_values < 1 || heads < 1 || heads_per_group < 1 || heads % heads_per_group) return -1;
    if (rot_dim < 0 || rot_dim > n_keys || (rot_dim & 1) || (rot_dim > 0 && (rope == nullptr || positions == nullptr))) return -1;
    ScanArgs a{(const elem_t*)q, q_stride, (const elem_t*)k, k_stride, (const elem_t*)v, v_stride, log_decay, decay_stride,
               v_scale, v_scale_stride, skip, out, live, stage, state_stride, seg_first, seg_count, slots, heads,
               heads_per_group, n_keys, n_values, decay_per_channel, write_state, q_scale, silu, rope, positions, rot_dim, piece_state,
               piece_decay, live == stage};
    if ((piece_state == nullptr) != (piece_decay == nullptr)) return -2;
    const int nr = (n_keys + SCAN_PARTS - 1) / SCAN_PARTS;
    if (nr <= 8) return launch_scan<8, 16>(a, segments, rows == segments, stream);
    if (nr <= 16) return launch_scan<16, 16>(a, segments, rows == segments, stream);
    if (nr <= 32) return launch_scan<32, 16>(a, segments, rows == segments, stream);
    return launch_scan<64, 8>(a, segments, rows == segments, stream);
}

int mlr_channel_log_decay(const float* z, const float* bias, const float* a_log, float* out, int rows, int heads, int n_keys,
                          hipStream_t stream) {
    if (rows <= 0) return 0;
    if (heads < 1 || n_keys < 1) return -1;
    const size_t width = (size_t)heads * n_keys, total = (size_t)rows * width;
    const size_t across = width >= 262144 ? 1 : 262144 / width;               // rows side by side: a quarter of a million threads
    const size_t stride = (across < (size_t)rows ? across : (size_t)rows) * width;
    channel_log_decay_kernel<<<(unsigned)((stride + 255) / 256), 256, 0, stream>>>(z, bias, a_log, out, total, stride, (int)width, n_keys);
    return (int)hipGetLastError();
}

// The delta rule over the step's requests (seg_first, seg_count: one entry a request).  A lane keeps at most 64 rows of
// its column of S: up to 64 key channels a lane holds a whole column (64 columns a wavefront), up to 128 two lanes share
// one, up to 256 four; heads of few value channels use the narrower layouts too, so that their lanes are not idle.
int mlr_delta_rule(const void* q, long q_stride, const void* k, long k_stride, const void* v, long v_stride,
                   const float* log_decay, const float* beta_raw, long beta_stride, float* out, const float* live, float* stage,
                   long state_stride, const int32_t* seg_first, const int32_t* seg_count, const int32_t* slots, int rows,
                   int segments, int heads, int heads_per_group, int n_keys, int n_values, int write_state, int unit_norm, float q_scale,
                   float unit_eps, int decay_per_head, hipStream_t stream) {
    if (segments <= 0) return 0;
    if (n_keys < 1 || n_keys > 256 || n_values < 1 || heads < 1 || heads > 65535 || heads_per_group < 1 ||
        heads % heads_per_group)
        return -1;
    DeltaArgs a{(const elem_t*)q, q_stride, (const elem_t*)k, k_stride, (const elem_t*)v, v_stride, log_decay, beta_raw,
                beta_stride, out, live, stage, state_stride, seg_first, seg_count, slots, heads, heads_per_group, n_keys,
                n_values, write_state, unit_norm, q_scale, unit_eps, decay_per_head, live == stage};
    int parts = n_keys > 128 ? 4 : n_keys > 64 ? 2 : 1;
    if (n_values <= 16 && parts < 4) parts = 4;
    else if (n_values <= 32 && parts < 2) parts = 2;
    const int nr = (n_keys + parts - 1) / parts;
#define MLR_DELTA(PARTS)                                                        \
    if (parts == PARTS) {                                                       \
        if (nr <= 8) return launch_delta<8, PARTS>(a, segments, rows == segments, stream);        \
        if (nr <= 16) return launch_delta<16, PARTS>(a, segments, rows == segments, stream);      \
        if (nr <= 32) return launch_delta<32, PARTS>(a, segments, rows == segments, stream);      \
        return launch_delta<64, PARTS>(a, segments, rows == segments, stream);                    \
    }
    MLR_DELTA(1)
    MLR_DELTA(2)
    MLR_DELTA(4)
#undef MLR_DELTA
    return -1;
}

// The delta rule in chunks (see delta_chunk_prepare_kernel): `chunk_first`/`chunk_count` name the step's chunks of at
// most DELTA_CHUNK tokens, a request's chunks one after the other and the requests in the order of `seg_first`;
// scratch: chunks * heads * mlr_delta_chunk_floats(n_keys, n_values) floats.  Up to 128 key channels a head.
long mlr_delta_chunk_floats(int n_keys, int n_values) { return (long)delta_chunk_floats(n_keys, n_values); }
int mlr_delta_chunk_tokens() { return DELTA_CHUNK; }

int mlr_delta_rule_chunked(const void* q, long q_stride, const void* k, long k_stride, const void* v, long v_stride,
                           const float* log_decay, const float* beta_raw, long beta_stride, float* out, const float* live,
                           float* stage, long state_stride, const int32_t* seg_first, const int32_t* seg_count,
                           const int32_t* slots, int segments, const int32_t* chunk_first, const int32_t* chunk_count, int chunks,
                           float* scratch, int heads, int heads_per_group, int n_keys, int n_values, int write_state,
                           int unit_norm, float q_scale, float unit_eps, int decay_per_head, hipStream_t stream) {
    if (segments <= 0 || chunks <= 0) return 0;
    if (n_keys < 1 || n_keys > 128 || n_values < 1 || heads < 1 || heads > 65535 || heads_per_group < 1 ||
        heads % heads_per_group || scratch == nullptr)
        return -1;
    DeltaChunkArgs g{{(const elem_t*)q, q_stride, (const elem_t*)k, k_stride, (const elem_t*)v, v_stride, log_decay, beta_raw,
                      beta_stride, out, live, stage, state_stride, seg_first, seg_count, slots, heads, heads_per_group, n_keys,
                      n_values, write_state, unit_norm, q_scale, unit_eps, decay_per_head, live == stage},
                     chunk_first, chunk_count, scratch};
    if ((reinterpret_cast<uintptr_t>(scratch) & 15) != 0) return -1;
    const int C = DELTA_CHUNK, Np = delta_padded(n_keys);
    const size_t lds = sizeof(float) * ((size_t)3 * C * (Np + 4) + (size_t)3 * C * (C + 4) + 4 * 2 * 256 + C);
    static const hipError_t allowed = hipFuncSetAttribute(reinterpret_cast<const void*>(&delta_chunk_prepare_kernel),
                                                          hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024);
    if (allowed != hipSuccess) return (int)allowed;
    delta_chunk_prepare_kernel<<<dim3(chunks, heads), 256, lds, stream>>>(g);
    int err = (int)hipGetLastError();
    if (err != 0) return err;
    const dim3 grid(segments, heads, (n_values + 15) / 16);
    // (two chunks of operands on their way while one is at work while no compute unit has a second workgroup, which the registers
    // would keep out: both kernels, one request of 2048 tokens of 16 heads of 128 x 128 172 us, without 194; but three of 700 165
    // and 148, four of 512 128 and 115, 64 of 32 245 and 178, 64 of 9 238 and 169)
    const bool ahead = (long)segments * heads * ((n_values + 15) / 16) <= 256;
    if (Np <= 64) {
        if (ahead) delta_chunk_scan_kernel<1, true><<<grid, 256, 0, stream>>>(g);
        else delta_chunk_scan_kernel<1, false><<<grid, 256, 0, stream>>>(g);
    } else {
        if (ahead) delta_chunk_scan_kernel<2, true><<<grid, 256, 0, stream>>>(g);
        else delta_chunk_scan_kernel<2, false><<<grid, 256, 0, stream>>>(g);
    }
    return (int)hipGetLastError();
}

}  // extern "C"
