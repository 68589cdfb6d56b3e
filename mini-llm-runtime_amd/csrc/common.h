// Shared device helpers for the gfx950 kernels: element type of the engine (bfloat16 or
// float, chosen at compile time with -DMLR_BF16=1/0), wavefront (64 lanes) and workgroup
// reductions, 16-byte vector access.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#ifndef MLR_BF16
#error "compile with -DMLR_BF16=0 (float engine) or -DMLR_BF16=1 (bfloat16 engine)"
#endif

#if MLR_BF16
typedef __bf16 elem_t;
#define MLR_VEC 8            // elements in a 16-byte access
#else
typedef float elem_t;
#define MLR_VEC 4
#endif

#define MLR_WAVE 64

__device__ __forceinline__ float to_float(float x) { return x; }
__device__ __forceinline__ float to_float(__bf16 x) { return (float)x; }
template <class T> __device__ __forceinline__ T from_float(float x);
template <> __device__ __forceinline__ float from_float<float>(float x) { return x; }
template <> __device__ __forceinline__ __bf16 from_float<__bf16>(float x) { return (__bf16)x; }

struct alignas(16) vec16 { uint32_t w[4]; };

// Load MLR_VEC consecutive elements (16 bytes, 16-byte aligned) as floats.
__device__ __forceinline__ void vec_values(const vec16& v, float* out) {
#if MLR_BF16
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        out[2 * i] = __uint_as_float(v.w[i] << 16);
        out[2 * i + 1] = __uint_as_float(v.w[i] & 0xffff0000u);
    }
#else
#pragma unroll
    for (int i = 0; i < 4; ++i) out[i] = __uint_as_float(v.w[i]);
#endif
}

__device__ __forceinline__ void load_vec(const elem_t* p, float* out) { vec_values(*reinterpret_cast<const vec16*>(p), out); }

__device__ __forceinline__ void store_vec(elem_t* p, const float* in) {
    alignas(16) elem_t tmp[MLR_VEC];
#pragma unroll
    for (int i = 0; i < MLR_VEC; ++i) tmp[i] = from_float<elem_t>(in[i]);
    *reinterpret_cast<vec16*>(p) = *reinterpret_cast<const vec16*>(tmp);
}

// The same bits whatever fused operations the compiler would choose: a token's key is written by one of three
// kernels (the general and the vector kernel of rope_kv.hip, the decode merge of attention.hip) and should not
// depend on which.  An empty asm makes an intermediate opaque, so that a product cannot be drawn into the
// sum that follows it; the fused multiply-adds that are meant are written out.
__device__ __forceinline__ float opaque(float v) {
    asm("" : "+v"(v));
    return v;
}
// (x, y) = (a, b) turned by the angle with cosine c and sine s
__device__ __forceinline__ float turn_x(float a, float b, float c, float s) { return __builtin_fmaf(a, c, -opaque(b * s)); }
__device__ __forceinline__ float turn_y(float a, float b, float c, float s) { return __builtin_fmaf(a, s, opaque(b * c)); }
// a^2 + b^2, to be added to a running sum
__device__ __forceinline__ float squares(float a, float b) { return opaque(__builtin_fmaf(a, a, opaque(b * b))); }

// Four floats a lane: register i of lane block b (lanes 16 b ..) becomes what register b of block i was, so that four
// neighbouring places of a row become the places 4 i + b, which is what a 16x16x4 matrix instruction wants.
template <typename V> __device__ __forceinline__ V turned(const V& v) {
    unsigned r[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = __float_as_uint(v[i]);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const auto x = __builtin_amdgcn_permlane32_swap(r[i], r[i + 2], false, false);
        r[i] = x[0];
        r[i + 2] = x[1];
    }
#pragma unroll
    for (int i = 0; i < 4; i += 2) {
        const auto x = __builtin_amdgcn_permlane16_swap(r[i], r[i + 1], false, false);
        r[i] = x[0];
        r[i + 1] = x[1];
    }
    return V{__uint_as_float(r[0]), __uint_as_float(r[1]), __uint_as_float(r[2]), __uint_as_float(r[3])};
}

// Values of other lanes without a trip through LDS, which a `__shfl_xor` is (a sum over a wavefront is a chain of six; one token of
// the 0.6B sizes 1019 -> 1000 us a step, Pamunex 2.55 -> 2.515 ms; the float engine, whose time is its products', the same):
// the lane i ^ OFF within 16 lanes by DPP; across rows of 16 both operands of a swap, of which one is the lane's own value and the
// other its partner's -- which is which does not matter to a sum or a maximum.  All lanes of the wavefront take part.
template <int OFF> __device__ __forceinline__ float row_xor(float v) {
    static_assert(OFF == 1 || OFF == 2 || OFF == 4 || OFF == 8, "within 16 lanes");
    const int x = __float_as_int(v);
    if (OFF == 4) {                                       // lanes 0-3 and 8-11 from four up, the others from four down
        const int up = __builtin_amdgcn_update_dpp(x, x, 0x104, 0xf, 0x5, false);
        return __int_as_float(__builtin_amdgcn_update_dpp(up, x, 0x114, 0xf, 0xa, false));
    }
    constexpr int CTRL = OFF == 1 ? 0xb1 : OFF == 2 ? 0x4e : 0x128;         // quad_perm [1, 0, 3, 2], [2, 3, 0, 1], row_ror:8
    return __int_as_float(__builtin_amdgcn_update_dpp(x, x, CTRL, 0xf, 0xf, false));
}
struct lane_pair { float a, b; };
template <int OFF> __device__ __forceinline__ lane_pair xor_pair(float v) {
    const unsigned x = __float_as_uint(v);
    if constexpr (OFF == 32) {
        const auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
        return {__uint_as_float(r[0]), __uint_as_float(r[1])};
    } else if constexpr (OFF == 16) {
        const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
        return {__uint_as_float(r[0]), __uint_as_float(r[1])};
    } else {
        return {v, row_xor<OFF>(v)};
    }
}
template <int OFF> __device__ __forceinline__ float xor_sum(float v) { const lane_pair p = xor_pair<OFF>(v); return p.a + p.b; }
template <int OFF> __device__ __forceinline__ float xor_max(float v) { const lane_pair p = xor_pair<OFF>(v); return fmaxf(p.a, p.b); }
// The sum of groups of `lanes` (a power of two) neighbouring lanes, added from the nearest partner to the farthest.
__device__ __forceinline__ float group_sum(float v, int lanes) {
    if (lanes > 1) v = xor_sum<1>(v);
    if (lanes > 2) v = xor_sum<2>(v);
    if (lanes > 4) v = xor_sum<4>(v);
    if (lanes > 8) v = xor_sum<8>(v);
    if (lanes > 16) v = xor_sum<16>(v);
    if (lanes > 32) v = xor_sum<32>(v);
    return v;
}

// The sum of the lanes FROM, 2 FROM, .. apart, likewise.
template <int FROM> __device__ __forceinline__ float far_sum(float v) {
    if constexpr (FROM < 64) return far_sum<2 * FROM>(xor_sum<FROM>(v));
    else return v;
}

__device__ __forceinline__ float wave_sum(float v) {
    return xor_sum<1>(xor_sum<2>(xor_sum<4>(xor_sum<8>(xor_sum<16>(xor_sum<32>(v))))));
}
__device__ __forceinline__ float wave_max(float v) {
    return xor_max<1>(xor_max<2>(xor_max<4>(xor_max<8>(xor_max<16>(xor_max<32>(v))))));
}

// Sum over a workgroup of up to 1024 threads (a multiple of 64); every thread gets the
// result.  `scratch` holds at least 16 floats of LDS.  The order of the additions depends on
// the workgroup size only.
__device__ __forceinline__ float block_sum(float v, float* scratch) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = (blockDim.x + 63) >> 6;
    v = wave_sum(v);
    __syncthreads();
    if (lane == 0) scratch[wave] = v;
    __syncthreads();
    float total = 0.f;
    for (int i = 0; i < waves; ++i) total += scratch[i];
    return total;
}

// The activation of a gated feed-forward's gate: ACT 0 silu(g) = g / (1 + exp(-g)); ACT 1 the tanh form of gelu,
// 0.5 g (1 + tanh(sqrt(2 / pi) (g + 0.044715 g^3))); ACT 2 max(g, 0).  32-bit.
template <int ACT>
__device__ __forceinline__ float gate_act(float g) {
    if (ACT == 2) return fmaxf(g, 0.f);
    if (ACT == 1) return 0.5f * g * (1.0f + tanhf(0.7978845608028654f * (g + 0.044715f * g * g * g)));
    return g / (1.0f + expf(-g));
}
// The activation of a feed-forward without a gate: ACT 0 relu(x)^2; ACT 1 the exact gelu, x Phi(x) with the normal
// distribution's function.  32-bit.
template <int ACT> __device__ __forceinline__ float plain_act(float x) {
    if (ACT == 1) return 0.5f * x * (1.0f + erff(x * 0.70710678118654752440f));
    const float r = fmaxf(x, 0.f);
    return r * r;
}
// The gate whose branches are clamped: g * sigmoid(slope * g) * (u + 1), g = min(gate, limit), u = clamp(up, -limit, limit).
__device__ __forceinline__ float clamped_glu(float gate, float up, float limit, float slope) {
    const float g = fminf(gate, limit), u = fminf(fmaxf(up, -limit), limit);
    return (g / (1.0f + expf(-slope * g))) * (u + 1.0f);
}
// This wavefront's loads but the last LEFT and all its LDS reads are done, and so are every other wavefront's: behind it the
// block that those loads filled may be read and the block that those reads took from may be filled again.  The compiler does
// not follow loads that go to LDS, so both waits are written out.
template <int LEFT> __device__ __forceinline__ void wide_arrive() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(LEFT) : "memory");
}
// Compute units of the current device, asked for once; -1 when the device does not say.
inline int compute_units() {
    static int units = 0;
    if (units == 0) {
        int device = 0;
        if (hipGetDevice(&device) != hipSuccess ||
            hipDeviceGetAttribute(&units, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || units <= 0)
            units = -1;
    }
    return units;
}
