// Softmax attention of prompt portions on the 32x32 matrix-core tiles of gfx950 (bfloat16) for keys and values of sizes of
// their own, row by row: with a mask rule, a sink, capped scores (see sink_attention.hip, whose kernel serves single tokens,
// short portions and other sizes), and with keys that are two parts -- one a head, one that all heads share.
//
// A workgroup serves one group: consecutive tokens of one request times head_block query heads of one kv head, as 32 NQ
// columns (token = column / head_block).  Its 2 NQ wavefronts are NQ column quarters times two key parities; keys are
// walked in blocks of 64 at absolute multiples of 64, staged once through LDS (two buffers, the next block in flight in
// registers), parity p takes keys 32 p .. 32 p + 31 of a block, and the two are merged through LDS at the end.
//
// Per tile of 32 keys, with v_mfma_f32_32x32x16_bf16 (lane = 32 h + n: A row n, k-slots 8 h .. 8 h + 7; B column n, the same
// k-slots; C column n, rows 8 j + 4 h + r):
//   S^T[key][column]  = K[key][d] . Q^T[d][column]         A from LDS as the rows lie, B = Q in registers
//   O^T[channel][column] += V^T[channel][key] . P^T[key][column]
// registers 8 m .. 8 m + 7 of S^T are the keys 16 m + 8 a + 4 h + r (a = 0, 1): B's layout as they lie, and A wants those
// keys of ONE channel side by side.  The values lie in LDS as rows all the same: ds_read_b64_tr_b16 gives a lane four keys
// of its channel (of 16 lanes, lane i names the i % 4-th four channels of key i / 4 and gets channel i of all four keys).
// The kernel that this one relieves (64 columns, 16x16 tiles: 16 columns a wavefront) reads the LDS twice as often a
// product and transposes values on their way in: 2048 tokens of 16 heads on 4 kv heads of 128 channels in a window of 1024
// 103 us a layer, here 36 (360 TFLOP/s); 1777 tokens in blocks of 1024 89 us, here 35.  What is left is the instructions of
// a tile (see attention_tiles.hip), the triangle's last workgroups, and, with keys in two parts, one workgroup a compute unit
// (91 KB of LDS): 16 heads over the 2048 keys of their own prompt 59 us, where 576 + 512 channels a pair out of one shared
// row took 546.
//
// Rows: paged ([page][kv_head][place][row]) or, SPLIT, contiguous by key: k1[(key * kv_heads + kvh)][k1_row], k2[key][k2_row],
// v[(key * kv_heads + kvh)][v_row].
#define MLR_BF16 1
#include "common.h"

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float floatx16;
typedef short s16x4 __attribute__((ext_vector_type(4)));

#define MASK_ALL 0
#define MASK_WINDOW 1
#define MASK_CHUNK 2
#define BLOCK 64               // keys of a block
#define TILE 32
#define PAGE_IDS 1024          // page ids of a group's keys that are kept in LDS
#define RAISE_BY 8.0f          // base-2 exponent by which a tile must exceed a column's reference maximum

struct PortionArgs {
    const __bf16* q1; long q1_row, q1_head;    // the first channels of a query: q1[m * q1_row + head * q1_head + d]
    const __bf16* q2; long q2_row, q2_head;    // the rest (SPLIT)
    const __bf16* k1; long k1_row;
    const __bf16* k2; long k2_row;
    const __bf16* v; long v_row;
    const int32_t* block_table; const int32_t* slots; const int32_t* positions;
    const int32_t* group_first; const int32_t* group_count;     // null: groups of `tokens` rows from row0 on, `rows` in all
    const float* sink;                         // [q_heads] or null
    __bf16* out; long out_row;                 // out[m * out_row + head * value_dim + c]
    int groups, row0, rows, tokens, key0;      // key0 (SPLIT): the position of the first row of k1, k2 and v
    int max_blocks, page_size, page_shift, q_heads, kv_heads, head_block, head_blocks, mask_kind, mask_size, keep_first;
    float scale, softcap;
};

__device__ __forceinline__ int first_seen(int pos, int kind, int size) {
    if (kind == MASK_WINDOW) return max(0, pos - size + 1);
    if (kind == MASK_CHUNK) return (pos / size) * size;
    return 0;
}

// max(a, b, c) in one instruction (scores are finite or -inf)
__device__ __forceinline__ float max3(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

template <int ND, int NV, int NQ, bool SPLIT>
struct Shape {
    static constexpr int D = 16 * ND, V = 32 * NV, THREADS = 128 * NQ;
    static constexpr int KP = D + 8;           // row pitch of staged keys: 32 lanes' 16-byte reads spread over the banks
    static constexpr int VP = V + 32;          // of values: the four keys of a transposing read in 16 banks each
    static constexpr int KN = BLOCK * 2 * ND / THREADS, VN = BLOCK * 4 * NV / THREADS;      // 16-byte chunks a thread stages
    static constexpr int NO = NV * 16 + 2;     // floats a lane hands over in the merge
    static constexpr size_t kv_bytes = 2 * (size_t)BLOCK * (KP + VP) * sizeof(__bf16);
    static constexpr size_t merge_bytes = NQ * (size_t)NO * 64 * sizeof(float);
    static constexpr size_t ids_bytes = SPLIT ? 0 : PAGE_IDS * sizeof(int32_t);
    static constexpr size_t lds_bytes = ids_bytes + (kv_bytes > merge_bytes ? kv_bytes : merge_bytes);
};

// ND: key channels / 16, of which the last ND2 are the shared part (SPLIT); NV: value channels / 32
template <int ND, int ND2, int NV, int NQ, bool SPLIT>
__global__ __launch_bounds__(128 * NQ, ND > 8 && NQ == 2 ? 1 : 2) void portion_attention_kernel(PortionArgs a) {
    using S = Shape<ND, NV, NQ, SPLIT>;
    constexpr int V = S::V, KP = S::KP, VP = S::VP, THREADS = S::THREADS, KN = S::KN, VN = S::VN, D1 = 16 * (ND - ND2);
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
    int32_t* page_lds = reinterpret_cast<int32_t*>(lds_raw);
    __bf16* k_lds = reinterpret_cast<__bf16*>(lds_raw + S::ids_bytes);              // [2][BLOCK][KP]
    __bf16* v_lds = k_lds + 2 * BLOCK * KP;                                          // [2][BLOCK][VP]
    float* merge_lds = reinterpret_cast<float*>(lds_raw + S::ids_bytes);

    // the workgroups of a kv head, which read the same rows, to the same XCD; a prompt's last groups, the longest, first
    const int total = gridDim.x * gridDim.y;
    int lin = blockIdx.x + gridDim.x * blockIdx.y;
    if (total % 8 == 0) lin = (lin % 8) * (total / 8) + lin / 8;
    const int grp = a.groups - 1 - lin % (int)gridDim.x, part = lin / gridDim.x;
    const int kvh = part / a.head_blocks, hb = part % a.head_blocks, hg = a.q_heads / a.kv_heads, P = a.page_size;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n = lane & 31, h = lane >> 5;
    const int cq = wave % NQ, kp = wave / NQ;
    const int row0 = a.group_first != nullptr ? a.group_first[grp] : a.row0 + grp * a.tokens;
    const int ntok = a.group_first != nullptr ? a.group_count[grp] : min(a.tokens, a.rows - grp * a.tokens);
    const int slot = a.slots[row0], pos0 = a.positions[row0];
    const int lo = first_seen(pos0, a.mask_kind, a.mask_size), ke = pos0 + ntok;     // the group's keys: lo .. ke - 1

    // this wavefront's tokens and this lane's column
    const int tf = 32 * cq / a.head_block, tl = min(ntok - 1, (32 * cq + 31) / a.head_block);
    const bool wave_active = tf < ntok;
    const int wave_first_kend = pos0 + tf + 1, wave_hi = wave_active ? pos0 + tl + 1 : 0;
    const int wave_lo = first_seen(pos0 + tf, a.mask_kind, a.mask_size);
    const int wave_last_lo = wave_active ? first_seen(pos0 + tl, a.mask_kind, a.mask_size) : 0;
    const int c = 32 * cq + n, tok = c / a.head_block, hi = hb * a.head_block + c % a.head_block;
    const bool col_ok = tok < ntok && hi < hg;
    const int kend = col_ok ? pos0 + tok + 1 : 0, kbegin = first_seen(pos0 + tok, a.mask_kind, a.mask_size);
    const int head = kvh * hg + (hi < hg ? hi : 0), m_row = row0 + (tok < ntok ? tok : 0);
    const bf16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
    bf16x8 qf[ND];
#pragma unroll
    for (int st = 0; st < ND; ++st) {
        const __bf16* p = st < ND - ND2 ? a.q1 + (size_t)m_row * a.q1_row + (size_t)head * a.q1_head + 16 * st + 8 * h
                                        : a.q2 + (size_t)m_row * a.q2_row + (size_t)head * a.q2_head + 16 * (st - (ND - ND2)) + 8 * h;
        const bf16x8 x = *reinterpret_cast<const bf16x8*>(p);
        qf[st] = col_ok ? x : zero8;
    }
    float m_ref = -INFINITY, l_run = 0.f;
    floatx16 o[NV];
#pragma unroll
    for (int db = 0; db < NV; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[db][i] = 0.f;

    // the blocks: those of the kept first keys, then those from the range's first (number i lies at block i, or i + gap)
    int kept = (min(a.keep_first, ke) + BLOCK - 1) / BLOCK;
    const int gap = max(0, lo / BLOCK - kept);
    if (gap == 0) kept = 0;
    const int b_first = kept > 0 || a.keep_first > 0 ? 0 : lo / BLOCK, b_end = (ke + BLOCK - 1) / BLOCK;
    const int skip = b_first > 0 ? 0 : gap;                         // (without kept keys the walk starts behind the gap)
    const int blocks = b_end - b_first - skip;
    auto block_at = [&](int i) { return b_first + i + (i >= kept ? skip : 0); };
    bool all_mapped = true;
    const int lead_pages = SPLIT ? 0 : (kept * BLOCK + P - 1) >> a.page_shift;       // page ids: the kept blocks', then the others'
    const int main_block = b_first + kept + skip, main_page = SPLIT ? 0 : (main_block * BLOCK) >> a.page_shift;
    if (!SPLIT) {
        const int32_t* table = a.block_table + (size_t)slot * a.max_blocks;
        const int n_pages = min(PAGE_IDS, lead_pages + ((ke + P - 1) >> a.page_shift) - main_page);
        int mine = 1;
        for (int i = tid; i < n_pages; i += THREADS) {
            const int blk = i < lead_pages ? i : main_page + i - lead_pages;
            const int id = blk < a.max_blocks ? table[blk] : -1;
            page_lds[i] = id;
            mine &= id >= 0 ? 1 : 0;
        }
        all_mapped = __syncthreads_and(mine) != 0;
    }

    // A thread stages the same places of every block.  Loads are never behind a branch (addresses are clamped, and values
    // that must read as zero are zeroed on their way to LDS).
    int k_key[KN], k_ch[KN], v_key[VN], v_ch[VN];
#pragma unroll
    for (int i = 0; i < KN; ++i) k_key[i] = (tid + THREADS * i) / (2 * ND), k_ch[i] = (tid + THREADS * i) % (2 * ND) * 8;
#pragma unroll
    for (int i = 0; i < VN; ++i) v_key[i] = (tid + THREADS * i) / (4 * NV), v_ch[i] = (tid + THREADS * i) % (4 * NV) * 8;
    struct Staged {
        bf16x8 k[KN], v[VN];
        unsigned ok;             // bit i: the key of value chunk i is written and mapped
        bool whole;
    };
    auto row_of = [&](int key, bool& ok) -> long long {              // row of k1 and v (SPLIT: the key's row, heads side by side)
        if (SPLIT) {
            ok = key < ke;
            return (long long)(max(min(key, ke - 1), a.key0) - a.key0) * a.kv_heads + kvh;
        }
        const int blk = key >> a.page_shift;
        const int idx = key < kept * BLOCK ? blk : lead_pages + blk - main_page;
        const int raw = page_lds[min(max(idx, 0), PAGE_IDS - 1)];
        const int id = key < ke ? raw : -1;
        ok = id >= 0;
        return ((long long)max(id, 0) * a.kv_heads + kvh) * P + (key & (P - 1));
    };
    auto fetch = [&](int blk, Staged& st) {
        const int tb = blk * BLOCK;
        st.whole = all_mapped && tb + BLOCK <= ke;
        unsigned bits = 0;
        bool ok;
#pragma unroll
        for (int i = 0; i < KN; ++i) {
            const int key = tb + k_key[i];
            const long long r = row_of(key, ok);
            const __bf16* p = a.k1 + r * a.k1_row + k_ch[i];
            if (SPLIT) p = k_ch[i] < D1 ? p : a.k2 + (long long)(max(min(key, ke - 1), a.key0) - a.key0) * a.k2_row + (k_ch[i] - D1);
            st.k[i] = *reinterpret_cast<const bf16x8*>(p);
        }
#pragma unroll
        for (int i = 0; i < VN; ++i) {
            const long long r = row_of(tb + v_key[i], ok);
            st.v[i] = *reinterpret_cast<const bf16x8*>(a.v + r * a.v_row + v_ch[i]);
            bits |= (ok ? 1u : 0u) << i;
        }
        st.ok = bits;
    };
    auto stash = [&](int buf, const Staged& st) {
#pragma unroll
        for (int i = 0; i < KN; ++i) *reinterpret_cast<bf16x8*>(k_lds + buf * BLOCK * KP + k_key[i] * KP + k_ch[i]) = st.k[i];
#pragma unroll
        for (int i = 0; i < VN; ++i)
            *reinterpret_cast<bf16x8*>(v_lds + buf * BLOCK * VP + v_key[i] * VP + v_ch[i]) = st.whole || ((st.ok >> i) & 1) ? st.v[i] : zero8;
    };

    const bool capped = a.softcap > 0.f;
    const float scale2 = a.scale * 1.44269504088896340736f;            // scores in the base-2 domain
    const float cap2 = a.softcap * 1.44269504088896340736f, slope = capped ? 2.0f * scale2 / a.softcap : 0.f;
    const float c2 = capped ? 1.0f : scale2;
    auto compute = [&](int blk, int buf) {
        const int tb = blk * BLOCK + TILE * kp;
        if (!wave_active || tb >= wave_hi || (tb + TILE <= wave_lo && tb >= a.keep_first)) return;
        const __bf16* kb = k_lds + buf * BLOCK * KP + (TILE * kp + n) * KP + 8 * h;
        bf16x8 kf[ND];
#pragma unroll
        for (int st = 0; st < ND; ++st) kf[st] = *reinterpret_cast<const bf16x8*>(kb + 16 * st);
        __builtin_amdgcn_sched_barrier(0);
        floatx16 sc;
#pragma unroll
        for (int i = 0; i < 16; ++i) sc[i] = 0.f;
#pragma unroll
        for (int st = 0; st < ND; ++st) sc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[st], qf[st], sc, 0, 0, 0);
        // lane i of a sixteen names key i / 4, channels 4 (i % 4) .. of its sixteen's block
        const __bf16* vb = v_lds + buf * BLOCK * VP + (TILE * kp + 4 * h + ((lane & 15) >> 2)) * VP + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
        bf16x8 vf[NV][2];
#pragma unroll
        for (int db = 0; db < NV; ++db)
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                s16x4 half[2];
#pragma unroll
                for (int s = 0; s < 2; ++s)
                    half[s] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                        (__attribute__((address_space(3))) s16x4*)(vb + (16 * m + 8 * s) * VP + 32 * db));
                vf[db][m] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(half[0], half[1], 0, 1, 2, 3, 4, 5, 6, 7));
            }
        __builtin_amdgcn_sched_barrier(0);
        if (capped)          // c tanh(s / c) = c - 2 c / (1 + e^(2 s / c)); an exponent beyond 32 bits gives c
#pragma unroll
            for (int i = 0; i < 16; ++i)
                sc[i] = cap2 - 2.0f * cap2 * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(sc[i] * slope));
        // a tile that every token of this wavefront sees whole needs no mask
        if (!(tb + TILE <= wave_first_kend && (tb >= wave_last_lo || tb + TILE <= a.keep_first))) {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int key = tb + 8 * (i >> 2) + 4 * h + (i & 3);
                sc[i] = (key >= kbegin || key < a.keep_first) && key < kend ? sc[i] : -INFINITY;
            }
        }
        float mx = max3(max3(sc[0], sc[1], sc[2]), max3(sc[3], sc[4], sc[5]), max3(sc[6], sc[7], sc[8]));
        mx = max3(mx, max3(sc[9], sc[10], sc[11]), max3(sc[12], sc[13], sc[14]));
        mx = fmaxf(mx, sc[15]) * c2;                                   // c2 > 0
        if (__builtin_amdgcn_ballot_w64(mx > m_ref + RAISE_BY) != 0) {
            const float full = xor_max<32>(mx);     // the column's maximum in this tile
            if (full > m_ref + RAISE_BY) {
                const float corr = __builtin_amdgcn_exp2f(m_ref - full);      // -inf - finite: 0
                l_run *= corr;
#pragma unroll
                for (int db = 0; db < NV; ++db)
#pragma unroll
                    for (int i = 0; i < 16; ++i) o[db][i] *= corr;
                m_ref = full;
            }
        }
        const float m_use = fmaxf(m_ref, -1e30f);       // a column with no key yet: exp2(-inf - finite) = 0, not NaN
        const bf16x2 ones = {(__bf16)1.0f, (__bf16)1.0f};
        bf16x8 pf[2];
        float psum = 0.f;
#pragma unroll
        for (int m = 0; m < 2; ++m) {
#pragma unroll
            for (int e = 0; e < 8; ++e) pf[m][e] = (__bf16)__builtin_amdgcn_exp2f(fmaf(sc[8 * m + e], c2, -m_use));
#pragma unroll
            for (int e = 0; e < 8; e += 2) psum = __builtin_amdgcn_fdot2_f32_bf16(bf16x2{pf[m][e], pf[m][e + 1]}, ones, psum, false);
        }
        l_run += psum;
#pragma unroll
        for (int db = 0; db < NV; ++db)
#pragma unroll
            for (int m = 0; m < 2; ++m) o[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[db][m], pf[m], o[db], 0, 0, 0);
    };
    // One barrier a block suffices with two buffers: the second write of a buffer comes behind the barrier that follows
    // every wavefront's read of it.
    {
        Staged st;
        fetch(block_at(0), st);
        for (int i = 0; i < blocks; ++i) {
            stash(i & 1, st);
            fetch(block_at(min(i + 1, blocks - 1)), st);
            __syncthreads();
            compute(block_at(i), i & 1);
        }
    }

    // the two key parities; the sink; the division
    l_run = xor_sum<32>(l_run);
    __syncthreads();
    float* mine = merge_lds + (size_t)cq * S::NO * 64 + lane;
    if (kp == 1) {
#pragma unroll
        for (int db = 0; db < NV; ++db)
#pragma unroll
            for (int i = 0; i < 16; ++i) mine[(db * 16 + i) * 64] = o[db][i];
        mine[(NV * 16) * 64] = m_ref;
        mine[(NV * 16 + 1) * 64] = l_run;
    }
    __syncthreads();
    if (kp != 0 || !col_ok) return;
    const float m1 = mine[(NV * 16) * 64], l1 = mine[(NV * 16 + 1) * 64];
    const float sink2 = a.sink != nullptr ? a.sink[head] * 1.44269504088896340736f : -INFINITY;
    const float top = fmaxf(fmaxf(m_ref, m1), sink2);
    const float w0 = m_ref > -INFINITY ? __builtin_amdgcn_exp2f(m_ref - top) : 0.f;
    const float w1 = m1 > -INFINITY ? __builtin_amdgcn_exp2f(m1 - top) : 0.f;
    const float l = l_run * w0 + l1 * w1 + (a.sink != nullptr ? __builtin_amdgcn_exp2f(sink2 - top) : 0.f);
    const float inv = l != 0.f ? 1.f / l : 0.f;                        // (a NaN sum must show)
    __bf16* dst = a.out + (size_t)m_row * a.out_row + (size_t)head * V;
#pragma unroll
    for (int db = 0; db < NV; ++db)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            bf16x4 w4;
#pragma unroll
            for (int r = 0; r < 4; ++r) w4[r] = (__bf16)((o[db][4 * j + r] * w0 + mine[(db * 16 + 4 * j + r) * 64] * w1) * inv);
            *reinterpret_cast<bf16x4*>(dst + 32 * db + 8 * j + 4 * h) = w4;
        }
}

template <int ND, int ND2, int NV, int NQ, bool SPLIT>
static int launch_portion(const PortionArgs& a, hipStream_t stream) {
    constexpr size_t lds = Shape<ND, NV, NQ, SPLIT>::lds_bytes;
    static const hipError_t allowed = hipFuncSetAttribute(reinterpret_cast<const void*>(&portion_attention_kernel<ND, ND2, NV, NQ, SPLIT>),
                                                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (allowed != hipSuccess) return (int)allowed;
    portion_attention_kernel<ND, ND2, NV, NQ, SPLIT><<<dim3(a.groups, a.kv_heads * a.head_blocks), 128 * NQ, lds, stream>>>(a);
    return (int)hipGetLastError();
}

// The cached rows of a key range as the products want them: latent parts side by side, shared key parts side by side.
__global__ __launch_bounds__(256) void latent_rows_kernel(const __bf16* __restrict__ pages, long row, const int32_t* __restrict__ block_table,
                                                          int max_blocks, const int32_t* __restrict__ slots, int m, int page_size,
                                                          int key0, int keys, int rank, int rot, __bf16* __restrict__ latent,
                                                          __bf16* __restrict__ shared) {
    // (a wavefront a row, which looks its page up once: 1777 rows of 576 values 3.7 us; 17 with a lookup for every 16 bytes)
    const int i = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (i >= keys) return;
    const int block = (key0 + i) / page_size;
    const int page = block < max_blocks ? block_table[(size_t)slots[m] * max_blocks + block] : -1;
    const __bf16* src = pages + ((long long)max(page, 0) * page_size + (key0 + i) % page_size) * row;
    for (int d = lane * 8; d < rank + rot; d += 512) {
        vec16 x = *reinterpret_cast<const vec16*>(src + d);
        if (page < 0) x = {{0, 0, 0, 0}};
        *reinterpret_cast<vec16*>(d < rank ? latent + (size_t)i * rank + d : shared + (size_t)i * rot + d - rank) = x;
    }
}

extern "C" {

// Groups of at most `columns` / head_block consecutive tokens of one request each (device vectors); head_block a power of
// two, query heads of one kv head.  key_dim 64 or 128 with as many or 128 value channels; pages of a power of two of at
// least 16 tokens; a group's keys on at most 1024 - 4 pages.  Returns 1 for sizes that are not this kernel's.
int mlr_portion_attention(const void* q, long q_row, const void* k_pages, long k_row, const void* v_pages, long v_row,
                          const int32_t* block_table, int max_blocks, const int32_t* slots, const int32_t* positions,
                          const float* sink, void* out, long out_row, const int32_t* group_first, const int32_t* group_count,
                          int groups, int columns, int head_block, int q_heads, int kv_heads, int key_dim, int value_dim, int page_size,
                          int mask_kind, int mask_size, int keep_first, float softcap, int max_context, float scale, hipStream_t stream) {
    if (groups <= 0) return 0;
    if (q_row % 8 != 0 || k_row % 8 != 0 || v_row % 8 != 0 || out_row % 4 != 0 || page_size < 16 || (page_size & (page_size - 1)) != 0) return 1;
    const long reach = mask_kind == MASK_ALL ? (long)max_context : (long)mask_size + 256 + keep_first;
    if (reach / page_size + 4 > PAGE_IDS) return 1;
    if (kv_heads <= 0 || q_heads % kv_heads != 0 || head_block < 1 || head_block > 32 || (head_block & (head_block - 1)) != 0 ||
        (columns != 64 && columns != 128) || (mask_kind != MASK_ALL && mask_size <= 0) || keep_first < 0 || !(softcap >= 0.f))
        return -1;
    const int hg = q_heads / kv_heads, head_blocks = (hg + head_block - 1) / head_block;
    if ((long)kv_heads * head_blocks > 65535) return -2;
    int shift = 0;
    while ((1 << shift) < page_size) ++shift;
    PortionArgs a{(const __bf16*)q, q_row, key_dim, nullptr, 0, 0, (const __bf16*)k_pages, k_row, nullptr, 0, (const __bf16*)v_pages, v_row,
                  block_table, slots, positions, group_first, group_count, sink, (__bf16*)out, out_row, groups, 0, 0, columns / head_block, 0,
                  max_blocks, page_size, shift, q_heads, kv_heads, head_block, head_blocks, mask_kind, mask_size, keep_first, scale, softcap};
    if (key_dim == 128 && value_dim == 128) return columns == 128 ? launch_portion<8, 0, 4, 4, false>(a, stream) : launch_portion<8, 0, 4, 2, false>(a, stream);
    if (key_dim == 64 && value_dim == 128) return columns == 128 ? launch_portion<4, 0, 4, 4, false>(a, stream) : launch_portion<4, 0, 4, 2, false>(a, stream);
    if (key_dim == 64 && value_dim == 64) return columns == 128 ? launch_portion<4, 0, 2, 4, false>(a, stream) : launch_portion<4, 0, 2, 2, false>(a, stream);
    return 1;
}

// Rows key0 .. key0 + keys - 1 of the request of batch row m.
int mlr_latent_rows(const void* pages, long row, const int32_t* block_table, int max_blocks, const int32_t* slots, int m, int page_size,
                    int key0, int keys, int rank, int rot, void* latent, void* shared, hipStream_t stream) {
    if (keys <= 0) return 0;
    if (rank % 8 != 0 || rot % 8 != 0 || row % 8 != 0 || key0 < 0) return -1;
    latent_rows_kernel<<<(unsigned)((keys + 3) / 4), 256, 0, stream>>>((const __bf16*)pages, row, block_table, max_blocks, slots, m, page_size,
                                                                          key0, keys, rank, rot, (__bf16*)latent, (__bf16*)shared);
    return (int)hipGetLastError();
}

// Batch rows row0 .. row0 + rows - 1, a portion of one request whose first token stands at position pos0, over its keys from
// position key0 on: k1 [keys, heads, 128], k2 [keys, 64], v [keys, heads, 128]; every head has keys and values of its own.
// Returns 1 for sizes that are not this kernel's.
int mlr_portion_attention_split(const void* q1, long q1_row, long q1_head, const void* q2, long q2_row, long q2_head, const void* k1,
                                const void* k2, const void* v, const int32_t* slots, const int32_t* positions, const float* sink, void* out,
                                long out_row, int row0, int rows, int key0, int columns, int heads, int plain_dim, int shared_dim, int value_dim,
                                int mask_kind, int mask_size, float scale, hipStream_t stream) {
    if (rows <= 0) return 0;
    if (plain_dim != 128 || shared_dim != 64 || value_dim != 128 || q1_row % 8 != 0 || q1_head % 8 != 0 || q2_row % 8 != 0 || q2_head % 8 != 0 ||
        out_row % 4 != 0)
        return 1;
    if (heads < 1 || heads > 65535 || (columns != 64 && columns != 128) || (mask_kind != MASK_ALL && mask_size <= 0) || key0 < 0) return -1;
    PortionArgs a{(const __bf16*)q1, q1_row, q1_head, (const __bf16*)q2, q2_row, q2_head, (const __bf16*)k1, plain_dim, (const __bf16*)k2, shared_dim,
                  (const __bf16*)v, value_dim, nullptr, slots, positions, nullptr, nullptr, sink, (__bf16*)out, out_row,
                  (rows + columns - 1) / columns, row0, rows, columns, key0, 0, 16, 4, heads, heads, 1, 1, mask_kind, mask_size, 0, scale, 0.f};
    return columns == 128 ? launch_portion<12, 4, 4, 4, true>(a, stream) : launch_portion<12, 4, 4, 2, true>(a, stream);
}

}  // extern "C"
