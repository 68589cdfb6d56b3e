// Attention for prompt portions on the 32x32 matrix-core tiles of gfx950 (bfloat16 cache and queries).
//
// A workgroup serves one group: consecutive tokens of one request for one kv head, as 32 NQ columns (token,
// head): 32 NQ / g tokens, g = query heads per kv head, NQ = 4 or 2 (the smaller workgroup is for batches
// that would not fill the GPU otherwise).  Keys are walked in blocks of 64 at absolute multiples of 64, brought to LDS once per
// workgroup (two buffers: one multiplied, one on its way); a wavefront owns 32 columns and takes a block's keys 0..31 or 32..63
// (two key parities, merged through LDS at the end) or, head size 128 and NQ = 4, both halves.
//
// Head size 128 (four wavefronts, two workgroups a compute unit): the blocks go to LDS by loads that do not pass registers, and
// the loop over the blocks that a wavefront sees whole has nothing to check.  What bounds it is what a SIMD can issue for a tile
// and how long a tile's chain is (first product, softmax, second product), not memory: per tile 16 matrix instructions (512
// cycles), 49 vector and some 25 scalar ones; counters at 10 000 keys of context (kernel of 237 us): matrix cores 42 % of the
// cycles, LDS 22 %, no bank conflicts.  Measured (16 query heads over 8, pages of 16; the kernel that staged through registers,
// eight wavefronts of 128 columns, in brackets): 2048 tokens 32.7 us with 64 columns (42.5), behind 10 240 keys 201 (232);
// 32 query heads over 8, 2048 tokens behind 8192 keys 292 us with 128 columns (332), 64 over 8, 1501 tokens 56.5 (77); 4096 tokens
// of 16 heads behind 8192 keys 333-351 (448).  A softmax's wavefront goes before the others of its SIMD (`s_setprio`, 3 %): its
// chain is the longer one.  Measured and taken out: wavefronts of the two parities half a turn apart, a barrier at every half, so
// that one multiplies while the other is in its softmax (250 us for 232); four blocks of LDS, three on their way, in
// one workgroup of eight wavefronts (237).
//
// Other head sizes: 4 NQ / 2 wavefronts, staged through registers: a thread stages 32 contiguous bytes per page lookup, blocks
// whose keys are all written are staged without checks.
//
// Per tile of 32 keys, with v_mfma_f32_32x32x16_bf16:
//   S^T[key][column]  = K[key][d] . Q^T[d][column]         A = 32 keys x 16 channels from LDS, B = Q (registers)
//   O^T[d][column]   += V^T[d][key] . P^T[key][column]     A = 32 channels x 16 keys from LDS (values are
//                                                           cached transposed), B = the probabilities, which
//                                                           sit in B's register layout already
// Register layouts of that instruction, lane = 32 h + n: A holds row n, k-slots 8 h .. 8 h + 7; B holds
// column n, the same k-slots; C holds column n, rows 8 j + 4 h + r for j, r in 0..3 (register 4 j + r).
// So registers 8 m .. 8 m + 7 of S^T are the rows 16 m + 8 a + 4 h + r (a = 0, 1) of the tile.  Staged through registers, row =
// key, and the values are laid out in LDS with those keys side by side (position 16 m + 8 h + 4 a + r); head size 128, the row
// is the key with bits 2 and 3 swapped, and the registers are neighbouring keys.  Either way one 16-byte read gives the
// matching A operand.
//
// Softmax in the base-2 domain, 32-bit.  A column's reference is the maximum of one of its tiles and is only raised when the
// probabilities that a lane makes of a tile sum up to more than 2^20 (each then stays below that, as far from overflow as a value below
// 2^107 leaves it; a probability has its eight bits at any size, and the quotient at the end does not depend on the reference): raising
// it means taking the tile's exponentials again and rescaling 64 accumulators for all 32 columns of a wavefront, of which some one
// would need it in many tiles otherwise.  From 2^8 on, scores that vary little gain as much but scores of a standard deviation
// of 4 (before the base-2 scale) lose: against a maximum taken in every tile, 16 heads of 64 channels, 1000 tokens 17.6 us at a deviation
// of 1, 19.3 at 4; with 2^8 17.7 and 22.3, now 17.7 and 17.8; heads of 128 behind 4000 keys 47.0 and 54.4, 45.1 and 59.7, now 44.9 and 45.2.
// The sum is there anyway, so most tiles never take a maximum: 49 vector instructions a tile for 58, and the exponentials need not
// wait for it (12 321 tokens of 16 heads in portions of 2048: 0.6 % of the whole prompt).  The decision is taken per
// column from the column's own scores, so a column's arithmetic does not depend on its neighbours.  It does depend on the
// workgroup's width where that is two ways over the keys: with head size 128 a column of 128 has one reference and one chain for both
// halves of its blocks, a column of 64 two that are merged, so the two round their probabilities otherwise (as key ranges do, below;
// both are the step's choice, by its number of rows).
// The sum of a column's probabilities is taken over their bfloat16 roundings, the values that the second
// product multiplies.
//
// Key splits (max_splits > 1), for a step whose groups alone would not fill the GPU (a short portion of a
// long context): workgroup (group, kv head, split s) takes the keys [s * split_keys, (s + 1) * split_keys),
// split_keys a multiple of 64, and leaves its columns' (values, maximum, sum) unnormalised in `partial`;
// `tiles_combine_kernel` merges a column's splits in ascending order.
//
// Not handled here (the caller uses the other kernels): head sizes above 128, page sizes that are no power
// of two, groups whose keys span more than PAGE_IDS pages.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float floatx16;

#define BLOCK_KEYS 64
#define TILE_KEYS 32
#define PAGE_IDS 2048
#define VPITCH (BLOCK_KEYS + 8)        // elements per channel row of a staged block of values
#define RAISE_AT 1048576.0f            // sum of a lane's probabilities in a tile from which the reference may be raised

struct TileArgs {
    const __bf16* q;             // [M, q_heads, head_dim]
    const __bf16* k_pages;       // [pages][kv_heads][page_size][head_dim]
    const __bf16* v_pages;       // [pages][kv_heads][head_dim][page_size]
    const int32_t* block_table;  // [slots, max_blocks]
    const int32_t* slots;        // [M]
    const int32_t* positions;    // [M]
    __bf16* out;                 // [M, q_heads, head_dim]
    const int32_t* group_row0;   // [groups] first batch row of a group
    const int32_t* group_ntok;   // [groups] its tokens (consecutive rows of one request)
    float* partial;              // [M, q_heads, max_splits, head_dim + 4] when max_splits > 1 (16-byte aligned)
    int groups, max_blocks, q_heads, kv_heads, head_dim, page_size, page_shift, window, split_keys, max_splits;
    float scale;
    int all_resident;            // the grid fits the GPU at once (two workgroups of 64 columns a compute unit)
    int single;                  // host: the caller's `pairing`; kernel: 1 every workgroup takes one group, 0 two (group i and group groups - 1 - i)
};

// DIRECT (head size 128): blocks go straight from memory to LDS (see `tile_group`).
template <int ND, int NQ>
struct TileShape {
    static constexpr bool DIRECT = ND == 8;
    static constexpr int TILES = DIRECT && NQ == 4 ? 2 : 1;   // tiles of a block that a wavefront takes
    static constexpr int PARITIES = 2 / TILES;
    static constexpr int D = 16 * ND;
    static constexpr int DB = (ND + 1) / 2;               // blocks of 32 channels
    static constexpr int THREADS = 64 * NQ * PARITIES;
    static constexpr int KPITCH = DIRECT ? D : D + 8;     // elements per key row of a staged block of keys
    static constexpr int KBUF = BLOCK_KEYS * KPITCH;      // elements
    static constexpr int VBUF = DIRECT ? BLOCK_KEYS * D : 32 * DB * VPITCH;
    static constexpr int LOADS = 16 / (THREADS / 64);           // DIRECT: a wavefront's loads of 1 KB for a block's keys, and as many for its values
    static constexpr int KSTEP = THREADS / ND;            // keys that the workgroup stages per pass
    static constexpr int VSTEP = THREADS / D;             // 16-key groups of values per pass
    static constexpr int K_PASSES = (BLOCK_KEYS + KSTEP - 1) / KSTEP;
    static constexpr int V_PASSES = (BLOCK_KEYS / 16 + VSTEP - 1) / VSTEP;
    static constexpr int NO = DB * 16 + 2;                // floats a lane hands over in the merge
    static constexpr size_t kv_bytes = 2 * (size_t)(KBUF + VBUF) * sizeof(__bf16);
    static constexpr size_t merge_bytes = NQ * (size_t)NO * 64 * sizeof(float);
    static constexpr size_t lds_bytes = PAGE_IDS * sizeof(int32_t) + (kv_bytes > merge_bytes ? kv_bytes : merge_bytes);
};

// This wavefront's loads to LDS and its LDS reads are done, and so are every other wavefront's (the compiler does not follow
// loads that go to LDS).
__device__ __forceinline__ void tile_arrive() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <int ND, int NQ>
__device__ __forceinline__ void tile_group(const TileArgs& a, int grp, int kvh, int split, unsigned char* lds_raw) {
    using S = TileShape<ND, NQ>;
    constexpr int D = S::D, DB = S::DB, KPITCH = S::KPITCH, THREADS = S::THREADS;
    int32_t* page_lds = reinterpret_cast<int32_t*>(lds_raw);
    __bf16* k_lds = reinterpret_cast<__bf16*>(lds_raw + PAGE_IDS * sizeof(int32_t));
    __bf16* v_lds = k_lds + 2 * S::KBUF;
    float* merge_lds = reinterpret_cast<float*>(lds_raw + PAGE_IDS * sizeof(int32_t));

    const int P = a.page_size, pshift = a.page_shift;
    const int g = a.q_heads / a.kv_heads, cap = (32 * NQ) / g;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = lane & 31, h = lane >> 5;
    const int cq = wave % NQ, kp = wave / NQ;                  // column quarter, key parity
    const int row0 = a.group_row0[grp], ntok = min(a.group_ntok[grp], cap);
    const int slot = a.slots[row0], pos0 = a.positions[row0];
    const int lo = a.window > 0 ? max(0, pos0 + 1 - a.window) : 0;    // first key any token of the group sees
    const int ke = pos0 + ntok;                                      // one past the last
    // the keys of this workgroup: all of them, or those of its split
    const bool splitting = a.max_splits > 1;
    const int lo_s = splitting ? max(lo, split * a.split_keys) : lo;
    const int ke_s = splitting ? min(ke, (split + 1) * a.split_keys) : ke;
    if (lo_s >= ke_s) return;                                        // no column of the group sees this split

    // this wavefront's tokens
    const int tf = (32 * cq) / g;
    const int tl = min(ntok - 1, (32 * cq + 31) / g);
    const bool wave_active = tf < ntok;
    const int wave_first_kend = pos0 + tf + 1;
    const int wave_hi = wave_active ? pos0 + tl + 1 : 0;
    const int wave_lo = a.window > 0 ? max(0, pos0 + tf + 1 - a.window) : 0;
    const int wave_last_kbegin = a.window > 0 ? max(0, pos0 + tl + 1 - a.window) : 0;

    // this lane's column
    const int c = 32 * cq + n;
    const int tok = c / g, hh = c % g;
    const bool col_valid = tok < ntok;
    const int kend_c = col_valid ? pos0 + tok + 1 : 0;
    const int kbegin_c = a.window > 0 ? max(0, kend_c - a.window) : 0;
    const bf16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
    bf16x8 qf[ND];
    {
        const __bf16* qrow = a.q + ((size_t)(row0 + (col_valid ? tok : 0)) * a.q_heads + kvh * g + hh) * D + 8 * h;
#pragma unroll
        for (int st = 0; st < ND; ++st) {
            const bf16x8 v = *reinterpret_cast<const bf16x8*>(qrow + 16 * st);
            qf[st] = col_valid ? v : zero8;
        }
    }
    float m_ref = -INFINITY, l_run = 0.f;
    float m_neg = 1e30f;             // -m_ref as it is added (a column with no key yet: exp2(-inf + finite) = 0, not NaN; the first key
                                     // that it sees gets exp2(1e30) = inf, a sum beyond RAISE_AT, which sets the reference)
    floatx16 o[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[db][i] = 0.f;

    // page ids of the group's key range, so that a block's loads do not wait for a load of the table
    const int blk_begin = lo_s / BLOCK_KEYS, blk_end = (ke_s + BLOCK_KEYS - 1) / BLOCK_KEYS;
    const int first_page = (blk_begin * BLOCK_KEYS) >> pshift;
    const int32_t* table = a.block_table + (size_t)slot * a.max_blocks;
    bool all_mapped;                                  // every page of the key range is there (none given back, none missing)
    {
        const int n_pages = min(PAGE_IDS, ((ke_s + P - 1) >> pshift) - first_page);
        // (an entry beyond the request's row of the table is no page, like an entry of -1)
        int mine_mapped = 1;
        for (int i = threadIdx.x; i < n_pages; i += THREADS) {
            const int id = first_page + i < a.max_blocks ? table[first_page + i] : -1;
            page_lds[i] = id;
            mine_mapped &= id >= 0 ? 1 : 0;
        }
        all_mapped = __syncthreads_and(mine_mapped) != 0;
    }

    const float c2 = a.scale * 1.44269504088896340736f;     // scores in the base-2 domain: one v_exp_f32 each
    // a tile's scores -> probabilities (as B operands), updating the column's reference, sum and accumulators
    auto softmax = [&](auto& sc, int tb, bool interior, auto& pf) {
        constexpr int T = sizeof(sc) / sizeof(sc[0]);         // tiles, one behind the other
        if (!interior) {
#pragma unroll
            for (int t = 0; t < T; ++t)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int key = tb + 32 * t + (S::DIRECT ? 16 * (i >> 3) + 8 * h + (i & 7) : 8 * (i >> 2) + 4 * h + (i & 3));
                    sc[t][i] = (key >= kbegin_c && key < kend_c) ? sc[t][i] : -INFINITY;
                }
        }
        // (the sum is taken over the probabilities as the second product sees them, rounded to bfloat16, two
        // at a time: v_dot2c_f32_bf16 with a pair of ones, half the instructions of single additions)
        const bf16x2 ones = {(__bf16)1.0f, (__bf16)1.0f};
        float psum;
        auto probabilities = [&]() {
            float sum[2] = {0.f, 0.f};                        // (two chains: each addition waits for the one before it)
#pragma unroll
            for (int t = 0; t < T; ++t)
#pragma unroll
                for (int m = 0; m < 2; ++m) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) pf[t][m][e] = (__bf16)__builtin_amdgcn_exp2f(fmaf(sc[t][8 * m + e], c2, m_neg));
#pragma unroll
                    for (int e = 0; e < 8; e += 2)
                        sum[m] = __builtin_amdgcn_fdot2_f32_bf16(bf16x2{pf[t][m][e], pf[t][m][e + 1]}, ones, sum[m], false);
                }
            psum = sum[0] + sum[1];
        };
        probabilities();
        // A lane's sum beyond RAISE_AT says that some score may lie too far above the reference: only then the maximum is taken (in
        // every tile it would be nine instructions, a wait for the first product's last result before anything else can begin, and a
        // branch in front of the exponentials).  Both lanes of a column see both sums, so a column is raised by its own scores.
        if (__builtin_amdgcn_ballot_w64(psum > RAISE_AT) != 0) {
            const float most = fmaxf(psum, __shfl_xor(psum, 32, 64));
            float mx = sc[0][0];
#pragma unroll
            for (int t = 0; t < T; ++t)
#pragma unroll
                for (int i = 0; i < 16; ++i) mx = fmaxf(mx, sc[t][i]);
            const float full = fmaxf(mx, __shfl_xor(mx, 32, 64)) * c2;        // the column's maximum in this tile (c2 > 0)
            if (most > RAISE_AT && full > m_ref) {
                const float corr = __builtin_amdgcn_exp2f(m_ref - full);      // -inf - finite: 0
                l_run *= corr;
#pragma unroll
                for (int db = 0; db < DB; ++db)
#pragma unroll
                    for (int i = 0; i < 16; ++i) o[db][i] *= corr;
                m_ref = full;
                m_neg = -fmaxf(full, -1e30f);
            }
            probabilities();
        }
        l_run += psum;
    };

    auto compute = [&](int blk, int buf) {
        const int tb = blk * BLOCK_KEYS + TILE_KEYS * kp;
        if (!wave_active || tb >= wave_hi || tb + TILE_KEYS <= wave_lo) return;      // nothing for this wavefront
        const __bf16* kb = k_lds + buf * S::KBUF + (TILE_KEYS * kp + n) * KPITCH + 8 * h;
        const __bf16* vb = v_lds + buf * S::VBUF + n * VPITCH + TILE_KEYS * kp + 8 * h;
        // all operands of a product are asked for before its first instruction, and the values before
        // the softmax: the LDS answers while the matrix cores and the softmax are busy
        bf16x8 kf[ND];
#pragma unroll
        for (int st = 0; st < ND; ++st) kf[st] = *reinterpret_cast<const bf16x8*>(kb + 16 * st);
        __builtin_amdgcn_sched_barrier(0);
        floatx16 sc[1];
#pragma unroll
        for (int i = 0; i < 16; ++i) sc[0][i] = 0.f;
#pragma unroll
        for (int st = 0; st < ND; ++st) sc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[st], qf[st], sc[0], 0, 0, 0);
        bf16x8 vf[DB][2];
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int m = 0; m < 2; ++m) vf[db][m] = *reinterpret_cast<const bf16x8*>(vb + 32 * db * VPITCH + 16 * m);
        __builtin_amdgcn_sched_barrier(0);
        // a tile that every token of this wavefront sees whole needs no mask (all but the last few)
        const bool interior = tb + TILE_KEYS <= wave_first_kend && tb >= wave_last_kbegin;
        bf16x8 pf[1][2];
        softmax(sc, tb, interior, pf);
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int m = 0; m < 2; ++m)
                o[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[db][m], pf[0][m], o[db], 0, 0, 0);
    };

    if constexpr (S::DIRECT) {
        // A block of 64 keys is 16 KB of keys and 16 KB of values, 32 loads of 1 KB that go from memory to LDS without passing
        // registers (`buffer_load_dwordx4 .. lds`: a lane's 16 bytes from an address of its own, the 64 lanes' side by side in
        // LDS); a wavefront's share is one run of 16 keys, so lies in one page.  What is permuted is which lane asks for what:
        // row r of the block (row r of a tile of the first product) is the key with bits 2 and 3 of r swapped, so that a
        // lane's probabilities are eight neighbouring keys and the values can stay as the cache holds them, and 16-byte
        // piece p of row r lies at place p ^ (r & 15); of a channel's two pieces of eight keys the first lies second
        // where bits 2 and 3 of the channel differ.  Lanes that the LDS serves together then read different banks.
        // While one block is multiplied the next is on its way; the loop's two turns have a buffer each, so that an operand's
        // address is a register that does not change and a constant.
        constexpr int LOADS = S::LOADS, BLOCK = S::KBUF + S::VBUF, T = S::TILES;
        uint32_t k_at[LOADS], v_at[LOADS];
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int r = 4 * i + (lane >> 4), d = 32 * i + (lane >> 1);        // of the run
            const int key = (r & 3) | (r & 4) << 1 | (r & 8) >> 1;
            k_at[i] = (uint32_t)(key * D + 8 * ((lane & 15) ^ r)) * 2u;
            v_at[i] = (uint32_t)(d * P + 8 * ((lane & 1) ^ ((d >> 2 ^ d >> 3) & 1))) * 2u;
        }
        const uint32_t head_bytes = (uint32_t)P * D * 2, page_bytes = head_bytes * a.kv_heads;   // (page strides below 2^24 elements)
        const unsigned char* k_head = reinterpret_cast<const unsigned char*>(a.k_pages) + (size_t)kvh * head_bytes;
        const unsigned char* v_head = reinterpret_cast<const unsigned char*>(a.v_pages) + (size_t)kvh * head_bytes;
        auto page_of = [&](int blk) {                     // (behind the range, or a page that is not there: page 0, cleared below)
            const int key0 = blk * BLOCK_KEYS + 16 * wave;
            return __builtin_amdgcn_readfirstlane(key0 < ke ? max(page_lds[min((key0 >> pshift) - first_page, PAGE_IDS - 1)], 0) : 0);
        };
        auto ask = [&](int blk, int page, int buf) {
            const int in_page = (blk * BLOCK_KEYS + 16 * wave) & (P - 1);
            const uint64_t at = (uint64_t)(uint32_t)page * page_bytes;
            const auto kr = __builtin_amdgcn_make_buffer_rsrc((void*)(k_head + at), 0, (int)head_bytes, 0x00027000);
            const auto vr = __builtin_amdgcn_make_buffer_rsrc((void*)(v_head + at), 0, (int)head_bytes, 0x00027000);
            __bf16* to = k_lds + buf * BLOCK + wave * LOADS * 512;
#pragma unroll
            for (int i = 0; i < LOADS; ++i)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(kr, (__attribute__((address_space(3))) void*)(to + i * 512), 16, (int)k_at[i], in_page * (D * 2), 0, 0);
#pragma unroll
            for (int i = 0; i < LOADS; ++i)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(vr, (__attribute__((address_space(3))) void*)(to + S::KBUF + i * 512), 16, (int)v_at[i], in_page * 2, 0, 0);
        };
        // Values of keys that are not written yet, or of a page that was given back (behind a window), count as zero: their
        // probability is zero, but zero times whatever the memory holds need not be.
        auto clear_values = [&](int blk, int buf) {
            __bf16* vb = k_lds + buf * BLOCK + S::KBUF;
            for (int piece = threadIdx.x; piece < S::VBUF / 8; piece += THREADS) {
                const int m = piece / (2 * D), d = piece / 2 % D, half = (piece & 1) ^ ((d >> 2 ^ d >> 3) & 1);
                const int key0 = blk * BLOCK_KEYS + 16 * m;
                const bool there = key0 < ke && page_lds[min((key0 >> pshift) - first_page, PAGE_IDS - 1)] >= 0;
                if (there && key0 + 8 * half + 8 <= ke) continue;
                bf16x8 v = *reinterpret_cast<const bf16x8*>(vb + piece * 8);
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (!there || key0 + 8 * half + e >= ke) v[e] = (__bf16)0.f;
                *reinterpret_cast<bf16x8*>(vb + piece * 8) = v;
            }
        };
        // (kept in registers: left to itself the compiler adds them up again for every tile)
        const uint32_t kv_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)k_lds;      // (a byte of LDS)
        uint32_t k_row[ND], v_row;
#pragma unroll
        for (int st = 0; st < ND; ++st) {
            k_row[st] = kv_base + (uint32_t)(((TILE_KEYS * kp + n) * D + 8 * ((2 * st + h) ^ (n & 15))) * 2);
            asm volatile("" : "+v"(k_row[st]));
        }
        v_row = kv_base + (uint32_t)((S::KBUF + TILE_KEYS * kp * D + n * 16 + 8 * (h ^ ((n >> 2 ^ n >> 3) & 1))) * 2);
        asm volatile("" : "+v"(v_row));
        auto operand = [&](uint32_t at, int plus) { return *(__attribute__((address_space(3))) const bf16x8*)(uintptr_t)(at + (uint32_t)plus); };
        auto tile = [&](int tb, bool interior, auto buf_) {
            constexpr int buf = decltype(buf_)::value;
            // all operands of a product are asked for before its first instruction, and the values before the softmax; the
            // products of two tiles are chains of their own, side by side
            bf16x8 kf[T][ND], vf[T][DB][2], pf[T][2];
#pragma unroll
            for (int st = 0; st < ND; ++st)
#pragma unroll
                for (int t = 0; t < T; ++t) kf[t][st] = operand(k_row[st], buf * BLOCK * 2 + t * TILE_KEYS * D * 2);
            __builtin_amdgcn_sched_barrier(0);
            floatx16 sc[T];
#pragma unroll
            for (int t = 0; t < T; ++t)
#pragma unroll
                for (int i = 0; i < 16; ++i) sc[t][i] = 0.f;
#pragma unroll
            for (int st = 0; st < ND; ++st)
#pragma unroll
                for (int t = 0; t < T; ++t) sc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[t][st], qf[st], sc[t], 0, 0, 0);
            auto values = [&](int t) {
#pragma unroll
                for (int m = 0; m < 2; ++m)
#pragma unroll
                    for (int db = 0; db < DB; ++db) vf[t][db][m] = operand(v_row, buf * BLOCK * 2 + ((2 * t + m) * 16 * D + 32 * 16 * db) * 2);
                __builtin_amdgcn_sched_barrier(0);
            };
            values(0);
            __builtin_amdgcn_s_setprio(1);
            softmax(sc, tb, interior, pf);
            __builtin_amdgcn_s_setprio(0);
#pragma unroll
            for (int t = 0; t < T; ++t) {
                if (t + 1 < T) values(t + 1);             // (not before: both tiles' values beside the scores are too many registers)
#pragma unroll
                for (int m = 0; m < 2; ++m)
#pragma unroll
                    for (int db = 0; db < DB; ++db) o[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[t][db][m], pf[t][m], o[db], 0, 0, 0);
            }
        };
        const bool whole_range = all_mapped && a.window <= 0;
        ask(blk_begin, page_of(blk_begin), 0);
        int page = page_of(blk_begin + 1);
        // The blocks that this wavefront sees whole, in pairs, as long as three more follow (the page of the block after next is
        // looked up, and all keys of every block but the last are there): nothing to check.
        int blk = blk_begin;
        if (whole_range && wave_active) {
            const int fast_end = min(blk_end - 3, wave_first_kend / BLOCK_KEYS);
            int key2 = (blk_begin + 2) * BLOCK_KEYS + 16 * wave;                // this wavefront's run of the block after next
            auto fast = [&](auto buf_) {
                tile_arrive();
                ask(blk + 1, page, decltype(buf_)::value ^ 1);
                const int after = page_lds[(key2 >> pshift) - first_page];
                tile(0, true, buf_);
                page = __builtin_amdgcn_readfirstlane(after);
                key2 += BLOCK_KEYS;
                ++blk;
            };
            while (blk + 2 <= fast_end) {
                fast(std::integral_constant<int, 0>{});
                fast(std::integral_constant<int, 1>{});
            }
        }
        auto turn = [&](auto buf_) {
            constexpr int buf = decltype(buf_)::value;
            tile_arrive();                                // the block is there, and everyone is done with the one before
            if (blk + 1 < blk_end) ask(blk + 1, page, buf ^ 1);
            page = page_of(blk + 2);
            const int tb0 = blk * BLOCK_KEYS, tb = tb0 + TILE_KEYS * kp;
            if (!whole_range || tb0 + BLOCK_KEYS > ke) {
                clear_values(blk, buf);
                __syncthreads();
            }
            ++blk;
            if (wave_active && tb < wave_hi && tb + T * TILE_KEYS > wave_lo)    // (else: nothing for this wavefront)
                tile(tb, tb + T * TILE_KEYS <= wave_first_kend && tb >= wave_last_kbegin, buf_);
        };
        while (blk < blk_end) {
            turn(std::integral_constant<int, 0>{});
            if (blk < blk_end) turn(std::integral_constant<int, 1>{});
        }
    } else {
        // What a thread stages per block and pass: 32 bytes of the keys (16 channels of one key) and 32 bytes of
        // the values (16 keys of one channel; a page's values of one kv head are contiguous in the order
        // (channel, key)), so one page id and one address serve two 16-byte loads each.
        constexpr int KSTEP = S::KSTEP, VSTEP = S::VSTEP, KN = S::K_PASSES, VN = S::V_PASSES;
        const int k_key0 = threadIdx.x / ND, k_c16 = threadIdx.x % ND;
        const bool k_thread = (int)threadIdx.x < KSTEP * ND;
        const int v_m0 = threadIdx.x / D, v_d = threadIdx.x % D;
        const bool v_thread = (int)threadIdx.x < VSTEP * D;
        const bool big_page = P > BLOCK_KEYS;                   // a block lies within one page
        const uint32_t page_stride = (uint32_t)a.kv_heads * P * D;      // elements; the host keeps offsets within 32 bits
        int k_key[KN], k_pageadd[KN], v_m16[VN], v_pageadd[VN];
        uint32_t k_off0[KN], v_off0[VN];
#pragma unroll
        for (int i = 0; i < KN; ++i) {
            k_key[i] = min(k_key0 + KSTEP * i, BLOCK_KEYS - 1);
            k_pageadd[i] = big_page ? 0 : k_key[i] >> pshift;
            k_off0[i] = (uint32_t)kvh * P * D + (big_page ? k_key[i] : (k_key[i] & (P - 1))) * D + 16 * k_c16;
        }
#pragma unroll
        for (int i = 0; i < VN; ++i) {
            v_m16[i] = min(v_m0 + VSTEP * i, BLOCK_KEYS / 16 - 1);
            v_pageadd[i] = big_page ? 0 : (16 * v_m16[i]) >> pshift;
            v_off0[i] = (uint32_t)kvh * P * D + v_d * P + (big_page ? 16 * v_m16[i] : ((16 * v_m16[i]) & (P - 1)));
        }
        struct Staged {
            bf16x8 k[KN][2], v[VN][2];
            int tb;
            unsigned v_ok;               // bit i: pass i's page is mapped and its first key written
            bool whole;                  // every key of the block is written and mapped: nothing to check or zero
        };
        // global -> registers.  No branch around a load (a load behind a branch makes the compiler wait for
        // every load in flight): addresses are clamped to valid memory, and what must read as zero is zeroed
        // when the registers go to LDS.  Only the pages of written keys were looked up: anything later counts
        // as not mapped.
        auto fetch = [&](int blk, Staged& st) {
            const int tb = blk * BLOCK_KEYS;
            st.tb = tb;
            const int pidx = (tb >> pshift) - first_page;
            const uint32_t inpage = big_page ? (tb & (P - 1)) : 0;
            // (all blocks but a group's last, unless a window has given pages back: the same for every thread)
            st.whole = all_mapped && a.window <= 0 && tb + BLOCK_KEYS <= ke;
            if (st.whole) {
#pragma unroll
                for (int i = 0; i < KN; ++i) {
                    const int pg = page_lds[pidx + k_pageadd[i]];
                    const __bf16* kptr = a.k_pages + (__umul24(pg, page_stride) + inpage * D + k_off0[i]);
                    st.k[i][0] = *reinterpret_cast<const bf16x8*>(kptr);
                    st.k[i][1] = *reinterpret_cast<const bf16x8*>(kptr + 8);
                }
#pragma unroll
                for (int i = 0; i < VN; ++i) {
                    const int pg = page_lds[pidx + v_pageadd[i]];
                    const __bf16* vptr = a.v_pages + (__umul24(pg, page_stride) + inpage + v_off0[i]);
                    st.v[i][0] = *reinterpret_cast<const bf16x8*>(vptr);
                    st.v[i][1] = *reinterpret_cast<const bf16x8*>(vptr + 8);
                }
                st.v_ok = ~0u;
                return;
            }
            unsigned ok = 0;
#pragma unroll
            for (int i = 0; i < KN; ++i) {
                const int raw = page_lds[min(pidx + k_pageadd[i], PAGE_IDS - 1)];
                const int pg = tb + k_key[i] < ke ? raw : 0;
                const __bf16* kptr = a.k_pages + (__umul24(max(pg, 0), page_stride) + inpage * D + k_off0[i]);
                st.k[i][0] = *reinterpret_cast<const bf16x8*>(kptr);
                st.k[i][1] = *reinterpret_cast<const bf16x8*>(kptr + 8);
            }
#pragma unroll
            for (int i = 0; i < VN; ++i) {
                const int raw = page_lds[min(pidx + v_pageadd[i], PAGE_IDS - 1)];
                const int pg = tb + 16 * v_m16[i] < ke ? raw : -1;
                ok |= (pg >= 0 ? 1u : 0u) << i;
                const __bf16* vptr = a.v_pages + (__umul24(max(pg, 0), page_stride) + inpage + v_off0[i]);
                st.v[i][0] = *reinterpret_cast<const bf16x8*>(vptr);
                st.v[i][1] = *reinterpret_cast<const bf16x8*>(vptr + 8);
            }
            st.v_ok = ok;
        };
        auto stash = [&](int buf, const Staged& st) {      // registers -> LDS
            if (k_thread) {
                __bf16* kb = k_lds + buf * S::KBUF + k_key0 * KPITCH + 16 * k_c16;
#pragma unroll
                for (int i = 0; i < KN; ++i) {
                    if (KN * KSTEP > BLOCK_KEYS && k_key0 + KSTEP * i >= BLOCK_KEYS) continue;
                    *reinterpret_cast<bf16x8*>(kb + KSTEP * i * KPITCH) = st.k[i][0];
                    *reinterpret_cast<bf16x8*>(kb + KSTEP * i * KPITCH + 8) = st.k[i][1];
                }
            }
            if (v_thread) {
                __bf16* vb = v_lds + buf * S::VBUF + v_d * VPITCH + 16 * v_m0;
#pragma unroll
                for (int i = 0; i < VN; ++i) {
                    if (VN * VSTEP > BLOCK_KEYS / 16 && v_m0 + VSTEP * i >= BLOCK_KEYS / 16) continue;
                    bf16x8 v0 = st.v[i][0], v1 = st.v[i][1];
                    const int key0 = st.tb + 16 * (v_m0 + VSTEP * i);
                    const bool ok = (st.v_ok >> i) & 1;
                    if (!st.whole && !(ok && key0 + 16 <= ke)) {
                        // values of keys that are not written yet, or of a page that was given back (behind a
                        // window), count as zero: their probability is zero, but zero times whatever the
                        // memory holds need not be
#pragma unroll
                        for (int e = 0; e < 8; ++e) {
                            if (!ok || key0 + e >= ke) v0[e] = (__bf16)0.f;
                            if (!ok || key0 + 8 + e >= ke) v1[e] = (__bf16)0.f;
                        }
                    }
                    // keys 8 a + 4 h + r of the 16 go to position 8 h + 4 a + r
                    *reinterpret_cast<bf16x8*>(vb + 16 * VSTEP * i) =
                        bf16x8{v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
                    *reinterpret_cast<bf16x8*>(vb + 16 * VSTEP * i + 8) =
                        bf16x8{v0[4], v0[5], v0[6], v0[7], v1[4], v1[5], v1[6], v1[7]};
                }
            }
        };

        // Two blocks are under way at any time: one being multiplied out of LDS, the next in flight from memory
        // into registers.  One barrier per block suffices with two LDS buffers: a wavefront can only reach the
        // second write of a buffer after the barrier that follows every wavefront's read of it.  Fetches are
        // unconditional, clamped to the last block.
        {
            Staged st;
            const int last = blk_end - 1;
            fetch(blk_begin, st);
            int buf = 0;
            for (int blk = blk_begin; blk < blk_end; ++blk) {
                stash(buf, st);
                fetch(min(blk + 1, last), st);
                __syncthreads();
                compute(blk, buf);
                buf ^= 1;
            }
        }
    }

    // merge of the two key parities: parity 1 hands over its state, parity 0 finishes the columns
    l_run += __shfl_xor(l_run, 32, 64);
    if (S::PARITIES > 1) __syncthreads();                // the staged blocks are not read any more
    float* mine = merge_lds + (size_t)cq * S::NO * 64 + lane;
    if (kp == 1) {
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int i = 0; i < 16; ++i) mine[(db * 16 + i) * 64] = o[db][i];
        mine[(DB * 16) * 64] = m_ref;
        mine[(DB * 16 + 1) * 64] = l_run;
    }
    if (S::PARITIES > 1) __syncthreads();
    auto theirs = [&](int i) { return S::PARITIES > 1 ? mine[i * 64] : 0.f; };
    if (kp == 0 && col_valid) {
        const float m1 = S::PARITIES > 1 ? theirs(DB * 16) : -INFINITY, l1 = theirs(DB * 16 + 1);
        const float m = fmaxf(m_ref, m1);
        const float w0 = m_ref > -INFINITY ? __builtin_amdgcn_exp2f(m_ref - m) : 0.f;
        const float w1 = m1 > -INFINITY ? __builtin_amdgcn_exp2f(m1 - m) : 0.f;
        const float l = l_run * w0 + l1 * w1;
        // A column whose keys all lie in this split is finished here; the merge passes it over.
        const bool whole = !splitting || (split * a.split_keys <= kbegin_c && kend_c <= (split + 1) * a.split_keys);
        if (!whole) {
            // only the splits that hold keys of this column are read by the merge
            if (split * a.split_keys >= kend_c || (split + 1) * a.split_keys <= kbegin_c) return;
            float* dst = a.partial + (((size_t)(row0 + tok) * a.q_heads + kvh * g + hh) * a.max_splits + split) * (D + 4);
#pragma unroll
            for (int db = 0; db < DB; ++db)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int d0 = 32 * db + 8 * j + 4 * h;
                    if (d0 >= D) continue;
                    float4 v;                           // (D + 4 floats a split: 16-byte stores)
                    v.x = o[db][4 * j] * w0 + theirs(db * 16 + 4 * j) * w1;
                    v.y = o[db][4 * j + 1] * w0 + theirs(db * 16 + 4 * j + 1) * w1;
                    v.z = o[db][4 * j + 2] * w0 + theirs(db * 16 + 4 * j + 2) * w1;
                    v.w = o[db][4 * j + 3] * w0 + theirs(db * 16 + 4 * j + 3) * w1;
                    *reinterpret_cast<float4*>(dst + d0) = v;
                }
            if (h == 0) {
                dst[D] = m;
                dst[D + 1] = l;
            }
            return;
        }
        const float inv = l != 0.f ? 1.f / l : 0.f;      // (a NaN sum must show, not read as "no key")
        __bf16* dst = a.out + ((size_t)(row0 + tok) * a.q_heads + kvh * g + hh) * D;
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int d0 = 32 * db + 8 * j + 4 * h;
                if (d0 >= D) continue;
                bf16x4 w4;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float other = theirs(db * 16 + 4 * j + r);
                    w4[r] = (__bf16)((o[db][4 * j + r] * w0 + other * w1) * inv);
                }
                *reinterpret_cast<bf16x4*>(dst + d0) = w4;
            }
    }
}

// The merge of key splits: one wavefront per (group, head, token of the group), four a workgroup; a lane takes
// the channels lane and lane + 64.  A channel's values are added over the splits in ascending order; the denominators, a split a lane
// (of more than 64, the lane's own first), by halves over the lanes.  A token whose keys lay in one split was finished by that
// split's workgroup.
// Bound by its chain of loads: with one split after the other, its values asked for behind its weight, the merge of 33 tokens in 49
// splits of 16 heads took 17.7 us, now 7.5.
__global__ __launch_bounds__(256) void tiles_combine_kernel(TileArgs a) {
    const int grp = blockIdx.x, head = blockIdx.y, j = blockIdx.z * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (j >= a.group_ntok[grp]) return;
    const int D = a.head_dim;
    const int m = a.group_row0[grp] + j;
    const int pos = a.positions[m];
    const int first = a.window > 0 ? max(0, pos + 1 - a.window) / a.split_keys : 0;
    const int last = min(a.max_splits - 1, pos / a.split_keys);
    if (first == last) return;                           // one split held all its keys and wrote the result itself
    const float* base = a.partial + (((size_t)m * a.q_heads + head) * a.max_splits) * (D + 4);
    float gmax = -INFINITY;
    for (int s = first + lane; s <= last; s += 64) gmax = fmaxf(gmax, base[(size_t)s * (D + 4) + D]);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) gmax = fmaxf(gmax, __shfl_xor(gmax, off, 64));
    const int d0 = min(lane, D - 1), d1 = min(lane + 64, D - 1);
    float den = 0.f, n0 = 0.f, n1 = 0.f;
    constexpr int AHEAD = 8;
    for (int s0 = first; s0 <= last; s0 += 64) {         // a lane a split's weight, and eight splits' values under way
        const float* mine = base + (size_t)min(s0 + lane, last) * (D + 4) + D;
        const float sm = mine[0], sum = mine[1];
        const float w = s0 + lane <= last && sm > -INFINITY ? __builtin_amdgcn_exp2f(sm - gmax) : 0.f;   // maxima are base-2 exponents
        den += s0 + lane <= last ? w * sum : 0.f;
        const int n = min(64, last + 1 - s0);
        for (int u0 = 0; u0 < n; u0 += AHEAD) {
            float v0[AHEAD], v1[AHEAD];
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) {            // (clamped: no branch around a load)
                const float* p = base + (size_t)min(s0 + u0 + u, last) * (D + 4);
                v0[u] = p[d0];
                v1[u] = p[d1];
            }
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) {
                const float of = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), u0 + u));
                n0 += of * v0[u];
                n1 += of * v1[u];
            }
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) den += __shfl_xor(den, off, 64);
    const float inv = den != 0.f ? 1.f / den : 0.f;
    __bf16* dst = a.out + ((size_t)m * a.q_heads + head) * D;
    if (lane < D) dst[lane] = (__bf16)(n0 * inv);
    if (lane + 64 < D) dst[lane + 64] = (__bf16)(n1 * inv);
}

// Workgroups of eight wavefronts (128 columns, other head sizes than 128) take two groups, one after the other: group i and group
// (groups - 1 - i).  Within a long prompt the groups' key ranges grow with their position, so every workgroup gets about the
// same work -- unless the pairs would be fewer than the compute units: then every group gets a workgroup of
// its own.  Workgroups of four wavefronts take one group each, the later (longer) groups first, and two of
// them share a compute unit.  When all of them fit the GPU at once, the order is: the later half of the
// groups, longest first, then the earlier half, shortest first, so that the longest group shares its compute
// unit with the shortest (measured at 2 048 tokens: 42.4 us for 44.1; with more workgroups than places the
// longest must simply start first).  Workgroups are dealt to the 8 XCDs round-robin by their linear index; the
// index is remapped so that the workgroups of one kv head, which read the same keys and values, share an
// XCD and its L2.
template <int ND, int NQ>
__global__ __launch_bounds__((TileShape<ND, NQ>::THREADS), (NQ == 2 || ND == 8 ? 2 : 1)) void attention_tiles_kernel(TileArgs a) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
    const int per_head = gridDim.x, total = gridDim.x * gridDim.y;
    int lin = blockIdx.x + per_head * blockIdx.y;
    if (total % 8 == 0) lin = (lin % 8) * (total / 8) + lin / 8;
    const int first = lin % per_head, kvh = lin / per_head;
    const int second = a.groups - 1 - first;
    int todo[2] = {first, -1};
    if (a.single) {                                     // one group a workgroup, the later ones first
        // (with splits: split by split, so that the workgroups under way at a time walk the same keys.
        // Measured at 2048 tokens in two splits: 53 us; a group's splits side by side: 60; no split: 44)
        const int half = (a.groups + 1) / 2;
        todo[0] = a.max_splits > 1 || !a.all_resident ? second : (first < half ? second : first - half);
    } else if (second > first) {
        todo[0] = second;
        todo[1] = first;
    }
#pragma unroll 1
    for (int i = 0; i < 2; ++i) {                       // (one copy of the code for both)
        const int grp = i == 0 ? todo[0] : todo[1];
        if (grp < 0) return;
        if (i > 0) __syncthreads();
        tile_group<ND, NQ>(a, grp, kvh, a.single ? blockIdx.z : 0, lds_raw);
    }
}

template <int ND, int NQ>
static int launch_tiles(const TileArgs& a, hipStream_t stream) {
    static bool prepared = false;
    const size_t lds = TileShape<ND, NQ>::lds_bytes;
    if (!prepared) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&attention_tiles_kernel<ND, NQ>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return (int)e;
        prepared = true;
    }
    static int compute_units = 0;
    if (compute_units == 0) {
        int device = 0;
        if (hipGetDevice(&device) != hipSuccess ||
            hipDeviceGetAttribute(&compute_units, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess)
            compute_units = -1;
    }
    // (pairs that would leave compute units idle are no gain: then every group gets a workgroup of its own)
    const bool few_pairs = (long)((a.groups + 1) / 2) * a.kv_heads < compute_units;
    const bool two = TileShape<ND, NQ>::THREADS == 256;         // two workgroups a compute unit
    const bool single = NQ == 2 || a.max_splits > 1 || a.single == 1 || (a.single == 0 && (two || few_pairs));
    dim3 grid(single ? a.groups : (a.groups + 1) / 2, a.kv_heads, a.max_splits);
    TileArgs b = a;
    b.single = single ? 1 : 0;
    b.all_resident = two && compute_units > 0 && (long)a.groups * a.kv_heads * a.max_splits <= 2L * compute_units;
    attention_tiles_kernel<ND, NQ><<<grid, TileShape<ND, NQ>::THREADS, lds, stream>>>(b);
    int err = (int)hipGetLastError();
    if (err != 0 || a.max_splits <= 1) return err;
    tiles_combine_kernel<<<dim3(a.groups, a.q_heads, ((32 * NQ) / (a.q_heads / a.kv_heads) + 3) / 4), 256, 0, stream>>>(a);
    return (int)hipGetLastError();
}

template <int NQ>
static int launch_tiles_dim(const TileArgs& a, hipStream_t stream) {
    switch (a.head_dim / 16) {
        case 1: return launch_tiles<1, NQ>(a, stream);
        case 2: return launch_tiles<2, NQ>(a, stream);
        case 3: return launch_tiles<3, NQ>(a, stream);
        case 4: return launch_tiles<4, NQ>(a, stream);
        case 5: return launch_tiles<5, NQ>(a, stream);
        case 6: return launch_tiles<6, NQ>(a, stream);
        case 7: return launch_tiles<7, NQ>(a, stream);
        default: return launch_tiles<8, NQ>(a, stream);
    }
}

// Groups: group_row0[i] = first batch row of group i, group_ntok[i] = its tokens (consecutive rows of one
// request, at most columns / (q_heads / kv_heads); columns = 128 or 64).  A group's keys must span at most
// PAGE_IDS pages (per key split, with splits).  The cache of num_pages pages must hold fewer than 2^32 elements.
// With max_splits > 1, `partial` holds M * q_heads * max_splits * (head_dim + 4) floats, 16-byte aligned, M the batch's rows.
// `pairing` (workgroups of 128 columns without splits): 0 two groups a workgroup where it has eight wavefronts, unless that would
// leave compute units idle, 1 always one group a workgroup, 2 always two.  Returns 0, a HIP error
// code, or a negative number for sizes this kernel does not take.
extern "C" int mlr_attention_tiles(
    const void* q, const void* k_pages, const void* v_pages, const int32_t* block_table, int max_blocks,
    const int32_t* slots, const int32_t* positions, void* out, const int32_t* group_row0,
    const int32_t* group_ntok, int groups, int columns, int q_heads, int kv_heads, int head_dim, int page_size,
    int num_pages, int window, float scale, int split_keys, int max_splits, float* partial, int pairing,
    hipStream_t stream) {
    if (groups <= 0) return 0;
    if (head_dim % 16 != 0 || head_dim < 16 || head_dim > 128 || q_heads % kv_heads != 0 ||
        (columns != 128 && columns != 64) || q_heads / kv_heads > columns || pairing < 0 || pairing > 2) return -1;
    if (page_size < 16 || (page_size & (page_size - 1)) != 0) return -2;
    if (max_splits < 1) max_splits = 1;
    if (max_splits > 1 && (partial == nullptr || split_keys <= 0 || split_keys % BLOCK_KEYS != 0 ||
                           max_splits > 65535 || groups > 65535)) return -4;
    // offsets into the cache are 32-bit element counts, a page's stride and id 24-bit factors
    const uint64_t stride = (uint64_t)kv_heads * page_size * head_dim;
    if (stride >= (1u << 24) || num_pages >= (1 << 24) || stride * (uint64_t)num_pages >= (1ull << 32)) return -3;
    int shift = 0;
    while ((1 << shift) < page_size) ++shift;
    TileArgs a{(const __bf16*)q, (const __bf16*)k_pages, (const __bf16*)v_pages, block_table, slots, positions,
               (__bf16*)out, group_row0, group_ntok, partial, groups, max_blocks, q_heads, kv_heads, head_dim,
               page_size, shift, window, split_keys, max_splits, scale, 0, pairing};
    return columns == 128 ? launch_tiles_dim<4>(a, stream) : launch_tiles_dim<2>(a, stream);
}
