// Paged attention for long segments (long prompts and their late portions) on the matrix cores, bfloat16, heads of 256,
// pages of 16, 32, 64, ... keys.  A workgroup of eight wavefronts is 128 rows of one (segment, key/value head): rows
// are (token, query head of the group) pairs, row r = token * G + head.  Two groups of four wavefronts hold the
// same 128 rows, 32 a wavefront, and take the blocks of 32 keys in turn, one the even, the other the odd ones; at the
// end their results meet in shared memory.
//
// Why so: a fragment of keys or values read from shared memory feeds two tiles of rows (with one, the reads took as long as the
// products), a block's loads and their addresses are shared by twice the rows, and the groups work half a step apart:
// while one has the matrix cores, the other is at its softmax.  The step of a group, with a barrier of the workgroup after
// each half:
//   S  softmax of block j; the values of block j + 1 and the keys of block j + 2 are asked for
//   P  the weighted values of block j are added up, then the scores of block j + 1 made (64 products)
// A group holds two blocks of keys and two of values.  Keys j + 2 overwrite keys j and values j + 1 overwrite values j - 1, which every
// wavefront of the group has read in the P before.  They are needed a whole step later; each wavefront waits at the end of S for what it
// asked for one S before, so the barrier behind says that the next P's operands are there.
//
// What bounds it: 7,777 rows of 8 heads on one over their own keys take 255 us (0.97 PFLOP/s; blocks of 64 rows 383).  A half step measures
// 1,700 clocks where its 64 products take 1,024: in S the softmax of two tiles 1,150 and eight loads 550, in P the products
// 1,400, as every pair of fragments waits for a trip to shared memory now and then (the registers leave room for two pairs
// ahead).  What it took: rescaling the accumulators only where a maximum has grown by a lot (346 to 264), the wavefronts at
// their softmax going before those at their products (400 to 309, with half of the loads moved), loads whose
// addresses are a scalar and a fixed offset (a load 65 clocks, 130 with an address worked out a lane).
//
// The products are those of `attention_mfma.hip` (v_mfma_f32_16x16x32_bf16, scores transposed so that a lane's values all
// belong to one query row, probabilities fed to the second product from the registers they were computed in).  Tiles go
// to shared memory straight from the cache (global_load_lds_dwordx4), every load from one page.  Chunk c (16 bytes) of key
// row r lies at c ^ (r % 16); row 16 t + 4 g + v of a key tile holds key 8 g + 4 t + v of the block, so that a lane's eight scores
// are the eight keys of its chunk g of a value row.  A tile of values is two halves of 16 keys, each [256 rows][2 chunks], chunk
// q of row d at q ^ ((d / 8) % 2).  The 16 lanes that read together so meet all banks once.  In the blocks at the edges of a request the stale keys' scores
// are masked, and their values (which may be anything, NaN too) are cleared once they have landed.
#include "common.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));

constexpr int kPromptRows = 128;         // rows a workgroup
constexpr int kPromptGroupWaves = 4;
constexpr int kPromptThreads = 2 * kPromptGroupWaves * kWave;
constexpr int kPromptKeys = 32;          // keys a block
constexpr int kPromptTablePages = 1024;  // pages one work item's keys may span (the host cuts items to fit)
constexpr int kPromptItemInts = 8;

union QPack {
    uint4 u;
    bf16x8_t v;
};

// 16 bytes a lane from base + offset into shared memory at `lds_address` + 16 * lane.  Assembly, and M0 put back as it was, so that
// the compiler makes no later read of shared memory wait for it: the kernel waits itself.
static __device__ __forceinline__ void load_to_shared(const void* base, uint32_t offset, uint32_t lds_address) {
    uint32_t saved_m0;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
                 : "=&s"(saved_m0) : "v"(offset), "s"(base), "s"(lds_address) : "memory");
}

template <int N>
static __device__ __forceinline__ void wait_loads() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

static __device__ __forceinline__ void meet() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
}

// The same number as one that the compiler knows nothing of: what is worked out from it in a loop stays in the loop (kept over
// the loop, such numbers cost the registers that the accumulators need, and came back from memory).
static __device__ __forceinline__ int here(int v) {
    asm volatile("" : "+v"(v));
    return v;
}

constexpr float kSlack = 8.f;             // powers of two by which a score may pass the maximum its weight is relative to
constexpr int HD = 256;                                    // head size
constexpr int kTile = kPromptKeys * HD * 2;                // bytes of a block's keys, and of its values
constexpr int kTiles = 2 * 4 * kTile;                      // [group][keys 0, keys 1, values 0, values 1]
constexpr int kTableAt = kTiles, kMlAt = kTableAt + kPromptTablePages * 4;
constexpr int kPromptShared = kMlAt + 2 * kPromptGroupWaves * 16 * 8;

template <bool V>
struct Flag {
    static constexpr bool value = V;
};

// items: seg, kvh, first row, first key, end key, partial slot (-1: the workgroup walks all the keys of its rows and writes
// the result itself), 2 unused.  Items that split the keys of a block of rows write, per tile of 16 rows, an unnormalised
// accumulator and (maximum, sum) into slot `partial slot + tile`.  SPLIT: the weights of the second product keep 16 bits
// (the rounded weight and what the rounding left out, two products).
template <bool SPLIT>
__global__ void __launch_bounds__(kPromptThreads, 2)
paged_attention_prompt_kernel(const bf16* __restrict__ qkv, const bf16* __restrict__ cache, const int* __restrict__ block_tables,
                              const int* __restrict__ items, const int* __restrict__ seg_q_start, const int* __restrict__ seg_q_len,
                              const int* __restrict__ seg_ctx_len, bf16* __restrict__ out, float* __restrict__ partial_o,
                              float* __restrict__ partial_ml, int num_heads, int num_kv_heads, int page_size, int max_pages,
                              float scale_log2e, int window, int q_stride, float cap_scale, float softcap,
                              const float* __restrict__ sinks) {
    constexpr int DC = HD / 32, DT = HD / 16, CPR = HD / 8;       // CPR: 16-byte chunks of a key row
    constexpr int KU = kPromptKeys * CPR / 64 / kPromptGroupWaves, VU = HD * 4 / 64 / kPromptGroupWaves;   // loads a wavefront
    extern __shared__ __align__(16) unsigned char shared[];
    int* table_s = reinterpret_cast<int*>(shared + kTableAt);
    float2* ml_s = reinterpret_cast<float2*>(shared + kMlAt);

    const int* item = items + static_cast<size_t>(blockIdx.x) * kPromptItemInts;
    const int seg = item[0], kvh = item[1], row_begin = item[2];
    const int key_begin = item[3], key_end = item[4], partial_slot = item[5];
    if (seg < 0) return;
    const int tid = threadIdx.x, lane = tid % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int side = wave / kPromptGroupWaves, wv = wave % kPromptGroupWaves;
    const int i = lane % 16, g = lane / 16;
    const int group = num_heads / num_kv_heads;
    const int q_start = seg_q_start[seg], q_len = seg_q_len[seg], ctx = seg_ctx_len[seg];
    const int total_rows = q_len * group;
    const int first_pos = ctx - q_len;
    const int seg_lo = lowest_key(first_pos, window);
    const size_t page_elems = static_cast<size_t>(2) * num_kv_heads * page_size * HD;
    const size_t k_off = static_cast<size_t>(kvh) * page_size * HD;
    const size_t v_off = (static_cast<size_t>(num_kv_heads) + kvh) * page_size * HD;

    // ---- this wavefront's two tiles of rows ----
    const int wr0 = row_begin + wv * 32;
    int pos[2];                          // of a lane's row in each tile; -1, which masks every key, beyond the segment's rows
    bf16x8_t qreg[2][DC];
    int t_pos_min[2], t_lo_max[2];       // of a tile's rows: the lowest position, the highest window start
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
        const int row = wr0 + rt * 16 + i;
        const bool valid = row < total_rows;
        const int tok = valid ? row / group : 0;
        const int head = kvh * group + (valid ? row % group : 0);
        pos[rt] = valid ? first_pos + tok : -1;
        const bf16* qrow = qkv + static_cast<size_t>(q_start + tok) * q_stride + static_cast<size_t>(head) * HD;
#pragma unroll
        for (int c = 0; c < DC; ++c) {
            QPack p;
            p.u = valid ? *reinterpret_cast<const uint4*>(qrow + c * 32 + 8 * g) : make_uint4(0, 0, 0, 0);
            qreg[rt][c] = p.v;
        }
        const int begin = wr0 + rt * 16, last = min(total_rows - 1, begin + 15);
        t_pos_min[rt] = begin < total_rows ? first_pos + begin / group : -1;
        t_lo_max[rt] = lowest_key(first_pos + max(last, 0) / group, window);
        if (last < begin + 15) t_pos_min[rt] = -1;      // a tile with rows beyond the segment always masks
    }
    const int b_last_row = min(total_rows - 1, row_begin + kPromptRows - 1);
    const int b_hi = first_pos + b_last_row / group + 1;
    const int b_lo = lowest_key(first_pos + row_begin / group, window);
    const int blk_first = max(b_lo, key_begin) / kPromptKeys;
    const int blk_end = (min(b_hi, key_end) + kPromptKeys - 1) / kPromptKeys;
    const int blocks = max(0, blk_end - blk_first);
    const int steps = (blocks + 1) / 2, own = (blocks + 1 - side) / 2;        // steps of the workgroup, blocks of this group
    const int page_base = blk_first * kPromptKeys / page_size;
    int table_last = 0;
    if (blocks > 0) {
        const int* table_g = block_tables + static_cast<size_t>(seg) * max_pages + page_base;
        const int page_last = (min(blk_end * kPromptKeys, ctx) - 1) / page_size;
        const int count = min(min(max_pages - 1, page_last) - page_base + 1, kPromptTablePages);
        for (int p = tid; p < count; p += kPromptThreads) table_s[p] = table_g[p];
        table_last = count - 1;
    }

    // ---- the loads of a block.  The page size is a power of two from 16 on and a block begins at a multiple of 32 keys, so the
    //      place of key kbase + rel splits into page (kbase >> shift) + (rel >> shift) of the request and slot
    //      (kbase & mask) + (rel & mask).  Every load of a wavefront is of one page, so its address is a scalar base and a lane's
    //      fixed offset.  A page index beyond the request's last page is clamped: whatever lies there is masked and cleared. ----
    const int shift = __builtin_ctz(page_size), mask = page_size - 1;
    const size_t page_bytes = page_elems * 2;
    const char* const keys_base = reinterpret_cast<const char*>(cache + k_off);
    const char* const values_base = reinterpret_cast<const char*>(cache + v_off);
    // keys: load u of wavefront wv carries the rows 2 (wv + 4 u) and the next of the tile (two keys): with r the first for u = 0, the
    // keys rel = 8 (r / 4) + r % 4, for u = 1 rel + 16, for u = 2 and 3 those 4 further on; row r + 8 exchanges its chunks by 8 more
    const int k_row = 2 * wv + lane / 32;
    const int k_rel = 8 * (k_row / 4) + k_row % 4;
    const uint32_t k_at = static_cast<uint32_t>((k_rel & mask) * HD + ((lane % 32) ^ k_row) * 8) * 2;
    // values: the tile is two halves of 16 keys, each [256 rows][2 chunks]; wavefront wv brings rows 128 (wv % 2) .. + 127 of
    // half wv / 2, 32 rows a load
    const int v_rel = 16 * (wv / 2);
    const int v_row = 128 * (wv % 2) + lane / 2, v_chunk = (lane % 2) ^ ((v_row / 8) % 2);
    const uint32_t v_at = static_cast<uint32_t>(v_row * page_size + v_chunk * 8) * 2;
    const uint32_t tiles_lds = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(
                                   reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) void*)shared))) +
                               side * 4 * kTile + wv * 1024;
    auto base_of = [&](int j) { return (blk_first + 2 * j + side) * kPromptKeys; };
    // the pages of a block's keys (the load's 0 and 2, and its 1 and 3) and of its values, read ahead of the loads
    auto page_at = [&](int kbase, int rel) { return table_s[min((kbase >> shift) - page_base + (rel >> shift), table_last)]; };
    auto ask_keys = [&](int j, int page0, int page1) {
        const int kbase = base_of(j);
        const char* const from[2] = {
            keys_base + static_cast<size_t>(static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(page0))) * page_bytes +
                static_cast<size_t>(kbase & mask) * HD * 2,
            keys_base + static_cast<size_t>(static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(page1))) * page_bytes +
                static_cast<size_t>((kbase & mask) + (page_size >= 32 ? 16 : 0)) * HD * 2};
#pragma unroll
        for (int u = 0; u < KU; ++u)
            load_to_shared(from[u % 2] + u / 2 * (4 * HD * 2), u % 2 ? k_at ^ 128 : k_at,
                           tiles_lds + (j & 1) * kTile + u * (kPromptGroupWaves * 1024));
    };
    auto ask_values = [&](int j, int page) {
        const char* const from = values_base + static_cast<size_t>(static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(page))) * page_bytes +
                                 static_cast<size_t>(base_of(j) & mask) * 2 + (page_size >= 32 ? v_rel * 2 : 0);
#pragma unroll
        for (int u = 0; u < VU; ++u)
            load_to_shared(from + static_cast<size_t>(u * 32 * 2) * page_size, v_at,
                           tiles_lds + (2 + (j & 1)) * kTile + 3 * wv * 1024 + u * 1024);
    };

    float4_t acc[2][DT];
    float m_run[2] = {-INFINITY, -INFINITY}, l_run[2] = {0.f, 0.f};
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
        for (int t = 0; t < DT; ++t) acc[rt][t] = float4_t{0.f, 0.f, 0.f, 0.f};
    float sv[2][8];
    QPack pv[2], pr[2];                  // pr (SPLIT): what the rounding of pv left out

    __syncthreads();      // the block table is in shared memory
    for (int j = 0; j < min(own, 2); ++j) ask_keys(j, page_at(base_of(j), 0), page_at(base_of(j), 16));
    if (own > 0) ask_values(0, page_at(base_of(0), v_rel));
    if (own > 1) wait_loads<KU + VU>();
    else wait_loads<0>();
    meet();

    // A lane's fragment reads: every address is the tile, the lane's offset and a constant.  With x what row i
    // exchanges by, chunk (4 c + g) ^ x of a key row is 4 (c ^ (x >> 2)) + (g ^ (x & 3)), and x >> 2 touches the
    // two low bits of c only: the offset of c is that of chunk 0 with 64 (c % 4) exchanged.
    const int k_lane = (i * CPR + 4 * (i >> 2) + (g ^ (i & 3))) * 16;
    const int v_lane = g / 2 * 8192 + i * 32 + ((g ^ (i / 8)) % 2) * 16;
    const unsigned char* tiles = shared + side * 4 * kTile;

    // The products of a step: the weighted values of block j (WEIGH), then the scores of block j + 1.  Fragments are read two at
    // a time, kAhead such pairs before their products, the first ones of the keys while the last values are multiplied.
    constexpr int kPair = 2, kAhead = 2, kRing = kAhead + 1;
    auto tile_of = [&](int j) { return min(j, own - 1) & 1; };     // (a group without a block j has no weights for it)
    auto products = [&](int j, auto weigh) {
        constexpr int kFirst = decltype(weigh)::value ? 0 : DT, kEnd = DT + 2 * DC;
        const unsigned char* v_s = tiles + (2 + tile_of(j)) * kTile + v_lane;
        const unsigned char* k_s = tiles + tile_of(j + 1) * kTile;
        const int k0 = here(k_lane);
        const int k_of[4] = {k0, k0 ^ 64, k0 ^ 128, k0 ^ 192};
        QPack f[kRing][kPair];
        auto read = [&](int n) {
#pragma unroll
            for (int e = n; e < n + kPair; ++e) {
                const int c = (e - DT) / 2, t2 = (e - DT) % 2;
                f[n / kPair % kRing][e - n].u = *reinterpret_cast<const uint4*>(
                    e < DT ? v_s + e * 512 : k_s + k_of[c & 3] + (16 * t2 * CPR + 4 * (c & ~3)) * 16);
            }
        };
        float4_t sc[2][2];
#pragma unroll
        for (int rt = 0; rt < 2; ++rt)
#pragma unroll
            for (int t2 = 0; t2 < 2; ++t2) sc[rt][t2] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int n = kFirst; n < kFirst + kAhead * kPair; n += kPair) read(n);
#pragma unroll
        for (int n = kFirst; n < kEnd; n += kPair) {
            __builtin_amdgcn_sched_barrier(0);
            if (n + kAhead * kPair < kEnd) read(n + kAhead * kPair);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int e = n; e < n + kPair; ++e) {
                const QPack& frag = f[n / kPair % kRing][e - n];
#pragma unroll
                for (int rt = 0; rt < 2; ++rt) {
                    if (e < DT) {
                        float4_t& a = acc[rt][e % DT];
                        a = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag.v, pv[rt].v, a, 0, 0, 0);
                        if (SPLIT) a = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag.v, pr[rt].v, a, 0, 0, 0);
                    } else {
                        float4_t& a = sc[rt][(e - DT) % 2];
                        a = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag.v, qreg[rt][(e - DT) / 2 % DC], a, 0, 0, 0);
                    }
                }
            }
        }
#pragma unroll
        for (int rt = 0; rt < 2; ++rt)
#pragma unroll
            for (int e = 0; e < 8; ++e) sv[rt][e] = sc[rt][e / 4][e % 4];
    };
    // In a block at the edge of a request: of the values that this wavefront brought (they have landed), those of keys that are
    // not the request's are cleared, each by the lane whose 16 bytes they are.
    auto clear_stale = [&](int j) {
        const int kbase = base_of(j);
        if (kbase + kPromptKeys <= ctx && kbase >= seg_lo) return;
        const int ln = here(lane), key0 = kbase + v_rel + 8 * ((ln % 2) ^ ((ln / 16) % 2));
        uint4* own_s = reinterpret_cast<uint4*>(shared + (side * 4 + 2 + (j & 1)) * kTile + wv * 4096 + ln * 16);
        uint32_t k[4];
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const int key = key0 + 2 * w;
            k[w] = (key < ctx && key >= seg_lo ? 0xffffu : 0u) | (key + 1 < ctx && key + 1 >= seg_lo ? 0xffff0000u : 0u);
        }
#pragma unroll
        for (int u = 0; u < VU; ++u) {
            const uint4 v = own_s[u * 64];
            own_s[u * 64] = make_uint4(v.x & k[0], v.y & k[1], v.z & k[2], v.w & k[3]);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    };
    auto softmax = [&](int j) {
        const int kbase = base_of(j);
        float top[2];
        bool grown = false;
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
            float* s = sv[rt];
            if (softcap > 0.f) {            // the score is scaled and bent here; `scale_log2e` is then log2(e) alone
#pragma unroll
                for (int e = 0; e < 8; ++e) s[e] = capped_score_fast(s[e] * cap_scale, softcap);
            }
            if (!(kbase + kPromptKeys - 1 <= t_pos_min[rt] && kbase >= t_lo_max[rt] && j < own)) {
                const int highest = j < own ? pos[rt] : -1;
                const int lowest = lowest_key(here(pos[rt]), window), key0 = kbase + 8 * (here(lane) / 16);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int key = key0 + e;
                    if (!(key <= highest && key >= lowest)) s[e] = -INFINITY;
                }
            }
            top[rt] = fmaxf(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3])), fmaxf(fmaxf(s[4], s[5]), fmaxf(s[6], s[7])));
            top[rt] = max_across(max_across(top[rt], 16), 32);
            grown = grown || top[rt] * scale_log2e > m_run[rt] * scale_log2e + kSlack;
        }
        // What a row's weights are relative to is its maximum so far, or less by up to kSlack: a factor that cancels in the end
        // and leaves every rounding's relative size as it is, while the accumulators are rescaled a few times in all.
        if (__any(grown)) {
#pragma unroll
            for (int rt = 0; rt < 2; ++rt) {
                const float m_new = fmaxf(m_run[rt], top[rt]);
                const float alpha = exp2_probability(fmaf(m_run[rt], scale_log2e, -((m_new == -INFINITY ? 0.f : m_new) * scale_log2e)));
                l_run[rt] *= alpha;
                m_run[rt] = m_new;
#pragma unroll
                for (int t = 0; t < DT; ++t) acc[rt][t] *= alpha;
            }
        }
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
            const float mc = (m_run[rt] == -INFINITY ? 0.f : m_run[rt]) * scale_log2e;
            float pe[8], psum = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                pe[e] = exp2_probability(fmaf(sv[rt][e], scale_log2e, -mc));       // exp2(-inf) = 0 for masked keys
                psum += pe[e];
            }
            pv[rt].u = make_uint4(pack2_bf16(pe[0], pe[1]), pack2_bf16(pe[2], pe[3]), pack2_bf16(pe[4], pe[5]), pack2_bf16(pe[6], pe[7]));
            if (SPLIT)
                pr[rt].u = make_uint4(pack2_bf16(bf16_remainder(pe[0]), bf16_remainder(pe[1])),
                                      pack2_bf16(bf16_remainder(pe[2]), bf16_remainder(pe[3])),
                                      pack2_bf16(bf16_remainder(pe[4]), bf16_remainder(pe[5])),
                                      pack2_bf16(bf16_remainder(pe[6]), bf16_remainder(pe[7])));
            l_run[rt] += psum;
        }
    };

    if (side == 1) meet();
    if (own > 0) {
        // (no branch around the products: where the accumulators pass one, the compiler keeps them twice)
        products(-1, Flag<false>());
        meet();
#pragma nounroll
        for (int j = 0; j < steps; ++j) {
            __builtin_amdgcn_s_setprio(1);
            const int next = base_of(j + 1), after = base_of(j + 2);
            const int v_page = page_at(next, v_rel), k_page0 = page_at(after, 0), k_page1 = page_at(after, 16);
            softmax(j);
            if (j + 1 < own) ask_values(j + 1, v_page);
            if (j + 2 < own) ask_keys(j + 2, k_page0, k_page1);
            if (j + 2 < own) wait_loads<KU + VU>();
            else if (j + 1 < own) wait_loads<VU>();
            else wait_loads<0>();
            if (j < own) clear_stale(j);
            __builtin_amdgcn_s_setprio(0);
            meet();
            products(j, Flag<true>());
            meet();
        }
    } else {
        for (int j = 0; j < 2 * steps + 1; ++j) meet();
    }
    if (side == 0) meet();               // every wavefront is done with the tiles

    // ---- the two groups' results meet: each finishes one of a pair's two tiles of rows ----
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) l_run[rt] = sum_across(sum_across(l_run[rt], 16), 32);
    float4_t* give = reinterpret_cast<float4_t*>(shared) + (side * kPromptGroupWaves + wv) * DT * 64 + lane;
    const float4_t* take = reinterpret_cast<const float4_t*>(shared) + ((1 - side) * kPromptGroupWaves + wv) * DT * 64 + lane;
    auto merge = [&](int rt) {           // rt: the tile this side finishes (a constant, so that registers are named by constants)
#pragma unroll
        for (int t = 0; t < DT; ++t) give[t * 64] = acc[1 - rt][t];
        if (g == 0) ml_s[(side * kPromptGroupWaves + wv) * 16 + i] = make_float2(m_run[1 - rt], l_run[1 - rt]);
        __syncthreads();
        const int row = wr0 + rt * 16 + i;
        if (row >= total_rows) return;
        const float2 ml = ml_s[((1 - side) * kPromptGroupWaves + wv) * 16 + i];
        const float m = fmaxf(m_run[rt], ml.x);
        const float mc = (m == -INFINITY ? 0.f : m) * scale_log2e;
        const float mine = exp2_probability(fmaf(m_run[rt], scale_log2e, -mc)), theirs = exp2_probability(fmaf(ml.x, scale_log2e, -mc));
        float l = l_run[rt] * mine + ml.y * theirs;
        if (partial_slot >= 0) {
            const size_t slot = static_cast<size_t>(partial_slot) + wv * 2 + rt;
            float* po = partial_o + (slot * 16 + i) * HD;
#pragma unroll
            for (int t = 0; t < DT; ++t)
                *reinterpret_cast<float4_t*>(po + t * 16 + 4 * g) = acc[rt][t] * mine + take[t * 64] * theirs;
            if (g == 0) *reinterpret_cast<float2*>(partial_ml + (slot * 16 + i) * 2) = make_float2(m, l);
            return;
        }
        const int tok = row / group, head = kvh * group + row % group;
        // a sink: exp(sink of the head) once more in the denominator of a row that is finished here
        if (sinks) l += exp2f(sinks[head] * 1.4426950408889634f - m * scale_log2e);
        const float inv = 1.f / l;
        bf16* orow = out + (static_cast<size_t>(q_start + tok) * num_heads + head) * HD;
#pragma unroll
        for (int t = 0; t < DT; ++t) {
            const float4_t o = (acc[rt][t] * mine + take[t * 64] * theirs) * inv;
            *reinterpret_cast<uint2*>(orow + t * 16 + 4 * g) = make_uint2(pack2_bf16(o[0], o[1]), pack2_bf16(o[2], o[3]));
        }
    };
    if (side == 0) merge(0);
    else merge(1);
}

// Returns 0, a HIP error code, or -1 for sizes this kernel does not take.
WLLM_API int wllm_paged_attention_prompt(const void* qkv, const void* cache, const int* block_tables, const int* items, int num_items,
                                         int rows_per_item, const int* seg_q_start, const int* seg_q_len, const int* seg_ctx_len,
                                         void* out, float* partial_o, float* partial_ml, int num_heads, int num_kv_heads,
                                         int head_dim, int page_size, int max_pages, float scale, int window, int q_stride,
                                         float softcap, int split_weights, const float* sinks, hipStream_t stream) {
    if (head_dim != HD || page_size < 16 || (page_size & (page_size - 1)) != 0 || num_heads % num_kv_heads != 0 ||
        rows_per_item != kPromptRows)
        return -1;
    if (q_stride < num_heads * head_dim || q_stride % 8 != 0 || softcap < 0.f) return -1;
    if (num_items <= 0) return 0;
    const float scale_log2e = (softcap > 0.f ? 1.f : scale) * 1.4426950408889634f;
    const float cap_scale = softcap > 0.f ? scale / softcap : 0.f;
#define LAUNCH(S)                                                                                                   \
    do {                                                                                                            \
        static bool roomy = false;     /* more than 64 KiB of shared memory must be asked for once */              \
        if (!roomy) {                                                                                               \
            if (hipFuncSetAttribute(reinterpret_cast<const void*>(&paged_attention_prompt_kernel<S>),           \
                                    hipFuncAttributeMaxDynamicSharedMemorySize, kPromptShared) != hipSuccess) \
                return launch_status();                                                                             \
            roomy = true;                                                                                           \
        }                                                                                                           \
        paged_attention_prompt_kernel<S><<<num_items, kPromptThreads, kPromptShared, stream>>>(      \
            static_cast<const bf16*>(qkv), static_cast<const bf16*>(cache), block_tables, items, seg_q_start,       \
            seg_q_len, seg_ctx_len, static_cast<bf16*>(out), partial_o, partial_ml, num_heads, num_kv_heads,        \
            page_size, max_pages, scale_log2e, window, q_stride, cap_scale, softcap, sinks);                        \
    } while (0)
    if (split_weights) LAUNCH(true);
    else LAUNCH(false);
#undef LAUNCH
    return launch_status();
}
