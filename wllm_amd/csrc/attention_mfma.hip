// Paged attention on the matrix cores for bfloat16, for segments of at most 16 query rows (decoded
// tokens, and portions short enough): head sizes 32..256 in steps of 32, pages of a multiple of 4
// tokens, any number of heads and groups, optional window.  Longer segments take the kernel of
// `attention_prefill.hip`, which shares the products' layout described here.
//
// Rows.  For one request (segment) and one key/value head, the query rows are the pairs (token,
// query head of the group): row r = token * G + head.  All rows of a tile read the same keys and
// values, so under multi-query attention the G heads of a token share one pass over the cache
// (the reference's kernel runs one workgroup per query head and reads the cache G times,
// src/wllm/kernels/csrc/paged_attention.cu:44-45,185).
//
// Work items.  The host cuts every (segment, key/value head) into work items, one workgroup of 4
// wavefronts each: a tile of 16 of the segment's rows (it has one, unless more than 16 query heads
// share a key/value head) and a chunk of keys that lies within one
// aligned group of 128 keys, cut to what the rows can need.  Each wavefront takes one of the
// chunk's four blocks of 32 keys; its loads of keys and values wait for the item and the block
// table only (the request's lengths and the queries are read while they are in flight), and the
// four are merged through shared memory.  A segment with more keys than a chunk is split over
// workgroups; those write partial results (maximum, sum, unnormalised accumulator) that
// `attention_reduce_kernel` combines.  Chunk boundaries depend on the key index only, never on
// the batch.  A captured graph launches a workgroup for every item its plan has room for and reads
// the number of live items, which come first, from device memory.
//
// Matrix products (v_mfma_f32_16x16x32_bf16, 64 lanes: i = lane % 16, g = lane / 16):
//   scores^T[key, row] = K[key, :] . Q[row, :]     A = K: lane (i, g) holds K[key_i][32c + 8g ..+8]
//                                                  B = Q: lane (i, g) holds Q[row_i][32c + 8g ..+8]
//                                                  C: lane (i, g) holds rows (keys) 4g..4g+3, column row_i
//   out^T[d, row] = V^T[d, keys] . P^T[keys, row]  A = V^T: lane (i, g) holds V^T[16t + i][8 keys of g]
//                                                  B = P^T: the lane's own 8 probabilities of row_i
// so every value a lane holds belongs to one query row, softmax needs two shuffles per tile, and the
// probabilities feed the second product from the registers they were computed in.  The cache holds
// keys as [page_size, head_dim] rows and values transposed as [head_dim, page_size] rows.  Values are
// loaded as fragments (16-byte loads when the page size is a multiple of 8: per instruction two runs
// of 512 bytes).  Keys are loaded as whole rows, 16 bytes a lane in the order they lie in the page,
// and become fragments in the wavefront's part of shared memory: a fragment load straight from the
// cache asks for 64-byte pieces of 16 rows, a pattern the memory system serves more slowly.
// Scores, maxima, sums and accumulators are float32.
#include "attention_portion.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef uint32_t uint4_t __attribute__((ext_vector_type(4)));     // 16 bytes as one value (no aggregate copy)

constexpr int kItemInts = 8;
constexpr int kRowsPerTile = 16;
constexpr int kKeysPerBlock = 32;

union Pack16 {
    uint4 u;
    bf16x8_t v;
    uint2 half[2];
    uint16_t s[8];
};

__device__ __forceinline__ uint16_t bf16_bits(float f) { return from_float<bf16>(f).bits; }

// Shared memory, a part for each wavefront, used four times: three workgroups share a compute
// unit's 160 KB.  The wavefront turns its block of keys, which it reads from the cache row by row
// (whole key rows: contiguous runs the memory system streams much faster than the 64-byte pieces
// a fragment load straight from the cache would ask for), into fragments, the 16 keys of the
// first score tile and then the 16 of the second: [16 keys][HD + 8] bfloat16, rows padded so that
// the fragment reads spread over the banks.  Then it leaves its sums there for the merge, one
// half of the head after the other: [16 rows][HD / 2 + 4] floats.
template <int HD>
struct FewRowsShared {
    static constexpr int kKeyStride = HD + 8;                                      // elements
    static constexpr int kPartBytes = 16 * kKeyStride * 2;
    static constexpr int kMergeStride = HD / 2 + 4;                                // floats
    static_assert(kRowsPerTile * kMergeStride * 4 <= kPartBytes, "half of the sums fits a wavefront's part");
    alignas(16) unsigned char raw[4 * kPartBytes];
    float row_max[4][kRowsPerTile], row_sum[4][kRowsPerTile];
};

// How a block of 32 keys lies in pages: pages of a multiple of 4 or of 8 tokens, of 16, or of a power of two from 32 on.  The last two are
// known to hold a block in two pages, or in one: its page numbers are then the wavefront's, two scalar loads, and a lane's addresses a page's begin and its
// own place, where the others divide, multiply and look a page up for every load.  A wavefront has a vector unit to itself in a step of few requests, so every instruction in front of the
// loads counts (2,377 in the kernel for heads of 256 and pages of any multiple of 8, 1,184 in this one; decode steps at Gemma-2B sizes of 1 / 8 / 64 requests
// 1,293 / 1,375 / 2,113 to 1,260 / 1,326 / 2,078 us, Tokuvik's of 8 1,998 to 1,978, Duvozen's of 24 2,629 to 2,598).  The same bits.
enum Pages { kPagesOf4, kPagesOf8, kPagesOf16, kPagesFrom32 };

// One work item, by the whole workgroup of 256 threads.
// SPLIT: the weights of the second product keep 16 bits (rounded weight and remainder, two products).
template <int HD, Pages PAGES, bool SPLIT>
__device__ __forceinline__ void
few_rows_item(FewRowsShared<HD>& shared, uint32_t index, const bf16* __restrict__ qkv, const bf16* __restrict__ cache,
              const int* __restrict__ block_tables, const int* __restrict__ items, const int* __restrict__ live_items, 
              bf16* __restrict__ out, float* __restrict__ partial_o, float* __restrict__ partial_ml, int num_heads,
              int num_kv_heads, int group, int page_size, int max_pages, float scale_log2e, int window, int q_stride, float cap_scale,
              float softcap, const float* __restrict__ sinks) {
    constexpr bool V16 = PAGES != kPagesOf4, kWhole = PAGES == kPagesOf16 || PAGES == kPagesFrom32;
    if (PAGES == kPagesOf16) page_size = 16;
    constexpr int DC = HD / 32;   // 32-wide chunks of the head for the score product
    constexpr int DT = HD / 16;   // 16-row tiles of out^T
    constexpr int kKeyStride = FewRowsShared<HD>::kKeyStride, kPartBytes = FewRowsShared<HD>::kPartBytes;
    constexpr int kMergeStride = FewRowsShared<HD>::kMergeStride;
    unsigned char* const shared_raw = shared.raw;
    auto& row_max_s = shared.row_max;
    auto& row_sum_s = shared.row_sum;

    // A captured graph launches as many workgroups as its plan has room for items; the live ones come
    // first.  The item is asked for together with their number, not after it (there is an item, live
    // or stale, for every workgroup of the launch), and brings the segment's lengths with it: one trip
    // to memory for all of them.
    const int* item = items + static_cast<size_t>(index) * kItemInts;
    const int seg = item[0], kvh = item[1] & 0xffff, q_len = item[2], q_start = item[3];
    const int key_begin = item[4], key_end = item[5], partial_slot = item[6], ctx = item[7];
    const int live = live_items != nullptr ? live_items[0] : 0x7fffffff;
    if (static_cast<int>(index) >= live) return;
    const int row_begin = (item[1] >> 16) * kRowsPerTile;      // the tile's first row: 0 unless a token has more than 16 heads a group
    if (seg < 0) return;    // padding item
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int i = lane % 16, g = lane / 16;

    // ---- This lane's queries are asked for first: they arrive while the addresses of the keys and
    //      values are worked out.  (A lane without a row asks for the last one's: nothing of it is kept.) ----
    const int width = q_stride;                     // elements between two tokens' query rows
    const int total_rows = q_len * group;
    const int first_pos = ctx - q_len;
    const int seg_lo = lowest_key(first_pos, window);   // keys below may be given back
    const int row = row_begin + i;
    const bool row_valid = row < total_rows;
    int tok = 0, in_group = min(row, total_rows - 1);
    if (q_len > 1) {
        tok = in_group / group;
        in_group -= tok * group;
    }
    const int head = kvh * group + in_group;
    const int pos = first_pos + tok;
    const int lo = q_len > 1 ? lowest_key(pos, window) : seg_lo;
    // An item's keys lie within one aligned group of 128 (the host's chunk), so each of the four
    // wavefronts has at most one block of 32 keys and nothing is carried from block to block.
    const int blk = static_cast<int>(static_cast<unsigned>(key_begin) / kKeysPerBlock) + wave;
    const bool has_block = blk * kKeysPerBlock < key_end;
    bf16x8_t qreg[DC];
    if (has_block) {
        const bf16* qrow = qkv + static_cast<size_t>(q_start + tok) * width + static_cast<size_t>(head) * HD + 8 * g;
#pragma unroll
        for (int c = 0; c < DC; ++c) {
            Pack16 p;
            p.u = *reinterpret_cast<const uint4*>(qrow + c * 32);
            qreg[c] = p.v;
        }
    }

    const size_t page_elems = static_cast<size_t>(2) * num_kv_heads * page_size * HD;
    const size_t k_off = static_cast<size_t>(kvh) * page_size * HD;
    const size_t v_off = (static_cast<size_t>(num_kv_heads) + kvh) * page_size * HD;
    const int* table = block_tables + static_cast<size_t>(seg) * max_pages;
    // a block's keys as the cache holds them: 32 rows of HD, 16 bytes a lane and load
    constexpr int kPieces = HD / 8;                 // 16-byte pieces of a key row
    uint4_t kraw[DT];                               // 32 * kPieces / 64 = HD / 16 loads a lane
    Pack16 va_[DT];
    const int kbase = blk * kKeysPerBlock;
    float4_t acc[DT];
    float m_run = -INFINITY, l_run = 0.f;
    uint16_t* stage = reinterpret_cast<uint16_t*>(shared_raw + wave * kPartBytes);
    if (has_block) {
        // All loads of the block are issued before the first product needs one, so a block costs
        // one trip to memory after the block table's.  Keys beyond the request are masked later;
        // their table entry is clamped to the table's width (entries beyond a request's pages name
        // a valid page), not to the length.  A key's page and slot come from its place within the
        // block and one division a wavefront: the quotient by the page size as a float product,
        // exact for the few hundred values it is asked for here.
        if constexpr (kWhole) {
            // (page sizes are powers of two: shifts and masks)
            const int base_page = kbase >> __builtin_ctz(page_size), base_slot = kbase & (page_size - 1);
            const uint32_t number0 = table[min(base_page, max_pages - 1)], number1 = PAGES == kPagesOf16 ? table[min(base_page + 1, max_pages - 1)] : 0;
            const bf16 *page0 = cache + number0 * page_elems, *page1 = cache + number1 * page_elems;
            // pieces of 16 bytes in the order of the rows: half of the loads in either page, or all in one
            const uint32_t klane = lane * 8 + (PAGES == kPagesOf16 ? 0 : base_slot * HD);
#pragma unroll
            for (int j = 0; j < DT; ++j) {
                const bool second = PAGES == kPagesOf16 && j >= DT / 2;
                kraw[j] = __builtin_nontemporal_load(reinterpret_cast<const uint4_t*>((second ? page1 : page0) + k_off + klane + (second ? j - DT / 2 : j) * 512));
            }
            const bf16* vpage = (PAGES == kPagesOf16 && g >= 2 ? page1 : page0) + v_off;
            const uint32_t vlane = PAGES == kPagesOf16 ? i * 16 + (g % 2) * 8 : i * page_size + base_slot + 8 * g;
            const uint32_t vstep = PAGES == kPagesOf16 ? 256 : 16 * page_size;
#pragma unroll
            for (int t = 0; t < DT; ++t) va_[t].u = load_streamed(vpage + vlane + t * vstep);
        } else {
            const int base_page = kbase / page_size, base_slot = kbase % page_size;     // the same for all lanes
            const float inv_page = 1.f / static_cast<float>(page_size);
            auto place = [&](int within, int& page_index, int& slot) {
                const int x = base_slot + within;                                  // < page_size + 32
                const int q = static_cast<int>((static_cast<float>(x) + 0.5f) * inv_page);
                page_index = min(base_page + q, max_pages - 1);
                slot = x - q * page_size;
            };
            const bf16* kpiece[DT];
#pragma unroll
            for (int j = 0; j < DT; ++j) {
                // piece f of the block: key f / kPieces, its 8 elements f % kPieces; a wavefront's load
                // covers whole consecutive rows
                const int f = j * kWave + lane;
                int page_index, slot;
                place(f / kPieces, page_index, slot);
                kpiece[j] = cache + static_cast<size_t>(table[page_index]) * page_elems + k_off +
                            static_cast<size_t>(slot) * HD + (f % kPieces) * 8;
            }
            int vpage0, vslot0, vpage1 = 0, vslot1 = 0;
            place(V16 ? 8 * g : 4 * g, vpage0, vslot0);
            if (!V16) place(16 + 4 * g, vpage1, vslot1);
            const bf16* vbase0 = cache + static_cast<size_t>(table[vpage0]) * page_elems + v_off + vslot0;
            const bf16* vbase1 = cache + static_cast<size_t>(V16 ? 0 : table[vpage1]) * page_elems + v_off + vslot1;
#pragma unroll
            for (int j = 0; j < DT; ++j) kraw[j] = __builtin_nontemporal_load(reinterpret_cast<const uint4_t*>(kpiece[j]));
#pragma unroll
            for (int t = 0; t < DT; ++t) {
                const size_t drow = static_cast<size_t>(t * 16 + i) * page_size;
                if (V16) {
                    va_[t].u = load_streamed(vbase0 + drow);
                } else {
                    va_[t].half[0] = load_streamed8(vbase0 + drow);
                    va_[t].half[1] = load_streamed8(vbase1 + drow);
                }
            }
        }
        const bool edge = kbase < seg_lo || kbase + kKeysPerBlock > ctx;
        // ---- the keys through this wavefront's part of shared memory, then the scores: one tile
        //      of 16 keys after the other.  Which keys row i of a tile's first operand is: see the
        //      header for why. ----
        float4_t s[2];
#pragma unroll
        for (int t2 = 0; t2 < 2; ++t2) {
#pragma unroll
            for (int j = 0; j < DT; ++j) {
                const int f = lane + j * kWave;
                const int key = f / kPieces;
                const int tile = V16 ? (key / 4) % 2 : key / 16;
                const int at = V16 ? 4 * (key / 8) + key % 4 : key % 16;
                if (tile == t2)
                    *reinterpret_cast<uint4_t*>(stage + at * kKeyStride + (f % kPieces) * 8) = kraw[j];
            }
            // Lanes read what other lanes of the wavefront wrote, with no barrier between (a
            // wavefront's accesses to shared memory run in order): the compiler has to be told
            // that the memory changed, or a lane that wrote nothing keeps what it read before.
            asm volatile("" ::: "memory");
            float4_t sc = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < DC; ++c) {
                Pack16 a;
                a.u = *reinterpret_cast<const uint4*>(stage + i * kKeyStride + c * 32 + 8 * g);
                sc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, qreg[c], sc, 0, 0, 0);
            }
            s[t2] = sc;
        }
        // ---- mask, maximum, probabilities ----
        float sv[8];
        bool ok[8];
        float tile_max = -INFINITY;
        const int first_key = max(lo, key_begin), end_key = row_valid ? min(pos + 1, key_end) : 0;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int t2 = e / 4, v = e % 4;
            const int key = kbase + (V16 ? 8 * g + 4 * t2 + v : 16 * t2 + 4 * g + v);
            ok[e] = key >= first_key && key < end_key;
            // with a cap the score is scaled and bent here, and `scale_log2e` is log2(e) alone
            sv[e] = softcap > 0.f ? capped_score_fast(s[t2][v] * cap_scale, softcap) : s[t2][v];
            if (ok[e]) tile_max = fmaxf(tile_max, sv[e]);
        }
        tile_max = max_across(max_across(tile_max, 16), 32);
        m_run = tile_max;
        const float mc = (tile_max == -INFINITY ? 0.f : tile_max) * scale_log2e;
        Pack16 pv;
        float pe[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            pe[e] = ok[e] ? exp2_probability(fmaf(sv[e], scale_log2e, -mc)) : 0.f;
            l_run += pe[e];
        }
        pv.u = make_uint4(pack2_bf16(pe[0], pe[1]), pack2_bf16(pe[2], pe[3]), pack2_bf16(pe[4], pe[5]),
                          pack2_bf16(pe[6], pe[7]));
        Pack16 pr;      // SPLIT: what the rounding left out
        if (SPLIT)
            pr.u = make_uint4(pack2_bf16(bf16_remainder(pe[0]), bf16_remainder(pe[1])),
                              pack2_bf16(bf16_remainder(pe[2]), bf16_remainder(pe[3])),
                              pack2_bf16(bf16_remainder(pe[4]), bf16_remainder(pe[5])),
                              pack2_bf16(bf16_remainder(pe[6]), bf16_remainder(pe[7])));
        // the row's sum over its four lanes
        l_run = sum_across(sum_across(l_run, 16), 32);
        // ---- out^T = V^T . P^T ----
        if (edge) {
            // keys outside the request (stale slots, pages given back) may hold anything,
            // NaN included; 0 * NaN would poison the sum, so they are cleared
            uint32_t keep[4] = {0, 0, 0, 0};
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int key = kbase + (V16 ? 8 * g + e : (e < 4 ? 4 * g + e : 16 + 4 * g + e - 4));
                if (key < ctx && key >= seg_lo) keep[e / 2] |= 0xffffu << (16 * (e % 2));
            }
#pragma unroll
            for (int t = 0; t < DT; ++t)
                va_[t].u = make_uint4(va_[t].u.x & keep[0], va_[t].u.y & keep[1], va_[t].u.z & keep[2], va_[t].u.w & keep[3]);
        }
#pragma unroll
        for (int t = 0; t < DT; ++t) {
            const Pack16 a = va_[t];
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, pv.v, float4_t{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
            if (SPLIT) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, pr.v, acc[t], 0, 0, 0);
        }
    } else {
#pragma unroll
        for (int t = 0; t < DT; ++t) acc[t] = float4_t{0.f, 0.f, 0.f, 0.f};
    }

    // ---- merge: every wavefront leaves its sums in its own part of shared memory (it has read its
    //      keys from there already), one half of the head after the other; of each half every
    //      wavefront takes every fourth tile of 16 elements and combines the four wavefronts' sums of
    //      that tile, always in the order 0, 1, 2, 3.
    //      lane (i, g) holds out^T[16t + 4g + v][row i]: elements d = 16t + 4g + v of row i ----
    float* mine = reinterpret_cast<float*>(stage);
    if (g == 0) {
        row_max_s[wave][i] = m_run;
        row_sum_s[wave][i] = l_run;
    }
    float f_of[4] = {0.f, 0.f, 0.f, 0.f};
    float m_all = -INFINITY, l_all = 0.f, inv = 0.f;
    bf16* orow = out + (static_cast<size_t>(q_start + tok) * num_heads + head) * HD;
    const size_t prow = static_cast<size_t>(max(partial_slot, 0)) * kRowsPerTile + (row - row_begin);
    float* po = partial_o + prow * HD;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        if (half) __syncthreads();          // the first half has been read
#pragma unroll
        for (int t = 0; t < DT / 2; ++t)
            *reinterpret_cast<float4_t*>(mine + i * kMergeStride + t * 16 + 4 * g) = acc[half * (DT / 2) + t];
        __syncthreads();
        if (!half) {
            float m_of[4], l_of[4];
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                m_of[w] = row_max_s[w][i];
                l_of[w] = row_sum_s[w][i];
                m_all = fmaxf(m_all, m_of[w]);
            }
            const float m_use = m_all == -INFINITY ? 0.f : m_all;
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                f_of[w] = exp2f((m_of[w] - m_use) * scale_log2e);       // 0 for a wavefront without keys
                l_all = fmaf(l_of[w], f_of[w], l_all);
            }
            // a sink: exp(sink of the head) once more in the denominator of a row that is finished here
            // (the maximum is held in the exponent's own units: times scale_log2e it is in powers of two)
            const float sink_term = (sinks && partial_slot < 0) ? exp2f(sinks[head] * 1.4426950408889634f - m_use * scale_log2e) : 0.f;
            inv = 1.f / (l_all + sink_term);
        }
        if (row_valid) {
#pragma unroll
            for (int t0 = 0; t0 < DT / 2; t0 += 4) {
                const int t = t0 + wave;
                if (t < DT / 2) {
                    float4_t sum = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int w = 0; w < 4; ++w) {
                        const float* part = reinterpret_cast<const float*>(shared_raw + w * kPartBytes);
                        const float4_t v = *reinterpret_cast<const float4_t*>(part + i * kMergeStride + t * 16 + 4 * g);
#pragma unroll
                        for (int e = 0; e < 4; ++e) sum[e] = fmaf(v[e], f_of[w], sum[e]);
                    }
                    const int d = (half * (DT / 2) + t) * 16 + 4 * g;
                    if (partial_slot < 0) {
                        uint2 w2;
                        w2.x = pack2_bf16(sum[0] * inv, sum[1] * inv);
                        w2.y = pack2_bf16(sum[2] * inv, sum[3] * inv);
                        *reinterpret_cast<uint2*>(orow + d) = w2;
                    } else {
                        *reinterpret_cast<float4_t*>(po + d) = sum;
                    }
                }
            }
        }
    }
    if (row_valid && partial_slot >= 0 && wave == 0 && g == 0) {
        partial_ml[prow * 2] = m_all;
        partial_ml[prow * 2 + 1] = l_all;
    }
}

// Three workgroups a compute unit (168 registers a lane) where the kernel fits them without spilling;
// two for the head sizes and page sizes whose staging needs more.
template <int HD, Pages PAGES, bool SPLIT>
__global__ void __launch_bounds__(256, (HD <= 160 || (HD == 256 && PAGES != kPagesOf4)) ? 3 : 2)
paged_attention_mfma_kernel(const int* __restrict__ items, const int* __restrict__ live_items, const int* __restrict__ block_tables,
                            const bf16* __restrict__ qkv, const bf16* __restrict__ cache, int group, int window, int q_stride, int max_pages,
                            int num_kv_heads, int page_size, bf16* __restrict__ out, float* __restrict__ partial_o,
                            float* __restrict__ partial_ml, int num_heads, float scale_log2e, float cap_scale, float softcap,
                            const float* __restrict__ sinks) {
    // (what stands in front of the loads is asked for first: sixteen words of arguments are in registers when a wavefront begins)
    __shared__ FewRowsShared<HD> shared;
    few_rows_item<HD, PAGES, SPLIT>(shared, blockIdx.x, qkv, cache, block_tables, items, live_items, out, partial_o, partial_ml,
                                    num_heads, num_kv_heads, group, page_size, max_pages, scale_log2e, window, q_stride,
                                    cap_scale, softcap, sinks);
}

// A step that carries both prompt portions and decoded tokens: the items of both kernels in one launch, each with the bits it
// has in its own.  A portion's items are few (at most two a compute unit) and a chain of blocks each, which waits for memory's
// latency and leaves its bandwidth idle; the decoded tokens' are many and bound by that bandwidth.  One after the other they took
// the sum of both (8 heads of 256 on one, a portion of 448 tokens over 448 to 1,000 keys beside 60 tokens over 1,500 each: 19.7 + 17.1 us), in one
// launch 23.5 us.  A compute unit holds two of its workgroups (shared memory and registers of the portions), where it held
// three of the decoded tokens' kernel; two are enough beside the portions.
// The kinds alternate in runs of workgroups, eight an XCD, portions first: with all portions in front (runs of 512), 30 tokens
// over 1,250 keys beside 448 over 896 (16 heads of 128 on four; with the sum of the pieces) took 30.4 us, in runs of 256 / 64
// 30.2 / 29.8, in runs of 8, one an XCD, 32.2; with few items all are the same.
// With heads of 64 a compute unit holds four workgroups, and a run of eight an XCD, whose 32 units take them in turn, would bring the same
// unit the same kind every time: four portions here, none there (448 tokens over 3,000 keys beside 24 over 800, 64 heads of 64 on eight: 97.7 us, in
// runs of one workgroup a unit 71.3, in two launches 78).
template <int HD> constexpr int kRoleRun = HD == 64 ? 256 : 64;

template <int HD, Pages PAGES, bool SPLIT>
__global__ void __launch_bounds__(kPrefillThreads, 2)
paged_attention_both_kernel(const bf16* __restrict__ qkv, const bf16* __restrict__ cache,
                            const int* __restrict__ block_tables, const int* __restrict__ portion_items, int num_portions,
                            const int* __restrict__ items, int num_items,
                            const int* __restrict__ live_items, const int* __restrict__ seg_q_start, const int* __restrict__ seg_q_len,
                            const int* __restrict__ seg_ctx_len, bf16* __restrict__ out,
                            float* __restrict__ partial_o, float* __restrict__ partial_ml, int num_heads,
                            int num_kv_heads, int group, int page_size, int max_pages, float scale_log2e, int window,
                            int q_stride, float cap_scale, float softcap, const float* __restrict__ sinks) {
    __shared__ union Either {
        PortionShared<HD> portion;
        FewRowsShared<HD> few;
    } shared;
    // runs of either kind in turn, then what is left of both lists
    const int b = blockIdx.x, shorter = min(num_portions, num_items) / kRoleRun<HD> * kRoleRun<HD>;
    bool portion;
    int index;
    if (b < 2 * shorter) {
        portion = b / kRoleRun<HD> % 2 == 0;
        index = b / (2 * kRoleRun<HD>) * kRoleRun<HD> + b % kRoleRun<HD>;
    } else {
        index = b - shorter;
        portion = index < num_portions;
        if (!portion) index = b - num_portions;
    }
    if (portion)
        portion_item<HD, SPLIT>(shared.portion, index, qkv, cache, block_tables, portion_items, seg_q_start, seg_q_len,
                                seg_ctx_len, out, partial_o, partial_ml, num_heads, num_kv_heads, page_size, max_pages,
                                scale_log2e, window, q_stride, cap_scale, softcap, sinks);
    else
        few_rows_item<HD, PAGES, SPLIT>(shared.few, index, qkv, cache, block_tables, items, live_items, out, partial_o, partial_ml,
                                        num_heads, num_kv_heads, group, page_size, max_pages, scale_log2e, window, q_stride,
                                        cap_scale, softcap, sinks);
}

// Combines the partial results of a (segment, key/value head) whose keys were split over workgroups.
// reduce items: seg, kvh, first partial slot, number of splits, first row, slots between splits, the segment's rows, the place of its
// first token (looked up by the segment they were a trip to memory and a division more: Tokuvik's decode step of 8 requests 1,978 to 1,960 us,
// Gemma-2B's of 1, 8 and 64 2 us less each).
template <int HD>
__global__ void __launch_bounds__(HD)
attention_reduce_kernel(const int* __restrict__ reduce_items, const float* __restrict__ partial_o, const float* __restrict__ partial_ml,
                             bf16* __restrict__ out, int group, int num_heads, float scale_log2e, const float* __restrict__ sinks) {
    // one workgroup per (item, row); one thread per element of the head; the loads of the
    // splits do not depend on each other.  Reduce items are 8 int32: segment, key/value head, first
    // slot, number of splits, first row of the tile within the segment, slots between two splits.
    const int* item = reduce_items + static_cast<size_t>(blockIdx.x) * kItemInts;
    const int seg = item[0], kvh = item[1], first = item[2], splits = item[3], row0 = item[4], rows = item[6], q_start = item[7];
    if (seg < 0) return;
    const size_t stride = static_cast<size_t>(item[5]) * kRowsPerTile;     // rows between two splits
    const int r = blockIdx.y, d = threadIdx.x;
    if (row0 + r >= rows) return;
    const float* ml = partial_ml + (static_cast<size_t>(first) * kRowsPerTile + r) * 2;
    const float* po = partial_o + (static_cast<size_t>(first) * kRowsPerTile + r) * HD + d;
    // One pass in groups of eight splits: all loads of a group are issued together, and the sums are
    // rescaled when a group raises the maximum, so the kernel makes one trip to memory per group.
    float m = -INFINITY, num = 0.f, den = 0.f;
    for (int s0 = 0; s0 < splits; s0 += 8) {
        float ms[8], ls[8], ps[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            // a split beyond the last reads the last one again (the same addresses) and does not count
            const bool ok = s0 + u < splits;
            const size_t at = static_cast<size_t>(ok ? s0 + u : splits - 1) * stride;
            const float m_at = ml[at * 2];
            ms[u] = ok ? m_at : -INFINITY;
            ls[u] = ml[at * 2 + 1];
            ps[u] = po[at * HD];
        }
        float m_new = m;
#pragma unroll
        for (int u = 0; u < 8; ++u) m_new = fmaxf(m_new, ms[u]);
        if (m_new == -INFINITY) continue;       // nothing seen yet
        const float keep = m == -INFINITY ? 0.f : exp2f((m - m_new) * scale_log2e);
        num *= keep;
        den *= keep;
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const float f = ms[u] == -INFINITY ? 0.f : exp2f((ms[u] - m_new) * scale_log2e);
            num = fmaf(ps[u], f, num);
            den = fmaf(ls[u], f, den);
        }
        m = m_new;
    }
    const int row = row0 + r, tok = rows > group ? row / group : 0, head = kvh * group + row - tok * group;
    if (sinks) den += exp2f(sinks[head] * 1.4426950408889634f - m * scale_log2e);
    out[(static_cast<size_t>(q_start + tok) * num_heads + head) * HD + d] = from_float<bf16>(num / den);
}

// The same sums for steps with many tiles to combine (the pieces of a long prompt): a thread takes
// four consecutive elements of a row (16-byte loads), a workgroup of HD threads four rows.  Every
// element goes through the operations of the kernel above in the same order, so which of the two
// runs changes no bit of the result.
template <int HD>
__global__ void __launch_bounds__(HD)
attention_reduce_wide_kernel(const int* __restrict__ reduce_items, const float* __restrict__ partial_o, const float* __restrict__ partial_ml,
                             bf16* __restrict__ out, int group, int num_heads, float scale_log2e, const float* __restrict__ sinks) {
    const int* item = reduce_items + static_cast<size_t>(blockIdx.x) * kItemInts;
    const int seg = item[0], kvh = item[1], first = item[2], splits = item[3], row0 = item[4], rows = item[6], q_start = item[7];
    if (seg < 0) return;
    const size_t stride = static_cast<size_t>(item[5]) * kRowsPerTile;     // rows between two splits
    constexpr int kQuads = HD / 4;
    const int r = blockIdx.y * 4 + threadIdx.x / kQuads, d = (threadIdx.x % kQuads) * 4;
    if (row0 + r >= rows) return;
    const float* ml = partial_ml + (static_cast<size_t>(first) * kRowsPerTile + r) * 2;
    const float* po = partial_o + (static_cast<size_t>(first) * kRowsPerTile + r) * HD + d;
    float m = -INFINITY, den = 0.f;
    float4_t num = float4_t{0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < splits; s0 += 8) {
        float ms[8], ls[8];
        float4_t ps[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const bool ok = s0 + u < splits;
            const size_t at = static_cast<size_t>(ok ? s0 + u : splits - 1) * stride;
            const float2 pair = *reinterpret_cast<const float2*>(ml + at * 2);
            ms[u] = ok ? pair.x : -INFINITY;
            ls[u] = pair.y;
            ps[u] = *reinterpret_cast<const float4_t*>(po + at * HD);
        }
        float m_new = m;
#pragma unroll
        for (int u = 0; u < 8; ++u) m_new = fmaxf(m_new, ms[u]);
        if (m_new == -INFINITY) continue;       // nothing seen yet
        const float keep = m == -INFINITY ? 0.f : exp2f((m - m_new) * scale_log2e);
        num *= keep;
        den *= keep;
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const float f = ms[u] == -INFINITY ? 0.f : exp2f((ms[u] - m_new) * scale_log2e);
#pragma unroll
            for (int v = 0; v < 4; ++v) num[v] = fmaf(ps[u][v], f, num[v]);
            den = fmaf(ls[u], f, den);
        }
        m = m_new;
    }
    const int row = row0 + r, tok = rows > group ? row / group : 0, head = kvh * group + row - tok * group;
    if (sinks) den += exp2f(sinks[head] * 1.4426950408889634f - m * scale_log2e);
    uint2 w;
    w.x = pack2_bf16(num[0] / den, num[1] / den);
    w.y = pack2_bf16(num[2] / den, num[3] / den);
    *reinterpret_cast<uint2*>(out + (static_cast<size_t>(q_start + tok) * num_heads + head) * HD + d) = w;
}

namespace {

struct AttentionArguments {
    const bf16* qkv;
    const bf16* cache;
    const int* block_tables;
    const int* portion_items;      // null: the step has none, or they have been launched by themselves
    int num_portions;
    const int* items;
    const int* live_items;
    int num_items;
    const int* reduce_items;
    int num_reduce_items;
    const int* seg_q_start;
    const int* seg_q_len;
    const int* seg_ctx_len;
    bf16* out;
    float* partial_o;
    float* partial_ml;
    int num_heads, num_kv_heads, page_size, max_pages;
    float scale_log2e;
    int window;
    int q_stride;
    float cap_scale, softcap;
    int split_weights;
    const float* sinks;
    hipStream_t stream;
};

template <int HD, Pages PAGES, bool SPLIT>
int launch_items(const AttentionArguments& a) {
    paged_attention_mfma_kernel<HD, PAGES, SPLIT><<<a.num_items, 256, 0, a.stream>>>(
        a.items, a.live_items, a.block_tables, a.qkv, a.cache, a.num_heads / a.num_kv_heads, a.window, a.q_stride, a.max_pages,
        a.num_kv_heads, a.page_size, a.out, a.partial_o, a.partial_ml, a.num_heads, a.scale_log2e, a.cap_scale, a.softcap, a.sinks);
    return 0;
}

template <int HD, Pages PAGES, bool SPLIT>
int launch_both(const AttentionArguments& a) {
    paged_attention_both_kernel<HD, PAGES, SPLIT><<<a.num_portions + a.num_items, kPrefillThreads, 0, a.stream>>>(
        a.qkv, a.cache, a.block_tables, a.portion_items, a.num_portions, a.items, a.num_items, a.live_items, a.seg_q_start,
        a.seg_q_len, a.seg_ctx_len, a.out, a.partial_o, a.partial_ml, a.num_heads, a.num_kv_heads, a.num_heads / a.num_kv_heads, a.page_size, a.max_pages,
        a.scale_log2e, a.window, a.q_stride, a.cap_scale, a.softcap, a.sinks);
    return 0;
}

template <int HD>
int launch_all(const AttentionArguments& a) {
    if (a.num_portions > 0) {
        if constexpr (HD == 64 || HD == 128 || HD == 256) {
            const int status = a.page_size == 16 ? (a.split_weights ? launch_both<HD, kPagesOf16, true>(a) : launch_both<HD, kPagesOf16, false>(a))
                                                 : (a.split_weights ? launch_both<HD, kPagesOf8, true>(a) : launch_both<HD, kPagesOf8, false>(a));
            if (status != 0) return status;
        } else {
            return -1;
        }
    } else if (a.num_items > 0) {
        const bool power = (a.page_size & (a.page_size - 1)) == 0;
#define ITEMS(PAGES) (a.split_weights ? launch_items<HD, PAGES, true>(a) : launch_items<HD, PAGES, false>(a))
        const int status = a.page_size == 16             ? ITEMS(kPagesOf16)
                           : power && a.page_size >= 32 ? ITEMS(kPagesFrom32)
                           : a.page_size % 8 == 0        ? ITEMS(kPagesOf8)
                                                         : ITEMS(kPagesOf4);
#undef ITEMS
        if (status != 0) return status;
    }
    if (a.num_reduce_items >= 64) {
        attention_reduce_wide_kernel<HD><<<dim3(a.num_reduce_items, kRowsPerTile / 4), HD, 0, a.stream>>>(
            a.reduce_items, a.partial_o, a.partial_ml, a.out, a.num_heads / a.num_kv_heads, a.num_heads, a.scale_log2e, a.sinks);
    } else if (a.num_reduce_items > 0) {
        attention_reduce_kernel<HD><<<dim3(a.num_reduce_items, kRowsPerTile), HD, 0, a.stream>>>(
            a.reduce_items, a.partial_o, a.partial_ml, a.out, a.num_heads / a.num_kv_heads, a.num_heads, a.scale_log2e, a.sinks);
    }
    return launch_status();
}

}  // namespace

// Returns 0, a HIP error code, or -1 for sizes these kernels do not take.  `live_items`: null, or a
// device int that says how many of the `num_items` items count (a captured graph's plan).
// `portion_items`: null, or the items of the prompt portions of the same step, which then run in the same launch: pages of a power
// of two from 8, heads of 64, 128 and 256.
WLLM_API int wllm_paged_attention_mfma(const void* qkv, const void* cache, const int* block_tables,
                                       const int* portion_items, int num_portions, const int* items,
                                       const int* live_items, int num_items, const int* reduce_items,
                                       int num_reduce_items, const int* seg_q_start, const int* seg_q_len,
                                       const int* seg_ctx_len, void* out, float* partial_o, float* partial_ml,
                                       int num_heads, int num_kv_heads, int head_dim, int page_size, int max_pages,
                                       float scale, int window, int q_stride, float softcap, int split_weights,
                                       const float* sinks, hipStream_t stream) {
    if (head_dim % 32 != 0 || head_dim < 32 || head_dim > 256 || page_size % 4 != 0 || num_heads % num_kv_heads != 0 ||
        num_heads >= (1 << 16))       // an item holds a key/value head and a tile's first row in 16 bits each
        return -1;
    if (q_stride < num_heads * head_dim || q_stride % 8 != 0 || softcap < 0.f) return -1;
    if (num_portions < 0 || (num_portions > 0 && (portion_items == nullptr || num_items <= 0 || page_size < 8 ||
                                                  (page_size & (page_size - 1)) != 0)))
        return -1;
    // with a cap the kernel scales and bends the score itself; the softmax then works on final scores
    const float in_exponent = softcap > 0.f ? 1.f : scale;
    const float cap_scale = softcap > 0.f ? scale / softcap : 0.f;
    const AttentionArguments a = {static_cast<const bf16*>(qkv), static_cast<const bf16*>(cache), block_tables,
                                  portion_items, num_portions, items, live_items, num_items, reduce_items, num_reduce_items, seg_q_start, seg_q_len,
                                  seg_ctx_len, static_cast<bf16*>(out), partial_o, partial_ml, num_heads, num_kv_heads,
                                  page_size, max_pages, in_exponent * 1.4426950408889634f, window, q_stride, cap_scale,
                                  softcap, split_weights, sinks, stream};
    switch (head_dim) {
        case 32: return launch_all<32>(a);
        case 64: return launch_all<64>(a);
        case 96: return launch_all<96>(a);
        case 128: return launch_all<128>(a);
        case 160: return launch_all<160>(a);
        case 192: return launch_all<192>(a);
        case 224: return launch_all<224>(a);
        case 256: return launch_all<256>(a);
        default: return -1;
    }
}
