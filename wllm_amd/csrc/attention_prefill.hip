// Paged attention for long segments (prompt portions) on the matrix cores, bfloat16: the keys
// and values of a block of 32 keys are staged through shared memory once per workgroup and read
// by all four wavefronts; a wavefront owns one tile of 16 query rows.  A workgroup is 64 rows of one
// (segment, key/value head): rows are (token, query head of the group) pairs, row r = token * G +
// head.  (With two tiles a wavefront, every fragment read from shared memory would feed two
// products, but the registers of 128 rows leave room for one workgroup a compute unit; with 64
// rows two workgroups share it and hide each other's waits, which measured a quarter faster.)
//
// The products are those of `attention_mfma.hip` (v_mfma_f32_16x16x32_bf16, scores transposed so
// that a lane's values all belong to one query row, probabilities fed to the second product from
// the registers they were computed in).  Staging: while the products of block b run from shared
// memory, the global loads of block b+1 are in flight into registers; they are written to shared
// memory after a barrier.  Keys land as [32][HD] rows (padded), values as [HD][32] rows whose 32
// keys are permuted so that the 8 keys a lane needs are contiguous.  Keys outside the request
// (stale slots of the last page, pages a window gave back) are cleared while staging, so that a
// NaN there cannot meet a zero probability.
#include "attention_portion.h"

template <int HD>
struct PrefillSmem {
    static constexpr int kStrideK = HD + 8;            // elements; the pad spreads rows over banks
    static constexpr int kStrideV = kBlockKeys + 8;
    static constexpr int kBytes = (kBlockKeys * kStrideK + HD * kStrideV) * 2;
};

// prefill items: seg, kvh, first row, first key, end key, partial slot (-1: the workgroup walks all
// the keys of its rows and writes the result itself), 2 unused.  Items that split the keys of a
// block of rows write, per tile of 16 rows, an unnormalised accumulator and (maximum, sum) into
// slot `partial slot + tile`, which `attention_reduce_kernel` combines.
// RTW: tiles of 16 rows per wavefront (1 or 2).  SPLIT: the weights of the second product keep 16 bits (the
// rounded weight and what the rounding left out, two products).
template <int HD, int RTW, bool SPLIT>
__global__ void __launch_bounds__(kPrefillThreads, RTW == 1 ? 2 : 1)
paged_attention_prefill_kernel(const bf16* __restrict__ qkv, const bf16* __restrict__ cache,
                               const int* __restrict__ block_tables, const int* __restrict__ items,
                               const int* __restrict__ seg_q_start, const int* __restrict__ seg_q_len,
                               const int* __restrict__ seg_ctx_len, bf16* __restrict__ out,
                               float* __restrict__ partial_o, float* __restrict__ partial_ml, int num_heads,
                               int num_kv_heads, int page_size, int max_pages, float scale_log2e, int window,
                               int q_stride, float cap_scale, float softcap, const float* __restrict__ sinks) {
    constexpr int DC = HD / 32, DT = HD / 16;
    constexpr int SK = PrefillSmem<HD>::kStrideK, SV = PrefillSmem<HD>::kStrideV;
    __shared__ __align__(16) uint16_t k_s[kBlockKeys * SK];
    __shared__ __align__(16) uint16_t v_s[HD * SV];
    __shared__ int table_s[kMaxTablePages];     // the pages of this item's keys: lookups never leave the CU

    const int* item = items + static_cast<size_t>(blockIdx.x) * kPrefillItemInts;
    const int seg = item[0], kvh = item[1], row_begin = item[2];
    const int key_begin = item[3], key_end = item[4], partial_slot = item[5];
    if (seg < 0) return;
    const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    const int i = lane % 16, g = lane / 16;
    const int group = num_heads / num_kv_heads;
    const int q_start = seg_q_start[seg], q_len = seg_q_len[seg], ctx = seg_ctx_len[seg];
    const int total_rows = q_len * group;
    const int first_pos = ctx - q_len;
    const int seg_lo = lowest_key(first_pos, window);
    const int width = q_stride;         // elements between two tokens' query rows
    const size_t page_elems = static_cast<size_t>(2) * num_kv_heads * page_size * HD;
    const size_t k_off = static_cast<size_t>(kvh) * page_size * HD;
    const size_t v_off = (static_cast<size_t>(num_kv_heads) + kvh) * page_size * HD;

    // this wavefront's two tiles of rows
    constexpr int kWaveRows = 16 * RTW, kPrefillRows = kPrefillWaves * kWaveRows;
    const int wr0 = row_begin + wave * kWaveRows;
    int row[RTW], tok[RTW], head[RTW], pos[RTW], lo[RTW];
    bool row_valid[RTW];
    bf16x8_t qreg[RTW][DC];
#pragma unroll
    for (int rt = 0; rt < RTW; ++rt) {
        row[rt] = wr0 + rt * 16 + i;
        row_valid[rt] = row[rt] < total_rows;
        tok[rt] = row_valid[rt] ? row[rt] / group : 0;
        head[rt] = kvh * group + (row_valid[rt] ? row[rt] % group : 0);
        pos[rt] = first_pos + tok[rt];
        lo[rt] = lowest_key(pos[rt], window);
        const bf16* qrow = qkv + static_cast<size_t>(q_start + tok[rt]) * width + static_cast<size_t>(head[rt]) * HD;
#pragma unroll
        for (int c = 0; c < DC; ++c) {
            PPack p;
            p.u = row_valid[rt] ? *reinterpret_cast<const uint4*>(qrow + c * 32 + 8 * g) : make_uint4(0, 0, 0, 0);
            qreg[rt][c] = p.v;
        }
    }
    // per row tile: the lowest position and the highest window start of its rows (wavefront-wide)
    int t_pos_min[RTW], t_lo_max[RTW];
#pragma unroll
    for (int rt = 0; rt < RTW; ++rt) {
        const int first = wr0 + rt * 16, last = min(total_rows - 1, first + 15);
        t_pos_min[rt] = first < total_rows ? first_pos + first / group : -1;
        const int pmax = first_pos + max(last, 0) / group;
        t_lo_max[rt] = lowest_key(pmax, window);
        if (last < first + 15) t_pos_min[rt] = -1;      // a tile with rows beyond the segment always masks
    }
    // keys the wavefront's rows can need
    const bool wave_active = wr0 < total_rows;
    const int w_last_row = min(total_rows - 1, wr0 + kWaveRows - 1);
    const int w_hi = wave_active ? first_pos + w_last_row / group + 1 : 0;                       // exclusive
    const int w_lo = lowest_key(first_pos + wr0 / group, window);
    // keys the workgroup stages: from the first wavefront's lowest to the last row's highest
    const int b_last_row = min(total_rows - 1, row_begin + kPrefillRows - 1);
    const int b_hi = first_pos + b_last_row / group + 1;
    const int b_lo = lowest_key(first_pos + row_begin / group, window);
    const int blk_first = max(b_lo, key_begin) / kBlockKeys;
    const int blk_end = (min(b_hi, key_end) + kBlockKeys - 1) / kBlockKeys;
    // the pages of keys blk_first * 32 .. blk_end * 32 (clamped to the request's keys)
    const int page_base = blk_first * kBlockKeys / page_size;
    if (blk_first < blk_end) {
        const int* table_g = block_tables + static_cast<size_t>(seg) * max_pages + page_base;
        const int page_last = (min(blk_end * kBlockKeys, ctx) - 1) / page_size;
        const int count = min(min(max_pages - 1, page_last) - page_base + 1, kMaxTablePages);
        for (int p = tid; p < count; p += kPrefillThreads) table_s[p] = table_g[p];
    }

    float4_t acc[RTW][DT];
    float m_run[RTW], l_run[RTW];
#pragma unroll
    for (int rt = 0; rt < RTW; ++rt) {
        m_run[rt] = -INFINITY;
        l_run[rt] = 0.f;
#pragma unroll
        for (int t = 0; t < DT; ++t) acc[rt][t] = float4_t{0.f, 0.f, 0.f, 0.f};
    }

    // ---- staging.  Keys: kTPK threads share a key row and take its 16-byte chunks in turn, so a
    //      thread looks up one page per block.  Values: a thread keeps one group of 4 keys (j) and
    //      walks the rows d of the transposed page, again one page lookup per block. ----
    constexpr int kTPK = kPrefillThreads / kBlockKeys;              // threads per key row
    constexpr int KCH = (HD / 8 + kTPK - 1) / kTPK;
    constexpr int kRowsPerPass = kPrefillThreads / 8;               // value rows staged per pass
    constexpr int VCH = (HD + kRowsPerPass - 1) / kRowsPerPass;
    const int k_key = tid / kTPK, k_lane = tid % kTPK;
    const int v_j = tid % 8, v_d0 = tid / 8;
    uint4 kreg_a[KCH];
    uint2 vreg_a[VCH];
    const int page_shift = (page_size & (page_size - 1)) == 0 ? __builtin_ctz(page_size) : -1;
    auto page_of = [&](int key, int& slot) -> int {
        if (page_shift >= 0) {
            slot = key & (page_size - 1);
            return table_s[(key >> page_shift) - page_base];
        }
        slot = key % page_size;
        return table_s[key / page_size - page_base];
    };
    auto fetch = [&](uint4* kreg, uint2* vreg, int kbase) {
        {
            const int key = kbase + k_key;
            const bool ok = key < ctx && key >= seg_lo;
            const int kk = min(key, ctx - 1);
            int slot;
            const int page = page_of(kk, slot);
            const bf16* src = cache + static_cast<size_t>(page) * page_elems + k_off + static_cast<size_t>(slot) * HD;
#pragma unroll
            for (int u = 0; u < KCH; ++u) {
                const int chunk = k_lane + u * kTPK;
                kreg[u] = (ok && chunk < HD / 8) ? *reinterpret_cast<const uint4*>(src + chunk * 8)
                                                 : make_uint4(0, 0, 0, 0);
            }
        }
        {
            const int key = kbase + 4 * v_j;                 // group v_j: keys key .. key + 3
            const int kk = min(key, ctx - 1) & ~3;
            int slot;
            const int page = page_of(kk, slot);
            const bf16* src = cache + static_cast<size_t>(page) * page_elems + v_off + slot;
            // keys of the group that are not the request's are cleared
            uint2 keep = make_uint2(0xffffffffu, 0xffffffffu);
            if (key + 3 >= ctx || key < seg_lo) {
                const bool k0 = key < ctx && key >= seg_lo, k1 = key + 1 < ctx && key + 1 >= seg_lo;
                const bool k2 = key + 2 < ctx && key + 2 >= seg_lo, k3 = key + 3 < ctx && key + 3 >= seg_lo;
                keep.x = (k0 ? 0x0000ffffu : 0u) | (k1 ? 0xffff0000u : 0u);
                keep.y = (k2 ? 0x0000ffffu : 0u) | (k3 ? 0xffff0000u : 0u);
            }
#pragma unroll
            for (int u = 0; u < VCH; ++u) {
                const int d = min(v_d0 + u * kRowsPerPass, HD - 1);
                uint2 v = *reinterpret_cast<const uint2*>(src + static_cast<size_t>(d) * page_size);
                v.x &= keep.x;
                v.y &= keep.y;
                vreg[u] = v;
            }
        }
    };
    auto stage = [&](const uint4* kreg, const uint2* vreg) {
#pragma unroll
        for (int u = 0; u < KCH; ++u) {
            const int chunk = k_lane + u * kTPK;
            if (chunk < HD / 8) *reinterpret_cast<uint4*>(&k_s[k_key * SK + chunk * 8]) = kreg[u];
        }
#pragma unroll
        for (int u = 0; u < VCH; ++u) {
            const int d = v_d0 + u * kRowsPerPass;
            // keys 4j..4j+3 go to positions 8*(j%4) + 4*(j/4): a lane's keys {4g..4g+3, 16+4g..} become contiguous
            if (d < HD) *reinterpret_cast<uint2*>(&v_s[d * SV + 8 * (v_j % 4) + 4 * (v_j / 4)]) = vreg[u];
        }
    };

    __syncthreads();      // the block table is in shared memory
    // the loads of the next block are in flight while the products of this one run
    if (blk_first < blk_end) fetch(kreg_a, vreg_a, blk_first * kBlockKeys);
    for (int blk = blk_first; blk < blk_end; ++blk) {
        const int kbase = blk * kBlockKeys;
        __syncthreads();                 // everyone is done with the previous block's tiles
        stage(kreg_a, vreg_a);
        __syncthreads();
        if (blk + 1 < blk_end) fetch(kreg_a, vreg_a, kbase + kBlockKeys);
        if (!wave_active || kbase >= w_hi || kbase + kBlockKeys <= w_lo) continue;
        // ---- scores: tile t2 holds keys kbase + 16*t2 + (0..15); lane (i, g) gets keys 16*t2 + 4g + v ----
        float4_t s[RTW][2];
#pragma unroll
        for (int t2 = 0; t2 < 2; ++t2) {
            float4_t sc[RTW];
#pragma unroll
            for (int rt = 0; rt < RTW; ++rt) sc[rt] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < DC; ++c) {
                PPack a;
                a.u = *reinterpret_cast<const uint4*>(&k_s[(16 * t2 + i) * SK + c * 32 + 8 * g]);
#pragma unroll
                for (int rt = 0; rt < RTW; ++rt)
                    sc[rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, qreg[rt][c], sc[rt], 0, 0, 0);
            }
#pragma unroll
            for (int rt = 0; rt < RTW; ++rt) s[rt][t2] = sc[rt];
        }
        // ---- softmax bookkeeping per row tile ----
        PPack pv[RTW], pr[RTW];
        float alpha[RTW];
        bool rescale[RTW];
#pragma unroll
        for (int rt = 0; rt < RTW; ++rt) {
            float sv[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) sv[e] = s[rt][e / 4][e % 4];
            if (softcap > 0.f) {        // the score is scaled and bent here; `scale_log2e` is then log2(e) alone
#pragma unroll
                for (int e = 0; e < 8; ++e) sv[e] = capped_score_fast(sv[e] * cap_scale, softcap);
            }
            // blocks that lie wholly inside every row's range need no mask (a wavefront-wide decision)
            const bool inside = kbase + kBlockKeys - 1 <= t_pos_min[rt] && kbase >= t_lo_max[rt];
            if (!inside) {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int key = kbase + 16 * (e / 4) + 4 * g + (e % 4);
                    if (!(row_valid[rt] && key <= pos[rt] && key >= lo[rt])) sv[e] = -INFINITY;
                }
            }
            float tile_max = fmaxf(fmaxf(fmaxf(sv[0], sv[1]), fmaxf(sv[2], sv[3])),
                                   fmaxf(fmaxf(sv[4], sv[5]), fmaxf(sv[6], sv[7])));
            tile_max = max_across(max_across(tile_max, 16), 32);
            const float m_new = fmaxf(m_run[rt], tile_max);
            const float m_use = m_new == -INFINITY ? 0.f : m_new;
            const float mc = m_use * scale_log2e;
            alpha[rt] = exp2_probability(fmaf(m_run[rt], scale_log2e, -mc));
            float pe[8], psum = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                pe[e] = exp2_probability(fmaf(sv[e], scale_log2e, -mc));       // exp2(-inf) = 0 for masked keys
                psum += pe[e];
            }
            pv[rt].u = make_uint4(pack2_bf16(pe[0], pe[1]), pack2_bf16(pe[2], pe[3]), pack2_bf16(pe[4], pe[5]),
                                  pack2_bf16(pe[6], pe[7]));
            if (SPLIT)
                pr[rt].u = make_uint4(pack2_bf16(bf16_remainder(pe[0]), bf16_remainder(pe[1])),
                                      pack2_bf16(bf16_remainder(pe[2]), bf16_remainder(pe[3])),
                                      pack2_bf16(bf16_remainder(pe[4]), bf16_remainder(pe[5])),
                                      pack2_bf16(bf16_remainder(pe[6]), bf16_remainder(pe[7])));
            l_run[rt] = l_run[rt] * alpha[rt] + psum;
            m_run[rt] = m_new;
            rescale[rt] = __any(alpha[rt] != 1.f);
        }
        // ---- out^T += V^T . P^T; the accumulators are rescaled only when some row's maximum moved ----
#pragma unroll
        for (int rt = 0; rt < RTW; ++rt) {
            if (__builtin_amdgcn_readfirstlane(rescale[rt])) {      // one branch for the wavefront, not a select per number
#pragma unroll
                for (int t = 0; t < DT; ++t) acc[rt][t] *= alpha[rt];
            }
        }
#pragma unroll
        for (int t = 0; t < DT; ++t) {
            PPack a;
            a.u = *reinterpret_cast<const uint4*>(&v_s[(16 * t + i) * SV + 8 * g]);
#pragma unroll
            for (int rt = 0; rt < RTW; ++rt)
            {
                acc[rt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, pv[rt].v, acc[rt][t], 0, 0, 0);
                if (SPLIT) acc[rt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, pr[rt].v, acc[rt][t], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int rt = 0; rt < RTW; ++rt) {
        float l = l_run[rt];
        l = sum_across(sum_across(l, 16), 32);
        if (!row_valid[rt]) continue;
        if (partial_slot >= 0) {
            // one slot per tile of 16 rows: [16][HD] accumulators and [16][2] (maximum, sum)
            const size_t slot = static_cast<size_t>(partial_slot) + wave * RTW + rt;
            float* po = partial_o + (slot * 16 + i) * HD;
#pragma unroll
            for (int t = 0; t < DT; ++t)
                *reinterpret_cast<float4*>(po + t * 16 + 4 * g) =
                    make_float4(acc[rt][t][0], acc[rt][t][1], acc[rt][t][2], acc[rt][t][3]);
            if (g == 0) *reinterpret_cast<float2*>(partial_ml + (slot * 16 + i) * 2) = make_float2(m_run[rt], l);
            continue;
        }
        // a sink: exp(sink of the head) once more in the denominator of a row that is finished here
        if (sinks) l += exp2f(sinks[head[rt]] * 1.4426950408889634f - m_run[rt] * scale_log2e);
        const float inv = 1.f / l;
        bf16* orow = out + (static_cast<size_t>(q_start + tok[rt]) * num_heads + head[rt]) * HD;
#pragma unroll
        for (int t = 0; t < DT; ++t) {
            uint2 w;
            w.x = pack2_bf16(acc[rt][t][0] * inv, acc[rt][t][1] * inv);
            w.y = pack2_bf16(acc[rt][t][2] * inv, acc[rt][t][3] * inv);
            *reinterpret_cast<uint2*>(orow + t * 16 + 4 * g) = w;
        }
    }
}

// ---- the items of `attention_portion.h`: tiles moved into shared memory by the memory pipeline ----
template <int HD, bool SPLIT>
__global__ void __launch_bounds__(kPrefillThreads, 2)
paged_attention_prefill_dma_kernel(const bf16* __restrict__ qkv, const bf16* __restrict__ cache,
                                   const int* __restrict__ block_tables, const int* __restrict__ items,
                                   const int* __restrict__ seg_q_start, const int* __restrict__ seg_q_len,
                                   const int* __restrict__ seg_ctx_len, bf16* __restrict__ out,
                                   float* __restrict__ partial_o, float* __restrict__ partial_ml, int num_heads,
                                   int num_kv_heads, int page_size, int max_pages, float scale_log2e, int window,
                                   int q_stride, float cap_scale, float softcap, const float* __restrict__ sinks) {
    __shared__ PortionShared<HD> shared;
    portion_item<HD, SPLIT>(shared, blockIdx.x, qkv, cache, block_tables, items, seg_q_start, seg_q_len, seg_ctx_len, out,
                            partial_o, partial_ml, num_heads, num_kv_heads, page_size, max_pages, scale_log2e, window,
                            q_stride, cap_scale, softcap, sinks);
}

// Returns 0, a HIP error code, or -1 for sizes this kernel does not take.
WLLM_API int wllm_paged_attention_prefill(const void* qkv, const void* cache, const int* block_tables,
                                          const int* items, int num_items, int rows_per_item, const int* seg_q_start,
                                          const int* seg_q_len, const int* seg_ctx_len, void* out, float* partial_o,
                                          float* partial_ml, int num_heads,
                                          int num_kv_heads, int head_dim, int page_size, int max_pages, float scale,
                                          int window, int q_stride, float softcap, int split_weights,
                                          const float* sinks, hipStream_t stream) {
    if (head_dim % 32 != 0 || head_dim < 32 || head_dim > 256 || page_size % 4 != 0 || num_heads % num_kv_heads != 0)
        return -1;
    if (rows_per_item != 64) return -1;
    if (q_stride < num_heads * head_dim || q_stride % 8 != 0 || softcap < 0.f) return -1;
    if (num_items <= 0) return 0;
    const float scale_log2e = (softcap > 0.f ? 1.f : scale) * 1.4426950408889634f;
    const float cap_scale = softcap > 0.f ? scale / softcap : 0.f;
    if (page_size >= 8 && (page_size & (page_size - 1)) == 0 && (head_dim == 64 || head_dim == 128 || head_dim == 256)) {
#define LAUNCH_DMA(HD)                                                                                              \
    if (split_weights) LAUNCH_DMA_S(HD, true); else LAUNCH_DMA_S(HD, false)
#define LAUNCH_DMA_S(HD, S)                                                                                         \
    paged_attention_prefill_dma_kernel<HD, S><<<num_items, kPrefillThreads, 0, stream>>>(                           \
        static_cast<const bf16*>(qkv), static_cast<const bf16*>(cache), block_tables, items, seg_q_start, seg_q_len, \
        seg_ctx_len, static_cast<bf16*>(out), partial_o, partial_ml, num_heads, num_kv_heads, page_size, max_pages, \
        scale_log2e, window, q_stride, cap_scale, softcap, sinks)
        if (head_dim == 64) { LAUNCH_DMA(64); }
        else if (head_dim == 128) { LAUNCH_DMA(128); }
        else { LAUNCH_DMA(256); }
#undef LAUNCH_DMA
#undef LAUNCH_DMA_S
        return launch_status();
    }
#define LAUNCH_RTW(HD, RTW)                                                                                         \
    if (split_weights) LAUNCH_RTW_S(HD, RTW, true); else LAUNCH_RTW_S(HD, RTW, false)
#define LAUNCH_RTW_S(HD, RTW, S)                                                                                    \
    paged_attention_prefill_kernel<HD, RTW, S><<<num_items, kPrefillThreads, 0, stream>>>(                          \
        static_cast<const bf16*>(qkv), static_cast<const bf16*>(cache), block_tables, items, seg_q_start, seg_q_len, \
        seg_ctx_len, static_cast<bf16*>(out), partial_o, partial_ml, num_heads, num_kv_heads, page_size, max_pages, \
        scale_log2e, window, q_stride, cap_scale, softcap, sinks)
#define LAUNCH(HD) LAUNCH_RTW(HD, 1)
    switch (head_dim) {
        case 32: LAUNCH(32); break;
        case 64: LAUNCH(64); break;
        case 96: LAUNCH(96); break;
        case 128: LAUNCH(128); break;
        case 160: LAUNCH(160); break;
        case 192: LAUNCH(192); break;
        case 224: LAUNCH(224); break;
        case 256: LAUNCH(256); break;
        default: return -1;
    }
#undef LAUNCH
#undef LAUNCH_RTW
#undef LAUNCH_RTW_S
    return launch_status();
}
