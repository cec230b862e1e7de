// Paged attention for long segments (prompt portions), the work items of `attention_prefill.hip`, with the
// tiles moved into shared memory by the memory pipeline itself.
// For head sizes 64, 128 and 256 and pages of 8, 16, 32, ... keys (a power of two, so that a key's
// place is a shift and a mask and most of a load's address is fixed for a lane: with divisions and a
// table look-up per load the address arithmetic was a third of the kernel's time; other page sizes
// take the kernel of `attention_prefill.hip`).  A lane's 16-byte load goes
// straight to shared memory (lane l of a wavefront to base + 16 l), so staging costs no registers,
// no writes to shared memory and no second barrier; two tiles of keys and values are held, and
// the loads of block b+1 run while block b is multiplied.  Since a lane chooses its address, the
// 16-byte chunks of a tile are placed so that fragment reads are free of bank conflicts: the 16
// lanes that read together (one chunk each of 16 rows) have to hit 16 different chunks of the 256
// bytes that the banks span.  Chunk c of key row r lies at position c ^ (r % 16) of the row (heads
// of 64, whose rows are 8 chunks and lie two to the 256 bytes: c ^ ((r / 2) % 8)), chunk q (8 keys)
// of value row d at q ^ ((d / 2) % 4).  Measured with a loop of such reads alone, eight wavefronts a
// compute unit: 4.0 clocks a read (256 bytes a clock), and 6.4 with c ^ (r % 8), where rows r and
// r + 8 meet in the same banks.  The keys of a block are staged in the order the second product wants them: row
// 16 t + 4 g + v of the tile holds key 8 g + 4 t + v, so that after the first product a lane's eight
// scores are the keys 8 g .. 8 g + 7 of its row, the same eight keys that chunk g of a value row holds.
// Nothing is cleared in flight: in the blocks at the edges of a request the stale keys' values are
// cleared in shared memory after they have landed (their scores are masked in any case).
// Two kernels run these items: alone, and beside the items of `attention_mfma.hip` in one launch.
#pragma once
#include "lds_load.h"

constexpr int kPrefillWaves = 4;       // wavefronts per workgroup
constexpr int kPrefillThreads = kPrefillWaves * 64;
constexpr int kBlockKeys = 32;
constexpr int kMaxTablePages = 1024;     // pages one work item's keys may span (the host cuts items to fit)
constexpr int kPrefillItemInts = 8;

union PPack {
    uint4 u;
    bf16x8_t v;
    uint2 half[2];
    uint16_t s[8];
};

template <int HD>
struct PortionShared {
    alignas(16) uint16_t k[2][kBlockKeys * HD];
    alignas(16) uint16_t v[2][HD * kBlockKeys];
    int table[kMaxTablePages];
};

// One work item, by the whole workgroup of kPrefillThreads threads.
template <int HD, bool SPLIT>
__device__ __forceinline__ void portion_item(PortionShared<HD>& shared, int index, const bf16* __restrict__ qkv,
                                             const bf16* __restrict__ cache, const int* __restrict__ block_tables,
                                             const int* __restrict__ items, const int* __restrict__ seg_q_start,
                                             const int* __restrict__ seg_q_len, const int* __restrict__ seg_ctx_len,
                                             bf16* __restrict__ out, float* __restrict__ partial_o,
                                             float* __restrict__ partial_ml, int num_heads, int num_kv_heads,
                                             int page_size, int max_pages, float scale_log2e, int window, int q_stride,
                                             float cap_scale, float softcap, const float* __restrict__ sinks) {
    constexpr int DC = HD / 32, DT = HD / 16, CPR = HD / 8;       // CPR: 16-byte chunks of a key row
    constexpr int kKeyInstr = kBlockKeys * CPR / 64, kValInstr = HD * 4 / 64;    // wavefront loads per tile
    uint16_t *const k_s0 = shared.k[0], *const k_s1 = shared.k[1], *const v_s0 = shared.v[0], *const v_s1 = shared.v[1];
    int* const table_s = shared.table;

    const int* item = items + static_cast<size_t>(index) * kPrefillItemInts;
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

    constexpr int kPrefillRows = kPrefillWaves * 16;
    const int wr0 = row_begin + wave * 16;
    const int row = wr0 + i;
    const bool row_valid = row < total_rows;
    const int tok = row_valid ? row / group : 0;
    const int head = kvh * group + (row_valid ? row % group : 0);
    const int pos = first_pos + tok;
    const int lo = lowest_key(pos, window);
    bf16x8_t qreg[DC];
    {
        const bf16* qrow = qkv + static_cast<size_t>(q_start + tok) * width + static_cast<size_t>(head) * HD;
#pragma unroll
        for (int c = 0; c < DC; ++c) {
            PPack p;
            p.u = row_valid ? *reinterpret_cast<const uint4*>(qrow + c * 32 + 8 * g) : make_uint4(0, 0, 0, 0);
            qreg[c] = p.v;
        }
    }
    // the lowest position and the highest window start of the wavefront's rows
    int t_pos_min, t_lo_max;
    {
        const int last = min(total_rows - 1, wr0 + 15);
        t_pos_min = wr0 < total_rows ? first_pos + wr0 / group : -1;
        const int pmax = first_pos + max(last, 0) / group;
        t_lo_max = lowest_key(pmax, window);
        if (last < wr0 + 15) t_pos_min = -1;      // a tile with rows beyond the segment always masks
    }
    const bool wave_active = wr0 < total_rows;
    const int w_last_row = min(total_rows - 1, wr0 + 15);
    const int w_hi = wave_active ? first_pos + w_last_row / group + 1 : 0;                       // exclusive
    const int w_lo = lowest_key(first_pos + wr0 / group, window);
    const int b_last_row = min(total_rows - 1, row_begin + kPrefillRows - 1);
    const int b_hi = first_pos + b_last_row / group + 1;
    const int b_lo = lowest_key(first_pos + row_begin / group, window);
    const int blk_first = max(b_lo, key_begin) / kBlockKeys;
    const int blk_end = (min(b_hi, key_end) + kBlockKeys - 1) / kBlockKeys;
    const int page_base = blk_first * kBlockKeys / page_size;
    if (blk_first < blk_end) {
        const int* table_g = block_tables + static_cast<size_t>(seg) * max_pages + page_base;
        const int page_last = (min(blk_end * kBlockKeys, ctx) - 1) / page_size;
        const int count = min(min(max_pages - 1, page_last) - page_base + 1, kMaxTablePages);
        for (int p = tid; p < count; p += kPrefillThreads) table_s[p] = table_g[p];
    }

    float4_t acc[DT];
    float m_run = -INFINITY, l_run = 0.f;
#pragma unroll
    for (int t = 0; t < DT; ++t) acc[t] = float4_t{0.f, 0.f, 0.f, 0.f};

    // ---- the loads of a block.  The page size is a power of two here and a block begins at a multiple
    //      of 32 keys, so the place of a lane's key kbase + rel splits into a part all lanes share and the
    //      lane's own, which is worked out once: page (kbase >> shift) + (rel >> shift) of the request,
    //      slot (kbase & mask) + (rel & mask).  Per block and load that leaves one look-up in the table
    //      and one multiply-add for the address.  A page index beyond the request's last page (the keys
    //      after the end of the last block) is clamped: whatever lies there is masked and cleared. ----
    const int shift = __builtin_ctz(page_size), mask = page_size - 1;
    static_assert(kKeyInstr % kPrefillWaves == 0 && kValInstr % kPrefillWaves == 0, "whole loads per wavefront");
    constexpr int KU = kKeyInstr / kPrefillWaves, VU = kValInstr / kPrefillWaves;
    const uint32_t page_bytes = static_cast<uint32_t>(page_elems * 2);
    // keys: wavefront load q = wave + 4 u of the tile carries the chunks 64 q .. 64 q + 63 of the tile in
    // shared-memory order
    auto k_swizzle = [](int r) { return CPR >= 16 ? r % 16 : (r / 2) % 8; };      // what row r exchanges its chunks by
    int k_page[KU];
    const char* k_src[KU];
#pragma unroll
    for (int u = 0; u < KU; ++u) {
        const int chunk_index = (wave + u * kPrefillWaves) * 64 + lane;       // position in the tile, in chunks
        const int r = chunk_index / CPR;                                      // row of the tile
        const int chunk = (chunk_index % CPR) ^ k_swizzle(r);                 // the chunk of the key's row that lies there
        const int rel = 8 * ((r % 16) / 4) + 4 * (r / 16) + r % 4;            // the key of the block that row r holds
        k_page[u] = rel >> shift;
        k_src[u] = reinterpret_cast<const char*>(cache + k_off + static_cast<size_t>(rel & mask) * HD + chunk * 8);
    }
    // values: a lane moves the same chunk of 8 keys in every load, of the rows d = 16 q + lane / 4
    const int v_rel = 8 * ((lane % 4) ^ ((lane / 8) % 4));
    const int v_page = v_rel >> shift;
    const char* v_src[VU];
#pragma unroll
    for (int u = 0; u < VU; ++u) {
        const int d = (wave + u * kPrefillWaves) * 16 + lane / 4;
        v_src[u] = reinterpret_cast<const char*>(cache + v_off + static_cast<size_t>(d) * page_size + (v_rel & mask));
    }
    const int table_last = blk_first < blk_end
                               ? min(min(max_pages - 1, (min(blk_end * kBlockKeys, ctx) - 1) / page_size) - page_base + 1,
                                     kMaxTablePages) - 1
                               : 0;
    // where this wavefront's loads land: tile + 1 KiB * (wave + 4 u)
    const uint32_t k_lds[2] = {shared_address(k_s0) + wave * 1024u, shared_address(k_s1) + wave * 1024u};
    const uint32_t v_lds[2] = {shared_address(v_s0) + wave * 1024u, shared_address(v_s1) + wave * 1024u};
    auto issue = [&](int which, int kbase) {
        const int pb = (kbase >> shift) - page_base;
        const uint32_t k_slot_bytes = static_cast<uint32_t>(kbase & mask) * HD * 2, v_slot_bytes = static_cast<uint32_t>(kbase & mask) * 2;
        int kp[KU];
#pragma unroll
        for (int u = 0; u < KU; ++u) kp[u] = table_s[min(pb + k_page[u], table_last)];
        const int vp = table_s[min(pb + v_page, table_last)];
#pragma unroll
        for (int u = 0; u < KU; ++u)
            load_lane_to_shared(k_src[u] + (static_cast<uint64_t>(static_cast<uint32_t>(kp[u])) * page_bytes + k_slot_bytes),
                              k_lds[which] + u * (kPrefillWaves * 1024u));
        const uint64_t v_page_bytes = static_cast<uint64_t>(static_cast<uint32_t>(vp)) * page_bytes + v_slot_bytes;
#pragma unroll
        for (int u = 0; u < VU; ++u) load_lane_to_shared(v_src[u] + v_page_bytes, v_lds[which] + u * (kPrefillWaves * 1024u));
    };

    __syncthreads();      // the block table is in shared memory
    if (blk_first < blk_end) issue(0, blk_first * kBlockKeys);
    // One block: its tiles are k_s and v_s, the next block's loads go to k_next and v_next.  The loop below
    // names the two pairs of tiles in turn, so every address in shared memory is a constant plus a lane's
    // fixed offset.
    // a lane's fragment reads: every address is the tile, the lane's offset and a constant.  With x what row i
    // exchanges by, chunk (4 c + g) ^ x of a key row is 4 (c ^ (x >> 2)) + (g ^ (x & 3)), and x >> 2 touches the
    // two low bits of c only: one offset for each c % 4.
    const int k_x = k_swizzle(i);
    int k_lane[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) k_lane[c] = (i * CPR + 4 * ((c ^ (k_x >> 2)) % DC) + (g ^ (k_x & 3))) * 8;
    const int v_lane = (i * 4 + (g ^ ((i / 2) % 4))) * 8;
    auto block = [&](int blk, const uint16_t* k_s, uint16_t* v_s, int next) {
        const int kbase = blk * kBlockKeys;
        __builtin_amdgcn_s_waitcnt(0);   // this lane's loads of the block have landed
        __syncthreads();                 // everyone's have, and everyone is done with the block before
        if (kbase + kBlockKeys > ctx || kbase < seg_lo) {
            // a block at the edge of the request: the values of keys that are not the request's are cleared
            if (tid < HD) {
                for (int kib = 0; kib < kBlockKeys; ++kib) {
                    const int key = kbase + kib;
                    if (key >= ctx || key < seg_lo) v_s[(tid * 4 + ((kib / 8) ^ ((tid / 2) % 4))) * 8 + kib % 8] = 0;
                }
            }
            __syncthreads();
        }
        // The order below is kept as written (nothing moves across a sched_barrier): all fragments of the keys
        // are asked for before the next block's loads are, the values' fragments before the softmax, so that
        // a product waits for no read that was asked for just before it.  Left to itself the compiler keeps two
        // reads in flight and every product waits a trip to shared memory.
        const bool active = wave_active && kbase < w_hi && kbase + kBlockKeys > w_lo;
        PPack kf[2 * DC], vf[DT];
        if (active) {
#pragma unroll
            for (int t2 = 0; t2 < 2; ++t2)
#pragma unroll
                for (int c = 0; c < DC; ++c)
                    kf[t2 * DC + c].u = *reinterpret_cast<const uint4*>(&k_s[k_lane[c % 4] + (16 * t2 * CPR + 4 * (c & ~3)) * 8]);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (blk + 1 < blk_end) issue(next, kbase + kBlockKeys);
        if (!active) return;
        __builtin_amdgcn_sched_barrier(0);
        // ---- scores: tile t2, lane (i, g) gets the keys 8 g + 4 t2 + v of the block ----
        float sv[8];
#pragma unroll
        for (int t2 = 0; t2 < 2; ++t2) {
            float4_t sc = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < DC; ++c) sc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[t2 * DC + c].v, qreg[c], sc, 0, 0, 0);
#pragma unroll
            for (int v = 0; v < 4; ++v) sv[4 * t2 + v] = sc[v];
        }
        if (softcap > 0.f) {            // the score is scaled and bent here; `scale_log2e` is then log2(e) alone
#pragma unroll
            for (int e = 0; e < 8; ++e) sv[e] = capped_score_fast(sv[e] * cap_scale, softcap);
        }
#pragma unroll
        for (int t = 0; t < DT; ++t) vf[t].u = *reinterpret_cast<const uint4*>(&v_s[v_lane + 16 * t * 4 * 8]);
        __builtin_amdgcn_sched_barrier(0);
        // ---- softmax bookkeeping ----
        const bool inside = kbase + kBlockKeys - 1 <= t_pos_min && kbase >= t_lo_max;
        if (!inside) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int key = kbase + 8 * g + e;
                if (!(row_valid && key <= pos && key >= lo)) sv[e] = -INFINITY;
            }
        }
        float tile_max = fmaxf(fmaxf(fmaxf(sv[0], sv[1]), fmaxf(sv[2], sv[3])), fmaxf(fmaxf(sv[4], sv[5]), fmaxf(sv[6], sv[7])));
        tile_max = max_across(max_across(tile_max, 16), 32);
        const float m_new = fmaxf(m_run, tile_max);
        const float m_use = m_new == -INFINITY ? 0.f : m_new;
        const float mc = m_use * scale_log2e;
        const float alpha = exp2_probability(fmaf(m_run, scale_log2e, -mc));
        float pe[8], psum = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            pe[e] = exp2_probability(fmaf(sv[e], scale_log2e, -mc));       // exp2(-inf) = 0 for masked keys
            psum += pe[e];
        }
        PPack pv;
        pv.u = make_uint4(pack2_bf16(pe[0], pe[1]), pack2_bf16(pe[2], pe[3]), pack2_bf16(pe[4], pe[5]), pack2_bf16(pe[6], pe[7]));
        PPack pr;       // SPLIT: what the rounding left out
        if (SPLIT)
            pr.u = make_uint4(pack2_bf16(bf16_remainder(pe[0]), bf16_remainder(pe[1])),
                              pack2_bf16(bf16_remainder(pe[2]), bf16_remainder(pe[3])),
                              pack2_bf16(bf16_remainder(pe[4]), bf16_remainder(pe[5])),
                              pack2_bf16(bf16_remainder(pe[6]), bf16_remainder(pe[7])));
        l_run = l_run * alpha + psum;
        m_run = m_new;
        // ---- out^T += V^T . P^T; the accumulators are rescaled only when some row's maximum moved: one
        // branch for the whole wavefront around all of them (a test per accumulator becomes a multiply and a
        // select for each of its 64 numbers, whether or not anything moved) ----
        if (__builtin_amdgcn_readfirstlane(__any(alpha != 1.f))) {
#pragma unroll
            for (int t = 0; t < DT; ++t) acc[t] *= alpha;
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < DT; ++t) {
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[t].v, pv.v, acc[t], 0, 0, 0);
            if (SPLIT) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[t].v, pr.v, acc[t], 0, 0, 0);
        }
    };
    for (int blk = blk_first; blk < blk_end; blk += 2) {
        block(blk, k_s0, v_s0, 1);
        if (blk + 1 < blk_end) block(blk + 1, k_s1, v_s1, 0);
    }
    float l = l_run;
    l = sum_across(sum_across(l, 16), 32);
    if (!row_valid) return;
    if (partial_slot >= 0) {
        const size_t slot = static_cast<size_t>(partial_slot) + wave;
        float* po = partial_o + (slot * 16 + i) * HD;
#pragma unroll
        for (int t = 0; t < DT; ++t)
            *reinterpret_cast<float4*>(po + t * 16 + 4 * g) = make_float4(acc[t][0], acc[t][1], acc[t][2], acc[t][3]);
        if (g == 0) *reinterpret_cast<float2*>(partial_ml + (slot * 16 + i) * 2) = make_float2(m_run, l);
        return;
    }
    if (sinks) l += exp2f(sinks[head] * 1.4426950408889634f - m_run * scale_log2e);
    const float inv = 1.f / l;
    bf16* orow = out + (static_cast<size_t>(q_start + tok) * num_heads + head) * HD;
#pragma unroll
    for (int t = 0; t < DT; ++t) {
        uint2 w;
        w.x = pack2_bf16(acc[t][0] * inv, acc[t][1] * inv);
        w.y = pack2_bf16(acc[t][2] * inv, acc[t][3] * inv);
        *reinterpret_cast<uint2*>(orow + t * 16 + 4 * g) = w;
    }
}
