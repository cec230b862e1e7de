// The query/key/value projection of a decode step, its bias, the rotation of queries and keys and
// the write of keys and values into their pages, in one kernel: for at most 32 tokens, bfloat16,
// heads whose size is a multiple of 32 and that are rotated whole.
//
// out[m, :] = x[m, :] . w^T as in `gemm_skinny.hip` (weights as the A operand of
// v_mfma_f32_16x16x32_bf16, read row by row or from the tile-major copy).  A workgroup owns two
// bands of 16 columns of one head that the rotation pairs: columns 16p .. 16p+15 and the same
// HD/2 further on.  Its eight wavefronts split the K axis, issue all their loads before the first
// product (a register is refilled as soon as its product is issued), and add their sums through
// shared memory in the order of the pieces.  The first wavefront then holds, per lane, four
// columns of both bands for one token: element j of the head and its partner j + HD/2, so the
// pair is turned in registers by position * inv_freq[j] (angle, sine, cosine in float32, made while the
// weights are on their way: behind the sums they cost 1.1 us of 7.2), written
// to the row of queries, keys and values, and keys go to the cache as [page_size, HD], values
// transposed as [HD, page_size].  Heads of values take the same path without the rotation.
// 17 to 32 tokens are two tiles of 16: every fragment of the weights then feeds two products.  (Three
// and four tiles were measured too: with fewer steps in flight to fit the registers they are no faster
// than the product and the rotation as two kernels.)
//
// HALVES: 128 or fewer pairs of bands leave half of the 256 compute units idle, and a workgroup waits for the 64 bytes a clock that a
// compute unit takes in (128 KiB of weights at 2,048 keys, and x).  Then a pair is two workgroups, one for rows 0 .. 7 of both bands
// and one for rows 8 .. 15: eight rows of the lower and eight of the upper band make one fragment of 16, lanes (i, g) and
// (i, g + 2) end up with four elements and their partners and exchange them.  Products, pieces and order of the sums are the
// same, so are the bits.  2,048 keys to 10 heads of 256 (80 pairs) for 1 / 8 / 16 / 32 tokens 6.7 / 7.4 / 8.2 / 11.0 to
// 5.8 / 6.3 / 7.2 / 9.7 us, to 32 heads of 128 (128 pairs) for 1 / 8 / 32 tokens 7.3 / 7.9 / 11.4 to 6.5 / 6.8 / 10.1;
// with more pairs the fragments of x are read twice as often for nothing (4,096 keys, 192 pairs: 13.5 / 13.7 / 19.0 to
// 14.0 / 16.1 / 27.6; 2,560 keys, 256 pairs: 10.0 to 10.7 for one token).  With more keys the runs of 128 bytes in which the
// weights are then read count (80 pairs for 1 / 8 tokens of 8,192 keys 17.6 / 18.9 to 20.1 / 20.8; 128 pairs of 4,096 11.5 / 12.4 to
// 11.5 / 11.8), so beyond 4,096 keys a pair is one workgroup.
#include "common.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));

union QFrag {
    uint4 u;
    bf16x8_t v;
};

constexpr int kQkvWaves = 8;

// What the first wavefront does with one token's sums of a pair of bands: bias, the rotation of the
// pair (element j of the head with j + HD/2), the row of queries, keys and values, and the cache.
// ONE_SIDE: the lane writes the elements, or (`upper`) their partners only.
template <bool ONE_SIDE>
__device__ __forceinline__ void finish_row(float4_t acc_lo, float4_t acc_hi, const float* __restrict__ bias, int col, int half,
                                           bool rotated, const float* sines, const float* cosines, bf16* __restrict__ qkv, int m, int width,
                                           bf16* __restrict__ cache, int head, int num_heads, int num_kv_heads, int slot,
                                           int page_size, long long num_pages, size_t page_elems, int HD, int j0, bool upper) {
    const bool write_lo = !ONE_SIDE || !upper, write_hi = !ONE_SIDE || upper;
    if (bias) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            acc_lo[v] += bias[col + v];
            acc_hi[v] += bias[col + half + v];
        }
    }
    if (rotated) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const float a = acc_lo[v], b = acc_hi[v];
            float ra, rb;
            rotate_pair(a, b, sines[v], cosines[v], ra, rb);
            acc_lo[v] = ra;
            acc_hi[v] = rb;
        }
    }
    uint2 plo, phi;
    plo.x = pack2_bf16(acc_lo[0], acc_lo[1]);
    plo.y = pack2_bf16(acc_lo[2], acc_lo[3]);
    phi.x = pack2_bf16(acc_hi[0], acc_hi[1]);
    phi.y = pack2_bf16(acc_hi[2], acc_hi[3]);
    bf16* row = qkv + static_cast<size_t>(m) * width + col;
    if (write_lo) *reinterpret_cast<uint2*>(row) = plo;
    if (write_hi) *reinterpret_cast<uint2*>(row + half) = phi;
    if (!cache || head < num_heads) return;
    const long long page = slot / page_size;
    const int off = slot % page_size;
    if (slot < 0 || page >= num_pages) return;
    bf16* kpage = cache + page * page_elems;
    if (head < num_heads + num_kv_heads) {
        bf16* dst = kpage + (static_cast<size_t>(head - num_heads) * page_size + off) * HD + j0;
        if (write_lo) *reinterpret_cast<uint2*>(dst) = plo;
        if (write_hi) *reinterpret_cast<uint2*>(dst + half) = phi;
    } else {
        bf16* vpage = kpage + static_cast<size_t>(num_kv_heads) * page_size * HD;
        const int vh = head - num_heads - num_kv_heads;
        const uint16_t el[4] = {static_cast<uint16_t>(plo.x & 0xffff), static_cast<uint16_t>(plo.x >> 16),
                                static_cast<uint16_t>(plo.y & 0xffff), static_cast<uint16_t>(plo.y >> 16)};
        const uint16_t eh[4] = {static_cast<uint16_t>(phi.x & 0xffff), static_cast<uint16_t>(phi.x >> 16),
                                static_cast<uint16_t>(phi.y & 0xffff), static_cast<uint16_t>(phi.y >> 16)};
        uint16_t* vp = reinterpret_cast<uint16_t*>(vpage);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            if (write_lo) vp[(static_cast<size_t>(vh) * HD + j0 + v) * page_size + off] = el[v];
            if (write_hi) vp[(static_cast<size_t>(vh) * HD + j0 + half + v) * page_size + off] = eh[v];
        }
    }
}

template <bool TILED, int MT, bool HALVES>
__global__ void __launch_bounds__(kQkvWaves * 64)
qkv_rope_kernel(const bf16* __restrict__ x, const bf16* __restrict__ w, const float* __restrict__ bias,
                const int* __restrict__ positions, const float* __restrict__ inv_freq, const int* __restrict__ slots,
                bf16* __restrict__ qkv, bf16* __restrict__ cache, int M, int K, int num_heads, int num_kv_heads, int HD,
                int page_size, long long num_pages) {
    constexpr int BANDS = HALVES ? 1 : 2;
    __shared__ float4_t red[(kQkvWaves - 1) * kWave * BANDS * MT];
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int i = lane % 16, g = lane / 16;
    const int pairs = HD / 32;                          // pairs of bands in a head
    const int pair = HALVES ? blockIdx.x / 2 : blockIdx.x, below = HALVES ? 8 * (blockIdx.x % 2) : 0;
    const int head = pair / pairs, p = pair % pairs;
    const int band_lo = head * (HD / 16) + p, band_hi = band_lo + pairs;
    const int steps = K / 32;
    const int per = (steps + kQkvWaves - 1) / kQkvWaves;
    const int s0 = wave * per, s1 = min(steps, s0 + per);
    constexpr int kStep = TILED ? 512 : 32;             // elements from one step of 32 keys to the next
    // HALVES: one fragment of eight rows of the lower band and eight of the upper
    const int row_lo = HALVES ? below + i % 8 : i, from = HALVES && i >= 8 ? band_hi : band_lo;
    const bf16* lo = TILED ? w + static_cast<size_t>(from) * steps * 512 + (g * 16 + row_lo) * 8
                           : w + (static_cast<size_t>(from) * 16 + row_lo) * K + 8 * g;
    const bf16* hi = TILED ? w + static_cast<size_t>(band_hi) * steps * 512 + lane * 8
                           : w + (static_cast<size_t>(band_hi) * 16 + i) * K + 8 * g;
    const bf16* xp[MT];
    bool x_row[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        xp[t] = x + static_cast<size_t>(min(16 * t + i, M - 1)) * K + 8 * g;
        x_row[t] = 16 * t + i < M;
    }
    // what the first wavefront needs after the sums, asked for now so that it has arrived by then
    const int j0 = p * 16 + (HALVES ? below + 4 * (g % 2) : 4 * g), half = HD / 2;
    const bool rotated = head < num_heads + num_kv_heads && inv_freq != nullptr;
    float pos[MT];
    float4 freq = make_float4(0.f, 0.f, 0.f, 0.f);
    int slot[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        pos[t] = 0.f;
        slot[t] = -1;
        if (wave == 0 && x_row[t]) {
            if (rotated) pos[t] = static_cast<float>(positions[16 * t + i]);
            if (cache && head >= num_heads) slot[t] = slots[16 * t + i];
        }
    }
    if (wave == 0 && rotated) freq = *reinterpret_cast<const float4*>(inv_freq + j0);
    constexpr int U = 8;        // steps of 32 keys whose loads a wavefront keeps in flight, per band
    QFrag cl[U], ch[U], cx[U][MT];
    auto load_step = [&](int u, int at) {
        const bool ok = at < s1;
        cl[u].u = ok ? load_streamed(lo + static_cast<size_t>(at) * kStep) : make_uint4(0, 0, 0, 0);
        if (!HALVES) ch[u].u = ok ? load_streamed(hi + static_cast<size_t>(at) * kStep) : make_uint4(0, 0, 0, 0);
#pragma unroll
        for (int t = 0; t < MT; ++t)
            cx[u][t].u = ok && x_row[t] ? *reinterpret_cast<const uint4*>(xp[t] + static_cast<size_t>(at) * 32) : make_uint4(0, 0, 0, 0);
    };
#pragma unroll
    for (int u = 0; u < U; ++u) load_step(u, s0 + u);
    // (the angles' sines while the weights are on their way, not behind the sums)
    float sines[MT][4], cosines[MT][4];
    if (wave == 0 && rotated) {
        const float fr[4] = {freq.x, freq.y, freq.z, freq.w};
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) sincosf(pos[t] * fr[v], &sines[t][v], &cosines[t][v]);
    }
    float4_t acc_lo[MT], acc_hi[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        acc_lo[t] = float4_t{0.f, 0.f, 0.f, 0.f};
        acc_hi[t] = float4_t{0.f, 0.f, 0.f, 0.f};
    }
    for (int s = s0; s < s1; s += U) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                acc_lo[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(cl[u].v, cx[u][t].v, acc_lo[t], 0, 0, 0);
                if (!HALVES) acc_hi[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ch[u].v, cx[u][t].v, acc_hi[t], 0, 0, 0);
            }
            load_step(u, s + U + u);
        }
    }
    if (wave > 0) {
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            float4_t* to = red + (((wave - 1) * kWave + lane) * MT + t) * BANDS;
            to[0] = acc_lo[t];
            if (!HALVES) to[BANDS - 1] = acc_hi[t];
        }
    }
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int q = 0; q < kQkvWaves - 1; ++q)
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            const float4_t* part = red + ((q * kWave + lane) * MT + t) * BANDS;
            acc_lo[t] += part[0];
            if (!HALVES) acc_hi[t] += part[BANDS - 1];
        }
    if (HALVES) {
        // lanes of g and g + 2 hold four elements and their partners: each side gets the other
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const float own = acc_lo[t][v], other = __shfl_xor(own, 32);
                acc_lo[t][v] = g < 2 ? own : other;
                acc_hi[t][v] = g < 2 ? other : own;
            }
    }
    const int width = (num_heads + 2 * num_kv_heads) * HD;
    const int col = head * HD + j0;
    const size_t page_elems = static_cast<size_t>(2) * num_kv_heads * page_size * HD;
    // lane (i, g): token m = 16 t + i, elements j .. j + 3 of the head and their partners
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        const int m = 16 * t + i;
        if (m >= M) continue;
        finish_row<HALVES>(acc_lo[t], acc_hi[t], bias, col, half, rotated, sines[t], cosines[t], qkv, m, width, cache, head, num_heads,
                   num_kv_heads, slot[t], page_size, num_pages, page_elems, HD, j0, g >= 2);
    }
}
// Returns 0, a HIP error code, or -1 for sizes this kernel does not take (the caller then runs the
// product and the rotation as two kernels).  `w` is the stacked [q; k; v] weight, row by row or
// (`tiled`) its tile-major copy.  inv_freq has HD/2 entries or is null (no rotation).
WLLM_API int wllm_qkv_rope(const void* x, const void* w, int tiled, const float* bias, const int* positions,
                           const float* inv_freq, const int* slots, void* qkv, void* cache, long long num_pages, int M,
                           int K, int num_heads, int num_kv_heads, int head_dim, int page_size, hipStream_t stream) {
    if (M < 1 || M > 32 || K < 32 || K % 32 != 0 || head_dim < 32 || head_dim % 32 != 0 || num_heads < 1 || num_kv_heads < 1 ||
        page_size < 1)
        return -1;
    const int grid = (num_heads + 2 * num_kv_heads) * (head_dim / 32);
    const bool halves = grid <= 128 && K <= 4096;       // twice as many workgroups have a compute unit each
#define LAUNCH(T, MT)                                                                                                  \
    do {                                                                                                               \
        if (halves) LAUNCH_BANDS(T, MT, true); else LAUNCH_BANDS(T, MT, false);                              \
    } while (0)
#define LAUNCH_BANDS(T, MT, HALVES)                                                                                    \
    qkv_rope_kernel<T, MT, HALVES><<<HALVES ? 2 * grid : grid, kQkvWaves * 64, 0, stream>>>(                           \
        static_cast<const bf16*>(x), static_cast<const bf16*>(w), bias, positions, inv_freq, slots, static_cast<bf16*>(qkv), \
        static_cast<bf16*>(cache), M, K, num_heads, num_kv_heads, head_dim, page_size, num_pages)
    if (tiled) {
        if (M <= 16) LAUNCH(true, 1);
        else LAUNCH(true, 2);
    } else {
        if (M <= 16) LAUNCH(false, 1);
        else LAUNCH(false, 2);
    }
#undef LAUNCH_BANDS
#undef LAUNCH
    return launch_status();
}
