// The two products of a mixture of experts where an expert has some tens of rows and more, bfloat16: tiles of 256 rows
// of one expert by 256 rows of its weights, as `wide_tile.h` makes them.  What differs from the product of one
// matrix: a plan (`moe_plan_kernel`) names the assignments in tiles of 128 rows of one expert, of which two that follow each
// other are the two halves of a tile here, and an expert's odd last one is a tile with one half; a tile's rows of x are gathered
// (the token's row of x for the first product, the assignment's row of act for the second), the weights are the
// tile's expert's, and a row's result goes where its assignment belongs.  A row's sums run over k in ascending stages
// whatever tile it lies in.
//
// What bounds it beside its products are the rows that fill no tile.  16 experts of 4,096 behind a width of
// 2,048, three a token, us, against tiles of 128 x 128 with two workgroups a compute unit (first product; second): 256 tokens 148, 140; 78,
// 68; 1,000 227, 156; 115, 97; 2,048 393, 244; 198, 109; 3,001 531, 351; 265, 194; 7,777 1,108, 722; 538, 420; 64 experts of
// 1,024, six a token, 1,500 tokens 222, 139; 172, 90.  16 of 1,408, four a token: 1,000 tokens 88, 55; 74, 41.  The activation in full, as the other
// kernels of the experts make it, costs 3 to 12% of the first product (by the hardware's exponential and reciprocal 137, 151, 238, 333 and 645 us).
#include "wide_tile.h"

constexpr int kBandPairs = 4;          // tiles of rows that share a tile of columns one after the other
constexpr int kMostTiles = 16000;      // tiles of the plan that a launch takes: its list of pairs lies behind the stages in shared memory

struct ExpertItem {
    int tile, n_base;                  // first of the plan's tiles, first column
    bool two;
};

// GATED: 0 the second product (out32[a % top][a / top][n] = weight[a] * sum), 1 + the activation's number the
// first (act[a][n] = activation(gate) * up; w holds an expert's N gate rows, then its N up rows).
// `weights`: of the second product the factor of a row's result, 1 if null; of the first the factor of a row's
// input, taken out of both sums, none if null.  The plan's tiles from `tile_begin` on, at most kMostTiles.  `vectors`: the result begins
// at a multiple of 16 bytes.  ODD: x or w begins at none.
template <int GATED, bool ODD>
__global__ void __launch_bounds__(512, 2)
moe_wide_kernel(const bf16* __restrict__ x, const bf16* __restrict__ w, const int* __restrict__ plan, int max_tiles,
                bf16* __restrict__ act, float* __restrict__ out32, const float* __restrict__ weights, int N, int K, int top,
                int tokens, int n_tiles, int tile_begin, bool vectors) {
    constexpr int kColumns = GATED ? kWideHalf : kWideRows;
    extern __shared__ __align__(16) unsigned char tiles_s[];
    uint16_t* pairs_s = reinterpret_cast<uint16_t*>(tiles_s + kWideShared);         // the plan's tile, and whether it is two in the top bit
    int* count_s = reinterpret_cast<int*>(tiles_s + kWideShared + kMostTiles * 2);
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int i = lane % 16, g = lane / 16;
    const int wm = wave / 4, wn = wave % 4;
    const int live = min(plan[0] - tile_begin, kMostTiles);
    if (live <= 0) return;
    const int* expert_of = plan + 1 + tile_begin;
    const int* rows = plan + 1 + max_tiles + static_cast<size_t>(tile_begin) * kWideHalf;

    // ---- the tiles of rows: every even one of an expert's tiles in the plan, with the odd one behind it ----
    if (wave == 0) {
        int begin = 0, count = 0;              // the first tile of the expert at hand, tiles listed
        for (int base = 0; base < live; base += kWave) {
            const int t = base + lane;
            const bool there = t < live;
            const int e = there ? expert_of[t] : -1;
            const bool starts = there && (t == 0 || expert_of[t - 1] != e);
            const unsigned long long start_mask = __ballot(starts), upto = start_mask & (~0ull >> (63 - lane));
            const int mine = upto ? base + 63 - __builtin_clzll(upto) : begin;
            const bool leads = there && (t - mine) % 2 == 0;
            const unsigned long long lead_mask = __ballot(leads);
            if (leads) {
                const bool two = t + 1 < live && expert_of[t + 1] == e;
                pairs_s[count + __popcll(lead_mask & ((1ull << lane) - 1))] = static_cast<uint16_t>(t | (two ? 0x8000 : 0));
            }
            if (start_mask) begin = base + 63 - __builtin_clzll(start_mask);
            count += __popcll(lead_mask);
        }
        if (lane == 0) *count_s = count;
    }
    __syncthreads();
    const int m_tiles = *count_s;
    const int items = m_tiles * n_tiles;
    const int xcd = blockIdx.x % 8, per_xcd = items / 8, left = items % 8;
    const int first = xcd * per_xcd + min(xcd, left), end = first + per_xcd + (xcd < left ? 1 : 0);
    if (first + static_cast<int>(blockIdx.x) / 8 >= end) return;

    auto place = [&](int it, WideSource& from) {
        const int band = it / (kBandPairs * n_tiles), in_band = it - band * kBandPairs * n_tiles;
        const int band_rows = min(kBandPairs, m_tiles - kBandPairs * band);
        const int n_tile = in_band / band_rows;
        // (each round of the band's items another of its tiles of rows, so that no workgroup makes tiles of one half alone, or of two: 16 experts of
        // 4,096 behind a width of 2,048, three a token, 3,001 tokens 332 us and 314.  Tiles of one half behind all others: 357, their weights read again.)
        const int of_band = (in_band - n_tile * band_rows + n_tile * band_rows / (static_cast<int>(gridDim.x) / 8)) % band_rows;
        const int pair = __builtin_amdgcn_readfirstlane(pairs_s[kBandPairs * band + of_band]);
        const ExpertItem at{pair & 0x7fff, n_tile * kColumns, (pair & 0x8000) != 0};
        from.stages = K / kWideKeys;
        from.two = at.two;
        from.x_bytes = reinterpret_cast<const unsigned char*>(x);
        from.w_bytes = reinterpret_cast<const unsigned char*>(w + static_cast<size_t>(expert_of[at.tile]) * (GATED ? 2 : 1) * N * K);
#pragma unroll
        for (int h = 0; h < 4; ++h)
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int r = wide_row(u);
                size_t row;
                if (h < 2) {
                    const int a = h == 0 || at.two ? rows[at.tile * kWideHalf + kWideHalf * h + r] : -1;
                    row = a < 0 ? 0 : GATED ? a / top : a;
                } else if (GATED) {
                    row = static_cast<size_t>(min(at.n_base + r, N - 1)) + (h == 3 ? N : 0);
                } else {
                    row = min(at.n_base + kWideHalf * (h - 2) + r, N - 1);
                }
                from.offset[h][u] = static_cast<uint32_t>((row * K + wide_chunk() * 8) * 2);
            }
        return at;
    };
    auto finish = [&](const ExpertItem& at, const WideSums& acc) {
#pragma unroll
        for (int xh = 0; xh < 2; ++xh) {
            if (xh == 1 && !at.two) break;
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const int asg = rows[at.tile * kWideHalf + xh * kWideHalf + wm * 64 + 16 * b + i];
                if (GATED) {
                    const float scale = weights && asg >= 0 ? weights[asg] : 1.f;
                    uint32_t q[2][2];
#pragma unroll
                    for (int a = 0; a < 2; ++a) {
                        float r[4];
#pragma unroll
                        for (int v = 0; v < 4; ++v)
                            r[v] = activate<(GATED > 0 ? GATED - 1 : 0)>(acc[xh][0][a][b][v] * scale) * (acc[xh][1][a][b][v] * scale);
                        q[a][0] = pack2_bf16(r[0], r[1]);
                        q[a][1] = pack2_bf16(r[2], r[3]);
                    }
                    const uint4 columns = wide_eight_columns(q);
                    if (asg < 0) continue;
                    const int n = at.n_base + wn * 32 + 16 * (g & 1) + 8 * (g >> 1);
                    bf16* to = act + static_cast<size_t>(asg) * N + n;
                    const uint32_t words[4] = {columns.x, columns.y, columns.z, columns.w};
                    if (vectors && n + 7 < N && N % 8 == 0) {
                        *reinterpret_cast<uint4*>(to) = columns;
                    } else {
#pragma unroll
                        for (int v = 0; v < 8; ++v)
                            if (n + v < N) to[v] = bf16{static_cast<uint16_t>(words[v / 2] >> (16 * (v % 2)))};
                    }
                } else {
                    if (asg < 0) continue;
                    const float weight = weights ? weights[asg] : 1.f;
                    float* o_row = out32 + (static_cast<size_t>(asg % top) * tokens + asg / top) * N;
#pragma unroll
                    for (int wh = 0; wh < 2; ++wh)
#pragma unroll
                        for (int a = 0; a < 2; ++a) {
                            const int n = at.n_base + wh * kWideHalf + wn * 32 + 16 * a + 4 * g;
                            const float4_t r = acc[xh][wh][a][b] * weight;
                            if (vectors && n + 3 < N && N % 4 == 0) {
                                *reinterpret_cast<float4_t*>(o_row + n) = r;
                            } else {
#pragma unroll
                                for (int v = 0; v < 4; ++v)
                                    if (n + v < N) o_row[n + v] = r[v];
                            }
                        }
                }
            }
        }
    };
    wide_products<true, ODD>(tiles_s, first + blockIdx.x / 8, end, gridDim.x / 8, place, finish);
}

// The first product (activation >= 0: `act` [assignments, N] from x [tokens, K] and w [experts, 2N, K]) or the second
// (activation < 0: out32 [top, tokens, N] from x = act [assignments, K] and w [experts, N, K]) over a plan of tiles of
// 128 rows.  Returns -1 for what it does not take (K no multiple of 64, x or an expert's w of 4 GiB).
WLLM_API int wllm_moe_wide(const void* x, const void* w, const int* plan, int max_tiles, void* act, float* out32,
                           const float* weights, int activation, int x_rows, int N, int K, int top, int tokens,
                           hipStream_t stream) {
    if (max_tiles <= 0 || x_rows <= 0) return 0;
    if (N <= 0 || K < kWideKeys || K % kWideKeys || top <= 0 || tokens <= 0 || activation >= kActivations) return -1;
    const bool gated = activation >= 0;
    if ((gated && !act) || (!gated && !out32)) return -1;
    if (static_cast<size_t>(gated ? 2 : 1) * N * K * 2 >= (size_t(1) << 32) || static_cast<size_t>(x_rows) * K * 2 >= (size_t(1) << 32))
        return -1;
    const bool odd = (reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) % 16 != 0;
    const bool vectors = reinterpret_cast<uintptr_t>(gated ? act : static_cast<void*>(out32)) % 16 == 0;
    const int columns = gated ? kWideHalf : kWideRows;
    const int n_tiles = (N + columns - 1) / columns;
    static int compute_units = 0;
    if (compute_units == 0) {
        int device = 0;
        if (hipGetDevice(&device) != hipSuccess ||
            hipDeviceGetAttribute(&compute_units, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess)
            return launch_status();
    }
    const int most = compute_units / 8 * 8 > 0 ? compute_units / 8 * 8 : 8;
    const long long items = static_cast<long long>(max_tiles) * n_tiles;
    if (items > 0x3fffffffLL) return -1;
    const int grid = items < most ? static_cast<int>((items + 7) / 8 * 8) : most;
    constexpr int kShared = kWideShared + kMostTiles * 2 + 16;
    const bf16* xp = static_cast<const bf16*>(x);
    const bf16* wp = static_cast<const bf16*>(w);
#define LAUNCH(GATED, ODD)                                                                                          \
    do {                                                                                                            \
        static bool roomy = false;     /* more than 64 KiB of shared memory must be asked for once */              \
        if (!roomy) {                                                                                               \
            if (hipFuncSetAttribute(reinterpret_cast<const void*>(&moe_wide_kernel<GATED, ODD>),                    \
                                    hipFuncAttributeMaxDynamicSharedMemorySize, kShared) != hipSuccess)             \
                return launch_status();                                                                             \
            roomy = true;                                                                                           \
        }                                                                                                           \
        for (int begin = 0; begin < max_tiles; begin += kMostTiles)                                                 \
            moe_wide_kernel<GATED, ODD><<<grid, 512, kShared, stream>>>(xp, wp, plan, max_tiles, static_cast<bf16*>(act), \
                                                                        out32, weights, N, K, top, tokens, n_tiles, \
                                                                        begin, vectors);                            \
    } while (0)
    if (!gated && odd) { LAUNCH(0, true); }
    else if (!gated) { LAUNCH(0, false); }
    else if (odd) { WLLM_BY_ACTIVATION(activation, LAUNCH(ACT + 1, true)) }
    else { WLLM_BY_ACTIVATION(activation, LAUNCH(ACT + 1, false)) }
#undef LAUNCH
    return launch_status();
}
