// A layer's token input for at most 16 rows, bfloat16, in one launch: out[r, :] = W_proj (act(W_gate x[r]) * table[ids[r], col0 : col0 + dim]) with dim
// 32 or 64: what the few-row product, `gated_lookup` and the few-row product make in three, with their roundings (the gate's product, and its product with the
// entry, to bfloat16) and their order of sums for a K axis in two pieces.
//
// A workgroup owns 128 columns of the result, a wavefront 16 of them.  Every workgroup makes the whole small product W_gate x for itself: its wavefronts take
// steps of 64 keys in turn (the first four the first half of the K axis, the others the second) and meet in shared memory, where each
// thread adds up its elements, bends them and multiplies them by their entries; then each wavefront multiplies by its band of W_proj.  The weights of both products and
// the entries are asked for at the beginning.
//
// What bounds it: the launch, and 256 KiB of W_gate into each compute unit that runs a workgroup (64 bytes a clock: 1.7 us of 2,048 keys); so the workgroups
// are few.  A launch costs 1.5 us by itself, and each of the three had a chain of its own: 64 columns of 2,048 keys and 2,048 of 64 at 1 / 8 / 16 rows 8.4 / 8.7 / 8.9 us
// in three and 5.9 / 6.7 / 7.4 in one, Tokuvik's decode step of 8 requests 1,960 and 1,889 us.  With two tiles of 16 rows a workgroup 17 / 32 rows took 9.0 / 10.4 us, the
// three 9.6 / 9.9.
#include "common.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));

union SideFragment {
    uint4 u;
    bf16x8_t v;
};

constexpr int kSideWaves = 8, kSideRows = 16, kSideSteps = 4;        // steps of 64 keys of a wavefront at most

// NB: bands of 16 of the small product's columns (dim = 16 NB).  TILED: both weights are their tile-major copies.
template <int NB, int ACT, bool TILED>
__global__ void __launch_bounds__(64 * kSideWaves)
token_side_kernel(const bf16* __restrict__ x, const bf16* __restrict__ w_gate, const int* __restrict__ ids, const bf16* __restrict__ table,
                  const bf16* __restrict__ w_proj, int M, int K, int N, long long table_stride, int col0, bf16* __restrict__ out) {
    constexpr int DIM = 16 * NB;
    __shared__ float4_t sums_s[kSideWaves][NB][kWave];
    __shared__ __align__(16) uint16_t side_s[16][DIM + 8];
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int i = lane % 16, g = lane / 16;
    const int half = wave / 4, steps = K / 128;                          // steps of a half of the K axis
    // the entries of this thread's elements (row e / DIM, column e % DIM)
    constexpr int kOwn = 16 * DIM / (64 * kSideWaves);
    static_assert(kOwn >= 1 && kOwn * 64 * kSideWaves == 16 * DIM, "whole elements a thread");
    int token[kOwn];
#pragma unroll
    for (int q = 0; q < kOwn; ++q) token[q] = ids[min((static_cast<int>(threadIdx.x) + q * 64 * kSideWaves) / DIM, M - 1)];
    const int n_band = blockIdx.x * kSideWaves + wave, bands = N / 16;
    SideFragment proj[NB / 2];
#pragma unroll
    for (int u = 0; u < NB / 2; ++u)
        proj[u].u = *reinterpret_cast<const uint4*>(
            TILED ? w_proj + (static_cast<size_t>(min(n_band, bands - 1)) * (DIM / 32) + u) * 512 + lane * 8
                  : w_proj + (static_cast<size_t>(min(n_band, bands - 1)) * 16 + i) * DIM + u * 32 + 8 * g);

    const bf16* xp = x + static_cast<size_t>(min(i, M - 1)) * K + 8 * g;
    // all of the wavefront's steps on their way at once
    SideFragment fw[kSideSteps][2][NB], fx[kSideSteps][2];
#pragma unroll
    for (int u = 0; u < kSideSteps; ++u) {
        const int step = 2 * (half * steps + min(wave % 4 + 4 * u, steps - 1));      // in steps of 32 keys
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int b = 0; b < NB; ++b)
                fw[u][h][b].u = *reinterpret_cast<const uint4*>(TILED ? w_gate + (static_cast<size_t>(b) * (K / 32) + step + h) * 512 + lane * 8
                                                                      : w_gate + (static_cast<size_t>(b) * 16 + i) * K + (step + h) * 32 + 8 * g);
            fx[u][h].u = *reinterpret_cast<const uint4*>(xp + (step + h) * 32);
        }
    }
    float entry[kOwn];
#pragma unroll
    for (int q = 0; q < kOwn; ++q)
        entry[q] = to_float(table[static_cast<size_t>(token[q]) * table_stride + col0 + (threadIdx.x + q * 64 * kSideWaves) % DIM]);
    // (here, not behind the conditions below, into which the compiler would move them)
#pragma unroll
    for (int u = 0; u < kSideSteps; ++u)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int b = 0; b < NB; ++b) asm volatile("" : "+v"(fw[u][h][b].v));
            asm volatile("" : "+v"(fx[u][h].v));
        }
    float4_t acc[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[b] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < kSideSteps; ++u) {
        if (wave % 4 + 4 * u >= steps) break;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int b = 0; b < NB; ++b) acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[u][h][b].v, fx[u][h].v, acc[b], 0, 0, 0);
    }
#pragma unroll
    for (int b = 0; b < NB; ++b) sums_s[wave][b][lane] = acc[b];
    __syncthreads();
    // lane 16 gg + ii of a tile holds columns 4 gg .. + 3 of row ii
#pragma unroll
    for (int q = 0; q < kOwn; ++q) {
        const int e = threadIdx.x + q * 64 * kSideWaves, r = e / DIM, c = e % DIM;
        const int b = c / 16, at = (c % 16 / 4) * 16 + r, v = c % 4;
        float piece[2];
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            piece[p] = sums_s[4 * p][b][at][v];
#pragma unroll
            for (int w = 1; w < 4; ++w) piece[p] += sums_s[4 * p + w][b][at][v];
        }
        const float gate = to_float(from_float<bf16>(piece[0] + piece[1]));
        side_s[r][c] = from_float<bf16>(activate<ACT>(gate) * entry[q]).bits;
    }
    __syncthreads();
    if (n_band >= bands) return;
    float4_t y = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < NB / 2; ++u) {
        SideFragment side;
        side.u = *reinterpret_cast<const uint4*>(&side_s[i][u * 32 + 8 * g]);
        y = __builtin_amdgcn_mfma_f32_16x16x32_bf16(proj[u].v, side.v, y, 0, 0, 0);
    }
    if (i < M)
        *reinterpret_cast<uint2*>(out + static_cast<size_t>(i) * N + n_band * 16 + 4 * g) = make_uint2(pack2_bf16(y[0], y[1]), pack2_bf16(y[2], y[3]));
}

// Whether `wllm_token_side` has a kernel: at most 16 rows, dim 32 or 64, hidden a multiple of 128 (two halves of whole steps of 64 keys) of at most 2,048 (the
// steps of a wavefront that lie in its registers; and a chain of sums no longer than the few-row product's, which cuts a longer axis more often).
WLLM_API int wllm_token_side_takes(int rows, int hidden, int dim) {
    return rows >= 1 && rows <= kSideRows && hidden >= 128 && hidden <= 2 * 4 * 64 * kSideSteps && hidden % 128 == 0 && (dim == 32 || dim == 64);
}

// x [rows, hidden], w_gate [dim, hidden], table rows of `table_stride` elements, w_proj [hidden, dim] (`tiled`: both tile-major copies), out [rows, hidden], all
// bfloat16 and at multiples of 16 bytes but for the table.  Returns 0, a HIP error code, or -1 for what it does not take.
WLLM_API int wllm_token_side(const void* x, const void* w_gate, const int* ids, const void* table, long long table_stride, int col0,
                             const void* w_proj, int tiled, void* out, int rows, int hidden, int dim, int activation, hipStream_t stream) {
    if (!wllm_token_side_takes(rows, hidden, dim) || activation < 0 || activation >= kActivations || col0 < 0 || col0 + dim > table_stride) return -1;
    if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w_gate) | reinterpret_cast<uintptr_t>(w_proj) | reinterpret_cast<uintptr_t>(out)) % 16 != 0)
        return -1;
    const int grid = (hidden / 16 + kSideWaves - 1) / kSideWaves;
#define LAUNCH(NB, T)                                                                                                                       \
    WLLM_BY_ACTIVATION(activation, (token_side_kernel<NB, ACT, T><<<grid, 64 * kSideWaves, 0, stream>>>(                                    \
                                       static_cast<const bf16*>(x), static_cast<const bf16*>(w_gate), ids, static_cast<const bf16*>(table), \
                                       static_cast<const bf16*>(w_proj), rows, hidden, hidden, table_stride, col0, static_cast<bf16*>(out))))
    if (dim == 64 && tiled) { LAUNCH(4, true); }
    else if (dim == 64) { LAUNCH(4, false); }
    else if (tiled) { LAUNCH(2, true); }
    else { LAUNCH(2, false); }
#undef LAUNCH
    return launch_status();
}
