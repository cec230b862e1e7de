// out[M, N] = x[M, K] . w[N, K]^T for bfloat16 with at most 64 rows and a K axis in pieces, and the gated form
// out[M, I] = act(x . Wg^T) * (x . Wu^T) with w = [Wg; Wu] for 33 to 64 rows, whose activation and product are made in the registers the
// sums are in.  Both are bound by reading w once from HBM.
//
// The kernels of few rows (`gemm_skinny.hip`) hold the weights on their way in registers; with three and four tiles of 16 rows
// the sums and the staged x leave them eight wavefronts a compute unit, and each pair of bands reads all of x again.  Here
// everything goes straight to shared memory (global_load_lds_dwordx4): a workgroup of four wavefronts has 64 rows of x and
// eight bands of 16 rows of w (gated: four bands of gate rows and the four of the up rows that belong to them), in stages of 64 keys,
// 8 + 16 KB each, three in turn, two of them on their way while one is multiplied, and two workgroups share a compute unit (96 KB
// on their way).  Six stages and one workgroup leave a launch of some more workgroups than compute units half empty: to 10,304
// columns 16.3 us against 13.9 at 64 rows, to 2 x 24,576 of 3,072 keys 56.9 against 54.0.
//
// Measured, us, the few-row kernels and this one: gated, 2,048 keys to 2 x 16,384 columns, 40 / 64 rows 28.3 / 33.2 and 25.8 / 26.0 (5.2 TB/s);
// 3,072 keys to 2 x 24,576 63.3 / 74.1 and 51.3 / 54.0; plain, 3,072 keys to 12,288 columns in two pieces at 8 / 24 / 64 rows 15.2 / 17.4 / 21.7 and
// 14.7 / 15.1 / 17.2; 1,024 to 16,384 8.9 / 9.5 / 11.8 and 8.3 / 8.8 / 10.0.  At 32 rows and below the gated few-row kernel is as fast (24 rows 25.8 and
// 25.5; 8 rows 24.8 and 26.3), and so many columns that no K axis is cut belong to the unsplit one (256,000 columns, 64 rows: 199 and 214).
// Fewer columns belong to the kernel that leaves fewer pieces (`gemm_pieces.hip`).
//
// A wavefront brings and reads its own two bands, so only x is waited for together: one barrier a stage, behind which
// the buffer of the stage before is free as well.  w is read from its tile-major copy (`wllm_tile_weight`: a band's 16 rows by 32
// keys are one KiB in lane order, a load and a fragment alike) or row by row (chunk c of 16 bytes of row r then lies at
// place c ^ (r % 8) of its row, as the chunks of x do).  v_mfma_f32_16x16x32_bf16, w the A operand, x the B operand:
// lane (i, g) ends with four consecutive columns of one output row.
//
// A plain product leaves float32 sums [splits, M, N], a piece of the K axis after the other.  Every element is summed over k in
// ascending order within a piece (gated: within a half), so the sums have the bits of the few-row kernels'.  The workgroups of
// a piece get indices that are equal modulo the pieces, so that (eight pieces and more) they run on one XCD and find
// their part of x in its L2.
#include "common.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));

constexpr int kStreamRows = 64, kStreamBands = 8, kStreamKeys = 64, kStreamStages = 3;
constexpr int kStreamX = kStreamRows * kStreamKeys * 2, kStreamW = kStreamBands * 16 * kStreamKeys * 2;
constexpr int kStreamStage = kStreamX + kStreamW;
constexpr int kStreamLoads = 6;              // loads a wavefront and stage: two of x, four of w

union SFrag {
    uint4 u;
    bf16x8_t v;
};

// 16 bytes a lane from base + offset into shared memory at `lds_address` + 16 * lane; M0 is put back as it was, and the
// kernel waits for these loads itself (the compiler does not see them).  KEPT false: what is read once is not kept in the caches.
template <bool KEPT>
static __device__ __forceinline__ void load_to_shared(const void* base, uint32_t offset, uint32_t lds_address) {
    uint32_t saved_m0;
    if (KEPT)
        asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
                     : "=&s"(saved_m0) : "v"(offset), "s"(base), "s"(lds_address) : "memory");
    else
        asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt\n\ts_mov_b32 m0, %0"
                     : "=&s"(saved_m0) : "v"(offset), "s"(base), "s"(lds_address) : "memory");
}

template <int N>
static __device__ __forceinline__ void wait_loads() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

// GATED: 0 plain, 1 + the gate's number.  N: rows of w (plain), or of gate rows (gated).
template <int GATED, bool TILED>
__global__ void __launch_bounds__(256, 2)
gemm_stream_kernel(const bf16* __restrict__ x, const bf16* __restrict__ w, bf16* __restrict__ out, float* __restrict__ sums, int M,
                   int N, int K, int out_stride, int splits, GateShape shape) {
    extern __shared__ __align__(16) unsigned char ring_s[];
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int i = lane % 16, g = lane / 16;
    constexpr int kColumns = GATED ? 64 : 128;
    const int piece = blockIdx.x % splits, n_base = blockIdx.x / splits * kColumns;
    const int piece_k = K / splits, k_begin = piece * piece_k;
    const int stages = piece_k / kStreamKeys;

    // ---- what this wavefront brings of a stage: x rows 8 (wave + 4 u) .. + 7, and its two bands of w, two loads each ----
    const int chunk = (lane % 8) ^ (lane / 8);
    uint32_t x_offset[2];
#pragma unroll
    for (int u = 0; u < 2; ++u)
        x_offset[u] = static_cast<uint32_t>((static_cast<size_t>(min(8 * (wave + 4 * u) + lane / 8, M - 1)) * K + k_begin + chunk * 8) * 2);
    const int bands = (N + 15) / 16;
    const unsigned char* w_base[2];              // a band's bytes at the piece's first key
    uint32_t w_offset[2][2];                     // [band][load] within it
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        const int row0 = GATED ? n_base + wave * 16 : n_base + (2 * wave + b) * 16;          // of the gate's (b 0), of the up's rows (b 1)
        if (TILED) {
            const size_t band = static_cast<size_t>(min(row0 / 16, bands - 1)) + (GATED && b == 1 ? bands : 0);
            w_base[b] = reinterpret_cast<const unsigned char*>(w) + (band * (K / 32) + k_begin / 32) * 1024;
#pragma unroll
            for (int u = 0; u < 2; ++u) w_offset[b][u] = u * 1024 + lane * 16;
        } else {
            w_base[b] = reinterpret_cast<const unsigned char*>(w) + static_cast<size_t>(k_begin) * 2 +
                        (GATED && b == 1 ? static_cast<size_t>(N) * K * 2 : 0);
#pragma unroll
            for (int u = 0; u < 2; ++u)
                w_offset[b][u] = static_cast<uint32_t>((static_cast<size_t>(min(row0 + 8 * u + lane / 8, N - 1)) * K + chunk * 8) * 2);
        }
    }
    const uint32_t lds_base = __builtin_amdgcn_readfirstlane(
        static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) void*)ring_s)));
    auto send = [&](int s, int slot) {
        const uint32_t to = lds_base + slot * kStreamStage;
        const unsigned char* xb = reinterpret_cast<const unsigned char*>(x) + static_cast<size_t>(s) * (kStreamKeys * 2);
        const size_t w_at = static_cast<size_t>(s) * (TILED ? 2048 : kStreamKeys * 2);
#pragma unroll
        for (int u = 0; u < 2; ++u) load_to_shared<true>(xb, x_offset[u], to + (wave + 4 * u) * 1024);
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int u = 0; u < 2; ++u)
                load_to_shared<false>(w_base[b] + w_at, w_offset[b][u], to + kStreamX + (wave * 2 + b) * 2048 + u * 1024);
    };

    float4_t acc[2][4];          // [band][16 rows of x]
    auto clear = [&] {
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int t = 0; t < 4; ++t) acc[b][t] = float4_t{0.f, 0.f, 0.f, 0.f};
    };
    clear();
#pragma unroll
    for (int p = 0; p < kStreamStages - 1; ++p)
        if (p < stages) send(p, p);
    int slot = 0;
    auto walk = [&](int from, int to) {
        for (int s = from; s < to; ++s) {
            // this wavefront's loads of the stage have landed: those of the stage behind it are not waited for
            if (s + 1 < stages) wait_loads<(kStreamStages - 2) * kStreamLoads>();
            else wait_loads<0>();
            __syncthreads();                                     // everyone's have, and everyone is done with the stage before
            if (s + kStreamStages - 1 < stages) send(s + kStreamStages - 1, slot == 0 ? kStreamStages - 1 : slot - 1);
            const unsigned char* xs = ring_s + slot * kStreamStage;
            const unsigned char* ws = xs + kStreamX + wave * 4096;
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const int place = ((4 * k + g) ^ (i % 8)) * 16;
                SFrag fw[2], fx[4];
#pragma unroll
                for (int b = 0; b < 2; ++b)
                    fw[b].u = *reinterpret_cast<const uint4*>(ws + b * 2048 + (TILED ? k * 1024 + lane * 16 : i * 128 + place));
#pragma unroll
                for (int t = 0; t < 4; ++t) fx[t].u = *reinterpret_cast<const uint4*>(xs + (16 * t + i) * 128 + place);
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int t = 0; t < 4; ++t) acc[b][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[b].v, fx[t].v, acc[b][t], 0, 0, 0);
            }
            slot = slot == kStreamStages - 1 ? 0 : slot + 1;
        }
    };
    if (GATED) {
        // the halves of the K axis are summed by themselves, as the kernel of fewer rows sums them
        walk(0, stages / 2);
        float4_t first[2][4];
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int t = 0; t < 4; ++t) first[b][t] = acc[b][t];
        clear();
        walk(stages / 2, stages);
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int t = 0; t < 4; ++t) acc[b][t] = first[b][t] + acc[b][t];
    } else {
        walk(0, stages);
    }

    // ---- lane (i, g) holds, of band b and tile t, output row 16 t + i and columns 4g .. 4g + 3 of the band ----
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const int m = 16 * t + i;
        if (m >= M) continue;
        if (GATED) {
            constexpr bool kPair = GATED == kGatePairSquaredRelu + 1;
            const int n = n_base + wave * 16 + 4 * g;
            float r[4], r2[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const float gate = acc[0][t][v], up = acc[1][t][v];
                if (kPair) {
                    r[v] = squared_relu(gate);
                    r2[v] = squared_relu(up);
                } else {
                    r[v] = gate_product<(GATED > 0 && !kPair ? GATED - 1 : 0)>(gate, up, shape);
                }
            }
            bf16* o = out + static_cast<size_t>(m) * out_stride + n;
            if (n + 3 < N && N % 4 == 0 && out_stride % 4 == 0 && reinterpret_cast<uintptr_t>(out) % 8 == 0) {
                *reinterpret_cast<uint2*>(o) = make_uint2(pack2_bf16(r[0], r[1]), pack2_bf16(r[2], r[3]));
                if (kPair) *reinterpret_cast<uint2*>(o + N) = make_uint2(pack2_bf16(r2[0], r2[1]), pack2_bf16(r2[2], r2[3]));
            } else {
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    if (n + v < N) {
                        o[v] = from_float<bf16>(r[v]);
                        if (kPair) o[N + v] = from_float<bf16>(r2[v]);
                    }
            }
        } else {
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const int n = n_base + (2 * wave + b) * 16 + 4 * g;
                float* o = sums + (static_cast<size_t>(piece) * M + m) * N + n;
                if (n + 3 < N && N % 4 == 0 && reinterpret_cast<uintptr_t>(sums) % 16 == 0) {
                    *reinterpret_cast<float4_t*>(o) = acc[b][t];
                } else {
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        if (n + v < N) o[v] = acc[b][t][v];
                }
            }
        }
    }
}

// The plain product (gated 0): float32 `sums` [splits, M, N].  The gated one (1 + the gate's number, with limit, slope and shift for the
// clamped swish; splits 1): bfloat16 `out`, `out_stride` elements from a row to the next; w [2N, K], gate rows first; with the
// paired squared relu out [M, 2N] = relu(x . w^T)^2.  `tiled`: w is the tile-major copy (gated: of the two halves, one after the other).  At most
// 64 rows, K a multiple of 64 * splits (gated: of 128), x and w at multiples of 16 bytes and below 4 GiB.  Returns 0, a HIP error code, or -1.
WLLM_API int wllm_gemm_stream(const void* x, const void* w, int tiled, void* out, float* sums, int M, int N, int K, int out_stride,
                              int splits, int gated, float limit, float slope, float shift, hipStream_t stream) {
    if (M < 1 || M > kStreamRows || N < 1 || splits < 1 || K < kStreamKeys * splits || K % (kStreamKeys * splits) != 0 || gated < 0 ||
        gated > kPairedGates || (gated && K % (2 * kStreamKeys) != 0))
        return -1;
    if (gated ? (out == nullptr || splits != 1 || out_stride < (gated == kGatePairSquaredRelu + 1 ? 2LL : 1LL) * N) : sums == nullptr) return -1;
    const size_t w_rows = static_cast<size_t>(gated ? 2 : 1) * N;
    if (w_rows * K * 2 >= (size_t(1) << 32) || static_cast<size_t>(M) * K * 2 >= (size_t(1) << 32)) return -1;
    if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) % 16 != 0) return -1;
    constexpr int kShared = kStreamStages * kStreamStage;
    const int columns = gated ? 64 : 128;
    const long long blocks = static_cast<long long>((N + columns - 1) / columns) * splits;
    if (blocks > 0x7fffffffLL) return -1;
    const bf16* xp = static_cast<const bf16*>(x);
    const bf16* wp = static_cast<const bf16*>(w);
    const GateShape shape{limit, slope, shift};
#define LAUNCH_T(GATED, T)                                                                                          \
    do {                                                                                                            \
        static bool roomy = false;     /* more than 64 KiB of shared memory must be asked for once */              \
        if (!roomy) {                                                                                               \
            if (hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_stream_kernel<GATED, T>),                   \
                                    hipFuncAttributeMaxDynamicSharedMemorySize, kShared) != hipSuccess)             \
                return launch_status();                                                                             \
            roomy = true;                                                                                           \
        }                                                                                                           \
        gemm_stream_kernel<GATED, T><<<static_cast<unsigned>(blocks), 256, kShared, stream>>>(                      \
            xp, wp, static_cast<bf16*>(out), sums, M, N, K, out_stride, splits, shape);                             \
    } while (0)
#define LAUNCH(GATED)                      \
    if (tiled) { LAUNCH_T(GATED, true); }   \
    else { LAUNCH_T(GATED, false); }
    if (gated == 0) { LAUNCH(0); }
    else { WLLM_BY_PAIRED_GATE(gated - 1, LAUNCH(GATE + 1)) }
#undef LAUNCH
#undef LAUNCH_T
    return launch_status();
}
