// out[M, N] = x[M, K] . w[N, K]^T for bfloat16 with at most 64 rows and a K axis in few pieces: the stack of the pieces' sums for a
// consumer that adds them (a norm, a rotation), or their sum.  Bound by reading w once from HBM, and by what reading the stack costs
// the consumer: a norm has a workgroup a row, and a compute unit takes some 20 GB/s from other chiplets' writes, so after a
// stack of 16 it took 6.6 us at 8 rows (8.4 at 64) where it takes 2.0 alone, 4.3 (5.3) of 8, 3.1 (3.7) of 4, 2.5 (3.0) of 2.
//
// So the K axis is cut among wavefronts first: a workgroup of four owns one to three bands of 16 columns and one piece, its wavefronts
// take the piece's steps of 64 keys in turn and join their sums in shared memory.  In turn, not each a quarter: the
// workgroup then reads one run of a band's bytes (16,384 keys to 2,048 columns at 8 rows 11.8 us; with quarters, four times as many runs
// that begin 32 KiB apart, 14.6, at any depth of loads).  A wavefront brings its own steps of x and w straight to
// shared memory (global_load_lds_dwordx4), two steps in turn, and waits for nobody until the end.  Three or six steps in turn are as
// fast or slower (2,560 columns of 2,048 keys 5.4 against 4.3: fewer workgroups share a compute unit).
//
// Measured, us, the kernels before (registers, or four wavefronts on one stage of eight bands) and this one, product and norm together, 8 / 24 / 64 rows:
// 2,048 keys to 2,048 columns 8.8 / 9.5 / 11.1 and 6.2 / 6.7 / 8.1; to 2,560 9.1 / 10.2 / 12.4 and 7.1 / 7.7 / 9.4; 4,096 to 2,048
// 11.7 / 12.6 / 15.3 and 7.8 / 8.5 / 10.3; 5,632 to 2,048 13.5 / 14.3 / 18.2 and 8.8 / 9.4 / 11.9; 16,384 to 2,048 18.3 / 19.1 / 22.4 and
// 15.0 / 16.1 / 20.5 (the product alone 11.9 / 12.3 / 14.0 and 12.0 / 12.8 / 16.7); 24,576 to 3,072 30.5 / 31.4 / 35.6 and 27.8 / 28.7 / 35.8.
// Row by row instead of the tile-major copy: 2,048 to 2,048 3.7 us alone against 4.3, but 16,384 to 2,048 16.2 against 12.4.
//
// w is read from its tile-major copy (`wllm_tile_weight`: a band's 16 rows by 32 keys are one KiB in lane order, a load and a
// fragment alike) or row by row.  v_mfma_f32_16x16x32_bf16, w the A operand, x the B operand: lane (i, g) ends with four consecutive
// columns of one output row.  One order of sums: a wavefront's steps ascending, the four wavefronts, the pieces; both forms of the
// result and both orders of w have the same bits.
#include "common.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));

constexpr int kPieceWaves = 4, kPieceKeys = 64, kPieceSlots = 2;

union PFrag {
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

// MT: tiles of 16 rows of x.  B: bands of 16 rows of w a workgroup.
template <int MT, int B, bool TILED>
__global__ void __launch_bounds__(64 * kPieceWaves, 2)
gemm_pieces_kernel(const bf16* __restrict__ x, const bf16* __restrict__ w, float* __restrict__ sums, bf16* __restrict__ out, int M, int N,
                   int K, int splits, int joined) {
    extern __shared__ __align__(16) unsigned char ring_s[];
    constexpr int kLoads = 2 * (MT + B), kStep = kLoads * 1024;          // of a step and wavefront
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int i = lane % 16, g = lane / 16;
    const int here = joined ? splits : 1;                                // pieces of this workgroup
    const int piece = joined ? 0 : blockIdx.x % splits, n_base = (joined ? blockIdx.x : blockIdx.x / splits) * (16 * B);
    const int piece_steps = K / splits / kPieceKeys, k_begin = (piece * piece_steps + wave) * kPieceKeys;
    const int steps = (piece_steps - wave + kPieceWaves - 1) / kPieceWaves;       // steps wave, wave + 4, ... of the piece

    // a load of rows: eight of 128 bytes, chunk c of 16 bytes of row r at place c ^ (r % 8) (fragment reads without bank conflicts)
    const int row = lane / 8, chunk = (lane % 8) ^ row;
    uint32_t x_offset[MT][2], w_offset[B][2];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int u = 0; u < 2; ++u)
            x_offset[t][u] = static_cast<uint32_t>((static_cast<size_t>(min(16 * t + 8 * u + row, M - 1)) * K + k_begin + chunk * 8) * 2);
    const int bands = (N + 15) / 16;
#pragma unroll
    for (int b = 0; b < B; ++b)
#pragma unroll
        for (int u = 0; u < 2; ++u)
            w_offset[b][u] = static_cast<uint32_t>(
                TILED ? (static_cast<size_t>(min(n_base / 16 + b, bands - 1)) * (K / 32) + k_begin / 32 + u) * 1024 + lane * 16
                      : (static_cast<size_t>(min(n_base + 16 * b + 8 * u + row, N - 1)) * K + k_begin + chunk * 8) * 2);
    const uint32_t lds_base = __builtin_amdgcn_readfirstlane(
        static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) void*)ring_s)) + wave * (kPieceSlots * kStep));
    const unsigned char* mine = ring_s + wave * (kPieceSlots * kStep);
    const int total = steps * here;
    int sent = 0, slot = 0;
    size_t step = 0;                             // of the next load, from this wavefront's first
    auto send = [&](int to_slot) {
        const uint32_t to = lds_base + to_slot * kStep;
        const unsigned char* xb = reinterpret_cast<const unsigned char*>(x) + step * (kPieceKeys * 2);
        const unsigned char* wb = reinterpret_cast<const unsigned char*>(w) + step * (TILED ? 2048 : kPieceKeys * 2);
#pragma unroll
        for (int b = 0; b < B; ++b)
#pragma unroll
            for (int u = 0; u < 2; ++u)
                load_to_shared<false>(wb, w_offset[b][u], to + (2 * (MT + b) + u) * 1024);
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int u = 0; u < 2; ++u) load_to_shared<true>(xb, x_offset[t][u], to + (2 * t + u) * 1024);
        step += kPieceWaves;
        if (++sent == steps) {                   // the next piece begins
            step += piece_steps - steps * kPieceWaves;
            sent = 0;
        }
    };

    float4_t acc[B][MT];
    auto multiply = [&] {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const unsigned char* at = mine + slot * kStep;
            const int place = i * 128 + ((4 * u + g) ^ (i % 8)) * 16;
            PFrag fx[MT], fw[B];
#pragma unroll
            for (int b = 0; b < B; ++b) fw[b].u = *reinterpret_cast<const uint4*>(at + (MT + b) * 2048 + (TILED ? u * 1024 + lane * 16 : place));
#pragma unroll
            for (int t = 0; t < MT; ++t) fx[t].u = *reinterpret_cast<const uint4*>(at + t * 2048 + place);
#pragma unroll
            for (int b = 0; b < B; ++b)
#pragma unroll
                for (int t = 0; t < MT; ++t) acc[b][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[b].v, fx[t].v, acc[b][t], 0, 0, 0);
        }
    };
    static_assert(kPieceSlots == 2, "the slots change by turns");
    send(0);
    if (total > 1) send(1);
    // the wavefronts' sums of a piece meet here: behind the rings, or, of the last piece, in their place
    float4_t* parts = reinterpret_cast<float4_t*>(ring_s + (here > 1 ? kPieceWaves * kPieceSlots * kStep : 0));
    constexpr int kTiles = (B * MT + kPieceWaves - 1) / kPieceWaves;     // of them this wavefront adds tiles wave, wave + 4, ...
    float4_t whole[kTiles];
    int at_step = 0;
    for (int p = 0; p < here; ++p) {
#pragma unroll
        for (int b = 0; b < B; ++b)
#pragma unroll
            for (int t = 0; t < MT; ++t) acc[b][t] = float4_t{0.f, 0.f, 0.f, 0.f};
        for (int s = 0; s < steps; ++s, ++at_step) {
            if (at_step + 1 < total) wait_loads<kLoads>();                 // the step after it is on its way
            else wait_loads<0>();
            multiply();
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");             // the slot has been read
            if (at_step + 2 < total) send(slot);
            slot ^= 1;
        }
        if (here == 1 || p > 0) __syncthreads();       // the rings have been read (one piece); the piece before has been added
#pragma unroll
        for (int b = 0; b < B; ++b)
#pragma unroll
            for (int t = 0; t < MT; ++t) parts[((wave * B + b) * MT + t) * kWave + lane] = acc[b][t];
        __syncthreads();
#pragma unroll
        for (int e = 0; e < kTiles; ++e) {
            const int at = wave + e * kPieceWaves;
            if (at >= B * MT) continue;
            float4_t sum = parts[at * kWave + lane];
#pragma unroll
            for (int q = 1; q < kPieceWaves; ++q) sum += parts[(q * B * MT + at) * kWave + lane];
            whole[e] = p == 0 ? sum : whole[e] + sum;
        }
    }
    const bool aligned = out ? reinterpret_cast<uintptr_t>(out) % 8 == 0 : reinterpret_cast<uintptr_t>(sums) % 16 == 0;
#pragma unroll
    for (int e = 0; e < kTiles; ++e) {
        const int at = wave + e * kPieceWaves;
        if (at >= B * MT) continue;
        const float4_t sum = whole[e];
        const int m = at % MT * 16 + i, n = n_base + at / MT * 16 + 4 * g;
        if (m >= M) continue;
        const size_t to = (static_cast<size_t>(piece) * M + m) * N + n;          // (joined: piece 0)
        if (n + 3 < N && N % 4 == 0 && aligned) {
            if (out) *reinterpret_cast<uint2*>(out + to) = make_uint2(pack2_bf16(sum[0], sum[1]), pack2_bf16(sum[2], sum[3]));
            else *reinterpret_cast<float4_t*>(sums + to) = sum;
        } else {
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                if (n + v >= N) continue;
                if (out) out[to + v] = from_float<bf16>(sum[v]);
                else sums[to + v] = sum[v];
            }
        }
    }
}

// x w^T of at most 64 rows, the K axis in `splits` pieces of at least 256 keys, multiples of 64.  `joined` 0: float32 `sums`
// [splits, M, N].  1: their sum in order, in float32 `sums` [M, N] or bfloat16 `out` [M, N].  `tiled`: w is the tile-major copy.
// `bands` (1 to 3) of 16 columns a workgroup.  x and w at multiples of 16 bytes and below 4 GiB.  Returns 0, a HIP error code, or -1.
WLLM_API int wllm_gemm_pieces(const void* x, const void* w, int tiled, float* sums, void* out, int M, int N, int K, int splits,
                              int joined, int bands, hipStream_t stream) {
    if (M < 1 || M > 64 || N < 1 || splits < 1 || K < 1 || K % (kPieceKeys * splits) != 0 || K / splits < kPieceKeys * kPieceWaves ||
        (sums == nullptr) == (out == nullptr) || (out && !joined) || bands < 1 || bands > 3)
        return -1;
    if ((static_cast<size_t>(N) + 15) * K * 2 >= (size_t(1) << 32) || static_cast<size_t>(M) * K * 2 >= (size_t(1) << 32)) return -1;
    if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) % 16 != 0) return -1;
    const long long blocks = (static_cast<long long>(N) + 16 * bands - 1) / (16 * bands) * (joined ? 1 : splits);
    if (blocks > 0x7fffffffLL) return -1;
    const bf16* xp = static_cast<const bf16*>(x);
    const bf16* wp = static_cast<const bf16*>(w);
    const bool behind = joined && splits > 1;          // the meeting place lies behind the rings
#define LAUNCH_T(MT, B, T)                                                                                          \
    do {                                                                                                            \
        constexpr int kRings = kPieceSlots * 2 * (MT + B) * 1024 * kPieceWaves, kMeet = B * MT * 1024 * kPieceWaves; \
        static_assert(kRings >= kMeet && kRings + kMeet <= 160 * 1024, "shared memory of a compute unit");           \
        static bool roomy = false;     /* more than 64 KiB of shared memory must be asked for once */              \
        if (!roomy) {                                                                                               \
            if (hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_pieces_kernel<MT, B, T>),                   \
                                    hipFuncAttributeMaxDynamicSharedMemorySize, kRings + kMeet) != hipSuccess)      \
                return launch_status();                                                                             \
            roomy = true;                                                                                           \
        }                                                                                                           \
        gemm_pieces_kernel<MT, B, T><<<static_cast<unsigned>(blocks), 64 * kPieceWaves, kRings + (behind ? kMeet : 0), stream>>>( \
            xp, wp, sums, static_cast<bf16*>(out), M, N, K, splits, joined);                                        \
    } while (0)
#define LAUNCH(MT, B)                       \
    do {                                    \
        if (tiled) LAUNCH_T(MT, B, true);   \
        else LAUNCH_T(MT, B, false);        \
    } while (0)
#define BY_B(MT)                            \
    switch (bands) {                        \
        case 1: LAUNCH(MT, 1); break;       \
        case 2: LAUNCH(MT, 2); break;       \
        default: LAUNCH(MT, 3); break;      \
    }
    switch ((M + 15) / 16) {
        case 1: BY_B(1) break;
        case 2: BY_B(2) break;
        case 3: BY_B(3) break;
        default: BY_B(4) break;
    }
#undef BY_B
#undef LAUNCH
#undef LAUNCH_T
    return launch_status();
}
