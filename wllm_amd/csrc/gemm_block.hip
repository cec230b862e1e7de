// out[M, N] = x[M, K] . w[N, K]^T for bfloat16 with more than 64 rows and few columns (a prompt's projections), on the matrix
// cores, in tiles of 64 to 192 rows of x by 64 or 128 rows of w: as many as make one round of a workgroup a compute unit (2,048 columns to 3,072 rows).
// And, where one round is enough, the stack of the sums of a long K axis in pieces, and the gated form out[M, I] = act(x . Wg^T) * (x . Wu^T) with
// w = [Wg; Wu], whose activation and product are made in the registers the sums are in: a tile's rows of w are then half gate rows, half
// the up rows that belong to them, and a wavefront has 16 of each.
//
// A workgroup of eight wavefronts walks the K axis in stages of 64 keys, a ring of them in shared memory.  A stage goes there straight from
// memory (global_load_lds_dwordx4: a wavefront's load is 8 rows of 8 chunks of 16 bytes; chunk c of row r lies at place c ^ (r % 8) of its
// row, so that the reads of a fragment meet no bank twice).  The wavefronts are TN / 32 across the rows of w, the others across those of x,
// each with 32 rows of w by its share of x (v_mfma_f32_16x16x32_bf16, w the A operand, x the B operand: lane (i, g) ends with four
// consecutive columns of one output row).  While it multiplies the fragments of a stage it reads those of the next into a second set of
// registers and sends its part of a stage further on, a read and a load between products each: reads in a row keep
// the products behind them waiting, as they issue no faster than shared memory serves them (with all reads in front 192 x 128 took 26.4 us for the 21.4 below).
//
// One barrier a stage.  In front of it a wavefront waits for its own loads of the next stage (at most D - 2 newer stages' are on their way) and
// for its reads of this one; behind it the next stage is whole, and the place of this one is free for stage s + D.
//
// What bounds it: the loads into shared memory, 64 bytes a clock and compute unit, the weights' first of them a trip to HBM, and the reads
// there.  us, weights from HBM, the library and this kernel, 2,048 keys to 2,048 columns at 100 / 256 / 508 / 1,024 / 1,500 / 2,048 rows
// 11.3 / 12.1 / 13.2 / 16.8 / 22.4 / 24.3 and 11.1 / 11.8 / 12.0 / 16.2 / 20.5 / 22.1; to 2,560 12.1 / 13.2 / 15.4 / 23.0 / 24.4 / 29.8 and
// 11.2 / 12.0 / 15.2 / 18.0 / 22.3 / 27.5; to 4,608 at 256 / 508 / 1,024 23.7 / 24.2 / 29.2 and 16.1 / 18.3 / 27.7; 768 keys to 2,048 at 508 / 1,500 7.8 / 10.0 and
// 6.3 / 9.2; 2,300 / 2,560 / 3,001 rows to 2,048 columns 29 / 26 / 28 and 26 / 26 / 28; rows in whole tiles of the library's and few of these lose up to an eighth
// (128 / 384 / 768 rows to 2,048 11.0 / 13.1 / 14.0 and 12.1 / 12.7 / 15.5).  Tiles of a second round find the machine half empty, and more rows are the library's
// (4,096 rows to 2,048 columns 34 and 41).  A call of the library costs the host 19 us where a launch costs 6, and a step of a few hundred rows waits for the host.
//
// Gated, 2,048 keys to 2 x 16,384 columns at 100 / 164 / 256 rows 35.3 / 37.4 / 42.1, in tiles of 128 37.0 / 44.3 / 48.7; to 2 x 4,096 13.2 / 16.1 / 17.6 and
// 24.1 / 23.7 / 24.6.  16,384 keys to 2,048 columns in 8 pieces at 65 / 164 rows 20.9 / 24.7 and 26.2 / 26.5.
//
// Tried: four wavefronts of 64 x 64 (25.4 for 19.8: nothing is left to multiply while one sends), loads by wavefronts of their own (as fast), rings of more
// than four stages (slower but for 64 x 64).  Every element is summed over k in ascending order (of a piece), whatever the tile.
#include "lds_load.h"

constexpr int kBlockKeys = 64;                       // keys a stage

template <int TM, int TN>
struct BlockShape {
    static constexpr int kWavesN = TN / 32, kWavesM = 8 / kWavesN;
    static constexpr int kXBlocks = TM / 16 / kWavesM;                          // blocks of 16 rows of x a wavefront has
    static constexpr int kStage = (TM + TN) * kBlockKeys * 2;                   // bytes
    static constexpr int kRing = TM + TN <= 128 ? 6 : (160 * 1024 / kStage < 4 ? 160 * 1024 / kStage : 4);
    static constexpr int kLoadsX = TM / 64, kLoadsW = TN / 64, kLoads = kLoadsX + kLoadsW;        // a wavefront and stage
    static_assert(TM % 64 == 0 && TN % 64 == 0 && kXBlocks >= 1 && kRing >= 3 && kRing * kStage <= 160 * 1024, "whole loads, and room for the ring");
};

// GATED: 0 plain, 1 + the gate's number for the gated product.  N is the number of rows of w (plain) or of gate rows (gated); `vectors`: a lane's
// neighbouring results (16 bytes, gated 8) lie at multiples of their size.
template <int TM, int TN, int GATED>
__global__ void __launch_bounds__(512, 2)
gemm_block_kernel(const bf16* __restrict__ x, const bf16* __restrict__ w, bf16* __restrict__ out, float* __restrict__ partial, int M, int N,
                  int K, int stride, bool vectors, int m_tiles, int n_tiles, int splits, GateShape shape) {
    using S = BlockShape<TM, TN>;
    constexpr int kColumns = GATED ? TN / 2 : TN;                    // output columns a tile
    constexpr bool kPair = GATED == kGatePairSquaredRelu + 1;
    constexpr int XB = S::kXBlocks, D = S::kRing, L = S::kLoads;
    extern __shared__ __align__(16) unsigned char ring_s[];
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int i = lane % 16, g = lane / 16;
    const int wm = wave / S::kWavesN, wn = wave % S::kWavesN;
    const uint32_t lds_base = shared_address(ring_s);

    // The items, at most one a workgroup, go to the XCDs in equal runs of an order in which 8 tiles of x rows share a tile of w rows.
    const int tiles = m_tiles * n_tiles, items = tiles * splits, all_stages = K / kBlockKeys;
    const int xcd = blockIdx.x % 8, per_xcd = items / 8, left = items % 8, in_run = blockIdx.x / 8;
    if (in_run >= per_xcd + (xcd < left ? 1 : 0)) return;
    const int item = xcd * per_xcd + min(xcd, left) + in_run;
    const int piece = item / tiles, tile = item - piece * tiles;
    const int begin = static_cast<int>(static_cast<long long>(piece) * all_stages / splits);
    const int stages = static_cast<int>(static_cast<long long>(piece + 1) * all_stages / splits) - begin;
    const int band = tile / (8 * n_tiles), in_band = tile - band * 8 * n_tiles;
    const int band_rows = min(8, m_tiles - 8 * band);
    const int n_tile = in_band / band_rows;
    const int m0 = (8 * band + in_band - n_tile * band_rows) * TM, n0 = n_tile * kColumns;

    // what this lane brings of a stage: rows 8 (wave + 8 u) + lane / 8 of the tiles, in bytes from the stage's first key
    uint32_t offset_x[S::kLoadsX], offset_w[S::kLoadsW];
    const int r0 = 8 * wave + lane / 8, c0 = (lane % 8) ^ (lane / 8);
#pragma unroll
    for (int u = 0; u < S::kLoadsX; ++u) offset_x[u] = (static_cast<uint32_t>(min(m0 + r0 + 64 * u, M - 1)) * K + c0 * 8) * 2;
#pragma unroll
    for (int u = 0; u < S::kLoadsW; ++u) {
        const int at = r0 + 64 * u;               // gated: the gate rows, then the up rows that belong to them
        const int row = !GATED || at < TN / 2 ? min(n0 + at, N - 1) : N + min(n0 + at - TN / 2, N - 1);
        offset_w[u] = (static_cast<uint32_t>(row) * K + c0 * 8) * 2;
    }
    auto send_one = [&](int s, int slot, int u) {
        const size_t at = static_cast<size_t>(begin + s) * (kBlockKeys * 2);
        const uint32_t to = lds_base + slot * S::kStage + wave * 1024;
        if (u < S::kLoadsX) load_to_shared(reinterpret_cast<const unsigned char*>(x) + at, offset_x[u < S::kLoadsX ? u : 0], to + u * 8192);
        else load_to_shared(reinterpret_cast<const unsigned char*>(w) + at, offset_w[u < S::kLoadsX ? 0 : u - S::kLoadsX],
                            to + TM * 128 + (u - S::kLoadsX) * 8192);
    };
#pragma unroll
    for (int s = 0; s < D; ++s)
        if (s < stages)
#pragma unroll
            for (int u = 0; u < L; ++u) send_one(s, s, u);
    const int place0 = (g ^ (i % 8)) * 16, place1 = ((4 + g) ^ (i % 8)) * 16;

    float4_t acc[2][XB];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < XB; ++b) acc[a][b] = float4_t{0.f, 0.f, 0.f, 0.f};
    Fragment fx[2][2][XB], fw[2][2][2];              // [set][32 keys][block]
    constexpr int kReads = 2 * (2 + XB), kProducts = 4 * XB;
    // fragment number r of a stage: w's and x's of its first 32 keys, then of the others
    auto read_one = [&](auto set, int slot, int r) {
        constexpr int F = decltype(set)::value ? 1 : 0;
        const int k = r / (2 + XB), f = r % (2 + XB);
        const unsigned char* from = ring_s + slot * S::kStage + (k ? place1 : place0);
        if (f < 2) fw[F][k][f].u = *reinterpret_cast<const uint4*>(from + TM * 128 + ((GATED ? f * (TN / 2) + wn * 16 : wn * 32 + f * 16) + i) * 128);
        else fx[F][k][f - 2].u = *reinterpret_cast<const uint4*>(from + ((wm * XB + f - 2) * 16 + i) * 128);
    };
    // stage s is in the registers `set`
    auto step = [&](auto set, auto other, int s, int slot, int next) {
        constexpr int F = decltype(set)::value ? 1 : 0;
        if (s + D - 1 < stages) wait_loads<(D - 2) * L>();
        else wait_loads<0>();
        // (through the builtin, so that the compiler knows that this stage's reads are done and does not wait for the next one's)
        __builtin_amdgcn_s_waitcnt(0xC07F);          // lgkmcnt(0)
        meet();
        const bool more = s + D < stages;
        int r = 0, u = 0;
#pragma unroll
        for (int p = 0; p < kProducts; ++p) {
            const int k = p / (2 * XB), b = p / 2 % XB, a = p % 2;
            acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[F][k][a].v, fx[F][k][b].v, acc[a][b], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (; r * kProducts < (p + 1) * kReads; ++r) read_one(other, next, r);
#pragma unroll
            for (; u * kProducts < (p + 1) * L; ++u)
                if (more) send_one(s + D, slot, u);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    if (stages >= D) wait_loads<(D - 1) * L>();
    else wait_loads<0>();
    meet();
#pragma unroll
    for (int r = 0; r < kReads; ++r) read_one(Flag<false>(), 0, r);
    int slot = 0;
    auto after = [](int q) { return q + 1 == D ? 0 : q + 1; };
    for (int s = 0; s < stages; s += 2) {
        // (behind the last stage a step reads its own once more, and nothing uses it)
        const int second = s + 1 < stages ? after(slot) : slot, third = s + 2 < stages ? after(second) : second;
        step(Flag<false>(), Flag<true>(), s, slot, second);
        if (s + 1 < stages) step(Flag<true>(), Flag<false>(), s + 1, second, third);
        slot = third;
    }
#pragma unroll
    for (int b = 0; b < XB; ++b) {
        const int m = m0 + (wm * XB + b) * 16 + i;
        if (m >= M) continue;
        if (GATED) {
            // a lane has four columns' gate and up sums
            const int n = n0 + wn * 16 + 4 * g;
            bf16* to = out + static_cast<size_t>(m) * stride + n;
#pragma unroll
            for (int h = 0; h < (kPair ? 2 : 1); ++h) {
                float r[4];
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    r[v] = kPair ? squared_relu(acc[h][b][v])
                                 : gate_product<(GATED > 0 && !kPair ? GATED - 1 : 0)>(acc[0][b][v], acc[1][b][v], shape);
                const uint32_t words[2] = {pack2_bf16(r[0], r[1]), pack2_bf16(r[2], r[3])};
                bf16* here = to + h * N;
                if (vectors && n + 3 < N) {
                    *reinterpret_cast<uint2*>(here) = make_uint2(words[0], words[1]);
                } else {
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        if (n + v < N) here[v] = bf16{static_cast<uint16_t>(words[v / 2] >> (16 * (v % 2)))};
                }
            }
            continue;
        }
        if (partial != nullptr) {
            float* row = partial + (static_cast<size_t>(piece) * M + m) * N;
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                const int n = n0 + wn * 32 + 16 * a + 4 * g;
                if (vectors && n + 3 < N) {
                    *reinterpret_cast<float4_t*>(row + n) = acc[a][b];
                } else {
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        if (n + v < N) row[n + v] = acc[a][b][v];
                }
            }
            continue;
        }
        uint32_t q[2][2];
#pragma unroll
        for (int a = 0; a < 2; ++a) {
            q[a][0] = pack2_bf16(acc[a][b][0], acc[a][b][1]);
            q[a][1] = pack2_bf16(acc[a][b][2], acc[a][b][3]);
        }
        // lanes g and g + 1 (g even) exchange halves, so that each has eight neighbouring columns of the 32
        typedef unsigned uint2_t __attribute__((ext_vector_type(2)));
        const uint2_t lo = __builtin_amdgcn_permlane16_swap(q[0][0], q[1][0], false, false);
        const uint2_t hi = __builtin_amdgcn_permlane16_swap(q[0][1], q[1][1], false, false);
        const uint32_t words[4] = {lo.x, hi.x, lo.y, hi.y};
        const int n = n0 + wn * 32 + 16 * (g & 1) + 8 * (g >> 1);
        bf16* to = out + static_cast<size_t>(m) * stride + n;
        if (vectors && n + 7 < N) {
            *reinterpret_cast<uint4*>(to) = make_uint4(words[0], words[1], words[2], words[3]);
        } else {
#pragma unroll
            for (int v = 0; v < 8; ++v)
                if (n + v < N) to[v] = bf16{static_cast<uint16_t>(words[v / 2] >> (16 * (v % 2)))};
        }
    }
}

// out = x w^T, rounded to bfloat16, in tiles of tile_m rows of x by tile_n rows of w (64, 128, 192 by 64, 128 and 192 by 128; gated 256 by 128 too); `stride` elements from a
// row of out to the next.  `splits` > 1: `out` is null and `partial` float32 [splits, M, N] takes the sums of the K axis's pieces.  `gated` = 1 + the
// gate's number (with limit, slope and shift for the clamped swish): the gated product, w [2N, K], gate rows first; with the paired squared
// relu out [M, 2N] = relu(x . w^T)^2.  K is a multiple of 64 and at least 64 * splits, x and w begin at multiples of 16 bytes and are smaller
// than 4 GiB, and tiles times pieces are at most 256, a round.  Returns 0, a HIP error code, or -1 for what it does not take.
WLLM_API int wllm_gemm_block(const void* x, const void* w, void* out, float* partial, int M, int N, int K, int stride, int splits, int gated,
                             float limit, float slope, float shift, int tile_m, int tile_n, hipStream_t stream) {
    if (M < 1 || N < 1 || K < kBlockKeys || K % kBlockKeys != 0 || splits < 1 || splits > K / kBlockKeys || gated < 0 || gated > kPairedGates ||
        tile_m < 64 || tile_n < 64)
        return -1;
    if ((splits > 1) != (partial != nullptr) || (splits > 1) != (out == nullptr) || (splits > 1 && gated != 0)) return -1;
    const bool pair = gated == kGatePairSquaredRelu + 1;
    if (out != nullptr && stride < (pair ? 2LL * N : N)) return -1;
    if (static_cast<size_t>(gated ? 2 : 1) * N * K * 2 >= (size_t(1) << 32) || static_cast<size_t>(M) * K * 2 >= (size_t(1) << 32)) return -1;
    if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) % 16 != 0) return -1;
    const bool vectors = partial ? reinterpret_cast<uintptr_t>(partial) % 16 == 0 && N % 4 == 0
                         : gated ? reinterpret_cast<uintptr_t>(out) % 8 == 0 && stride % 4 == 0 && (!pair || N % 4 == 0)
                                 : reinterpret_cast<uintptr_t>(out) % 16 == 0 && stride % 8 == 0;
    const int columns = gated ? tile_n / 2 : tile_n;
    const int m_tiles = (M - 1) / tile_m + 1, n_tiles = (N - 1) / columns + 1;
    const long long items = static_cast<long long>(m_tiles) * n_tiles * splits;
    if (items > 256) return -1;
    const int grid = static_cast<int>((items + 7) / 8 * 8);
    const int longest = (K / kBlockKeys + splits - 1) / splits;          // stages of an item
    const GateShape shape{limit, slope, shift};
#define LAUNCH(TM, TN, GATED)                                                                                                     \
    if (tile_m == TM && tile_n == TN) {                                                                                            \
        using S = BlockShape<TM, TN>;                                                                                              \
        static bool roomy = false;     /* more than 64 KiB of shared memory must be asked for once */                             \
        if (!roomy) {                                                                                                              \
            if (hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_block_kernel<TM, TN, GATED>),                              \
                                    hipFuncAttributeMaxDynamicSharedMemorySize, S::kRing * S::kStage) != hipSuccess)               \
                return launch_status();                                                                                            \
            roomy = true;                                                                                                          \
        }                                                                                                                          \
        gemm_block_kernel<TM, TN, GATED><<<grid, 512, (longest < S::kRing ? longest : S::kRing) * S::kStage, stream>>>(            \
            static_cast<const bf16*>(x), static_cast<const bf16*>(w), static_cast<bf16*>(out), partial, M, N, K, stride, vectors,  \
            m_tiles, n_tiles, splits, shape);                                                                                      \
        return launch_status();                                                                                                    \
    }
#define TILES(GATED)                                                                                    \
    do {                                                                                                \
        LAUNCH(64, 64, GATED) LAUNCH(128, 64, GATED) LAUNCH(192, 64, GATED)                             \
        LAUNCH(128, 128, GATED) LAUNCH(192, 128, GATED)                                                 \
        if (GATED) { LAUNCH(256, 128, (GATED ? GATED : 1)) }                                            \
    } while (0)
    if (gated == 0) { TILES(0); }
    else { WLLM_BY_PAIRED_GATE(gated - 1, TILES(GATE + 1)) }
#undef TILES
#undef LAUNCH
    return -1;
}
