// out[M, N] = x[M, K] * w[N, K]^T for float32 and bfloat16 operands, accumulated in float32.  It is
// the product of the float32 path, and the product of last resort for bfloat16 (shapes the
// bfloat16 matrix-core kernels do not take, float32 results from bfloat16 operands).  No
// reduced-precision mode is involved anywhere: float32 operands are multiplied and added as float32,
// on the matrix cores' float32 instruction where the K axis is a multiple of 4 (below), with fused
// multiply-adds on the vector units otherwise (this kernel).
//
// A workgroup of 256 threads makes a 64x64 tile of the result; the K axis is walked in steps of
// 16 through shared memory; a thread holds a 4x4 block.  The K axis is cut into segments of kSegment
// keys counted from 0, a segment is summed over k in ascending order of fused multiply-adds from
// zero, and the segments' sums are added in ascending order: an order fixed by K alone, so a row's
// result does not depend on the other rows of the batch.
#include "common.h"

constexpr int kTile = 64;
constexpr int kStep = 16;
constexpr int kSegment = 2048;

template <typename TI, typename TO>
__global__ void __launch_bounds__(256)
gemm_nt_kernel(const TI* __restrict__ x, const TI* __restrict__ w, TO* __restrict__ out, int M, int N, int K) {
    __shared__ float xs[kStep][kTile + 4];
    __shared__ float ws[kStep][kTile + 4];
    const int tid = threadIdx.x;
    const int row0 = blockIdx.y * kTile, col0 = blockIdx.x * kTile;
    const int tr = (tid / 16) * 4, tc = (tid % 16) * 4;
    float acc[4][4], total[4][4];
    // each thread stages 4 elements of x and 4 of w per step: row = tid / 4, k = (tid % 4) * 4 ..
    const int lr = tid / 4, lk = (tid % 4) * 4;
    for (int seg0 = 0; seg0 < K; seg0 += kSegment) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;
    for (int k0 = seg0; k0 < min(K, seg0 + kSegment); k0 += kStep) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int k = k0 + lk + e;
            const int xr = row0 + lr, wr = col0 + lr;
            xs[lk + e][lr] = (xr < M && k < K) ? to_float(x[static_cast<size_t>(xr) * K + k]) : 0.f;
            ws[lk + e][lr] = (wr < N && k < K) ? to_float(w[static_cast<size_t>(wr) * K + k]) : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kStep; ++k) {
            float a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = xs[k][tr + i];
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = ws[k][tc + j];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
        }
        __syncthreads();
    }
    // the segment's sum joins the sums of the segments before it
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) total[i][j] = seg0 == 0 ? acc[i][j] : total[i][j] + acc[i][j];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = row0 + tr + i;
        if (r >= M) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int c = col0 + tc + j;
            if (c < N) out[static_cast<size_t>(r) * N + c] = from_float<TO>(total[i][j]);
        }
    }
}

// ---- float32 on the matrix cores ----------------------------------------------------------------
// v_mfma_f32_16x16x4_f32 multiplies and accumulates IEEE float32 (no narrower format is involved), at
// twice the rate that unpacked vector multiply-adds reach.  Both kernels below make an element of the
// result by the same instructions on the same numbers in the same order, whatever the rows and columns
// beside it, so a token's projection has the same bits in a decode step as inside a prompt:
//   the K axis is cut into segments of kF32Segment keys counted from 0; within a segment the keys go
//   in chunks of 16; a chunk is four instructions, the t-th of which takes the keys 16 q + 4 g + t
//   (g = 0..3, the lane's group) and accumulates into the segment's sum, which starts at zero; the
//   segments' sums are added in ascending order.
// A lane (i, g) of a wavefront holds, of a chunk, w[n0 + i][16 q + 4 g .. + 3] and x[m0 + i][the same
// keys]: one 16-byte load each, whose t-th element goes to the t-th instruction.  The first operand is
// w, so a lane's four results are four consecutive columns of one row of out.
typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int kF32Segment = 512;
constexpr int kF32Chunk = 16;

__device__ __forceinline__ f32x4 mfma_chunk(const f32x4 a, const f32x4 b, f32x4 acc) {
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[0], b[0], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[1], b[1], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[2], b[2], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[3], b[3], acc, 0, 0, 0);
    return acc;
}

// At most 64 rows (the decode steps of the float32 path): the weights stream from memory straight
// into the lanes that multiply them, a wavefront a band of 16 columns, `U` chunks of it in flight at a
// time; x comes through the caches (all wavefronts read the same few rows).  MT tiles of 16 rows: a
// fragment of the weights feeds MT products, each row's sums in the one order (the tiled kernel below
// took 300 us for the gate and up projections of 64 rows at the 2B sizes, this one streams them).  SPLIT: a wavefront takes
// one segment of the K axis (blockIdx.y) and leaves its sum in partial[segment]; a second kernel adds
// the segments in ascending order.  Otherwise it walks all segments and adds as it goes.
// TILED: w is the weight's tile-major copy (`tile_weight_f32_kernel`): per band of 16 rows and chunk
// of 16 keys one KiB in lane order, so that a wavefront's load is one contiguous KiB and its walk along
// K one contiguous run (gate and up at Gemma-2B sizes: 76 us from the row-major weight, whose loads
// touch 16 rows of 64 bytes each, 49 us from the copy).
template <bool SPLIT, bool TILED, int MT>
__global__ void __launch_bounds__(256)
gemm_f32_few_rows_kernel(const float* __restrict__ x, const float* __restrict__ w, float* __restrict__ out, int M, int N,
                         int K) {
    constexpr int U = MT <= 2 ? 8 : 4;
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int i = lane % 16, g = lane / 16;
    const int n0 = (blockIdx.x * 4 + wave) * 16;
    if (n0 >= N) return;
    const int chunks_of_row = (K + kF32Chunk - 1) / kF32Chunk;
    const float* wrow = TILED ? w + (static_cast<size_t>(n0 / 16) * chunks_of_row * 64 + lane) * 4
                              : w + static_cast<size_t>(min(n0 + i, N - 1)) * K;
    const float* xrow[MT];
    bool x_live[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        xrow[t] = x + static_cast<size_t>(min(16 * t + i, M - 1)) * K;
        x_live[t] = 16 * t + i < M;
    }
    const int segments = (K + kF32Segment - 1) / kF32Segment;
    const int seg_first = SPLIT ? blockIdx.y : 0, seg_end = SPLIT ? blockIdx.y + 1 : segments;
    f32x4 total[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) total[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int seg = seg_first; seg < seg_end; ++seg) {
        const int k_begin = seg * kF32Segment, k_end = min(K, k_begin + kF32Segment);
        f32x4 acc[MT];
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        for (int k0 = k_begin; k0 < k_end; k0 += U * kF32Chunk) {
            f32x4 a[U], b[MT][U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                // every lane loads, from a clamped address; what lies beyond the segment becomes zero
                const int k = k0 + u * kF32Chunk + 4 * g;
                // (a chunk beyond the row's last is clamped to the last: what it holds becomes zero below)
                a[u] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(
                    TILED ? wrow + static_cast<size_t>(min(k0 / kF32Chunk + u, chunks_of_row - 1)) * 256 : wrow + min(k, K - 4)));
#pragma unroll
                for (int t = 0; t < MT; ++t) b[t][u] = *reinterpret_cast<const f32x4*>(xrow[t] + min(k, K - 4));
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int k = k0 + u * kF32Chunk + 4 * g;
                const bool live = k < k_end;
                const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
                const f32x4 av = live ? a[u] : zero;
                if (k0 + u * kF32Chunk < k_end) {     // the same for all lanes
#pragma unroll
                    for (int t = 0; t < MT; ++t) acc[t] = mfma_chunk(av, live && x_live[t] ? b[t][u] : zero, acc[t]);
                }
            }
        }
#pragma unroll
        for (int t = 0; t < MT; ++t) total[t] = seg == seg_first ? acc[t] : total[t] + acc[t];
    }
    // lane (i, g) holds out[row 16 t + i][n0 + 4 g .. + 3]
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        if (!x_live[t]) continue;
        float* dst = out + (SPLIT ? static_cast<size_t>(blockIdx.y) * M * N : 0) + static_cast<size_t>(16 * t + i) * N + n0 + 4 * g;
        if (N % 4 == 0 && n0 + 4 * g + 3 < N) {
            *reinterpret_cast<f32x4*>(dst) = total[t];
        } else {
#pragma unroll
            for (int v = 0; v < 4; ++v)
                if (n0 + 4 * g + v < N) dst[v] = total[t][v];
        }
    }
}

// More rows: a workgroup of four wavefronts (2 x 2) makes 32 WM rows by 32 WN columns; the tiles of
// x and w of a chunk go through shared memory, the next chunks' loads in flight while this one is
// multiplied.  Rows of a tile are padded to 20 floats, so that the 16-byte fragment reads of 8 lanes
// fall into different banks.  What lies beyond the K axis becomes zero when it is put into shared memory
// and not when it is loaded: a choice made on a load's result waits for the load at once (with it there,
// 4,096 x 4,096 x 4,096 ran at 109 TFLOP/s, every chunk a trip to memory).
// SPLIT: a workgroup (blockIdx.z) takes `per_group` segments of the K axis and leaves each one's sum in
// out[segment]; the kernel below adds them in the order in which the unsplit walk does.
// PART: the last tile's blocks of 16 rows that lie beyond the rows are left out, a branch in front of each block's products.  A wavefront
// has every second block, so that both halves of the workgroup get less to do (333 rows of 2,048 keys to 32,768 columns 423 to 400 us, 260 rows 421
// to 352, 140 rows 231 to 192; 16,384 keys to 2,048 columns, 333 rows, 241 to 227).
template <int WM, int WN, bool SPLIT, bool PART>
__global__ void __launch_bounds__(256, 2)
gemm_f32_tile_kernel(const float* __restrict__ x, const float* __restrict__ w, float* __restrict__ out, int M, int N, int K,
                     int per_group) {
    constexpr int TM = 32 * WM, TN = 32 * WN, kStride = kF32Chunk + 4;
    constexpr int XP = TM * 4 / 256, WP = TN * 4 / 256;       // 16-byte pieces of a chunk's tiles per thread
    static_assert(XP * 256 == TM * 4 && WP * 256 == TN * 4, "whole pieces per thread");
    __shared__ __align__(16) float xs[2][TM * kStride];
    __shared__ __align__(16) float ws[2][TN * kStride];
    const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    const int i = lane % 16, g = lane / 16;
    const int m0 = blockIdx.y * TM, n0 = blockIdx.x * TN;
    // a wavefront has every second block of 16 rows, so that the rows that the last tile has not are left out by both halves
    const int wm0 = wave / 2 * 16, wn0 = (wave % 2) * (TN / 2);
    const int live = __builtin_amdgcn_readfirstlane(min(WM, (M - m0 - wm0 + 31) / 32));       // of its blocks, those with rows
    // a thread's pieces: row tid / 4 (+ 64 per further piece), keys 4 (tid % 4) ..
    const int p_row = tid / 4, p_k = (tid % 4) * 4;
    const float* xsrc[XP];
    const float* wsrc[WP];
#pragma unroll
    for (int p = 0; p < XP; ++p) xsrc[p] = x + static_cast<size_t>(min(m0 + p_row + 64 * p, M - 1)) * K;
#pragma unroll
    for (int p = 0; p < WP; ++p) wsrc[p] = w + static_cast<size_t>(min(n0 + p_row + 64 * p, N - 1)) * K;
    // two sets of registers for chunks on their way: a chunk is asked for two chunks before it is
    // multiplied, so a trip to memory has two chunks' products to hide behind
    f32x4 xr[2][XP], wr[2][WP];
    auto fetch = [&](f32x4 (&xq)[XP], f32x4 (&wq)[WP], int k0) {
        const int k = min(k0 + p_k, K - 4);
#pragma unroll
        for (int p = 0; p < XP; ++p) xq[p] = *reinterpret_cast<const f32x4*>(xsrc[p] + k);
#pragma unroll
        for (int p = 0; p < WP; ++p) wq[p] = *reinterpret_cast<const f32x4*>(wsrc[p] + k);
    };
    auto stage = [&](int buf, f32x4 (&xq)[XP], f32x4 (&wq)[WP], int k0) {
        if (k0 + kF32Chunk > K && k0 + p_k >= K) {
            const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int p = 0; p < XP; ++p) xq[p] = zero;
#pragma unroll
            for (int p = 0; p < WP; ++p) wq[p] = zero;
        }
#pragma unroll
        for (int p = 0; p < XP; ++p) *reinterpret_cast<f32x4*>(&xs[buf][(p_row + 64 * p) * kStride + p_k]) = xq[p];
#pragma unroll
        for (int p = 0; p < WP; ++p) *reinterpret_cast<f32x4*>(&ws[buf][(p_row + 64 * p) * kStride + p_k]) = wq[p];
    };
    f32x4 acc[WM][WN], total[WM][WN];
#pragma unroll
    for (int jm = 0; jm < WM; ++jm)
#pragma unroll
        for (int jn = 0; jn < WN; ++jn) acc[jm][jn] = total[jm][jn] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto put = [&](float* to, const f32x4 (&value)[WM][WN]) {
#pragma unroll
        for (int jm = 0; jm < WM; ++jm) {
            const int m = m0 + wm0 + 32 * jm + i;
            if (m >= M) continue;
#pragma unroll
            for (int jn = 0; jn < WN; ++jn) {
                const int n = n0 + wn0 + 16 * jn + 4 * g;
                float* dst = to + static_cast<size_t>(m) * N + n;
                if (N % 4 == 0 && n + 3 < N) {
                    *reinterpret_cast<f32x4*>(dst) = value[jm][jn];
                } else {
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        if (n + v < N) dst[v] = value[jm][jn][v];
                }
            }
        }
    };
    constexpr int kChunksPerSegment = kF32Segment / kF32Chunk;
    const int all_chunks = (K + kF32Chunk - 1) / kF32Chunk;
    const int first = SPLIT ? blockIdx.z * per_group * kChunksPerSegment : 0;
    const int chunks = SPLIT ? min(all_chunks, first + per_group * kChunksPerSegment) : all_chunks;   // one past the last
    // chunk q: multiplied from tile q % 2 of shared memory; chunk q + 1 waits in the registers (q + 1) % 2
    // and goes to the other tile when the products of chunk q are issued; chunk q + 2 is asked for
    auto step = [&](int q, int buf, f32x4 (&x_next)[XP], f32x4 (&w_next)[WP], f32x4 (&x_ask)[XP], f32x4 (&w_ask)[WP]) {
        if (q + 2 < chunks) fetch(x_ask, w_ask, (q + 2) * kF32Chunk);
        f32x4 a[WN], b[WM];
#pragma unroll
        for (int jn = 0; jn < WN; ++jn) a[jn] = *reinterpret_cast<const f32x4*>(&ws[buf][(wn0 + 16 * jn + i) * kStride + 4 * g]);
#pragma unroll
        for (int jm = 0; jm < WM; ++jm) b[jm] = *reinterpret_cast<const f32x4*>(&xs[buf][(wm0 + 32 * jm + i) * kStride + 4 * g]);
        if (PART) {
#pragma unroll
            for (int jm = 0; jm < WM; ++jm) {
                if (jm >= live) break;
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int jn = 0; jn < WN; ++jn)
                        acc[jm][jn] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[jn][t], b[jm][t], acc[jm][jn], 0, 0, 0);
            }
        } else {
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int jm = 0; jm < WM; ++jm)
#pragma unroll
                    for (int jn = 0; jn < WN; ++jn)
                        acc[jm][jn] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[jn][t], b[jm][t], acc[jm][jn], 0, 0, 0);
        }
        if ((q + 1) % kChunksPerSegment == 0 || q + 1 == chunks) {
            // a segment ends: its sum joins the sums of the segments before it, or goes to its own place
            const bool alone = q < kChunksPerSegment;
            if (SPLIT) put(out + static_cast<size_t>(q / kChunksPerSegment) * M * N, acc);
#pragma unroll
            for (int jm = 0; jm < WM; ++jm)
#pragma unroll
                for (int jn = 0; jn < WN; ++jn) {
                    if (!SPLIT) total[jm][jn] = alone ? acc[jm][jn] : total[jm][jn] + acc[jm][jn];
                    acc[jm][jn] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
        }
        if (q + 1 < chunks) stage(buf ^ 1, x_next, w_next, (q + 1) * kF32Chunk);
        __syncthreads();
    };
    fetch(xr[0], wr[0], first * kF32Chunk);
    stage(0, xr[0], wr[0], first * kF32Chunk);
    if (first + 1 < chunks) fetch(xr[1], wr[1], (first + 1) * kF32Chunk);
    __syncthreads();
    for (int q = first; q < chunks; q += 2) {
        step(q, 0, xr[1], wr[1], xr[0], wr[0]);
        if (q + 1 < chunks) step(q + 1, 1, xr[0], wr[0], xr[1], wr[1]);
    }
    if (!SPLIT) put(out, total);
}

// out[i] = partial[0][i] + partial[1][i] + ... in ascending order of the segments; VEC consecutive elements a thread
// (four where the count and the addresses allow it), eight segments asked for before the first is added.
template <int VEC>
__global__ void __launch_bounds__(256)
gemm_segments_sum_kernel(const float* __restrict__ partial, float* __restrict__ out, long long count, int segments) {
    typedef float floats __attribute__((ext_vector_type(VEC)));
    const long long i = (static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x) * VEC;
    if (i >= count) return;
    floats total = *reinterpret_cast<const floats*>(partial + i);
    for (int s0 = 1; s0 < segments; s0 += 8) {
        floats t[8];
#pragma unroll
        for (int j = 0; j < 8; ++j)
            t[j] = *reinterpret_cast<const floats*>(partial + static_cast<size_t>(min(s0 + j, segments - 1)) * count + i);
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (s0 + j < segments) total = total + t[j];
    }
    *reinterpret_cast<floats*>(out + i) = total;
}

namespace {
// Whether the few-row kernel gives every segment of the K axis a wavefront of its own: where the bands
// of 16 columns alone are too few wavefronts to keep the memory busy.
bool few_rows_split(int N, int K) { return K > kF32Segment && (N + 15) / 16 < 1024; }
bool f32_by_matrix_cores(int in_bf16, int out_bf16, int K) { return !in_bf16 && !out_bf16 && K % 4 == 0 && K >= 4; }

int sum_segments(const float* partial, float* out, long long count, int segments, hipStream_t stream) {
    const bool fours = count % 4 == 0 && (reinterpret_cast<uintptr_t>(partial) | reinterpret_cast<uintptr_t>(out)) % 16 == 0;
    const int vec = fours ? 4 : 1;
    const long long blocks = (count / vec + 255) / 256;
    if (blocks > 0x7fffffffLL) return -1;
    if (vec == 4)
        gemm_segments_sum_kernel<4><<<static_cast<unsigned>(blocks), 256, 0, stream>>>(partial, out, count, segments);
    else
        gemm_segments_sum_kernel<1><<<static_cast<unsigned>(blocks), 256, 0, stream>>>(partial, out, count, segments);
    return launch_status();
}

// How a product of more than 64 rows is cut: tiles of 32 wm by 32 wn, and `per_group` segments of the K axis a
// workgroup (0: all of them, no partial sums).  Every choice gives the same bits, so the cheapest by this estimate
// is taken: a compute unit that holds two or more workgroups works off one's tile and segment in the first time
// below, one that holds a single workgroup in the second (measured, in us: 132, 117 and 110 TFLOP/s with all
// compute units full, 110, 92 and 75 with one workgroup each), and partial sums are written and read at
// 4 TB/s by a further launch.  333 rows, by the estimate against tiles chosen by their number alone:
// K 16,384 to 2,048 columns 596 to 260 us, 2,048 to 2,560 84 to 49, 2,048 to 2,048 80 to 42; 100 rows, 16,384 to
// 2,048: 596 to 94.
struct F32Cut {
    int wm, wn, per_group;
    bool part;                   // the last tile's blocks without rows are left out
};
constexpr long long kMostPartials = 64LL << 20;       // floats of partial sums a product may leave (256 MiB)

F32Cut f32_cut(int M, int N, int K, bool may_split) {
    constexpr struct { int wm, wn; float shared, alone, part; } kTiles[] = {
        {4, 4, 32.6f, 38.f, 1.02f}, {4, 2, 18.4f, 22.7f, 0.95f}, {2, 4, 18.4f, 22.7f, 0.95f}, {2, 2, 9.7f, 14.3f, 0.97f}};
    constexpr int kUnits = 256;
    const int segments = (K + kF32Segment - 1) / kF32Segment;
    F32Cut best{4, 4, 0, false};
    float least = 3.4e38f;
    // With all blocks first.  Then with the blocks left out that the last tiles have no rows for: these tiles cost 0.3 and 0.7 of what they have rows
    // for, and the branches make the others slower or faster (measured, `part`).  A launch is shorter for it only where the compute units get about the
    // same share of such tiles: where all are, two to a unit and more; where each unit has five and more; or two, one with all rows and one without (as
    // many columns of tiles as units: 140 rows of 2,048 keys to 32,768 columns 237 to 195 us).  Else it ends with the units that have none (2,048 keys,
    // two to a unit, 333 rows to 2,048 and 2,560 columns 38.7 and 46.6 to 47.7 and 49.1, 192 to 8,192 74 to 102; four to a unit, 400 rows of 16,384
    // keys to 2,048 294 to 322).  3% are left for what the estimate does not see (600 rows to 32,768 columns 689 to 716), 6% where other tiles in pieces
    // would take the place of the best without (192 rows of 16,384 keys to 2,560 173 to 197).  Tiles of 64 x 64 gain only where four and more share a unit.
    for (const bool part : {false, true}) {
        const F32Cut whole = best;
        for (const auto& t : kTiles) {
            const int row_tiles = (M + 32 * t.wm - 1) / (32 * t.wm), column_tiles = (N + 32 * t.wn - 1) / (32 * t.wn);
            const int in_last = (M - 1) % (32 * t.wm) / 32 + 1;
            if (part && in_last == t.wm) continue;
            const float shorter = t.part * (1.f - 0.7f * (t.wm - in_last) / t.wm / row_tiles);
            for (int per_group = segments; per_group >= 1; per_group = per_group == 1 ? 0 : (per_group + 1) / 2) {
                const int groups = (segments + per_group - 1) / per_group;
                const bool split = groups > 1;
                if (split && (!may_split || groups > 65535 || static_cast<long long>(segments) * M * N > kMostPartials)) break;
                const long long on_a_unit = (static_cast<long long>(row_tiles) * column_tiles * groups + kUnits - 1) / kUnits;
                float us = per_group * ((on_a_unit & ~1LL) * t.shared + (on_a_unit & 1) * t.alone);
                if (part) {
                    const bool evenly = row_tiles == 1 ? on_a_unit > 1 : on_a_unit > 4 || (on_a_unit == 2 && !split && column_tiles >= kUnits);
                    if (!evenly || (t.wm + t.wn == 4 && on_a_unit < 4)) continue;
                    const bool other = t.wm != whole.wm || t.wn != whole.wn || (split ? per_group : 0) != whole.per_group;
                    us *= shorter * (row_tiles == 1 ? 1.f : other && split ? 1.06f : 1.03f);
                }
                if (split) us += 4.f + 2e-6f * segments * M * N;
                if (us < least) {
                    least = us;
                    best = F32Cut{t.wm, t.wn, split ? per_group : 0, part};
                }
            }
        }
    }
    return best;
}
}  // namespace

// The tile-major copy of a float32 weight [N, K] (K a multiple of 4): for band b of 16 rows and chunk q
// of 16 keys, lane 16 g + i finds w[16 b + i][16 q + 4 g .. + 3] at ((b * chunks + q) * 64 + lane) * 4;
// rows beyond N and keys beyond K are zeros.
__global__ void __launch_bounds__(256)
tile_weight_f32_kernel(const float* __restrict__ w, float* __restrict__ tiles, int N, int K, int chunks, long long pieces) {
    const long long piece = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (piece >= pieces) return;
    const int lane = piece % 64, i = lane % 16, g = lane / 16;
    const long long tile = piece / 64;
    const int q = tile % chunks;
    const long long row = tile / chunks * 16 + i;
    const int k = 16 * q + 4 * g;
    f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
    if (row < N && k < K) v = *reinterpret_cast<const f32x4*>(w + row * K + k);
    *reinterpret_cast<f32x4*>(tiles + piece * 4) = v;
}

// Elements of the tile-major copy of a float32 weight [N, K].
WLLM_API long long wllm_tiled_size_f32(int N, int K) {
    return static_cast<long long>((N + 15) / 16) * 16 * ((K + kF32Chunk - 1) / kF32Chunk) * kF32Chunk;
}

WLLM_API int wllm_tile_weight_f32(const float* w, float* tiles, int N, int K, hipStream_t stream) {
    if (N < 1 || K < 4 || K % 4 != 0) return -1;
    const int chunks = (K + kF32Chunk - 1) / kF32Chunk;
    const long long pieces = static_cast<long long>((N + 15) / 16) * chunks * 64;
    const long long blocks = (pieces + 255) / 256;
    if (blocks > 0x7fffffffLL) return -1;
    tile_weight_f32_kernel<<<static_cast<unsigned>(blocks), 256, 0, stream>>>(w, tiles, N, K, chunks, pieces);
    return launch_status();
}

// Into how many partial sums [segments, M, N] a float32 product of these sizes is split (1: it is not).
// `wllm_gemm_generic` needs `partial` to hold them (at most 64 rows; with more rows it runs unsplit without); of at most
// 64 rows it leaves them there for a consumer that adds them in ascending order if `out` is null.
WLLM_API int wllm_gemm_f32_segments(int M, int N, int K) {
    if (M < 1 || N < 1 || K < 4 || K % 4 != 0) return 1;
    if (M <= 64 ? !few_rows_split(N, K) : f32_cut(M, N, K, true).per_group == 0) return 1;
    return (K + kF32Segment - 1) / kF32Segment;
}

// Whether the product of these sizes, of more than 64 rows, leaves out the blocks of 16 rows that its last tiles have no rows for.
WLLM_API int wllm_gemm_f32_leaves_out(int M, int N, int K) {
    return M > 64 && N > 0 && K >= 4 && K % 4 == 0 && f32_cut(M, N, K, true).part;
}

// `tiles`: null, or the tile-major copy of a float32 w (`wllm_tile_weight_f32`), which the few-row kernel
// streams faster; everything else reads w.
WLLM_API int wllm_gemm_generic(const void* x, const void* w, const void* tiles, int in_bf16, void* out, int out_bf16,
                               void* partial, int M, int N, int K, hipStream_t stream) {
    if (M < 1 || N < 1 || K < 1) return -1;
    if (f32_by_matrix_cores(in_bf16, out_bf16, K)) {
        const float* xf = static_cast<const float*>(x);
        const float* wf = static_cast<const float*>(w);
        const float* tf = static_cast<const float*>(tiles);
        float* of = static_cast<float*>(out);
        if (M <= 64) {
            const int bands = (N + 15) / 16, groups = (bands + 3) / 4;
            const int mt = (M + 15) / 16;
#define FEW_ROWS(SPLIT, GRID, DST)                                                                                      \
    do {                                                                                                                \
        if (tf) {                                                                                                       \
            if (mt == 1) gemm_f32_few_rows_kernel<SPLIT, true, 1><<<GRID, 256, 0, stream>>>(xf, tf, DST, M, N, K);       \
            else if (mt == 2) gemm_f32_few_rows_kernel<SPLIT, true, 2><<<GRID, 256, 0, stream>>>(xf, tf, DST, M, N, K);  \
            else if (mt == 3) gemm_f32_few_rows_kernel<SPLIT, true, 3><<<GRID, 256, 0, stream>>>(xf, tf, DST, M, N, K);  \
            else gemm_f32_few_rows_kernel<SPLIT, true, 4><<<GRID, 256, 0, stream>>>(xf, tf, DST, M, N, K);               \
        } else {                                                                                                        \
            if (mt == 1) gemm_f32_few_rows_kernel<SPLIT, false, 1><<<GRID, 256, 0, stream>>>(xf, wf, DST, M, N, K);      \
            else if (mt == 2) gemm_f32_few_rows_kernel<SPLIT, false, 2><<<GRID, 256, 0, stream>>>(xf, wf, DST, M, N, K); \
            else if (mt == 3) gemm_f32_few_rows_kernel<SPLIT, false, 3><<<GRID, 256, 0, stream>>>(xf, wf, DST, M, N, K); \
            else gemm_f32_few_rows_kernel<SPLIT, false, 4><<<GRID, 256, 0, stream>>>(xf, wf, DST, M, N, K);              \
        }                                                                                                               \
    } while (0)
            if (few_rows_split(N, K)) {
                const int segments = (K + kF32Segment - 1) / kF32Segment;
                if (!partial || segments > 65535) return -1;
                float* pf = static_cast<float*>(partial);
                FEW_ROWS(true, dim3(groups, segments), pf);
                if (int err = launch_status()) return err;
                if (of) return sum_segments(pf, of, static_cast<long long>(M) * N, segments, stream);
            } else {
                if (!of) return -1;
                FEW_ROWS(false, dim3(groups), of);
            }
#undef FEW_ROWS
            return launch_status();
        }
        if (!of) return -1;
        float* pf = static_cast<float*>(partial);
        const F32Cut cut = f32_cut(M, N, K, pf != nullptr);
        const int segments = (K + kF32Segment - 1) / kF32Segment;
        const dim3 grid((N + 32 * cut.wn - 1) / (32 * cut.wn), (M + 32 * cut.wm - 1) / (32 * cut.wm),
                        cut.per_group ? (segments + cut.per_group - 1) / cut.per_group : 1);
        if (grid.y > 65535) return -1;
#define TILES_P(WM, WN, PART)                                                                                                  \
    do {                                                                                                                        \
        if (cut.per_group) gemm_f32_tile_kernel<WM, WN, true, PART><<<grid, 256, 0, stream>>>(xf, wf, pf, M, N, K, cut.per_group); \
        else gemm_f32_tile_kernel<WM, WN, false, PART><<<grid, 256, 0, stream>>>(xf, wf, of, M, N, K, 0);                       \
    } while (0)
#define TILES(WM, WN)                           \
    do {                                        \
        if (cut.part) TILES_P(WM, WN, true);    \
        else TILES_P(WM, WN, false);            \
    } while (0)
        if (cut.wm == 4 && cut.wn == 4) TILES(4, 4);
        else if (cut.wm == 4) TILES(4, 2);
        else if (cut.wn == 4) TILES(2, 4);
        else TILES(2, 2);
#undef TILES
#undef TILES_P
        if (const int err = launch_status()) return err;
        return cut.per_group ? sum_segments(pf, of, static_cast<long long>(M) * N, segments, stream) : 0;
    }
    const dim3 grid((N + kTile - 1) / kTile, (M + kTile - 1) / kTile);
    if (grid.y > 65535) return -1;
#define LAUNCH(TI, TO)                                                                                  \
    gemm_nt_kernel<TI, TO><<<grid, 256, 0, stream>>>(static_cast<const TI*>(x), static_cast<const TI*>(w), \
                                                     static_cast<TO*>(out), M, N, K)
    if (in_bf16 && out_bf16) LAUNCH(bf16, bf16);
    else if (in_bf16) LAUNCH(bf16, float);
    else if (!out_bf16) LAUNCH(float, float);
    else return -1;
#undef LAUNCH
    return launch_status();
}
