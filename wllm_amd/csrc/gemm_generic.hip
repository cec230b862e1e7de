// out[M, N] = x[M, K] * w[N, K]^T for float32 and bfloat16 operands, accumulated in float32.  It is
// the product of the float32 path, and the product of last resort for bfloat16 (shapes the
// bfloat16 matrix-core kernels do not take, float32 results from bfloat16 operands).  float32 operands are multiplied and added with
// float32's precision: where the K axis is a multiple of 4 on the matrix cores, each number as the sum of three bfloat16 numbers (below), with fused
// multiply-adds on the vector units otherwise (this kernel).
//
// A workgroup of 256 threads makes a 64x64 tile of the result; the K axis is walked in steps of
// 16 through shared memory; a thread holds a 4x4 block.  The K axis is cut into segments of kSegment
// keys counted from 0, a segment is summed over k in ascending order of fused multiply-adds from
// zero, and the segments' sums are added in ascending order: an order fixed by K alone, so a row's
// result does not depend on the other rows of the batch.
#include "split_product.h"

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
// Every number as three of bfloat16, a product of two as six on the bfloat16 instruction (`split_product.h`), which runs at 16 times the
// rate of v_mfma_f32_16x16x4_f32.  us, that instruction and here: 333 rows of 2,048 keys to 32,768 columns 400 and 273, of 16,384 to 2,048 223 and 143, of 2,048 to
// 2,560 46 and 32; 100 rows 159 and 109, 80 and 51; 2,048 rows 2,100 and 1,500 (183 TFLOP/s), 1,103 and 792; 8 rows of 2,048 keys to 2,560 columns 10.7 and 7.8, to 32,768, where the weights
// are the bound, 49.4 and 48.6 (the logits' 256,000 columns 339 and 346).  What bounds many rows: the card's power (1.77 GHz at 2,048 rows, matrix cores busy
// 66% of the cycles); few rows: the weights.
//
// Both kernels below make an element of the
// result by the same instructions on the same numbers in the same order, whatever the rows and columns
// beside it, so a token's projection has the same bits in a decode step as inside a prompt:
//   the K axis is cut into segments of kF32Segment keys counted from 0; within a segment the keys go
//   in steps of 32; a step is six instructions, the smallest products first, that accumulate into the segment's sum, which starts at zero; the
//   segments' sums are added in ascending order.
// (Sums that are not finite are made again, over what a kernel has of the K axis.)
// A lane (i, g) of a wavefront holds, of a step's two chunks of 16 keys, w[n0 + i][16 q + 4 g .. + 3] and x[m0 + i][the same
// keys]: a 16-byte load each.  The first operand is
// w, so a lane's four results are four consecutive columns of one row of out.
typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int kF32Segment = 512;
constexpr int kF32Chunk = 16;
constexpr int kF32Step = 2 * kF32Chunk;

// At most 64 rows (the decode steps of the float32 path): the weights stream from memory straight
// into the lanes that multiply them, a wavefront a band of 16 columns, U chunks of it and of x on their way while the U before them are split and multiplied
// (one after the other a wavefront waited for both: 8 rows of 2,048 keys to 32,768 columns, two wavefronts a vector unit, 62 us); x comes through the
// caches (all wavefronts read the same few rows).  MT tiles of 16 rows: a
// fragment of the weights feeds MT products, each row's sums in the one order.  SPLIT: a wavefront takes
// one segment of the K axis (blockIdx.y) and leaves its sum in partial[segment]; a second kernel adds
// the segments in ascending order.  Otherwise it walks all segments and adds as it goes.
// TILED: w is the weight's tile-major copy (`tile_weight_f32_kernel`): per band of 16 rows and chunk
// of 16 keys one KiB in lane order, so that a wavefront's load is one contiguous KiB and its walk along
// K one contiguous run (with the float32 instruction gate and up at Gemma-2B sizes took 76 us from the row-major weight, whose loads
// touch 16 rows of 64 bytes each, 49 us from the copy).
template <bool SPLIT, bool TILED, int MT>
__global__ void __launch_bounds__(256)
gemm_f32_few_rows_kernel(const float* __restrict__ x, const float* __restrict__ w, float* __restrict__ out, int M, int N,
                         int K) {
    constexpr int U = 4, kBatch = U * kF32Chunk;
    static_assert(kF32Segment % (2 * kBatch) == 0, "a segment ends behind two batches");
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int i = lane % 16, g = lane / 16;
    const int n0 = (blockIdx.x * 4 + wave) * 16;
    if (n0 >= N) return;
    const int chunks_of_row = (K + kF32Chunk - 1) / kF32Chunk;
    const float* wrow = TILED ? w + (static_cast<size_t>(n0 / 16) * chunks_of_row * 64 + lane) * 4
                              : w + static_cast<size_t>(min(n0 + i, N - 1)) * K;
    // (rows beyond the last are the last again: nothing of theirs is written)
    const float* xrow[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) xrow[t] = x + static_cast<size_t>(min(16 * t + i, M - 1)) * K;
    const int begin = SPLIT ? blockIdx.y * kF32Segment : 0, end = SPLIT ? min(K, begin + kF32Segment) : K;
    const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
    f32x4 total[MT], acc[MT], a[2][U], b[2][MT][U];
#pragma unroll
    for (int t = 0; t < MT; ++t) total[t] = acc[t] = zero;
    auto fetch = [&](f32x4 (&aq)[U], f32x4 (&bq)[MT][U], int k0) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            // every lane loads, from a clamped address; what lies beyond the K axis becomes zero when it is split
            const int k = min(k0 + u * kF32Chunk + 4 * g, K - 4);
            aq[u] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(
                TILED ? wrow + static_cast<size_t>(min(k0 / kF32Chunk + u, chunks_of_row - 1)) * 256 : wrow + k));
#pragma unroll
            for (int t = 0; t < MT; ++t) bq[t][u] = *reinterpret_cast<const f32x4*>(xrow[t] + k);
        }
    };
    auto multiply = [&](f32x4 (&aq)[U], f32x4 (&bq)[MT][U], int k0) {
#pragma unroll
        for (int u = 0; u < U; u += 2) {
            const int k = k0 + u * kF32Chunk;
            if (k >= end) break;                        // the same for all lanes
            if (k + kF32Step > K) {
                if (k + 4 * g >= K) aq[u] = zero;
                if (k + kF32Chunk + 4 * g >= K) aq[u + 1] = zero;
            }
            SplitFragment wf, xf;
            split_eight(aq[u], aq[u + 1], wf);
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                split_eight(bq[t][u], bq[t][u + 1], xf);
#pragma unroll
                for (int p = 0; p < kSplitProducts; ++p) acc[t] = split_product(wf, xf, acc[t], p);
            }
        }
    };
    // (behind the last batch the last one again, which the caches have: a branch would make the products wait)
    const int last = begin + (end - 1 - begin) / kBatch * kBatch;
    fetch(a[0], b[0], begin);
    for (int k0 = begin; k0 < end; k0 += 2 * kBatch) {
        fetch(a[1], b[1], min(k0 + kBatch, last));
        multiply(a[0], b[0], k0);
        fetch(a[0], b[0], min(k0 + 2 * kBatch, last));
        multiply(a[1], b[1], k0 + kBatch);
        if ((k0 + 2 * kBatch) % kF32Segment == 0 || k0 + 2 * kBatch >= end) {
            const bool alone = SPLIT || k0 < kF32Segment;
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                total[t] = alone ? acc[t] : total[t] + acc[t];
                acc[t] = zero;
            }
        }
    }
    // lane (i, g) holds out[row 16 t + i][n0 + 4 g .. + 3]
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        if (16 * t + i >= M) continue;
        float* dst = out + (SPLIT ? static_cast<size_t>(blockIdx.y) * M * N : 0) + static_cast<size_t>(16 * t + i) * N + n0 + 4 * g;
        if (N % 4 == 0 && n0 + 4 * g + 3 < N) {
            *reinterpret_cast<f32x4*>(dst) = total[t];
        } else {
#pragma unroll
            for (int v = 0; v < 4; ++v)
                if (n0 + 4 * g + v < N) dst[v] = total[t][v];
        }
        if (finite_probe(total[t]) != 0.f) {
#pragma unroll 1
            for (int v = 0; v < 4; ++v)
                if (n0 + 4 * g + v < N && !__builtin_isfinite(dst[v]))
                    dst[v] = plain_product<TILED>(xrow[t], w, n0 + 4 * g + v, K, chunks_of_row, begin, end, kF32Segment);
        }
    }
}

// More rows: a tile of a workgroup of four wavefronts is 16 MB rows by 64 NB columns, each wavefront all rows by 16 NB columns.  A wavefront takes its rows of w
// straight into the lanes that multiply them and splits them there, each number once; x is split on its way to shared memory, once a workgroup, in
// three planes of 64 bytes a row and step: chunk g (the keys of lanes (., g)) of row r lies at place (4 (r % 2) + g) ^ (r / 2 % 4) of the 128 bytes of two rows, so that eight
// rows' reads meet no bank twice.
// While a wavefront multiplies a step it splits the next one's numbers, a few vector instructions behind each product, and asks for those of the step after it into the registers that
// these leave.
// SPLIT: a workgroup (blockIdx.z) takes `per_group` segments of the K axis and leaves each one's sum in
// out[segment]; the kernel below adds them in the order in which the unsplit walk does.
// (w is read row by row: its tile-major copy is no faster here, 333 rows of 2,048 keys to 32,768 columns 280 us from it and 262 from the rows.)
constexpr int f32_plane(int mb) { return (mb + 1) / 2 * 32 * 64; }       // bytes of a plane of x: whole pieces a thread

template <int MB, int NB, bool SPLIT>
static __device__ __forceinline__ void f32_tile(unsigned char (*planes_s)[3][f32_plane(MB)], const float* __restrict__ x, const float* __restrict__ w,
                                                float* __restrict__ out, int M, int N, int K, int per_group, int m0) {
    constexpr int TN = 64 * NB;
    constexpr int XP = (MB + 1) / 2;                          // 16-byte pieces of a step's x per thread
    const int tid = threadIdx.x, lane = tid % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int i = lane % 16, g = lane / 16;
    const int n0 = blockIdx.x * TN + wave * 16 * NB;
    // a thread's pieces of x: row tid / 8 (+ 32 per further piece), keys 4 (tid % 8) .., from the tile's first row
    const int p_row = tid / 8, p_k = tid % 8 * 4;
    auto place = [](int row, int chunk) { return row / 2 * 128 + (((row % 2) * 4 + chunk) ^ (row / 2 % 4)) * 16; };
    const float* xbase = x + static_cast<size_t>(m0) * K;
    uint32_t xoff[XP];
#pragma unroll
    for (int p = 0; p < XP; ++p) xoff[p] = static_cast<uint32_t>(min(p_row + 32 * p, M - 1 - m0)) * K;
    // this wavefront's bands of w (beyond the last one: the last one again), and in them this lane's place
    const int first_band = min(n0 / 16, (N - 1) / 16);
    const float* wbase = w + static_cast<size_t>(first_band) * 16 * K;
    uint32_t woff[NB];
#pragma unroll
    for (int a = 0; a < NB; ++a)
        woff[a] = static_cast<uint32_t>(min(n0 + 16 * a + i, N - 1) - first_band * 16) * K;
    // The numbers of a step that this lane splits, four at a time: 2 NB of w (band q / 2, chunk q % 2 of 16 keys), then XP of x.
    constexpr int kQuads = 2 * NB + XP;
    f32x4 raw[kQuads];
    auto fetch = [&](int q, int s) {
        const float* from = q < 2 * NB ? wbase + woff[q / 2 % NB] + static_cast<uint32_t>(min(s * kF32Step + 16 * (q % 2) + 4 * g, K - 4))
                                       : xbase + xoff[q < 2 * NB ? 0 : q - 2 * NB] + static_cast<uint32_t>(min(s * kF32Step + p_k, K - 4));
        raw[q] = *reinterpret_cast<const f32x4*>(from);
    };
    const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
    SplitFragment fw[2][NB];
    const int write0 = place(p_row, tid % 4) + tid / 4 % 2 * 8;          // (32 rows are 2,048 bytes)
    // Quad q of step s into the fragments `to` or the buffer `buf`.  What lies beyond the K axis: w's numbers become zero, x's are then any
    // (where they are not finite, the sums are made again).
    auto split_quad = [&](int q, int s, SplitFragment (&to)[NB], int buf) {
        uint32_t words[3][2];
        f32x4 v = raw[q];
        if (q < 2 * NB && s * kF32Step + 16 * (q % 2) + 4 * g >= K) v = zero;
        split_numbers(v[0], v[1], words[0][0], words[1][0], words[2][0]);
        split_numbers(v[2], v[3], words[0][1], words[1][1], words[2][1]);
        // (made here, between this step's products: the compiler would move what only the next step uses there)
        if (q < 2 * NB)
            asm volatile("" : "+v"(words[0][0]), "+v"(words[0][1]), "+v"(words[1][0]), "+v"(words[1][1]), "+v"(words[2][0]), "+v"(words[2][1]));
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            if (q >= 2 * NB) {
                *reinterpret_cast<uint2*>(&planes_s[buf][r][write0 + (q - 2 * NB) * 2048]) = make_uint2(words[r][0], words[r][1]);
            } else if (q % 2 == 0) {
                to[q / 2 % NB].part[r].u.x = words[r][0];
                to[q / 2 % NB].part[r].u.y = words[r][1];
            } else {
                to[q / 2 % NB].part[r].u.z = words[r][0];
                to[q / 2 % NB].part[r].u.w = words[r][1];
            }
        }
    };
    f32x4 acc[MB][NB];
    float probe = 0.f;
#pragma unroll
    for (int b = 0; b < MB; ++b)
#pragma unroll
        for (int a = 0; a < NB; ++a) acc[b][a] = zero;
    // a segment's sums to `to`, or (add) to those that this lane put there before
    auto put = [&](float* to, bool add) __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < MB; ++b) {
            const int m = m0 + 16 * b + i;
            if (m >= M) continue;
#pragma unroll
            for (int a = 0; a < NB; ++a) {
                const int n = n0 + 16 * a + 4 * g;
                float* dst = to + static_cast<size_t>(m) * N + n;
                if (N % 4 == 0 && n < N) {
                    f32x4 v = acc[b][a];
                    if (add) v = *reinterpret_cast<const f32x4*>(dst) + v;
                    *reinterpret_cast<f32x4*>(dst) = v;
                } else {
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        if (n + v < N) dst[v] = add ? dst[v] + acc[b][a][v] : acc[b][a][v];
                }
            }
        }
    };
    constexpr int kStepsPerSegment = kF32Segment / kF32Step;
    const int all_steps = (K + kF32Step - 1) / kF32Step;
    const int first = SPLIT ? blockIdx.z * per_group * kStepsPerSegment : 0;
    const int steps = SPLIT ? min(all_steps, first + per_group * kStepsPerSegment) : all_steps;   // one past the last
    const int read0 = place(i, g);                  // (16 rows are 1,024 bytes)
    SplitFragment fx[2];
    auto read_part = [&](int buf, int b, int r) { fx[b % 2].part[r].u = *reinterpret_cast<const uint4*>(&planes_s[buf][r][read0 + b * 1024]); };
    // step s: its x lies in buffer s % 2 and its w, split, in fw[F]; behind the last step what is split and staged is the last step's again and nothing uses it
    auto step = [&](auto set, int s, int buf) __attribute__((always_inline)) {
        constexpr int F = decltype(set)::value ? 1 : 0;
        const int next = min(s + 1, steps - 1), after = min(s + 2, steps - 1);
#pragma unroll
        for (int r = 0; r < 3; ++r) read_part(buf, 0, r);
#pragma unroll
        for (int b = 0; b < MB; ++b) {
            if (b + 1 < MB)
#pragma unroll
                for (int r = 0; r < 3; ++r) read_part(buf, b + 1, r);
#pragma unroll
            for (int q = b * kQuads / MB; q < (b + 1) * kQuads / MB; ++q) {
                split_quad(q, next, fw[1 - F], buf ^ 1);
                fetch(q, after);
            }
#pragma unroll
            for (int p = 0; p < kSplitProducts; ++p)
#pragma unroll
                for (int a = 0; a < NB; ++a) acc[b][a] = split_product(fw[F][a], fx[b % 2], acc[b][a], p);
            // the reads first, then some of the splitting between two products
            if (b == 0) __builtin_amdgcn_sched_group_barrier(0x100, 6, 0);
            else __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
#pragma unroll
            for (int q = 0; q < kSplitProducts * NB; ++q) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if (NB == 1) __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
                else __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        wait_reads();                   // (and writes)
        meet();
        if ((s + 1) % kStepsPerSegment == 0 || s + 1 == steps) {
            // a segment ends: its sum joins the sums of the segments before it, or goes to its own place
            float* to = out + (SPLIT ? static_cast<size_t>(s / kStepsPerSegment) * M * N : 0);
            put(to, !SPLIT && s >= kStepsPerSegment);
#pragma unroll
            for (int b = 0; b < MB; ++b)
#pragma unroll
                for (int a = 0; a < NB; ++a) {
                    probe += finite_probe(acc[b][a]);
                    acc[b][a] = zero;
                }
        }
    };
#pragma unroll
    for (int q = 0; q < kQuads; ++q) fetch(q, first);
#pragma unroll
    for (int q = 0; q < kQuads; ++q) {
        split_quad(q, first, fw[0], 0);
        fetch(q, min(first + 1, steps - 1));
    }
    __syncthreads();
    for (int s = first; s < steps; s += 2) {
        step(Flag<false>(), s, 0);
        if (s + 1 < steps) step(Flag<true>(), s + 1, 1);
    }
    if (probe != 0.f) {
        // some of this lane's sums are not finite
        const int segments = SPLIT ? (steps - first + kStepsPerSegment - 1) / kStepsPerSegment : 1;
#pragma unroll 1
        for (int e = 0; e < segments * MB * NB * 4; ++e) {
            const int segment = SPLIT ? first / kStepsPerSegment + e / (MB * NB * 4) : 0;
            const int m = m0 + e / (NB * 4) % MB * 16 + i, n = n0 + e / 4 % NB * 16 + 4 * g + e % 4;
            if (m >= M || n >= N) continue;
            float* here = out + (static_cast<size_t>(segment) * M + m) * N + n;
            if (!__builtin_isfinite(*here))
                *here = plain_product<false>(x + static_cast<size_t>(m) * K, w, n, K, 0, segment * kF32Segment,
                                             SPLIT ? min(K, (segment + 1) * kF32Segment) : K, kF32Segment);
        }
    }
}

// The first `high` tiles have MB blocks of 16 rows, the others one less, so that rows of any number fill their tiles.
template <int MB, int NB, bool SPLIT>
__global__ void __launch_bounds__(256, 2)
gemm_f32_tile_kernel(const float* __restrict__ x, const float* __restrict__ w, float* __restrict__ out, int M, int N, int K,
                     int per_group, int high) {
    __shared__ __align__(16) unsigned char planes_s[2][3][f32_plane(MB)];
    const int tile = blockIdx.y, m0 = 16 * (tile * MB - max(0, tile - high));
    if (tile < high) f32_tile<MB, NB, SPLIT>(planes_s, x, w, out, M, N, K, per_group, m0);
    else f32_tile<MB - 1, NB, SPLIT>(reinterpret_cast<unsigned char (*)[3][f32_plane(MB - 1)]>(planes_s), x, w, out, M, N, K, per_group, m0);
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

// How a product of more than 64 rows is cut: tiles of `mb` blocks of 16 rows by 64 nb columns, and `per_group` segments of the K axis a
// workgroup (0: all of them, no partial sums).  Every choice gives the same bits, so the cheapest by this estimate
// is taken: a compute unit that holds two or more workgroups works off one's tile and segment in the first time
// below, one that holds a single workgroup in the second (us, measured), and partial sums are written and read at
// 4 TB/s by a further launch.  Heights by the rows (`part`) where there are enough workgroups that a launch gets shorter by it: 333 rows to 32,768 columns in tiles of 8
// and of 7 blocks 285 and 262 us, 140 rows in 8 and 5 165 and 138; with a workgroup or two a compute unit a launch is as long as its longest (2,048 keys, 333 rows to 2,048
// and 192 to 8,192 columns 27.0 and 44.7 to 26.1 and 43.9; 400 rows of 4,096 keys to 2,048 43.6 to 42.5), which leaves them to whole tiles.
struct F32Cut {
    int mb, nb, per_group, row_tiles, high;
    bool part;                   // tiles' heights by the rows: the first `high` have mb blocks of 16 rows, the others one less, and no block is without rows
};
constexpr long long kMostPartials = 64LL << 20;       // floats of partial sums a product may leave (256 MiB)

F32Cut f32_cut(int M, int N, int K, bool may_split) {
    constexpr struct { int mb, nb; float shared, alone; } kTiles[] = {{8, 2, 22.0f, 25.5f}, {8, 1, 13.0f, 17.2f}, {4, 2, 13.4f, 17.2f}, {4, 1, 7.6f, 11.0f}};
    constexpr int kUnits = 256;
    const int segments = (K + kF32Segment - 1) / kF32Segment, blocks = (M + 15) / 16;
    F32Cut best{8, 2, 0, (blocks + 7) / 8, (blocks + 7) / 8, false};
    float least = 3.4e38f;
    for (const bool part : {false, true}) {
        const F32Cut whole = best;
        for (const auto& t : kTiles) {
            const int row_tiles = (blocks + t.mb - 1) / t.mb, column_tiles = (N + 64 * t.nb - 1) / (64 * t.nb);
            const int mb = part ? (blocks + row_tiles - 1) / row_tiles : t.mb;
            const int high = part ? blocks - row_tiles * (mb - 1) : row_tiles;
            if (part && mb == t.mb && high == row_tiles) continue;
            const float height = part ? 0.18f + 0.82f * blocks / (row_tiles * t.mb) : 1.f;
            for (int per_group = segments; per_group >= 1; per_group = per_group == 1 ? 0 : (per_group + 1) / 2) {
                const int groups = (segments + per_group - 1) / per_group;
                const bool split = groups > 1;
                if (split && (!may_split || groups > 65535 || static_cast<long long>(segments) * M * N > kMostPartials)) break;
                const long long on_a_unit = (static_cast<long long>(row_tiles) * column_tiles * groups + kUnits - 1) / kUnits;
                float us = per_group * ((on_a_unit & ~1LL) * t.shared + (on_a_unit & 1) * t.alone) * height;
                if (part) {
                    const bool evenly = row_tiles == 1 ? on_a_unit > 1 : on_a_unit > 4 || (on_a_unit >= 2 && !split && column_tiles >= kUnits);
                    if (!evenly || (t.mb + 4 * (t.nb - 1) == 4 && on_a_unit < 4)) continue;
                    const bool other = t.mb != whole.mb || t.nb != whole.nb || (split ? per_group : 0) != whole.per_group;
                    us *= row_tiles == 1 ? 1.f : other && split ? 1.06f : 1.03f;
                }
                if (split) us += 4.f + 2e-6f * segments * M * N;
                if (us < least) {
                    least = us;
                    best = F32Cut{mb, t.nb, split ? per_group : 0, row_tiles, high, part};
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
        const dim3 grid((N + 64 * cut.nb - 1) / (64 * cut.nb), cut.row_tiles,
                        cut.per_group ? (segments + cut.per_group - 1) / cut.per_group : 1);
        if (grid.y > 65535) return -1;
#define TILES(MB)                                                                                                             \
    case MB:                                                                                                                  \
        if (cut.nb == 2 && cut.per_group) gemm_f32_tile_kernel<MB, 2, true><<<grid, 256, 0, stream>>>(xf, wf, pf, M, N, K, cut.per_group, cut.high);  \
        else if (cut.nb == 2) gemm_f32_tile_kernel<MB, 2, false><<<grid, 256, 0, stream>>>(xf, wf, of, M, N, K, 0, cut.high);           \
        else if (cut.per_group) gemm_f32_tile_kernel<MB, 1, true><<<grid, 256, 0, stream>>>(xf, wf, pf, M, N, K, cut.per_group, cut.high); \
        else gemm_f32_tile_kernel<MB, 1, false><<<grid, 256, 0, stream>>>(xf, wf, of, M, N, K, 0, cut.high);                            \
        break;
        switch (cut.mb) {
            TILES(3) TILES(4) TILES(5) TILES(6) TILES(7) TILES(8)
            default: return -1;
        }
#undef TILES
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
