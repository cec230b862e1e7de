// out[M, N] = x[M, K] . w[N, K]^T for bfloat16 with many rows (prompts), on the matrix cores, and the gated
// form out[M, I] = act(x . Wg^T) * (x . Wu^T) with w = [Wg; Wu], whose activation and product are made in
// the registers the sums are in, so that only [M, I] is written.
//
// A workgroup of eight wavefronts makes tiles of 256 rows of x by 256 rows of w (gated: 128 gate rows and the 128 up rows that
// belong to them, so that a lane holds a column's gate and up sums), as `wide_tile.h` says.
//
// A launch has at most a workgroup a compute unit; each takes items (tile, piece of the K axis) one after
// the other, and sends the first stages of its next item before it writes the results of the last.  The items
// go to the XCDs in equal runs of an order in which 8 tiles of x rows share a tile of w rows, so that the 32
// items that an XCD has under way read 8 tiles of x and 4 of w.
//
// What bounds it: the card's power.  With numbers as models have them 4,096^3 runs at 1.45 PFLOP/s and 8,192^3 at 1.54 (the
// library: 1.49 and 1.60), with zeros at 2.0, where a slot of 512 cycles of products takes 640 with its barrier.  2,048 rows
// by 2 x 16,384 columns of 2,048 keys with the activation: 211 us, against 193 for the library's product that
// writes both streams and 41 for the pass that reads them; 16,384 keys to 2,048 columns in four pieces: 97 us against
// 133, as the library's tiles for 2,048 columns are no more than 128 rows and columns.  Slots of 16 products
// (a quarter each) took 1.24 PFLOP/s at 8,192^3, a workgroup an item 237 us for the gated product, a barrier before the
// last 2 to 8 products of a slot the same to 5% more.
//
// `splits` > 1 leaves float32 partial sums [splits, M, N], for the consumer to add in order.  Every output element
// is summed over k in ascending order within a piece; pieces depend on K and `splits` alone.
#include "wide_tile.h"

struct WideItem {
    int m_base, n_base, piece;
};

// GATED: 0 plain, 1 + the gate's number for the gated product.  N is the number of rows of w (plain) or of gate rows
// (gated); `stride` elements from a row of `out` to the next.  `vectors`: rows of `out` begin at multiples of 16 bytes.
template <int GATED>
__global__ void __launch_bounds__(512, 2)
gemm_wide_kernel(const bf16* __restrict__ x, const bf16* __restrict__ w, bf16* __restrict__ out, float* __restrict__ partial,
                 int M, int N, int K, int stride, bool vectors, int m_tiles, int n_tiles, int splits, GateShape shape) {
    constexpr int kColumns = GATED ? kWideHalf : kWideRows;         // output columns a tile
    constexpr bool kPair = GATED == kGatePairSquaredRelu + 1;
    extern __shared__ __align__(16) unsigned char tiles_s[];
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int i = lane % 16, g = lane / 16;
    const int wm = wave / 4, wn = wave % 4;

    const int tiles = m_tiles * n_tiles, items = tiles * splits, all_stages = K / kWideKeys;
    const int xcd = blockIdx.x % 8, per_xcd = items / 8, left = items % 8;
    const int first = xcd * per_xcd + min(xcd, left), end = first + per_xcd + (xcd < left ? 1 : 0);
    if (first + static_cast<int>(blockIdx.x) / 8 >= end) return;

    auto place = [&](int it, WideSource& from) {
        WideItem at;
        at.piece = it / tiles;
        const int t = it - at.piece * tiles;
        const int band = t / (8 * n_tiles), in_band = t - band * 8 * n_tiles;
        const int band_rows = min(8, m_tiles - 8 * band);
        const int n_tile = in_band / band_rows;
        at.m_base = (8 * band + in_band - n_tile * band_rows) * kWideRows;
        at.n_base = n_tile * kColumns;
        const int begin = static_cast<int>(static_cast<long long>(at.piece) * all_stages / splits);
        from.stages = static_cast<int>(static_cast<long long>(at.piece + 1) * all_stages / splits) - begin;
        from.two = true;
        from.x_bytes = reinterpret_cast<const unsigned char*>(x) + static_cast<size_t>(begin) * (kWideKeys * 2);
        from.w_bytes = reinterpret_cast<const unsigned char*>(w) + static_cast<size_t>(begin) * (kWideKeys * 2);
#pragma unroll
        for (int h = 0; h < 4; ++h)
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int r = wide_row(u);
                size_t row;
                if (h < 2) row = min(at.m_base + kWideHalf * h + r, M - 1);
                else if (GATED) row = static_cast<size_t>(min(at.n_base + r, N - 1)) + (h == 3 ? N : 0);
                else row = min(at.n_base + kWideHalf * (h - 2) + r, N - 1);
                from.offset[h][u] = static_cast<uint32_t>((row * K + wide_chunk() * 8) * 2);
            }
        return at;
    };
    // lane (i, g) holds, of quarter (xh, wh) and tile (a, b), output row 16 b + i and columns 4g .. 4g + 3
    auto finish = [&](const WideItem& at, const WideSums& acc) {
#pragma unroll
        for (int xh = 0; xh < 2; ++xh)
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const int m = at.m_base + xh * kWideHalf + wm * 64 + 16 * b + i;
                if (m >= M) continue;
                if (!GATED && partial != nullptr) {
                    float* row = partial + (static_cast<size_t>(at.piece) * M + m) * N;
#pragma unroll
                    for (int wh = 0; wh < 2; ++wh)
#pragma unroll
                        for (int a = 0; a < 2; ++a) {
                            const int n = at.n_base + wh * kWideHalf + wn * 32 + 16 * a + 4 * g;
                            if (n + 3 < N && N % 4 == 0) {
                                *reinterpret_cast<float4_t*>(row + n) = acc[xh][wh][a][b];
                            } else {
#pragma unroll
                                for (int v = 0; v < 4; ++v)
                                    if (n + v < N) row[n + v] = acc[xh][wh][a][b][v];
                            }
                        }
                    continue;
                }
                bf16* row = out + static_cast<size_t>(m) * stride;
#pragma unroll
                for (int wh = 0; wh < (GATED && !kPair ? 1 : 2); ++wh) {
                    uint32_t q[2][2];               // [16 columns][pair]
#pragma unroll
                    for (int a = 0; a < 2; ++a) {
                        float r[4];
#pragma unroll
                        for (int v = 0; v < 4; ++v) {
                            const float own = acc[xh][wh][a][b][v];
                            if (kPair) r[v] = squared_relu(own);
                            else if (GATED) r[v] = gate_product_fast<(GATED > 0 && !kPair ? GATED - 1 : 0)>(own, acc[xh][1][a][b][v], shape);
                            else r[v] = own;
                        }
                        q[a][0] = pack2_bf16(r[0], r[1]);
                        q[a][1] = pack2_bf16(r[2], r[3]);
                    }
                    const uint4 columns = wide_eight_columns(q);
                    const int n = at.n_base + (GATED ? 0 : wh * kWideHalf) + wn * 32 + 16 * (g & 1) + 8 * (g >> 1);
                    bf16* to = row + (kPair && wh == 1 ? N : 0) + n;
                    const uint32_t words[4] = {columns.x, columns.y, columns.z, columns.w};
                    if (vectors && n + 7 < N) {
                        *reinterpret_cast<uint4*>(to) = columns;
                    } else {
#pragma unroll
                        for (int v = 0; v < 8; ++v)
                            if (n + v < N) to[v] = bf16{static_cast<uint16_t>(words[v / 2] >> (16 * (v % 2)))};
                    }
                }
            }
    };
    wide_products<false>(tiles_s, first + blockIdx.x / 8, end, gridDim.x / 8, place, finish);
}

// out[M, N] = x . w^T (gated 0, w [N, K]), or the gated product (gated = 1 + the gate's number, with limit, slope and
// shift for the clamped swish; w [2N, K], gate rows first; with the paired squared relu out [M, 2N] = relu(x . w^T)^2);
// `stride` elements from a row of `out` to the next.  splits > 1 (plain only): `out` is null and `partial` float32
// [splits, M, N] takes the pieces' sums.  K must be a multiple of 64 and at least 64 * splits, x and w begin at
// multiples of 16 bytes and be smaller than 4 GiB.  Returns 0, a HIP error code, or -1 for what it does not take.
WLLM_API int wllm_gemm_wide(const void* x, const void* w, void* out, float* partial, int M, int N, int K, int stride, int splits,
                            int gated, float limit, float slope, float shift, hipStream_t stream) {
    if (M < 1 || N < 1 || K < kWideKeys || K % kWideKeys != 0 || splits < 1 || splits > K / kWideKeys || gated < 0 ||
        gated > kPairedGates)
        return -1;
    if ((splits > 1) != (partial != nullptr) || (splits > 1) != (out == nullptr) || (splits > 1 && gated != 0)) return -1;
    const bool pair = gated == kGatePairSquaredRelu + 1;
    if (out != nullptr && stride < (pair ? 2LL * N : N)) return -1;
    const size_t w_rows = static_cast<size_t>(gated ? 2 : 1) * N;
    if (w_rows * K * 2 >= (size_t(1) << 32) || static_cast<size_t>(M) * K * 2 >= (size_t(1) << 32)) return -1;
    if (reinterpret_cast<uintptr_t>(x) % 16 != 0 || reinterpret_cast<uintptr_t>(w) % 16 != 0 ||
        reinterpret_cast<uintptr_t>(partial) % 16 != 0)
        return -1;
    const bool vectors = reinterpret_cast<uintptr_t>(out) % 16 == 0 && stride % 8 == 0 && (!pair || N % 8 == 0);
    const int m_tiles = (M + kWideRows - 1) / kWideRows;
    const int columns = gated ? kWideHalf : kWideRows;
    const int n_tiles = (N + columns - 1) / columns;
    const long long items = static_cast<long long>(m_tiles) * n_tiles * splits;
    if (items > 0x3fffffffLL) return -1;
    static int compute_units = 0;
    if (compute_units == 0) {
        int device = 0;
        if (hipGetDevice(&device) != hipSuccess ||
            hipDeviceGetAttribute(&compute_units, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess)
            return launch_status();
    }
    // a multiple of 8, so that a workgroup's items stay in its XCD's run (an XCD of fewer items has idle workgroups)
    const int most = compute_units / 8 * 8 > 0 ? compute_units / 8 * 8 : 8;
    const int grid = items < most ? static_cast<int>((items + 7) / 8 * 8) : most;
    const bf16* xp = static_cast<const bf16*>(x);
    const bf16* wp = static_cast<const bf16*>(w);
    bf16* op = static_cast<bf16*>(out);
    const GateShape shape{limit, slope, shift};
#define LAUNCH(GATED)                                                                                               \
    do {                                                                                                            \
        static bool roomy = false;     /* more than 64 KiB of shared memory must be asked for once */              \
        if (!roomy) {                                                                                               \
            if (hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_wide_kernel<GATED>),                        \
                                    hipFuncAttributeMaxDynamicSharedMemorySize, kWideShared) != hipSuccess)         \
                return launch_status();                                                                             \
            roomy = true;                                                                                           \
        }                                                                                                           \
        gemm_wide_kernel<GATED><<<grid, 512, kWideShared, stream>>>(xp, wp, op, partial, M, N, K, stride, vectors,  \
                                                                    m_tiles, n_tiles, splits, shape);               \
    } while (0)
    if (gated == 0) { LAUNCH(0); }
    else { WLLM_BY_PAIRED_GATE(gated - 1, LAUNCH(GATE + 1)) }
#undef LAUNCH
    return launch_status();
}
