// out[M, N] = x[M, K] . w[N, K]^T for bfloat16 with many rows (prompts), on the matrix cores, and the gated
// form out[M, I] = act(x . Wg^T) * (x . Wu^T) with w = [Wg; Wu], whose activation and product are made in
// the registers the sums are in, so that only [M, I] is written.
//
// A workgroup of eight wavefronts makes a tile of 256 rows of x by 256 rows of w (gated: 128 gate rows and
// the 128 up rows that belong to them).  The tile is two halves of 128 rows of x by two halves of 128 rows
// of w; wavefront (wm, wn) of the 2 x 4 makes, of each of the four quarters, the 64 x 32 at (64 wm, 32 wn),
// as products v_mfma_f32_16x16x32_bf16 (w is the A operand, x the B operand: lane (i, g) ends with four
// consecutive columns of one output row).  In the gated form a lane so holds a column's gate and up sums.
//
// The K axis is walked in stages of 64 keys, two stages of 64 KB in shared memory.  A stage's halves (16 KB
// each) go there straight from memory (global_load_lds_dwordx4, 8 rows of 8 chunks of 16 bytes a load;
// chunk c of row r lies at place c ^ (r % 8) of its row, so that the reads of a fragment meet no bank
// twice).  The two wavefronts of a vector unit (wave and wave + 4) work half a step apart: while one reads
// fragments and sends loads, the other has the matrix cores for 32 products.  The step of one stage:
//   A  read both w halves and the first x half; send the second x half of the next stage
//   B  32 products (first x half)
//   C  read the second x half; send the first x half and both w halves of the stage after the next
//   D  32 products (second x half)
// with a barrier after each; the second group of wavefronts is one barrier behind the first.  Why the
// buffers are safe: a half is sent over only after a barrier that follows the last read of it by either group
// (each waits for its reads before the barrier that ends A and C), and it is read only after a barrier that
// follows both groups' wait for their loads of it: in front of a read at most 8 newer loads a lane may be
// on their way (vmcnt counts in order), which is what the order of sending leaves.  A load has about
// a stage and a half to arrive.
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
#include "common.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));

constexpr int kWideRows = 256;                       // rows of x, and rows of w, a tile
constexpr int kWideHalf = kWideRows / 2;
constexpr int kWideKeys = 64;                        // keys a stage
constexpr int kHalfBytes = kWideHalf * kWideKeys * 2;
constexpr int kWideStage = 4 * kHalfBytes;           // x halves, w halves
constexpr int kWideShared = 2 * kWideStage;

union WFrag {
    uint4 u;
    bf16x8_t v;
};

// 16 bytes a lane from base + offset into shared memory at `lds_address` + 16 * lane.  M0 is put back as it
// was: naming it as clobbered instead makes the compiler wait for every load in flight before the
// next read of shared memory.  The compiler does not see these loads; the kernel waits for them itself.
static __device__ __forceinline__ void load_to_shared(const void* base, uint32_t offset, uint32_t lds_address) {
    uint32_t saved_m0;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
                 : "=&s"(saved_m0) : "v"(offset), "s"(base), "s"(lds_address) : "memory");
}

// Until at most N of this lane's loads into shared memory are on their way.
template <int N>
static __device__ __forceinline__ void wait_loads() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

static __device__ __forceinline__ void wait_reads() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// A barrier that nothing is moved across (the products before it stay before it, and the reads behind it behind).
static __device__ __forceinline__ void meet() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
}

// GATED: 0 plain, 1 + the gate's number for the gated product.  N is the number of rows of w (plain) or of gate rows
// (gated); `stride` elements from a row of `out` to the next.  `vectors`: rows of `out` begin at multiples of 16 bytes.
template <int GATED>
__global__ void __launch_bounds__(512, 2)
gemm_wide_kernel(const bf16* __restrict__ x, const bf16* __restrict__ w, bf16* __restrict__ out, float* __restrict__ partial,
                 int M, int N, int K, int stride, bool vectors, int m_tiles, int n_tiles, int splits, GateShape shape) {
    constexpr int kColumns = GATED ? kWideHalf : kWideRows;         // output columns a tile
    constexpr bool kPair = GATED == kGatePairSquaredRelu + 1;
    extern __shared__ __align__(16) unsigned char tiles_s[];        // [2 stages][x half, x half, w half, w half]
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int i = lane % 16, g = lane / 16;
    const int wm = wave / 4, wn = wave % 4;                          // wm is also the group: waves of one vector unit are 4 apart

    const int tiles = m_tiles * n_tiles, items = tiles * splits, all_stages = K / kWideKeys;
    const int xcd = blockIdx.x % 8, per_xcd = items / 8, left = items % 8;
    const int first = xcd * per_xcd + min(xcd, left), end = first + per_xcd + (xcd < left ? 1 : 0);
    const int step = gridDim.x / 8;
    int item = first + blockIdx.x / 8;
    if (item >= end) return;

    const int chunk = (lane % 8) ^ (lane / 8);
    const uint32_t lds_base = __builtin_amdgcn_readfirstlane(
        static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) void*)tiles_s)));
    uint32_t offset[4][2];      // what this lane brings of each half: rows 8 (wave + 8 u) + lane / 8
    int m_base, n_base, piece, stages;
    const unsigned char *x_bytes, *w_bytes;
    auto place_item = [&](int it) {
        piece = it / tiles;
        const int t = it - piece * tiles;
        const int band = t / (8 * n_tiles), in_band = t - band * 8 * n_tiles;
        const int band_rows = min(8, m_tiles - 8 * band);
        const int n_tile = in_band / band_rows;
        m_base = (8 * band + in_band - n_tile * band_rows) * kWideRows;
        n_base = n_tile * kColumns;
        const int begin = static_cast<int>(static_cast<long long>(piece) * all_stages / splits);
        stages = static_cast<int>(static_cast<long long>(piece + 1) * all_stages / splits) - begin;
        x_bytes = reinterpret_cast<const unsigned char*>(x) + static_cast<size_t>(begin) * (kWideKeys * 2);
        w_bytes = reinterpret_cast<const unsigned char*>(w) + static_cast<size_t>(begin) * (kWideKeys * 2);
#pragma unroll
        for (int h = 0; h < 4; ++h)
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int r = 8 * (wave + 8 * u) + lane / 8;
                size_t row;
                if (h < 2) row = min(m_base + kWideHalf * h + r, M - 1);
                else if (GATED) row = static_cast<size_t>(min(n_base + r, N - 1)) + (h == 3 ? N : 0);
                else row = min(n_base + kWideHalf * (h - 2) + r, N - 1);
                offset[h][u] = static_cast<uint32_t>((row * K + chunk * 8) * 2);
            }
    };
    auto send = [&](int h, int s) {
        const unsigned char* base = (h < 2 ? x_bytes : w_bytes) + static_cast<size_t>(s) * (kWideKeys * 2);
        const uint32_t to = lds_base + (s & 1) * kWideStage + h * kHalfBytes + wave * 1024;
#pragma unroll
        for (int u = 0; u < 2; ++u) load_to_shared(base, offset[h][u], to + u * 8192);
    };
    auto send_first = [&] {
        send(0, 0);
        send(2, 0);
        send(3, 0);
        send(1, 0);
        if (stages > 1) {
            send(0, 1);
            send(2, 1);
            send(3, 1);
        }
    };

    WFrag fx[4][2], fw[2][2][2];         // [16 rows of the x half][32 keys], [w half][16 rows][32 keys]
    const int place0 = (g ^ (i % 8)) * 16, place1 = ((4 + g) ^ (i % 8)) * 16;
    auto read_x = [&](int s, int h) {
        const unsigned char* p = tiles_s + (s & 1) * kWideStage + h * kHalfBytes + (wm * 64 + i) * 128;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            fx[b][0].u = *reinterpret_cast<const uint4*>(p + b * 2048 + place0);
            fx[b][1].u = *reinterpret_cast<const uint4*>(p + b * 2048 + place1);
        }
    };
    auto read_w = [&](int s, int h) {
        const unsigned char* p = tiles_s + (s & 1) * kWideStage + (2 + h) * kHalfBytes + (wn * 32 + i) * 128;
#pragma unroll
        for (int a = 0; a < 2; ++a) {
            fw[h][a][0].u = *reinterpret_cast<const uint4*>(p + a * 2048 + place0);
            fw[h][a][1].u = *reinterpret_cast<const uint4*>(p + a * 2048 + place1);
        }
    };

    place_item(item);
    send_first();
    for (;;) {
        float4_t acc[2][2][2][4];        // [x half][w half][16 rows of w][16 rows of x]
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int c = 0; c < 2; ++c)
#pragma unroll
                    for (int d = 0; d < 4; ++d) acc[a][b][c][d] = float4_t{0.f, 0.f, 0.f, 0.f};
        auto products = [&](int xh) {
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int wh = 0; wh < 2; ++wh)
#pragma unroll
                for (int k = 0; k < 2; ++k)
#pragma unroll
                    for (int a = 0; a < 2; ++a)
#pragma unroll
                        for (int b = 0; b < 4; ++b)
                            acc[xh][wh][a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[wh][a][k].v, fx[b][k].v,
                                                                                        acc[xh][wh][a][b], 0, 0, 0);
            __builtin_amdgcn_s_setprio(0);
        };
        const int n_stages = stages;
        if (n_stages > 1) wait_loads<8>();         // stage 0's first x half and w halves, 3 of the 7 halves sent, and more
        else wait_loads<0>();
        meet();
        if (wm == 1) meet();
        for (int s = 0; s < n_stages; ++s) {
            read_w(s, 0);
            read_x(s, 0);
            read_w(s, 1);
            if (s + 1 < n_stages) {
                send(1, s + 1);
                wait_loads<8>();                   // behind x's second half of this stage: the next stage's four halves
            } else {
                wait_loads<0>();
            }
            wait_reads();
            meet();
            products(0);
            meet();
            read_x(s, 1);
            if (s + 2 < n_stages) {
                send(0, s + 2);
                send(2, s + 2);
                send(3, s + 2);
                wait_loads<8>();                   // behind the next stage's first three halves: its fourth, and these three
            } else {
                wait_loads<0>();
            }
            wait_reads();
            meet();
            products(1);
            meet();
        }
        if (wm == 0) meet();                       // every wavefront is done with the shared memory

        const int m_now = m_base, n_now = n_base, piece_now = piece;
        item += step;
        const bool again = item < end;
        if (again) {
            place_item(item);
            send_first();
        }
        // ---- lane (i, g) holds, of quarter (xh, wh) and tile (a, b), output row 16 b + i and columns 4g .. 4g + 3 ----
#pragma unroll
        for (int xh = 0; xh < 2; ++xh)
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const int m = m_now + xh * kWideHalf + wm * 64 + 16 * b + i;
                if (m >= M) continue;
                if (!GATED && partial != nullptr) {
                    float* row = partial + (static_cast<size_t>(piece_now) * M + m) * N;
#pragma unroll
                    for (int wh = 0; wh < 2; ++wh)
#pragma unroll
                        for (int a = 0; a < 2; ++a) {
                            const int n = n_now + wh * kWideHalf + wn * 32 + 16 * a + 4 * g;
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
                    // the lanes g and g + 1 (g even) exchange, so that each holds eight neighbouring columns: of the 32, the
                    // even lane 8 (g / 2) .. + 7, the odd one those 16 further on
                    typedef unsigned uint2_t __attribute__((ext_vector_type(2)));
                    const uint2_t lo = __builtin_amdgcn_permlane16_swap(q[0][0], q[1][0], false, false);
                    const uint2_t hi = __builtin_amdgcn_permlane16_swap(q[0][1], q[1][1], false, false);
                    const int n = n_now + (GATED ? 0 : wh * kWideHalf) + wn * 32 + 16 * (g & 1) + 8 * (g >> 1);
                    bf16* to = row + (kPair && wh == 1 ? N : 0) + n;
                    const uint32_t words[4] = {lo.x, hi.x, lo.y, hi.y};
                    if (vectors && n + 7 < N) {
                        *reinterpret_cast<uint4*>(to) = make_uint4(words[0], words[1], words[2], words[3]);
                    } else {
#pragma unroll
                        for (int v = 0; v < 8; ++v)
                            if (n + v < N) to[v] = bf16{static_cast<uint16_t>(words[v / 2] >> (16 * (v % 2)))};
                    }
                }
            }
        if (!again) break;
    }
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
