// The walk over the K axis that the products of many rows share (`gemm_wide.hip`, and the experts' in `moe_wide.hip`): a workgroup of
// eight wavefronts makes tiles of 256 rows of x by 256 rows of w from operands that it brings to shared memory itself.
//
// The tile is two halves of 128 rows of x by two halves of 128 rows of w; wavefront (wm, wn) of the 2 x 4 makes, of each
// of the four quarters, the 64 x 32 at (64 wm, 32 wn), as products v_mfma_f32_16x16x32_bf16 (w is the A operand, x the B
// operand: lane (i, g) ends with four consecutive columns of one output row).
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
// a stage and a half to arrive.  A tile without a second half of x (6 newer loads) leaves out its reads, loads and products.
#pragma once
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

template <bool V>
struct WideFlag {
    static constexpr bool value = V;
};

// Where a tile's operands are: what this lane brings of each half (x, x, w, w), rows 8 (wave + 8 u) + lane / 8 of the half, in
// bytes from `x_bytes` or `w_bytes` at the stage's first key; `two`: there is a second half of x.
struct WideSource {
    uint32_t offset[4][2];
    const unsigned char *x_bytes, *w_bytes;
    int stages;
    bool two;
};

typedef float4_t WideSums[2][2][2][4];       // [x half][w half][16 rows of w][16 rows of x]

// The row of a half, and the chunk of 16 bytes of it, that this lane's load `u` brings.
static __device__ __forceinline__ int wide_row(int u) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    return 8 * (wave + 8 * u) + threadIdx.x % kWave / 8;
}
static __device__ __forceinline__ int wide_chunk() { return (threadIdx.x % 8) ^ (threadIdx.x % kWave / 8); }

// Lanes g and g + 1 (g even) of a row exchange halves of what they hold (four neighbouring columns of each of two tiles of 16), so that
// each has eight neighbouring columns of the 32: the even lane 8 (g / 2) .. + 7, the odd one those 16 further on.
static __device__ __forceinline__ uint4 wide_eight_columns(const uint32_t q[2][2]) {
    typedef unsigned uint2_t __attribute__((ext_vector_type(2)));
    const uint2_t lo = __builtin_amdgcn_permlane16_swap(q[0][0], q[1][0], false, false);
    const uint2_t hi = __builtin_amdgcn_permlane16_swap(q[0][1], q[1][1], false, false);
    return make_uint4(lo.x, hi.x, lo.y, hi.y);
}

// Items `item`, item + step, ... below `end`, one after the other; the first stages of the next one are sent before the results
// of the last are written.  `place(item, source)` says where an item's operands are and returns what `finish(what, sums)` needs to
// write its results.  ONE: items may have one half of x.
template <bool ONE, typename Place, typename Finish>
static __device__ __forceinline__ void wide_products(unsigned char* tiles_s, int item, int end, int step, Place place, Finish finish) {
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int i = lane % 16, g = lane / 16;
    const int wm = wave / 4, wn = wave % 4;                          // wm is also the group: waves of one vector unit are 4 apart
    const uint32_t lds_base = __builtin_amdgcn_readfirstlane(
        static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) void*)tiles_s)));
    WideSource from;
    auto send = [&](int h, int s) {
        const unsigned char* base = (h < 2 ? from.x_bytes : from.w_bytes) + static_cast<size_t>(s) * (kWideKeys * 2);
        const uint32_t to = lds_base + (s & 1) * kWideStage + h * kHalfBytes + wave * 1024;
#pragma unroll
        for (int u = 0; u < 2; ++u) load_to_shared(base, from.offset[h][u], to + u * 8192);
    };
    auto send_first = [&] {
        send(0, 0);
        send(2, 0);
        send(3, 0);
        if (!ONE || from.two) send(1, 0);
        if (from.stages > 1) {
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

    auto now = place(item, from);
    send_first();
    for (;;) {
        WideSums acc;
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
        const int stages = from.stages;
        if (stages <= 1) wait_loads<0>();
        else if (!ONE || from.two) wait_loads<8>();        // stage 0's first x half and w halves are 3 of the 7 (or 6) halves sent
        else wait_loads<6>();
        meet();
        if (wm == 1) meet();
        auto walk = [&](auto both) {
            constexpr bool kTwo = decltype(both)::value;
            for (int s = 0; s < stages; ++s) {
                read_w(s, 0);
                read_x(s, 0);
                read_w(s, 1);
                if (kTwo) {
                    if (s + 1 < stages) {
                        send(1, s + 1);
                        wait_loads<8>();           // behind x's second half of this stage: the next stage's four halves
                    } else {
                        wait_loads<0>();
                    }
                }
                wait_reads();
                meet();
                products(0);
                meet();
                if (kTwo) read_x(s, 1);
                if (s + 2 < stages) {
                    send(0, s + 2);
                    send(2, s + 2);
                    send(3, s + 2);
                    wait_loads<kTwo ? 8 : 6>();    // behind the next stage's first three halves: its fourth, and these three
                } else {
                    wait_loads<0>();
                }
                wait_reads();
                meet();
                if (kTwo) products(1);
                meet();            // (also where D is empty: the other group's wait in C stands between a stage's loads and A)
            }
        };
        if (!ONE || from.two) walk(WideFlag<true>());
        else walk(WideFlag<false>());
        if (wm == 0) meet();                       // every wavefront is done with the shared memory

        const auto done = now;
        item += step;
        const bool again = item < end;
        if (again) {
            now = place(item, from);
            send_first();
        }
        finish(done, acc);
        if (!again) break;
    }
}
