// Products of float32 numbers on the bfloat16 matrix instruction, with float32's precision: a number is the sum of three bfloat16 numbers,
//   hi = round(v), mid = round(v - hi), lo = round(v - hi - mid),
// each subtraction exact, and of the nine products of two such sums the six largest are taken.  lo holds what hi and mid leave to the last bit (8 bits
// of 24 each, down to 2^-133), and the three products left out are less than 2^-25 of the whole product, half of what rounding one float32 number loses.  The products of bfloat16
// numbers are exact in float32, and the sums are float32's.
//
// The instruction adds 32 keys' products before it rounds to the accumulator where the float32 instruction adds 4, so the chain of roundings of a sum is
// shorter.  Off from 64 bits (normal x and w, 2-norm, and the worst element over the sum of the absolute products): 2,048 keys 3.41e-7 and 8.8e-8 where the
// float32 instruction's products in the same segments are off by 4.08e-7 and 1.16e-7, 16,384 keys 3.82e-7 and 2.4e-8 for 4.20e-7 and 2.6e-8.  (It cuts off where the float32 instruction rounds: a mean
// of -1.8e-9 of the absolute products, within those figures.)
//
// Numbers that are not finite, and finite ones above 3.39e38 that round to infinity in bfloat16, make mid or lo a NaN, and so the sum they enter.  A sum that is not finite is therefore
// made again from the float32 numbers (`plain_product`), which gives infinities and NaN where float32's own sums have them.
#pragma once
#include "lds_load.h"

// Eight float32 numbers as three fragments of eight bfloat16 numbers: a's four, then b's.
static __device__ __forceinline__ void split_numbers(float v0, float v1, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
    hi = pack2_bf16(v0, v1);
    const float r0 = v0 - __uint_as_float(hi << 16), r1 = v1 - __uint_as_float(hi & 0xffff0000u);
    mid = pack2_bf16(r0, r1);
    lo = pack2_bf16(r0 - __uint_as_float(mid << 16), r1 - __uint_as_float(mid & 0xffff0000u));
}

struct SplitFragment {
    Fragment part[3];              // hi, mid, lo
};

static __device__ __forceinline__ void split_eight(const float4_t a, const float4_t b, SplitFragment& to) {
    uint32_t words[3][4];
    split_numbers(a[0], a[1], words[0][0], words[1][0], words[2][0]);
    split_numbers(a[2], a[3], words[0][1], words[1][1], words[2][1]);
    split_numbers(b[0], b[1], words[0][2], words[1][2], words[2][2]);
    split_numbers(b[2], b[3], words[0][3], words[1][3], words[2][3]);
#pragma unroll
    for (int p = 0; p < 3; ++p) to.part[p].u = make_uint4(words[p][0], words[p][1], words[p][2], words[p][3]);
}

// The six products, smallest first: (part of w, part of x) of product number p.
constexpr int kSplitProducts = 6;
static __device__ __forceinline__ constexpr int split_w(int p) { constexpr int t[] = {2, 0, 1, 1, 0, 0}; return t[p]; }
static __device__ __forceinline__ constexpr int split_x(int p) { constexpr int t[] = {0, 2, 1, 0, 1, 0}; return t[p]; }

static __device__ __forceinline__ float4_t split_product(const SplitFragment& w, const SplitFragment& x, float4_t acc, int p) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.part[split_w(p)].v, x.part[split_x(p)].v, acc, 0, 0, 0);
}

// 0 if four sums are finite, else NaN.
static __device__ __forceinline__ float finite_probe(const float4_t v) { return v[0] * 0.f + v[1] * 0.f + (v[2] * 0.f + v[3] * 0.f); }

// The product of row `x` and row n of w over keys k_begin .. k_end - 1, multiplied and added in float32 by ascending keys, in segments of `segment`
// keys whose sums are added in order.  `w` is the weight row by row or (TILED) its tile-major copy, `chunks` of 16 keys a row.
template <bool TILED>
static __device__ __forceinline__ float plain_product(const float* x, const float* w, int n, int K, int chunks, int k_begin, int k_end, int segment) {
    const float* row = TILED ? w + static_cast<size_t>(n / 16) * chunks * 256 + n % 16 * 4 : w + static_cast<size_t>(n) * K;
    float total = 0.f;
    for (int k0 = k_begin; k0 < k_end; k0 += segment) {
        float sum = 0.f;
        for (int k = k0; k < min(k_end, k0 + segment); ++k)
            sum = __builtin_fmaf(x[k], row[TILED ? static_cast<size_t>(k / 16) * 256 + k % 16 / 4 * 64 + k % 4 : k], sum);
        total = k0 == k_begin ? sum : total + sum;
    }
    return total;
}
