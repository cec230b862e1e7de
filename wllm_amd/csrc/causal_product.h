// What the recurrences walked in chunks of 16 tokens share: the part of a chunk's results that its own tokens make.
#pragma once
#include "common.h"

constexpr int kChunk = 16;           // tokens of a chunk

// The place of a segment's first chunk in the scratch, for segments of `from` tokens (16 at least) and more: chunk c lies c
// places further.  No two chunks share a place, whatever order the segments come in: a segment of n >= from tokens has at most
// n / 16 + 1 chunks, and the first place of what begins n tokens later is at least n / 16 + 1 further.  The last place of a step
// of t tokens is t / 16 + t / from - 1.
__host__ __device__ __forceinline__ int first_place(int q_start, int from) { return q_start / kChunk + q_start / from; }
__host__ __device__ __forceinline__ int chunk_places(int tokens, int from) { return tokens / kChunk + tokens / from; }

typedef float causal_float4 __attribute__((ext_vector_type(4)));

// part + N x on v_mfma_f32_16x16x4_f32 for the four tokens s = token_of(0 .. 3): lane (i, g) holds n = N[i][token_of(g)] and
// x = column i of token_of(g), and gets the rows t = 4g .. 4g + 3 of column i.  N is zero where the key s is later than the
// row t, but 0 x inf is NaN: a value of x that is not finite is taken out of the product and given to the rows from its
// own token on alone, so that the tokens before it are what they are without it.  (One comparison and a branch no wave
// takes otherwise; every other sum has the same bits with it and without.)
template <typename TOKEN>
__device__ __forceinline__ causal_float4 add_causal_product(float n, float x, causal_float4 part, int i, int g, TOKEN token_of) {
    constexpr float kLargest = 3.402823466e38f;
    const bool finite = fabsf(x) <= kLargest;
    part = __builtin_amdgcn_mfma_f32_16x16x4f32(n, finite ? x : 0.f, part, 0, 0, 0);
    if (__ballot(!finite)) {
        // (places that the compiler knows nothing of: it would work out all of them ahead of the loop over the chunks, in
        // registers that cost ssm_chunk_scan_kernel its second workgroup on a compute unit)
        asm volatile("" : "+v"(i), "+v"(g));
#pragma unroll 1
        for (int q = 0; q < 4; ++q) {
            const float value = __shfl(x, 16 * q + i);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int t = 4 * g + u;
                const float weight = __shfl(n, 16 * q + t);
                if (!(fabsf(value) <= kLargest) && t >= token_of(q)) part[u] = fmaf(weight, value, part[u]);
            }
        }
    }
    return part;
}
