// A selective state-space mixer (the recurrence of Mamba-2) on a flat batch of segments: the short
// causal convolution with its carried inputs, the recurrence with its carried state, and the gated
// norm in groups behind it.  A segment is the next tokens of one request; what a request carries from
// step to step lies in one float32 row of `state` per request (row state_slots[segment]):
//   [heads, N, P] the recurrence's state S, then [taps - 1, channels] the convolution's last inputs
//   (the oldest first).
// A fresh request's row is all zeros, which is both "S starts at zero" and "zeros before the start".
// Everything that enters the recurrence is float32: step sizes, decays, the state, the sums.
#include "causal_product.h"
#include "common.h"
#include "short_conv.h"

// ---- convolution: out[t, c] = silu(bias[c] + sum_k w[c, k] * in[t - (taps - 1) + k, c]), the inputs
// before the segment's first token taken from the carried rows.  in is a band of a wider row. ----
template <typename T>
__global__ void __launch_bounds__(256)
causal_conv_kernel(const T* __restrict__ in, long long in_stride, const float* __restrict__ weight,
                   const float* __restrict__ bias, const float* __restrict__ state, long long state_stride,
                   long long carried_offset, const int* __restrict__ token_segment, const int* __restrict__ seg_q_start,
                   const int* __restrict__ state_slots, T* __restrict__ out, int channels, int taps) {
    const int token = blockIdx.x;
    const int seg = token_segment[token];
    const int local = token - seg_q_start[seg];
    const float* carried = state + static_cast<size_t>(state_slots[seg]) * state_stride + carried_offset;
    for (int c = blockIdx.y * blockDim.x + threadIdx.x; c < channels; c += gridDim.y * blockDim.x) {
        float acc = bias[c];
        for (int k = 0; k < taps; ++k) {
            const int src = local - (taps - 1) + k;          // place in the segment; negative: a carried input
            const float v = src >= 0 ? to_float(in[static_cast<size_t>(token - local + src) * in_stride + c])
                                     : carried[static_cast<size_t>(taps - 1 + src) * channels + c];
            acc = fmaf(weight[static_cast<size_t>(c) * taps + k], v, acc);
        }
        out[static_cast<size_t>(token) * channels + c] = from_float<T>(acc / (1.f + expf(-acc)));
    }
}

// The same sums for steps of a token a segment and fewer: a workgroup walks a segment's tokens in order, each thread its channels with the
// carried rows in registers (TAPS; 0: any number, the rows in memory), and writes the new rows behind them: no launch behind this one.  A decode
// step's chain is two launches otherwise: 8 tokens of 6,144 channels 5.0 and 4.7 us, now 4.8.
template <typename T, int TAPS>
__global__ void __launch_bounds__(256)
causal_conv_segment_kernel(const T* __restrict__ in, long long in_stride, const float* __restrict__ weight,
                           const float* __restrict__ bias, float* __restrict__ state, long long state_stride,
                           long long carried_offset, const int* __restrict__ seg_q_start, const int* __restrict__ seg_q_len,
                           const int* __restrict__ state_slots, T* __restrict__ out, int channels, int taps) {
    const int seg = blockIdx.x, begin = seg_q_start[seg], len = seg_q_len[seg];
    if (len <= 0) return;
    float* carried = state + static_cast<size_t>(state_slots[seg]) * state_stride + carried_offset;
    for (int c = blockIdx.y * blockDim.x + threadIdx.x; c < channels; c += gridDim.y * blockDim.x) {
        const float* w = weight + static_cast<size_t>(c) * taps;
        const float b = bias[c];
        float rows[TAPS > 1 ? TAPS - 1 : 1], by[TAPS > 0 ? TAPS : 1];
#pragma unroll
        for (int k = 0; k < TAPS; ++k) {
            by[k] = w[k];
            if (k + 1 < TAPS) rows[k] = carried[static_cast<size_t>(k) * channels + c];
        }
        for (int t = begin; t < begin + len; ++t) {
            const float now = to_float(in[static_cast<size_t>(t) * in_stride + c]);
            float acc = b;
            if (TAPS > 0) {
#pragma unroll
                for (int k = 0; k + 1 < TAPS; ++k) {
                    acc = fmaf(by[k], rows[k], acc);
                    rows[k] = k + 2 < TAPS ? rows[k + 1] : now;
                }
                acc = fmaf(by[TAPS > 0 ? TAPS - 1 : 0], now, acc);
            } else {
                for (int k = 0; k + 1 < taps; ++k) {
                    const float v = carried[static_cast<size_t>(k) * channels + c];
                    acc = fmaf(w[k], v, acc);
                    if (k > 0) carried[static_cast<size_t>(k - 1) * channels + c] = v;
                }
                acc = fmaf(w[taps - 1], now, acc);
                if (taps > 1) carried[static_cast<size_t>(taps - 2) * channels + c] = now;
            }
            out[static_cast<size_t>(t) * channels + c] = from_float<T>(acc / (1.f + expf(-acc)));
        }
#pragma unroll
        for (int k = 0; k + 1 < TAPS; ++k) carried[static_cast<size_t>(k) * channels + c] = rows[k];
    }
}

// The same sums for the many tokens of a prompt's portion and convolutions of kSlideTaps taps: a thread takes four
// consecutive channels and walks kSlideTokens tokens with the last inputs in registers, so a row is read once and not
// once a tap, in 8-byte (float32: 16-byte) pieces (6,144 channels of 1,500 tokens: 62 to 17 us).
// Fewer elements than `many_elements` are bound by a launch's chain, which is longer here (the kernel a token and the one for the
// carried rows behind it, against this one, us: 256 channels of 200 tokens 5.1 and 5.5, 2,048 of 64 5.4 and 6.0, of 200 6.6 and 6.1, 6,144 of
// 64 6.4 and 6.2), and tokens that each begin a segment are a chain of their own (6,144 channels of 96 segments of one token 9.2 and
// 10.1, 2,048 of 200 segments of two 12.5 and 8.2).
constexpr int kSlideTaps = 4, kSlideTokens = 8, kSlideFrom = 64;
static bool slides(int tokens, int segments, int channels, long long many_elements) {
    return tokens >= kSlideFrom && tokens >= 2LL * segments && static_cast<long long>(tokens) * channels >= many_elements;
}
template <typename T> struct alignas(4 * sizeof(T)) ConvFour { T v[4]; };

template <typename T>
__device__ __forceinline__ float4 conv_four(const T* p) {
    const ConvFour<T> r = *reinterpret_cast<const ConvFour<T>*>(p);
    return make_float4(to_float(r.v[0]), to_float(r.v[1]), to_float(r.v[2]), to_float(r.v[3]));
}

// Walks the tokens of a tile of kSlideTokens from `token0`, four channels at `in`: calls make(token, rows) with the rows
// of the last kSlideTaps inputs, the oldest first.  Inputs before a segment's first token are its request's carried rows.
// The carried rows of a segment are read by its first three tokens only, and these always belong to the tile of the
// first: a tile that begins at a segment's second or third token leaves them to the tile before it, which walks up to
// kSlideOver tokens more.  So the thread that has read a request's carried rows is the only one that will, and writes
// the new ones (the segment's last inputs) without a launch behind this one.  2,048 channels of 3,001 float32 tokens: 9.3
// us and 3.0 in a launch behind it, now 10.0.
constexpr int kSlideOver = kSlideTaps - 2;
template <typename T, typename MAKE>
__device__ __forceinline__ void slide(const T* in, long long in_stride, float* state, long long state_stride,
                                      long long carried_offset, const int* token_segment, const int* seg_q_start,
                                      const int* seg_q_len, const int* state_slots, int channels, int token0, int tokens,
                                      MAKE make) {
    constexpr int kWalk = kSlideTokens + kSlideOver, kCarried = kSlideTaps - 1;
    float4 rows[kSlideTaps];
    auto begin_segment = [&](int seg, int start) {
        float* carried = state + static_cast<size_t>(state_slots[seg]) * state_stride + carried_offset;
        const int len = seg_q_len[seg];
        float4 last[kCarried];
#pragma unroll
        for (int k = 0; k < kCarried; ++k) {
            rows[k + 1] = *reinterpret_cast<const float4*>(carried + static_cast<size_t>(k) * channels);
            last[k] = conv_four(in + static_cast<size_t>(start + max(len - kCarried + k, 0)) * in_stride);
        }
#pragma unroll
        for (int k = 0; k < kCarried; ++k) {           // a segment of fewer tokens keeps some of the rows, moved up
            float4 v = last[k];
#pragma unroll
            for (int n = 1; n < kCarried; ++n)
                if (len == n && k + n < kCarried) v = rows[k + n + 1];
            if (len > 0) *reinterpret_cast<float4*>(carried + static_cast<size_t>(k) * channels) = v;
        }
    };
    ConvFour<T> now[kWalk];
    int segs[kWalk];
#pragma unroll
    for (int t = 0; t < kWalk; ++t) {
        const int token = min(token0 + t, tokens - 1);
        now[t] = *reinterpret_cast<const ConvFour<T>*>(in + static_cast<size_t>(token) * in_stride);
        segs[t] = token_segment[token];
    }
    const int local0 = token0 - seg_q_start[segs[0]];
    int local = local0;
#pragma unroll
    for (int k = 0; k < kSlideTaps; ++k)
        rows[k] = k > 0 && local0 - kSlideTaps + k >= 0 ? conv_four(in + static_cast<size_t>(token0 - kSlideTaps + k) * in_stride)
                                                        : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int t = 0; t < kWalk; ++t) {
        if (token0 + t >= tokens) break;
        if (t > 0) local = segs[t] != segs[t - 1] ? token0 + t - seg_q_start[segs[t]] : local + 1;
        if (t >= kSlideTokens && (local == 0 || local >= kCarried)) break;
        if (local == 0) begin_segment(segs[t], token0 + t);
#pragma unroll
        for (int k = 0; k + 1 < kSlideTaps; ++k) rows[k] = rows[k + 1];
        rows[kSlideTaps - 1] = make_float4(to_float(now[t].v[0]), to_float(now[t].v[1]), to_float(now[t].v[2]), to_float(now[t].v[3]));
        if (local == t + local0 && local0 > 0 && local < kCarried) continue;       // a token of the tile before
        make(token0 + t, rows);
    }
}

template <typename T>
__global__ void __launch_bounds__(256)
causal_conv_slide_kernel(const T* __restrict__ in, long long in_stride, const float* __restrict__ weight,
                         const float* __restrict__ bias, float* __restrict__ state, long long state_stride,
                         long long carried_offset, const int* __restrict__ token_segment, const int* __restrict__ seg_q_start,
                         const int* __restrict__ seg_q_len, const int* __restrict__ state_slots, T* __restrict__ out, int tokens,
                         int channels) {
    const int c = (blockIdx.y * 256 + threadIdx.x) * 4, token0 = blockIdx.x * kSlideTokens;
    if (c >= channels) return;
    float4 w[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) w[u] = *reinterpret_cast<const float4*>(weight + static_cast<size_t>(c + u) * kSlideTaps);
    const float4 b = *reinterpret_cast<const float4*>(bias + c);
    slide(in + c, in_stride, state, state_stride, carried_offset + c, token_segment, seg_q_start, seg_q_len, state_slots, channels,
          token0, tokens, [&](int token, const float4 (&rows)[kSlideTaps]) {
        float acc[4] = {b.x, b.y, b.z, b.w};
        const float* wf = reinterpret_cast<const float*>(w);
#pragma unroll
        for (int k = 0; k < kSlideTaps; ++k) {
            acc[0] = fmaf(wf[k], rows[k].x, acc[0]);
            acc[1] = fmaf(wf[4 + k], rows[k].y, acc[1]);
            acc[2] = fmaf(wf[8 + k], rows[k].z, acc[2]);
            acc[3] = fmaf(wf[12 + k], rows[k].w, acc[3]);
        }
        ConvFour<T> r;
#pragma unroll
        for (int u = 0; u < 4; ++u) r.v[u] = from_float<T>(acc[u] / (1.f + expf(-acc[u])));
        *reinterpret_cast<ConvFour<T>*>(out + static_cast<size_t>(token) * channels + c) = r;
    });
}

// Whether the channels and the addresses let a thread take four channels of a row at once.
template <typename T>
static bool in_fours(const void* in, long long in_stride, const float* weight, const float* bias, const float* state,
                     long long state_stride, long long carried_offset, const void* out, int channels) {
    const uintptr_t vectors = reinterpret_cast<uintptr_t>(weight) | reinterpret_cast<uintptr_t>(bias) | reinterpret_cast<uintptr_t>(state);
    return channels % 4 == 0 && in_stride % 4 == 0 && state_stride % 4 == 0 && carried_offset % 4 == 0 && vectors % 16 == 0 &&
           (reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) % (4 * sizeof(T)) == 0;
}

WLLM_API int wllm_causal_conv(const void* in, long long in_stride, const float* weight, const float* bias, float* state,
                              long long state_stride, long long carried_offset, const int* token_segment,
                              const int* seg_q_start, const int* seg_q_len, const int* state_slots, void* out,
                              int is_bf16, int tokens, int segments, int channels, int taps, hipStream_t stream) {
    if (tokens <= 0 || segments <= 0) return 0;
    if (channels <= 0 || taps < 1 || taps > 64) return -1;
    const int tiles = (channels + 255) / 256 < 64 ? (channels + 255) / 256 : 64;
    const dim3 grid(tokens, tiles), carry_grid(segments, tiles);
    const dim3 slide_grid((tokens + kSlideTokens - 1) / kSlideTokens, (channels / 4 + 255) / 256);
#define SLIDE(T)                                                                                                        \
    causal_conv_slide_kernel<T><<<slide_grid, 256, 0, stream>>>(static_cast<const T*>(in), in_stride, weight, bias, state, \
                                                                state_stride, carried_offset, token_segment, seg_q_start, \
                                                                seg_q_len, state_slots, static_cast<T*>(out), tokens, \
                                                                channels)
    const bool many = taps == kSlideTaps && slides(tokens, segments, channels, 3LL << 17);   // (these keep the carried rows themselves)
    if (many && is_bf16 && in_fours<bf16>(in, in_stride, weight, bias, state, state_stride, carried_offset, out, channels))
        return SLIDE(bf16), launch_status();
    if (many && !is_bf16 && in_fours<float>(in, in_stride, weight, bias, state, state_stride, carried_offset, out, channels))
        return SLIDE(float), launch_status();
#undef SLIDE
    if (tokens <= segments) {
#define LAUNCH(T, TAPS)                                                                                                    \
    causal_conv_segment_kernel<T, TAPS><<<carry_grid, 256, 0, stream>>>(                                                   \
        static_cast<const T*>(in), in_stride, weight, bias, state, state_stride, carried_offset, seg_q_start, seg_q_len,   \
        state_slots, static_cast<T*>(out), channels, taps)
        if (is_bf16) { if (taps == kSlideTaps) LAUNCH(bf16, kSlideTaps); else LAUNCH(bf16, 0); }
        else { if (taps == kSlideTaps) LAUNCH(float, kSlideTaps); else LAUNCH(float, 0); }
#undef LAUNCH
        return launch_status();
    }
    if (is_bf16)
        causal_conv_kernel<bf16><<<grid, 256, 0, stream>>>(static_cast<const bf16*>(in), in_stride, weight, bias, state,
                                                           state_stride, carried_offset, token_segment, seg_q_start,
                                                           state_slots, static_cast<bf16*>(out), channels, taps);
    else
        causal_conv_kernel<float><<<grid, 256, 0, stream>>>(static_cast<const float*>(in), in_stride, weight, bias, state,
                                                            state_stride, carried_offset, token_segment, seg_q_start,
                                                            state_slots, static_cast<float*>(out), channels, taps);
    if (const int err = launch_status()) return err;
    if (taps == 1) return 0;
    if (is_bf16)
        conv_carry_kernel<bf16><<<carry_grid, 256, 0, stream>>>(static_cast<const bf16*>(in), in_stride, state, state_stride,
                                                                carried_offset, seg_q_start, seg_q_len, state_slots, channels,
                                                                taps);
    else
        conv_carry_kernel<float><<<carry_grid, 256, 0, stream>>>(static_cast<const float*>(in), in_stride, state,
                                                                 state_stride, carried_offset, seg_q_start, seg_q_len,
                                                                 state_slots, channels, taps);
    return launch_status();
}

// ---- the same convolution on the residual stream itself, in front of a sublayer that reads the stream:
// out[t, c] = x[t, c] + sum_k w[k, c] * x[t - (taps - 1) + k, c] (w a row a tap, [taps, channels]), float32 sums in this order, no bias and no
// activation; x float32 [tokens, channels], out the activation type.  The carried rows (the request's last
// taps - 1 rows of x, the oldest first) are kept by `conv_carry_kernel` (by `slide`), as above; or, CARRY (a step of single
// tokens, where no other token of the launch reads a request's carried rows), by the token's own threads, each
// moving its channel's rows up by one as it reads them: one launch instead of two, the same sums. ----
template <typename T, bool CARRY>
__global__ void __launch_bounds__(256)
stream_conv_kernel(const float* __restrict__ x, const float* __restrict__ weight, float* __restrict__ state,
                   long long state_stride, long long carried_offset, const int* __restrict__ token_segment,
                   const int* __restrict__ seg_q_start, const int* __restrict__ state_slots, T* __restrict__ out,
                   int channels, int taps) {
    const int token = blockIdx.x;
    const int seg = token_segment[token];
    const int local = token - seg_q_start[seg];
    float* carried = state + static_cast<size_t>(state_slots[seg]) * state_stride + carried_offset;
    for (int c = blockIdx.y * blockDim.x + threadIdx.x; c < channels; c += gridDim.y * blockDim.x) {
        float acc = x[static_cast<size_t>(token) * channels + c];
        if (CARRY) {
            // the segment is this one token: every earlier input is a carried row
            const float now = acc;
            for (int k = 0; k + 1 < taps; ++k) {
                const float v = carried[static_cast<size_t>(k) * channels + c];
                acc = fmaf(weight[static_cast<size_t>(k) * channels + c], v, acc);
                if (k > 0) carried[static_cast<size_t>(k - 1) * channels + c] = v;
            }
            acc = fmaf(weight[static_cast<size_t>(taps - 1) * channels + c], now, acc);
            if (taps > 1) carried[static_cast<size_t>(taps - 2) * channels + c] = now;
            out[static_cast<size_t>(token) * channels + c] = from_float<T>(acc);
            continue;
        }
        for (int k = 0; k < taps; ++k) {
            const int src = local - (taps - 1) + k;
            const float v = src >= 0 ? x[static_cast<size_t>(token - local + src) * channels + c]
                                     : carried[static_cast<size_t>(taps - 1 + src) * channels + c];
            acc = fmaf(weight[static_cast<size_t>(k) * channels + c], v, acc);
        }
        out[static_cast<size_t>(token) * channels + c] = from_float<T>(acc);
    }
}

// The same sums, four consecutive channels a thread with 16-byte loads of x and of the carried rows (a prompt's
// portion: the kernel is bound by what it moves).  Channels, the carried rows' offset and the state's row are
// multiples of four floats.
template <typename T>
__global__ void __launch_bounds__(256)
stream_conv_four_kernel(const float* __restrict__ x, const float* __restrict__ weight, const float* __restrict__ state,
                        long long state_stride, long long carried_offset, const int* __restrict__ token_segment,
                        const int* __restrict__ seg_q_start, const int* __restrict__ state_slots, T* __restrict__ out,
                        int channels, int taps) {
    const int token = blockIdx.x;
    const int seg = token_segment[token];
    const int local = token - seg_q_start[seg];
    const float* carried = state + static_cast<size_t>(state_slots[seg]) * state_stride + carried_offset;
    for (int c = (blockIdx.y * blockDim.x + threadIdx.x) * 4; c < channels; c += gridDim.y * blockDim.x * 4) {
        const float4 now = *reinterpret_cast<const float4*>(x + static_cast<size_t>(token) * channels + c);
        float acc[4] = {now.x, now.y, now.z, now.w};
        for (int k = 0; k < taps; ++k) {
            const int src = local - (taps - 1) + k;
            const float4 v = *reinterpret_cast<const float4*>(
                src >= 0 ? x + static_cast<size_t>(token - local + src) * channels + c
                         : carried + static_cast<size_t>(taps - 1 + src) * channels + c);
            const float4 w = *reinterpret_cast<const float4*>(weight + static_cast<size_t>(k) * channels + c);
            acc[0] = fmaf(w.x, v.x, acc[0]);
            acc[1] = fmaf(w.y, v.y, acc[1]);
            acc[2] = fmaf(w.z, v.z, acc[2]);
            acc[3] = fmaf(w.w, v.w, acc[3]);
        }
        ConvFour<T> r;
#pragma unroll
        for (int u = 0; u < 4; ++u) r.v[u] = from_float<T>(acc[u]);
        *reinterpret_cast<ConvFour<T>*>(out + static_cast<size_t>(token) * channels + c) = r;
    }
}

// The same for convolutions of kSlideTaps taps over many tokens: every row of x read once (see `slide`;
// 2,048 channels of 3,001 tokens: 19.2 to 9.5 us).
template <typename T>
__global__ void __launch_bounds__(256)
stream_conv_slide_kernel(const float* __restrict__ x, const float* __restrict__ weight, float* __restrict__ state,
                         long long state_stride, long long carried_offset, const int* __restrict__ token_segment,
                         const int* __restrict__ seg_q_start, const int* __restrict__ seg_q_len,
                         const int* __restrict__ state_slots, T* __restrict__ out, int tokens, int channels) {
    const int c = (blockIdx.y * 256 + threadIdx.x) * 4, token0 = blockIdx.x * kSlideTokens;
    if (c >= channels) return;
    float4 w[kSlideTaps];
#pragma unroll
    for (int k = 0; k < kSlideTaps; ++k) w[k] = *reinterpret_cast<const float4*>(weight + static_cast<size_t>(k) * channels + c);
    slide(x + c, static_cast<long long>(channels), state, state_stride, carried_offset + c, token_segment, seg_q_start, seg_q_len,
          state_slots, channels, token0, tokens, [&](int token, const float4 (&rows)[kSlideTaps]) {
        float4 acc = rows[kSlideTaps - 1];
#pragma unroll
        for (int k = 0; k < kSlideTaps; ++k) {
            acc.x = fmaf(w[k].x, rows[k].x, acc.x);
            acc.y = fmaf(w[k].y, rows[k].y, acc.y);
            acc.z = fmaf(w[k].z, rows[k].z, acc.z);
            acc.w = fmaf(w[k].w, rows[k].w, acc.w);
        }
        ConvFour<T> r;
        r.v[0] = from_float<T>(acc.x);
        r.v[1] = from_float<T>(acc.y);
        r.v[2] = from_float<T>(acc.z);
        r.v[3] = from_float<T>(acc.w);
        *reinterpret_cast<ConvFour<T>*>(out + static_cast<size_t>(token) * channels + c) = r;
    });
}

WLLM_API int wllm_stream_conv(const float* x, const float* weight, float* state, long long state_stride,
                              long long carried_offset, const int* token_segment, const int* seg_q_start,
                              const int* seg_q_len, const int* state_slots, void* out, int out_bf16, int tokens,
                              int segments, int channels, int taps, int single_tokens, hipStream_t stream) {
    if (tokens <= 0 || segments <= 0) return 0;
    if (channels <= 0 || taps < 1 || taps > 64) return -1;
    if (single_tokens && tokens != segments) return -1;      // `single_tokens`: every segment is one token
    const int tiles = (channels + 255) / 256 < 64 ? (channels + 255) / 256 : 64;
    const dim3 grid(tokens, tiles), carry_grid(segments, tiles);
    const bool four = !single_tokens && channels % 4 == 0 && state_stride % 4 == 0 && carried_offset % 4 == 0 &&
                      reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(state) % 16 == 0 &&
                      reinterpret_cast<uintptr_t>(weight) % 16 == 0 &&
                      reinterpret_cast<uintptr_t>(out) % 16 == 0;
    if (four) {
        const dim3 grid4(tokens, (channels / 4 + 255) / 256);
        const dim3 slide_grid((tokens + kSlideTokens - 1) / kSlideTokens, (channels / 4 + 255) / 256);
        // (the kernel that it replaces reads in fours too, and its chain is no shorter: beside many single tokens only, 2,048
        // channels of 60 and a segment of 448, 6.2 us and here 6.8, 6,144 channels of them 14.6 and 11.2)
        if (taps == kSlideTaps && slides(tokens, segments, channels, tokens >= 16LL * segments ? 0 : 1 << 21)) {
            if (out_bf16)
                stream_conv_slide_kernel<bf16><<<slide_grid, 256, 0, stream>>>(x, weight, state, state_stride, carried_offset,
                                                                               token_segment, seg_q_start, seg_q_len, state_slots,
                                                                               static_cast<bf16*>(out), tokens, channels);
            else
                stream_conv_slide_kernel<float><<<slide_grid, 256, 0, stream>>>(x, weight, state, state_stride, carried_offset,
                                                                                token_segment, seg_q_start, seg_q_len, state_slots,
                                                                                static_cast<float*>(out), tokens, channels);
            return launch_status();
        }
        if (out_bf16)
            stream_conv_four_kernel<bf16><<<grid4, 256, 0, stream>>>(x, weight, state, state_stride, carried_offset,
                                                                     token_segment, seg_q_start, state_slots,
                                                                     static_cast<bf16*>(out), channels, taps);
        else
            stream_conv_four_kernel<float><<<grid4, 256, 0, stream>>>(x, weight, state, state_stride, carried_offset,
                                                                      token_segment, seg_q_start, state_slots,
                                                                      static_cast<float*>(out), channels, taps);
        if (const int err = launch_status()) return err;
        if (taps == 1) return 0;
        conv_carry_kernel<float><<<carry_grid, 256, 0, stream>>>(x, channels, state, state_stride, carried_offset, seg_q_start,
                                                                 seg_q_len, state_slots, channels, taps);
        return launch_status();
    }
#define LAUNCH(T, CARRY)                                                                                              \
    stream_conv_kernel<T, CARRY><<<grid, 256, 0, stream>>>(x, weight, state, state_stride, carried_offset, token_segment, \
                                                           seg_q_start, state_slots, static_cast<T*>(out), channels, taps)
    if (out_bf16) { if (single_tokens) LAUNCH(bf16, true); else LAUNCH(bf16, false); }
    else { if (single_tokens) LAUNCH(float, true); else LAUNCH(float, false); }
#undef LAUNCH
    if (const int err = launch_status()) return err;
    if (taps == 1 || single_tokens) return 0;
    conv_carry_kernel<float><<<carry_grid, 256, 0, stream>>>(x, channels, state, state_stride, carried_offset, seg_q_start,
                                                             seg_q_len, state_slots, channels, taps);
    return launch_status();
}

// ---- the recurrence.  Per head h (group g = h / (heads / groups)), token by token:
//   dt = softplus(dt_in + dt_bias[h]);  S = exp(-exp(A_log[h]) * dt) * S + dt * B_t x_t^T;  y_t = S^T C_t + D[h] x_t
// with S [N, P], B_t and C_t [N] of the group, x_t [P] of the head.  xbc [tokens, heads*P + 2*groups*N]
// holds x, then B, then C.  The step sizes and decays of all tokens and heads are made first, by a
// kernel of their own (`ssm_steps_kernel`: softplus and two exponentials a value, out of the token
// loop).  Then a workgroup owns (head, segment, 16 columns of P) and walks the segment's tokens in
// order.  N is cut into 32 slices: a lane is (column, one of four slices), a wavefront four slices,
// the workgroup's eight wavefronts all of them; a lane keeps its R rows of its column of S in
// registers.  So a head of 64 columns is four workgroups, a prompt's 64 heads fill 256 compute units
// with two wavefronts a SIMD (one multiplies while the other waits for shared memory), and a lane's
// chain of dependent multiply-adds a token is R long (4 at N = 128).  Measured at 64 heads of 64 with
// 128 rows of state, a prompt of 2,048 tokens / 64 decoded tokens / 8 portions of 256: four wavefronts
// a workgroup 787 / 83 / 290 us, eight 572 / 88 / 291, sixteen 682 / 113 / 466; eight with 32 tokens a
// chunk 564 / 105 / 335; 8 columns a workgroup (a lane's 32 bytes of a row of S are half a memory
// transaction) 654 / 134 / 409.  Tokens are staged 16 at a time through shared memory
// (B, C, x, step, decay), the next 16 fetched into registers meanwhile; a token's y is the slices'
// partial sums added in a fixed order (within the wavefront, then wavefront by wavefront), so it has
// the same bits whether the token came alone or inside a prompt.  In float32 it takes every segment; in bfloat16 those of
// fewer than `shorter_than` tokens, the others being walked in chunks further down, which add in another order. ----
constexpr int kScanTokens = 16;
constexpr int kScanWaves = 8;
constexpr int kScanCols = 16;                       // columns of P a workgroup owns
constexpr int kScanLaneSlices = kWave / kScanCols;  // slices of N side by side in a wavefront
constexpr int kScanSlices = kScanWaves * kScanLaneSlices;
constexpr int kScanFetchers = kWave * kScanWaves / kScanTokens;    // threads that fetch one token's B, C and x of a chunk
static_assert(kScanFetchers >= kScanCols && (kScanLaneSlices == 4 || kScanLaneSlices == 8),
              "a token's fetchers cover its columns of x; the lane sums below are for 4 or 8 slices");

__device__ __forceinline__ float softplus(float z) { return fmaxf(z, 0.f) + log1pf(expf(-fabsf(z))); }

// steps[0][t][h] = softplus(dt_in[t][h] + dt_bias[h]); steps[1][t][h] = exp(-exp(a_log[h]) * steps[0][t][h])
template <typename T>
__global__ void ssm_steps_kernel(const T* __restrict__ dt_in, long long dt_stride, const float* __restrict__ dt_bias,
                                 const float* __restrict__ a_log, float* __restrict__ steps, int tokens, int heads) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= tokens * heads) return;
    const int t = e / heads, h = e - t * heads;
    const float dt = softplus(to_float(dt_in[static_cast<size_t>(t) * dt_stride + h]) + dt_bias[h]);
    steps[e] = dt;
    steps[static_cast<size_t>(tokens) * heads + e] = expf(-expf(a_log[h]) * dt);
}

// VEC: N is a multiple of 4 and so is R, so a lane's rows of B and C are runs of float4 in shared memory.
// F: elements of B (of C) one of a token's 16 fetchers brings.
template <typename T, int R, int F, bool VEC>
__global__ void __launch_bounds__(kWave * kScanWaves)
ssm_scan_kernel(const T* __restrict__ xbc, const float* __restrict__ steps, int tokens,
                const float* __restrict__ d_skip, float* __restrict__ state, long long state_stride, const int* __restrict__ seg_q_start,
                const int* __restrict__ seg_q_len, const int* __restrict__ state_slots, float* __restrict__ y, int heads,
                int groups, int n_state, int p_dim, int shorter_than) {
    extern __shared__ __align__(16) float smem[];
    const int h = blockIdx.x, seg = blockIdx.y, p0 = blockIdx.z * kScanCols;
    const int q_len = seg_q_len[seg], q_start = seg_q_start[seg];
    if (q_len <= 0 || q_len >= shorter_than) return;
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int col = lane % kScanCols, slice = wave * kScanLaneSlices + lane / kScanCols;
    const int p = p0 + col;
    const bool live = p < p_dim;
    const int g = h / (heads / groups);
    const int inner = heads * p_dim, channels = inner + 2 * groups * n_state;
    const int b_col = inner + g * n_state, c_col = inner + groups * n_state + g * n_state;
    const int n_pad = (n_state + 3) / 4 * 4;             // a token's row of B (of C) in shared memory
    float* b_s = smem;                                   // [kScanTokens][n_pad]
    float* c_s = b_s + kScanTokens * n_pad;              // [kScanTokens][n_pad]
    float* x_s = c_s + kScanTokens * n_pad;              // [kScanTokens][kScanCols]
    float* dt_s = x_s + kScanTokens * kScanCols;         // [kScanTokens]
    float* decay_s = dt_s + kScanTokens;                 // [kScanTokens]
    float* part_s = decay_s + kScanTokens;               // [kScanTokens][kScanWaves][kScanCols]
    float* s_rows = state + static_cast<size_t>(state_slots[seg]) * state_stride + static_cast<size_t>(h) * n_state * p_dim;
    const int n0 = slice * R;
    float s[R];
#pragma unroll
    for (int i = 0; i < R; ++i) s[i] = (live && n0 + i < n_state) ? s_rows[static_cast<size_t>(n0 + i) * p_dim + p] : 0.f;
    const float skip = d_skip[h];
    // What a thread fetches of a chunk of 16 tokens, into registers while the chunk before is worked on:
    // of token `ft` of the chunk, F elements of B and of C (thread = 16 ft + fq takes the fq-th run), one
    // element of x, and (the first 16 threads) a token's step size and decay.
    const int ft = threadIdx.x / kScanFetchers, fq = threadIdx.x % kScanFetchers;
    float pb[F], pc[F], px = 0.f, pdt = 0.f, pdecay = 0.f;
    auto fetch = [&](int t0) {
        const int count = min(kScanTokens, q_len - t0);
        if (ft < count) {
            const T* row = xbc + static_cast<size_t>(q_start + t0 + ft) * channels;
#pragma unroll
            for (int i = 0; i < F; ++i) {
                const int n = fq * F + i;
                pb[i] = n < n_state ? to_float(row[b_col + n]) : 0.f;
                pc[i] = n < n_state ? to_float(row[c_col + n]) : 0.f;
            }
            px = (fq < kScanCols && p0 + fq < p_dim) ? to_float(row[h * p_dim + p0 + fq]) : 0.f;
        }
        if (threadIdx.x < count) {
            const size_t at = static_cast<size_t>(q_start + t0 + threadIdx.x) * heads + h;
            pdt = steps[at];
            pdecay = steps[static_cast<size_t>(tokens) * heads + at];
        }
    };
    fetch(0);
    for (int t0 = 0; t0 < q_len; t0 += kScanTokens) {
        const int count = min(kScanTokens, q_len - t0);
        __syncthreads();                                 // the chunk before is read out
        if (ft < count) {
#pragma unroll
            for (int i = 0; i < F; ++i) {
                const int n = fq * F + i;
                if (n < n_pad) {
                    b_s[ft * n_pad + n] = pb[i];
                    c_s[ft * n_pad + n] = pc[i];
                }
            }
            if (fq < kScanCols) x_s[ft * kScanCols + fq] = px;
        }
        if (threadIdx.x < count) {
            dt_s[threadIdx.x] = pdt;
            decay_s[threadIdx.x] = pdecay;
        }
        __syncthreads();
        if (t0 + kScanTokens < q_len) fetch(t0 + kScanTokens);      // in flight while this chunk is worked on
        // (unrolled: a token's reads of shared memory are asked for while the token before it is multiplied)
#pragma unroll 4
        for (int t = 0; t < count; ++t) {
            const float decay = decay_s[t], dx = dt_s[t] * x_s[t * kScanCols + col];
            const float* bt = b_s + t * n_pad + n0;
            const float* ct = c_s + t * n_pad + n0;
            float part = 0.f;
            if (VEC) {
#pragma unroll
                for (int i = 0; i < R; i += 4) {
                    if (n0 + i < n_state) {              // whole groups of four: N and R are multiples of 4
                        const float4 bv = *reinterpret_cast<const float4*>(bt + i), cv = *reinterpret_cast<const float4*>(ct + i);
                        s[i] = fmaf(decay, s[i], dx * bv.x);
                        s[i + 1] = fmaf(decay, s[i + 1], dx * bv.y);
                        s[i + 2] = fmaf(decay, s[i + 2], dx * bv.z);
                        s[i + 3] = fmaf(decay, s[i + 3], dx * bv.w);
                        part = fmaf(s[i], cv.x, part);
                        part = fmaf(s[i + 1], cv.y, part);
                        part = fmaf(s[i + 2], cv.z, part);
                        part = fmaf(s[i + 3], cv.w, part);
                    }
                }
            } else {
#pragma unroll
                for (int i = 0; i < R; ++i) {
                    if (n0 + i < n_state) {
                        s[i] = fmaf(decay, s[i], dx * bt[i]);
                        part = fmaf(s[i], ct[i], part);
                    }
                }
            }
            // the wavefront's slices of this column, in a fixed order
            part = sum_across(sum_across(part, 32), 16);
            if (kScanLaneSlices == 8) part += row_permuted<0x128>(part);
            if (lane < kScanCols) part_s[(t * kScanWaves + wave) * kScanCols + col] = part;
        }
        __syncthreads();
        for (int e = threadIdx.x; e < count * kScanCols; e += blockDim.x) {
            const int t = e / kScanCols, l = e % kScanCols;
            if (p0 + l >= p_dim) continue;
            float total = part_s[(t * kScanWaves) * kScanCols + l];
#pragma unroll
            for (int w = 1; w < kScanWaves; ++w) total += part_s[(t * kScanWaves + w) * kScanCols + l];
            total = fmaf(skip, x_s[e], total);
            y[static_cast<size_t>(q_start + t0 + t) * inner + h * p_dim + p0 + l] = total;
        }
    }
    if (live) {
#pragma unroll
        for (int i = 0; i < R; ++i)
            if (n0 + i < n_state) s_rows[static_cast<size_t>(n0 + i) * p_dim + p] = s[i];
    }
}

// ---- the same recurrence over many tokens, 16 at a time on the matrix cores.  With f_t, d_t the decay and the step of
// a head's token t, pre_t the product of a chunk's decays up to t, and suf_s that of the decays behind s,
//   y_t = pre_t (C_t . S0) + sum over s <= t of N_ts x_s + D x_t,   S = pre_16 S0 + B^T (suf_s d_s x_s),
//   N_ts = (C_t . B_s) (the decays s < r <= t) d_s.
// bfloat16 inputs only: in the 32-bit path a token's bits do not depend on how its prompt was cut.
// A product of decays is formed from the decays it is made of (never as a quotient or a difference of logarithms), so
// the numbers are those of the walk token by token up to the order of float32 sums.  Nothing but S0 depends on the
// tokens before, so `ssm_chunk_kernel` makes all else for every chunk at once: per (chunk, group) the rows C_t and the
// transposed B, per (chunk, head) N, pre, suf d and pre_16; and `ssm_chunk_scan_kernel` walks a segment's chunks with
// v_mfma_f32_16x16x4_f32 (float32 in and out), 17 of them a wavefront and chunk.  A chunk begins every 16 tokens of a
// segment; the last one is filled with tokens that change nothing (d = 0, f = 1, B = C = 0).
// The walk token by token is bound by its chain (0.27 us a token).  64 heads of 64 with 128 rows of state: 1,500 tokens
// 410 us token by token, 13 and 73 us for the two kernels here (a chunk takes 0.75 us, of which the products are a third);
// 64 tokens 21 us against 7 and 9, one line between the two ways; of more heads a group it lies further on. ----
constexpr int kChunkHeadFloats = kChunk * kChunk + 3 * kChunk;       // N, pre, suf d, pre_16 (and padding)

// The operands of a chunk and a group: 28 us at 8 heads a group with a thread an entry of N that multiplied its decays one
// after the other as it read them, 7 (6 chunks) to 13 (95) with a head a wavefront, a lane's 16 decays read at once and the products C_t . B_s
// on the matrix cores.
typedef float ssm_float4 __attribute__((ext_vector_type(4)));

template <int TILES>        // C = 64 TILES: the rows of state, padded
__global__ void __launch_bounds__(256)
ssm_chunk_kernel(const bf16* __restrict__ xbc, const bf16* __restrict__ dt_in, long long dt_stride, const float* __restrict__ dt_bias,
                 const float* __restrict__ a_log, const int* __restrict__ seg_q_start, const int* __restrict__ seg_q_len,
                 int segments, float* __restrict__ of_head, bf16* __restrict__ of_group, int heads, int groups, int n_state,
                 int p_dim, int from) {
    constexpr int C = 64 * TILES, kRow = C + 4;
    __shared__ __align__(16) float b_s[kChunk * kRow], c_s[kChunk * kRow];
    __shared__ __align__(16) float f_s[kChunk][kChunk], dt_s[kChunk][kChunk];          // [head of sixteen][token]
    __shared__ ssm_float4 g_s[4][kWave];
    __shared__ int found;
    const int place = blockIdx.x, g = blockIdx.y, tid = threadIdx.x;
    if (tid == 0) found = -1;
    __syncthreads();
    for (int s = tid; s < segments; s += 256) {
        const int first = first_place(seg_q_start[s], from), len = seg_q_len[s];
        if (len >= from && place >= first && place < first + (len + kChunk - 1) / kChunk) found = s;
    }
    __syncthreads();
    const int seg = found;
    if (seg < 0) return;
    const int q_start = seg_q_start[seg], local = (place - first_place(q_start, from)) * kChunk;
    const int count = min(kChunk, seg_q_len[seg] - local), token = q_start + local;
    const int inner = heads * p_dim, channels = inner + 2 * groups * n_state;
    const int b_col = inner + g * n_state, c_col = b_col + groups * n_state;
    bf16* rows = of_group + (static_cast<size_t>(place) * groups + g) * 2 * kChunk * C;
    constexpr int kEach = kChunk * C / 256;
    bf16 b[kEach], c[kEach];
#pragma unroll
    for (int k = 0; k < kEach; ++k) {
        const int t = (tid + 256 * k) / C, n = (tid + 256 * k) % C;
        const bf16* row = xbc + static_cast<size_t>(token + min(t, count - 1)) * channels + min(n, n_state - 1);
        b[k] = row[b_col];
        c[k] = row[c_col];
    }
#pragma unroll
    for (int k = 0; k < kEach; ++k) {
        const int t = (tid + 256 * k) / C, n = (tid + 256 * k) % C;
        const bool there = t < count && n < n_state;
        const bf16 bv = there ? b[k] : from_float<bf16>(0.f), cv = there ? c[k] : from_float<bf16>(0.f);
        b_s[t * kRow + n] = to_float(bv);
        c_s[t * kRow + n] = to_float(cv);
        rows[tid + 256 * k] = cv;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kEach; ++k) {
        const int e = tid + 256 * k;
        rows[kChunk * C + e] = from_float<bf16>(b_s[e % kChunk * kRow + e / kChunk]);
    }
    const int lane = tid % kWave, wave = tid / kWave, i = lane % 16, q = lane / 16;
    {
        // lane (i, q) takes what every wavefront's quarter of the rows gives of B_s . C_t for t = i, s = 4q .. 4q + 3
        ssm_float4 part = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < TILES; ++j) {
            const int n = (wave * TILES + j) * 16 + 4 * q;
            const ssm_float4 bv = *reinterpret_cast<const ssm_float4*>(b_s + i * kRow + n);
            const ssm_float4 cv = *reinterpret_cast<const ssm_float4*>(c_s + i * kRow + n);
#pragma unroll
            for (int u = 0; u < 4; ++u) part = __builtin_amdgcn_mfma_f32_16x16x4f32(bv[u], cv[u], part, 0, 0, 0);
        }
        g_s[wave][lane] = part;
    }
    const int per_group = heads / groups;
    for (int h0 = 0; h0 < per_group; h0 += kChunk) {
        {
            const int hh = tid / kChunk, t = tid % kChunk, h = g * per_group + h0 + hh;
            float step = 0.f, decay = 1.f;
            if (h0 + hh < per_group && t < count) {
                step = softplus(to_float(dt_in[static_cast<size_t>(token + t) * dt_stride + h]) + dt_bias[h]);
                decay = expf(-expf(a_log[h]) * step);
            }
            if (h0 > 0) __syncthreads();                  // the sixteen heads before are done with
            dt_s[hh][t] = step;
            f_s[hh][t] = decay;
        }
        __syncthreads();
        ssm_float4 dot = g_s[0][lane];
#pragma unroll
        for (int w = 1; w < 4; ++w) dot += g_s[w][lane];
        for (int hh = wave; hh < min(kChunk, per_group - h0); hh += 4) {
            float* out = of_head + (static_cast<size_t>(place) * heads + g * per_group + h0 + hh) * kChunkHeadFloats;
            float f[kChunk];
#pragma unroll
            for (int r = 0; r < kChunk; r += 4) *reinterpret_cast<ssm_float4*>(f + r) = *reinterpret_cast<const ssm_float4*>(&f_s[hh][r]);
            const ssm_float4 step = *reinterpret_cast<const ssm_float4*>(&dt_s[hh][4 * q]);
            // the decays between s and t = i for s = 4q + 3, and from there down.  (Products in 64 bits, rounded once: a
            // whole row of sums shares their error, where the walk token by token rounds every element for itself.)
            double between = 1.0;
#pragma unroll
            for (int r = 4; r < kChunk; ++r) between *= r > 4 * q + 3 && r <= i ? f[r] : 1.f;
            ssm_float4 n;
#pragma unroll
            for (int u = 3; u >= 0; --u) {
                const int s = 4 * q + u;
                n[u] = s <= i ? dot[u] * static_cast<float>(between * step[u]) : 0.f;
                between *= s <= i ? f_s[hh][s] : 1.f;
            }
            *reinterpret_cast<ssm_float4*>(out + i * kChunk + 4 * q) = n;
            // lanes of q = 0: the decays up to token i; of q = 1: those behind it, times its step; of q = 2: all of them
            double v = q == 1 ? dt_s[hh][i] : 1.f;
#pragma unroll
            for (int r = 0; r < kChunk; ++r) v *= q == 2 || (q == 0 ? r <= i : r > i) ? f[r] : 1.f;
            if (q < 3) out[kChunk * kChunk + q * kChunk + i] = static_cast<float>(v);
        }
    }
}

// A workgroup owns (head, segment, 16 columns of P); its first four wavefronts cut the rows of state, each with TILES tiles of
// 16: lane (i, g) holds the rows 4g .. 4g + 3 of a tile in column i, which is what a product leaves and, row by row, what
// it takes (the k-th of four products takes the rows 4g + k), so the state never moves between lanes.  They keep the state and read it for
// every chunk; what is left of a chunk's results (the part that its own tokens make, the sum over the wavefronts, the stores) is the other four's, a chunk
// and two chunks behind, beside them on their SIMDs.  One barrier a chunk, two places of shared memory in turn.  The operands of a chunk are asked
// for kAhead chunks before they are used, while the products that free their registers run.
// What bounds it: the chain of a chunk in one wavefront, of which the products (32 clocks each, 8 TILES) should be all
// (16 of them 0.25 us of a chunk's 0.7; with the other wavefronts' work in the same chain 83 us for 1,500 tokens of 64 heads of 64 with 128 rows of state, now
// 73; without the loads of B and C and their conversions 52).
struct alignas(8) SsmFour { bf16 v[4]; };

template <int TILES>
__global__ void __launch_bounds__(512, TILES <= 2 ? 4 : 2)
ssm_chunk_scan_kernel(const float* of_head, const bf16* of_group, const bf16* xbc, const float* __restrict__ d_skip,
                      float* __restrict__ state, long long state_stride, const int* __restrict__ seg_q_start,
                      const int* __restrict__ seg_q_len, const int* __restrict__ state_slots, float* __restrict__ y, int heads,
                      int groups, int n_state, int p_dim, int from) {
    constexpr int C = 64 * TILES, kAhead = 3, kOwnAhead = 6;
    __shared__ ssm_float4 read_s[2][4][kWave], part_s[2][4][kWave];
    const int h = blockIdx.x, seg = blockIdx.y, p0 = blockIdx.z * 16;
    const int q_len = seg_q_len[seg], q_start = seg_q_start[seg];
    if (q_len < from) return;
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave) % 4;
    const bool keeps = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave) < 4;
    const int i = lane % 16, g = lane / 16;
    const int p = p0 + i;
    const bool live = p < p_dim;
    const int inner = heads * p_dim, channels = inner + 2 * groups * n_state;
    const size_t first = static_cast<size_t>(first_place(q_start, from));
    const unsigned col = static_cast<unsigned>(min(p, p_dim - 1)), x_row = 2 * static_cast<unsigned>(channels);
    // Where the next chunk's operands lie: addresses that are the same in all lanes, moved on by a sum a chunk (and not beyond the last chunk); a lane's
    // offsets beside them are bytes in 32 bits.  (Worked out from the chunk's number: 76 us a scan, now 73.)
    struct Place {
        const char *x, *of, *rows;
        int left;                                        // tokens from this chunk on
    };
    auto move_on = [&](Place& at) __attribute__((always_inline)) {
        const bool more = at.left > kChunk;
        at.x += more ? static_cast<size_t>(kChunk) * x_row : 0;
        at.of += more ? static_cast<size_t>(heads) * kChunkHeadFloats * sizeof(float) : 0;
        at.rows += more ? static_cast<size_t>(groups) * 2 * kChunk * C * sizeof(bf16) : 0;
        at.left -= more ? kChunk : 0;
    };
    // (beyond the last token, that token's once more: what it is multiplied by is zero)
    auto x_of = [&](const Place& at, unsigned row_at) __attribute__((always_inline)) {
        return *reinterpret_cast<const bf16*>(at.x + (min(row_at, static_cast<unsigned>(min(kChunk, at.left) - 1) * x_row) + 2 * col));
    };
    Place next = {reinterpret_cast<const char*>(xbc + static_cast<size_t>(q_start) * channels + h * p_dim),
                  reinterpret_cast<const char*>(of_head + (first * heads + h) * kChunkHeadFloats),
                  reinterpret_cast<const char*>(of_group + (first * groups + h / (heads / groups)) * 2 * kChunk * C), q_len};
    const int count = (q_len + kChunk - 1) / kChunk;
    // (a barrier for what lies in shared memory alone: the operands of the chunks ahead stay on their way)
    auto meet = [&]() __attribute__((always_inline)) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    if (!keeps) {
        // wavefront w: the part of the tokens 4g + w as keys, then their sums
        const float skip = d_skip[h];
        float* y_first = y + static_cast<size_t>(q_start) * inner + h * p_dim;
        struct Own { ssm_float4 pre; float n; bf16 x; };
        const unsigned n_at = 4 * (i * kChunk + 4 * g + wave), pre_at = 4 * (kChunk * kChunk + 4 * g), x_at = (4 * g + wave) * x_row;
        auto load = [&]() __attribute__((always_inline)) {
            const Own o = {*reinterpret_cast<const ssm_float4*>(next.of + pre_at), *reinterpret_cast<const float*>(next.of + n_at), x_of(next, x_at)};
            move_on(next);
            return o;
        };
        float mine[2];
        auto add_own = [&](int c, int place, const Own& now) __attribute__((always_inline)) {
            mine[place] = c * kChunk + 4 * g + wave < q_len ? to_float(now.x) : 0.f;
            part_s[place][wave][lane] = add_causal_product(now.n, mine[place], read_s[place][wave][lane] * now.pre, i, g, [&](int q) { return 4 * q + wave; });
        };
        auto finish = [&](int c, int place) __attribute__((always_inline)) {
            const float* parts = reinterpret_cast<const float*>(&part_s[place][0][lane]) + wave;
            float o = parts[0];
#pragma unroll
            for (int w = 1; w < 4; ++w) o += parts[w * 4 * kWave];
            const int t = 4 * g + wave;
            if (live && c * kChunk + t < q_len)
                (y_first + static_cast<size_t>(c) * kChunk * inner)[t * static_cast<unsigned>(inner) + col] = fmaf(skip, mine[place], o);
        };
        // (kOwnAhead chunks ahead: a wait for these loads is one for the stores in front of them, too)
        Own ring[kOwnAhead];
#pragma unroll
        for (int a = 0; a < kOwnAhead; ++a) {
            ring[a] = load();
            __builtin_amdgcn_sched_barrier(0);           // (in this order, which the waits of the loop count on)
        }
        auto step = [&](int c, int a) __attribute__((always_inline)) {
            add_own(c + a, a % 2, ring[a]);
            __builtin_amdgcn_sched_barrier(0);
            ring[a] = load();
            __builtin_amdgcn_sched_barrier(0);
            if (c + a > 0) finish(c + a - 1, 1 - a % 2);
            meet();
        };
        meet();                                                              // chunk 0 has read the state
        int c = 0;
        for (; c + kOwnAhead <= count; c += kOwnAhead) {
#pragma unroll
            for (int a = 0; a < kOwnAhead; ++a) step(c, a);
        }
#pragma unroll
        for (int a = 0; a < kOwnAhead - 1; ++a)
            if (c + a < count) step(c, a);
        if (count % 2) finish(count - 1, 0);
        else finish(count - 1, 1);
        return;
    }
    float* s_rows = state + static_cast<size_t>(state_slots[seg]) * state_stride + static_cast<size_t>(h) * n_state * p_dim + p;
    const int n0 = wave * 16 * TILES;
    ssm_float4 s[TILES];
#pragma unroll
    for (int j = 0; j < TILES; ++j)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int n = n0 + 16 * j + 4 * g + u;
            s[j][u] = live && n < n_state ? s_rows[static_cast<size_t>(n) * p_dim] : 0.f;
        }
    struct Operands {
        SsmFour c[TILES], b[TILES];
        ssm_float4 suf;
        float all;
        bf16 x[4];
    };
    // where this lane's operands lie in a chunk's, in bytes
    const unsigned c_at = 2 * (i * C + n0 + 4 * g), b_at = 2 * (kChunk * C + (n0 + i) * kChunk + 4 * g), suf_at = 4 * (kChunk * kChunk + kChunk + 4 * g);
    unsigned x_at[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) x_at[u] = (4 * g + u) * x_row;
    auto load = [&]() __attribute__((always_inline)) {
        Operands o;
#pragma unroll
        for (int u = 0; u < 4; ++u) o.x[u] = x_of(next, x_at[u]);
        o.suf = *reinterpret_cast<const ssm_float4*>(next.of + suf_at);
        o.all = *reinterpret_cast<const float*>(next.of + 4 * (kChunk * kChunk + 2 * kChunk));
#pragma unroll
        for (int j = 0; j < TILES; ++j) {
            o.c[j] = *reinterpret_cast<const SsmFour*>(next.rows + c_at + 32 * j);
            o.b[j] = *reinterpret_cast<const SsmFour*>(next.rows + b_at + 32 * kChunk * j);
        }
        move_on(next);
        return o;
    };
    auto walk = [&](int c, Operands& now) __attribute__((always_inline)) {
        ssm_float4 x, read[TILES];
#pragma unroll
        for (int u = 0; u < 4; ++u) x[u] = c * kChunk + 4 * g + u < q_len ? to_float(now.x[u]) : 0.f;
        // (a sum a tile, added in the end: short chains of products, and of roundings)
#pragma unroll
        for (int j = 0; j < TILES; ++j) read[j] = ssm_float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int j = 0; j < TILES; ++j)
                read[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(to_float(now.c[j].v[u]), s[j][u], read[j], 0, 0, 0);
        const ssm_float4 moved = x * now.suf;
        const float all = now.all;
        // (the chunk's own sum first, from zero, and the state joins it with one rounding a chunk)
        ssm_float4 own[TILES];
#pragma unroll
        for (int j = 0; j < TILES; ++j) own[j] = ssm_float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int j = 0; j < TILES; ++j)
                own[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(to_float(now.b[j].v[u]), moved[u], own[j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        now = load();
        __builtin_amdgcn_sched_barrier(0);
        ssm_float4 part = read[0];
#pragma unroll
        for (int j = 1; j < TILES; ++j) part += read[j];
        read_s[c % 2][wave][lane] = part;                                    // a wavefront's part: its rows of the state
#pragma unroll
        for (int j = 0; j < TILES; ++j)
#pragma unroll
            for (int u = 0; u < 4; ++u) s[j][u] = fmaf(all, s[j][u], own[j][u]);
        meet();
    };
    // the operands of kAhead chunks in turn (beyond the last chunk: the last's once more).  The loads stay where they are
    // written: the scratch and xbc may alias y as far as the compiler knows, and the empty statements touch memory.
    Operands ring[kAhead];
#pragma unroll
    for (int d = 0; d < kAhead; ++d) {
        ring[d] = load();
        __builtin_amdgcn_sched_barrier(0);               // (in this order, which the waits of the loop count on)
    }
    int c = 0;
    for (; c + kAhead <= count; c += kAhead) {
#pragma unroll
        for (int d = 0; d < kAhead; ++d) walk(c + d, ring[d]);
    }
#pragma unroll
    for (int d = 0; d < kAhead - 1; ++d)
        if (c + d < count) walk(c + d, ring[d]);
    meet();                                                                  // the others' last sums
#pragma unroll
    for (int j = 0; j < TILES; ++j)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int n = n0 + 16 * j + 4 * g + u;
            if (live && n < n_state) s_rows[static_cast<size_t>(n) * p_dim] = s[j][u];
        }
}

// `steps`: scratch of 2 * tokens * heads floats (the step sizes, then the decays).  `from` tokens (16 at least; 0: no
// segment, as in float32) is what a segment needs to be walked in chunks, out of the scratch `chunks`: `chunk_places`
// places, first [place][head] of kChunkHeadFloats floats, then [place][group] of
// 32 x (the rows of state padded to a multiple of 64) elements.  `shortest`: the caller's word that no segment has fewer
// tokens (0: it has none); with it at `from` or above nothing is launched for shorter ones.
WLLM_API int wllm_ssm_scan(const void* xbc, const void* dt_in, long long dt_stride, const float* dt_bias, const float* a_log,
                           const float* d_skip, float* state, long long state_stride, const int* seg_q_start,
                           const int* seg_q_len, const int* state_slots, float* y, float* steps, int is_bf16, int tokens,
                           int segments, int heads, int groups, int n_state, int p_dim, float* chunks, int from, int shortest,
                           hipStream_t stream) {
    if (segments <= 0 || tokens <= 0) return 0;
    if (!steps) return -1;
    if (heads <= 0 || groups <= 0 || heads % groups != 0 || n_state <= 0 || n_state > 16 * kScanSlices || p_dim <= 0) return -1;
    if (segments > 65535 || (p_dim + kScanCols - 1) / kScanCols > 65535) return -1;
    const dim3 grid(heads, segments, (p_dim + kScanCols - 1) / kScanCols);
    // (a segment of `from` tokens leaves room for the others' single tokens)
    // (what the chunks' kernels do not take goes token by token: more channels than 16 rows' bytes in 32 bits allow, too)
    const bool in_chunks = from > 0 && tokens - (segments - 1) >= from && n_state <= 256 && groups <= 65535 &&
                           static_cast<long long>(heads) * p_dim + 2LL * groups * n_state <= 0x07ffffffLL;
    if (in_chunks) {
        if (!is_bf16 || !chunks || from < kChunk || reinterpret_cast<uintptr_t>(chunks) % 16) return -1;
        const int places = chunk_places(tokens, from);
        const dim3 chunk_grid(places, groups);
        bf16* of_group = reinterpret_cast<bf16*>(chunks + static_cast<size_t>(places) * heads * kChunkHeadFloats);
#define LAUNCH(TILES)                                                                                                  \
    do {                                                                                                               \
        ssm_chunk_kernel<TILES><<<chunk_grid, 256, 0, stream>>>(                                                       \
            static_cast<const bf16*>(xbc), static_cast<const bf16*>(dt_in), dt_stride, dt_bias, a_log, seg_q_start, seg_q_len, \
            segments, chunks, of_group, heads, groups, n_state, p_dim, from);                                          \
        if (const int err = launch_status()) return err;                                                               \
        ssm_chunk_scan_kernel<TILES><<<grid, 512, 0, stream>>>(                                                        \
            chunks, of_group, static_cast<const bf16*>(xbc), d_skip, state, state_stride, seg_q_start, seg_q_len, state_slots, y, \
            heads, groups, n_state, p_dim, from);                                                                      \
    } while (0)
        if (n_state <= 64) LAUNCH(1);
        else if (n_state <= 128) LAUNCH(2);
        else if (n_state <= 192) LAUNCH(3);
        else LAUNCH(4);
#undef LAUNCH
        if (const int err = launch_status()) return err;
        if (shortest >= from) return 0;
    }
    const int shorter_than = in_chunks ? from : 0x7fffffff;
    const int r = (n_state + kScanSlices - 1) / kScanSlices;
    {
        const int total = tokens * heads, blocks = (total + 255) / 256;
        if (is_bf16)
            ssm_steps_kernel<bf16><<<blocks, 256, 0, stream>>>(static_cast<const bf16*>(dt_in), dt_stride, dt_bias, a_log, steps,
                                                               tokens, heads);
        else
            ssm_steps_kernel<float><<<blocks, 256, 0, stream>>>(static_cast<const float*>(dt_in), dt_stride, dt_bias, a_log,
                                                                steps, tokens, heads);
        if (const int err = launch_status()) return err;
    }
    const int n_pad = (n_state + 3) / 4 * 4;
    const size_t smem = sizeof(float) * (2 * kScanTokens * n_pad + kScanTokens * kScanCols + 2 * kScanTokens +
                                         kScanTokens * kScanWaves * kScanCols);
#define LAUNCH(T, R, V)                                                                                             \
    ssm_scan_kernel<T, R, (R * kScanSlices + kScanFetchers - 1) / kScanFetchers, V><<<grid, kWave * kScanWaves, smem, stream>>>( \
        static_cast<const T*>(xbc), steps, tokens, d_skip, state, state_stride, seg_q_start, seg_q_len, state_slots, y, \
        heads, groups, n_state, p_dim, shorter_than)
#define LAUNCH_R(T)                                                                          \
    if (r <= 1) LAUNCH(T, 1, false);                                                         \
    else if (r <= 2) LAUNCH(T, 2, false);                                                    \
    else if (r <= 4) { if (n_state % 4 == 0) LAUNCH(T, 4, true); else LAUNCH(T, 4, false); }   \
    else if (r <= 8) { if (n_state % 4 == 0) LAUNCH(T, 8, true); else LAUNCH(T, 8, false); }   \
    else { if (n_state % 4 == 0) LAUNCH(T, 16, true); else LAUNCH(T, 16, false); }
    if (is_bf16) { LAUNCH_R(bf16) } else { LAUNCH_R(float) }
#undef LAUNCH_R
#undef LAUNCH
    return launch_status();
}

// ---- out = rms_norm_in_groups(y * silu(z)) * weight: the recurrence's result (float32) gated by
// z (a band of a wider row, the activation type), then every one of `groups` equal parts of the row
// divided by its own root mean square, times the weight; out in the activation type.  One workgroup
// a (token, part). ----
template <typename T>
__global__ void __launch_bounds__(256)
gated_group_norm_kernel(const float* __restrict__ y, const T* __restrict__ z, long long z_stride,
                        const float* __restrict__ weight, T* __restrict__ out, int width, int groups, float eps) {
    __shared__ float scratch[16];
    const int token = blockIdx.x, part = blockIdx.y;
    const int size = width / groups, c0 = part * size;
    const float* yr = y + static_cast<size_t>(token) * width + c0;
    const T* zr = z + static_cast<size_t>(token) * z_stride + c0;
    float ss = 0.f;
    for (int i = threadIdx.x; i < size; i += blockDim.x) {
        const float zv = to_float(zr[i]);
        const float v = yr[i] * (zv / (1.f + expf(-zv)));
        ss += v * v;
    }
    const float inv = 1.f / sqrtf(block_sum(ss, scratch) / static_cast<float>(size) + eps);
    T* o = out + static_cast<size_t>(token) * width + c0;
    for (int i = threadIdx.x; i < size; i += blockDim.x) {
        const float zv = to_float(zr[i]);
        const float v = yr[i] * (zv / (1.f + expf(-zv)));
        o[i] = from_float<T>(v * inv * weight[c0 + i]);
    }
}

// The same, the same bits, for many (token, part)s of at most 256 PER columns: a wavefront each, which holds its columns in registers and adds them up as
// the four wavefronts above do (lane by lane every 256th column, each 64 lanes by themselves, then those four sums).  No barrier, one pass over memory, and
// all loads at once.  1,500 tokens of 8 parts of 512, bfloat16: 21.5 us and 14.0 (the bytes: 10).
template <typename T, int PER>
__global__ void __launch_bounds__(256)
gated_group_norm_wave_kernel(const float* __restrict__ y, const T* __restrict__ z, long long z_stride, const float* __restrict__ weight,
                             T* __restrict__ out, int width, int groups, float eps) {
    const int lane = threadIdx.x % kWave, part = blockIdx.y * 4 + threadIdx.x / kWave;
    if (part >= groups) return;
    const size_t token = blockIdx.x;
    const int size = width / groups, c0 = part * size;
    const float* yr = y + token * width + c0;
    const T* zr = z + token * z_stride + c0;
    float yv[4][PER], v[4][PER];
    T zv[4][PER];
#pragma unroll
    for (int w = 0; w < 4; ++w)
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int i = min(64 * w + lane + 256 * j, size - 1);
            yv[w][j] = yr[i];
            zv[w][j] = zr[i];
        }
    float total = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        float ss = 0.f;
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const float g = to_float(zv[w][j]);
            v[w][j] = yv[w][j] * (g / (1.f + expf(-g)));
            if (64 * w + lane + 256 * j < size) ss += v[w][j] * v[w][j];
        }
        total += wave_sum(ss);
    }
    const float inv = 1.f / sqrtf(total / static_cast<float>(size) + eps);
    T* o = out + token * width + c0;
#pragma unroll
    for (int w = 0; w < 4; ++w)
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int i = 64 * w + lane + 256 * j;
            if (i < size) o[i] = from_float<T>(v[w][j] * inv * weight[c0 + i]);
        }
}

WLLM_API int wllm_gated_group_norm(const float* y, const void* z, long long z_stride, const float* weight, void* out,
                                   int is_bf16, int tokens, int width, int groups, float eps, hipStream_t stream) {
    if (tokens <= 0) return 0;
    if (width <= 0 || groups <= 0 || width % groups != 0 || groups > 65535) return -1;
    const int size = width / groups;
    // (a wavefront a compute unit's SIMD twice over: of fewer parts the kernel with four wavefronts a part is done sooner)
    if (size <= 1024 && static_cast<long long>(tokens) * groups >= 2048) {
        const dim3 grid(tokens, (groups + 3) / 4);
#define LAUNCH(T, PER)                                                                                                     \
    gated_group_norm_wave_kernel<T, PER><<<grid, 256, 0, stream>>>(y, static_cast<const T*>(z), z_stride, weight,          \
                                                                   static_cast<T*>(out), width, groups, eps)
        if (size <= 256) { if (is_bf16) LAUNCH(bf16, 1); else LAUNCH(float, 1); }
        else if (size <= 512) { if (is_bf16) LAUNCH(bf16, 2); else LAUNCH(float, 2); }
        else { if (is_bf16) LAUNCH(bf16, 4); else LAUNCH(float, 4); }
#undef LAUNCH
        return launch_status();
    }
    const dim3 grid(tokens, groups);
    if (is_bf16)
        gated_group_norm_kernel<bf16><<<grid, 256, 0, stream>>>(y, static_cast<const bf16*>(z), z_stride, weight,
                                                                static_cast<bf16*>(out), width, groups, eps);
    else
        gated_group_norm_kernel<float><<<grid, 256, 0, stream>>>(y, static_cast<const float*>(z), z_stride, weight,
                                                                 static_cast<float*>(out), width, groups, eps);
    return launch_status();
}
