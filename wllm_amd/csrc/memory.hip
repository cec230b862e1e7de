// A recurrent mixer whose state is a matrix a head (linear attention in its recurrent form) on a flat
// batch of segments.  A segment is the next tokens of one request; what a request carries from step to
// step lies in one float32 row of `state` per request (row state_slots[segment]):
//   [heads, D, P] the memory S, then (exponential gating only) [heads, D] the normaliser n and [heads] the
//   running maximum m.
// A fresh request's row is all zeros: S, n and m all start at zero.  Per head and token
//   S_t = a_t S_(t-1) + b_t k_t v_t^T,    o_t = S_t^T q_t / den_t
// with (a, b) either (the head's fixed decay, 1) and den = 1, or made from the two gates by `memory_gates`; then
// the normaliser n_t = a_t n_(t-1) + b_t k_t is one more column of the memory (a value that is always 1), the
// recurrence leaves n_t . q_t beside the columns' sums, and den_t = max(|n_t . q_t|, exp(-m_t)) + eps divides them
// where the heads are normed (`head_norm_gate`).
// Everything that enters the recurrence is float32: the rotated queries and keys, the gates, their
// exponentials, the maximum, the normaliser, the state and every sum.
#include "causal_product.h"
#include "common.h"

// ---- queries and keys as the recurrence takes them: qk[0] = q_scale * rot(q), qk[1] = k_scale * rot(k), float32.
// row [n, >= 2 * heads * D] begins with the query heads, then the key heads.  The first rot_dims elements
// of a head turn by position * inv_freq[j], element j paired with j + rot_dims / 2. ----
template <typename T>
__global__ void __launch_bounds__(256)
memory_inputs_kernel(const T* __restrict__ row, long long row_stride, const int* __restrict__ positions,
                     const float* __restrict__ inv_freq, float* __restrict__ qk, int tokens, int heads, int d, int rot_dims,
                     float q_scale, float k_scale) {
    const int token = blockIdx.x;
    const int width = heads * d, half = rot_dims / 2;
    const float pos = static_cast<float>(positions[token]);
    const T* r = row + static_cast<size_t>(token) * row_stride;
    for (int e = blockIdx.y * blockDim.x + threadIdx.x; e < 2 * width; e += gridDim.y * blockDim.x) {
        const int which = e / width, j = e % d;
        float v = to_float(r[e]);
        if (j < rot_dims) {
            const int f = j < half ? j : j - half;
            float sn, cs, ra, rb;
            sincosf(pos * inv_freq[f], &sn, &cs);
            if (j < half) {
                rotate_pair(v, to_float(r[e + half]), sn, cs, ra, rb);
                v = ra;
            } else {
                rotate_pair(to_float(r[e - half]), v, sn, cs, ra, rb);
                v = rb;
            }
        }
        qk[static_cast<size_t>(which) * tokens * width + static_cast<size_t>(token) * width + (e - which * width)] =
            v * (which ? k_scale : q_scale);
    }
}

WLLM_API int wllm_memory_inputs(const void* row, long long row_stride, const int* positions, const float* inv_freq,
                                float* qk, int is_bf16, int tokens, int heads, int d, int rot_dims, float q_scale,
                                float k_scale, hipStream_t stream) {
    if (tokens <= 0) return 0;
    if (heads <= 0 || d <= 0 || rot_dims < 0 || rot_dims > d || rot_dims % 2 || (rot_dims && !inv_freq)) return -1;
    const int tiles = (2 * heads * d + 255) / 256 < 64 ? (2 * heads * d + 255) / 256 : 64;
    const dim3 grid(tokens, tiles);
    if (is_bf16)
        memory_inputs_kernel<bf16><<<grid, 256, 0, stream>>>(static_cast<const bf16*>(row), row_stride, positions, inv_freq,
                                                             qk, tokens, heads, d, rot_dims, q_scale, k_scale);
    else
        memory_inputs_kernel<float><<<grid, 256, 0, stream>>>(static_cast<const float*>(row), row_stride, positions,
                                                              inv_freq, qk, tokens, heads, d, rot_dims, q_scale, k_scale);
    return launch_status();
}

// ---- a forget gate a channel that also decides what is written (the gating of HGRN2): from a row that begins
// with the query heads and then the forget gate's projection z (heads * D columns each),
//   f = lower + (1 - lower) * sigmoid(z + bias),   qkf[0] = act(q) (0: as it is, 1: silu),   qkf[1] = 1 - f,   qkf[2] = f
// all float32: the recurrence S_t = diag(f_t) S_(t-1) + (1 - f_t) v_t^T then is `memory_scan` with 1 - f in the
// keys' place and f as a decay a row. ----
template <typename T>
__global__ void __launch_bounds__(256)
memory_forget_inputs_kernel(const T* __restrict__ row, long long row_stride, const float* __restrict__ bias,
                            const float* __restrict__ lower, float* __restrict__ qkf, int tokens, int width, int q_act) {
    const int token = blockIdx.x;
    const T* r = row + static_cast<size_t>(token) * row_stride;
    const size_t plane = static_cast<size_t>(tokens) * width;
    for (int e = blockIdx.y * blockDim.x + threadIdx.x; e < width; e += gridDim.y * blockDim.x) {
        const float q = to_float(r[e]);
        const float z = to_float(r[width + e]) + (bias ? bias[e] : 0.f);
        const float l = lower ? lower[e] : 0.f;
        const float f = l + (1.f - l) * (1.f / (1.f + expf(-z)));
        const size_t at = static_cast<size_t>(token) * width + e;
        qkf[at] = q_act == 1 ? q / (1.f + expf(-q)) : q;
        qkf[plane + at] = 1.f - f;
        qkf[2 * plane + at] = f;
    }
}

WLLM_API int wllm_memory_forget_inputs(const void* row, long long row_stride, const float* bias, const float* lower,
                                       float* qkf, int is_bf16, int tokens, int width, int q_act, hipStream_t stream) {
    if (tokens <= 0) return 0;
    if (width <= 0 || q_act < 0 || q_act > 1) return -1;
    const int tiles = (width + 255) / 256 < 64 ? (width + 255) / 256 : 64;
    const dim3 grid(tokens, tiles);
    if (is_bf16)
        memory_forget_inputs_kernel<bf16><<<grid, 256, 0, stream>>>(static_cast<const bf16*>(row), row_stride, bias, lower,
                                                                    qkf, tokens, width, q_act);
    else
        memory_forget_inputs_kernel<float><<<grid, 256, 0, stream>>>(static_cast<const float*>(row), row_stride, bias, lower,
                                                                     qkf, tokens, width, q_act);
    return launch_status();
}

// ---- exponential gates held in range by a running maximum.  Per head and token, with the gate
// projections z_i, z_f (a band [n, 2 * heads] of a wider row: the input gates, then the forget gates):
//   i = cap * tanh((z_i + bias_i) / cap)                 (cap <= 0: no cap)
//   f = logsigmoid(cap * tanh((z_f + bias_f) / cap))
//   m_t = max(f + m_(t-1), i);  a = exp(f + m_(t-1) - m_t);  b = exp(i - m_t);  floor = exp(-m_t)
// steps[0], [1], [2] [n, heads] take a, b and floor; m is read from and left in the request's row (one float a
// head from `m_offset`).  One wavefront a (head, segment), 64 tokens at a time: a lane bends its token's gates,
// the chain of maxima (an addition and a maximum a token, the same operations in the same order however the
// tokens are cut into steps) runs over the 64 in turn with every lane following it, and a lane takes the
// exponentials of its own token. ----
__device__ __forceinline__ float from_lane(float v, int lane) {      // `lane` is the same in every lane
    return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), lane));
}
__device__ __forceinline__ float bent(float z, float cap) { return cap > 0.f ? cap * tanhf(z / cap) : z; }
__device__ __forceinline__ float log_sigmoid(float z) { return fminf(z, 0.f) - log1pf(expf(-fabsf(z))); }

template <typename T>
__global__ void __launch_bounds__(kWave)
memory_gates_kernel(const T* __restrict__ gates, long long gates_stride, const float* __restrict__ i_bias,
                    const float* __restrict__ f_bias, float cap, float* __restrict__ state, long long state_stride,
                    long long m_offset, const int* __restrict__ seg_q_start, const int* __restrict__ seg_q_len,
                    const int* __restrict__ state_slots, float* __restrict__ steps, int tokens, int heads) {
    const int h = blockIdx.x, seg = blockIdx.y, lane = threadIdx.x;
    const int q_len = seg_q_len[seg], q_start = seg_q_start[seg];
    if (q_len <= 0) return;
    const size_t all = static_cast<size_t>(tokens) * heads;
    float* m_at = state + static_cast<size_t>(state_slots[seg]) * state_stride + m_offset + h;
    float m = *m_at;
    const float bi = i_bias ? i_bias[h] : 0.f, bf = f_bias ? f_bias[h] : 0.f;
    for (int t0 = 0; t0 < q_len; t0 += kWave) {
        const int count = min(kWave, q_len - t0);
        float li = 0.f, lf = 0.f;
        if (lane < count) {
            const T* g = gates + static_cast<size_t>(q_start + t0 + lane) * gates_stride;
            li = bent(to_float(g[h]) + bi, cap);
            lf = log_sigmoid(bent(to_float(g[heads + h]) + bf, cap));
        }
        float m_before = 0.f, m_mine = 0.f;
        auto follow = [&](int t) {
            const float m_new = fmaxf(from_lane(lf, t) + m, from_lane(li, t));
            if (lane == t) {
                m_before = m;
                m_mine = m_new;
            }
            m = m_new;
        };
        if (count == kWave) {
#pragma unroll
            for (int t = 0; t < kWave; ++t) follow(t);
        } else {
            for (int t = 0; t < count; ++t) follow(t);
        }
        if (lane < count) {
            const size_t at = static_cast<size_t>(q_start + t0 + lane) * heads + h;
            steps[at] = expf(lf + m_before - m_mine);
            steps[all + at] = expf(li - m_mine);
            steps[2 * all + at] = expf(-m_mine);
        }
    }
    if (lane == 0) *m_at = m;
}

WLLM_API int wllm_memory_gates(const void* gates, long long gates_stride, const float* i_bias, const float* f_bias, float cap,
                               float* state, long long state_stride, long long m_offset, const int* seg_q_start,
                               const int* seg_q_len, const int* state_slots, float* steps, int is_bf16, int tokens,
                               int segments, int heads, hipStream_t stream) {
    if (tokens <= 0 || segments <= 0) return 0;
    if (heads <= 0 || segments > 65535) return -1;
    const dim3 grid(heads, segments);
    if (is_bf16)
        memory_gates_kernel<bf16><<<grid, kWave, 0, stream>>>(static_cast<const bf16*>(gates), gates_stride, i_bias, f_bias, cap,
                                                              state, state_stride, m_offset, seg_q_start, seg_q_len,
                                                              state_slots, steps, tokens, heads);
    else
        memory_gates_kernel<float><<<grid, kWave, 0, stream>>>(static_cast<const float*>(gates), gates_stride, i_bias, f_bias,
                                                               cap, state, state_stride, m_offset, seg_q_start, seg_q_len,
                                                               state_slots, steps, tokens, heads);
    return launch_status();
}

// ---- the recurrence itself.  A workgroup owns (head, segment, 16 columns of P) and walks the segment's
// tokens in order.  D is cut into 32 slices: a lane is (column, one of four slices), a wavefront four
// slices, the workgroup's eight wavefronts all of them; a lane keeps its R rows of its column of S in
// registers.  Tokens go 16 at a time through shared memory (q, k, v, a, b), the next 16 fetched into registers
// while these are walked; a token's sum is the slices' partial sums added in a fixed order (within the
// wavefront, then wavefront by wavefront), so it has the same bits whether the token came alone or inside a
// prompt.  With values in float32 it takes every segment; in bfloat16 those of fewer than `shorter_than` tokens, the others
// being walked in chunks further down, which add in another order.  With `steps` the column behind the last (p = P) is the normaliser: its value is 1 for every token,
// its rows lie at `n_offset` of the request's row, and its sums go to `nq` [tokens, heads]. ----
constexpr int kMemTokens = 16;
constexpr int kMemWaves = 8;
constexpr int kMemCols = 16;
constexpr int kMemSlices = kMemWaves * (kWave / kMemCols);
constexpr int kMemThreads = kWave * kMemWaves;

template <typename T, int R, bool ROWS>
__global__ void __launch_bounds__(kMemThreads)
memory_scan_kernel(const float* __restrict__ qk, const T* __restrict__ v, long long v_stride, const float* __restrict__ steps,
                   const float* __restrict__ decays, float* __restrict__ state, long long state_stride, long long n_offset,
                   const int* __restrict__ seg_q_start, const int* __restrict__ seg_q_len, const int* __restrict__ state_slots,
                   float* __restrict__ y, float* __restrict__ nq, int tokens, int heads, int d, int p_dim, int shorter_than) {
    constexpr int kRow = kMemSlices * R;                   // a token's row of q (and of k) in shared memory: d and zeros
    constexpr int kPasses = kMemTokens * kRow / kMemThreads;      // elements of q (and of k) a thread stages: R
    constexpr int kRowsPass = kMemThreads / kRow;          // tokens a pass covers
    __shared__ __align__(16) float q_s[kMemTokens * kRow];
    __shared__ __align__(16) float k_s[kMemTokens * kRow];
    __shared__ __align__(16) float f_s[ROWS ? kMemTokens * kRow : 1];      // ROWS: a decay a row of S and token
    __shared__ float v_s[kMemTokens * kMemCols];
    __shared__ float a_s[kMemTokens], b_s[kMemTokens];
    __shared__ float part_s[kMemTokens * kMemWaves * kMemCols];
    const int h = blockIdx.x, seg = blockIdx.y, p0 = blockIdx.z * kMemCols;
    const int q_len = seg_q_len[seg], q_start = seg_q_start[seg];
    if (q_len <= 0 || q_len >= shorter_than) return;
    const int tid = threadIdx.x;
    const int lane = tid % kWave, wave = tid / kWave;
    const int col = lane % kMemCols, slice = wave * (kWave / kMemCols) + lane / kMemCols;
    const int p = p0 + col;
    const bool norm_col = steps != nullptr && p == p_dim;
    const bool live = p < p_dim || norm_col;
    const size_t width = static_cast<size_t>(heads) * d, all = static_cast<size_t>(tokens) * heads;
    float* request = state + static_cast<size_t>(state_slots[seg]) * state_stride;
    // this lane's column of the state: rows p_dim apart in S, or the normaliser's rows one after the other
    float* s_rows = norm_col ? request + n_offset + static_cast<size_t>(h) * d : request + static_cast<size_t>(h) * d * p_dim + p;
    const size_t s_step = norm_col ? 1 : p_dim;
    const int n0 = slice * R;
    float s[R];
#pragma unroll
    for (int i = 0; i < R; ++i) s[i] = (live && n0 + i < d) ? s_rows[static_cast<size_t>(n0 + i) * s_step] : 0.f;
    const float fixed = decays ? decays[h] : 1.f;

    // what this thread stages of every 16 tokens: element `sj` of the rows of tokens st, st + kRowsPass, ... of q and of
    // k (zeros beyond d: a row of S that is not there stays zero and adds nothing), one value of v, one token's a and b
    const int sj = tid % kRow, st = tid / kRow;
    const int vt = tid / kMemCols, vc = tid % kMemCols;
    float q_r[kPasses], k_r[kPasses], f_r[ROWS ? kPasses : 1], v_r = 0.f, a_r = 1.f, b_r = 1.f;
    auto fetch = [&](int t0) {
        const int count = min(kMemTokens, q_len - t0);
#pragma unroll
        for (int u = 0; u < kPasses; ++u) {
            const int t = st + u * kRowsPass;
            q_r[u] = k_r[u] = 0.f;
            if (ROWS) f_r[u] = 0.f;
            if (sj < d && t < count) {
                const size_t at = static_cast<size_t>(q_start + t0 + t) * width + static_cast<size_t>(h) * d + sj;
                q_r[u] = qk[at];
                k_r[u] = qk[static_cast<size_t>(tokens) * width + at];
                if (ROWS) f_r[u] = qk[2 * static_cast<size_t>(tokens) * width + at];
            }
        }
        if (tid < kMemTokens * kMemCols) {
            v_r = 0.f;
            if (vt < count) {
                if (p0 + vc < p_dim)
                    v_r = to_float(v[static_cast<size_t>(q_start + t0 + vt) * v_stride + static_cast<size_t>(h) * p_dim + p0 + vc]);
                else if (steps != nullptr && p0 + vc == p_dim)
                    v_r = 1.f;
            }
        }
        if (tid < count) {
            const size_t at = static_cast<size_t>(q_start + t0 + tid) * heads + h;
            a_r = steps ? steps[at] : fixed;
            b_r = steps ? steps[all + at] : 1.f;
        }
    };
    auto place = [&]() {
#pragma unroll
        for (int u = 0; u < kPasses; ++u) {
            q_s[(st + u * kRowsPass) * kRow + sj] = q_r[u];
            k_s[(st + u * kRowsPass) * kRow + sj] = k_r[u];
            if (ROWS) f_s[(st + u * kRowsPass) * kRow + sj] = f_r[u];
        }
        if (tid < kMemTokens * kMemCols) v_s[tid] = v_r;
        if (tid < kMemTokens) {
            a_s[tid] = a_r;
            b_s[tid] = b_r;
        }
    };
    auto token = [&](int t) {
        const float a = a_s[t], bv = b_s[t] * v_s[t * kMemCols + col];
        const float* kt = k_s + t * kRow + n0;
        const float* qt = q_s + t * kRow + n0;
        const float* ft = f_s + (ROWS ? t * kRow + n0 : 0);
        float part = 0.f;
#pragma unroll
        for (int i = 0; i < R; ++i) {
            s[i] = fmaf(ROWS ? ft[i] : a, s[i], bv * kt[i]);
            part = fmaf(s[i], qt[i], part);
        }
        part = sum_across(sum_across(part, 32), 16);      // the wavefront's four slices of this column
        if (lane < kMemCols) part_s[(t * kMemWaves + wave) * kMemCols + col] = part;
    };

    fetch(0);
    for (int t0 = 0; t0 < q_len; t0 += kMemTokens) {
        const int count = min(kMemTokens, q_len - t0);
        place();
        __syncthreads();
        if (t0 + kMemTokens < q_len) fetch(t0 + kMemTokens);     // on their way while these 16 are walked
        if (count == kMemTokens) {
#pragma unroll
            for (int t = 0; t < kMemTokens; ++t) token(t);
        } else {
            for (int t = 0; t < count; ++t) token(t);
        }
        __syncthreads();
        for (int e = tid; e < count * kMemCols; e += kMemThreads) {
            const int t = e / kMemCols, l = e % kMemCols;
            if (p0 + l > p_dim || (p0 + l == p_dim && steps == nullptr)) continue;
            float total = part_s[(t * kMemWaves) * kMemCols + l];
#pragma unroll
            for (int w = 1; w < kMemWaves; ++w) total += part_s[(t * kMemWaves + w) * kMemCols + l];
            if (p0 + l == p_dim) nq[static_cast<size_t>(q_start + t0 + t) * heads + h] = total;
            else y[static_cast<size_t>(q_start + t0 + t) * heads * p_dim + static_cast<size_t>(h) * p_dim + p0 + l] = total;
        }
        // (the next round's `place` writes q, k, v, a, b, which nobody reads any more; its barrier stands between
        // these reads of the partial sums and the next writes to them)
    }
    if (live) {
#pragma unroll
        for (int i = 0; i < R; ++i)
            if (n0 + i < d) s_rows[static_cast<size_t>(n0 + i) * s_step] = s[i];
    }
}

// ---- the same recurrence over many tokens, 16 at a time on the matrix cores.  Per head, with f_t the decays of token t (a
// number a channel; the same in all channels unless the decays are a row's own) and k_t the key times its b_t,
//   y_t = (P_t q_t) . S0 + sum over s <= t of N_ts v_s,   S = P_16 S0 + Kh^T V,   N_ts = q_t . (the decays s < r <= t) k_s,
// P_t the product of a chunk's decays up to t, Kh_s = k_s times the decays behind s.  A product of decays is formed from
// the decays it is made of, never as a quotient, so the numbers are those of the walk token by token up to the order of
// float32 sums.  Nothing but S0 depends on the tokens before: `memory_chunk_kernel` makes P q, Kh, P_16 and N for every
// chunk and head at once ([16][C], [C][16], [C], [16][16] floats, C = the channels padded to a multiple of 64; and [C][4]:
// what the last four of a chunk's Kh, which weigh most, lost in being rounded to 32 bits), and
// `memory_chunk_scan_kernel` walks a segment's chunks with v_mfma_f32_16x16x4_f32 (float32 in and out).  A chunk begins
// every 16 tokens of a segment; the last one is its last 16 tokens, those of the chunk before it as tokens that change
// nothing (q = k = 0, f = 1).  Values in bfloat16 only: in the 32-bit path a token's bits do not depend on how its prompt
// was cut.
// Three segments of 500, 1,000 and 1,501 tokens, 16 heads of 128 by 128 with decays a row: 301 us token by token, 34 and
// 156 for the two kernels here; 2,048 tokens of 8 heads of 128 by 256 with a decay a head 305 against 19 and 127, with
// exponential gates and the normaliser 297 against 19 and 125; 64 tokens 12.6 against 7 and 9 (where a segment
// gains is the caller's rule, `from`).  Off the result in 64 bits (y; the memory left behind), here and token by token: decays a head 2.0e-7; 2.0e-7 and
// 3.1e-7; 3.2e-7, decays a row 8.1e-8; 4.5e-8 and 9.1e-8; 4.5e-8, exponential gates 8.7e-8; 5.3e-8 and 9.9e-8; 5.7e-8.  With N
// in 32 bits (27 us) and without the rest of Kh (138 us) decays a row are off by 9.4e-8; 4.8e-8, so both stay. ----
typedef float memory_float4 __attribute__((ext_vector_type(4)));

static __host__ __device__ __forceinline__ size_t chunk_floats(int c) { return static_cast<size_t>(2 * kChunk + 5) * c + kChunk * kChunk; }

// The sum over a row of 16 lanes, in every lane.
__device__ __forceinline__ float row_of_16_sum(float v) {
    v += row_permuted<0x128>(v);
    v += row_permuted<0x124>(v);
    v += row_permuted<0x4E>(v);
    v += row_permuted<0xB1>(v);
    return v;
}

template <int R>        // C = 64 R
__global__ void __launch_bounds__(256)
memory_chunk_kernel(const float* __restrict__ qk, const float* __restrict__ steps, const float* __restrict__ decays,
                    const int* __restrict__ seg_q_start, const int* __restrict__ seg_q_len, int segments,
                    float* __restrict__ chunks, int tokens, int heads, int d, int row_decays, int from) {
    constexpr int C = 64 * R, kEach = kChunk * C / 256;
    __shared__ __align__(16) float k_s[kChunk * C], q_s[kChunk * C], f_s[kChunk * C];
    __shared__ float b_s[kChunk];
    __shared__ int found;
    const int place = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
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
    // (a segment's last chunk is its last 16 tokens, of which those that the chunk before it holds are left out)
    const int begin = min(local, seg_q_len[seg] - kChunk), out_of = local - begin, token = q_start + begin;
    float* out = chunks + (static_cast<size_t>(place) * heads + h) * chunk_floats(C);
    const size_t width = static_cast<size_t>(heads) * d, plane = static_cast<size_t>(tokens) * width;
    float q[kEach], k[kEach], f[kEach];
#pragma unroll
    for (int j = 0; j < kEach; ++j) {
        // (every load from a place that is there: what is not is put right below)
        const int t = (tid + 256 * j) / C, i = min((tid + 256 * j) % C, d - 1);
        const size_t at = static_cast<size_t>(token + t) * width + static_cast<size_t>(h) * d + i;
        const size_t th = static_cast<size_t>(token + t) * heads + h;
        q[j] = qk[at];
        k[j] = qk[plane + at];
        f[j] = row_decays ? qk[2 * plane + at] : steps ? steps[th] : decays[h];
    }
    if (tid < kChunk)
        b_s[tid] = steps ? steps[static_cast<size_t>(tokens) * heads + static_cast<size_t>(token + tid) * heads + h] : 1.f;
#pragma unroll
    for (int j = 0; j < kEach; ++j) {
        const int e = tid + 256 * j;
        const bool there = e / C >= out_of && e % C < d;
        q_s[e] = there ? q[j] : 0.f;
        k_s[e] = there ? k[j] : 0.f;
        f_s[e] = there ? f[j] : 1.f;
    }
    __syncthreads();
    {
        // N: 16 lanes hold the key of token s, which decays as t goes on (decayed keys and a lane's sums in 64 bits)
        const int s = tid / kChunk, sl = tid % kChunk;
        double r[R][4];
#pragma unroll
        for (int j = 0; j < R; ++j) {
            const memory_float4 key = *reinterpret_cast<const memory_float4*>(k_s + s * C + 64 * j + 4 * sl);
#pragma unroll
            for (int u = 0; u < 4; ++u) r[j][u] = static_cast<double>(key[u]) * b_s[s];
        }
        float mine = 0.f;                              // N of token sl and key s
#pragma unroll
        for (int t = 0; t < kChunk; ++t) {
            double sum = 0.0;
#pragma unroll
            for (int j = 0; j < R; ++j) {
                const int at = t * C + 64 * j + 4 * sl;
                const memory_float4 qt = *reinterpret_cast<const memory_float4*>(q_s + at), ft = *reinterpret_cast<const memory_float4*>(f_s + at);
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    if (t > s) r[j][u] *= ft[u];
                    sum = fma(r[j][u], static_cast<double>(qt[u]), sum);
                }
            }
            const float dot = row_of_16_sum(static_cast<float>(sum));
            if (sl == t && t >= s) mine = dot;
        }
        out[(2 * kChunk + 5) * C + sl * kChunk + s] = mine;
    }
    // the decays up to and behind every token, a channel a thread.  (Products in 64 bits, rounded once: where the decays
    // are the head's, all channels share their error, which the walk token by token spreads over the state's elements.)
    for (int c = tid; c < C; c += 256) {
        double decay = 1.0, behind = 1.0;
        float kh[kChunk], rest[4];
#pragma unroll
        for (int t = 0; t < kChunk; ++t) {
            decay *= f_s[t * C + c];
            out[t * C + c] = static_cast<float>(q_s[t * C + c] * decay);
        }
        out[2 * kChunk * C + c] = static_cast<float>(decay);
#pragma unroll
        for (int t = kChunk - 1; t >= 0; --t) {
            const double key = static_cast<double>(k_s[t * C + c]) * b_s[t] * behind;
            kh[t] = static_cast<float>(key);
            // (a key that 32 bits do not hold is infinite, and has no remainder: inf - inf would be NaN)
            if (t >= kChunk - 4) rest[t - (kChunk - 4)] = fabsf(kh[t]) <= 3.402823466e38f ? static_cast<float>(key - kh[t]) : 0.f;
            behind *= f_s[t * C + c];
        }
        // (token 4u + g at place 4g + u: the u-th product of the walk then takes the tokens 4u .. 4u + 3, the oldest first)
#pragma unroll
        for (int g = 0; g < 4; ++g)
            *reinterpret_cast<memory_float4*>(out + kChunk * C + c * kChunk + 4 * g) = memory_float4{kh[g], kh[4 + g], kh[8 + g], kh[12 + g]};
        *reinterpret_cast<memory_float4*>(out + (2 * kChunk + 1) * C + 4 * c) = memory_float4{rest[0], rest[1], rest[2], rest[3]};
    }
}

// A workgroup owns (head, segment, 16 columns of P; the column behind the last is the normaliser's, as above).  Its first four
// wavefronts cut the channels, each with TILES tiles of 16: lane (i, g) holds the channels 4g .. 4g + 3 of a tile in column
// i, which is what a product leaves and, channel by channel, what it takes (the k-th of four products takes the channels
// 4g + k), so the memory never moves between lanes.  They keep the memory and read it for every chunk; what is left of a chunk's results
// (the part that its own tokens make, the sum over the wavefronts, the stores) is the other four's, a chunk and two chunks behind, beside them
// on their SIMDs.  One barrier a chunk, two places of shared memory in turn.  The operands of a chunk are asked for kAhead chunks before they are used, while
// the products that free their registers run.
// What bounds it: the chain of a chunk in one wavefront, of which the products (32 clocks each, 8 TILES + TILES) should be all. (Three prompts of 3,001
// tokens, 16 heads of 128 by 128, us: with the others' work in the same chain, and so many registers that a compute unit ran one workgroup, 157; now 115.)
template <int TILES>
__global__ void __launch_bounds__(512, TILES <= 2 ? 4 : 2)
memory_chunk_scan_kernel(const float* chunks, const bf16* v, long long v_stride, float* __restrict__ state, long long state_stride,
                         long long n_offset, const int* __restrict__ seg_q_start, const int* __restrict__ seg_q_len,
                         const int* __restrict__ state_slots, float* __restrict__ y, float* __restrict__ nq, int heads, int d,
                         int p_dim, int from) {
    constexpr int C = 64 * TILES, kAhead = 2, kOwnAhead = 6;
    __shared__ memory_float4 read_s[2][4][kWave], part_s[2][4][kWave];
    const int h = blockIdx.x, seg = blockIdx.y, p0 = blockIdx.z * 16;
    const int q_len = seg_q_len[seg], q_start = seg_q_start[seg];
    if (q_len < from) return;
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave) % 4;
    const bool keeps = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave) < 4;
    const int i = lane % 16, g = lane / 16;
    const int p = p0 + i;
    const bool norm_col = nq != nullptr && p == p_dim;
    const bool live = p < p_dim || norm_col;
    const float* first = chunks + (static_cast<size_t>(first_place(q_start, from)) * heads + h) * chunk_floats(C);
    const bf16* v_first = v + static_cast<size_t>(q_start) * v_stride + static_cast<size_t>(h) * p_dim;
    const unsigned col = static_cast<unsigned>(min(p, p_dim - 1)), row = static_cast<unsigned>(v_stride);
    auto begins = [&](int c) { return min(c * kChunk, q_len - kChunk); };      // (the last chunk: the last 16 tokens)
    const int count = (q_len + kChunk - 1) / kChunk;
    // (a barrier for what lies in shared memory alone: the operands of the chunks ahead stay on their way)
    auto meet = [&]() __attribute__((always_inline)) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    if (!keeps) {
        // wavefront w: the part of the tokens 4w .. 4w + 3 as keys; then the sums of the tokens 4g + w
        struct Own { float n; bf16 v; };
        const unsigned n_at = (2 * kChunk + 5) * C + i * kChunk + 4 * wave + g;
        auto load = [&](int c) __attribute__((always_inline)) {
            return Own{(first + static_cast<size_t>(c) * heads * chunk_floats(C))[n_at],
                       (v_first + static_cast<size_t>(begins(c)) * v_stride)[(4 * wave + g) * row + col]};
        };
        auto add_own = [&](int c, const Own& now) __attribute__((always_inline)) {
            const float x = begins(c) + 4 * wave + g >= c * kChunk ? (norm_col ? 1.f : to_float(now.v)) : 0.f;
            part_s[c % 2][wave][lane] = add_causal_product(now.n, x, read_s[c % 2][wave][lane], i, g, [&](int q) { return 4 * wave + q; });
        };
        auto finish = [&](int c) __attribute__((always_inline)) {
            const float* parts = reinterpret_cast<const float*>(&part_s[c % 2][0][lane]) + wave;
            float o = parts[0];
#pragma unroll
            for (int w = 1; w < 4; ++w) o += parts[w * 4 * kWave];
            const int t = begins(c) + 4 * g + wave;
            if (live && t >= c * kChunk) {
                if (norm_col) nq[static_cast<size_t>(q_start + t) * heads + h] = o;
                else y[static_cast<size_t>(q_start + t) * heads * p_dim + static_cast<size_t>(h) * p_dim + p] = o;
            }
        };
        // (kOwnAhead chunks ahead: a wait for these loads is one for the stores in front of them, too)
        Own ring[kOwnAhead];
#pragma unroll
        for (int a = 0; a < kOwnAhead; ++a) {
            ring[a] = load(min(a, count - 1));
            __builtin_amdgcn_sched_barrier(0);           // (in this order, which the waits of the loop count on)
        }
        auto step = [&](int c, int a) __attribute__((always_inline)) {
            add_own(c + a, ring[a]);
            __builtin_amdgcn_sched_barrier(0);
            ring[a] = load(min(c + a + kOwnAhead, count - 1));
            __builtin_amdgcn_sched_barrier(0);
            if (c + a > 0) finish(c + a - 1);
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
        finish(count - 1);
        return;
    }
    float* request = state + static_cast<size_t>(state_slots[seg]) * state_stride;
    float* s_rows = norm_col ? request + n_offset + static_cast<size_t>(h) * d : request + static_cast<size_t>(h) * d * p_dim + p;
    const size_t s_step = norm_col ? 1 : p_dim;
    const int ch0 = wave * 16 * TILES;
    memory_float4 s[TILES];
#pragma unroll
    for (int j = 0; j < TILES; ++j)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int ch = ch0 + 16 * j + 4 * g + u;
            s[j][u] = live && ch < d ? s_rows[static_cast<size_t>(ch) * s_step] : 0.f;
        }
    struct Operands {
        memory_float4 q[TILES], k[TILES], f[TILES];
        float rest[TILES];
        bf16 v[4];
    };
    // where this lane's operands lie in a chunk's (unsigned: a lane's offset beside an address that is the same in all lanes)
    const unsigned q_at = i * C + ch0 + 4 * g, k_at = kChunk * C + (ch0 + i) * kChunk + 4 * g, f_at = 2 * kChunk * C + ch0 + 4 * g;
    const unsigned rest_at = (2 * kChunk + 1) * C + (ch0 + i) * 4 + g;
    // what the products read, and (asked for behind the products' results, for a copy of it would wait for it) the decays
    auto load = [&](int c, Operands& o) __attribute__((always_inline)) {
        const float* at = first + static_cast<size_t>(c) * heads * chunk_floats(C);
        const bf16* v_chunk = v_first + static_cast<size_t>(begins(c)) * v_stride;
#pragma unroll
        for (int u = 0; u < 4; ++u) o.v[u] = v_chunk[(4 * u + g) * row + col];
#pragma unroll
        for (int j = 0; j < TILES; ++j) {
            o.q[j] = *reinterpret_cast<const memory_float4*>(at + q_at + 16 * j);
            o.k[j] = *reinterpret_cast<const memory_float4*>(at + k_at + 16 * kChunk * j);
            o.rest[j] = at[rest_at + 64 * j];
        }
    };
    auto load_decays = [&](int c, Operands& o) __attribute__((always_inline)) {
        const float* at = first + static_cast<size_t>(c) * heads * chunk_floats(C);
#pragma unroll
        for (int j = 0; j < TILES; ++j) o.f[j] = *reinterpret_cast<const memory_float4*>(at + f_at + 16 * j);
    };
    auto walk = [&](int c, Operands& now) __attribute__((always_inline)) {
        memory_float4 x, read[TILES];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            x[u] = begins(c) + 4 * u + g >= c * kChunk ? (norm_col ? 1.f : to_float(now.v[u])) : 0.f;
        // (a sum a tile, added in the end: short chains of products, and of roundings)
#pragma unroll
        for (int j = 0; j < TILES; ++j) read[j] = memory_float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int j = 0; j < TILES; ++j) read[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(now.q[j][u], s[j][u], read[j], 0, 0, 0);
        // (the chunk's own sum first, from what its newest keys lost in rounding, and the memory joins it with one rounding)
        memory_float4 own[TILES];
#pragma unroll
        for (int j = 0; j < TILES; ++j)
            own[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(now.rest[j], x[3], memory_float4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int j = 0; j < TILES; ++j) own[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(now.k[j][u], x[u], own[j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        load(min(c + kAhead, count - 1), now);
        __builtin_amdgcn_sched_barrier(0);
        memory_float4 part = read[0];
#pragma unroll
        for (int j = 1; j < TILES; ++j) part += read[j];
        read_s[c % 2][wave][lane] = part;                                    // a wavefront's part: its channels of the memory
#pragma unroll
        for (int j = 0; j < TILES; ++j)
#pragma unroll
            for (int u = 0; u < 4; ++u) s[j][u] = fmaf(now.f[j][u], s[j][u], own[j][u]);
        __builtin_amdgcn_sched_barrier(0);
        load_decays(min(c + kAhead, count - 1), now);
        meet();
    };
    // the operands of kAhead chunks in turn (beyond the last chunk: the last's once more).  The loads stay where they are
    // written: the scratch and v may alias y as far as the compiler knows, and the empty statements touch memory.
    Operands ring[kAhead];
#pragma unroll
    for (int a = 0; a < kAhead; ++a) {
        load(min(a, count - 1), ring[a]);
        __builtin_amdgcn_sched_barrier(0);
        load_decays(min(a, count - 1), ring[a]);
        __builtin_amdgcn_sched_barrier(0);               // (in this order, which the waits of the loop count on)
    }
    int c = 0;
    for (; c + kAhead <= count; c += kAhead) {
#pragma unroll
        for (int a = 0; a < kAhead; ++a) walk(c + a, ring[a]);
    }
#pragma unroll
    for (int a = 0; a < kAhead - 1; ++a)
        if (c + a < count) walk(c + a, ring[a]);
    meet();                                                                  // the others' last sums
#pragma unroll
    for (int j = 0; j < TILES; ++j)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int ch = ch0 + 16 * j + 4 * g + u;
            if (live && ch < d) s_rows[static_cast<size_t>(ch) * s_step] = s[j][u];
        }
}

// `steps` (float32 [3, tokens, heads], of which a and b are read; then `nq` float32 [tokens, heads] takes the
// normaliser's sums and the normaliser lies at `n_offset` of a request's row) or, if null, `decays` (float32 [heads]; b = 1),
// or, with `row_decays`, neither: then qk has a third plane [tokens, heads * d] of decays a row and token (b = 1).
// `from` tokens (16 at least; 0: no segment, as in float32) is what a segment needs to be walked in chunks, out of the
// scratch `chunks`: `chunk_places` places of heads * chunk_floats(the channels padded to a multiple of 64) floats.
// `shortest`: the caller's word that no segment has fewer tokens (0: it has none); with it at `from` or above nothing is
// launched for shorter ones.
WLLM_API int wllm_memory_scan(const float* qk, const void* v, long long v_stride, const float* steps, const float* decays,
                              float* state, long long state_stride, long long n_offset, const int* seg_q_start,
                              const int* seg_q_len, const int* state_slots, float* y, float* nq, int is_bf16, int tokens,
                              int segments, int heads, int d, int p_dim, int row_decays, float* chunks, int from, int shortest,
                              hipStream_t stream) {
    if (segments <= 0 || tokens <= 0) return 0;
    if (row_decays ? (steps || decays) : ((!steps) == (!decays) || (steps && !nq))) return -1;
    if (heads <= 0 || d <= 0 || d > 8 * kMemSlices || p_dim <= 0) return -1;
    if (segments > 65535 || (p_dim + kMemCols) / kMemCols > 65535) return -1;
    const int r = (d + kMemSlices - 1) / kMemSlices;
    const int columns = p_dim + (steps ? 1 : 0);
    const dim3 grid(heads, segments, (columns + kMemCols - 1) / kMemCols);
    // (a segment of `from` tokens leaves room for the others' single tokens)
    // (what the chunks' kernels do not take goes token by token)
    const bool in_chunks = from > 0 && tokens - (segments - 1) >= from && d <= 256 && heads <= 65535 && v_stride <= 0x0fffffffLL;
    if (in_chunks) {
        if (!is_bf16 || !chunks || from < kChunk || reinterpret_cast<uintptr_t>(chunks) % 16) return -1;
        const dim3 chunk_grid(chunk_places(tokens, from), heads);
#define LAUNCH(R)                                                                                                      \
    do {                                                                                                               \
        memory_chunk_kernel<R><<<chunk_grid, 256, 0, stream>>>(qk, steps, decays, seg_q_start, seg_q_len, segments, chunks, \
                                                               tokens, heads, d, row_decays, from);                    \
        if (const int err = launch_status()) return err;                                                               \
        memory_chunk_scan_kernel<R><<<grid, 512, 0, stream>>>(chunks, static_cast<const bf16*>(v), v_stride, state,    \
                                                              state_stride, n_offset, seg_q_start, seg_q_len, state_slots, y, \
                                                              steps ? nq : nullptr, heads, d, p_dim, from);            \
    } while (0)
        if (d <= 64) LAUNCH(1);
        else if (d <= 128) LAUNCH(2);
        else if (d <= 192) LAUNCH(3);
        else LAUNCH(4);
#undef LAUNCH
        if (const int err = launch_status()) return err;
        if (shortest >= from) return 0;
    }
    const int shorter_than = in_chunks ? from : 0x7fffffff;
#define LAUNCH(T, R, ROWS)                                                                                          \
    memory_scan_kernel<T, R, ROWS><<<grid, kMemThreads, 0, stream>>>(qk, static_cast<const T*>(v), v_stride, steps, decays, \
                                                                     state, state_stride, n_offset, seg_q_start, seg_q_len, \
                                                                     state_slots, y, nq, tokens, heads, d, p_dim, shorter_than)
#define LAUNCH_R(T, ROWS)                  \
    if (r <= 1) LAUNCH(T, 1, ROWS);        \
    else if (r <= 2) LAUNCH(T, 2, ROWS);   \
    else if (r <= 4) LAUNCH(T, 4, ROWS);   \
    else LAUNCH(T, 8, ROWS);
    if (row_decays) {
        if (is_bf16) { LAUNCH_R(bf16, true) } else { LAUNCH_R(float, true) }
    } else {
        if (is_bf16) { LAUNCH_R(bf16, false) } else { LAUNCH_R(float, false) }
    }
#undef LAUNCH_R
#undef LAUNCH
    return launch_status();
}

// ---- out = o / rms_of_the_head(o) * weight * act(gate) * scale with o = y / den: the recurrence's sums (float32),
// divided by the head's denominator den = max(|nq|, floor) + den_eps if there is one (nq, floor float32 [tokens, heads]),
// every head divided by its own root mean square (eps inside the root), times a weight over the whole row (if
// any), times the gate's activation (0: sigmoid, 1: silu; 2: there is no gate) of a band of a wider row; out (the activation
// type) may be a band too.  One wavefront a (token, head), kNormHeads of them a workgroup (a workgroup each, the launching of workgroups bounds it: 3,001 tokens of 16
// heads of 128, bfloat16, 18.1 us and 12.9; the bytes: 10); of heads of at most 64 HELD columns the sums stay in registers (HELD 0: they are read twice). ----
constexpr int kNormHeads = 4;

template <typename T, int GATE, int HELD>
__global__ void __launch_bounds__(kWave * kNormHeads)
head_norm_gate_kernel(const float* __restrict__ y, const T* __restrict__ gate, long long gate_stride,
                      const float* __restrict__ weight, T* __restrict__ out, long long out_stride,
                      const float* __restrict__ nq, const float* __restrict__ floor, float den_eps, int heads, int p_dim,
                      float eps, float scale) {
    const int token = blockIdx.x, lane = threadIdx.x % kWave;
    const int h = blockIdx.y * (blockDim.x / kWave) + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    if (h >= heads) return;
    const float* yr = y + (static_cast<size_t>(token) * heads + h) * p_dim;
    const size_t th = static_cast<size_t>(token) * heads + h;
    const T* g = GATE == 2 ? nullptr : gate + static_cast<size_t>(token) * gate_stride + static_cast<size_t>(h) * p_dim;
    T* o = out + static_cast<size_t>(token) * out_stride + static_cast<size_t>(h) * p_dim;
    float held[HELD > 0 ? HELD : 1];
    T held_gate[HELD > 0 ? HELD : 1];
#pragma unroll
    for (int k = 0; k < HELD; ++k) {
        const int i = min(lane + k * kWave, p_dim - 1);
        held[k] = yr[i];
        if (GATE != 2) held_gate[k] = g[i];
    }
    const float den = nq ? fmaxf(fabsf(nq[th]), floor[th]) + den_eps : 1.f;
    float ss = 0.f;
    if (HELD > 0) {
#pragma unroll
        for (int k = 0; k < HELD; ++k) {
            held[k] = held[k] / den;
            if (lane + k * kWave < p_dim) ss = fmaf(held[k], held[k], ss);
        }
    } else {
        for (int i = lane; i < p_dim; i += kWave) {
            const float part = yr[i] / den;
            ss = fmaf(part, part, ss);
        }
    }
    const float inv = 1.f / sqrtf(wave_sum(ss) / static_cast<float>(p_dim) + eps);
    auto finish = [&](int i, float part, T gate_value) __attribute__((always_inline)) {
        float val = part * inv;
        if (weight) val *= weight[h * p_dim + i];
        if (GATE != 2) {
            const float z = to_float(gate_value);
            const float sg = 1.f / (1.f + expf(-z));
            val *= GATE == 0 ? sg : z * sg;
        }
        o[i] = from_float<T>(val * scale);
    };
    if (HELD > 0) {
#pragma unroll
        for (int k = 0; k < HELD; ++k)
            if (lane + k * kWave < p_dim) finish(lane + k * kWave, held[k], held_gate[k]);
    } else {
        for (int i = lane; i < p_dim; i += kWave) finish(i, yr[i] / den, GATE == 2 ? T{} : g[i]);
    }
}

WLLM_API int wllm_head_norm_gate(const float* y, const void* gate, long long gate_stride, const float* weight, void* out,
                                 long long out_stride, const float* nq, const float* floor, float den_eps, int is_bf16,
                                 int gate_kind, int tokens, int heads, int p_dim, float eps, float scale, hipStream_t stream) {
    if (tokens <= 0) return 0;
    if (heads <= 0 || heads > 65535 || p_dim <= 0 || gate_kind < 0 || gate_kind > 2 || (!nq) != (!floor)) return -1;
    if (gate_kind != 2 && !gate) return -1;
    // (few tokens: a workgroup a head, for the compute units that would have none)
    const int together = static_cast<long long>(tokens) * heads >= 4096 ? kNormHeads : 1;
    const dim3 grid(tokens, (heads + together - 1) / together);
#define LAUNCH_HELD(T, G, HELD)                                                                                        \
    head_norm_gate_kernel<T, G, HELD><<<grid, kWave * together, 0, stream>>>(                                          \
        y, static_cast<const T*>(gate), gate_stride, weight, static_cast<T*>(out), out_stride, nq, floor, den_eps, heads, p_dim, eps, scale)
#define LAUNCH(T, G)                                                                                                   \
    do {                                                                                                               \
        if (p_dim <= 2 * kWave) LAUNCH_HELD(T, G, 2);                                                                  \
        else if (p_dim <= 4 * kWave) LAUNCH_HELD(T, G, 4);                                                             \
        else LAUNCH_HELD(T, G, 0);                                                                                     \
    } while (0)
    if (is_bf16) { if (gate_kind == 0) LAUNCH(bf16, 0); else if (gate_kind == 1) LAUNCH(bf16, 1); else LAUNCH(bf16, 2); }
    else { if (gate_kind == 0) LAUNCH(float, 0); else if (gate_kind == 1) LAUNCH(float, 1); else LAUNCH(float, 2); }
#undef LAUNCH_HELD
#undef LAUNCH
    return launch_status();
}
