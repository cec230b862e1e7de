// The entry point of `head_prepare.hip`, for the kernels that hand their work to it.
#pragma once
#include "common.h"

WLLM_API int wllm_head_prepare(void* rows, int is_bf16, int row_width, const float* parts, int splits,
                               long long split_stride, const float* bias, int bias_width, const int* positions,
                               const float* inv_freq, const int* slots, void* cache, long long num_pages, int n,
                               int num_heads, int num_kv_heads, int head_dim, int rotary_dim, int interleaved,
                               float norm_eps, int norm_dim, int values_are_keys, int page_size, const float* pre_q,
                               const float* pre_k, float pre_eps, float rot_scale, float temp_coef, int temp_every,
                               hipStream_t stream);
