// Attention over the paged cache for the 32-bit path, on the matrix cores (attn_float.hip).
#pragma once
#include "common.h"

// Whether the kernel takes the sizes: heads of 64 or 128, pages of a multiple of four tokens, 16-byte aligned pointers.
bool attn_float_takes(const void* q, const void* out, const void* cache_base, int hd, int page_size);
void attn_float_launch(const float* q, float* out, const PagedCache& cache, const int* positions, const int* tok_seq,
                       const int* block_table, int max_blocks, int n, int nh, float scale, int window, float softcap,
                       const float* sink, hipStream_t stream);
