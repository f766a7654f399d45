// Attention over cached latent rows on the matrix cores (bfloat16 pools), and the small products per
// head around it.
//
// A wave takes one token and up to 16 of its heads; every head of a token sees the same rows, so a
// loaded row serves all 16.  Everything is computed transposed, as in the other attention kernels of
// this library: S^T[key][head] = C[key][:] . Qa[head][:] (A = rows of the page, B = the folded queries,
// held in registers for the whole walk) and Z^T[dim][head] += C^T[dim][key] P^T[key][head] (A = the
// page's transposed copy, B = the weights, which are the lanes' own score accumulators: the rows of
// the score tiles are dealt out so that a lane's eight values of two tiles are eight keys in a row).
// A head is a lane column, so maxima, sums and rescaling need no broadcast.  Waves share nothing:
// rows of different requests may lie in one block.  Keys beyond the query's position are given weight
// zero and their values are set to zero before they are multiplied, so what an unused or reused page
// holds (a NaN too) never reaches a sum.
//
// A row is K values wide as a key and R as a value (its first R values; K > R where a rotated key part stands behind
// the latent); folded queries are K wide, the weighted sums R.
// sink (float [H], or null): a score per head that joins the denominator once, not scaled, with no key and no value.
//
// A kernel is compiled for the most steps of 32 values it takes and runs that many whatever K and R are: a step beyond
// K multiplies zeros of the query with the row's first values, one beyond R fills sums that nobody reads.  A branch
// around a load would make the compiler wait for every load before it issues the next.
#include "common.h"
#include "api.h"
#include "recordable.h"
#include "query_tail.h"

#define LT_WAVES 4
#define LT_CHUNK 64

// v with the values of the keys outside first_visible .. last_visible set to zero (v holds eight keys from first_key on)
__device__ __forceinline__ bf16x8 keep_keys(bf16x8 v, int first_key, int first_visible, int last_visible) {
#pragma unroll
    for (int e = 0; e < 8; ++e)
        v[e] = first_key + e > last_visible || first_key + e < first_visible ? (bf16_t)0.f : v[e];
    return v;
}

// qa: bfloat16 [n][H][K]; z: float [n][H][R]; pool: [n_pages][page_size * (K + R)]; K = 32 * nk, nk <= NK, R = 32 * ns, ns <= NS.
// n_split > 1: the keys of every token are dealt out to that many waves, which leave their sums in
// part_o [n * groups * n_split * 16][R] and (maximum, sum of weights) in part_ml [...][2]; a second kernel adds them.
template <int NK, int NS>
__global__ __launch_bounds__(64 * LT_WAVES) void latent_attention_mfma_kernel(
    const bf16_t* __restrict__ qa, float* __restrict__ z, const bf16_t* __restrict__ pool,
    const int* __restrict__ positions, const int* __restrict__ tok_seq, const int* __restrict__ block_table,
    int max_blocks, int n, int H, int K, int R, int page_size, int n_pages, float scale, int window, int groups_per_token,
    int n_split, float* __restrict__ part_o, float* __restrict__ part_ml, const float* __restrict__ sink) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int unit = blockIdx.x * LT_WAVES + wave;                 // (token, group of 16 heads, part of the keys)
    if (unit >= n * groups_per_token * n_split) return;
    const int split = unit % n_split, tg = unit / n_split;
    const int token = tg / groups_per_token, h0 = (tg - token * groups_per_token) * 16;
    const int col = lane & 15, g = lane >> 4;                      // col: head (B columns) or row of an A tile
    const int nk = K >> 5, ns = R >> 5;
    const int p = positions[token];
    const int* table = block_table + (size_t)tok_seq[token] * max_blocks;
    const int lo = window > 0 ? max(0, p - window + 1) : 0;
    const size_t page_stride = (size_t)page_size * (K + R);
    const bool head_live = h0 + col < H;

    // the folded queries of this lane's head: B operand of every score product
    bf16x8 qreg[NK];
    {
        const bf16_t* qr = qa + ((size_t)token * H + h0 + (head_live ? col : 0)) * K;
#pragma unroll
        for (int s = 0; s < NK; ++s) {
            if (s < nk && head_live) {
                qreg[s] = *(const bf16x8*)(qr + 32 * s + 8 * g);
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) qreg[s][e] = (bf16_t)0.f;
            }
        }
    }
    f32x4 o[2 * NS];                                               // Z^T tiles: dims 16 t + 4 g + r of head `col`
#pragma unroll
    for (int t = 0; t < 2 * NS; ++t) o[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;

    int first = lo & ~(LT_CHUNK - 1);                              // chunks are aligned, so a tile of 16 keys lies in one page
    int last = p;
    if (n_split > 1) {
        // this part's chunks: the token's chunks dealt out in equal runs (a short context leaves late parts empty)
        const int chunks = (p - first) / LT_CHUNK + 1, per = (chunks + n_split - 1) / n_split;
        last = min(p, first + (split + 1) * per * LT_CHUNK - 1);
        first += split * per * LT_CHUNK;
    }
    for (int t0 = first; t0 <= last; t0 += LT_CHUNK) {
        // ---- scores of 64 keys: four tiles of 16; tile 2 q + b, row i <-> key t0 + 32 q + 8 (i / 4) + 4 b + i % 4
        f32x4 sacc[4];
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            sacc[a] = (f32x4){0.f, 0.f, 0.f, 0.f};
            const int key = t0 + 32 * (a >> 1) + 8 * (col >> 2) + 4 * (a & 1) + (col & 3);
            const int kc = min(key, p);                            // a key beyond p: any loadable row, masked below
            int page = table[kc / page_size];
            page = min(max(page, 0), n_pages - 1);
            const bf16_t* row = pool + (size_t)page * page_stride + (size_t)(kc % page_size) * K + 8 * g;
#pragma unroll
            for (int s = 0; s < NK; ++s)
                sacc[a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8*)(row + (s < nk ? 32 * s : 0)), qreg[s], sacc[a], 0, 0, 0);
        }
        // lane (head col, g): sacc[2 q + b][e] is key t0 + 32 q + 8 g + 4 b + e
        float cmax = -INFINITY;
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int key = t0 + 32 * (a >> 1) + 8 * g + 4 * (a & 1) + e;
                sacc[a][e] = key > p || key < lo ? -INFINITY : sacc[a][e] * scale;
                cmax = fmaxf(cmax, sacc[a][e]);
            }
        cmax = fmaxf(cmax, __shfl_xor(cmax, 16, FL_WAVE));
        cmax = fmaxf(cmax, __shfl_xor(cmax, 32, FL_WAVE));
        const float m_new = fmaxf(m, cmax);                        // finite: every chunk holds a visible key
        const float corr = expf(m - m_new);
        m = m_new;
        bf16x8 pb[2];
        float lsum = 0.f;
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const bf16_t w = (bf16_t)expf(sacc[a][e] - m_new);
                pb[a >> 1][4 * (a & 1) + e] = w;
                lsum += (float)w;                                  // the sum of the weights as they are multiplied
            }
        lsum += __shfl_xor(lsum, 16, FL_WAVE);
        lsum += __shfl_xor(lsum, 32, FL_WAVE);
        l = l * corr + lsum;
        // ---- weighted sum: Z^T[dim][head] += C^T[dim][keys] P^T[keys][head], 32 keys a step
        const bool edge = t0 + LT_CHUNK - 1 > p || t0 < lo;
        const bf16_t* cols[2];
        int key0[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            key0[q] = t0 + 32 * q + 8 * g;
            const int kc = min(key0[q], p);
            int page = table[kc / page_size];
            page = min(max(page, 0), n_pages - 1);
            cols[q] = pool + (size_t)page * page_stride + (size_t)page_size * K + (key0[q] % page_size);
        }
#pragma unroll
        for (int t = 0; t < 2 * NS; ++t) {
            o[t] *= corr;
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                bf16x8 v = *(const bf16x8*)(cols[q] + (size_t)((t < 2 * ns ? 16 * t : 0) + col) * page_size);
                if (edge) v = keep_keys(v, key0[q], lo, p);
                o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v, pb[q], o[t], 0, 0, 0);
            }
        }
    }
    if (n_split > 1) {
        // unnormalised sums relative to this part's own maximum; fl_latent_attention_mfma's second kernel adds the parts
        float* po = part_o + ((size_t)unit * 16 + col) * R;
#pragma unroll
        for (int t = 0; t < 2 * NS; ++t)
            if (t < 2 * ns) *(f32x4*)(po + 16 * t + 4 * g) = o[t];
        if (g == 0) {
            part_ml[((size_t)unit * 16 + col) * 2] = m;
            part_ml[((size_t)unit * 16 + col) * 2 + 1] = l;
        }
        return;
    }
    if (!head_live) return;
    const float inv = sink ? softmax_factor_with_sink(m, l, sink[h0 + col]) : l > 0.f ? 1.0f / l : 0.f;
    float* zr = z + ((size_t)token * H + h0 + col) * R;
#pragma unroll
    for (int t = 0; t < 2 * NS; ++t)
        if (t < 2 * ns) *(f32x4*)(zr + 16 * t + 4 * g) = o[t] * inv;
}

// z[token][head][:] = sum_s o_s exp(m_s - M) / sum_s l_s exp(m_s - M), M = max_s m_s, over the parts of the keys
// (rising s; an empty part left zeros and has weight 0).  A block takes 256 dims of one (token, head): its
// first wave makes the parts' weights, then every thread adds its dim's parts, all loads independent.
__global__ __launch_bounds__(256) void latent_merge_kernel(const float* __restrict__ part_o, const float* __restrict__ part_ml,
                                                           float* __restrict__ z, int H, int R, int groups, int n_split,
                                                           const float* __restrict__ sink) {
    __shared__ float ws[64];
    __shared__ float inv_l;
    const int unit = blockIdx.x, d = blockIdx.y * 256 + threadIdx.x;
    const int token = unit / H, h = unit - token * H;
    const size_t base = ((size_t)(token * groups + (h >> 4)) * n_split) * 16 + (h & 15);        // part 0; parts are 16 rows apart
    if (threadIdx.x < 64) {
        const int lane = threadIdx.x;
        const float ms = lane < n_split ? part_ml[(base + (size_t)lane * 16) * 2] : -INFINITY;
        const float ls = lane < n_split ? part_ml[(base + (size_t)lane * 16) * 2 + 1] : 0.f;
        const float M = wave_max(ms);
        const float w = ms > -INFINITY ? expf(ms - M) : 0.f;
        const float L = wave_sum(ls * w);
        ws[lane] = w;
        if (lane == 0) inv_l = sink ? softmax_factor_with_sink(M, L, sink[h]) : L > 0.f ? 1.0f / L : 0.f;
    }
    __syncthreads();
    if (d >= R) return;
    float acc = 0.f;
#pragma unroll 8
    for (int s = 0; s < n_split; ++s) acc = fmaf(part_o[(base + (size_t)s * 16) * R + d], ws[s], acc);
    z[(size_t)unit * R + d] = acc * inv_l;
}

// Whether the kernels take a pool's shape: values of a multiple of 32 up to 512, keys as wide or one or two steps of
// 32 wider, pages of a multiple of 16 rows.
extern "C" int fl_latent_attention_mfma_takes(int K, int R, int page_size) {
    return R > 0 && R % 32 == 0 && R <= 512 && K % 32 == 0 && K >= R && K <= R + 64 && page_size > 0 && page_size % 16 == 0;
}

extern "C" int fl_latent_attention_mfma(const void* qa, float* z, const void* pool, const int* positions,
                                        const int* tok_seq, const int* block_table, int max_blocks, int n, int H, int K, int R,
                                        int page_size, int n_pages, float scale, int window, int n_split, float* part_o,
                                        float* part_ml, const float* sink, hipStream_t stream) {
    FL_CHECK(n >= 0 && H > 0 && n_pages > 0 && max_blocks > 0, "latent_attention_mfma: bad sizes");
    FL_CHECK(n_split >= 1 && n_split <= 64 && (n_split == 1 || (part_o && part_ml)), "latent_attention_mfma: %d parts of the keys (at most 64) need a workspace", n_split);
    FL_CHECK(fl_latent_attention_mfma_takes(K, R, page_size), "latent_attention_mfma: rows of %d and %d values in pages of %d are not taken", K, R, page_size);
    FL_CHECK((uintptr_t)qa % 16 == 0 && (uintptr_t)pool % 16 == 0 && (uintptr_t)z % 16 == 0, "latent_attention_mfma: operands must be 16-byte aligned");
    FL_CHECK(window >= 0, "latent_attention_mfma: negative window");
    if (n == 0) return 0;
    const int groups = ceil_div(H, 16);
    const long units = (long)n * groups * n_split;
    FL_CHECK(units < (1L << 30), "latent_attention_mfma: too many rows");
    const int blocks = (int)((units + LT_WAVES - 1) / LT_WAVES);
    const int ns = R / 32;
#define FL_LT(NK, NS)                                                                                                       \
    latent_attention_mfma_kernel<NK, NS><<<blocks, 64 * LT_WAVES, 0, stream>>>((const bf16_t*)qa, z, (const bf16_t*)pool,  \
                                                                           positions, tok_seq, block_table, max_blocks, \
                                                                           n, H, K, R, page_size, n_pages, scale, window, groups, \
                                                                           n_split, part_o, part_ml, sink)
    if (K == R) {
        if (ns <= 2) FL_LT(2, 2);
        else if (ns <= 4) FL_LT(4, 4);
        else if (ns <= 8) FL_LT(8, 8);
        else FL_LT(16, 16);
    } else {
        if (ns <= 2) FL_LT(4, 2);
        else if (ns <= 4) FL_LT(6, 4);
        else if (ns <= 8) FL_LT(10, 8);
        else FL_LT(18, 16);
    }
#undef FL_LT
    FL_LAUNCH_CHECK();
    if (n_split > 1) {
        dim3 mgrid(n * H, ceil_div(R, 256));
        latent_merge_kernel<<<mgrid, 256, 0, stream>>>(part_o, part_ml, z, H, R, groups, n_split, sink);
        FL_LAUNCH_CHECK();
    }
    return 0;
}
FL_RECORDABLE(fl_latent_attention_mfma)


// The same walk for prompt portions, four waves to a block that share their keys: a tile (from the host:
// first token, tokens, first group of 16 heads, groups; tokens x groups <= 4, all of one request) loads
// every chunk of 64 rows once into LDS, as it is and transposed, and its waves read their operands from
// there.  Without this every wave fetches every row itself and the kernel runs at the rate of the
// caches, 16 flops a byte.  Rows are padded by 16 bytes so that the 16 rows (or dims) of an operand
// start in different banks.  A wave whose token lies before a chunk sits the chunk out.
template <int NK, int NS>
__global__ __launch_bounds__(64 * LT_WAVES) void latent_attention_shared_kernel(
    const bf16_t* __restrict__ qa, float* __restrict__ z, const bf16_t* __restrict__ pool,
    const int* __restrict__ positions, const int* __restrict__ tok_seq, const int* __restrict__ block_table,
    int max_blocks, int H, int K, int R, int page_size, int n_pages, float scale, int window, const int* __restrict__ tiles,
    const float* __restrict__ sink) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lt_smem[];
    const int stride_r = K + 8, stride_c = LT_CHUNK + 8;
    bf16_t* ks = (bf16_t*)lt_smem;                                  // [64 keys][K + 8]
    bf16_t* vs = ks + (size_t)LT_CHUNK * stride_r;                  // [R dims][64 + 8]
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int t_first = tiles[4 * blockIdx.x], n_tok = tiles[4 * blockIdx.x + 1];
    const int g_first = tiles[4 * blockIdx.x + 2], n_grp = tiles[4 * blockIdx.x + 3];
    const int tw = wave / n_grp, gw = wave - tw * n_grp;
    const bool active = tw < n_tok;
    const int token = t_first + (active ? tw : 0), h0 = (g_first + gw) * 16;
    const int col = lane & 15, g = lane >> 4;
    const int nk = K >> 5, ns = R >> 5;
    const int p = active ? positions[token] : -1;
    const int p_max = positions[t_first + n_tok - 1];              // a request's tokens of a step stand in rising order
    const int* table = block_table + (size_t)tok_seq[t_first] * max_blocks;
    const int lo = window > 0 ? max(0, p - window + 1) : 0;
    const int lo_min = window > 0 ? max(0, positions[t_first] - window + 1) : 0;
    const size_t page_stride = (size_t)page_size * (K + R);
    const bool head_live = active && h0 + col < H;
    bf16x8 qreg[NK];
    {
        const bf16_t* qr = qa + ((size_t)token * H + (head_live ? h0 + col : 0)) * K;
#pragma unroll
        for (int s = 0; s < NK; ++s) {
            if (s < nk && head_live) {
                qreg[s] = *(const bf16x8*)(qr + 32 * s + 8 * g);
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) qreg[s][e] = (bf16_t)0.f;
            }
        }
    }
    f32x4 o[2 * NS];
#pragma unroll
    for (int t = 0; t < 2 * NS; ++t) o[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;
    const int pieces_r = K >> 3;                                    // 16-byte pieces of a row
    for (int t0 = lo_min & ~(LT_CHUNK - 1); t0 <= p_max; t0 += LT_CHUNK) {
        // ---- the chunk into LDS: rows as they are, and the pages' transposed copies dim by dim.  The pages of the
        // chunk's four runs of 16 keys are looked up first (pages hold a multiple of 16 rows), so that all copies
        // of a thread are in flight at once; a run beyond the newest token takes that token's page and is masked.
        const bf16_t* run_rows[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int kc = min(t0 + 16 * j, p_max & ~15);
            int page = table[kc / page_size];
            page = min(max(page, 0), n_pages - 1);
            run_rows[j] = pool + (size_t)page * page_stride + (size_t)(kc % page_size) * K;       // row kc of the page; the transposed values begin behind the page's page_size rows
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) {                             // wave w copies rows w, w + 4, ...: row 4 i + w lies in run i / 4
            const int row = 4 * i + wave;
            const bf16_t* src = run_rows[i >> 2] + (size_t)(row & 15) * K;
            for (int c = lane; c < pieces_r; c += 64) *(bf16x8*)(ks + (size_t)row * stride_r + 8 * c) = *(const bf16x8*)(src + 8 * c);
        }
        {
            const int k8 = threadIdx.x & 7;                        // this thread's 8 keys of every dim: run k8 / 2, its first or second half
            const int kc = min(t0 + 16 * (k8 >> 1), p_max & ~15);
            const bf16_t* src = run_rows[0];
#pragma unroll
            for (int j = 1; j < 4; ++j) src = (k8 >> 1) == j ? run_rows[j] : src;
            src += (size_t)(page_size - (kc % page_size)) * K + (kc % page_size) + 8 * (k8 & 1);    // from row kc of the page to column kc (+ 8) of its transposed copy
            for (int dim = threadIdx.x >> 3; dim < R; dim += 32)
                *(bf16x8*)(vs + (size_t)dim * stride_c + 8 * k8) = *(const bf16x8*)(src + (size_t)dim * page_size);
        }
        __syncthreads();
        if (active && t0 <= p && t0 + LT_CHUNK - 1 >= lo) {
            f32x4 sacc[4];
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                sacc[a] = (f32x4){0.f, 0.f, 0.f, 0.f};
                const bf16_t* row = ks + (size_t)(32 * (a >> 1) + 8 * (col >> 2) + 4 * (a & 1) + (col & 3)) * stride_r + 8 * g;
#pragma unroll
                for (int s = 0; s < NK; ++s)
                    sacc[a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8*)(row + (s < nk ? 32 * s : 0)), qreg[s], sacc[a], 0, 0, 0);
            }
            float cmax = -INFINITY;
#pragma unroll
            for (int a = 0; a < 4; ++a)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int key = t0 + 32 * (a >> 1) + 8 * g + 4 * (a & 1) + e;
                    sacc[a][e] = key > p || key < lo ? -INFINITY : sacc[a][e] * scale;
                    cmax = fmaxf(cmax, sacc[a][e]);
                }
            cmax = fmaxf(cmax, __shfl_xor(cmax, 16, FL_WAVE));
            cmax = fmaxf(cmax, __shfl_xor(cmax, 32, FL_WAVE));
            // The base of the exponents follows the maximum lazily: it moves only when a score exceeds it by more
            // than 8 (weights stay below e^8, exact enough in bfloat16 and float), so that in most chunks nothing
            // is rescaled and the sums can stay where the matrix cores accumulate them.
            const float m_new = (cmax > m + 8.0f) ? cmax : m;      // finite after the first chunk: it holds a key this wave sees
            const bool moved = __any(m_new != m);
            const float corr = expf(m - m_new);
            m = m_new;
            bf16x8 pb[2];
            float lsum = 0.f;
#pragma unroll
            for (int a = 0; a < 4; ++a)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const bf16_t w = (bf16_t)expf(sacc[a][e] - m_new);
                    pb[a >> 1][4 * (a & 1) + e] = w;
                    lsum += (float)w;
                }
            lsum += __shfl_xor(lsum, 16, FL_WAVE);
            lsum += __shfl_xor(lsum, 32, FL_WAVE);
            l = l * corr + lsum;
            if (moved) {
#pragma unroll
                for (int t = 0; t < 2 * NS; ++t) o[t] *= corr;
            }
            const bool edge = t0 + LT_CHUNK - 1 > p || t0 < lo;
#pragma unroll
            for (int t = 0; t < 2 * NS; ++t) {
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    bf16x8 v = *(const bf16x8*)(vs + (size_t)((t < 2 * ns ? 16 * t : 0) + col) * stride_c + 32 * q + 8 * g);
                    if (edge) v = keep_keys(v, t0 + 32 * q + 8 * g, lo, p);
                    o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v, pb[q], o[t], 0, 0, 0);
                }
            }
        }
        __syncthreads();
    }
    if (!head_live) return;
    const float inv = sink ? softmax_factor_with_sink(m, l, sink[h0 + col]) : l > 0.f ? 1.0f / l : 0.f;
    float* zr = z + ((size_t)token * H + h0 + col) * R;
#pragma unroll
    for (int t = 0; t < 2 * NS; ++t)
        if (t < 2 * ns) *(f32x4*)(zr + 16 * t + 4 * g) = o[t] * inv;
}

// The same tiles for latents of 128, 256 or 512 values, up to eight units (token, group of 16 heads) to a tile and eight waves to a
// block: a wave is a unit, with its folded queries and its weighted sums in registers and its weights formed and used in
// place (a wave behind the tile's units only copies).  Chunks of 32 keys lie in LDS twice, the next one on its way (memory straight to
// LDS, one barrier per chunk) while this one is read: rows as they are, the pages' transposed copies run by run of 16 keys, 16-byte
// pieces exchanged so that the reads of an operand meet no bank twice.
//
// A key whose score is the base has a weight of exactly one, and where a few keys have most of the weight, that is most of what rounding the weights to 16
// bits costs: the base follows the maximum for the first LT_FOLLOW keys.  Distance from 64 bits (2-norms, 32 heads of 576 and 512, 600 tokens, scores of deviation 0.18, 0.7
// and 2.1): 1.290e-3, 1.220e-3 and 0.89e-3; following it for the first 32 keys alone 1.282e-3, 1.263e-3 and 1.06e-3, for 64 (the kernel before) 1.294e-3, 1.248e-3 and
// 1.00e-3, for all of them 1.292e-3, 1.206e-3 and 0.71e-3 but 3 to 8 % slower.
//
// Bound by LDS: an operand of a kilobyte serves one matrix instruction, 4,352 clocks per chunk of eight units of 576 and 512 values where
// the matrix cores take 2,176; a chunk takes about 6,700 (5,450 without its copies, 3,400 the copies alone).  Why not eight waves that
// deal out the keys, the steps and the dims of 64 rows, as it was: their chunks' 137 KB for half the rows came in 5.6 us.  Microseconds,
// before and now: 32 heads of 576 and 512 values, 2,048 tokens 329 / 191, 1,024 95 / 78, 512 47 / 38, 512 behind 2,048 183 / 134, 4,096
// 1,200 / 635; 16 heads of 320 and 256, 2,048 123 / 86, 300 22 / 18.  The asks ahead of an operand's use, three to five, make no
// difference; the compiler's own order, one at a time, takes 242 where this takes 183.
#define LT_FOLLOW 128
template <int KB, int NS>                                           // steps of 64 values of a row as a key, of 32 as a value
__global__ __launch_bounds__(512, 2) void latent_attention_units_kernel(
    const bf16_t* __restrict__ qa, float* __restrict__ z, const bf16_t* __restrict__ pool,
    const int* __restrict__ positions, const int* __restrict__ tok_seq, const int* __restrict__ block_table,
    int max_blocks, int H, int K, int page_size, int n_pages, float scale, int window, const int* __restrict__ tiles,
    const float* __restrict__ sink) {
    constexpr int R = 32 * NS, NK = 2 * KB, CHUNK = 32, AHEAD = 4;
    constexpr int KEYS = CHUNK * KB * 64, VALUES = R * CHUNK;       // values of a chunk in LDS
    constexpr int K_COPIES = 4 * KB, V_COPIES = 2 * NS;             // copies of a kilobyte by one wave
    constexpr int KU = (K_COPIES + 7) / 8, VU = (V_COPIES + 7) / 8;
    extern __shared__ __attribute__((aligned(16))) unsigned char lt_smem[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int col = lane & 15, g = lane >> 4;
    const int tile = gridDim.x - 1 - blockIdx.x;                    // (a prompt's last tokens see the most keys: first)
    const int t_first = tiles[4 * tile], n_tok = tiles[4 * tile + 1], g_first = tiles[4 * tile + 2], n_grp = tiles[4 * tile + 3];
    const int tw = wave / n_grp, gw = wave - tw * n_grp;
    const bool active = tw < n_tok;
    const int token = t_first + (active ? tw : 0), h0 = (g_first + gw) * 16;
    const int p = active ? positions[token] : -1;
    const int p_max = positions[t_first + n_tok - 1];
    const int* table = block_table + (size_t)tok_seq[t_first] * max_blocks;
    const int lo = window > 0 ? max(0, p - window + 1) : 0;
    const int lo_min = window > 0 ? max(0, positions[t_first] - window + 1) : 0;
    const size_t page_stride = (size_t)page_size * (K + R);
    const bool head_live = active && h0 + col < H;

    bf16x8 qreg[NK];
    {
        const bf16_t* qr = qa + ((size_t)token * H + (head_live ? h0 + col : 0)) * K;
        const bf16x8 zero = {(bf16_t)0.f, (bf16_t)0.f, (bf16_t)0.f, (bf16_t)0.f, (bf16_t)0.f, (bf16_t)0.f, (bf16_t)0.f, (bf16_t)0.f};
#pragma unroll
        for (int st = 0; st < NK; ++st) {
            const bool inside = head_live && 32 * st < K;
            const bf16x8 v = *(const bf16x8*)(qr + (32 * st < K ? 32 * st : 0) + 8 * g);
            qreg[st] = inside ? v : zero;
        }
    }
    // the runs of 16 keys whose copies are sent next, two at a time (behind the newest token's run: that one again, masked below)
    const int t_begin = lo_min & ~(CHUNK - 1), runs_of_page = page_size / 16, last_run = p_max / 16;
    int run = min(t_begin / 16, last_run), page_at = run / runs_of_page, in_run = run - page_at * runs_of_page;
    int page[2], in_page[2];
    auto next_runs = [&]() {
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            page[r] = min(max(__builtin_amdgcn_readfirstlane(table[page_at]), 0), n_pages - 1);
            in_page[r] = 16 * in_run;
            if (run < last_run) {
                ++run;
                if (++in_run == runs_of_page) {
                    in_run = 0;
                    ++page_at;
                }
            }
        }
    };
    auto send = [&](int at) {
        const auto first = __builtin_amdgcn_make_buffer_rsrc((void*)(pool + (size_t)page[0] * page_stride), 0, (int)(page_stride * 2), 0x00020000);
        const auto second = __builtin_amdgcn_make_buffer_rsrc((void*)(pool + (size_t)page[1] * page_stride), 0, (int)(page_stride * 2), 0x00020000);
        unsigned char* ks = lt_smem + at * (KEYS + VALUES) * 2;
        unsigned char* vs = ks + KEYS * 2;
        int l = lane;                                               // (where a lane's 16 bytes come from is formed anew each time: no register is left to keep it)
        asm volatile("" : "+v"(l));
#pragma unroll
        for (int u = 0; u < KU; ++u) {
            const int c = wave + 8 * u;
            if (K_COPIES % 8 != 0 && c >= K_COPIES) break;
            const int slot = c % (2 * KB) * 64 + l, row = slot / (8 * KB), piece = slot % (8 * KB) ^ ((row & 3) | (row >> 1 & 4));
            const unsigned from = 8 * piece < K ? (unsigned)(row * K + 8 * piece) * 2 : 0x80000000u;      // (beyond the range: zeros)
            if (c < 2 * KB) __builtin_amdgcn_raw_ptr_buffer_load_lds(first, (__attribute__((address_space(3))) void*)(ks + c * 1024), 16, from, in_page[0] * K * 2, 0, 0);
            else __builtin_amdgcn_raw_ptr_buffer_load_lds(second, (__attribute__((address_space(3))) void*)(ks + c * 1024), 16, from, in_page[1] * K * 2, 0, 0);
        }
        const unsigned v_from = (unsigned)((l >> 1) * page_size + 8 * ((l & 1) ^ (l >> 3 & 1))) * 2;      // of 32 dims
#pragma unroll
        for (int u = 0; u < VU; ++u) {
            const int c = wave + 8 * u;
            if (V_COPIES % 8 != 0 && c >= V_COPIES) break;
            const int from = (page_size * (K + c % NS * 32) + in_page[c / NS]) * 2;
            if (c < NS) __builtin_amdgcn_raw_ptr_buffer_load_lds(first, (__attribute__((address_space(3))) void*)(vs + c * 1024), 16, v_from, from, 0, 0);
            else __builtin_amdgcn_raw_ptr_buffer_load_lds(second, (__attribute__((address_space(3))) void*)(vs + c * 1024), 16, v_from, from, 0, 0);
        }
    };
    f32x4 o[2 * NS];
#pragma unroll
    for (int t = 0; t < 2 * NS; ++t) o[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;                                   // (l: of the keys that this lane weighs)
    next_runs();
    send(0);
    next_runs();
    int at = 0;
    const float scale2 = scale * 1.4426950408889634f;               // (scores in powers of two)
    // a chunk; EDGE: some token of the tile does not see all of it
    auto chunk = [&](int t0, auto EDGE) {
        constexpr bool edge = decltype(EDGE)::value;
        __builtin_amdgcn_s_waitcnt(0x0F70);                         // this wave's copies of the chunk are there ...
        asm volatile("s_barrier" ::: "memory");                     // ... everyone's, and the other half is read
        if (t0 + CHUNK <= p_max) {
            send(at ^ 1);
            next_runs();
        }
        if (active && (!edge || (t0 <= p && t0 + CHUNK - 1 >= lo))) {
            const bf16_t* ks = (const bf16_t*)(lt_smem + at * (KEYS + VALUES) * 2);
            const bf16_t* vs = ks + KEYS;
            // row i of tile a is key 8 (i / 4) + 4 a + i % 4, so that lane (g, head col) gets keys 8 g + 4 a + e in sacc[a][e]
            int lc = lane;                                          // (as above)
            asm volatile("" : "+v"(lc));
            const int c = lc & 15, q = lc >> 4;
            const bf16_t* row = ks + (8 * (c >> 2) + (c & 3)) * KB * 64;
            const bf16_t* even = row + (q ^ (c & 7)) * 8;           // its 16 bytes of steps 0, 2, ..., and of 1, 3, ...
            const bf16_t* odd = row + ((4 + q) ^ (c & 7)) * 8;
            const bf16_t* dims = vs + ((q >> 1) * R + c) * 16 + ((q & 1) ^ (c >> 2 & 1)) * 8;
            // the operands of the scores and, behind them, of the sums, in the order of their use, AHEAD of them on their way (left to
            // itself the compiler, short of registers, asks for one and waits for it)
            auto operand = [&](auto J) {
                constexpr int j = decltype(J)::value, t = j - 2 * NK;
                if constexpr (t < 0) return *(const bf16x8*)((j & 2 ? odd : even) + (j >> 2) * 64 + (j & 1) * 4 * KB * 64);
                else return *(const bf16x8*)(dims + t * 256);
            };
            bf16x8 ring[AHEAD];
            static_for<AHEAD>([&](auto J) { ring[J] = operand(J); });
            f32x4 sacc[2];
#pragma unroll
            for (int a = 0; a < 2; ++a) sacc[a] = (f32x4){0.f, 0.f, 0.f, 0.f};
            static_for<2 * NK>([&](auto J) {
                constexpr int j = decltype(J)::value;
                sacc[j & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ring[j % AHEAD], qreg[j >> 1], sacc[j & 1], 0, 0, 0);
                ring[j % AHEAD] = operand(std::integral_constant<int, j + AHEAD>{});
                __builtin_amdgcn_sched_barrier(0);
            });
            float cmax = -INFINITY;
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int key = t0 + 8 * q + 4 * a + e;
                    sacc[a][e] = edge && (key > p || key < lo) ? -INFINITY : sacc[a][e] * scale2;
                    cmax = fmaxf(cmax, sacc[a][e]);
                }
            cmax = fmaxf(cmax, __shfl_xor(cmax, 16, FL_WAVE));
            cmax = fmaxf(cmax, __shfl_xor(cmax, 32, FL_WAVE));
            // (the base of the exponents follows the maximum, behind the first LT_FOLLOW keys lazily: weights stay below 2^11.5)
            const float m_new = cmax > (t0 < t_begin + LT_FOLLOW ? m : m + 11.5f) ? cmax : m;
            const float base = m_new == -INFINITY ? 0.f : m_new;
            if (__any(m_new != m)) {
                const float corr = __builtin_amdgcn_exp2f(m - base);
                l *= corr;
#pragma unroll
                for (int t = 0; t < 2 * NS; ++t) o[t] *= corr;
                m = m_new;
            }
            bf16x8 pb;
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    pb[4 * a + e] = (bf16_t)__builtin_amdgcn_exp2f(sacc[a][e] - base);
                    l += (float)pb[4 * a + e];                      // the sum of the weights as they are multiplied
                }
            // values of keys that the token does not see are zero, whatever the page holds
            u32x4 keep = {};
            if constexpr (edge) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int key = t0 + 8 * q + 2 * e;
                    keep[e] = (key > p || key < lo ? 0u : 0xffffu) | (key + 1 > p || key + 1 < lo ? 0u : 0xffff0000u);
                }
            }
            static_for<2 * NS>([&](auto T) {
                constexpr int t = decltype(T)::value, j = 2 * NK + t;
                bf16x8 v = ring[j % AHEAD];
                if constexpr (edge) v = __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, v) & keep);
                o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v, pb, o[t], 0, 0, 0);
                if constexpr (t + AHEAD < 2 * NS) ring[j % AHEAD] = operand(std::integral_constant<int, j + AHEAD>{});
                __builtin_amdgcn_sched_barrier(0);
            });
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");          // (the reads are done before the barrier lets anyone copy into their place)
        at ^= 1;
    };
    const int p_least = positions[t_first], lo_most = window > 0 ? max(0, p_max - window + 1) : 0;
    int t0 = t_begin;
    for (; t0 <= p_max && t0 < lo_most; t0 += CHUNK) chunk(t0, std::true_type{});
    for (; t0 + CHUNK - 1 <= p_least; t0 += CHUNK) chunk(t0, std::false_type{});
    for (; t0 <= p_max; t0 += CHUNK) chunk(t0, std::true_type{});
    if (!head_live) return;
    l += __shfl_xor(l, 16, FL_WAVE);
    l += __shfl_xor(l, 32, FL_WAVE);
    const float inv = sink ? softmax_factor_with_sink(m * 0.6931471805599453f, l, sink[h0 + col]) : l > 0.f ? 1.0f / l : 0.f;
    float* zr = z + ((size_t)token * H + h0 + col) * R;
#pragma unroll
    for (int t = 0; t < 2 * NS; ++t) *(f32x4*)(zr + 16 * t + 4 * g) = o[t] * inv;
}

template <int KB, int NS>
static int launch_units(const void* qa, float* z, const void* pool, const int* positions, const int* tok_seq, const int* block_table,
                        int max_blocks, int H, int K, int page_size, int n_pages, float scale, int window, const int* tiles, int n_tiles,
                        const float* sink, hipStream_t stream) {
    constexpr int LDS = 2 * 32 * (KB * 64 + NS * 32) * 2;
    static bool sized = false;
    if (!sized) {
        hipError_t e_ = hipFuncSetAttribute((const void*)latent_attention_units_kernel<KB, NS>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
        FL_CHECK(e_ == hipSuccess, "latent_attention_units: %s", hipGetErrorString(e_));
        sized = true;
    }
    latent_attention_units_kernel<KB, NS><<<n_tiles, 512, LDS, stream>>>((const bf16_t*)qa, z, (const bf16_t*)pool, positions, tok_seq, block_table,
                                                                         max_blocks, H, K, page_size, n_pages, scale, window, tiles, sink);
    return 0;
}

extern "C" long fl_latent_attention_shared_lds(int K, int R) { return (long)LT_CHUNK * (K + 8) * 2 + (long)R * (LT_CHUNK + 8) * 2; }

// how many units (token, group of 16 heads) a tile of the kernel below may hold (eight: in pages that lie within a 31-bit offset)
extern "C" int fl_latent_attention_units(int K, int R, int page_size) {
    return (R == 128 || R == 256 || R == 512) && (long)page_size * (K + R) < (1l << 30) ? 8 : 4;
}

// tiles [n_tiles][4] = (first token, tokens, first group of 16 heads, groups): tokens x groups <= fl_latent_attention_units, the tokens of one request
extern "C" int fl_latent_attention_shared(const void* qa, float* z, const void* pool, const int* positions,
                                          const int* tok_seq, const int* block_table, int max_blocks, int H, int K, int R,
                                          int page_size, int n_pages, float scale, int window, const int* tiles, int n_tiles,
                                          const float* sink, hipStream_t stream) {
    FL_CHECK(n_tiles >= 0 && H > 0 && n_pages > 0 && max_blocks > 0, "latent_attention_shared: bad sizes");
    FL_CHECK(fl_latent_attention_mfma_takes(K, R, page_size), "latent_attention_shared: rows of %d and %d values in pages of %d are not taken", K, R, page_size);
    FL_CHECK((uintptr_t)qa % 16 == 0 && (uintptr_t)pool % 16 == 0 && (uintptr_t)z % 16 == 0, "latent_attention_shared: operands must be 16-byte aligned");
    FL_CHECK(window >= 0, "latent_attention_shared: negative window");
    if (n_tiles == 0) return 0;
    if (fl_latent_attention_units(K, R, page_size) == 8) {
#define FL_LUN(KB, NS) launch_units<KB, NS>(qa, z, pool, positions, tok_seq, block_table, max_blocks, H, K, page_size, n_pages, scale, window, tiles, n_tiles, sink, stream)
        const int rc = R == 128 ? (K == R ? FL_LUN(2, 4) : FL_LUN(3, 4)) : R == 256 ? (K == R ? FL_LUN(4, 8) : FL_LUN(5, 8)) : K == R ? FL_LUN(8, 16) : FL_LUN(9, 16);
#undef FL_LUN
        if (rc != 0) return rc;
        FL_LAUNCH_CHECK();
        return 0;
    }
    const size_t lds = (size_t)fl_latent_attention_shared_lds(K, R);
    const int ns = R / 32;
#define FL_LTS(NK, NS)                                                                                                     \
    do {                                                                                                               \
        static bool sized = false;                                                                                     \
        if (!sized) {                                                                                                  \
            hipError_t e_ = hipFuncSetAttribute((const void*)latent_attention_shared_kernel<NK, NS>,                      \
                                                hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);              \
            FL_CHECK(e_ == hipSuccess, "latent_attention_shared: %s", hipGetErrorString(e_));                          \
            sized = true;                                                                                              \
        }                                                                                                              \
        latent_attention_shared_kernel<NK, NS><<<n_tiles, 64 * LT_WAVES, lds, stream>>>(                                  \
            (const bf16_t*)qa, z, (const bf16_t*)pool, positions, tok_seq, block_table, max_blocks, H, K, R, page_size,   \
            n_pages, scale, window, tiles, sink);                                                                            \
    } while (0)
    if (K == R) {
        if (ns <= 2) FL_LTS(2, 2);
        else if (ns <= 4) FL_LTS(4, 4);
        else if (ns <= 8) FL_LTS(8, 8);
        else FL_LTS(16, 16);
    } else {
        if (ns <= 2) FL_LTS(4, 2);
        else if (ns <= 4) FL_LTS(6, 4);
        else if (ns <= 8) FL_LTS(10, 8);
        else FL_LTS(18, 16);
    }
#undef FL_LTS
    FL_LAUNCH_CHECK();
    return 0;
}
FL_RECORDABLE(fl_latent_attention_shared)


// The same walk for steps of few rows (decoding), where a wave that holds all of a latent's dims has no register
// left for reads in flight and waits for every operand: the four waves of a block take one (token, 16 heads, part
// of the keys) together and deal the latent's steps of 32 dims out among them (wave w: steps w, w + 4, ...).
// Each forms its share of the scores, the shares are added through LDS in a fixed order (every wave gets the
// same sums, hence the same maxima and weights), and each adds the weighted rows of its own dims.  A wave then
// holds a quarter of the accumulators and queries, and the reads of a chunk are all in flight at once.
template <int NKW, int NSW>
__global__ __launch_bounds__(64 * LT_WAVES) void latent_attention_dealt_kernel(
    const bf16_t* __restrict__ qa, float* __restrict__ z, const bf16_t* __restrict__ pool,
    const int* __restrict__ positions, const int* __restrict__ tok_seq, const int* __restrict__ block_table,
    int max_blocks, int n, int H, int K, int R, int page_size, int n_pages, float scale, int window, int groups_per_token,
    int n_split, float* __restrict__ part_o, float* __restrict__ part_ml, const float* __restrict__ sink) {
    __shared__ f32x4 sx[LT_WAVES][4][64];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int unit = blockIdx.x;                                   // (token, group of 16 heads, part of the keys)
    const int split = unit % n_split, tg = unit / n_split;
    const int token = tg / groups_per_token, h0 = (tg - token * groups_per_token) * 16;
    const int col = lane & 15, g = lane >> 4;
    const int nk = K >> 5, ns = R >> 5;
    const int p = positions[token];
    const int* table = block_table + (size_t)tok_seq[token] * max_blocks;
    const int lo = window > 0 ? max(0, p - window + 1) : 0;
    const size_t page_stride = (size_t)page_size * (K + R);
    const bool head_live = h0 + col < H;
    bf16x8 qreg[NKW];
    {
        const bf16_t* qr = qa + ((size_t)token * H + h0 + (head_live ? col : 0)) * K;
#pragma unroll
        for (int i = 0; i < NKW; ++i) {
            const int s = wave + LT_WAVES * i;
            if (s < nk && head_live) {
                qreg[i] = *(const bf16x8*)(qr + 32 * s + 8 * g);
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) qreg[i][e] = (bf16_t)0.f;
            }
        }
    }
    f32x4 o[2 * NSW];                                              // dims 32 s + 16 u + 4 g + r of the wave's steps s, u = 0, 1
#pragma unroll
    for (int t = 0; t < 2 * NSW; ++t) o[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;
    int first = lo & ~(LT_CHUNK - 1), last = p;
    if (n_split > 1) {
        const int chunks = (p - first) / LT_CHUNK + 1, per = (chunks + n_split - 1) / n_split;
        last = min(p, first + (split + 1) * per * LT_CHUNK - 1);
        first += split * per * LT_CHUNK;
    }
    for (int t0 = first; t0 <= last; t0 += LT_CHUNK) {
        // the values do not wait for the scores: all of a chunk's reads are asked for at its start
        int key0[2];
        bf16x8 vreg[2 * NSW][2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            key0[q] = t0 + 32 * q + 8 * g;
            const int kc = min(key0[q], p);
            int page = table[kc / page_size];
            page = min(max(page, 0), n_pages - 1);
            const bf16_t* cols = pool + (size_t)page * page_stride + (size_t)page_size * K + (key0[q] % page_size);
#pragma unroll
            for (int t = 0; t < 2 * NSW; ++t) {
                const int s = wave + LT_WAVES * (t >> 1);
                vreg[t][q] = *(const bf16x8*)(cols + (size_t)((s < ns ? 32 * s : 0) + 16 * (t & 1) + col) * page_size);
            }
        }
        f32x4 sacc[4];
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            sacc[a] = (f32x4){0.f, 0.f, 0.f, 0.f};
            const int key = t0 + 32 * (a >> 1) + 8 * (col >> 2) + 4 * (a & 1) + (col & 3);
            const int kc = min(key, p);
            int page = table[kc / page_size];
            page = min(max(page, 0), n_pages - 1);
            const bf16_t* row = pool + (size_t)page * page_stride + (size_t)(kc % page_size) * K + 8 * g;
#pragma unroll
            for (int i = 0; i < NKW; ++i) {
                const int s = wave + LT_WAVES * i;
                sacc[a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8*)(row + (s < nk ? 32 * s : 0)), qreg[i], sacc[a], 0, 0, 0);
            }
            sx[wave][a][lane] = sacc[a];
        }
        __syncthreads();
        float cmax = -INFINITY;
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            sacc[a] = (sx[0][a][lane] + sx[1][a][lane]) + (sx[2][a][lane] + sx[3][a][lane]);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int key = t0 + 32 * (a >> 1) + 8 * g + 4 * (a & 1) + e;
                sacc[a][e] = key > p || key < lo ? -INFINITY : sacc[a][e] * scale;
                cmax = fmaxf(cmax, sacc[a][e]);
            }
        }
        __syncthreads();                                           // (the next chunk's shares overwrite sx)
        cmax = fmaxf(cmax, __shfl_xor(cmax, 16, FL_WAVE));
        cmax = fmaxf(cmax, __shfl_xor(cmax, 32, FL_WAVE));
        const float m_new = fmaxf(m, cmax);
        const float corr = expf(m - m_new);
        m = m_new;
        bf16x8 pb[2];
        float lsum = 0.f;
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const bf16_t w = (bf16_t)expf(sacc[a][e] - m_new);
                pb[a >> 1][4 * (a & 1) + e] = w;
                lsum += (float)w;
            }
        lsum += __shfl_xor(lsum, 16, FL_WAVE);
        lsum += __shfl_xor(lsum, 32, FL_WAVE);
        l = l * corr + lsum;
        const bool edge = t0 + LT_CHUNK - 1 > p || t0 < lo;
#pragma unroll
        for (int t = 0; t < 2 * NSW; ++t) {
            o[t] *= corr;
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                bf16x8 v = vreg[t][q];
                if (edge) v = keep_keys(v, key0[q], lo, p);
                o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v, pb[q], o[t], 0, 0, 0);
            }
        }
    }
    if (n_split > 1) {
        float* po = part_o + ((size_t)unit * 16 + col) * R;
#pragma unroll
        for (int t = 0; t < 2 * NSW; ++t) {
            const int s = wave + LT_WAVES * (t >> 1);
            if (s < ns) *(f32x4*)(po + 32 * s + 16 * (t & 1) + 4 * g) = o[t];
        }
        if (wave == 0 && g == 0) {
            part_ml[((size_t)unit * 16 + col) * 2] = m;
            part_ml[((size_t)unit * 16 + col) * 2 + 1] = l;
        }
        return;
    }
    if (!head_live) return;
    const float inv = sink ? softmax_factor_with_sink(m, l, sink[h0 + col]) : l > 0.f ? 1.0f / l : 0.f;
    float* zr = z + ((size_t)token * H + h0 + col) * R;
#pragma unroll
    for (int t = 0; t < 2 * NSW; ++t) {
        const int s = wave + LT_WAVES * (t >> 1);
        if (s < ns) *(f32x4*)(zr + 32 * s + 16 * (t & 1) + 4 * g) = o[t] * inv;
    }
}

// fl_latent_attention_mfma with a block of four waves per (token, 16 heads, part of the keys): for steps of few rows
extern "C" int fl_latent_attention_dealt(const void* qa, float* z, const void* pool, const int* positions,
                                         const int* tok_seq, const int* block_table, int max_blocks, int n, int H, int K, int R,
                                         int page_size, int n_pages, float scale, int window, int n_split, float* part_o,
                                         float* part_ml, const float* sink, hipStream_t stream) {
    FL_CHECK(n >= 0 && H > 0 && n_pages > 0 && max_blocks > 0, "latent_attention_dealt: bad sizes");
    FL_CHECK(n_split >= 1 && n_split <= 64 && (n_split == 1 || (part_o && part_ml)), "latent_attention_dealt: %d parts of the keys (at most 64) need a workspace", n_split);
    FL_CHECK(fl_latent_attention_mfma_takes(K, R, page_size), "latent_attention_dealt: rows of %d and %d values in pages of %d are not taken", K, R, page_size);
    FL_CHECK((uintptr_t)qa % 16 == 0 && (uintptr_t)pool % 16 == 0 && (uintptr_t)z % 16 == 0, "latent_attention_dealt: operands must be 16-byte aligned");
    FL_CHECK(window >= 0, "latent_attention_dealt: negative window");
    if (n == 0) return 0;
    const int groups = ceil_div(H, 16);
    const long units = (long)n * groups * n_split;
    FL_CHECK(units < (1L << 30), "latent_attention_dealt: too many rows");
    const int nkw = ceil_div(K / 32, LT_WAVES), nsw = ceil_div(R / 32, LT_WAVES);
#define FL_LTD(NKW, NSW)                                                                                                       \
    latent_attention_dealt_kernel<NKW, NSW><<<(unsigned)units, 64 * LT_WAVES, 0, stream>>>((const bf16_t*)qa, z, (const bf16_t*)pool, \
                                                                                      positions, tok_seq, block_table, max_blocks, \
                                                                                      n, H, K, R, page_size, n_pages, scale, window,  \
                                                                                      groups, n_split, part_o, part_ml, sink)
    if (nkw <= 1) FL_LTD(1, 1);
    else if (nkw <= 2) FL_LTD(2, 2);
    else if (nsw <= 2 && nkw <= 3) FL_LTD(3, 2);
    else if (nkw <= 4) FL_LTD(4, 4);
    else FL_LTD(5, 4);
#undef FL_LTD
    FL_LAUNCH_CHECK();
    if (n_split > 1) {
        dim3 mgrid(n * H, ceil_div(R, 256));
        latent_merge_kernel<<<mgrid, 256, 0, stream>>>(part_o, part_ml, z, H, R, groups, n_split, sink);
        FL_LAUNCH_CHECK();
    }
    return 0;
}
FL_RECORDABLE(fl_latent_attention_dealt)

// ------------------------------------------------------------------ one product per head on the matrix cores
// out[t][h][j] = sum_k x[t][h][k] w[h][j][k]   (x float or bfloat16 rows ldx apart, head h at h * hx; w bfloat16
// [H][J][K], K a multiple of 8, J of 16; heads ho apart in out), optionally times sigmoid(gate[t][gate_col0 + h]); tail:
// what stands behind a head's J results (query_tail.h).  A wave takes 16 tokens of one head: its x is
// the B operand, held in registers for all of K; the weights are the A operand, so a lane ends with four
// consecutive outputs of one token.
template <typename TX, typename TOut, int NS>
__global__ __launch_bounds__(64 * LT_WAVES) void heads_matmul_mfma_kernel(
    const TX* __restrict__ x, int ldx, int hx, const bf16_t* __restrict__ w, TOut* __restrict__ out, int ho, int n, int H, int K, int J,
    const float* __restrict__ gate, int ldg, int gate_col0, int j_parts, QueryTail tail) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    // a wave takes 16 tokens and every j_parts-th tile of 16 output columns (few tokens: many parts, so that
    // a decode step still fills the chip)
    const int unit = blockIdx.x * LT_WAVES + wave;
    const int t0 = (unit / j_parts) * 16, j_first = unit % j_parts, h = blockIdx.y;
    if (t0 >= n) return;
    const int col = lane & 15, g = lane >> 4;
    const int token = t0 + col;
    const bool live = token < n;
    bf16x8 xreg[NS];
    {
        const TX* xr = x + (size_t)(live ? token : t0) * ldx + (size_t)h * hx;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const bool inside = 32 * s + 8 * g < K;
            const TX* src = xr + (inside ? 32 * s + 8 * g : 0);        // (no branch around a load: what lies beyond K or n is set to zero afterwards)
            TX v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = src[e];
#pragma unroll
            for (int e = 0; e < 8; ++e) xreg[s][e] = inside && live ? (bf16_t)to_f32(v[e]) : (bf16_t)0.f;
        }
    }
    const float gv = (gate && live) ? 1.0f / (1.0f + expf(-gate[(size_t)token * ldg + gate_col0 + h])) : 1.0f;
    const bf16_t* wh = w + (size_t)h * J * K;
#pragma unroll 4
    for (int jt = j_first; jt < J / 16; jt += j_parts) {
        f32x4 acc = (f32x4){0.f, 0.f, 0.f, 0.f};
        const bf16_t* row = wh + (size_t)(16 * jt + col) * K + 8 * g;
#pragma unroll
        for (int s = 0; s < NS; ++s)
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8*)(32 * s + 8 * g < K ? row + 32 * s : row - 8 * g), xreg[s], acc, 0, 0, 0);      // (beyond K: finite weights against zeros)
        if (live) {
            TOut* dst = out + ((size_t)token * H + h) * ho + 16 * jt + 4 * g;
#pragma unroll
            for (int r = 0; r < 4; ++r) dst[r] = from_f32<TOut>(acc[r] * gv);
        }
    }
    if constexpr (std::is_same<TX, float>::value) {
        if (tail.width > 0 && j_first == 0)
            for (int e = lane; e < 16 * tail.width; e += 64) {
                const int i = e / tail.width, d = e - i * tail.width;
                if (t0 + i < n)
                    out[((size_t)(t0 + i) * H + h) * ho + J + d] =
                        from_f32<TOut>(query_tail_value(tail, x + (size_t)(t0 + i) * ldx + (size_t)h * hx, t0 + i, d));
            }
    }
}

// The same products for many tokens: a block of four waves takes 64 TW tokens of one head and a part of its columns.  The
// weights pass through LDS once per block, in chunks of 16 KB through a ring of three (copied as they lie, a row's 16-byte pieces
// exchanged by row % 8, with which the operand reads meet no bank twice; a range in place of conditions: what lies beyond K or J
// arrives as zeros); a wave holds its x for all of K in registers, as above, and sums in the same order: the same bits.
// What bounded the kernel above at 2,048 tokens of 32 heads were its weights, fetched by every 16 tokens from the L2 (537 MB), and its results, stored
// value by value: 128 -> 512 values per head 79 us, now 43 (2.9 TB/s of rows and results); 512 -> 128 76 us, now 39 (3.9 TB/s).
template <typename TX, typename TOut, int NS, int TW>
__global__ __launch_bounds__(256, 2) void heads_matmul_tiled_kernel(
    const TX* __restrict__ x, int ldx, int hx, const bf16_t* __restrict__ w, TOut* __restrict__ out, int ho, int n, int H, int K, int J,
    const float* __restrict__ gate, int ldg, int gate_col0, int chunks_per_part, int by_four, QueryTail tail) {
    constexpr int PK = 4 * NS, JR = 256 / NS, COPIES = 4;            // pieces of a row in LDS, rows of a chunk, copies of a wave per chunk
    // A tile's rows are not 16 neighbours but four of every 4 Q (row i of tile q: 4 Q (i / 4) + 4 q + i % 4 of 16 Q), so that a lane ends
    // with 4 Q neighbouring results and stores 16 bytes at a time.
    constexpr int Q = !std::is_same<TOut, bf16_t>::value ? 1 : JR / 16 < 4 ? JR / 16 : 4;      // (float results are 16 bytes by themselves)
    auto turn = [](int r) { return (r & 3) | ((r / (4 * Q) & 1) << 2); };
    __shared__ __attribute__((aligned(16))) bf16_t ring[3][JR * PK * 8];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int col = lane & 15, g = lane >> 4, h = blockIdx.y;
    const int t0 = (blockIdx.x * 4 + wave) * 16 * TW;
    bf16x8 xreg[TW][NS];
    float gv[TW];
#pragma unroll
    for (int u = 0; u < TW; ++u) {
        const int token = t0 + 16 * u + col;
        const bool live = token < n;
        const TX* xr = x + (size_t)(live ? token : 0) * ldx + (size_t)h * hx;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const bool inside = 32 * s + 8 * g < K;
            const TX* src = xr + (inside ? 32 * s + 8 * g : 0);        // (no branch around a load: what lies beyond K or n is set to zero afterwards)
            TX v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = src[e];
#pragma unroll
            for (int e = 0; e < 8; ++e) xreg[u][s][e] = inside && live ? (bf16_t)to_f32(v[e]) : (bf16_t)0.f;
            if (s % 8 == 7) __builtin_amdgcn_sched_barrier(0);         // (so many float values at a time beside those kept)
        }
        gv[u] = (gate && live) ? 1.0f / (1.0f + expf(-gate[(size_t)token * ldg + gate_col0 + h])) : 1.0f;
    }
    const int c_end = min((blockIdx.z + 1) * chunks_per_part, (J + JR - 1) / JR);
    const unsigned bytes = (unsigned)J * K * 2;
    const auto rows = __builtin_amdgcn_make_buffer_rsrc((void*)(w + (size_t)h * J * K), 0, bytes, 0x00020000);
    unsigned at[COPIES];
#pragma unroll
    for (int u = 0; u < COPIES; ++u) {
        const int slot = (wave * COPIES + u) * 64 + lane, r = slot / PK, piece = (slot % PK) ^ turn(r);
        at[u] = 8 * piece < K ? (unsigned)(r * K + 8 * piece) * 2 : 0x80000000u;
    }
    auto send = [&](int c) {
        if (c >= c_end) return;
#pragma unroll
        for (int u = 0; u < COPIES; ++u)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rows, (__attribute__((address_space(3))) void*)(ring[c % 3] + (wave * COPIES + u) * 512), 16,
                                                     at[u] + (unsigned)c * (JR * K * 2), 0, 0, 0);
    };
    const int c_begin = blockIdx.z * chunks_per_part;
    send(c_begin);
    send(c_begin + 1);
    for (int c = c_begin; c < c_end; ++c) {
        // this chunk is there when at most the next one's copies are under way (stores in between only make the wait longer)
        if (c + 1 < c_end) __builtin_amdgcn_s_waitcnt(0x0F70 | COPIES);
        else __builtin_amdgcn_s_waitcnt(0x0F70);
        asm volatile("s_barrier" ::: "memory");
        send(c + 2);                                                   // (into the place of the chunk that all have read)
        const bf16_t* chunk = ring[c % 3];
#pragma unroll
        for (int j1 = 0; j1 < JR; j1 += 16 * Q) {
            const int j0 = c * JR + j1 + 4 * Q * g;                     // this lane's first result
            f32x4 acc[TW][Q];
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                const int r = j1 + 4 * Q * (col >> 2) + 4 * q + (col & 3);
#pragma unroll
                for (int u = 0; u < TW; ++u) acc[u][q] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int s = 0; s < NS; ++s) {
                    const bf16x8 wv = *(const bf16x8*)(chunk + (r * PK + ((4 * s + g) ^ turn(r))) * 8);
#pragma unroll
                    for (int u = 0; u < TW; ++u) acc[u][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv, xreg[u][s], acc[u][q], 0, 0, 0);
                }
            }
#pragma unroll
            for (int u = 0; u < TW; ++u) {
                const int token = t0 + 16 * u + col;
                if (token >= n) continue;
                TOut* dst = out + ((size_t)token * H + h) * ho + j0;
#pragma unroll
                for (int q = 0; q < Q; ++q) acc[u][q] *= gv[u];
                if (by_four && j0 + 4 * Q <= J) {
                    if constexpr (std::is_same<TOut, bf16_t>::value && Q > 1) {
#pragma unroll
                        for (int q = 0; q < Q; q += 2)
                            *(bf16x8*)(dst + 4 * q) = (bf16x8){(bf16_t)acc[u][q][0], (bf16_t)acc[u][q][1], (bf16_t)acc[u][q][2], (bf16_t)acc[u][q][3],
                                                              (bf16_t)acc[u][q + 1][0], (bf16_t)acc[u][q + 1][1], (bf16_t)acc[u][q + 1][2], (bf16_t)acc[u][q + 1][3]};
                    } else if constexpr (std::is_same<TOut, bf16_t>::value) {
                        *(bf16x4*)dst = (bf16x4){(bf16_t)acc[u][0][0], (bf16_t)acc[u][0][1], (bf16_t)acc[u][0][2], (bf16_t)acc[u][0][3]};
                    } else {
#pragma unroll
                        for (int q = 0; q < Q; ++q) *(f32x4*)(dst + 4 * q) = acc[u][q];
                    }
                } else {
#pragma unroll
                    for (int q = 0; q < Q; ++q)
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            if (j0 + 4 * q + r < J) dst[4 * q + r] = from_f32<TOut>(acc[u][q][r]);
                }
            }
        }
        // (the operand reads are done before the next barrier lets anyone copy into their place)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    if constexpr (std::is_same<TX, float>::value) {
        if (tail.width > 0 && blockIdx.z == 0)
            for (int e = lane; e < 16 * TW * tail.width; e += 64) {
                const int i = e / tail.width, d = e - i * tail.width;
                if (t0 + i < n)
                    out[((size_t)(t0 + i) * H + h) * ho + J + d] =
                        from_f32<TOut>(query_tail_value(tail, x + (size_t)(t0 + i) * ldx + (size_t)h * hx, t0 + i, d));
            }
    }
}

extern "C" int fl_heads_matmul_mfma_takes(int K, int J) { return K > 0 && K % 8 == 0 && K <= 512 && J > 0 && J % 16 == 0; }

extern "C" int fl_heads_matmul_mfma(const void* x, int x_dtype, int ldx, int hx, const void* w, void* out, int out_dtype, int ho,
                                    int n, int H, int K, int J, const float* gate, int ldg, int gate_col0, int rot_dim, int rot,
                                    int interleaved, const float* cs, int rot_at, hipStream_t stream) {
    FL_CHECK(n >= 0 && H > 0 && hx >= K + rot_dim && ho >= J && (long)ldx >= (long)(H - 1) * hx + K + rot_dim, "heads_matmul_mfma: bad sizes");
    FL_CHECK(rot_dim >= 0 && rot >= 0 && rot % 2 == 0 && rot <= rot_dim && (rot == 0 || cs) && (rot_dim == 0 || (rot_at >= J && rot_at + rot_dim <= ho)),
             "heads_matmul_mfma: a rotated part of %d (%d turned) at %d of %d", rot_dim, rot, rot_at, ho);
    FL_CHECK(ho == J || x_dtype == FL_F32, "heads_matmul_mfma: what stands behind a head's results is made of float rows");
    const QueryTail tail = {ho - J, K, rot_at - J, rot_dim, rot, interleaved, cs};
    FL_CHECK(fl_heads_matmul_mfma_takes(K, J), "heads_matmul_mfma: %d x %d per head is not taken", J, K);
    FL_CHECK((uintptr_t)w % 16 == 0, "heads_matmul_mfma: the weights must be 16-byte aligned");
    FL_CHECK(!gate || ldg >= gate_col0 + H, "heads_matmul_mfma: gate columns beyond rows %d wide", ldg);
    if (n == 0) return 0;
    FL_CHECK(H <= 65535, "heads_matmul_mfma: too many heads");
    // Where there is enough to do for the blocks' way through LDS: 128 -> 256 with 16 heads 128 tokens 9.2 us above and 9.4 here, 200 tokens 10.5 and
    // 9.5; with rows of more than 256 values a block of every 64 tokens per unit (512 -> 128 with 32 heads: 200 tokens 15.2 and 15.8, 500 tokens 24.4 and 18.9;
    // 448 -> 112 with eight heads: 1,024 tokens 13.7 and 14.9, 2,048 tokens 20.8 and 15.9).
    const long tiles64 = (long)ceil_div(n, 64) * H;
    if (n > 64 && (K > 256 ? tiles64 >= fl_units() : tiles64 * K * J >= 1 << 21) && (long)J * K < (1L << 30)) {
        // two token tiles a wave where that leaves two blocks a unit and the registers hold their rows; else one, and the columns in parts
        const int ns = K <= 64 ? 2 : K <= 128 ? 4 : K <= 256 ? 8 : 16, chunks = ceil_div(J, 256 / ns);
        const bool two = K <= 256 && (long)ceil_div(n, 128) * H >= 2 * fl_units();
        const int blocks = ceil_div(n, two ? 128 : 64);
        int parts = (2 * fl_units()) / (blocks * H);
        parts = parts < 1 ? 1 : (parts > chunks ? chunks : parts);
        const int per = ceil_div(chunks, parts);
        dim3 grid(blocks, H, ceil_div(chunks, per));
        const int by_four = ho % 8 == 0 && (uintptr_t)out % 16 == 0;               // (16-byte stores)
#define FL_HMT(TX, TO, NS, TW) heads_matmul_tiled_kernel<TX, TO, NS, TW><<<grid, 256, 0, stream>>>((const TX*)x, ldx, hx, (const bf16_t*)w, (TO*)out, ho, n, H, K, J, gate, ldg, gate_col0, per, by_four, tail)
#define FL_HMT_NS(TX, TO, TW)                       \
    do {                                            \
        if (ns == 2) FL_HMT(TX, TO, 2, TW);         \
        else if (ns == 4) FL_HMT(TX, TO, 4, TW);    \
        else if (ns == 8) FL_HMT(TX, TO, 8, TW);    \
        else FL_HMT(TX, TO, 16, TW);                \
    } while (0)
#define FL_HMT_TW(TX, TO) do { if (two) FL_HMT_NS(TX, TO, 2); else FL_HMT_NS(TX, TO, 1); } while (0)
        if (x_dtype == FL_F32 && out_dtype == FL_BF16) FL_HMT_TW(float, bf16_t);
        else if (x_dtype == FL_F32 && out_dtype == FL_F32) FL_HMT_TW(float, float);
        else if (x_dtype == FL_BF16 && out_dtype == FL_BF16) FL_HMT_TW(bf16_t, bf16_t);
        else FL_CHECK(false, "heads_matmul_mfma: unsupported dtypes x=%d out=%d", x_dtype, out_dtype);
#undef FL_HMT_TW
#undef FL_HMT_NS
#undef FL_HMT
        FL_LAUNCH_CHECK();
        return 0;
    }
    // enough waves for four per compute unit, as far as the column tiles go
    const int groups = ceil_div(n, 16);
    int j_parts = (4 * fl_units()) / (groups * H);
    j_parts = j_parts < 1 ? 1 : (j_parts > J / 16 ? J / 16 : j_parts);
    dim3 grid(ceil_div(groups * j_parts, LT_WAVES), H);
    const int ns = (K + 31) / 32;
#define FL_HMM(TX, TO, NS) heads_matmul_mfma_kernel<TX, TO, NS><<<grid, 64 * LT_WAVES, 0, stream>>>((const TX*)x, ldx, hx, (const bf16_t*)w, (TO*)out, ho, n, H, K, J, gate, ldg, gate_col0, j_parts, tail)
#define FL_HMM_NS(TX, TO)                      \
    do {                                       \
        if (ns <= 2) FL_HMM(TX, TO, 2);        \
        else if (ns <= 4) FL_HMM(TX, TO, 4);   \
        else if (ns <= 8) FL_HMM(TX, TO, 8);   \
        else FL_HMM(TX, TO, 16);               \
    } while (0)
    if (x_dtype == FL_F32 && out_dtype == FL_BF16) FL_HMM_NS(float, bf16_t);
    else if (x_dtype == FL_F32 && out_dtype == FL_F32) FL_HMM_NS(float, float);
    else if (x_dtype == FL_BF16 && out_dtype == FL_BF16) FL_HMM_NS(bf16_t, bf16_t);
    else FL_CHECK(false, "heads_matmul_mfma: unsupported dtypes x=%d out=%d", x_dtype, out_dtype);
#undef FL_HMM_NS
#undef FL_HMM
    FL_LAUNCH_CHECK();
    return 0;
}
FL_RECORDABLE(fl_heads_matmul_mfma)
