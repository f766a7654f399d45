// Split-K grouped-query attention over the paged cache for single query rows (decode rows, and
// the rows of short prompt portions): bf16 storage, float arithmetic, matrix cores.
//
// Work item = (query row, kv head, split); a query row comes as (row, position, request, 0), or, with
// splits of its own, once per split as (row, position, request, split + 256 * splits): the caller
// then gives long contexts more splits than short ones, and the blocks take about equally long
// (with one number of splits for all, the longest context of a ragged batch ends the kernel alone).  A
// block of four waves handles the (up to 16) query heads that share one kv head over the keys of
// its split, 32 keys per wave at a time:
//
//   S^T[key][head] = K[key][:] . Q[head][:]     v_mfma_f32_16x16x32_bf16, A = K rows read
//                                               straight from the cache pages (head dims are
//                                               contiguous), B = Q (kept in registers)
//   per head (one lane column): running max and sum; scores and their exponentials never leave
//   the lane that owns the column, so no broadcast is needed to rescale
//   O^T[d][head]  += V^T[d][key] . P^T[key][head]   A = values, which the cache stores transposed
//                                               inside a page (keys contiguous: one 16-byte load
//                                               per lane), B = P from the S^T accumulator without
//                                               any data movement
//
// The four waves' states are merged through LDS; with more than one split the block writes a
// partial (max, sum, O) and a second kernel merges the splits (same rule: exp(m_c - m_max)).
// (Merging in the block that finishes last was tried twice: with a device-wide release fence in every
// block it is far slower, since each fence writes the L2 back, one block after the other; with
// device-scope loads and stores and a relaxed counter instead of fences it takes as long as the second
// kernel that it saves.)  Keys and values are loaded with the non-temporal hint: a step reads each
// byte of them once, and streaming reads are a tenth faster with the hint.
// Which keys a row sees depends on its own position only: [max(0, p - window + 1), p].
//
// Reference: crates/kernels-hip/src/kernels/attention_decode_f16_paged.cu:49-158 (paged decode),
// attention_decode_f16_splitk.cu:31-256 (partials and merge).
#include "common.h"
#include "api.h"
#include "recordable.h"
#include "attn_decode.h"
#include <mutex>

template <int HDP>
__global__ __launch_bounds__(256, HDP <= 128 ? 2 : 1) void attn_decode_kernel(
    const bf16_t* __restrict__ q, bf16_t* __restrict__ out, float* part_o,
    float* part_ml, PagedCache cache, const int4* __restrict__ items,
    const int* __restrict__ block_table, int max_blocks, int nh, float scale, int window,
    int n_split, int q_tiles, int ps_shift, int item_base, float softcap, const float* __restrict__ sink) {
    __shared__ DecodeLds<HDP> lds;
    attn_decode_block<HDP>(lds, {blockIdx.x, blockIdx.y, blockIdx.z}, q, out, part_o, part_ml, cache, items, block_table, max_blocks, nh, scale, window, n_split,
                           q_tiles, ps_shift, item_base, softcap, sink);
}

// Merge of the splits: one block per (item, head) (attn_merge.h).
__global__ __launch_bounds__(256) void attn_decode_merge_kernel(const float* __restrict__ part_o,
                                                                const float* __restrict__ part_ml,
                                                                bf16_t* __restrict__ out,
                                                                const int4* __restrict__ items, int nh,
                                                                int hd, int hdp, int n_split) {
    const int item = blockIdx.x, head = blockIdx.y;
    const int token = items[item].x;
    attn_merge_splits(part_o, part_ml, out + ((size_t)token * nh + head) * hd, ((size_t)item * nh + head) * n_split, hd, hdp,
                      n_split);
}

// The same for items with splits of their own, which lie nh slots apart: one block per (row, head); firsts[r] =
// (row, index of the row's first item, its splits, 0).
__global__ __launch_bounds__(256) void attn_decode_merge_items_kernel(const float* __restrict__ part_o,
                                                                      const float* __restrict__ part_ml,
                                                                      bf16_t* __restrict__ out,
                                                                      const int4* __restrict__ items,
                                                                      const int4* __restrict__ firsts, int nh,
                                                                      int hd, int hdp, const float* __restrict__ sink) {
    const int head = blockIdx.y;
    const int4 row = firsts[blockIdx.x];
    const int first = row.y, n_split = row.z;
    if (n_split <= 1) return;
    attn_merge_splits(part_o, part_ml, out + ((size_t)row.x * nh + head) * hd, (size_t)first * nh + head, hd, hdp, n_split,
                      (size_t)nh, sink ? sink + head : nullptr);
}

extern "C" int fl_attn_decode_workspace(int n_items, int nh, int hd, int n_split, long* o_floats,
                                        long* ml_floats) {
    const int hdp = ceil_div(hd, 32) * 32;
    *o_floats = (long)n_items * nh * n_split * hdp;
    *ml_floats = (long)n_items * nh * n_split * 2;
    return 0;
}

int attn_decode_prepare(const char* who, const int* items, int n_items, int nh, int nkv, int hd, int page_size, int window, int n_split, bool own_splits,
                        const float* part_o, const float* part_ml, const float* sink, int* ps_shift) {
    FL_CHECK(n_items >= 0 && nh > 0 && nkv > 0 && nh % nkv == 0, "%s: bad head counts %d/%d", who, nh, nkv);
    FL_CHECK(hd > 0 && hd <= 256 && hd % 8 == 0, "%s: head size %d must be a multiple of 8 up to 256", who, hd);
    FL_CHECK(page_size % 8 == 0, "%s: page size %d must be a multiple of 8", who, page_size);
    FL_CHECK(n_split >= 1 && n_split <= 256, "%s: %d splits", who, n_split);
    FL_CHECK(n_split == 1 || (part_o && part_ml), "%s: splits need a workspace", who);
    FL_CHECK(window >= 0, "%s: negative window", who);
    FL_CHECK(!sink || own_splits, "%s: a sink comes with rows that have splits of their own", who);
    FL_CHECK((uintptr_t)items % 16 == 0, "%s: the items must be 16-byte aligned", who);
    *ps_shift = -1;
    if ((page_size & (page_size - 1)) == 0)
        for (*ps_shift = 0; (1 << *ps_shift) < page_size; ++*ps_shift) {}
    return 0;
}

static int attn_decode_launch(const char* who, const void* q, void* out, float* part_o, float* part_ml,
                              const void* cache_base, const int* items, int n_items, const int* block_table,
                              int max_blocks, int nh, int nkv, int hd, int page_size, int n_pages,
                              float scale, int window, int n_split, hipStream_t stream, bool own_splits = false,
                              const int* firsts = nullptr, int n_rows = 0, float softcap = 0.f, const float* sink = nullptr) {
    int ps_shift;
    if (attn_decode_prepare(who, items, n_items, nh, nkv, hd, page_size, window, n_split, own_splits, part_o, part_ml, sink, &ps_shift)) return -1;
    if (n_items == 0) return 0;
    PagedCache c{(void*)cache_base, nkv, page_size, hd, n_pages};
    const int G = nh / nkv;
    const int q_tiles = ceil_div(G, 16);
    const int hdp = ceil_div(hd, 32) * 32;
    // a grid's slow index holds 65,535 places: longer lists of items take several launches
    for (int item_base = 0; item_base < n_items; item_base += 65535) {
        dim3 grid(nkv * q_tiles, min(n_items - item_base, 65535), own_splits ? 1 : n_split);
#define FL_DEC(HDP_)                                                                                  \
    attn_decode_kernel<HDP_><<<grid, 256, 0, stream>>>((const bf16_t*)q, (bf16_t*)out, part_o, part_ml, c,       \
                                                       (const int4*)items, block_table, max_blocks, nh, scale,   \
                                                       window, n_split, q_tiles, ps_shift, item_base, softcap, sink)
        switch (hdp) {
            case 32: FL_DEC(32); break;
            case 64: FL_DEC(64); break;
            case 96: FL_DEC(96); break;
            case 128: FL_DEC(128); break;
            case 160: FL_DEC(160); break;
            case 192: FL_DEC(192); break;
            case 224: FL_DEC(224); break;
            default: FL_DEC(256); break;
        }
#undef FL_DEC
        FL_LAUNCH_CHECK();
    }
    if (own_splits) {
        if (firsts && n_rows > 0) {              // (without: the caller knows that no row has more than one split)
            FL_CHECK((uintptr_t)firsts % 16 == 0, "%s: the rows' first items must be 16-byte aligned", who);
            dim3 mg(n_rows, nh);
            attn_decode_merge_items_kernel<<<mg, 256, 0, stream>>>(part_o, part_ml, (bf16_t*)out, (const int4*)items,
                                                                   (const int4*)firsts, nh, hd, hdp, sink);
            FL_LAUNCH_CHECK();
        }
    } else if (n_split > 1) {
        dim3 mg(n_items, nh);
        attn_decode_merge_kernel<<<mg, 256, 0, stream>>>(
            part_o, part_ml, (bf16_t*)out, (const int4*)items, nh, hd, hdp, n_split);
        FL_LAUNCH_CHECK();
    }
    return 0;
}

extern "C" int fl_attn_decode(const void* q, void* out, float* part_o, float* part_ml,
                              const void* cache_base, const int* items, int n_items, const int* block_table,
                              int max_blocks, int nh, int nkv, int hd, int page_size, int n_pages,
                              float scale, int window, int n_split, hipStream_t stream) {
    return attn_decode_launch("attn_decode", q, out, part_o, part_ml, cache_base, items, n_items, block_table, max_blocks,
                              nh, nkv, hd, page_size, n_pages, scale, window, n_split, stream);
}
FL_RECORDABLE(fl_attn_decode)

// Items with splits of their own: items[i] = (row, position, request, split + 256 * splits), the splits of
// a row one after the other from split 0 on (up to 255), row < 0 for a place that is not used.  part_o
// holds n_items * nh * (head size rounded up to 32) floats, part_ml n_items * nh * 2.  firsts[r] = (row,
// index of the row's first item, its splits, 0) for the n_rows rows; without it no row has more
// than one split (a list with a place per row and no more) and the kernel that merges is left out.
extern "C" int fl_attn_decode_items(const void* q, void* out, float* part_o, float* part_ml, const void* cache_base,
                                    const int* items, int n_items, const int* block_table, int max_blocks, int nh,
                                    int nkv, int hd, int page_size, int n_pages, float scale, int window,
                                    const int* firsts, int n_rows, hipStream_t stream) {
    FL_CHECK(!firsts || (part_o && part_ml), "attn_decode_items: needs a workspace");
    return attn_decode_launch("attn_decode_items", q, out, part_o, part_ml, cache_base, items, n_items, block_table, max_blocks,
                              nh, nkv, hd, page_size, n_pages, scale, window, 1, stream, true, firsts, n_rows);
}
FL_RECORDABLE(fl_attn_decode_items)

// the same with the scores capped, score <- softcap * tanh(score / softcap) before the softmax (softcap > 0; 0: as they
// are), and with a sink per query head in the denominator (sink float [nh], or null)
extern "C" int fl_attn_decode_items_capped(const void* q, void* out, float* part_o, float* part_ml, const void* cache_base,
                                           const int* items, int n_items, const int* block_table, int max_blocks, int nh,
                                           int nkv, int hd, int page_size, int n_pages, float scale, int window,
                                           float softcap, const float* sink, const int* firsts, int n_rows, hipStream_t stream) {
    FL_CHECK(!firsts || (part_o && part_ml), "attn_decode_items: needs a workspace");
    FL_CHECK(softcap >= 0.f, "attn_decode_items: negative cap");
    return attn_decode_launch("attn_decode_items", q, out, part_o, part_ml, cache_base, items, n_items, block_table, max_blocks,
                              nh, nkv, hd, page_size, n_pages, scale, window, 1, stream, true, firsts, n_rows, softcap, sink);
}
FL_RECORDABLE(fl_attn_decode_items_capped)

// ---- the same without any allocation: the splits' partial results go to an array that is part of
// the library's image on every GPU.  `scratch` is a host-side stand-in for that array, not a device
// address; its address on the current device is asked for once per device and kept.
static __device__ __align__(256) float scratch[FL_ATTN_DECODE_STATIC_FLOATS];

#define FL_MAX_DEVICES 64
static float* g_scratch_ptr[FL_MAX_DEVICES];       // per device: where `scratch` lies there
static std::mutex g_scratch_mutex;

static int static_scratch(float** ptr) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    FL_CHECK(e == hipSuccess, "attn_decode_static: hipGetDevice failed: %s", hipGetErrorString(e));
    FL_CHECK(dev >= 0 && dev < FL_MAX_DEVICES, "attn_decode_static: device %d, at most %d are known", dev, FL_MAX_DEVICES);
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        float* p = nullptr;
        e = hipGetSymbolAddress((void**)&p, HIP_SYMBOL(scratch));
        FL_CHECK(e == hipSuccess && p, "attn_decode_static: hipGetSymbolAddress failed on device %d: %s", dev,
                 hipGetErrorString(e));
        g_scratch_ptr[dev] = p;
    }
    *ptr = g_scratch_ptr[dev];
    return 0;
}

extern "C" long fl_attn_decode_static_capacity(void) { return (long)FL_ATTN_DECODE_STATIC_FLOATS; }

extern "C" int fl_attn_decode_static(const void* q, void* out, const void* cache_base, const int* items, int n_items,
                                     const int* block_table, int max_blocks, int nh, int nkv, int hd, int page_size,
                                     int n_pages, float scale, int window, int n_split, hipStream_t stream) {
    float* part_o = nullptr;
    float* part_ml = nullptr;
    if (n_split > 1 && n_items > 0) {
        FL_CHECK(nh > 0 && hd > 0 && hd <= 256 && n_split <= 256, "attn_decode_static: bad sizes (%d heads, head size %d, %d splits)",
                 nh, hd, n_split);
        const long hdp = ceil_div(hd, 32) * 32;
        const long slots = (long)n_items * nh * n_split;
        const long o_floats = (slots * hdp + 63) / 64 * 64;          // the pairs start 256-byte aligned
        const long need = o_floats + slots * 2;
        FL_CHECK(need <= (long)FL_ATTN_DECODE_STATIC_FLOATS,
                 "attn_decode_static: %d rows x %d heads x %d splits need %ld floats of scratch, the static array holds %ld "
                 "(use fl_attn_decode with a workspace, or fewer splits)",
                 n_items, nh, n_split, need, (long)FL_ATTN_DECODE_STATIC_FLOATS);
        float* base = nullptr;
        if (static_scratch(&base) != 0) return -1;
        part_o = base;
        part_ml = base + o_floats;
    }
    return attn_decode_launch("attn_decode_static", q, out, part_o, part_ml, cache_base, items, n_items, block_table,
                              max_blocks, nh, nkv, hd, page_size, n_pages, scale, window, n_split, stream);
}
FL_RECORDABLE(fl_attn_decode_static)
