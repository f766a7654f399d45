// Tiled grouped-query attention over the paged cache for prompt portions: bf16 storage, float
// softmax, matrix cores (v_mfma_f32_16x16x32_bf16).
//
// A block of four waves takes 64 consecutive query tokens of one request (16 per wave) and, for
// one kv head, QT of the query heads that share it (QT = 4, 2 or 1, a divisor of the group size):
// each wave holds QT query tiles and reuses every key/value operand it reads from LDS QT times.
// Keys are walked in stages of 64 from the first key any of the block's queries may see to the
// last, through a ring of LDS stages filled straight from the cache pages
// (global_load_lds_dwordx4: each lane names its own 16 bytes, the wave's kilobyte lands in tile
// order), one bare barrier per stage.  The block's part of the block table sits in LDS.
//
// Everything is computed transposed, so that a query is a lane column:
//   S^T[key][query] = K . Q^T        A = K tile (LDS, stored as matrix-core tiles), B = Q (registers)
//   softmax per column: the base m of the exponents and the sum l live in the lanes that own the
//       column; rescaling the output needs no broadcast and happens only when a base moves, which
//       it does lazily (when a score exceeds it by more than a factor of 256): the usual chunk
//       costs no exchange between lanes
//   O^T[d][query] += V^T . P^T       A = V^T tile (the cache stores values transposed inside a
//       page, so its rows are runs of keys), B = P straight from the S^T accumulator
// Scores are scaled by scale * log2(e) and exponentiated with exp2.  Query at position p sees keys
// [max(0, p - window + 1), p]; keys outside are excluded, never scored.
//
// Reference: crates/kernels-hip/src/kernels/attention_prefill_flash_tile_f16.cu:43-330 (tiled
// prefill, 4 query rows per tile), attention_prefill_f16_paged.cu:50-150 (paged addressing).
#include "common.h"
#include "api.h"
#include "recordable.h"
#include "attn_prefill.h"

template <int HDP, int QT, int NS>
__global__ __launch_bounds__(256, QT * HDP <= 256 ? 2 : 1) void attn_prefill_kernel(
    const bf16_t* __restrict__ q, bf16_t* __restrict__ out, PagedCache cache,
    const int* __restrict__ tiles, const int* __restrict__ positions,
    const int* __restrict__ block_table, int max_blocks, int nh, float scale_log2e, float cap_raw, int window,
    int log2_ps, int mirror_from, float* __restrict__ part_o, float* __restrict__ part_ml, const float* __restrict__ sink) {
    attn_prefill_block<HDP, QT, NS>({blockIdx.x, blockIdx.y, blockIdx.z}, {gridDim.x, gridDim.y, gridDim.z}, q, out, cache, tiles, positions, block_table,
                                    max_blocks, nh, scale_log2e, cap_raw, window, log2_ps, mirror_from, part_o, part_ml, sink);
}

template <int HDP, int QT, int NS>
static void launch_prefill_one(dim3 grid, hipStream_t stream, const bf16_t* q, bf16_t* out, PagedCache c,
                               const int* tiles, const int* positions, const int* block_table, int max_blocks,
                               int nh, float scale_log2e, float cap_raw, int window, int log2_ps, float* part_o, float* part_ml, int lds_pages, const float* sink) {
    // blocks that the chip holds at one time: one or two per compute unit
    const int units = fl_units();
    const int total = (int)(grid.x * grid.y * grid.z);
    constexpr int RING = attn_prefill_ring<HDP, NS>();
    const int lds = RING + lds_pages * (int)sizeof(int);
    const int resident = units * ((QT * HDP <= 256 && 2 * lds <= PF_LDS_BYTES) ? 2 : 1);
    // (whole rows of the grid: every tile of a head group is taken exactly once either way)
    const int mirror_from = (resident == 2 * units && grid.z == 1 && total <= resident && total > units) ? (int)((grid.y / 2) * grid.x)
                            : (grid.z == 1 && total > resident) ? -1 : (int)(grid.x * grid.y);
    static bool configured = false;
    auto kern = attn_prefill_kernel<HDP, QT, NS>;
    if (!configured) {
        (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                  min(RING + PF_MAX_PAGES * (int)sizeof(int), PF_LDS_BYTES));
        configured = true;
    }
    kern<<<grid, 256, lds, stream>>>(q, out, c, tiles, positions, block_table, max_blocks, nh, scale_log2e, cap_raw, window, log2_ps, mirror_from, part_o, part_ml, sink);
}

template <int HDP, int NS>
static void launch_prefill(int qt, dim3 grid, hipStream_t stream, const bf16_t* q, bf16_t* out, PagedCache c,
                           const int* tiles, const int* positions, const int* block_table, int max_blocks, int nh,
                           float scale_log2e, float cap_raw, int window, int log2_ps, float* part_o, float* part_ml, int lds_pages, const float* sink) {
    if constexpr (HDP <= 64) {            // four heads per wave only where two blocks still fit a compute unit
        if (qt == 4) {
            launch_prefill_one<HDP, 4, NS>(grid, stream, q, out, c, tiles, positions, block_table, max_blocks, nh, scale_log2e, cap_raw, window, log2_ps, part_o, part_ml, lds_pages, sink);
            return;
        }
    }
    if (qt >= 2)
        launch_prefill_one<HDP, 2, NS>(grid, stream, q, out, c, tiles, positions, block_table, max_blocks, nh, scale_log2e, cap_raw, window, log2_ps, part_o, part_ml, lds_pages, sink);
    else
        launch_prefill_one<HDP, 1, NS>(grid, stream, q, out, c, tiles, positions, block_table, max_blocks, nh, scale_log2e, cap_raw, window, log2_ps, part_o, part_ml, lds_pages, sink);
}

// Query heads per wave (QT, a divisor of the group size) and parts of the keys for a batch of n_tiles
// tiles whose longest context has max_keys keys.
//  * At most as many heads as leave room for two blocks per compute unit (two waves per SIMD hide each
//    other's waits: 906 against 1314 us at 8192 tokens with 2 heads instead of 4 at head size 128).
//  * A grid of fewer than two blocks per unit is filled by splitting the keys, as long as every part keeps
//    12 stages of 64 keys or so, rather than by fewer heads per wave: a block of two heads reads its keys
//    and values once for both (512 tokens behind 7,680 keys: 99 us with two heads and 4 parts against 125
//    with one head and 2; behind 32,256: 314 against 422; 64 tokens behind 32,704: 83 against 115).
//  * Where the keys are too few for that (a whole prompt of 1,024 tokens: 16 stages at most), fewer heads
//    per wave give the blocks (29 us with one head, 35 with two).
//  * Blocks of single rows that run beside (fl_attn_both) may have one of a unit's two places (beside = units): the grid then is as many
//    blocks fewer (512 tokens behind up to 1,536 beside 16 rows of 500 to 4,096 keys: 57 us with 4 parts of the keys, 51 with 2, merges
//    and all; 1: 55).  When they have is the caller's rule: beside few rows' keys half a grid is the slower one.
struct PrefillPlan { int qt, splits; };
static PrefillPlan pf_plan(int n_tiles, int nh, int nkv, int hd, int max_keys, int beside) {
    const int G = nh / nkv;
    const int hdp = ceil_div(hd, 32) * 32;
    int qt = (G % 4 == 0) ? 4 : (G % 2 == 0 ? 2 : 1);
    const int qt_max = hdp <= 64 ? 4 : 2;
    while (qt > qt_max) qt /= 2;
    const int slots = 2 * fl_units() - min(max(beside, 0), fl_units());
    const int by_keys = max(1, ceil_div(max(max_keys, 1), PF_STAGE) / 12);
    for (;; qt /= 2) {
        const int blocks = max(1, n_tiles * nkv * (G / qt));
        if (blocks >= slots) return {qt, 1};
        const int splits = max(1, min(min(slots / blocks, by_keys), 16));
        // (at the most parts there are, fewer heads would only read the keys more often)
        if (qt == 1 || splits == 16 || blocks * splits >= slots * 5 / 8) return {qt, splits};
    }
}

// query heads per wave for fl_attn_prefill: qt_hint (1, 2 or 4) at most that many; else what goes with
// the parts the caller has chosen
static int pf_heads_per_wave(int n_tiles, int nh, int nkv, int hd, int qt_hint, int n_split) {
    const int G = nh / nkv;
    const int hdp = ceil_div(hd, 32) * 32;
    int qt = (G % 4 == 0) ? 4 : (G % 2 == 0 ? 2 : 1);
    const int qt_max = hdp <= 64 ? 4 : 2;
    while (qt > qt_max) qt /= 2;
    if (qt_hint == 1 || qt_hint == 2 || qt_hint == 4) {
        while (qt > qt_hint) qt /= 2;
        return qt;
    }
    while (qt > 1 && n_tiles * nkv * (G / qt) * n_split < 3 * fl_units() / 2) qt /= 2;
    return qt;
}

// Query heads per wave for a batch of this shape (what fl_attn_prefill takes as its hint), and into how
// many parts its keys are split (1: not at all); `beside`: blocks of single rows in the same launch (fl_attn_both).
extern "C" int fl_attn_prefill_heads(int n_tiles, int nh, int nkv, int hd, int max_keys, int beside) {
    if (n_tiles <= 0 || nh <= 0 || nkv <= 0 || nh % nkv) return 1;
    return pf_plan(n_tiles, nh, nkv, hd, max_keys, beside).qt;
}
extern "C" int fl_attn_prefill_splits(int n_tiles, int nh, int nkv, int hd, int max_keys, int beside) {
    if (n_tiles <= 0 || nh <= 0 || nkv <= 0 || nh % nkv) return 1;
    return pf_plan(n_tiles, nh, nkv, hd, max_keys, beside).splits;
}

// Block-table entries per request that the kernel takes at a head size: the table of a request sits in
// LDS beside the ring of two stages of 64 keys and values (256 bytes per padded head dim and stage).
extern "C" int fl_attn_prefill_max_pages(int hd) {
    if (hd <= 0 || hd > 256) return 0;
    const int hdp = ceil_div(hd, 32) * 32;
    return min(PF_MAX_PAGES, (PF_LDS_BYTES - 2 * hdp * 256) / (int)sizeof(int));
}

// Entries of a request's table that a block may need: all of them, or with a window the pages of the
// window + 63 keys that its 64 queries see between them.
static int pf_table_need(int max_blocks, int page_size, int window) {
    if (window <= 0) return max_blocks;
    return min(max_blocks, (window + PF_TOKENS - 2) / page_size + 2);
}

// Whether fl_attn_prefill takes a cache of this shape with block tables max_blocks wide.
extern "C" int fl_attn_prefill_takes(int hd, int page_size, int max_blocks, int window) {
    if (hd <= 0 || hd > 256 || hd % 8 || page_size < 8 || (page_size & (page_size - 1)) || max_blocks < 0 || window < 0) return 0;
    return pf_table_need(max_blocks, page_size, window) <= fl_attn_prefill_max_pages(hd) ? 1 : 0;
}

// Workspace of the split form, in floats: part_o and part_ml for n_rows rows of tiles.
extern "C" int fl_attn_prefill_workspace(int n_rows, int nh, int hd, int n_split, long* o_floats, long* ml_floats) {
    const int hdp = ceil_div(hd, 32) * 32;
    *o_floats = (long)n_rows * nh * n_split * hdp;
    *ml_floats = (long)n_rows * nh * n_split * 2;
    return 0;
}

__global__ __launch_bounds__(256) void attn_prefill_merge_kernel(const float* __restrict__ part_o,
                                                                 const float* __restrict__ part_ml,
                                                                 bf16_t* __restrict__ out, const int* __restrict__ tiles,
                                                                 int nh, int hd, int hdp, int n_split, int blocks_per_tile,
                                                                 const float* __restrict__ sink) {
    attn_prefill_merge_block(blockIdx.x, part_o, part_ml, out, tiles, nh, hd, hdp, n_split, blocks_per_tile, sink);
}

int attn_prefill_prepare(const char* who, int n_tiles, int max_blocks, int nh, int nkv, int hd, int page_size, float scale, int window, int qt_hint,
                         const float* part_o, const float* part_ml, int n_split, float softcap, PrefillLaunch* launch) {
    FL_CHECK(n_tiles >= 0 && nh > 0 && nkv > 0 && nh % nkv == 0, "%s: bad head counts %d/%d", who, nh, nkv);
    FL_CHECK(hd > 0 && hd <= 256 && hd % 8 == 0, "%s: head size %d must be a multiple of 8 up to 256", who, hd);
    FL_CHECK(page_size >= 8 && (page_size & (page_size - 1)) == 0,
             "%s: page size %d must be a power of two, at least 8", who, page_size);
    FL_CHECK((long long)2 * nkv * page_size * hd < (1ll << 31), "%s: a page of %d heads x %d keys x %d is too large (2^31 values)", who, nkv, page_size, hd);
    FL_CHECK(window >= 0, "%s: negative window", who);
    const int lds_pages = pf_table_need(max_blocks, page_size, window);
    FL_CHECK(lds_pages <= fl_attn_prefill_max_pages(hd), "%s: %d pages per request in reach of a block, at most %d with heads of %d", who,
             lds_pages, fl_attn_prefill_max_pages(hd), hd);
    FL_CHECK(scale > 0.f, "%s: the score scale must be positive", who);
    FL_CHECK(n_split >= 1 && n_split <= 16, "%s: %d splits (at most 16)", who, n_split);
    FL_CHECK(n_split == 1 || (part_o && part_ml && (uintptr_t)part_o % 16 == 0), "%s: splits need a 16-byte aligned workspace", who);
    FL_CHECK(n_split == 1 || (long long)n_tiles * PF_TOKENS * nh * (ceil_div(hd, 32) * 8) / 256 < (1ll << 31),
             "%s: %d tiles are too many to split", who, n_tiles);
    const int hdp = ceil_div(hd, 32) * 32;
    int log2_ps = 0;
    while ((1 << log2_ps) < page_size) ++log2_ps;
    const int qt = pf_heads_per_wave(n_tiles, nh, nkv, hd, qt_hint, n_split);
    *launch = {dim3(n_tiles, nkv * (nh / nkv / qt), n_split), qt, hdp, lds_pages, log2_ps, ceil_div(PF_TOKENS * nh * (hdp / 4), 256),
               scale * 1.4426950408889634f, softcap > 0.f ? softcap / scale : 0.f};
    return 0;
}

// tiles[n_tiles][4] = (row of the request in the block table, first row, rows (at most 64), index of
// the first row among all rows of tiles).  n_split > 1 (fl_attn_prefill_splits): the keys are split,
// part_o and part_ml hold fl_attn_prefill_workspace floats.
static int attn_prefill_launch(const void* q, void* out, const void* cache_base, const int* tiles,
                               int n_tiles, const int* positions, const int* block_table,
                               int max_blocks, int nh, int nkv, int hd, int page_size, int n_pages,
                               float scale, int window, int qt_hint, float* part_o, float* part_ml, int n_split,
                               float softcap, const float* sink, hipStream_t stream) {
    PrefillLaunch l;
    if (attn_prefill_prepare("attn_prefill", n_tiles, max_blocks, nh, nkv, hd, page_size, scale, window, qt_hint, part_o, part_ml, n_split, softcap, &l)) return -1;
    if (n_tiles == 0) return 0;
    PagedCache c{(void*)cache_base, nkv, page_size, hd, n_pages};
    // a ring of two stages: two blocks then fit a compute unit (three stages were no faster)
#define FL_PF(HDP_)                                                                                            \
    launch_prefill<HDP_, 2>(l.heads_per_wave, l.grid, stream, (const bf16_t*)q, (bf16_t*)out, c, tiles, positions, block_table, \
                            max_blocks, nh, l.scale_log2e, l.cap_raw, window, l.log2_page, part_o, part_ml, l.lds_pages, sink)
    switch (l.hdp) {
        case 32: FL_PF(32); break;
        case 64: FL_PF(64); break;
        case 96: FL_PF(96); break;
        case 128: FL_PF(128); break;
        case 160: FL_PF(160); break;
        case 192: FL_PF(192); break;
        case 224: FL_PF(224); break;
        default: FL_PF(256); break;
    }
#undef FL_PF
    FL_LAUNCH_CHECK();
    if (n_split > 1) {
        attn_prefill_merge_kernel<<<n_tiles * l.merge_blocks_per_tile, 256, 0, stream>>>(part_o, part_ml, (bf16_t*)out, tiles, nh, hd, l.hdp, n_split,
                                                                                         l.merge_blocks_per_tile, sink);
        FL_LAUNCH_CHECK();
    }
    return 0;
}

extern "C" int fl_attn_prefill(const void* q, void* out, const void* cache_base, const int* tiles,
                               int n_tiles, const int* positions, const int* block_table,
                               int max_blocks, int nh, int nkv, int hd, int page_size, int n_pages,
                               float scale, int window, int qt_hint, float* part_o, float* part_ml, int n_split,
                               hipStream_t stream) {
    return attn_prefill_launch(q, out, cache_base, tiles, n_tiles, positions, block_table, max_blocks, nh, nkv, hd, page_size,
                               n_pages, scale, window, qt_hint, part_o, part_ml, n_split, 0.f, nullptr, stream);
}
FL_RECORDABLE(fl_attn_prefill)

// the same with the scores capped, score <- softcap * tanh(score / softcap) before the softmax (softcap > 0; 0: as they
// are), and with a sink per query head in the denominator (sink float [nh], or null)
extern "C" int fl_attn_prefill_capped(const void* q, void* out, const void* cache_base, const int* tiles,
                                      int n_tiles, const int* positions, const int* block_table,
                                      int max_blocks, int nh, int nkv, int hd, int page_size, int n_pages,
                                      float scale, int window, float softcap, const float* sink, int qt_hint, float* part_o, float* part_ml,
                                      int n_split, hipStream_t stream) {
    FL_CHECK(softcap >= 0.f, "attn_prefill: negative cap");
    return attn_prefill_launch(q, out, cache_base, tiles, n_tiles, positions, block_table, max_blocks, nh, nkv, hd, page_size,
                               n_pages, scale, window, qt_hint, part_o, part_ml, n_split, softcap, sink, stream);
}
FL_RECORDABLE(fl_attn_prefill_capped)
