// Attention of a step that holds prompt portions and single rows (decoding requests beside a prompt): the tiles of attn_prefill.hip and the items of
// attn_decode.hip in ONE launch, their merges in another.
//
// The tiles fill the vector unit, the single rows wait for the lines that a compute unit has in flight; one behind the other each leaves the other half
// idle and has a slow end and a launch of its own.  Here a unit, which holds two blocks, mostly has one of either kind: kinds take turns after as many
// blocks as there are units, in proportion to their numbers (a unit's first and second block are that far apart; changed every 8 blocks, units got two of
// one kind: 47 us, every 256 blocks 45, every 512 49).  The tiles' keys are then split over fewer blocks (pf_plan), which leaves less to merge.
// What bounds it: the lines in flight, which the tiles' keys and values share: of 512 tokens behind up to 1,536 beside 16 rows of 500 to 4,096 keys the
// kernels of their own take 24 + 27 us and 9 + 6 of merges, these 42 + 10.  A layer's attention apart and in one: 64 tokens behind 2,000 beside one row of 1,500
// 42 / 34 us, 128 behind 4,000 beside 16 of 1,000 53 / 40, 512 behind 1,536 beside 16 of 2,000 67 / 49, 1,024 behind 2,000 beside 32 of 4,000 158 / 113, a prompt of
// 2,048 beside one row of 300 72 / 66 (whose tiles run longest first here: in the order of attn_prefill.hip, mirrored, 69, beside more rows up to 30 % slower), of 1,280 59 / 45.
//
// Both are the code of the kernels of their own, so results are the same bits.
#include "common.h"
#include "api.h"
#include "recordable.h"
#include "attn_prefill.h"
#include "attn_decode.h"

struct BothTiles {
    const int* tiles;
    const int* positions;
    float scale_log2e, cap_raw;
    int log2_page, mirror_from;
    float* part_o;
    float* part_ml;
    dim3 grid;
};
struct BothItems {
    const int4* items;
    float scale, softcap;
    int q_tiles, per_item, n;              // per_item: blocks of an item
    float* part_o;
    float* part_ml;
};

template <int HDP, int QT>
__global__ __launch_bounds__(256, 2) void attn_both_kernel(const bf16_t* __restrict__ q, bf16_t* __restrict__ out, PagedCache cache,
                                                           const int* __restrict__ block_table, int max_blocks, int nh, int window,
                                                           const float* __restrict__ sink, BothTiles t, BothItems r, unsigned turn, unsigned tile_turns, unsigned item_turns) {
    static_assert(QT * HDP <= 256 && HDP <= 128);          // (both kernels of their own hold two blocks to a unit)
    extern __shared__ __attribute__((aligned(16))) bf16_t ring[];
    const unsigned at = blockIdx.x / turn, within = blockIdx.x % turn, all = tile_turns + item_turns;
    const unsigned items_before = at * item_turns / all;
    if ((at + 1) * item_turns / all > items_before) {
        const unsigned b = items_before * turn + within;
        if (b >= (unsigned)r.n * r.per_item) return;
        attn_decode_block<HDP>(*(DecodeLds<HDP>*)ring, {b % r.per_item, b / r.per_item, 0}, q, out, r.part_o, r.part_ml, cache, r.items, block_table, max_blocks, nh,
                               r.scale, window, 1, r.q_tiles, t.log2_page, 0, r.softcap, sink);
    } else {
        const unsigned b = (at - items_before) * turn + within;
        const unsigned plane = t.grid.x * t.grid.y;
        if (b >= plane * t.grid.z) return;
        attn_prefill_block<HDP, QT, 2>({b % t.grid.x, b % plane / t.grid.x, b / plane}, {t.grid.x, t.grid.y, t.grid.z}, q, out, cache, t.tiles, t.positions, block_table,
                                       max_blocks, nh, t.scale_log2e, t.cap_raw, window, t.log2_page, t.mirror_from, t.part_o, t.part_ml, sink);
    }
}

// The merges of both: first the blocks of the tiles' (none where their keys are in one part), then a block per (row, head) of the single rows' (none where no row is split).
__global__ __launch_bounds__(256) void attn_both_merge_kernel(const float* __restrict__ tile_o, const float* __restrict__ tile_ml, const int* __restrict__ tiles,
                                                              int n_split, int blocks_per_tile, int tile_blocks, const float* __restrict__ row_o,
                                                              const float* __restrict__ row_ml, const int4* __restrict__ firsts, bf16_t* __restrict__ out, int nh,
                                                              int hd, int hdp, const float* __restrict__ sink) {
    if ((int)blockIdx.x < tile_blocks) {
        attn_prefill_merge_block(blockIdx.x, tile_o, tile_ml, out, tiles, nh, hd, hdp, n_split, blocks_per_tile, sink);
        return;
    }
    const int at = blockIdx.x - tile_blocks, head = at % nh;
    const int4 row = firsts[at / nh];
    if (row.z <= 1) return;
    attn_merge_splits(row_o, row_ml, out + ((size_t)row.x * nh + head) * hd, (size_t)row.y * nh + head, hd, hdp, row.z, (size_t)nh, sink ? sink + head : nullptr);
}

template <int HDP, int QT>
static void launch_both(const PrefillLaunch& l, hipStream_t stream, const bf16_t* q, bf16_t* out, PagedCache c, const int* block_table, int max_blocks, int nh,
                        int window, const float* sink, BothTiles t, const BothItems& r) {
    const int lds = max(attn_prefill_ring<HDP, 2>() + l.lds_pages * (int)sizeof(int), (int)sizeof(DecodeLds<HDP>));
    static bool configured = false;
    auto kern = attn_both_kernel<HDP, QT>;
    if (!configured) {
        (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                  min(max(attn_prefill_ring<HDP, 2>() + PF_MAX_PAGES * (int)sizeof(int), (int)sizeof(DecodeLds<HDP>)), PF_LDS_BYTES));
        configured = true;
    }
    const unsigned turn = fl_units(), tile_turns = ceil_div(l.grid.x * l.grid.y * l.grid.z, turn), item_turns = ceil_div(r.n * r.per_item, turn);
    // (longest tiles first, unless parts of the keys even them out; the mirrored order of attn_prefill.hip is for a chip that the tiles have to themselves)
    t.mirror_from = l.grid.z == 1 ? -1 : (int)(l.grid.x * l.grid.y);
    kern<<<(tile_turns + item_turns) * turn, 256, lds, stream>>>(q, out, c, block_table, max_blocks, nh, window, sink, t, r, turn, tile_turns, item_turns);
}

// fl_attn_prefill(_capped) of the tiles and fl_attn_decode_items(_capped) of the items (splits of their own) at once; tile_* are the workspaces, parts and heads of the
// former, row_* and firsts those of the latter.  Heads beyond 128 run one behind the other: there a unit has one block of either.  So do tables that
// leave a unit one block, where the tiles fill the chip by themselves (6,000 pages, a prompt of 2,048 tokens beside one row of 1,500 keys 81 us joined, 79 apart, beside 16
// of 2,000 94 and 97; with fewer blocks or parts of the keys joined is the faster one there too: 512 tokens 31 and 35).
extern "C" int fl_attn_both(const void* q, void* out, const void* cache_base, const int* block_table, int max_blocks, int nh, int nkv, int hd, int page_size,
                            int n_pages, float scale, int window, float softcap, const float* sink, const int* tiles, int n_tiles, const int* positions, int qt_hint,
                            float* tile_part_o, float* tile_part_ml, int tile_splits, const int* items, int n_items, float* row_part_o, float* row_part_ml,
                            const int* firsts, int n_rows, hipStream_t stream) {
    FL_CHECK(softcap >= 0.f, "attn_both: negative cap");
    FL_CHECK(!firsts || (row_part_o && row_part_ml && (uintptr_t)firsts % 16 == 0), "attn_both: rows that are split need a workspace and aligned firsts");
    PrefillLaunch l;
    int log2_page;
    if (attn_prefill_prepare("attn_both", n_tiles, max_blocks, nh, nkv, hd, page_size, scale, window, qt_hint, tile_part_o, tile_part_ml, tile_splits, softcap, &l)) return -1;
    if (attn_decode_prepare("attn_both", items, n_items, nh, nkv, hd, page_size, window, 1, true, row_part_o, row_part_ml, sink, &log2_page)) return -1;
    const int q_tiles = ceil_div(nh / nkv, 16), per_item = nkv * q_tiles;
    const int row_rows = firsts ? n_rows : 0;
    const long long merges = (tile_splits > 1 ? (long long)n_tiles * l.merge_blocks_per_tile : 0) + (long long)row_rows * nh;
    const long long tile_blocks_all = (long long)l.grid.x * l.grid.y * l.grid.z;
    const bool in_range = tile_blocks_all + (long long)n_items * per_item < (1ll << 23) && merges < (1ll << 23);        // (a grid has 2^32 threads)
    const bool one_place = 2 * (2 * 256 * l.hdp + l.lds_pages * (long long)sizeof(int)) > PF_LDS_BYTES;        // (a table of more than 4,096 pages with heads of 128)
    if (l.hdp > 128 || n_tiles == 0 || n_items == 0 || !in_range || (one_place && tile_splits == 1 && tile_blocks_all > fl_units())) {
        const int rc = fl_attn_prefill_capped(q, out, cache_base, tiles, n_tiles, positions, block_table, max_blocks, nh, nkv, hd, page_size, n_pages, scale, window,
                                              softcap, sink, qt_hint, tile_part_o, tile_part_ml, tile_splits, stream);
        if (rc) return rc;
        return fl_attn_decode_items_capped(q, out, row_part_o, row_part_ml, cache_base, items, n_items, block_table, max_blocks, nh, nkv, hd, page_size, n_pages, scale,
                                           window, softcap, sink, firsts, n_rows, stream);
    }
    const PagedCache c{(void*)cache_base, nkv, page_size, hd, n_pages};
    const BothTiles t = {tiles, positions, l.scale_log2e, l.cap_raw, l.log2_page, 0, tile_part_o, tile_part_ml, l.grid};
    const BothItems r = {(const int4*)items, scale, softcap, q_tiles, per_item, n_items, row_part_o, row_part_ml};
#define FL_BOTH(HDP_, QT_) launch_both<HDP_, QT_>(l, stream, (const bf16_t*)q, (bf16_t*)out, c, block_table, max_blocks, nh, window, sink, t, r)
    switch (l.hdp * 8 + l.heads_per_wave) {
        case 32 * 8 + 1: FL_BOTH(32, 1); break;
        case 32 * 8 + 2: FL_BOTH(32, 2); break;
        case 32 * 8 + 4: FL_BOTH(32, 4); break;
        case 64 * 8 + 1: FL_BOTH(64, 1); break;
        case 64 * 8 + 2: FL_BOTH(64, 2); break;
        case 64 * 8 + 4: FL_BOTH(64, 4); break;
        case 96 * 8 + 1: FL_BOTH(96, 1); break;
        case 96 * 8 + 2: FL_BOTH(96, 2); break;
        case 128 * 8 + 1: FL_BOTH(128, 1); break;
        default: FL_BOTH(128, 2); break;
    }
#undef FL_BOTH
    FL_LAUNCH_CHECK();
    if (merges > 0) {
        const int tile_blocks = tile_splits > 1 ? n_tiles * l.merge_blocks_per_tile : 0;
        attn_both_merge_kernel<<<(unsigned)merges, 256, 0, stream>>>(tile_part_o, tile_part_ml, tiles, tile_splits, l.merge_blocks_per_tile, tile_blocks, row_part_o,
                                                                             row_part_ml, (const int4*)firsts, (bf16_t*)out, nh, hd, l.hdp, sink);
        FL_LAUNCH_CHECK();
    }
    return 0;
}
FL_RECORDABLE(fl_attn_both)
