// A block of the attention of single rows (attn_decode.hip: what it does and what bounds it), for the kernel of its own and the one that takes
// prompt portions beside it (attn_both.hip).
#pragma once
#include "common.h"
#include "attn_merge.h"

#define DEC_WAVES 4
#define DEC_CHUNK 32

// items[i] = (row of q and out, position, request, 0 or split + 256 * splits): everything a block needs
// to find its keys comes with one load.  `block`: as the launch of a kernel of its own has it, (kv head and 16 query heads, item, split).
template <int HDP>
struct DecodeLds {
    float m[DEC_WAVES][16], l[DEC_WAVES][16];
    f32x4 o[DEC_WAVES - 1][HDP / 16][64];            // wave 0 keeps its own in registers
};
template <int HDP>
__device__ __forceinline__ void attn_decode_block(
    DecodeLds<HDP>& lds, uint3 block, const bf16_t* __restrict__ q, bf16_t* __restrict__ out, float* part_o,
    float* part_ml, PagedCache cache, const int4* __restrict__ items,
    const int* __restrict__ block_table, int max_blocks, int nh, float scale, int window,
    int n_split, int q_tiles, int ps_shift, int item_base, float softcap, const float* __restrict__ sink) {
    constexpr int QS = HDP / 32;     // k-steps of the score product
    constexpr int DT = HDP / 16;     // 16-wide tiles of head dims in the output
    constexpr bool PIPELINED = HDP <= 128;       // two chunks of keys and values fit the registers
    auto& s_m = lds.m;
    auto& s_l = lds.l;
    auto& s_o = lds.o;

    // (the items are the slow index of the grid: the places of a list that no row uses come last)
    const int item = item_base + block.y;
    const int kvh = block.x / q_tiles, qt = block.x % q_tiles;
    const int4 it = items[item];
    if (it.x < 0) return;                              // a place in the list that no row uses
    // an item with splits of its own says which split it is; its partial result lies in the slot of the item
    const bool own_splits = it.w != 0;
    const int split = own_splits ? (it.w & 255) : (int)block.z;
    if (own_splits) n_split = it.w >> 8;
    const int token = it.x, p = it.y;
    const int hd = cache.head_dim, ps = cache.page_size;
    const int G = nh / cache.n_kv_heads;
    const int* table = block_table + (size_t)it.z * max_blocks;
    const int lo = window > 0 ? max(0, p - window + 1) : 0;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);      // the same for the whole wave: what depends on it is scalar
    const int li = lane & 15, g = lane >> 4;
    const bf16_t* kv = (const bf16_t*)cache.base;
    const bf16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};

    // this split's chunks of 32 keys
    const int c_lo = lo / DEC_CHUNK, c_hi = p / DEC_CHUNK;
    const int per = (c_hi - c_lo + n_split) / n_split;
    const int c0 = c_lo + split * per, c1 = min(c_hi + 1, c0 + per);

    // Q as B operand: lane (head li, group g) holds Q[head][32 s + 8 g .. +7]
    const int head = kvh * G + qt * 16 + li;
    const bool head_ok = qt * 16 + li < G;
    bf16x8 qreg[QS];
#pragma unroll
    for (int s = 0; s < QS; ++s) {
        const int d = 32 * s + 8 * g;
        qreg[s] = (head_ok && d + 8 <= hd) ? *(const bf16x8*)(q + ((size_t)token * nh + head) * hd + d) : zero8;
    }

    f32x4 o[DT];
#pragma unroll
    for (int t = 0; t < DT; ++t) o[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;

    // Row i of score tile a is key t0 + 8 (i / 4) + i % 4, of tile b the same + 4: a lane (head, g)
    // of the accumulators then owns the 8 consecutive keys t0 + 8 g .. + 7, one 16-byte run of a
    // row of the transposed values.  The two keys of a lane lie in one page (pages hold multiples of 8).
    const int k_off = 8 * (li >> 2) + (li & 3), v_off = 8 * g;
    struct Chunk { bf16x8 xa[QS], xb[QS], wv[DT]; };
    auto page_of = [&](int key) { return ps_shift >= 0 ? key >> ps_shift : key / ps; };
    auto row_of = [&](int key) { return ps_shift >= 0 ? key & (ps - 1) : key % ps; };
    // Loads carry no conditions (a branch around a load would make every wait a wait for all loads
    // in flight): keys outside [lo, p] are clamped into it, page ids outside the pool to a page of
    // the pool, chunks beyond the split to its last chunk; what such a load brings is masked in
    // compute().  Pages of chunk c for this lane: of its two keys and of its eight values.
    const int c_last = c1 - 1;
    auto page_ids = [&](int c, int& pk, int& pv) {
        c = min(c, c_last);
        const int ka = min(max(c * DEC_CHUNK + k_off, lo), p), vk = min(max(c * DEC_CHUNK + v_off, lo), p);
        pk = table[page_of(ka)];
        pv = table[page_of(vk)];
    };
    auto load_chunk = [&](Chunk& f, int c, int pk, int pv) {
        c = min(c, c_last);
        const int ka = c * DEC_CHUNK + k_off, vk = c * DEC_CHUNK + v_off;
        pk = (int)min((unsigned)pk, (unsigned)cache.n_pages - 1u);
        pv = (int)min((unsigned)pv, (unsigned)cache.n_pages - 1u);
        const bf16_t* rowa = kv + cache_k_offset(cache, pk, kvh, row_of(ka), 0);
        const bf16_t* rowb = rowa + 4 * hd;          // key ka + 4: the same page
#pragma unroll
        for (int s = 0; s < QS; ++s) {
            const int d = min(32 * s + 8 * g, hd - 8);       // head dims beyond hd: q is zero there
            f.xa[s] = __builtin_nontemporal_load((const bf16x8*)(rowa + d));
            f.xb[s] = __builtin_nontemporal_load((const bf16x8*)(rowb + d));
        }
        const bf16_t* vrow = kv + cache_v_offset(cache, pv, kvh, row_of(vk), 0);
#pragma unroll
        for (int t = 0; t < DT; ++t) {
            const int d = min(16 * t + li, hd - 1);          // rows beyond hd are never stored
            f.wv[t] = __builtin_nontemporal_load((const bf16x8*)(vrow + (size_t)d * ps));
        }
    };
    auto compute = [&](const Chunk& f, int c) {
        const int t0 = c * DEC_CHUNK;
        f32x4 sa = {0.f, 0.f, 0.f, 0.f}, sb = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < QS; ++s) {
            sa = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.xa[s], qreg[s], sa, 0, 0, 0);
            sb = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.xb[s], qreg[s], sb, 0, 0, 0);
        }
        // online softmax; this lane holds keys t0 + 8 g + r (tile a) and + 4 + r (tile b) for head li
        float mt = -INFINITY;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int ka = t0 + 8 * g + r, kb = ka + 4;
            float va = sa[r] * scale, vb = sb[r] * scale;
            if (softcap > 0.f) {                             // scores capped smoothly at +-softcap
                va = softcap * fast_tanh(va / softcap);
                vb = softcap * fast_tanh(vb / softcap);
            }
            sa[r] = (ka >= lo && ka <= p) ? va : -INFINITY;
            sb[r] = (kb >= lo && kb <= p) ? vb : -INFINITY;
            mt = fmaxf(mt, fmaxf(sa[r], sb[r]));
        }
        mt = fmaxf(mt, __shfl_xor(mt, 16, 64));
        mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
        const float m_new = fmaxf(m, mt);          // finite: every chunk holds a visible key
        const float corr = expf(m - m_new);
        bf16x8 pb8;
        float ls = 0.f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float ea = expf(sa[r] - m_new), eb = expf(sb[r] - m_new);
            ls += ea + eb;
            pb8[r] = (bf16_t)ea;
            pb8[4 + r] = (bf16_t)eb;
        }
        l = l * corr + ls;
        m = m_new;
        if (t0 < lo || t0 + DEC_CHUNK - 1 > p) {
            // a chunk at an end of the range: values of keys outside it (whatever the page holds
            // there) are zeroed, since 0 * NaN would not be 0
            u32x4 keep;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int k0 = t0 + 8 * g + 2 * e;
                keep[e] = ((k0 >= lo && k0 <= p) ? 0x0000FFFFu : 0u) | ((k0 + 1 >= lo && k0 + 1 <= p) ? 0xFFFF0000u : 0u);
            }
#pragma unroll
            for (int t = 0; t < DT; ++t) {
                o[t] *= corr;
                const u32x4 v = __builtin_bit_cast(u32x4, f.wv[t]) & keep;
                o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, v), pb8, o[t], 0, 0, 0);
            }
        } else {
#pragma unroll
            for (int t = 0; t < DT; ++t) {
                o[t] *= corr;
                o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.wv[t], pb8, o[t], 0, 0, 0);
            }
        }
    };

    // The wave's chunks are c0 + wave, + 4, ...  What bounds a short split is the chain page id ->
    // key and value loads -> arithmetic, so the chain is pipelined: page ids two chunks ahead, keys
    // and values one chunk ahead, in two register sets that swap roles.  The loop body has no
    // branch, so the compiler's count of the loads in flight is exact.
    int c = c0 + wave;
    if (c < c1) {
        if (PIPELINED) {
            Chunk fa, fb;
            int pk0, pv0, pk1, pv1;
            page_ids(c, pk0, pv0);
            page_ids(c + DEC_WAVES, pk1, pv1);
            load_chunk(fa, c, pk0, pv0);
            for (; c + 2 * DEC_WAVES < c1; c += 2 * DEC_WAVES) {
                page_ids(c + 2 * DEC_WAVES, pk0, pv0);
                load_chunk(fb, c + DEC_WAVES, pk1, pv1);
                compute(fa, c);
                page_ids(c + 3 * DEC_WAVES, pk1, pv1);
                load_chunk(fa, c + 2 * DEC_WAVES, pk0, pv0);
                compute(fb, c + DEC_WAVES);
            }
            if (c + DEC_WAVES < c1) {               // two chunks left
                load_chunk(fb, c + DEC_WAVES, pk1, pv1);
                compute(fa, c);
                compute(fb, c + DEC_WAVES);
            } else {
                compute(fa, c);
            }
        } else {
            Chunk f;
            for (; c < c1; c += DEC_WAVES) {
                int pk, pv;
                page_ids(c, pk, pv);
                load_chunk(f, c, pk, pv);
                compute(f, c);
            }
        }
    }
    // sum over the four key groups of a head
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);

    // ---- merge the waves
    if (g == 0) { s_m[wave][li] = m; s_l[wave][li] = l; }
    if (wave > 0) {
#pragma unroll
        for (int t = 0; t < DT; ++t) s_o[wave - 1][t][lane] = o[t];
    }
    __syncthreads();
    if (wave == 0) {
        float mm = -INFINITY;
#pragma unroll
        for (int w = 0; w < DEC_WAVES; ++w) mm = fmaxf(mm, s_m[w][li]);
        float f[DEC_WAVES], ll = 0.f;
#pragma unroll
        for (int w = 0; w < DEC_WAVES; ++w) {
            f[w] = s_m[w][li] == -INFINITY ? 0.f : expf(s_m[w][li] - mm);
            ll += s_l[w][li] * f[w];
        }
        // lane (head li, group g) holds dims 16 t + 4 g + r
        if (head_ok && n_split == 1) {
            const float inv = sink ? softmax_factor_with_sink(mm, ll, sink[head]) : ll > 0.f ? 1.0f / ll : 0.f;
            bf16_t* orow = out + ((size_t)token * nh + head) * hd;
#pragma unroll
            for (int t = 0; t < DT; ++t) {
                f32x4 acc = o[t] * f[0];
#pragma unroll
                for (int w = 1; w < DEC_WAVES; ++w) acc += s_o[w - 1][t][lane] * f[w];
                const int d = 16 * t + 4 * g;
                if (d + 4 <= hd) {
                    bf16x4 ov = {(bf16_t)(acc[0] * inv), (bf16_t)(acc[1] * inv), (bf16_t)(acc[2] * inv), (bf16_t)(acc[3] * inv)};
                    *(bf16x4*)(orow + d) = ov;
                }
            }
        } else if (head_ok) {
            const size_t slot = own_splits ? (size_t)item * nh + head : ((size_t)item * nh + head) * n_split + split;
            if (g == 0) { part_ml[slot * 2] = mm; part_ml[slot * 2 + 1] = ll; }
            float* prow = part_o + slot * HDP;
#pragma unroll
            for (int t = 0; t < DT; ++t) {
                f32x4 acc = o[t] * f[0];
#pragma unroll
                for (int w = 1; w < DEC_WAVES; ++w) acc += s_o[w - 1][t][lane] * f[w];
                *(f32x4*)(prow + 16 * t + 4 * g) = acc;
            }
        }
    }
}

// Checks the arguments of a launch (0: they are in order); *ps_shift: log2 of the page size, -1 where it is no power of two.
int attn_decode_prepare(const char* who, const int* items, int n_items, int nh, int nkv, int hd, int page_size, int window, int n_split, bool own_splits,
                        const float* part_o, const float* part_ml, const float* sink, int* ps_shift);
