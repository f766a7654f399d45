// Attention over the paged cache for the 32-bit path: floats in, floats out, every product on the matrix cores
// (v_mfma_f32_16x16x4_f32), precise expf.  The same result, to the bit, whatever tokens run beside a token.
//
// What a (token, query head) is: its keys in blocks of 64 counted from position 0.  A block's scores (chains of 8
// head dims, added in a tree), their maximum m, the weights e^(score - m), their sum l and the weighted sum a of the
// values (chains of 16 keys, added in pairs); then (M, L, A) over the blocks in rising order,
//     M' = max(M, m),  L <- L e^(M - M') + l e^(m - M'),  A <- A e^(M - M') + a e^(m - M').
// Keys outside the row's range weigh nothing (their scores are not looked at), and a block without a key of the row
// leaves (M, L, A) as it is.  So neither the rows of a tile, nor how a prompt is cut, nor who forms a block shows.
// A block's weights add up to at least 1 where it has a score above minus infinity, and to NaN where a score is NaN (or
// plus infinity), which a maximum would pass by: the sum tells whether a block counts, never the maximum.  A row
// whose scores are all minus infinity is NaN, as the formula has it.  A value that is no finite number reaches the rows
// that see its key and no other, although a tile's rows share the values: where a block's sums are not all finite
// they are formed again, such values as zero and then row by row (add_unbounded).
// A row whose keys fit into AF_FEW positions (from a multiple of four on) is a wave's own work instead
// (attn_float_few): whether it is one, the row's position and the window alone decide.
//
// Block of threads = a tile of up to 16 rows (token, query head) that read one key/value head: T tokens by its query
// heads (T = 1 in steps of few tokens, where the heads alone have to fill the chip).  Eight waves form eight blocks of
// keys at a time and leave (m, l, a) in LDS, where all threads add them in order, four head dims of a row each.  The
// tokens of a tile may belong to several requests: their blocks of keys are one list that the waves share.
// No operand passes through LDS.  Scores are computed transposed, S^T = K Q^T, so that a lane holds scores of one row:
// instruction (c, e) takes head dims 16 c + 4 g + e of lane group g = lane / 16, four neighbouring dims of a row being one
// 16-byte load for four instructions.  S^T leaves lane (g, row) with keys 16 t + 4 g + r, which is just what it has to
// give as an operand of O^T = V^T P^T if instruction (t, r) takes those keys, and the values of four neighbouring keys
// are 16 bytes of the transposed page.
//
// Bound by the chain look-up of the page, loads, 256 matrix instructions of 32 clocks, adding up.  Microseconds with 32
// heads of 128 over 8 (attn_plain_kernel, a block per token and head that goes through its keys one by one): a prompt of
// 333 tokens 48.6 (527), of 100 14.8 (67); one token behind 340 19.7 (88), behind 4,000 137 (1,526); 64 tokens behind 340
// 36 (213), behind 17 6.8 (15.7), behind 1 5.3 (4.8).  With a key head for each of the 32 heads, 64 tokens behind 100
// 44 (72).  Error against 64 bits beside that kernel's: 0.96 to 1.0 up to 64 keys, 0.92, 0.72, 0.56, 0.43 at 100, 340,
// 1,000, 4,000.
#include "attn_float.h"
#include "lanes.h"

#define AF_WAVES 8
#define AF_ROWS 16
#define AF_KEYS 64
// Rows of 33 to 48 keys: 6.1 us against 11.7 on the matrix cores (eight tokens, as above), and 0.97 against 1.07 times the
// plain kernel's error; with 64 a prompt of 100 tokens took 16.9 us instead of 14.8 (a tile's rows share matrix
// instructions, here a wave has one or two rows after the other).
#define AF_FEW 48

// The scores of 16 keys: chains of two instructions from zero, their results added in a tree.  Longer chains lose
// more: the error against 64 bits, beside the plain kernel's, was 0.98, 0.92, 0.72 and 0.56 times at 64, 100, 340 and
// 1,000 keys, with chains of 16 products 1.05, 1.03, 0.89, 0.63, with chains of 32 (and the values of a block in one
// chain) 1.41, 1.30, 1.11, 0.76.  A result is added two chains after its own, so that no addition waits for the
// matrix unit.
template <int NC>
__device__ __forceinline__ f32x4 scores(const f32x4 (&kf)[NC], const f32x4 (&qv)[NC]) {
    constexpr int N = 2 * NC, LATE = 2;
    f32x4 sum[N];
#pragma unroll
    for (int n = 0; n < N + LATE; ++n) {
        if (n < N) {
            sum[n] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int e = 2 * (n & 1); e < 2 * (n & 1) + 2; ++e)
                sum[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[n / 2][e], qv[n / 2][e], sum[n], 0, 0, 0);
        }
        const int d = n - LATE;                       // (a binary counter: d's trailing ones are complete pairs)
#pragma unroll
        for (int w = 1; w < N; w *= 2) {
            if (d < 0 || !(d & w)) break;
            sum[d & ~(2 * w - 1)] += sum[(d & ~(2 * w - 1)) + w];
        }
        __builtin_amdgcn_sched_barrier(0);            // (in this order: all chains first would hold all their results)
    }
    return sum[0];
}

// o[e], the sum of lane (g, row j) for dim 4 g + e, plus weight times value for the values of `v` that are no finite
// numbers: v of lane (g, d) belongs to dim d and to the key whose weights for the rows (g, 0) .. (g, 15) are in `weight`
// of those lanes; `sees`: whether the row's range holds that key.
__device__ __forceinline__ void add_unbounded(f32x4& o, float v, float weight, bool sees) {
    const int lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4;
    for (unsigned long long rest = __ballot(!isfinite(v)); rest; rest &= rest - 1) {
        const int from = __ffsll(rest) - 1, d = from & 15;
        const float value = __shfl(v, from, 64), p = __shfl(weight, (from & 48) + j, 64);
        if (__shfl((int)sees, (from & 48) + j, 64) && g == d >> 2) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (e == (d & 3)) o[e] += p * value;
        }
    }
}

// The result of one row with at most AF_FEW keys from position lo4 on (lo rounded down to a multiple of four), by one
// wave on the vector unit: 256 matrix instructions for a handful of keys, most of them for nothing, take 7 us.  Lane
// (g, j) forms a share of four dims in 64 of the scores of keys 4 i + g, i = 0 .. 15, keeps that of i = j, and holds two
// (one) of the head dims when the values are added, in four chains of every fourth key.
template <int HD>
__device__ __forceinline__ void attn_float_few(const float* __restrict__ q, float* __restrict__ out, const PagedCache& cache,
                                               const int* __restrict__ table, int kvh, int lo, int p, float scale, float softcap,
                                               const float* __restrict__ sink) {
    constexpr int NV = HD / 64;                                       // pieces of four dims of a key, and dims of a value, per lane
    const int lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4;
    const int lo4 = lo & ~3, groups = (p - lo4 + 4) >> 2;             // groups of four keys, which share a page
    const size_t block = (size_t)cache.page_size * HD;
    const int at = lo4 + 4 * min(j, groups - 1);
    const int page = table[at / cache.page_size], row = at % cache.page_size;
    const bool there = page >= 0 && page < cache.n_pages;
    const int held = there ? page : 0;                                // (lane i knows group i's page and row)
    const bool seen = there && j < groups && lo4 + 4 * j + g >= lo && lo4 + 4 * j + g <= p;
    f32x4 qv[NV];
#pragma unroll
    for (int c = 0; c < NV; ++c) qv[c] = *(const f32x4*)(q + 64 * c + 4 * j);
    auto base_of = [&](int i, int is_v) {
        return (const float*)cache.base + (((size_t)__builtin_amdgcn_readlane(held, i) * 2 + is_v) * cache.n_kv_heads + kvh) * block;
    };
    f32x4 vf[4][NV];
    auto values = [&](int i0) {                                       // of four groups (behind the last one it is that one again)
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const int i = min(i0 + a, groups - 1);
            const float* v = base_of(i, 1) + __builtin_amdgcn_readlane(row, i);
#pragma unroll
            for (int d = 0; d < NV; ++d) vf[a][d] = *(const f32x4*)(v + (size_t)(64 * d + lane) * cache.page_size);
        }
    };
    float s = 0.f;
    for (int i0 = 0; i0 < groups; i0 += 4) {
        f32x4 kf[4][NV];
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const int i = min(i0 + a, groups - 1);
            const float* k = base_of(i, 0) + (size_t)(__builtin_amdgcn_readlane(row, i) + g) * HD;
#pragma unroll
            for (int d = 0; d < NV; ++d) kf[a][d] = *(const f32x4*)(k + 64 * d + 4 * j);
        }
        if (i0 == 0) values(0);
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            float part[NV];
#pragma unroll
            for (int d = 0; d < NV; ++d) {
                part[d] = kf[a][d][0] * qv[d][0];
#pragma unroll
                for (int r = 1; r < 4; ++r) part[d] = fmaf(kf[a][d][r], qv[d][r], part[d]);
            }
            const float sum = row_sum16(NV == 2 ? part[0] + part[NV - 1] : part[0]);
            if (i0 + a == j) s = sum;
        }
    }
    s *= scale;
    if (softcap > 0.f) s = softcap * tanhf(s / softcap);              // scores capped smoothly at +-softcap
    const float m = wave_max(seen ? s : -INFINITY), base = m == -INFINITY ? 0.f : m;
    const float weight = seen ? expf(s - base) : 0.f;
    const float l = wave_sum(weight);
    const unsigned long long sees = __ballot(seen);
    f32x4 acc[NV];
#pragma unroll
    for (int c = 0; c < NV; ++c) acc[c] = (f32x4){0.f, 0.f, 0.f, 0.f};
    for (int i0 = 0; i0 < groups; i0 += 4) {
        if (i0) values(i0);
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int from = 16 * e + i0 + a;                     // (behind the last group: seen by nobody)
                const float w = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(weight), from));
                const bool counts = (sees >> from) & 1;
#pragma unroll
                for (int d = 0; d < NV; ++d) acc[d][e] = fmaf(w, counts ? vf[a][d][e] : 0.f, acc[d][e]);
            }
    }
    const float none = sees ? NAN : 0.f;                              // every score minus infinity, or no key at all
    const float inv = sink ? softmax_factor_with_sink(m, l, *sink) : l == 0.f ? none : 1.0f / l;
#pragma unroll
    for (int c = 0; c < NV; ++c) out[64 * c + lane] = ((acc[c][0] + acc[c][1]) + (acc[c][2] + acc[c][3])) * inv;
}

template <int HD>
__global__ __launch_bounds__(64 * AF_WAVES, 2) void attn_float_kernel(const float* __restrict__ q, float* __restrict__ out,
                                                                      PagedCache cache, const int* __restrict__ positions,
                                                                      const int* __restrict__ tok_seq,
                                                                      const int* __restrict__ block_table, int max_blocks, int n,
                                                                      int nh, int tokens, int heads, int head_tiles, float scale,
                                                                      int window, float softcap, const float* __restrict__ sink) {
    constexpr int NC = HD / 16, LD = HD + 4, FOURS = HD / 4, AHEAD = 2;
    constexpr int MINE = AF_ROWS * FOURS / (64 * AF_WAVES);           // groups of four dims a thread adds up
    static_assert(AF_ROWS * FOURS % (64 * AF_WAVES) == 0 || AF_ROWS * FOURS < 64 * AF_WAVES, "rows must divide among the threads");
    constexpr int SUMS = MINE > 0 ? MINE : 1;
    __shared__ __attribute__((aligned(16))) float part_a[AF_WAVES][AF_ROWS][LD];
    __shared__ float part_m[AF_WAVES][AF_ROWS], part_l[AF_WAVES][AF_ROWS];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, j = lane & 15, g = lane >> 4;
    const int kvh = blockIdx.y / head_tiles, group = nh / cache.n_kv_heads;
    const int h0 = (blockIdx.y % head_tiles) * heads;                 // first query head of the tile within the group
    const int tok0 = blockIdx.x * tokens, n_tok = min(tokens, n - tok0);
    const int n_heads = min(heads, group - h0);
    // row j: token j / heads, query head j % heads of the tile
    const int my_tok = j / heads, my_head = j % heads;
    const int at_tok = tok0 + min(my_tok, n_tok - 1), at_head = kvh * group + h0 + min(my_head, n_heads - 1);
    const int my_p = positions[at_tok], my_lo = window > 0 ? max(0, my_p - window + 1) : 0;
    const bool my_row = my_tok < n_tok && my_head < n_heads && my_p - (my_lo & ~3) >= AF_FEW;
    // Rows of few keys, a wave each.  (Lane `row` knows whether that row is one.)
    const unsigned few = (unsigned)__ballot(g == 0 && my_tok < n_tok && my_head < n_heads && my_p - (my_lo & ~3) < AF_FEW);
    int dealt = 0;
    for (unsigned rest = few; rest; rest &= rest - 1, ++dealt) {
        if (dealt % AF_WAVES != wave) continue;
        const int row = __ffs(rest) - 1, tok = tok0 + row / heads, head = kvh * group + h0 + row % heads;
        const int p = __builtin_amdgcn_readlane(my_p, row), lo = __builtin_amdgcn_readlane(my_lo, row);
        const size_t at = ((size_t)tok * nh + head) * HD;
        attn_float_few<HD>(q + at, out + at, cache, block_table + (size_t)tok_seq[tok] * max_blocks, kvh, lo, p, scale, softcap,
                           sink ? sink + head : nullptr);
    }
    if (!__any(my_row)) return;                                       // (the same in every wave)
    f32x4 qv[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) qv[c] = *(const f32x4*)(q + ((size_t)at_tok * nh + at_head) * HD + 16 * c + 4 * g);
    // what this thread adds up: row a_row[u], head dims a_d[u] ..+ 3
    float M[SUMS], L[SUMS];
    f32x4 A[SUMS];
    bool low[SUMS];                                                   // a block of the row had keys, all at minus infinity
#pragma unroll
    for (int u = 0; u < SUMS; ++u) {
        M[u] = -INFINITY;
        L[u] = 0.f;
        low[u] = false;
        A[u] = (f32x4){0.f, 0.f, 0.f, 0.f};
    }
    const size_t block = (size_t)cache.page_size * HD;                // floats of a (page, K or V, head)
    // The tile's requests, one after the other, each from the first to the last block of keys that its tokens see: lane r
    // keeps the r-th of them, and every wave takes the next block of the whole list (not of one request: 16 requests of
    // one token are two rounds instead of 16).
    const int last_tok = min(lane & (AF_ROWS - 1), n_tok - 1);
    const int lane_seq = tok_seq[tok0 + last_tok], lane_p = positions[tok0 + last_tok];
    int blocks = 0, requests = 0, r_seq = 0, r_max = 0, r_min = 0, r_from = 0, r_to = 0, r_end = 0;
    for (int from = 0, to; from < n_tok; from = to) {
        const int seq = __builtin_amdgcn_readlane(lane_seq, from);
        int p_max = -1, p_min = 0x7fffffff;
        for (to = from; to < n_tok && __builtin_amdgcn_readlane(lane_seq, to) == seq; ++to) {
            const int p = __builtin_amdgcn_readlane(lane_p, to);
            if (p - ((window > 0 ? max(0, p - window + 1) : 0) & ~3) < AF_FEW) continue;
            p_max = max(p_max, p);
            p_min = min(p_min, p);
        }
        if (p_max < 0) continue;
        const int lo_min = window > 0 ? max(0, p_min - window + 1) : 0;
        blocks += p_max / AF_KEYS - lo_min / AF_KEYS + 1;
        if (lane == requests) {
            r_seq = seq;
            r_max = p_max;
            r_min = lo_min;
            r_from = from;
            r_to = to;
            r_end = blocks;
        }
        ++requests;
    }
    const int slot = (wave + AF_WAVES - dealt % AF_WAVES) % AF_WAVES;  // (first the waves that had a row of few keys less)
    for (int b0 = 0; b0 < blocks; b0 += AF_WAVES) {
        const int b = b0 + slot;
        if (b < blocks) {
            const int r = __ffsll(__ballot(lane < requests && r_end > b)) - 1;
            const int p_max = __builtin_amdgcn_readlane(r_max, r), lo_min = __builtin_amdgcn_readlane(r_min, r);
            const int* table = block_table + (size_t)__builtin_amdgcn_readlane(r_seq, r) * max_blocks;
            const bool in_turn = my_row && my_tok >= __builtin_amdgcn_readlane(r_from, r) && my_tok < __builtin_amdgcn_readlane(r_to, r);
            const int key0 = (p_max / AF_KEYS - (__builtin_amdgcn_readlane(r_end, r) - 1 - b)) * AF_KEYS;
            // S^T: lane (g, row j) gets the scores of keys key0 + 16 t + 4 g + r
            f32x4 S[4];
            bool there[4];                                        // keys 16 t + 4 g .. + 3 have a page (all four or none)
            const float* vals[4];                                 // their values of head dim 0
            const float* keys[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int key = min(key0 + 16 * t + j, p_max);    // (beyond the last key: that one again, not looked at)
                const int page = table[key / cache.page_size];
                const int held = page >= 0 && page < cache.n_pages ? page : 0;
                keys[t] = (const float*)cache.base + ((size_t)held * 2 * cache.n_kv_heads + kvh) * block +
                          (size_t)(key % cache.page_size) * HD + 4 * g;
                const int key4 = key0 + 16 * t + 4 * g;           // (pages hold a multiple of four tokens)
                const int page4 = key4 <= p_max ? table[key4 / cache.page_size] : -1;
                there[t] = page4 >= 0 && page4 < cache.n_pages;
                vals[t] = (const float*)cache.base + ((size_t)(there[t] ? page4 : 0) * 2 * cache.n_kv_heads + cache.n_kv_heads + kvh) * block +
                          (there[t] ? key4 % cache.page_size : 0) + (size_t)j * cache.page_size;
            }
            // 16 keys at a time, the next 16 on their way (a wait for all of them at once would take the registers of 64)
            f32x4 kf[2][NC];
#pragma unroll
            for (int c = 0; c < NC; ++c) kf[0][c] = *(const f32x4*)(keys[0] + 16 * c);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                if (t < 3) {
#pragma unroll
                    for (int c = 0; c < NC; ++c) kf[(t + 1) & 1][c] = *(const f32x4*)(keys[t + 1] + 16 * c);
                }
                __builtin_amdgcn_sched_barrier(0);
                S[t] = scores<NC>(kf[t & 1], qv);
                __builtin_amdgcn_sched_barrier(0);
            }
            f32x4 vf[AHEAD][4];                                   // values of 16 head dims, AHEAD times 16 on their way
            auto fetch = [&](int d0, f32x4* to) {
#pragma unroll
                for (int t = 0; t < 4; ++t) to[t] = *(const f32x4*)(vals[t] + (size_t)d0 * cache.page_size);
            };
#pragma unroll
            for (int a = 0; a < AHEAD; ++a) fetch(16 * a, vf[a]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < 4; ++t) S[t] *= scale;
            if (softcap > 0.f) {                                  // scores capped smoothly at +-softcap
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r) S[t][r] = softcap * tanhf(S[t][r] / softcap);
            }
            auto sees = [&](int t, int r) {                       // whether the row looks at key 16 t + 4 g + r
                const int key = key0 + 16 * t + 4 * g + r;
                return in_turn && there[t] && key >= my_lo && key <= my_p;
            };
            float m = -INFINITY;
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (sees(t, r)) m = fmaxf(m, S[t][r]);
            m = fmaxf(m, __shfl_xor(m, 16, 64));
            m = fmaxf(m, __shfl_xor(m, 32, 64));
            const float base = m == -INFINITY ? 0.f : m;
            bool any = false;
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const bool seen = sees(t, r);
                    S[t][r] = seen ? expf(S[t][r] - base) : 0.f;
                    any = any || seen;
                }
            const f32x4 four = (S[0] + S[1]) + (S[2] + S[3]);
            float l = (four[0] + four[1]) + (four[2] + four[3]);
            l += __shfl_xor(l, 16, 64);
            l += __shfl_xor(l, 32, 64);
            // lanes j, j + 16, j + 32, j + 48 hold row j's keys; -1: there are some, and every score is minus infinity
            if (l == 0.f && ((__ballot(any) >> j) & 0x0001000100010001ull)) l = -1.f;
            // O^T: four chains of 16 keys, instruction (t, r) the keys 16 t + 4 g + r; whatever lies behind a weight of zero
            // counts only if it is no finite number, and then it shows in the sums
            bool finite = true;
#pragma unroll
            for (int d0 = 0; d0 < HD; d0 += 16) {
                f32x4 part[4];
                f32x4* now = vf[d0 / 16 % AHEAD];
#pragma unroll
                for (int t = 0; t < 4; ++t) part[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int t = 0; t < 4; ++t) part[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(now[t][r], S[t][r], part[t], 0, 0, 0);
                if (d0 + 16 * AHEAD < HD) fetch(d0 + 16 * AHEAD, now);
                const f32x4 o = (part[0] + part[1]) + (part[2] + part[3]);
#pragma unroll
                for (int r = 0; r < 4; ++r) finite = finite && isfinite(o[r]);
                *(f32x4*)&part_a[slot][j][d0 + 4 * g] = o;
                __builtin_amdgcn_sched_barrier(0);
            }
            if (__any(!finite)) {
#pragma unroll 1
                for (int d0 = 0; d0 < HD; d0 += 16) {
                    f32x4 val[4], part[4];
                    fetch(d0, val);
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        part[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            part[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(isfinite(val[t][r]) ? val[t][r] : 0.f, S[t][r], part[t], 0, 0, 0);
                    }
                    f32x4 o = (part[0] + part[1]) + (part[2] + part[3]);
#pragma unroll
                    for (int t = 0; t < 4; ++t)
#pragma unroll
                        for (int r = 0; r < 4; ++r) add_unbounded(o, val[t][r], S[t][r], sees(t, r));
                    *(f32x4*)&part_a[slot][j][d0 + 4 * g] = o;
                }
            }
            if (g == 0) {
                part_m[slot][j] = m;
                part_l[slot][j] = l;
            }
        }
        __syncthreads();
        const int formed = min(AF_WAVES, blocks - b0);
#pragma unroll
        for (int u = 0; u < SUMS; ++u) {
            const int e = threadIdx.x + 64 * AF_WAVES * u, row = e / FOURS, d = 4 * (e % FOURS);
            if (row < AF_ROWS) {
                for (int w = 0; w < formed; ++w) {
                    const float m = part_m[w][row], l = part_l[w][row];
                    if (l == 0.f) continue;                           // no key of this row in the block
                    if (l < 0.f) {
                        low[u] = true;
                        continue;
                    }
                    const float top = fmaxf(M[u], m), old = expf(M[u] - top), now = expf(m - top);
                    const f32x4 a = *(const f32x4*)&part_a[w][row][d];
                    L[u] = L[u] * old + l * now;
#pragma unroll
                    for (int r = 0; r < 4; ++r) A[u][r] = A[u][r] * old + a[r] * now;
                    M[u] = top;
                }
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int u = 0; u < SUMS; ++u) {
        const int e = threadIdx.x + 64 * AF_WAVES * u, row = e / FOURS, d = 4 * (e % FOURS);
        const int tok = row / heads, hh = row % heads;
        if (row >= AF_ROWS || tok >= n_tok || hh >= n_heads || ((few >> row) & 1)) continue;
        const int head = kvh * group + h0 + hh;
        const float none = low[u] ? NAN : 0.f;                        // (NaN, or no key at all)
        const float inv = sink ? softmax_factor_with_sink(M[u], L[u], sink[head]) : L[u] == 0.f ? none : 1.0f / L[u];
        f32x4 o;
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = A[u][r] * inv;
        *(f32x4*)(out + ((size_t)(tok0 + tok) * nh + head) * HD + d) = o;
    }
}

bool attn_float_takes(const void* q, const void* out, const void* cache_base, int hd, int page_size) {
    return (hd == 64 || hd == 128) && page_size % 4 == 0 && (((uintptr_t)q | (uintptr_t)out | (uintptr_t)cache_base) % 16) == 0;
}

void attn_float_launch(const float* q, float* out, const PagedCache& cache, const int* positions, const int* tok_seq,
                       const int* block_table, int max_blocks, int n, int nh, float scale, int window, float softcap,
                       const float* sink, hipStream_t stream) {
    const int group = nh / cache.n_kv_heads, heads = min(group, AF_ROWS), head_tiles = ceil_div(group, heads);
    // A unit holds one thread block at a time: as few tokens per tile as still give every unit at most one, up to what
    // fills the rows.
    const int per_head = fl_units() / (cache.n_kv_heads * head_tiles);
    const int tokens = per_head > 0 ? min(AF_ROWS / heads, ceil_div(n, per_head)) : AF_ROWS / heads;
    const dim3 grid(ceil_div(n, tokens), cache.n_kv_heads * head_tiles);
    if (cache.head_dim == 64)
        attn_float_kernel<64><<<grid, 64 * AF_WAVES, 0, stream>>>(q, out, cache, positions, tok_seq, block_table, max_blocks, n, nh,
                                                                  tokens, heads, head_tiles, scale, window, softcap, sink);
    else
        attn_float_kernel<128><<<grid, 64 * AF_WAVES, 0, stream>>>(q, out, cache, positions, tok_seq, block_table, max_blocks, n, nh,
                                                                   tokens, heads, head_tiles, scale, window, softcap, sink);
}
