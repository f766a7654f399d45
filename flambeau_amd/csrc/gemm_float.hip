// The 32-bit matrix product on the matrix cores: out[m][n] = sum_k x[m][k] w[n][k], floats in, floats out,
// the same bits as gemm_plain_kernel (plain.hip) gives.
//
// What an output element is: its k in rising groups of 32, a group three chains of 12, 8 and 12 fused multiply-adds from zero,
// (12 + 8) + 12 added in 32 bits, the groups in rising order in 64; k behind K are zeros.  A v_mfma_f32_16x16x4_f32 is such a chain
// of four (rising k, one rounding each: 1 M random results and products below the smallest normal number are bit for bit those of
// fmaf).  Nothing else about the sum is free: K cannot be split, but groups are independent of one another up to their addition.
// How far the sums are from the exact ones (2-norm of the difference over 2-norm of the exact sums, x normal, w normal times 0.02), and
// in brackets chains of 16 with a compensated addition in 32 bits: K 14336 7.55e-8 (8.14e-8), 4096 7.55e-8 (8.14e-8), 100 7.47e-8 (7.98e-8);
// of absolute values, whose sums grow, K 4096 2.153e-8 (2.154e-8), 1000 2.323e-8 (2.326e-8), 100 3.74e-8 (3.75e-8).  Groups of 64 whose
// halves were joined in 32 bits were further off than the latter: 2.18e-8, 2.43e-8, 4.44e-8.
// Additions and 32-bit matrix instructions share the vector unit, at 2.7 clocks an addition in 32 bits, 5.4 one in 64 or a
// conversion to it, and 32.3 a matrix instruction (measured, any number of waves): 258 clocks of products and 65 of
// additions per 16 x 16 x 32, where chains of 16 took 86 of additions in either way (four compensated in 32 bits, or two in 64).
//
// Operand of the instruction for the k = 4 s .. 4 s + 3 of a group (s = 0 .. 7): lane l gives row l % 16 at
// k = 4 s + l / 16.  Rows lie in LDS as in memory, an odd multiple of 4 floats apart (68 or 36): 16 such rows
// begin at 16 different multiples of 4 of the 64 banks, so that the 16 rows x 4 neighbours of a read meet no bank twice.
//
// Two kernels: `few` streams w for a few rows of x (bound by HBM), `many` tiles both (bound by the vector unit, which 32-bit matrix
// instructions share: 125 of 157 TFLOP/s at most).  The bits do not depend on which one runs.
#include "common.h"
#include "gemm_float.h"

// Instruction s of a group's eight: the next four k of its chain (of 12, 8 and 12).
__device__ __forceinline__ void gf_chain(float w, float x, int s, f32x4* part) {
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4& p = part[(s >= 3) + (s >= 5)];
    p = __builtin_amdgcn_mfma_f32_16x16x4f32(w, x, s == 0 || s == 3 || s == 5 ? zero : p, 0, 0, 0);
}
__device__ __forceinline__ f32x4 gf_group(const f32x4* part) { return (part[0] + part[1]) + part[2]; }

// ------------------------------------------------------------------ few rows of x
// Block = 16 rows of w x 16 MT rows of x, four waves.  A step is 128 GROUPS k: wave v forms GROUPS groups of it, the ones
// from v GROUPS on, of rows of w and x that it fetches itself (AHEAD steps ahead, in registers; a row's piece by
// neighbouring lanes, every line asked for once) and turns into operands through LDS of its own; their sums
// go to LDS, one barrier, and every thread adds those of its own output elements in their order, while other
// waves are already in the next step.  Bound by the stream of w and, at 4096 rows of w, by a block's chain of steps (one block to a
// unit).  Measured with weights from HBM, one row of x (chains of 16, whose sums all went through LDS, in brackets):
// 28672 x 4096 91 us = 5.2 TB/s (99), 4096 x 14336 46 (53), 6144 x 4096 25.6 (29.4), 4096 x 4096 20.6 (21.2); 16 rows: 100 (111),
// 59 (72), 30 (33.5), 22 (24).  Three and four steps ahead are up to 10 % slower but at 4096 x 14336 (up to 6 % faster).
template <int MT, int GROUPS, int XF, int AHEAD>
__global__ __launch_bounds__(256, 2) void gemm_float_few_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                                float* __restrict__ out, int M, int N, int K) {
    constexpr int STEP = 128 * GROUPS, WK = 32 * GROUPS;   // k per step, and of a wave
    constexpr int LD = WK + 4;                       // floats between rows in LDS
    constexpr int LANES = WK / 4, ROWS = 64 / LANES; // a fetch: ROWS rows by LANES lanes each
    constexpr int F = 16 / ROWS;                     // fetches per 16 rows
    __shared__ __attribute__((aligned(16))) float ws[4][16 * LD];
    __shared__ __attribute__((aligned(16))) float xs[4][MT][16 * LD];
    __shared__ __attribute__((aligned(16))) float sums[2][MT][4 * GROUPS * 256];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int n0 = blockIdx.x * 16, i = lane & 15, g = lane >> 4;
    const int fr = lane / LANES, fk = 4 * (lane % LANES);
    const int steps = (K + STEP - 1) / STEP;
    const float* xrow[XF];
    const float* wrow[F];
#pragma unroll
    for (int u = 0; u < F; ++u) wrow[u] = w + (size_t)min(n0 + ROWS * u + fr, N - 1) * K;
#pragma unroll
    for (int u = 0; u < XF; ++u) xrow[u] = x + (size_t)min(ROWS * u + fr, M - 1) * K;
    f32x4 pw[AHEAD][F], px[AHEAD][XF];
    // (no condition on a load, so that the waits for them stay exact: k behind K is clamped, and zeroed on its way to LDS)
    auto fetch = [&](int step, f32x4* fw, f32x4* fx) {
        const int k = min(step * STEP + WK * wave + fk, K - 4);
#pragma unroll
        for (int u = 0; u < F; ++u) fw[u] = __builtin_nontemporal_load((const f32x4*)(wrow[u] + k));
#pragma unroll
        for (int u = 0; u < XF; ++u) fx[u] = *(const f32x4*)(xrow[u] + k);
    };
    double acc[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = 0.0;
#pragma unroll
    for (int a = 0; a < AHEAD; ++a) fetch(a, pw[a], px[a]);
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < steps; s0 += AHEAD) {
#pragma unroll
        for (int a = 0; a < AHEAD; ++a) {
            const int step = s0 + a;                 // (what lies behind K, a step behind the last too, is zeros: they add nothing)
            const bool in = step * STEP + WK * wave + fk < K;
#pragma unroll
            for (int u = 0; u < F; ++u) *(f32x4*)&ws[wave][(ROWS * u + fr) * LD + fk] = in ? pw[a][u] : zero;
#pragma unroll
            for (int u = 0; u < XF; ++u) *(f32x4*)&xs[wave][u / F][((ROWS * u + fr) & 15) * LD + fk] = in ? px[a][u] : zero;
            fetch(step + AHEAD, pw[a], px[a]);
            wave_fence();
            f32x4 part[GROUPS][MT][3];
#pragma unroll
            for (int s = 0; s < 8; ++s)
#pragma unroll
                for (int h = 0; h < GROUPS; ++h) {
                    const float wv = ws[wave][i * LD + 32 * h + 4 * s + g];
#pragma unroll
                    for (int t = 0; t < MT; ++t) gf_chain(wv, xs[wave][t][i * LD + 32 * h + 4 * s + g], s, part[h][t]);
                }
            wave_fence();
            float(*to)[4 * GROUPS * 256] = sums[step & 1];
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int h = 0; h < GROUPS; ++h) *(f32x4*)&to[t][(GROUPS * wave + h) * 256 + 4 * lane] = gf_group(part[h][t]);
            __syncthreads();                         // (who writes these sums again has passed the next barrier, behind these reads)
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                float v[4 * GROUPS];
#pragma unroll
                for (int c = 0; c < 4 * GROUPS; ++c) v[c] = to[t][c * 256 + threadIdx.x];
#pragma unroll
                for (int c = 0; c < 4 * GROUPS; ++c) acc[t] += v[c];
            }
        }
    }
    // element 4 l + r of the sums: lane l's register r of the product, w row 4 (l / 16) + r, x row l % 16
    const int n = n0 + 4 * (threadIdx.x >> 6) + (threadIdx.x & 3);
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        const int m = 16 * t + ((threadIdx.x >> 2) & 15);
        if (m < M && n < N) out[(size_t)m * N + n] = (float)acc[t];
    }
}

// ------------------------------------------------------------------ many rows of x
// Block = 64 rows of w x 16 TM rows of x, wave v the 16 rows of w from 16 v on against all of x's.  Stages of 32 k in
// two LDS slots, two stages asked for (into registers) before the products of this one.  3 TM chains are in flight
// per wave.  Measured at 333 rows (chains of 16 in brackets, and the groups of 64): 28672 x 4096 766 us = 102 TFLOP/s (828, 750),
// 4096 x 14336 443 us (520, 435), 6144 x 4096 184 (207, 181), 4096 x 4096 136 (153, 131).  No faster: four stages ahead, the next stage's first operands read and this
// one's sums added behind the barrier, 32 rows of w to a wave, waves side by side along x.
#define GF_K 32
#define GF_LDM 36

template <int TM>
__global__ __launch_bounds__(256, 2) void gemm_float_many_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                                 float* __restrict__ out, int M, int N, int K, int m_tiles, int tiles,
                                                                 int per_die) {
    constexpr int AHEAD = 2;
    constexpr int XR = 16 * TM, XF = (XR * 8 + 255) / 256;           // float4 of x per thread and stage
    __shared__ __attribute__((aligned(16))) float ws[2][64 * GF_LDM];
    __shared__ __attribute__((aligned(16))) float xs[2][XR * GF_LDM];
    // blocks go to the eight dies in turn: a die gets a run of neighbouring tiles, those of one stretch of w side by side
    const int tile = (blockIdx.x & 7) * per_die + (blockIdx.x >> 3);
    if (tile >= tiles) return;
    const int n0 = (tile / m_tiles) * 64, m0 = (tile % m_tiles) * XR;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
    const int row = threadIdx.x >> 3, kq = 4 * (threadIdx.x & 7);
    // rows by a 32-bit offset from the block's first (at most 63 rows of K < 2^24 floats)
    const char* wb = (const char*)(w + (size_t)n0 * K);
    const char* xb = (const char*)(x + (size_t)m0 * K);
    unsigned wo[2], xo[XF];
#pragma unroll
    for (int u = 0; u < 2; ++u) wo[u] = 4u * ((unsigned)min(row + 32 * u, N - 1 - n0) * (unsigned)K + (unsigned)kq);
#pragma unroll
    for (int u = 0; u < XF; ++u) xo[u] = 4u * ((unsigned)min(min(row + 32 * u, XR - 1), M - 1 - m0) * (unsigned)K + (unsigned)kq);
    const int last = (K - 1) / GF_K * GF_K;          // first k of the last stage
    f32x4 pw[AHEAD][2], px[AHEAD][XF];
    auto fetch = [&](int k0, f32x4* fw, f32x4* fx) {
        // (no condition on a load: behind the last stage it is that one again)
        const unsigned k = 4u * (unsigned)min(k0, last);
        const bool beyond = k0 >= last && last + kq >= K;          // a piece behind K reads the row's first one instead ...
        const unsigned back = beyond ? 4u * (unsigned)(last + kq) : 0u;
#pragma unroll
        for (int u = 0; u < 2; ++u) fw[u] = *(const f32x4*)(wb + (wo[u] + k - back));
#pragma unroll
        for (int u = 0; u < XF; ++u) fx[u] = *(const f32x4*)(xb + (xo[u] + k - back));
    };
    auto put = [&](int slot, int k0, f32x4* fw, f32x4* fx) {
        if (k0 + GF_K > K) {                         // ... and is zeroed on its way to LDS
            const bool in = k0 + kq < K;
            const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int u = 0; u < 2; ++u) fw[u] = in ? fw[u] : zero;
#pragma unroll
            for (int u = 0; u < XF; ++u) fx[u] = in ? fx[u] : zero;
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) *(f32x4*)&ws[slot][(row + 32 * u) * GF_LDM + kq] = fw[u];
#pragma unroll
        for (int u = 0; u < XF; ++u)
            if (XR % 32 == 0 || row + 32 * u < XR) *(f32x4*)&xs[slot][(row + 32 * u) * GF_LDM + kq] = fx[u];
    };
    double acc[TM][4];
#pragma unroll
    for (int t = 0; t < TM; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[t][r] = 0.0;
    const int stages = (K + GF_K - 1) / GF_K;
    fetch(0, pw[0], px[0]);
    put(0, 0, pw[0], px[0]);
#pragma unroll
    for (int a = 0; a < AHEAD; ++a) fetch((a + 1) * GF_K, pw[a], px[a]);
    __syncthreads();
    for (int s0 = 0; s0 < stages; s0 += AHEAD) {
#pragma unroll
        for (int a = 0; a < AHEAD; ++a) {
            const int st = s0 + a;                   // (one behind the last is zeros and adds nothing)
            const int slot = a;
            f32x4 part[TM][3];
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                const int at = i * GF_LDM + 4 * s + g;
                const float wv = ws[slot][16 * wave * GF_LDM + at];
#pragma unroll
                for (int t = 0; t < TM; ++t) gf_chain(wv, xs[slot][16 * t * GF_LDM + at], s, part[t]);
            }
            put(slot ^ 1, (st + 1) * GF_K, pw[a], px[a]);
            fetch((st + 1 + AHEAD) * GF_K, pw[a], px[a]);
#pragma unroll
            for (int t = 0; t < TM; ++t) {
                const f32x4 sum = gf_group(part[t]);
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[t][r] += sum[r];
            }
            __syncthreads();
        }
    }
    const int n = n0 + 16 * wave + 4 * g;
#pragma unroll
    for (int t = 0; t < TM; ++t) {
        const int m = m0 + 16 * t + i;
        if (m >= M) continue;
        if (n + 3 < N && N % 4 == 0) {
            *(f32x4*)(out + (size_t)m * N + n) = (f32x4){(float)acc[t][0], (float)acc[t][1], (float)acc[t][2], (float)acc[t][3]};
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (n + r < N) out[(size_t)m * N + n + r] = (float)acc[t][r];
        }
    }
}

// Which of the two kernels takes a product: to 16 rows `few`, to 48 where `many` would have too few blocks.  Microseconds, few against
// many: 17 rows 28672 x 4096 125 / 109, 32 rows 28672 x 4096 128 / 102, 4096 x 14336 92 / 153, 6144 x 4096 43 / 46, 4096 x 4096 30 / 46; 48 rows 190 / 138,
// 127 / 153, 59 / 61, 40 / 46.
static bool gf_few(int M, int N) { return M <= 16 || (M <= 48 && N <= 8192); }

// Tiles of 16 rows of x to a block of `many`: what a stage takes by the blocks that a unit gets, r.  Fitted to 43 products of 17 to
// 1,000 rows with 4096 to 32768 rows of w; of 108 with 2048 to 32768 none takes more than 2 % longer than with the best number (100 and 128 rows of
// 4096 x 4096, 63 us with one tile and 62 with two).  Four tiles were nowhere more than 2 % faster.  `full` blocks share a
// unit; to two rounds of those the unit with the most blocks decides.
static int gf_tiles(int M, int N) {
    static const struct { float stage, tile; int full; } cost[3] = {{0.193f, 0.153f, 6}, {0.241f, 0.259f, 4}, {0.281f, 0.381f, 3}};
    int best = 1;
    float least = 0.f;
    for (int tm = 1; tm <= 3; ++tm) {
        const auto& c = cost[tm - 1];
        const long blocks = (long)ceil_div(M, 16 * tm) * ceil_div(N, 64), units = fl_units();
        const float r = (float)blocks / units, most = r <= 2 * c.full ? (float)((blocks + units - 1) / units) : r;
        const float t = c.stage * (r > c.full ? r / c.full : 1.f) + c.tile * most;
        if (tm == 1 || t < least) {
            best = tm;
            least = t;
        }
    }
    return best;
}

bool gemm_float_takes(const void* x, const void* w, const void* out, int M, int N, int K) {
    // 16-byte pieces of rows; a grid of fewer than 2^31 blocks, and 64 rows within a 32-bit offset
    const bool fits = K % 4 == 0 && ((uintptr_t)x | (uintptr_t)w | (uintptr_t)out) % 16 == 0 && K < (1 << 24) &&
                      (long)(N / 64 + 1) * (M / 32 + 1) < (1l << 30);
    if (!fits) return false;
    // A block's beginning and end take as long as some ten k, so a K that is short beside the number of blocks is left to
    // gemm_plain_kernel, the same bits.  Microseconds here / there, for few rows: one row 32768 x 16 12.0 / 3.7, x 64 12.0 / 9.1, x 128 12.4 / 19.8,
    // 8192 x 32 4.8 / 4.9, 16384 x 32 7.3 / 5.0, x 64 7.4 / 7.8; 40 rows 6144 x 32 6.3 / 5.7, x 48 6.4 / 8.4, 4096 x 20 4.6 / 5.7.  For many: K up to 16 0.7 to 0.95
    // of the time there to 2^20 results (64 rows 6144 x 16 3.9 / 4.7, 17 of 32768 4.5 / 4.5), 1.03 to 1.25 of it beyond (65 of 16384 5.8 / 5.1, 1,000 of 4096 12.0 /
    // 10.6); from 20 on 0.5 to 1.0.
    const bool few = gf_few(M, N);
    if (K <= 16) return !few && (long)M * N <= (1l << 20);
    if (!few) return true;
    return M <= 32 ? 256l * K >= N : N <= 4096 || K > 32;
}

void gemm_float_launch(const float* x, const float* w, float* out, int M, int N, int K, hipStream_t stream) {
    const int blocks = ceil_div(N, 16);
    const int tm = gf_tiles(M, N);
    const int m_tiles = ceil_div(M, 16 * tm), tiles = m_tiles * ceil_div(N, 64), per_die = ceil_div(tiles, 8);
#define GF_FEW(MT, GROUPS, XF) gemm_float_few_kernel<MT, GROUPS, XF, 2><<<blocks, 256, 0, stream>>>(x, w, out, M, N, K)
#define GF_MANY(TM) gemm_float_many_kernel<TM><<<8 * per_die, 256, 0, stream>>>(x, w, out, M, N, K, m_tiles, tiles, per_die)
    if (M <= 4) GF_FEW(1, 2, 1);
    else if (M <= 16) GF_FEW(1, 2, 4);
    else if (gf_few(M, N) && M <= 32) GF_FEW(2, 1, 4);
    else if (gf_few(M, N)) GF_FEW(3, 1, 6);
    else if (tm == 3) GF_MANY(3);
    else if (tm == 2) GF_MANY(2);
    else GF_MANY(1);
#undef GF_FEW
#undef GF_MANY
}
