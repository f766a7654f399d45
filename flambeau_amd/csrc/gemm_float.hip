// The 32-bit matrix product on the matrix cores: out[m][n] = sum_k x[m][k] w[n][k], floats in, floats out,
// the same bits as gemm_plain_kernel (plain.hip) gives.
//
// What an output element is: its k in rising chunks of 16, every chunk a chain of 16 fused multiply-adds
// from zero, the chunks' sums added in rising order with a compensated (Kahan) addition.  A
// v_mfma_f32_16x16x4_f32 is such a chain of four (rising k, one rounding each: 1 M random results and
// products below the smallest normal number are bit for bit those of fmaf), so four of them on one
// accumulator are a chunk.  Nothing else about the sum is free: K cannot be split, but the chunks' chains
// are independent of one another; only the compensated addition, four operations per chunk, is serial.
//
// Operand of the instruction for the chunk's k = 4 s .. 4 s + 3 (s = 0 .. 3): lane l gives row l % 16 at
// k = 4 s + l / 16.  Rows lie in LDS as in memory, an odd multiple of 4 floats apart (68 or 36): 16 such rows
// begin at 16 different multiples of 4 of the 64 banks, so that the 16 rows x 4 neighbours of a read meet no bank twice.
//
// Two kernels: `few` streams w for a few rows of x (bound by HBM), `many` tiles both (bound by the matrix and the
// vector unit, which 32-bit matrix instructions share: 128 clocks of products and 64 of compensated additions per
// 16 x 16 x 16, so 105 of 157 TFLOP/s at most).  The bits do not depend on which one runs.
#include "common.h"
#include "gemm_float.h"

#define GF_CHUNK 16

// One compensated addition of a chunk's sum to (acc, lost).
__device__ __forceinline__ void gf_add(float part, float& acc, float& lost) {
    const float y = part - lost;
    const float t = acc + y;
    lost = (t - acc) - y;
    acc = t;
}

// ------------------------------------------------------------------ few rows of x
// Block = 16 rows of w x 16 MT rows of x, four waves.  A step is 64 CH k: wave v forms CH chunks of it, the ones
// from v CH on, of rows of w and x that it fetches itself (AHEAD steps ahead, in registers; a row's piece by
// neighbouring lanes, every line asked for once) and turns into operands through LDS of its own; the chunks' sums
// go to LDS, one barrier, and every thread adds the sums of its own output elements in their order, while other
// waves are already in the next step.  Bound by the stream of w up to 16 rows, by the sums' way through LDS beyond.
// Measured with weights from HBM, one row of x (gemm_plain_kernel in brackets): 28672 x 4096 98.7 us = 4.8 TB/s (832),
// 4096 x 14336 53.4 us (2,650), 6144 x 4096 29.4 us (747), 4096 x 4096 21.2 us (739); 16 rows: 111, 72, 33.5, 24 us.
template <int MT, int CH, int XF, int AHEAD>
__global__ __launch_bounds__(256, 2) void gemm_float_few_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                                float* __restrict__ out, int M, int N, int K) {
    constexpr int STEP = 64 * CH, WK = 16 * CH;      // k per step, and of a wave
    constexpr int LD = WK + 4;                       // floats between rows in LDS
    constexpr int LANES = WK / 4, ROWS = 64 / LANES; // a fetch: ROWS rows by LANES lanes each
    constexpr int F = 16 / ROWS;                     // fetches per 16 rows
    __shared__ __attribute__((aligned(16))) float ws[4][16 * LD];
    __shared__ __attribute__((aligned(16))) float xs[4][MT][16 * LD];
    __shared__ __attribute__((aligned(16))) float sums[2][MT][4 * CH * 256];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int n0 = blockIdx.x * 16, i = lane & 15, g = lane >> 4;
    const int fr = lane / LANES, fk = 4 * (lane % LANES);
    const int steps = (K + STEP - 1) / STEP, chunks = (K + GF_CHUNK - 1) / GF_CHUNK;
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
    float acc[MT], lost[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = lost[t] = 0.f;
#pragma unroll
    for (int a = 0; a < AHEAD; ++a) fetch(a, pw[a], px[a]);
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < steps; s0 += AHEAD) {
#pragma unroll
        for (int a = 0; a < AHEAD; ++a) {
            const int step = s0 + a;                 // (one behind the last adds nothing: cnt is 0 or less)
            const bool in = step * STEP + WK * wave + fk < K;
#pragma unroll
            for (int u = 0; u < F; ++u) *(f32x4*)&ws[wave][(ROWS * u + fr) * LD + fk] = in ? pw[a][u] : zero;
#pragma unroll
            for (int u = 0; u < XF; ++u) *(f32x4*)&xs[wave][u / F][((ROWS * u + fr) & 15) * LD + fk] = in ? px[a][u] : zero;
            fetch(step + AHEAD, pw[a], px[a]);
            wave_fence();
            f32x4 part[MT][CH];
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int c = 0; c < CH; ++c) {
                    const float wv = ws[wave][i * LD + 16 * c + 4 * s + g];
#pragma unroll
                    for (int t = 0; t < MT; ++t) {
                        const float xv = xs[wave][t][i * LD + 16 * c + 4 * s + g];
                        const f32x4 from = s ? part[t][c] : (f32x4){0.f, 0.f, 0.f, 0.f};
                        part[t][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv, xv, from, 0, 0, 0);
                    }
                }
            wave_fence();
            float(*to)[4 * CH * 256] = sums[step & 1];
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int c = 0; c < CH; ++c) *(f32x4*)&to[t][(CH * wave + c) * 256 + 4 * lane] = part[t][c];
            __syncthreads();                         // (who writes these sums again has passed the next barrier, behind these reads)
            const int cnt = min(4 * CH, chunks - step * 4 * CH);
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                float v[4 * CH];
#pragma unroll
                for (int c = 0; c < 4 * CH; ++c) v[c] = to[t][c * 256 + threadIdx.x];
                if (cnt == 4 * CH) {
#pragma unroll
                    for (int c = 0; c < 4 * CH; ++c) gf_add(v[c], acc[t], lost[t]);
                } else {
#pragma unroll
                    for (int c = 0; c < 4 * CH; ++c)
                        if (c < cnt) gf_add(v[c], acc[t], lost[t]);
                }
            }
        }
    }
    // element 4 l + r of the sums: lane l's register r of the product, w row 4 (l / 16) + r, x row l % 16
    const int n = n0 + 4 * (threadIdx.x >> 6) + (threadIdx.x & 3);
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        const int m = 16 * t + ((threadIdx.x >> 2) & 15);
        if (m < M && n < N) out[(size_t)m * N + n] = acc[t];
    }
}

// ------------------------------------------------------------------ many rows of x
// Block = 64 rows of w x 16 TM rows of x, wave v the 16 rows of w from 16 v on against all of x's.  Stages of 32 k in
// two LDS slots, AHEAD stages asked for (into registers) before the products of this one.  2 TM chains are in flight
// per wave.  Counters at 28672 x 4096 x 333: matrix unit busy 67 % of the time, vector unit 41 %.  Measured at 333 rows
// (gemm_plain_kernel in brackets): 28672 x 4096 837 us = 93 TFLOP/s (1,948), 4096 x 14336 538 us (2,624), 6144 x 4096
// 222 us (736), 4096 x 4096 163 us (691); at 1,000 rows 81 to 100 TFLOP/s.
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
    f32x4 acc[TM], lost[TM];
#pragma unroll
    for (int t = 0; t < TM; ++t) acc[t] = lost[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
    const int stages = (K + GF_K - 1) / GF_K;
    const int chunks = (K + GF_CHUNK - 1) / GF_CHUNK;
    fetch(0, pw[0], px[0]);
    put(0, 0, pw[0], px[0]);
#pragma unroll
    for (int a = 0; a < AHEAD; ++a) fetch((a + 1) * GF_K, pw[a], px[a]);
    __syncthreads();
    for (int s0 = 0; s0 < stages; s0 += AHEAD) {
#pragma unroll
        for (int a = 0; a < AHEAD; ++a) {
            const int st = s0 + a;                   // (one behind the last adds nothing)
            const int slot = a & 1;
            f32x4 part[2][TM];
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    const int at = i * GF_LDM + 16 * c + 4 * s + g;
                    const float wv = ws[slot][16 * wave * GF_LDM + at];
#pragma unroll
                    for (int t = 0; t < TM; ++t) {
                        const f32x4 from = s ? part[c][t] : (f32x4){0.f, 0.f, 0.f, 0.f};
                        part[c][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv, xs[slot][16 * t * GF_LDM + at], from, 0, 0, 0);
                    }
                }
            put(slot ^ 1, (st + 1) * GF_K, pw[a], px[a]);
            fetch((st + 1 + AHEAD) * GF_K, pw[a], px[a]);
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                if (2 * st + c >= chunks) break;
#pragma unroll
                for (int t = 0; t < TM; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        float sum = acc[t][r], l = lost[t][r];
                        gf_add(part[c][t][r], sum, l);
                        acc[t][r] = sum;
                        lost[t][r] = l;
                    }
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
            *(f32x4*)(out + (size_t)m * N + n) = acc[t];
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (n + r < N) out[(size_t)m * N + n + r] = acc[t][r];
        }
    }
}

// Which of the two kernels takes a product (gemm_float_launch says why).
static bool gf_few(int M, int N) { return M <= 32 || (M <= 64 && N <= 8192); }

bool gemm_float_takes(const void* x, const void* w, const void* out, int M, int N, int K) {
    // 16-byte pieces of rows; a grid of fewer than 2^31 blocks, and 64 rows within a 32-bit offset
    const bool fits = K % 4 == 0 && ((uintptr_t)x | (uintptr_t)w | (uintptr_t)out) % 16 == 0 && K < (1 << 24) &&
                      (long)(N / 64 + 1) * (M / 32 + 1) < (1l << 30);
    if (!fits) return false;
    // A block's beginning and end take as long as some hundred k, so a K that is short beside the number of blocks is left to
    // gemm_plain_kernel, the same bits.  Microseconds here / there, one row: 32768 x 4 15.0 / 4.3, x 32 14.8 / 6.5, x 64 14.9 / 10.9, x 128
    // 15 / 20; 16384 x 32 1.27 times as long, x 64 0.73; 131072 x 128 1.5 times; 64 rows: 8192 x 32 1.5 times, x 64 0.93, 4096 x 20
    // 0.89; 1,000 rows: 4096 x 16 1.13 times, 1024 x 16 0.95, 4096 x 20 0.96.
    if (K <= 16) return !gf_few(M, N) && (long)M * N <= (1l << 20);
    if (!gf_few(M, N)) return true;
    return M <= 32 ? 256l * K >= N : N <= 4096 || K >= 64;
}

void gemm_float_launch(const float* x, const float* w, float* out, int M, int N, int K, hipStream_t stream) {
    const int blocks = ceil_div(N, 16);
    // rows of x per block: 32, 48 or 64, whichever leaves the fewest empty (the larger of two that leave as many: w is
    // read by fewer blocks)
    int best = 4;
    for (int tm = 3; tm >= 2; --tm)
        if (ceil_div(M, 16 * tm) * tm < ceil_div(M, 16 * best) * best) best = tm;
    const int m_tiles = ceil_div(M, 16 * best), tiles = m_tiles * ceil_div(N, 64), per_die = ceil_div(tiles, 8);
    // 33 to 64 rows of x: a narrow matrix gives `many` too few blocks (N / 64) and goes to `few` (N / 16).  Microseconds at
    // 33 / 64 rows, few against many: 4096 x 4096 52 / 64 against 131 / 146, 4096 x 14336 172 / 218 against 461 / 507, 6144 x
    // 4096 97 / 122 against 133 / 148, 28672 x 4096 339 / 424 against 170 / 224.  17 to 32 rows: 28672 x 4096 few 172, many 170.
#define GF_FEW(MT, CH, XF) gemm_float_few_kernel<MT, CH, XF, 2><<<blocks, 256, 0, stream>>>(x, w, out, M, N, K)
#define GF_MANY(TM) gemm_float_many_kernel<TM><<<8 * per_die, 256, 0, stream>>>(x, w, out, M, N, K, m_tiles, tiles, per_die)
    if (M <= 4) GF_FEW(1, 4, 1);
    else if (M <= 16) GF_FEW(1, 4, 4);
    else if (M <= 32) GF_FEW(2, 2, 4);
    else if (gf_few(M, N) && M <= 48) GF_FEW(3, 2, 6);
    else if (gf_few(M, N)) GF_FEW(4, 2, 8);
    else if (best == 4) GF_MANY(4);
    else if (best == 3) GF_MANY(3);
    else GF_MANY(2);
#undef GF_FEW
#undef GF_MANY
}
