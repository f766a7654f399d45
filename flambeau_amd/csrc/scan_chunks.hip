// Linear recurrences over long runs of tokens, a chunk of 64 at a time on the 32-bit matrix cores.
//
// linear_scan.hip walks S <- g S + k u^T, o = S^T q token by token; its time is the tokens' chain, 0.15 us each, whatever the
// chip has left.  Over a chunk of tokens the same sums are
//     o_i = p_i S^T q_i + sum_{j <= i} d_ij (q_i . k_j) u_j,      S <- p_last S + sum_j d_last,j k_j u_j^T
// with d_ij the product of the decays behind j up to i and p_i that of the chunk's decays up to i.  Two kernels:
//   scan_pairs: everything that does not wait for the state, for every chunk and head at once: d_ij (q_i . k_j) and the products
//     of decays, one record per chunk and head in the workspace;
//   scan_chunks: a block per request, head and 16 columns of S walks the chunks: per chunk and wave 16 tokens' outputs and
//     D / 4 rows of S, the next chunk's operands on their way in registers meanwhile.
// The delta rule writes u_i = beta_i (v_i - what the state before it holds at k_i), so that a chunk's u depend on each other:
//     (I + L) U = diag(beta) V - diag(beta p) K S,      L_ij = beta_i d_ij (k_i . k_j) for j < i;
// scan_pairs_delta forms T = (I + L)^-1 (unit lower triangular), T diag(beta) and T diag(beta p) K for every chunk at once, and the
// walk makes U from v and S, exchanges it between the waves through LDS, and goes on with it in the place of v.
// Measured, 2,048 tokens of one request alone on the device, the walk and the chunks: a decay per head, 16 heads of 128 x 128, 304 and 103
// us; with write strengths, 32 heads of 128 x 64, 310 and 106; a decay per key dim, 32 heads of 128 x 128, 311 and 150; the delta rule, 32
// heads of 128 x 128, 355 and 189; traced in a model's prompt the pairs and the walk over chunks take 16 + 99, 24 + 98, 57 + 113 and 73 +
// 150.  A chunk of the second kernel is 2.6 to 4.7 us where its matrix instructions are 1.2 to 2.0.  Error
// against 64 bits (2-norm) 7.6e-7 -> 1.4e-7, 3.7e-7 -> 1.0e-7, 1.4e-7 -> 1.2e-7, 3.7e-7 -> 1.7e-7.
// Products of decays are formed by multiplying, never through logarithms or quotients: a decay of zero is one, and their rounding
// is the walk's.  All values and sums are 32-bit; a chunk's sums are added to the state once, where the walk rounds the state at
// every token, so results are nearer to 64 bits than the walk's.
//
// A value that is no finite number reaches the tokens behind it and no token before it: entries above the diagonal are not
// multiplied (tiles of 16 tokens above it are left out; in the tile on it a wave that finds such a value adds its tokens one by one).
#include "common.h"
#include "api.h"
#include "scan_chunks.h"

__device__ __forceinline__ int scan_chunks_of(int len, int min_len) { return len >= min_len ? (len + SC_CHUNK - 1) / SC_CHUNK : 0; }

// Records are numbered request by request.  The first record of request s, summed by one wave (all of its lanes call this).
__device__ __forceinline__ int scan_first_record(const int* lens, int s, int min_len) {
    const int lane = threadIdx.x & 63;
    int n = 0;
    for (int i = lane; i < s; i += 64) n += scan_chunks_of(lens[i], min_len);
#pragma unroll
    for (int m = 1; m < 64; m *= 2) n += __shfl_xor(n, m, 64);
    return n;
}
// Which request and which of its chunks record `slot` is; a request of -1: no such record.
__device__ __forceinline__ int2 scan_find(const int* lens, int n_seqs, int min_len, int slot) {
    const int lane = threadIdx.x & 63;
    int base = 0;
    for (int s0 = 0; s0 < n_seqs; s0 += 64) {
        const int n = s0 + lane < n_seqs ? scan_chunks_of(lens[s0 + lane], min_len) : 0;
        int incl = n;
#pragma unroll
        for (int m = 1; m < 64; m *= 2) {
            const int below = __shfl_up(incl, m, 64);
            if (lane >= m) incl += below;
        }
        const int total = __builtin_amdgcn_readlane(incl, 63);       // (what blocks address by is uniform: scalars)
        if (slot < base + total) {
            const int l = __ffsll((unsigned long long)__ballot(base + incl > slot)) - 1;
            return {s0 + l, slot - (base + __builtin_amdgcn_readlane(incl - n, l))};
        }
        base += total;
    }
    return {-1, 0};
}

__device__ __forceinline__ f32x4 mfma_f32(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// Loads carry a range instead of a condition: rows behind the request's last are zeros.
template <int NT>
__device__ __forceinline__ auto scan_load(__amdgpu_buffer_rsrc_t rows, unsigned voff, unsigned soff) {
    typedef __attribute__((ext_vector_type(NT))) float fNT;
    if constexpr (NT == 1) return (fNT)__uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rows, voff, soff, 0));
    else if constexpr (NT == 2) return __builtin_bit_cast(fNT, __builtin_amdgcn_raw_buffer_load_b64(rows, voff, soff, 0));
    else return __builtin_bit_cast(fNT, __builtin_amdgcn_raw_buffer_load_b128(rows, voff, soff, 0));
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t scan_rows(const float* base, int count, int ld, int width) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, ((count - 1) * ld + width) * 4, 0x00020000);
}

// (eight short chains instead of a long one: their rounding is what the results' error is made of)
__device__ __forceinline__ f32x4 sum_of_8(const f32x4 (&s)[8]) { return ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7])); }

// Block = (record, head), four waves; a wave forms the pairs of 16 tokens with all before them.  What bounds it are the matrix instructions, which the blocks on a unit share: 10 tiles of D / 4.
template <int D>
__global__ __launch_bounds__(256) void scan_pairs_kernel(ScanChunks a) {
    __shared__ float decay[SC_CHUNK], write[SC_CHUNK], between[SC_CHUNK][SC_CHUNK + 1];
    const int2 at = scan_find(a.seq_q_len, a.n_seqs, a.min_len, blockIdx.x);
    const int s = at.x, c = at.y;
    if (s < 0) return;
    const int head = blockIdx.y, qk_head = head / (a.H / a.G);
    const int t0 = a.seq_q_start[s] + c * SC_CHUNK, cnt = min(SC_CHUNK, a.seq_q_len[s] - c * SC_CHUNK);
    const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    float* rec = a.records + ((size_t)blockIdx.x * a.H + head) * SC_RECORD;
    if (tid < SC_CHUNK) {
        const size_t row = (size_t)(t0 + min(tid, cnt - 1)) * a.ldg + head;
        const float own = a.tok_decay ? a.tok_decay[row] : a.head_decay[head];
        decay[tid] = tid < cnt ? own : 1.f;
        write[tid] = a.write ? a.write[row] : 1.f;
    }
    __syncthreads();
    if (wave == 0) {                               // lane j: the decays behind token j, up to every later one
        double p = 1.0;
        for (int i = 0; i < SC_CHUNK; ++i) {
            if (i > lane) p *= decay[i];
            between[i][lane] = (float)p;
        }
        rec[SC_SUF + lane] = (float)(p * write[lane]);
    } else if (wave == 1) {                        // lane i: the chunk's decays up to token i
        double p = 1.0;
        for (int m = 0; m < SC_CHUNK; ++m)
            if (m <= lane) p *= decay[m];
        rec[SC_PRE + lane] = (float)p;
        if (lane == SC_CHUNK - 1) rec[SC_REST] = p == p && p <= 1e30 ? (float)(p - (double)(float)p) : 0.f;
    }
    const int I = (wave + blockIdx.x) & 3;         // the wave's 16 tokens (its work grows with them: not the same SIMD's in every block)
    const auto qrows = scan_rows(a.q + (size_t)t0 * a.ldq + qk_head * D, cnt, a.ldq, D), krows = scan_rows(a.k + (size_t)t0 * a.ldk + qk_head * D, cnt, a.ldk, D);
    f32x4 q[D / 16], pair[4];
#pragma unroll
    for (int u = 0; u < D / 16; ++u) q[u] = scan_load<4>(qrows, 4 * ((16 * I + n) * a.ldq + 4 * g), 64 * u);
#pragma unroll
    for (int J = 0; J < 4; ++J) {
        if (J > I) break;
        f32x4 sum[8] = {}, k[D / 16];
#pragma unroll
        for (int u = 0; u < D / 16; ++u) k[u] = scan_load<4>(krows, 4 * ((16 * J + n) * a.ldk + 4 * g), 64 * u);
        __builtin_amdgcn_sched_barrier(0);         // (all of them on their way before the first product)
#pragma unroll
        for (int u = 0; u < D / 16; ++u)
#pragma unroll
            for (int r = 0; r < 4; ++r) sum[4 * (u & 1) + r] = mfma_f32(q[u][r], k[u][r], sum[4 * (u & 1) + r]);
        pair[J] = sum_of_8(sum);
    }
    __syncthreads();
#pragma unroll
    for (int J = 0; J < 4; ++J) {
        if (J > I) break;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = 16 * I + 4 * g + r, j = 16 * J + n;
            const float factor = between[i][j] * write[j];
            rec[i * SC_CHUNK + j] = j <= i && j < cnt ? pair[J][r] * factor : 0.f;
        }
    }
}

// The same for a decay per token, head and key dim, and the rows that scan_chunks reads instead of q and k: q_i times the chunk's
// decays up to i, k_j times those behind j.  d_ij is a vector over the key dims then, so the pairs are sums of three factors.  Of 16
// tokens with 16 before them (a tile off the diagonal) the products of decays split where the later tokens begin: matrix
// instructions over q_i times the decays from there to i, and k_j times those behind j up to there (times whole tiles' decays
// between).  In the tiles on the diagonal a lane takes one token j and a quarter of the dims and carries k_j times the decays behind
// it from token to token: 2 x 16 x D / 4 multiplications a lane, which with the matrix instructions is what bounds this kernel.
// Products of decays run in 64 bits and are rounded once.
template <int D>
__global__ __launch_bounds__(256) void scan_pairs_channel_kernel(ScanChunks a) {
    constexpr int ROW = D + 4;
    extern __shared__ __attribute__((aligned(16))) float lds[];
    float* qs = lds;                               // [64][ROW] q, then times the decays of its 16 tokens up to its own
    float* gs = lds + SC_CHUNK * ROW;              // [64][ROW] decays, then k times the decays of its 16 tokens behind its own
    float* ts = gs + SC_CHUNK * ROW;               // [4][D] the decays of 16 tokens
    double* whole = (double*)(ts + 4 * D);         // [4][D] the same, not rounded
    const int2 at = scan_find(a.seq_q_len, a.n_seqs, a.min_len, blockIdx.x);
    const int s = at.x, c = at.y;
    if (s < 0) return;
    const int head = blockIdx.y, qk_head = head / (a.H / a.G);
    const int t0 = a.seq_q_start[s] + c * SC_CHUNK, cnt = min(SC_CHUNK, a.seq_q_len[s] - c * SC_CHUNK);
    const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    float* rec = a.records + ((size_t)blockIdx.x * a.H + head) * SC_CHANNEL_RECORD(D);
    const auto qrows = scan_rows(a.q + (size_t)t0 * a.ldq + qk_head * D, cnt, a.ldq, D), krows = scan_rows(a.k + (size_t)t0 * a.ldk + qk_head * D, cnt, a.ldk, D),
               frows = scan_rows(a.chan_decay + (size_t)t0 * a.ldc + head * D, cnt, a.ldc, D);
#pragma unroll
    for (int u = 0; u < SC_CHUNK * D / 4 / 256; ++u) {
        const int e = tid + 256 * u, t = e / (D / 4), d = 4 * (e % (D / 4));
        const f32x4 q = scan_load<4>(qrows, 4 * (t * a.ldq + d), 0), f = scan_load<4>(frows, 4 * (t * a.ldc + d), 0);
        const float none = t < cnt ? 0.f : 1.f;    // (the decay of no token: zero as loaded, one as it counts)
        *(f32x4*)(qs + t * ROW + d) = q;
        *(f32x4*)(gs + t * ROW + d) = (f32x4){f[0] + none, f[1] + none, f[2] + none, f[3] + none};
    }
    {   // the tile on the diagonal of this wave's 16 tokens: lane (j = n, dims 16 u + 4 g .. + 3)
        const int j = 16 * wave + n;
        f32x4 run[D / 16];
#pragma unroll
        for (int u = 0; u < D / 16; ++u) run[u] = scan_load<4>(krows, 4 * (j * a.ldk + 4 * g), 64 * u);
        __syncthreads();
#pragma unroll 1
        for (int i0 = 0; i0 < 16; i0 += 4) {
            float part[4];                         // this lane's dims of the pairs (i0 .. i0 + 3, j)
#pragma unroll
            for (int r0 = 0; r0 < 4; ++r0) {
                const float* qrow = qs + (16 * wave + i0 + r0) * ROW + 4 * g;
                const float* grow = gs + (16 * wave + i0 + r0) * ROW + 4 * g;
                f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int u = 0; u < D / 16; ++u) {
                    const f32x4 f = *(const f32x4*)(grow + 16 * u), q = *(const f32x4*)(qrow + 16 * u);
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        run[u][r] *= i0 + r0 > n ? f[r] : 1.f;
                        sum[r] = fmaf(q[r], run[u][r], sum[r]);
                    }
                }
                part[r0] = (sum[0] + sum[1]) + (sum[2] + sum[3]);
                __builtin_amdgcn_sched_barrier(0); // (a token's reads at a time: the registers hold no more)
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) part[r] += __shfl_xor(part[r], 16, 64);
#pragma unroll
            for (int r = 0; r < 4; ++r) part[r] += __shfl_xor(part[r], 32, 64);
            if (4 * g == i0)
#pragma unroll
                for (int r = 0; r < 4; ++r) rec[(16 * wave + i0 + r) * SC_CHUNK + j] = n <= i0 + r ? part[r] : 0.f;
        }
    }
    __syncthreads();
    for (int e = tid; e < 4 * D; e += 256) {       // a dim of 16 tokens
        const int I = e / D, d = e % D;
        float k[16], f[16], q[16];                 // (all read before the first is written)
#pragma unroll
        for (int t = 0; t < 16; ++t) k[t] = scan_load<1>(krows, 4 * ((16 * I + t) * a.ldk + d), 0)[0];
#pragma unroll
        for (int t = 0; t < 16; ++t) { f[t] = gs[(16 * I + t) * ROW + d]; q[t] = qs[(16 * I + t) * ROW + d]; }
        double p = 1.0;
#pragma unroll
        for (int t = 0; t < 16; ++t) {
            p *= f[t];
            q[t] *= (float)p;
        }
        ts[I * D + d] = (float)p;
        whole[I * D + d] = p;
        p = 1.0;
#pragma unroll
        for (int t = 15; t >= 0; --t) {
            k[t] *= (float)p;
            p *= f[t];
        }
#pragma unroll
        for (int t = 0; t < 16; ++t) { qs[(16 * I + t) * ROW + d] = q[t]; gs[(16 * I + t) * ROW + d] = k[t]; }
    }
    __syncthreads();
    auto tile = [&](int I, int J) {                // I > J
        f32x4 sum[8] = {};
#pragma unroll
        for (int u = 0; u < D / 16; ++u) {
            f32x4 q = *(const f32x4*)(qs + (16 * I + n) * ROW + 16 * u + 4 * g);
            const f32x4 k = *(const f32x4*)(gs + (16 * J + n) * ROW + 16 * u + 4 * g);
            for (int m = J + 1; m < I; ++m) q *= *(const f32x4*)(ts + m * D + 16 * u + 4 * g);
#pragma unroll
            for (int r = 0; r < 4; ++r) sum[4 * (u & 1) + r] = mfma_f32(q[r], k[r], sum[4 * (u & 1) + r]);
        }
        const f32x4 pair = sum_of_8(sum);
#pragma unroll
        for (int r = 0; r < 4; ++r) rec[(16 * I + 4 * g + r) * SC_CHUNK + 16 * J + n] = pair[r];
    };
    if (wave == 0) { tile(1, 0); tile(2, 0); }
    else if (wave == 1) { tile(2, 1); tile(3, 1); }
    else if (wave == 2) tile(3, 2);
    else tile(3, 0);
    float* q_out = rec + SC_CHANNEL_Q;
    float* k_out = q_out + SC_CHUNK * D;
#pragma unroll 4
    for (int e = tid; e < SC_CHUNK * D / 4; e += 256) {
        const int t = e / (D / 4), d = 4 * (e % (D / 4)), I = t >> 4;
        f32x4 q = *(const f32x4*)(qs + t * ROW + d), k = *(const f32x4*)(gs + t * ROW + d);
        for (int m = I - 1; m >= 0; --m) q *= *(const f32x4*)(ts + m * D + d);
        for (int m = I + 1; m < 4; ++m) k *= *(const f32x4*)(ts + m * D + d);
        *(f32x4*)(q_out + t * D + d) = q;
        *(f32x4*)(k_out + t * D + d) = k;
    }
    if (tid < D) {                                 // the chunk's decay, and what its rounding to 32 bits left
        const double p = (whole[tid] * whole[D + tid]) * (whole[2 * D + tid] * whole[3 * D + tid]);
        k_out[SC_CHUNK * D + tid] = (float)p;
        k_out[SC_CHUNK * D + D + tid] = p == p && p <= 1e30 ? (float)(p - (double)(float)p) : 0.f;
    }
}

// The delta rule's pairs, T diag(beta) and T diag(beta p) K.  T by tiles of 16 tokens: the four on the diagonal by substitution, a
// column per lane; the others from those before them, T_IJ = -T_II sum_{J <= M < I} L_IM T_MJ, by their distance from the diagonal.  A
// chunk whose keys, decays or strengths are not all finite, or whose products are not, substitutes throughout, so that what is no number
// reaches no token before it.
template <int D>
__global__ __launch_bounds__(256) void scan_pairs_delta_kernel(ScanChunks a) {
    constexpr int ROW = D + 4, LT = SC_CHUNK + 4;
    extern __shared__ __attribute__((aligned(16))) float lds[];
    float* ks = lds;                               // [64][ROW] keys
    float* L = ks + SC_CHUNK * ROW;                // [64][LT]
    float* T = L + SC_CHUNK * LT;                  // [64][LT]: the decays between tokens first, then T
    float* X = T + SC_CHUNK * LT;                  // [4][16][20] a wave's tile on its way from one operand form to the other
    float* decay = X + 4 * 16 * 20;                // [64] each
    float* beta = decay + SC_CHUNK;
    float* pre = beta + SC_CHUNK;
    __shared__ int odd;
    const int2 at = scan_find(a.seq_q_len, a.n_seqs, a.min_len, blockIdx.x);
    const int s = at.x, c = at.y;
    if (s < 0) return;
    const int head = blockIdx.y, qk_head = head / (a.H / a.G);
    const int t0 = a.seq_q_start[s] + c * SC_CHUNK, cnt = min(SC_CHUNK, a.seq_q_len[s] - c * SC_CHUNK);
    const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    float* rec = a.records + ((size_t)blockIdx.x * a.H + head) * SC_DELTA_RECORD(D);
    const auto qrows = scan_rows(a.q + (size_t)t0 * a.ldq + qk_head * D, cnt, a.ldq, D), krows = scan_rows(a.k + (size_t)t0 * a.ldk + qk_head * D, cnt, a.ldk, D);
    const int I = (wave + blockIdx.x) & 3;         // the wave's 16 tokens
    f32x4 q[D / 16];
#pragma unroll
    for (int u = 0; u < D / 16; ++u) q[u] = scan_load<4>(qrows, 4 * ((16 * I + n) * a.ldq + 4 * g), 64 * u);
    if (tid == 0) odd = 0;
    float strange = 0.f;                           // NaN where something loaded is no finite number
#pragma unroll
    for (int u = 0; u < SC_CHUNK * D / 4 / 256; ++u) {
        const int e = tid + 256 * u, t = e / (D / 4), d = 4 * (e % (D / 4));
        const f32x4 k = scan_load<4>(krows, 4 * (t * a.ldk + d), 0);
        strange += ((k[0] - k[0]) + (k[1] - k[1])) + ((k[2] - k[2]) + (k[3] - k[3]));
        *(f32x4*)(ks + t * ROW + d) = k;
    }
    if (tid < SC_CHUNK) {
        const size_t row = (size_t)(t0 + min(tid, cnt - 1)) * a.ldg + head;
        const float own = a.tok_decay[row], strength = a.write[row];
        decay[tid] = tid < cnt ? own : 1.f;
        beta[tid] = tid < cnt ? strength : 0.f;
        strange += (own - own) + (strength - strength);
    }
    __syncthreads();
    if (strange != 0.f) odd = 1;
    if (wave == 0) {                               // lane j: the decays behind token j, up to every later one
        double p = 1.0;
        for (int i = 0; i < SC_CHUNK; ++i) {
            if (i > lane) p *= decay[i];
            T[i * LT + lane] = (float)p;
        }
        rec[SC_SUF + lane] = (float)p;
    } else if (wave == 1) {                        // lane i: the chunk's decays up to token i
        double p = 1.0;
        for (int m = 0; m < SC_CHUNK; ++m)
            if (m <= lane) p *= decay[m];
        pre[lane] = (float)p;
        rec[SC_PRE + lane] = (float)p;
        if (lane == SC_CHUNK - 1) rec[SC_REST] = p == p && p <= 1e30 ? (float)(p - (double)(float)p) : 0.f;
    }
    f32x4 pair[4], same[4];                        // q_i . k_j and k_i . k_j
#pragma unroll
    for (int J = 0; J < 4; ++J) {
        if (J > I) break;
        f32x4 sum[8] = {}, own[8] = {};
#pragma unroll
        for (int u = 0; u < D / 16; ++u) {
            const f32x4 k = *(const f32x4*)(ks + (16 * J + n) * ROW + 16 * u + 4 * g), ki = *(const f32x4*)(ks + (16 * I + n) * ROW + 16 * u + 4 * g);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                sum[4 * (u & 1) + r] = mfma_f32(q[u][r], k[r], sum[4 * (u & 1) + r]);
                own[4 * (u & 1) + r] = mfma_f32(ki[r], k[r], own[4 * (u & 1) + r]);
            }
        }
        pair[J] = sum_of_8(sum);
        same[J] = sum_of_8(own);
    }
    __syncthreads();
#pragma unroll
    for (int J = 0; J < 4; ++J)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = 16 * I + 4 * g + r, j = 16 * J + n;
            const float between = J <= I ? T[i * LT + j] : 0.f;
            if (J <= I) rec[i * SC_CHUNK + j] = j <= i && j < cnt ? pair[J][r] * between : 0.f;
            const float l = J <= I && j < i ? beta[i] * (same[J][r] * between) : 0.f;
            L[i * LT + j] = l;
            if (l - l != 0.f) odd = 1;             // (keys too large to multiply)
        }
    __syncthreads();                               // (the decays between tokens have been read: their room is T's)
    if (!odd) {
        {   // the tile on the diagonal: lane n has column n (all four lanes g the same)
            float t[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                float row[16];
#pragma unroll
                for (int j = 0; j < 16; j += 4) *(f32x4*)(row + j) = *(const f32x4*)(L + (16 * wave + i) * LT + 16 * wave + j);
                float sum = i == n ? 1.f : 0.f;
#pragma unroll
                for (int j = 0; j < i; ++j) sum = fmaf(-row[j], t[j], sum);
                t[i] = sum;
            }
#pragma unroll
            for (int i = 0; i < 16; ++i)
                if (g == i >> 2) T[(16 * wave + i) * LT + 16 * wave + n] = t[i];
        }
        __syncthreads();
        float* x = X + wave * 16 * 20;
#pragma unroll
        for (int away = 1; away < 4; ++away) {
            if (wave + away < 4) {
                const int J = wave, R = wave + away;
                f32x4 sum = {0.f, 0.f, 0.f, 0.f};
                for (int M = J; M < R; ++M) {
                    const f32x4 l = *(const f32x4*)(L + (16 * R + n) * LT + 16 * M + 4 * g);
#pragma unroll
                    for (int e = 0; e < 4; ++e) sum = mfma_f32(l[e], T[(16 * M + 4 * g + e) * LT + 16 * J + n], sum);
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) x[(4 * g + r) * 20 + n] = sum[r];
                if (((sum[0] - sum[0]) + (sum[1] - sum[1])) + ((sum[2] - sum[2]) + (sum[3] - sum[3])) != 0.f) odd = 1;      // (too large for 32 bits: its rows meet the others' zeros next)
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                f32x4 out = {0.f, 0.f, 0.f, 0.f};
                const f32x4 t = *(const f32x4*)(T + (16 * R + n) * LT + 16 * R + 4 * g);
#pragma unroll
                for (int e = 0; e < 4; ++e) out = mfma_f32(-t[e], x[(4 * g + e) * 20 + n], out);
#pragma unroll
                for (int r = 0; r < 4; ++r) T[(16 * R + 4 * g + r) * LT + 16 * J + n] = out[r];
            }
            __syncthreads();
        }
    }
    if (odd) {
        if (tid < SC_CHUNK) {                      // column tid, row by row; nothing above the diagonal is multiplied
            for (int i = 0; i < SC_CHUNK; ++i) {
                float t = i == tid ? 1.f : 0.f;
                if (i > tid)
                    for (int j = tid; j < i; ++j) t = fmaf(-L[i * LT + j], T[j * LT + tid], t);
                T[i * LT + tid] = t;
            }
        }
        __syncthreads();
        for (int d = tid; d < D; d += 256)
            for (int i = 0; i < SC_CHUNK; ++i) {
                float w = 0.f;
                for (int j = 0; j <= i; ++j) w = fmaf(T[i * LT + j] * (beta[j] * pre[j]), ks[j * ROW + d], w);
                rec[SC_DELTA_W + i * D + d] = w;
            }
    } else {
        // T diag(beta p) K for the wave's 16 tokens
        f32x4 t[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            t[b] = (f32x4){0.f, 0.f, 0.f, 0.f};
            if (b < I) t[b] = *(const f32x4*)(T + (16 * I + n) * LT + 16 * b + 4 * g);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int j = 16 * b + 4 * g + e;
                if (b == I) t[b][e] = 4 * g + e <= n ? T[(16 * I + n) * LT + j] : 0.f;
                t[b][e] *= beta[j] * pre[j];
            }
        }
#pragma unroll 2
        for (int dt = 0; dt < D / 16; ++dt) {
            f32x4 sum[4] = {};
#pragma unroll
            for (int b = 0; b < 4; ++b)
                if (b <= I) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) sum[e] = mfma_f32(t[b][e], ks[(16 * b + 4 * g + e) * ROW + 16 * dt + n], sum[e]);
                }
            const f32x4 w = (sum[0] + sum[1]) + (sum[2] + sum[3]);
#pragma unroll
            for (int r = 0; r < 4; ++r) rec[SC_DELTA_W + (16 * I + 4 * g + r) * D + 16 * dt + n] = w[r];
        }
    }
    for (int e = tid; e < SC_CHUNK * SC_CHUNK; e += 256) {
        const int i = e >> 6, j = e & 63;
        rec[SC_DELTA_T + e] = j <= i ? T[i * LT + j] * beta[j] : 0.f;
    }
}

// Block = (head, columns j0 .. j0 + 15, request), four waves (neighbouring blocks are neighbouring heads: the blocks of a head, which
// read the same q and k, share a die's L2 where the number of heads is a multiple of eight).  Wave w has the outputs of the chunk's
// tokens 16 w .. 16 w + 15 and the rows d = D / 4 w + NT n + i of S (n = lane % 16, i < NT) as S^T, whose operand form all waves
// read from LDS.  Token 16 b + 4 g + e (g = lane / 16) is the k of a matrix instruction (b, e): one load of v serves the outputs (as
// B) and the state (as A), and q, the pairs and S come in 16-byte pieces.  Every operand is asked for again, for the next chunk,
// right behind its last use in this one, into the same registers: the trip hides behind the rest of the chunk (a second set of
// registers did not fit: the compiler moved them through the accumulators, each move a wait).
template <int D, bool CHAN, bool DELTA>
__global__ __launch_bounds__(256, 1) void scan_chunks_kernel(ScanChunks a) {
    constexpr int NT = D / 64, ROW = D + 4;
    typedef __attribute__((ext_vector_type(NT))) float fNT;
    __shared__ __attribute__((aligned(16))) float st_lds[2][SC_COLS * ROW], u_lds[DELTA ? SC_COLS * (SC_CHUNK + 4) : 1];
    const int s = blockIdx.z, len = a.seq_q_len[s];
    if (len < a.min_len || len == 0) return;
    const int head = blockIdx.x, qk_head = head / (a.H / a.G), j0 = blockIdx.y * SC_COLS;
    const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int start = a.seq_q_start[s], n_chunks = (len + SC_CHUNK - 1) / SC_CHUNK;
    constexpr int RECORD = CHAN ? SC_CHANNEL_RECORD(D) : DELTA ? SC_DELTA_RECORD(D) : SC_RECORD;
    const size_t rec_step = (size_t)a.H * RECORD;
    const float* rec0 = a.records + ((size_t)scan_first_record(a.seq_q_len, s, a.min_len) * a.H + head) * RECORD;
    float* st = a.state + (size_t)a.seq_slots[s] * a.slot_stride + (size_t)head * D * a.Dv;
    const int d0 = 16 * NT * w + NT * n;
    f32x4 S[NT];                                   // S[i][r]: column j0 + 4 g + r, row d0 + i
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const fNT part = *(const fNT*)(st + (size_t)(j0 + 4 * g + r) * D + d0);
#pragma unroll
        for (int i = 0; i < NT; ++i) S[i][r] = part[i];
    }
    const float skip = a.skip ? a.skip[head] : 0.f;

    f32x4 q[D / 16], pairs[4], suf[4], pre;
    f32x4 wk[DELTA ? D / 16 : 1], tb[DELTA ? 4 : 1];           // T diag(beta p) k of the wave's tokens, T diag(beta)
    float v[4][4];
    fNT k[4][4], last, rest;                       // last: the whole chunk's decay, rest: what its rounding left
    const int ldq = CHAN ? D : a.ldq, ldk = CHAN ? D : a.ldk;
    const unsigned q_at = 4 * ((16 * w + n) * ldq + 4 * g), k_at = 4 * (4 * g * ldk + d0), v_at = 4 * (4 * g * a.ldv + n);
    struct Chunk {
        __amdgpu_buffer_rsrc_t q, k, v;
        const float* rec;
    };
    auto chunk = [&](int c) {
        const int t0 = start + c * SC_CHUNK, cnt = min(SC_CHUNK, len - c * SC_CHUNK);
        const float* rec = rec0 + (size_t)c * rec_step;
        const float* qrows = CHAN ? rec + SC_CHANNEL_Q : a.q + (size_t)t0 * a.ldq + qk_head * D;
        const float* krows = CHAN ? rec + SC_CHANNEL_Q + SC_CHUNK * D : a.k + (size_t)t0 * a.ldk + qk_head * D;
        return Chunk{scan_rows(qrows, cnt, ldq, D), scan_rows(krows, cnt, ldk, D),
                     scan_rows(a.v + (size_t)t0 * a.ldv + head * a.Dv + j0, cnt, a.ldv, SC_COLS), rec};
    };
    auto load_q = [&](const Chunk& c, int u) { q[u] = scan_load<4>(c.q, q_at, 64 * u); };
    auto load_v = [&](const Chunk& c, int b, int e) { v[b][e] = scan_load<1>(c.v, v_at, 4 * (16 * b + e) * a.ldv)[0]; };
    auto load_rows = [&](const Chunk& c, int b, int e) {
        if (!DELTA) load_v(c, b, e);
        k[b][e] = scan_load<NT>(c.k, k_at, 4 * (16 * b + e) * ldk);
    };
    auto load_pairs = [&](const Chunk& c) {
#pragma unroll
        for (int b = 0; b < 4; ++b) pairs[b] = *(const f32x4*)(c.rec + (16 * w + n) * SC_CHUNK + 16 * min(b, w) + 4 * g);
    };
    auto load_wk = [&](const Chunk& c, int u) { wk[DELTA ? u : 0] = *(const f32x4*)(c.rec + SC_DELTA_W + (16 * w + n) * D + 16 * u + 4 * g); };
    auto load_tb = [&](const Chunk& c) {
#pragma unroll
        for (int b = 0; b < (DELTA ? 4 : 1); ++b) tb[b] = *(const f32x4*)(c.rec + SC_DELTA_T + (16 * w + n) * SC_CHUNK + 16 * min(b, w) + 4 * g);
    };
    auto load_decays = [&](const Chunk& c) {
        if constexpr (CHAN) {
            const float* whole = c.rec + SC_CHANNEL_Q + 2 * SC_CHUNK * D + d0;
            last = *(const fNT*)whole;
            rest = *(const fNT*)(whole + D);
        } else {
#pragma unroll
            for (int b = 0; b < 4; ++b) suf[b] = *(const f32x4*)(c.rec + SC_SUF + 16 * b + 4 * g);
            pre = *(const f32x4*)(c.rec + SC_PRE + 16 * w + 4 * g);
#pragma unroll
            for (int i = 0; i < NT; ++i) { last[i] = c.rec[SC_PRE + SC_CHUNK - 1]; rest[i] = c.rec[SC_REST]; }
        }
    };
    {
        const Chunk first = chunk(0);
        if constexpr (DELTA) {
#pragma unroll
            for (int u = 0; u < D / 16; ++u) load_wk(first, u);
            __builtin_amdgcn_sched_barrier(0);
            load_tb(first);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int b = 0; b < 4; ++b)
#pragma unroll
                for (int e = 0; e < 4; ++e) load_v(first, b, e);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int u = 0; u < D / 16; ++u) load_q(first, u);
        __builtin_amdgcn_sched_barrier(0);         // (in the order of the loop: what a wait counts there holds for the first chunk too)
        load_pairs(first);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) load_rows(first, b, e);
        __builtin_amdgcn_sched_barrier(0);
        load_decays(first);
        __builtin_amdgcn_sched_barrier(0);
    }
    // A lower triangular matrix (this wave's 16 rows of it, the tiles' columns left of the diagonal in `rows`) times the chunk's `x`;
    // own: x of this wave's tokens.  The tile on the diagonal is not to meet values above it that are no numbers.
    auto lower = [&](const auto& rows, const float (&x)[4][4], f32x4& own) {
        f32x4 sum[4] = {}, row = rows[0];
        own = (f32x4){x[0][0], x[0][1], x[0][2], x[0][3]};
#pragma unroll
        for (int b = 0; b < 3; ++b)
            if (b < w) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    sum[e] = mfma_f32(rows[b][e], x[b][e], sum[e]);
                    own[e] = x[b + 1][e];
                }
                row = rows[b + 1];
            }
        const f32x4 none = own - own;              // zero for finite values, NaN for others
        const unsigned long long odd = __ballot((none[0] + none[1]) + (none[2] + none[3]) != 0.f);
        f32x4 apart = sum[0];                      // of a column with such a value: the tile's tokens one by one, none of them before its own
        if (odd != 0) {
#pragma unroll 1
            for (int t = 0; t < 16; ++t) {
                const float xt = __shfl((t & 2) ? ((t & 1) ? own[3] : own[2]) : ((t & 1) ? own[1] : own[0]), 16 * (t >> 2) + n, 64);
                const float rt = (t & 2) ? ((t & 1) ? row[3] : row[2]) : ((t & 1) ? row[1] : row[0]);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float p = __shfl(rt, 16 * (t >> 2) + 4 * g + r, 64);
                    if (t <= 4 * g + r) apart[r] = fmaf(p, xt, apart[r]);
                }
            }
        }
        apart += (sum[1] + sum[2]) + sum[3];
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[e] = mfma_f32(row[e], own[e], sum[e]);
        const bool is_odd = (odd >> n | odd >> (16 + n) | odd >> (32 + n) | odd >> (48 + n)) & 1;
        f32x4 all = (sum[0] + sum[1]) + (sum[2] + sum[3]);
#pragma unroll
        for (int r = 0; r < 4; ++r) all[r] = is_odd ? apart[r] : all[r];
        return all;
    };
    for (int c = 0; c < n_chunks; ++c) {
        const Chunk next = chunk(min(c + 1, n_chunks - 1));    // (no branch: the compiler would wait for every load behind one)
        float* lds = st_lds[c & 1];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            fNT part;
#pragma unroll
            for (int i = 0; i < NT; ++i) part[i] = S[i][r];
            *(fNT*)(lds + (4 * g + r) * ROW + d0) = part;
        }
        // (not __syncthreads(), which would wait for the loads on their way; two buffers: the next chunk's writes do not meet this one's reads)
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        f32x4 sb[D / 16];
#pragma unroll
        for (int u = 0; u < D / 16; ++u) sb[u] = *(const f32x4*)(lds + n * ROW + 16 * u + 4 * g);
        float u[4][4];                             // what the chunk's tokens write
        if constexpr (DELTA) {
            f32x4 held[8] = {};                    // T diag(beta p) K S
#pragma unroll
            for (int i = 0; i < D / 16; ++i) {
#pragma unroll
                for (int e = 0; e < 4; ++e) held[4 * (i & 1) + e] = mfma_f32(wk[DELTA ? i : 0][e], sb[i][e], held[4 * (i & 1) + e]);
                __builtin_amdgcn_sched_barrier(0); // (loads go out where they are written)
                load_wk(next, i);
            }
            f32x4 own;
            f32x4 mine = lower(tb, v, own);
            __builtin_amdgcn_sched_barrier(0);
            load_tb(next);
#pragma unroll
            for (int b = 0; b < 4; ++b)
#pragma unroll
                for (int e = 0; e < 4; ++e) load_v(next, b, e);
            mine -= sum_of_8(held);
            *(f32x4*)(u_lds + n * (SC_CHUNK + 4) + 16 * w + 4 * g) = mine;
        }
        // the state's part of the outputs
        f32x4 seen[8] = {};
#pragma unroll
        for (int i = 0; i < D / 16; ++i) {
#pragma unroll
            for (int e = 0; e < 4; ++e) seen[4 * (i & 1) + e] = mfma_f32(q[i][e], sb[i][e], seen[4 * (i & 1) + e]);
            __builtin_amdgcn_sched_barrier(0);     // (loads go out where they are written)
            load_q(next, i);
        }
        if constexpr (DELTA) {
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const f32x4 four = *(const f32x4*)(u_lds + n * (SC_CHUNK + 4) + 16 * b + 4 * g);
#pragma unroll
                for (int e = 0; e < 4; ++e) u[b][e] = four[e];
            }
        } else {
#pragma unroll
            for (int b = 0; b < 4; ++b)
#pragma unroll
                for (int e = 0; e < 4; ++e) u[b][e] = v[b][e];
        }
        f32x4 own;
        const f32x4 mine = lower(pairs, u, own);
        __builtin_amdgcn_sched_barrier(0);
        load_pairs(next);
        // the state: this chunk's sums apart, 16 tokens a chain, added once
        f32x4 sum[4][NT] = {};
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float behind = CHAN ? u[b][e] : u[b][e] * suf[b][e];
#pragma unroll
                for (int i = 0; i < NT; ++i) sum[b][i] = mfma_f32(behind, k[b][e][i], sum[b][i]);
                __builtin_amdgcn_sched_barrier(0);
                load_rows(next, b, e);
            }
        const int t0 = start + c * SC_CHUNK, cnt = min(SC_CHUNK, len - c * SC_CHUNK);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float num = ((seen[0][r] + seen[1][r]) + (seen[2][r] + seen[3][r])) + ((seen[4][r] + seen[5][r]) + (seen[6][r] + seen[7][r]));
            float y = (CHAN ? num + mine[r] : fmaf(num, pre[r], mine[r])) * a.o_scale;
            if (a.skip) y = fmaf(skip, own[r], y);
            const int t = 16 * w + 4 * g + r;
            if (t < cnt) a.out[((size_t)(t0 + t) * a.H + head) * a.Dv + j0 + n] = y;
#pragma unroll
            for (int i = 0; i < NT; ++i) {
                const float bounded = __builtin_isinf(S[i][r]) ? 0.f : S[i][r];            // (an infinity stays one, as in the walk: `rest` is zero or of either sign)
                S[i][r] = fmaf(S[i][r], last[i], fmaf(bounded, rest[i], (sum[0][i][r] + sum[1][i][r]) + (sum[2][i][r] + sum[3][i][r])));
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        load_decays(next);
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        fNT part;
#pragma unroll
        for (int i = 0; i < NT; ++i) part[i] = S[i][r];
        *(fNT*)(st + (size_t)(j0 + 4 * g + r) * D + d0) = part;
    }
}

template <int D>
static void scan_launch(const ScanChunks& a, int n_chunks, hipStream_t stream) {
    const dim3 pairs(n_chunks, a.H), walk(a.H, a.Dv / SC_COLS, a.n_seqs);
    if (a.chan_decay) {
        constexpr int LDS = (2 * SC_CHUNK * (D + 4) + 12 * D) * 4;
        static const bool configured = hipFuncSetAttribute((const void*)scan_pairs_channel_kernel<D>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS) == hipSuccess;
        (void)configured;
        scan_pairs_channel_kernel<D><<<pairs, 256, LDS, stream>>>(a);
        scan_chunks_kernel<D, true, false><<<walk, 256, 0, stream>>>(a);
    } else if (a.corrects) {
        constexpr int LDS = (SC_CHUNK * (D + 4) + 2 * SC_CHUNK * (SC_CHUNK + 4) + 4 * 16 * 20 + 3 * SC_CHUNK) * 4;
        static const bool configured = hipFuncSetAttribute((const void*)scan_pairs_delta_kernel<D>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS) == hipSuccess;
        (void)configured;
        scan_pairs_delta_kernel<D><<<pairs, 256, LDS, stream>>>(a);
        scan_chunks_kernel<D, false, true><<<walk, 256, 0, stream>>>(a);
    } else {
        scan_pairs_kernel<D><<<pairs, 256, 0, stream>>>(a);
        scan_chunks_kernel<D, false, false><<<walk, 256, 0, stream>>>(a);
    }
}
void scan_chunks_launch(const ScanChunks& a, int D, int n_chunks, hipStream_t stream) {
    if (D == 64) scan_launch<64>(a, n_chunks, stream);
    else if (D == 128) scan_launch<128>(a, n_chunks, stream);
    else scan_launch<256>(a, n_chunks, stream);
}
