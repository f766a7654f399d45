// Row-wise operations on the residual stream and on mixers' outputs that need no matrix product:
// the Dynamic Tanh norm, an embedding look-up with a factor, a gated activation of choice, the
// weighted sum of two normed rows, and a gate (with compaction) on heads side by side.
// All arithmetic is float; only the stores are in the storage type.
#include "common.h"
#include "api.h"
#include "recordable.h"

// ------------------------------------------------------------------ Dynamic Tanh
// out[r][i] = tanh(alpha * s) * w[i] + b[i], s = x[row][i] (+ delta[row][i]); with resid_out the sum is
// written back.  No mean, no variance: nothing crosses the elements of a row.
// A thread takes four neighbouring values of a row (one 16-byte load where the width allows it); a row is
// spread over as many blocks as it has thousands of values, so that a step of few rows still fills units.
template <typename TOut>
__global__ __launch_bounds__(256) void dyt_kernel(const float* __restrict__ x, const float* __restrict__ delta,
                                                  float* __restrict__ resid_out, const int* __restrict__ rows,
                                                  const float* __restrict__ alpha, const float* __restrict__ w,
                                                  const float* __restrict__ b, TOut* __restrict__ out, int H) {
    const int r = blockIdx.x;
    const size_t row = rows ? (size_t)rows[r] : (size_t)r;
    const float a = alpha[0];
    const int i0 = (blockIdx.y * 256 + threadIdx.x) * 4;
    if (i0 >= H) return;
    float s[4];
    if ((H & 3) == 0) {
        const f32x4 v = *(const f32x4*)(x + row * H + i0);
        s[0] = v[0]; s[1] = v[1]; s[2] = v[2]; s[3] = v[3];
        if (delta) {
            const f32x4 d = *(const f32x4*)(delta + row * H + i0);
            s[0] += d[0]; s[1] += d[1]; s[2] += d[2]; s[3] += d[3];
        }
        if (resid_out) *(f32x4*)(resid_out + row * H + i0) = (f32x4){s[0], s[1], s[2], s[3]};
    } else {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int i = i0 + u;
            s[u] = i < H ? x[row * H + i] + (delta ? delta[row * H + i] : 0.f) : 0.f;
            if (resid_out && i < H) resid_out[row * H + i] = s[u];
        }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int i = i0 + u;
        if (i < H) out[(size_t)r * H + i] = from_f32<TOut>(tanhf(a * s[u]) * w[i] + (b ? b[i] : 0.f));
    }
}

extern "C" int fl_dyt(const float* x, const float* delta, float* resid_out, const int* rows, const float* alpha,
                      const float* w, const float* b, void* out, int out_dtype, int n_rows, int H, hipStream_t stream) {
    FL_CHECK(n_rows >= 0 && H > 0, "dyt: bad sizes");
    FL_CHECK(alpha && w, "dyt: needs alpha and a gain");
    FL_CHECK(!(rows && resid_out), "dyt: picked rows are not stored back");
    if (n_rows == 0) return 0;
    FL_CHECK(ceil_div(H, 1024) <= 65535, "dyt: rows of %d values are more than one grid takes", H);
    dim3 grid(n_rows, ceil_div(H, 1024));
    if (out_dtype == FL_F32)
        dyt_kernel<float><<<grid, 256, 0, stream>>>(x, delta, resid_out, rows, alpha, w, b, (float*)out, H);
    else if (out_dtype == FL_BF16)
        dyt_kernel<bf16_t><<<grid, 256, 0, stream>>>(x, delta, resid_out, rows, alpha, w, b, (bf16_t*)out, H);
    else
        FL_CHECK(false, "dyt: unknown dtype %d", out_dtype);
    FL_LAUNCH_CHECK();
    return 0;
}
FL_RECORDABLE(fl_dyt)

// ------------------------------------------------------------------ embedding with a factor
// (a row over several blocks, four values a thread where rows are whole pieces of four: one trip to memory instead of one per 256
// values; 8 rows of 4096 in bfloat16 10.1 -> 3.5 us, 2,048 rows 18.9 -> 14.1)
template <typename T>
__global__ __launch_bounds__(256) void embed_scaled_kernel(const T* __restrict__ table, const int* __restrict__ tokens,
                                                           float* __restrict__ out, int H, int V, float scale, int pieces) {
    int tok = tokens[blockIdx.x];
    if (tok < 0 || tok >= V) tok = 0;  // the host rejects such ids before the launch
    const T* src = table + (size_t)tok * H;
    float* dst = out + (size_t)blockIdx.x * H;
    const int first = blockIdx.y * 256 + threadIdx.x, step = gridDim.y * 256;
    if (pieces) {
        for (int i = 4 * first; i < H; i += 4 * step) {
            T v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = src[i + u];
            *(f32x4*)(dst + i) = (f32x4){to_f32(v[0]) * scale, to_f32(v[1]) * scale, to_f32(v[2]) * scale, to_f32(v[3]) * scale};
        }
    } else {
        for (int i = first; i < H; i += step) dst[i] = to_f32(src[i]) * scale;
    }
}

extern "C" int fl_embed_scaled(const void* table, int dtype, const int* tokens, float* out, int n, int H, int V, float scale,
                               hipStream_t stream) {
    FL_CHECK(n >= 0 && H > 0 && V > 0, "embed_scaled: bad sizes");
    if (n == 0) return 0;
    const int pieces = H % 4 == 0 && (uintptr_t)table % 16 == 0 && (uintptr_t)out % 16 == 0;
    // (value by value, a row over several blocks while the chip holds them all: 2,048 rows of 4,098 8.5 us a block each, 9.4 over five)
    const dim3 grid(n, pieces || (long)n * ceil_div(H, 1024) <= 16 * fl_units() ? min(ceil_div(H, 1024), 64) : 1);
    if (dtype == FL_F32)
        embed_scaled_kernel<float><<<grid, 256, 0, stream>>>((const float*)table, tokens, out, H, V, scale, pieces);
    else if (dtype == FL_BF16)
        embed_scaled_kernel<bf16_t><<<grid, 256, 0, stream>>>((const bf16_t*)table, tokens, out, H, V, scale, pieces);
    else
        FL_CHECK(false, "embed_scaled: unknown dtype %d", dtype);
    FL_LAUNCH_CHECK();
    return 0;
}
FL_RECORDABLE(fl_embed_scaled)

// ------------------------------------------------------------------ gated activation
// kinds as in fl_activation: 0 gelu (error function), 1 gelu (tanh form), 2 silu
__device__ __forceinline__ float activate(float z, int kind) {
    if (kind == 0) return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f));
    if (kind == 1) return 0.5f * z * (1.0f + tanhf(0.79788456080286536f * (z + 0.044715f * z * z * z)));
    return z / (1.0f + expf(-z));
}

// out[r][i] = act(gu[r][i]) * gu[r][I + i]
template <typename TOut>
__global__ __launch_bounds__(256) void gated_act_kernel(const float* __restrict__ gu, TOut* __restrict__ out, int I, int kind) {
    const float* row = gu + (size_t)blockIdx.x * 2 * I;
    const int i0 = (blockIdx.y * 256 + threadIdx.x) * 4;        // four neighbouring values per thread, a row over several blocks
    if (i0 >= I) return;
    if ((I & 3) == 0) {
        const f32x4 g = *(const f32x4*)(row + i0), u = *(const f32x4*)(row + I + i0);
#pragma unroll
        for (int e = 0; e < 4; ++e) out[(size_t)blockIdx.x * I + i0 + e] = from_f32<TOut>(activate(g[e], kind) * u[e]);
    } else {
        for (int i = i0; i < min(i0 + 4, I); ++i) out[(size_t)blockIdx.x * I + i] = from_f32<TOut>(activate(row[i], kind) * row[I + i]);
    }
}

extern "C" int fl_gated_act(const float* gu, void* out, int out_dtype, int n, int I, int kind, hipStream_t stream) {
    FL_CHECK(n >= 0 && I > 0, "gated_act: bad sizes");
    FL_CHECK(kind >= 0 && kind <= 2, "gated_act: unknown activation %d", kind);
    if (n == 0) return 0;
    FL_CHECK(ceil_div(I, 1024) <= 65535, "gated_act: rows of %d values are more than one grid takes", I);
    dim3 grid(n, ceil_div(I, 1024));
    if (out_dtype == FL_F32)
        gated_act_kernel<float><<<grid, 256, 0, stream>>>(gu, (float*)out, I, kind);
    else if (out_dtype == FL_BF16)
        gated_act_kernel<bf16_t><<<grid, 256, 0, stream>>>(gu, (bf16_t*)out, I, kind);
    else
        FL_CHECK(false, "gated_act: unknown dtype %d", out_dtype);
    FL_LAUNCH_CHECK();
    return 0;
}
FL_RECORDABLE(fl_gated_act)

// ------------------------------------------------------------------ clamped gated activation
// out[r][i] = g sigmoid(alpha g) (u + shift), g = min(gu[r][i], limit), u = clamp(gu[r][I + i], -limit, limit)
template <typename TOut>
__global__ __launch_bounds__(256) void clamped_gate_kernel(const float* __restrict__ gu, TOut* __restrict__ out, int I, float alpha,
                                                           float limit, float shift) {
    const float* row = gu + (size_t)blockIdx.x * 2 * I;
    const int i0 = (blockIdx.y * 256 + threadIdx.x) * 4;
    if (i0 >= I) return;
    if ((I & 3) == 0) {
        const f32x4 g = *(const f32x4*)(row + i0), u = *(const f32x4*)(row + I + i0);
#pragma unroll
        for (int e = 0; e < 4; ++e) out[(size_t)blockIdx.x * I + i0 + e] = from_f32<TOut>(clamped_gate(g[e], u[e], alpha, limit, shift));
    } else {
        for (int i = i0; i < min(i0 + 4, I); ++i) out[(size_t)blockIdx.x * I + i] = from_f32<TOut>(clamped_gate(row[i], row[I + i], alpha, limit, shift));
    }
}

extern "C" int fl_clamped_gate(const float* gu, void* out, int out_dtype, int n, int I, float alpha, float limit, float shift,
                               hipStream_t stream) {
    FL_CHECK(n >= 0 && I > 0 && limit > 0.f, "clamped_gate: bad sizes or a limit that is not positive");
    if (n == 0) return 0;
    FL_CHECK(ceil_div(I, 1024) <= 65535, "clamped_gate: rows of %d values are more than one grid takes", I);
    dim3 grid(n, ceil_div(I, 1024));
    if (out_dtype == FL_F32)
        clamped_gate_kernel<float><<<grid, 256, 0, stream>>>(gu, (float*)out, I, alpha, limit, shift);
    else if (out_dtype == FL_BF16)
        clamped_gate_kernel<bf16_t><<<grid, 256, 0, stream>>>(gu, (bf16_t*)out, I, alpha, limit, shift);
    else
        FL_CHECK(false, "clamped_gate: unknown dtype %d", out_dtype);
    FL_LAUNCH_CHECK();
    return 0;
}
FL_RECORDABLE(fl_clamped_gate)

// ------------------------------------------------------------------ weighted sum of two normed rows
// out[t][i] = ca * a[t][i] / rms(a[t]) * wa[i] + cb * b[t][i] / rms(b[t]) * wb[i], rms with eps inside the root.
// PIECES: the 16-byte pieces of each row that a thread holds in registers between the sums and the results (0: any sizes, rows read
// twice a value at a time, a trip to memory per 256 values: 8 rows of 4096 10.5 us, 2,048 rows 27.7; with four pieces 4.6 and 18.9).
template <int PIECES>
__global__ __launch_bounds__(256) void norm_mix_kernel(const float* __restrict__ a, const float* __restrict__ wa, float ca,
                                                       const float* __restrict__ b, const float* __restrict__ wb, float cb,
                                                       float* __restrict__ out, int H, float eps) {
    __shared__ float lds[8];
    const float* ar = a + (size_t)blockIdx.x * H;
    const float* br = b + (size_t)blockIdx.x * H;
    float* dst = out + (size_t)blockIdx.x * H;
    float sa = 0.f, sb = 0.f;
    if constexpr (PIECES > 0) {
        f32x4 va[PIECES], vb[PIECES];
#pragma unroll
        for (int p = 0; p < PIECES; ++p) {
            const int i = 4 * (threadIdx.x + 256 * p);
            const bool in = i < H;
            va[p] = *(const f32x4*)(ar + (in ? i : 0));
            vb[p] = *(const f32x4*)(br + (in ? i : 0));
        }
#pragma unroll
        for (int p = 0; p < PIECES; ++p)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (4 * (threadIdx.x + 256 * p) < H) {
                    sa = fmaf(va[p][r], va[p][r], sa);
                    sb = fmaf(vb[p][r], vb[p][r], sb);
                }
        sa = block_sum<4>(sa, lds);
        sb = block_sum<4>(sb, lds + 4);
        const float ia = ca / sqrtf(sa / (float)H + eps), ib = cb / sqrtf(sb / (float)H + eps);
#pragma unroll
        for (int p = 0; p < PIECES; ++p) {
            const int i = 4 * (threadIdx.x + 256 * p);
            if (i < H) {
                const f32x4 ga = *(const f32x4*)(wa + i), gb = *(const f32x4*)(wb + i);
                f32x4 o;
#pragma unroll
                for (int r = 0; r < 4; ++r) o[r] = va[p][r] * ia * ga[r] + vb[p][r] * ib * gb[r];
                *(f32x4*)(dst + i) = o;
            }
        }
    } else {
        for (int i = threadIdx.x; i < H; i += 256) {
            sa = fmaf(ar[i], ar[i], sa);
            sb = fmaf(br[i], br[i], sb);
        }
        sa = block_sum<4>(sa, lds);
        sb = block_sum<4>(sb, lds + 4);
        const float ia = ca / sqrtf(sa / (float)H + eps), ib = cb / sqrtf(sb / (float)H + eps);
        for (int i = threadIdx.x; i < H; i += 256) dst[i] = ar[i] * ia * wa[i] + br[i] * ib * wb[i];
    }
}

extern "C" int fl_norm_mix(const float* a, const float* wa, float ca, const float* b, const float* wb, float cb, float* out,
                           int n, int H, float eps, hipStream_t stream) {
    FL_CHECK(n >= 0 && H > 0, "norm_mix: bad sizes");
    if (n == 0) return 0;
    const bool whole = H % 4 == 0 && ((uintptr_t)a | (uintptr_t)wa | (uintptr_t)b | (uintptr_t)wb | (uintptr_t)out) % 16 == 0;
    const int pieces = whole ? ceil_div(H, 1024) : 9;
    if (pieces <= 1) norm_mix_kernel<1><<<n, 256, 0, stream>>>(a, wa, ca, b, wb, cb, out, H, eps);       // (2,048 rows of 100 3.8 us, with two pieces 4.05)
    else if (pieces <= 2) norm_mix_kernel<2><<<n, 256, 0, stream>>>(a, wa, ca, b, wb, cb, out, H, eps);
    else if (pieces <= 4) norm_mix_kernel<4><<<n, 256, 0, stream>>>(a, wa, ca, b, wb, cb, out, H, eps);
    else if (pieces <= 8) norm_mix_kernel<8><<<n, 256, 0, stream>>>(a, wa, ca, b, wb, cb, out, H, eps);
    else norm_mix_kernel<0><<<n, 256, 0, stream>>>(a, wa, ca, b, wb, cb, out, H, eps);
    FL_LAUNCH_CHECK();
    return 0;
}
FL_RECORDABLE(fl_norm_mix)

// ------------------------------------------------------------------ gate on heads side by side
// out[t][h * Dv + j] = x[t][h * ldh + j] * g(gate[t][gate_col0 + h * Dv + j]) for j < Dv: the heads of x may be
// wider than Dv (padded); g: 0 none, 1 sigmoid, 2 silu.
template <typename T>
__global__ __launch_bounds__(256) void heads_gate_kernel(const T* __restrict__ x, int ldh, const float* __restrict__ gate, int ldg,
                                                         int gate_col0, int kind, int per_head, float scale, T* __restrict__ out,
                                                         int ldo, int H, int Dv, int pieces) {
    const size_t t = blockIdx.x;
    // (a token's values are spread over blocks, so that a step of few tokens still fills units; pieces: four values a thread, 2,048
    // tokens of 32 heads of 128 24.5 -> 17.3 us)
    if (pieces) {
        for (int e = 4 * (blockIdx.y * 256 + threadIdx.x); e < H * Dv; e += 1024 * gridDim.y) {
            const int h = e / Dv, j = e - h * Dv;
            T v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = x[(t * H + h) * ldh + j + r];
            float z[4] = {0.f, 0.f, 0.f, 0.f};
            if (kind) {
#pragma unroll
                for (int r = 0; r < 4; ++r) z[r] = gate[t * ldg + gate_col0 + (per_head ? h : e + r)];
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float o = to_f32(v[r]) * scale;
                if (kind) o *= kind == 1 ? 1.0f / (1.0f + expf(-z[r])) : z[r] / (1.0f + expf(-z[r]));
                out[t * ldo + e + r] = from_f32<T>(o);
            }
        }
        return;
    }
    for (int e = blockIdx.y * 256 + threadIdx.x; e < H * Dv; e += 256 * gridDim.y) {
        const int h = e / Dv, j = e - h * Dv;
        float v = to_f32(x[(t * H + h) * ldh + j]) * scale;
        if (kind) {
            const float z = gate[t * ldg + gate_col0 + (per_head ? h : e)];
            v *= kind == 1 ? 1.0f / (1.0f + expf(-z)) : z / (1.0f + expf(-z));
        }
        out[t * ldo + e] = from_f32<T>(v);
    }
}

extern "C" int fl_heads_gate(const void* x, int dtype, int ldh, const float* gate, int ldg, int gate_col0, int kind, int per_head,
                             float scale, void* out, int ldo, int n, int H, int Dv, hipStream_t stream) {
    FL_CHECK(n >= 0 && H > 0 && Dv > 0 && ldh >= Dv, "heads_gate: bad sizes");
    FL_CHECK(kind >= 0 && kind <= 2 && (kind == 0 || (gate && ldg >= gate_col0 + (per_head ? H : H * Dv))), "heads_gate: gate %d over rows %d wide", kind, ldg);
    FL_CHECK(ldo >= H * Dv, "heads_gate: output rows of %d values for %d heads of %d", ldo, H, Dv);
    if (n == 0) return 0;
    const size_t piece = dtype == FL_F32 ? 16 : 8;                     // four values of x and of out, and of the gate
    const int pieces = Dv % 4 == 0 && ldh % 4 == 0 && ldo % 4 == 0 && (uintptr_t)x % piece == 0 && (uintptr_t)out % piece == 0 &&
                       (!kind || per_head || (ldg % 4 == 0 && gate_col0 % 4 == 0 && (uintptr_t)gate % 16 == 0));
    // (value by value, two a thread: a trip to memory each, 8 tokens of 32 heads of 126 2.65 us, with four 3.35; four once there are
    // more blocks than the chip holds at a time, 2,048 tokens 20.6 and 19.4)
    const int each = pieces || (long)n * ceil_div(H * Dv, 512) > 16 * fl_units() ? 1024 : 512;
    const dim3 grid(n, min(ceil_div(H * Dv, each), 64));
    if (dtype == FL_F32)
        heads_gate_kernel<float><<<grid, 256, 0, stream>>>((const float*)x, ldh, gate, ldg, gate_col0, kind, per_head, scale, (float*)out, ldo, H, Dv, pieces);
    else if (dtype == FL_BF16)
        heads_gate_kernel<bf16_t><<<grid, 256, 0, stream>>>((const bf16_t*)x, ldh, gate, ldg, gate_col0, kind, per_head, scale, (bf16_t*)out, ldo, H, Dv, pieces);
    else
        FL_CHECK(false, "heads_gate: unknown dtype %d", dtype);
    FL_LAUNCH_CHECK();
    return 0;
}
FL_RECORDABLE(fl_heads_gate)
