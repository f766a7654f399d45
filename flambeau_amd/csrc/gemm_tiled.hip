// Tiled bf16 matrix product for prompt portions: out[m, n] = sum_k x[m, k] w[n, k] with many
// rows m, on the matrix cores (v_mfma_f32_16x16x32_bf16, float accumulation).  Here: the choice of block and parts, and
// the entry points; the kernel and what bounds it: gemm_tiled.h.
//
//  * w arrives packed (kernels/packing.py): a tile of 16 features x 32 k is 1 KB in lane order.
//    Operand tiles of both matrices go from memory straight into LDS (no staging registers, no ds_write): of w a wave copies
//    tiles as they lie, of the row-major x 8 rows of 128 bytes.  A wave
//    then reads an operand from LDS with one ds_read_b128 per lane (w at consecutive addresses, x
//    through an exchange of pieces that keeps the banks apart);
//  * the w tile is the A operand and the x tile the B operand: C[feature][token] leaves each
//    lane with four consecutive features of one token;
//  * blocks of four waves, one block per compute unit, 96 to 288 tokens by 128 to 256 features;
//    blocks are handed to the eight dies in turn, each die working on a compact patch of tiles;
//  * with few rows and a narrow matrix even that grid is small: K is then split over
//    blockIdx.z, the parts are written as float partial sums and a second kernel adds them in
//    a fixed order;
//  * epilogues: plain; SwiGLU over gate/up rows interleaved in fours; rotate and store q and the
//    cache rows (rope_store.h); add to the residual stream and leave the next norm in factors.
//    Every one can scale a token's results by the factor of a norm left that way (TiledFusion).
//
// The reference's nearest kernel multiplies a 64 x 8 tile per 64-thread block without matrix
// cores (crates/kernels-hip/src/kernels/mmq_f16_tile.cu:33-107).
#include "gemm_tiled.h"
extern template void launch_tiled<float, TG_PLAIN>(int, int, hipStream_t, const bf16_t*, const bf16_t*, float*, int, int, int, int, int, int, const RopeStore&, const TiledFusion&);
extern template void launch_tiled<bf16_t, TG_PLAIN>(int, int, hipStream_t, const bf16_t*, const bf16_t*, bf16_t*, int, int, int, int, int, int, const RopeStore&, const TiledFusion&);
extern template void launch_tiled<bf16_t, TG_SWIGLU>(int, int, hipStream_t, const bf16_t*, const bf16_t*, bf16_t*, int, int, int, int, int, int, const RopeStore&, const TiledFusion&);
extern template void launch_tiled<float, TG_SWIGLU>(int, int, hipStream_t, const bf16_t*, const bf16_t*, float*, int, int, int, int, int, int, const RopeStore&, const TiledFusion&);
extern template void launch_tiled<bf16_t, TG_ROPE>(int, int, hipStream_t, const bf16_t*, const bf16_t*, bf16_t*, int, int, int, int, int, int, const RopeStore&, const TiledFusion&);
extern template void launch_tiled<float, TG_RESIDUAL>(int, int, hipStream_t, const bf16_t*, const bf16_t*, float*, int, int, int, int, int, int, const RopeStore&, const TiledFusion&);

template <typename TOut>
__global__ __launch_bounds__(256) void gemm_splitk_reduce_kernel(const float* __restrict__ part,
                                                                 TOut* __restrict__ out, size_t total,
                                                                 int splits) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= total) return;
    float s = part[i];
    for (int z = 1; z < splits; ++z) s += part[(size_t)z * total + i];
    out[i] = from_f32<TOut>(s);
}

// Shape of the block, features x tokens: 3 = 128 x 256, 6 = 128 x 224, 7 = 192 x 224, 8 = 128 x 128, 10 = 256 x 256,
// 11 = 256 x 224, 12 = 192 x 128, 13 = 128 x 160, 14 = 256 x 160, 15 = 128 x 288, 16 = 224 x 288, 17 = 128 x 96; 0 = chosen
// here, together with the number of K-splits.  The entry points whose names end in _ex take either from the caller,
// for tests and measurements.
//
// What a shape costs, in us.  A block has its unit to itself.  Blocks go to the dies in turn, a die's share of the tiles times the parts of
// K: the unit with the most blocks is one of that die.  Per block 7.6 and 0.094 per tile of a wave (its first copies, its epilogue), and its steps, whose cost
// by shape stands in the list (a step with few units at work): more with all units at work, because the chip lowers its clock (256 x 256
// 0.49 us a step on 128 units, 0.63 on 256), more where few tiles of tokens share a tile of w, which then comes from HBM more often and
// with all units at work no faster than HBM gives it, less where a tile's rows are none, which are not fetched.  Splitting K adds the parts'
// way to memory and back and the kernel that sums them: 0.6 us, and 1.2 per million values and part.
// The constants are those that pick best among twelve shapes, chosen from 29 (features 128 to 256, tokens 96 to 384) as those
// whose best is nearest to the best of all: 20 products (7B, 12B and 24B sizes and layers of width 2,048 and 3,072, each with the epilogue
// that it runs with: rotation and stores, sum into the stream, activation, none; where K is split with the kernel that adds the parts) at 51 row
// counts from 65 to 4,001, weights from HBM, shapes and 1 to 6 and 8 parts, 19,600 timings launched back to back.  Picks take 0.9 %
// more time than the best on average; over another 384 products (twelve matrices, 32 row counts) 2.4 % and 19 % at worst.  Where they are known to be wrong: 97 to 128 rows
// of a narrow matrix, which 128 x 96 takes in two tiles of tokens (4096 x 4096 at 97 rows 18.9 us in four parts, 16.5 in six of 128 x 128), narrow matrices in more
// parts than pay, and splits count less than they cost with what stands behind them (7168 x 5120 at 400 rows with the rotation 49 us in two parts, 42 whole in
// 128 x 128; 6144 x 4096 at 512 rows 46 and 42).
struct TileShape { int variant, features, tokens, tiles; float step; };       // tiles: of a wave; step: us per k-step
#define TG_SHAPE(variant, FT, TT, WT, NSW, XP, step) {variant, 64 / WT * FT, 16 * WT * TT, FT * TT, step},
static const TileShape g_shapes[] = {TG_SHAPES(TG_SHAPE)};
#undef TG_SHAPE
static const TileShape& tile_shape(int variant) {
    for (const TileShape& t : g_shapes)
        if (t.variant == variant) return t;
    return g_shapes[0];
}
static bool tiled_known(int variant) { return variant == 0 || tile_shape(variant).variant == variant; }

// k-steps of a part of K: an even number, so that only K's last pair of steps is half empty
static int tiled_steps(int K, int splits) { return 2 * ceil_div(ceil_div(K, 32), 2 * splits); }

static float tiled_cost(const TileShape& t, int splits, int M, int N, int K) {
    const int units = fl_units();
    const int steps = tiled_steps(K, splits);
    const int m_tiles = ceil_div(M, t.tokens);
    const long tiles = (long)ceil_div(N, t.features) * m_tiles, blocks = tiles * splits;
    const int die_units = max(units / 8, 1);
    const long most = ((tiles + 7) / 8 * splits + die_units - 1) / die_units;              // blocks of the unit with the most
    const float busy = (float)blocks / (units * most), empty = 1.f - (float)M / ((long)m_tiles * t.tokens);     // share of the units' rounds that have a block; of the tiles' rows that are none
    const float step = t.step * (1.f + 0.2861f * busy) * (1.f - 0.0126f * empty) + 0.0044f * (t.features / 32) / m_tiles * (1.f + 7.6147f * busy) - 0.0270f * empty * (t.tokens / 32);
    float us = most * (steps * step + 7.6465f + 0.0943f * t.tiles);
    if (splits > 1) us += 0.6108f + 1.2332e-6f * M * N * splits;
    return us;
}

struct TilePlan { int variant, splits; };
// forced_variant / forced_splits: 0 = free; may_split: the epilogue allows parts of K.  The number of
// splits never depends on a forced shape (a caller sizes the workspace from the sizes alone).
static TilePlan tiled_plan(int M, int N, int K, bool may_split, int forced_variant, int forced_splits) {
    const int steps = ceil_div(K, 32);
    int splits = 1;
    if (forced_splits > 0) {
        splits = max(1, min(forced_splits, steps / 8));
    } else if (may_split) {
        float best_us = 0.f;
        for (const TileShape& t : g_shapes) {
            // (any number of parts up to 6, or 8: three fill two rounds where four start a third; 7 and more
            // than 8 measured worse than the formula says, their partial sums no longer stay in the caches)
            for (int s = 1; s <= 8 && (s == 1 || steps / s >= 8); s += (s == 6 ? 2 : 1)) {
                const float us = tiled_cost(t, s, M, N, K);
                if (best_us == 0.f || us < best_us * 0.999f) { best_us = us; splits = s; }
            }
        }
    }
    if (K > TG_MOST_K) return {8, splits};                 // (whichever is asked for: the block whose kernel has 64-bit addresses)
    if (forced_variant) return {forced_variant, splits};
    TilePlan best = {3, splits};
    float best_us = 0.f;
    for (const TileShape& t : g_shapes) {
        const float us = tiled_cost(t, splits, M, N, K);
        if (best_us == 0.f || us < best_us * 0.999f) { best_us = us; best.variant = t.variant; }
    }
    return best;
}

// A product whose blocks leave most of the last round's units idle may go in two launches: as many whole rounds of its first features as
// there are, the rest in smaller blocks that make one more, shorter round (28672 x 4096 at 2,048 rows: 896 blocks of 256 x 256 are
// 3.5 rounds, 366 us; 768 of them and 256 of 128 x 256 for the rest 352; 28672 x 5120 at 800 rows 213 and 194, at 3,072 rows 678 and 649).  0: one launch.  The rest's shape goes to *rest.
static int tiled_first_features(int M, int N, int K, int variant, int* rest) {
    const TileShape& t = tile_shape(variant);
    const int units = fl_units(), m_tiles = ceil_div(M, t.tokens), n_tiles = ceil_div(N, t.features);
    const int rounds = (int)((long)n_tiles * m_tiles / units), first = (int)((long)rounds * units / m_tiles);
    if (rounds < 1 || first < 1 || first >= n_tiles) return 0;
    const int features = first * t.features;
    float best = tiled_cost(t, 1, M, N, K) * 0.98f - 2.5f - tiled_cost(t, 1, M, features, K);      // (2.5: the way from one launch to the next)
    int found = 0;
    for (const TileShape& r : g_shapes) {
        const float us = tiled_cost(r, 1, M, N - features, K);
        if (us < best) { best = us; *rest = r.variant; found = features; }
    }
    return found;
}

// The features of the first launch (0: all in one) of a product with the activation.
extern "C" int fl_gemm_tiled_gate_first(int M, int N, int K) {
    int rest = 0;
    return tiled_first_features(M, N, K, tiled_plan(M, N, K, false, 0, 1).variant, &rest);
}

// Parts in which the residual epilogue leaves a token's sum of squares: one per tile of features.
extern "C" int fl_gemm_tiled_parts_ex(int M, int N, int K, int variant) {
    return ceil_div(N, tile_shape(tiled_plan(M, N, K, false, variant, 0).variant).features);
}
extern "C" int fl_gemm_tiled_parts(int M, int N, int K) { return fl_gemm_tiled_parts_ex(M, N, K, 0); }

// How many ways K is split for a product of this shape (forced > 0: that many, as far as K allows).
extern "C" int fl_gemm_tiled_splits_ex(int M, int N, int K, int forced) {
    return tiled_plan(M, N, K, true, 0, forced).splits;
}
extern "C" int fl_gemm_tiled_splits(int M, int N, int K) { return fl_gemm_tiled_splits_ex(M, N, K, 0); }
// The block shape chosen for a product of this shape (may_split = 0: an epilogue that takes whole sums only).
extern "C" int fl_gemm_tiled_shape(int M, int N, int K, int may_split) { return tiled_plan(M, N, K, may_split != 0, 0, 0).variant; }

// epilogue 0: out[M, N] = x w^T.  epilogue 1 (SwiGLU): out[M, out_cols] = silu(gate) * up from the
// N interleaved gate/up rows of w (K is not split then).  in_ssq (or null): [M, in_parts] partial sums of
// squares of the rows that x was made from; every token's results are multiplied by rsqrt(sum / K + eps).
static int tiled_entry(const void* x, const void* w_packed, void* out, float* workspace, int out_dtype, int M, int N, int K,
                       int epilogue, int out_cols, const float* in_ssq, int in_parts, float eps, int variant,
                       int forced_splits, const GateConstants& gate, hipStream_t stream) {
    FL_CHECK(M >= 0 && N > 0 && K > 0, "gemm_tiled: bad sizes M=%d N=%d K=%d", M, N, K);
    FL_CHECK(K % 8 == 0, "gemm_tiled: K=%d is no multiple of 8 (16-byte loads)", K);
    FL_CHECK(out_dtype == FL_F32 || out_dtype == FL_BF16, "gemm_tiled: unknown output dtype %d", out_dtype);
    const int gate_kind = epilogue >> 4;          // the bits above the low four: the activation of the gate (epilogue 1)
    epilogue &= 15;
    FL_CHECK(epilogue == 0 || epilogue == 1, "gemm_tiled: unknown epilogue %d", epilogue);
    FL_CHECK(gate_kind >= 0 && (gate_kind <= FL_GATE_GELU_ERF || (gate_kind == FL_GATE_CLAMPED && gate.limit > 0.f)) && (gate_kind == 0 || epilogue == 1), "gemm_tiled: gate activation %d", gate_kind);
    FL_CHECK(epilogue == 0 ? out_cols == N : (N % 16 == 0 && out_cols > 0 && out_cols <= N / 2),
             "gemm_tiled: %d output columns do not fit %d rows of w", out_cols, N);
    FL_CHECK(((uintptr_t)x % 16 == 0) && ((uintptr_t)w_packed % 16 == 0) && ((uintptr_t)out % 16 == 0),
             "gemm_tiled: operands must be 16-byte aligned");
    FL_CHECK(!in_ssq || in_parts > 0, "gemm_tiled: a row scale over %d parts", in_parts);
    if (M == 0) return 0;
    const int n_steps = ceil_div(K, 32);
    FL_CHECK(tiled_known(variant), "gemm_tiled: block shape %d (0, 3, 6, 7, 8 or 10 to 17)", variant);
    const TilePlan plan = tiled_plan(M, N, K, !epilogue, variant, epilogue ? 1 : forced_splits);
    const int splits = plan.splits, v = plan.variant;
    FL_CHECK(splits == 1 || workspace, "gemm_tiled: this shape splits K %d ways and needs a workspace", splits);
    const int per = tiled_steps(K, splits);
    const bf16_t* xb = (const bf16_t*)x;
    const bf16_t* wb = (const bf16_t*)w_packed;
    const RopeStore none{};
    const TiledFusion fu = {in_ssq, in_parts, eps, nullptr, nullptr, nullptr, nullptr, gate_kind, nullptr, nullptr, gate, 0};
    if (epilogue) {
        auto launch = [&](int shape, int first, int features, int cols) {             // the results of a range of w's rows
            TiledFusion part = fu;
            part.out_ld = out_cols;
            const bf16_t* w = wb + (size_t)(first / 16) * n_steps * 512;
            if (out_dtype == FL_F32)
                launch_tiled<float, TG_SWIGLU>(shape, 1, stream, xb, w, (float*)out + first / 2, M, features, K, n_steps, per, cols, none, part);
            else
                launch_tiled<bf16_t, TG_SWIGLU>(shape, 1, stream, xb, w, (bf16_t*)out + first / 2, M, features, K, n_steps, per, cols, none, part);
        };
        int rest = 0;
        const int first = variant ? 0 : tiled_first_features(M, N, K, v, &rest);
        if (first > 0 && out_cols > first / 2) {
            launch(v, 0, first, first / 2);
            FL_LAUNCH_CHECK();
            launch(rest, first, N - first, out_cols - first / 2);
        } else {
            launch(v, 0, N, out_cols);
        }
    } else if (splits > 1) {
        launch_tiled<float, TG_PLAIN>(v, splits, stream, xb, wb, workspace, M, N, K, n_steps, per, N, none, fu);
        FL_LAUNCH_CHECK();
        const size_t total = (size_t)M * N;
        const unsigned rb = (unsigned)((total + 255) / 256);
        if (out_dtype == FL_F32)
            gemm_splitk_reduce_kernel<float><<<rb, 256, 0, stream>>>(workspace, (float*)out, total, splits);
        else
            gemm_splitk_reduce_kernel<bf16_t><<<rb, 256, 0, stream>>>(workspace, (bf16_t*)out, total, splits);
    } else if (out_dtype == FL_F32) {
        launch_tiled<float, TG_PLAIN>(v, 1, stream, xb, wb, (float*)out, M, N, K, n_steps, per, N, none, fu);
    } else {
        launch_tiled<bf16_t, TG_PLAIN>(v, 1, stream, xb, wb, (bf16_t*)out, M, N, K, n_steps, per, N, none, fu);
    }
    FL_LAUNCH_CHECK();
    return 0;
}
extern "C" int fl_gemm_tiled_ex(const void* x, const void* w_packed, void* out, float* workspace,
                                int out_dtype, int M, int N, int K, int epilogue, int out_cols,
                                const float* in_ssq, int in_parts, float eps, int variant, int forced_splits,
                                hipStream_t stream) {
    return tiled_entry(x, w_packed, out, workspace, out_dtype, M, N, K, epilogue, out_cols, in_ssq, in_parts, eps, variant, forced_splits,
                       GateConstants{}, stream);
}
FL_RECORDABLE(fl_gemm_tiled_ex)

// epilogue 1 with the clamped gate (fl_gemm_skinny_clamped)
extern "C" int fl_gemm_tiled_clamped(const void* x, const void* w_packed, void* out, int out_dtype, int M, int N, int K,
                                     int out_cols, float alpha, float limit, float shift, hipStream_t stream) {
    return tiled_entry(x, w_packed, out, nullptr, out_dtype, M, N, K, 1 | (FL_GATE_CLAMPED << 4), out_cols, nullptr, 0, 0.f, 0, 0,
                       GateConstants{alpha, limit, shift}, stream);
}
FL_RECORDABLE(fl_gemm_tiled_clamped)

extern "C" int fl_gemm_tiled_scaled(const void* x, const void* w_packed, void* out, float* workspace,
                                    int out_dtype, int M, int N, int K, int epilogue, int out_cols,
                                    const float* in_ssq, int in_parts, float eps, hipStream_t stream) {
    return fl_gemm_tiled_ex(x, w_packed, out, workspace, out_dtype, M, N, K, epilogue, out_cols, in_ssq, in_parts, eps, 0, 0, stream);
}
FL_RECORDABLE(fl_gemm_tiled_scaled)

extern "C" int fl_gemm_tiled(const void* x, const void* w_packed, void* out, float* workspace,
                             int out_dtype, int M, int N, int K, int epilogue, int out_cols,
                             hipStream_t stream) {
    return fl_gemm_tiled_ex(x, w_packed, out, workspace, out_dtype, M, N, K, epilogue, out_cols, nullptr, 0, 0.f, 0, 0, stream);
}
FL_RECORDABLE(fl_gemm_tiled)

// resid[M, N] += x w^T (float, in place), xg[M, N] = bf16(resid * g), out_ssq[M, fl_gemm_tiled_residual_parts(M, N, K)]
// = the sums of resid^2 in parts: the factors of the norm that follows.  Where K is not split the
// product's epilogue does it (one part per tile of features); where it is, the partial sums go to
// the workspace (fl_gemm_tiled_splits(M, N, K) * M * N floats) and the kernel that adds them does it
// (one part per 4096 features, fl_reduce_residual).
extern "C" int fl_gemm_tiled_residual_ex(const void* x, const void* w_packed, float* workspace, int M, int N, int K,
                                         float* resid, const float* g, void* xg, float* out_ssq, int variant,
                                         hipStream_t stream) {
    FL_CHECK(tiled_known(variant), "gemm_tiled_residual: block shape %d (0, 3, 6, 7, 8 or 10 to 17)", variant);
    FL_CHECK(M >= 0 && N > 0 && K > 0, "gemm_tiled_residual: bad sizes M=%d N=%d K=%d", M, N, K);
    FL_CHECK(K % 8 == 0, "gemm_tiled_residual: K=%d is no multiple of 8 (16-byte loads)", K);
    FL_CHECK(N % 4 == 0, "gemm_tiled_residual: N=%d is no multiple of 4 (16-byte accesses to the residual rows)", N);
    FL_CHECK(resid && g && xg && out_ssq, "gemm_tiled_residual: needs resid, g, xg and out_ssq");
    FL_CHECK(((uintptr_t)x % 16 == 0) && ((uintptr_t)w_packed % 16 == 0) && ((uintptr_t)resid % 16 == 0) &&
             ((uintptr_t)g % 16 == 0) && ((uintptr_t)xg % 8 == 0), "gemm_tiled_residual: operands must be aligned (16 bytes, xg 8)");
    if (M == 0) return 0;
    const int n_steps = ceil_div(K, 32);
    const TilePlan plan = tiled_plan(M, N, K, true, variant, 0);
    const int splits = plan.splits;
    if (splits > 1) {
        FL_CHECK(workspace && (uintptr_t)workspace % 16 == 0, "gemm_tiled_residual: this shape splits K %d ways and needs a workspace", splits);
        launch_tiled<float, TG_PLAIN>(plan.variant, splits, stream, (const bf16_t*)x, (const bf16_t*)w_packed, workspace, M, N, K,
                                      n_steps, tiled_steps(K, splits), N, RopeStore{}, TiledFusion{});
        FL_LAUNCH_CHECK();
        return fl_reduce_residual(workspace, resid, g, xg, out_ssq, M, N, splits, stream);
    }
    const TiledFusion fu = {nullptr, 0, 0.f, resid, g, (bf16_t*)xg, out_ssq};
    launch_tiled<float, TG_RESIDUAL>(plan.variant, 1, stream, (const bf16_t*)x, (const bf16_t*)w_packed, resid, M, N, K,
                                     n_steps, n_steps, N, RopeStore{}, fu);
    FL_LAUNCH_CHECK();
    return 0;
}
FL_RECORDABLE(fl_gemm_tiled_residual_ex)

// resid[M, N] += x w^T with the Dynamic Tanh norm of the sum in the same epilogue, xn = bf16(tanh(alpha[0] * resid)
// * g + bias), as fl_gemm_skinny_dyt; for shapes whose K the plan does not split (fl_gemm_tiled_splits(M, N, K) == 1).
extern "C" int fl_gemm_tiled_dyt(const void* x, const void* w_packed, int M, int N, int K, float* resid,
                                 const float* alpha, const float* g, const float* bias, void* xn, hipStream_t stream) {
    FL_CHECK(M >= 0 && N > 0 && K > 0, "gemm_tiled_dyt: bad sizes M=%d N=%d K=%d", M, N, K);
    FL_CHECK(K % 8 == 0, "gemm_tiled_dyt: K=%d is no multiple of 8 (16-byte loads)", K);
    FL_CHECK(N % 4 == 0, "gemm_tiled_dyt: N=%d is no multiple of 4 (16-byte accesses to the residual rows)", N);
    FL_CHECK(resid && alpha && g && xn, "gemm_tiled_dyt: needs resid, alpha, g and xn");
    FL_CHECK(((uintptr_t)x % 16 == 0) && ((uintptr_t)w_packed % 16 == 0) && ((uintptr_t)resid % 16 == 0) &&
             ((uintptr_t)g % 16 == 0) && (!bias || (uintptr_t)bias % 16 == 0) && ((uintptr_t)xn % 8 == 0),
             "gemm_tiled_dyt: operands must be aligned (16 bytes, xn 8)");
    if (M == 0) return 0;
    const int n_steps = ceil_div(K, 32);
    const TilePlan plan = tiled_plan(M, N, K, true, 0, 0);
    FL_CHECK(plan.splits == 1, "gemm_tiled_dyt: this shape splits K %d ways; run product and norm apart", plan.splits);
    const TiledFusion fu = {nullptr, 0, 0.f, resid, g, (bf16_t*)xn, nullptr, 0, alpha, bias};
    launch_tiled<float, TG_RESIDUAL>(plan.variant, 1, stream, (const bf16_t*)x, (const bf16_t*)w_packed, resid, M, N, K,
                                     n_steps, n_steps, N, RopeStore{}, fu);
    FL_LAUNCH_CHECK();
    return 0;
}
FL_RECORDABLE(fl_gemm_tiled_dyt)

extern "C" int fl_gemm_tiled_residual(const void* x, const void* w_packed, float* workspace, int M, int N, int K,
                                      float* resid, const float* g, void* xg, float* out_ssq, hipStream_t stream) {
    return fl_gemm_tiled_residual_ex(x, w_packed, workspace, M, N, K, resid, g, xg, out_ssq, 0, stream);
}
FL_RECORDABLE(fl_gemm_tiled_residual)

// Parts in which fl_gemm_tiled_residual leaves a token's sum of squares.
extern "C" int fl_gemm_tiled_residual_parts(int M, int N, int K) {
    return fl_gemm_tiled_splits(M, N, K) > 1 ? fl_gemm_mid_parts(N) : fl_gemm_tiled_parts(M, N, K);
}

// The K-splits of x w^T left apart: workspace[splits][M][N] (splits = fl_gemm_tiled_splits(M, N, K), at
// least one) for a kernel that adds them with work of its own (the rotation kernel does).  in_ssq as
// in fl_gemm_tiled_scaled: every part is scaled, so that their sum is.
extern "C" int fl_gemm_tiled_partials(const void* x, const void* w_packed, float* workspace, int M, int N, int K,
                                      const float* in_ssq, int in_parts, float eps, hipStream_t stream) {
    FL_CHECK(M >= 0 && N > 0 && K > 0, "gemm_tiled_partials: bad sizes M=%d N=%d K=%d", M, N, K);
    FL_CHECK(K % 8 == 0, "gemm_tiled_partials: K=%d is no multiple of 8 (16-byte loads)", K);
    FL_CHECK(workspace && ((uintptr_t)x % 16 == 0) && ((uintptr_t)w_packed % 16 == 0) && ((uintptr_t)workspace % 16 == 0),
             "gemm_tiled_partials: operands must be 16-byte aligned");
    FL_CHECK(!in_ssq || in_parts > 0, "gemm_tiled_partials: a row scale over %d parts", in_parts);
    if (M == 0) return 0;
    const int n_steps = ceil_div(K, 32);
    const TilePlan plan = tiled_plan(M, N, K, true, 0, 0);
    const TiledFusion fu = {in_ssq, in_parts, eps, nullptr, nullptr, nullptr, nullptr};
    launch_tiled<float, TG_PLAIN>(plan.variant, plan.splits, stream, (const bf16_t*)x, (const bf16_t*)w_packed, workspace, M, N, K,
                                  n_steps, tiled_steps(K, plan.splits), N, RopeStore{}, fu);
    FL_LAUNCH_CHECK();
    return 0;
}
FL_RECORDABLE(fl_gemm_tiled_partials)

// The joined q/k/v projection of many rows with its rows in paired order: q is rotated and written to
// q_out[M, nh * hd], k rotated and v as it is into the cache pages at the tokens' positions; cs[M,
// rot / 2, 2] are the step's cosines and sines.  K is never split here (shapes whose K the plain
// product would split go to that product and the rotation kernel).  in_ssq as in
// fl_gemm_tiled_scaled.
extern "C" int fl_gemm_tiled_rope_ex(const void* x, const void* w_packed, int M, int N, int K, const float* in_ssq,
                                     int in_parts, float eps, const int* positions, const int* tok_seq,
                                     const int* block_table, int max_blocks, const float* cs, void* q_out,
                                     void* cache_base, int nh, int nkv, int hd, int page_size, int n_pages, int rot,
                                     int write_cache, int variant, hipStream_t stream) {
    FL_CHECK(tiled_known(variant), "gemm_tiled_rope: block shape %d (0, 3, 6, 7, 8 or 10 to 17)", variant);
    FL_CHECK(M >= 0 && N > 0 && K > 0, "gemm_tiled_rope: bad sizes M=%d N=%d K=%d", M, N, K);
    FL_CHECK(K % 8 == 0, "gemm_tiled_rope: K=%d is no multiple of 8 (16-byte loads)", K);
    FL_CHECK(positions && tok_seq && block_table && cs && q_out && cache_base,
             "gemm_tiled_rope: needs positions, requests, block table, angles, q and the cache");
    FL_CHECK(hd % 16 == 0 && rot % 16 == 0 && rot <= hd && N == (nh + 2 * nkv) * hd,
             "gemm_tiled_rope: %d features with heads of %d (%d rotated), %d + 2 x %d heads", N, hd, rot, nh, nkv);
    FL_CHECK(((uintptr_t)x % 16 == 0) && ((uintptr_t)w_packed % 16 == 0), "gemm_tiled_rope: operands must be 16-byte aligned");
    FL_CHECK(!in_ssq || in_parts > 0, "gemm_tiled_rope: a row scale over %d parts", in_parts);
    if (M == 0) return 0;
    const RopeStore rs = {positions, tok_seq, block_table, max_blocks, (const float2*)cs, (bf16_t*)q_out,
                          PagedCache{cache_base, nkv, page_size, hd, n_pages}, nh, rot, write_cache};
    const TiledFusion fu = {in_ssq, in_parts, eps, nullptr, nullptr, nullptr, nullptr};
    const int n_steps = ceil_div(K, 32);
    launch_tiled<bf16_t, TG_ROPE>(tiled_plan(M, N, K, false, variant, 0).variant, 1, stream, (const bf16_t*)x, (const bf16_t*)w_packed, (bf16_t*)q_out,
                                  M, N, K, n_steps, n_steps, N, rs, fu);
    FL_LAUNCH_CHECK();
    return 0;
}
FL_RECORDABLE(fl_gemm_tiled_rope_ex)

extern "C" int fl_gemm_tiled_rope(const void* x, const void* w_packed, int M, int N, int K, const float* in_ssq,
                                  int in_parts, float eps, const int* positions, const int* tok_seq,
                                  const int* block_table, int max_blocks, const float* cs, void* q_out,
                                  void* cache_base, int nh, int nkv, int hd, int page_size, int n_pages, int rot,
                                  int write_cache, hipStream_t stream) {
    return fl_gemm_tiled_rope_ex(x, w_packed, M, N, K, in_ssq, in_parts, eps, positions, tok_seq, block_table, max_blocks, cs,
                                 q_out, cache_base, nh, nkv, hd, page_size, n_pages, rot, write_cache, 0, stream);
}
FL_RECORDABLE(fl_gemm_tiled_rope)
