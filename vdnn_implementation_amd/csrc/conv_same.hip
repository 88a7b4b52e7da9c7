// Launchers of the float convolutions on the bfloat16 matrix cores at float precision (conv_same_f32x3.h).
#include "conv_launch.h"
#include "conv_same_f32x3.h"
#include "wgrad_same.h"

namespace vdnn {

// ---- float layers: 3x3 and 5x5 at stride 1, output planes as large as the input's, on the bfloat16 matrix cores at float
// precision (conv_same_f32x3.h): the filter in three parts at the front of the staging area, where half of that stays free.
//
// Where it pays: a tile has 64 rows and 256 pixels, and short reductions leave it mostly prologue and epilogue; below, the float
// engine's 64x64 tiles are faster (1 x 64 x 56 x 56, 128 of 3x3 forward 17.2 us there, 20.9 here; 16 x 16 x 81 x 81, 80 of 3x3 54 and 58).
// Of 1200 calls of 1 to 128 samples and 16 to 576 channels timed on both, those beyond the lines gained 89.5 ms together and
// lost 0.04, by 15 % at most; at 1e9 operations and any depth 90.6 and 1.3.
constexpr double kX3LeastOps = 2.5e9;
constexpr int kX3LeastDepth = 288;
static bool x3_pays(const ConvGeo& g, int rows, int reduced) {
    return reduced * g.R * g.S >= kX3LeastDepth && 2.0 * rows * (double)g.N * g.H * g.W * reduced * g.R * g.S >= kX3LeastOps;
}
// Layers of more than kSmallTileOps operations keep the order of their sums, as on the tile engine (mfma_gemm.h): OverFeat at batch 128, whose
// steps take 103 ms here for 118, saturates its softmax, and in one of ten drawn steps its parameters came out 3.6e-5 from the float
// instruction's.
//
// Layers of the float filter-row kernel (3x3, even rows of fourteen pixels or more, input channels in blocks of 64: every layer of VGG16
// but the first) keep the float instruction in all three passes, where they run at 0.8 to 0.9 of its peak, although these kernels take
// 0.6 to 0.65 of the time there too (64 x 256 x 56 x 56, 256 filters, forward 1755 and 1074 us, backward data 1765 and 1083, backward
// filter 1845 and 1190): deep stacks of such layers train to other parameters in the last places when the order of any sum changes.
// A pre-activation that falls on the other side of zero opens or shuts a unit for a sample; with backward data and filter alone
// on these kernels, in 7 of 34 drawn pairs of VGG16 steps at batch 128 a weight of the fully connected layers moved by 2.5e-5 to 8e-5
// of itself against the float instruction's step (AlexNet at batches of 7 and 32, OverFeat at 24: 1.9e-5 at most in 18).
static bool x3_layer(const ConvGeo& g) {
    return 2.0 * g.K * (double)g.N * g.H * g.W * g.C * g.R * g.S <= kSmallTileOps && (g.R == 3 || g.R == 5) && g.S == g.R && g.ph == g.R / 2 && g.pw == g.ph && g.sh == 1 && g.sw == 1 && !wgrad3x3_f32_ok(g);
}

static bool same_x3_ok(const ConvGeo& g, int mode) {
    const int reduced = mode == 0 ? g.C : g.K, rows = mode == 0 ? g.K : g.C;
    return x3_layer(g) && reduced % X3_CH == 0 && g.C > 4 &&
           (long)rows * reduced * g.R * g.S * 6 < 0x7FFF0000l && pixel_tile_span_ok((long)reduced * g.H * g.W, g.H * g.W, X3_TN, 4) && x3_pays(g, rows, reduced);
}

// How the reduction is split. A compute unit takes a filter row of sixteen channels (S steps) of one workgroup in kAlone us per
// three steps, of two together in kPair (measured on 1 to 784 tiles over 12 to 96 filter rows: 2.05 and 3.15); prologue and
// epilogue are about 4.5 such rows. Either every tile is split, or only those behind the first full_tiles, which are
// whole rounds of one workgroup a unit: 128 x 512 x 14 x 14, 512 filters of 3x3, 784 tiles 629 us unsplit, 554 with sixteen of them split.
struct X3Plan { int splits = 1; long full_tiles = 0; double us = 0.0; };
static X3Plan x3_plan(int M, int N, int filter_rows, int S, size_t room, int num_cu) {
    constexpr double kAlone = 2.05, kPair = 3.15, kEnds = 4.5, kSum = 5.0, kBytes = 4e6; // us, us, filter rows, us, bytes per us
    const double per_row = S / 3.0;
    auto rounds_us = [&](long per_cu, double rows) { return ((double)(per_cu / 2) * kPair + (double)(per_cu % 2) * kAlone) * (rows * per_row + kEnds); };
    auto per_cu = [&](long blocks) { return (blocks + num_cu - 1) / num_cu; };
    const long tiles = (long)((M + X3_TM - 1) / X3_TM) * ((N + X3_TN - 1) / X3_TN), most = filter_rows / 2 > 1 ? filter_rows / 2 : 1;
    const double out_bytes = 4.0 * M * N, tile_bytes = 4.0 * X3_TM * X3_TN;
    X3Plan best;
    best.us = rounds_us(per_cu(tiles), filter_rows);
    for (long s = 2; s <= most && s * out_bytes <= (double)room && tiles * s <= 8l * num_cu; s++) {
        const double us = rounds_us(per_cu(tiles * s), (double)((filter_rows + s - 1) / s)) + kSum + 1.2 * s * out_bytes / kBytes;
        if (us < best.us) { best.splits = (int)s; best.us = us; best.full_tiles = 0; }
    }
    for (long rounds = tiles / num_cu; rounds >= 1 && rounds >= tiles / num_cu - 1; rounds--) {
        const long rem = tiles - rounds * num_cu;
        for (long s = 2; rem > 0 && s <= most && s * rem * tile_bytes <= (double)room && rem * s <= 4l * num_cu; s++) {
            const double us = rounds_us(rounds, filter_rows) + rounds_us(per_cu(rem * s), (double)((filter_rows + s - 1) / s)) + kSum + 1.2 * s * rem * tile_bytes / kBytes;
            if (us < best.us) { best.splits = (int)s; best.us = us; best.full_tiles = rounds * num_cu; }
        }
    }
    return best;
}

template <int MODE>
static int launch_same_x3(vdnn_ctx* ctx, hipStream_t st, StagingCarve& carve, const ConvGeo& g, const float* src, const float* w, StoreNCHW<float> ep, bool* taken) {
    *taken = false;
    if (!same_x3_ok(g, MODE)) return VDNN_OK;
    const int rows = MODE == 0 ? g.K : g.C, reduced = MODE == 0 ? g.C : g.K, RS = g.R * g.S;
    const int M = rows, N = g.N * g.H * g.W, K = reduced * RS, DEPTH = X3_CH * g.S;
    const size_t bank = (size_t)rows * K * 6;
    unsigned short* packed = (unsigned short*)packed_filter_place(ctx, carve, bank);
    if (!packed) return VDNN_OK;
    *taken = true;
    const int row_stride = MODE == 0 ? g.C * RS : RS, red_stride = MODE == 0 ? RS : g.C * RS;
    {
        const long total = (long)rows * K;
        ProfScope prof(ctx, st, "conv_pack_filter", 0.0, 10.0 * (double)total);
        hipLaunchKernelGGL(pack_filter_split3_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, w, packed, reduced, RS, row_stride, red_stride, total);
        VDNN_LAUNCH_CHECK();
    }
    ep.partial = ctx->reduce_scratch;
    const size_t room = ctx->reduce_scratch_bytes;
    const X3Plan plan = x3_plan(M, N, reduced * g.R / X3_CH, g.S, room, ctx->num_cu);
    GemmDims d = make_dims(M, N, K, X3_TM, X3_TN, plan.splits, DEPTH);
    const long tiles = (long)d.mtiles * d.ntiles;
    if (plan.full_tiles > 0 && d.splits > 1) d.full_tiles = (int)plan.full_tiles;
    const long blocks = d.full_tiles > 0 ? d.full_tiles + (tiles - d.full_tiles) * d.splits : tiles * d.splits;
    if (blocks <= 0 || blocks >= (1l << 31)) { set_error("convolution: grid of %ld workgroups out of range", blocks); return VDNN_EINVAL; }
    const ConvSameX3 geo{src, packed, w, (unsigned)bank, row_stride, red_stride, g.H, g.W, reduced, (long)reduced * g.H * g.W, g.N};
    {
        ProfScope prof(ctx, st, MODE == 0 ? "conv_fwd_x3_64x256" : "conv_bwd_data_x3_64x256", 2.0 * g.N * (double)g.K * g.C * RS * g.P * g.Q, 0.0);
        const dim3 grid((unsigned)blocks);
        if (g.S == 3 && g.W % 2 == 0) hipLaunchKernelGGL((conv_same_f32x3_kernel<MODE, 3, true>), grid, dim3(NT), 0, st, geo, ep, d);
        else if (g.S == 3) hipLaunchKernelGGL((conv_same_f32x3_kernel<MODE, 3, false>), grid, dim3(NT), 0, st, geo, ep, d);
        else if (g.W % 2 == 0) hipLaunchKernelGGL((conv_same_f32x3_kernel<MODE, 5, true>), grid, dim3(NT), 0, st, geo, ep, d);
        else hipLaunchKernelGGL((conv_same_f32x3_kernel<MODE, 5, false>), grid, dim3(NT), 0, st, geo, ep, d);
        VDNN_LAUNCH_CHECK();
    }
    if (d.splits == 1) return VDNN_OK;
    if (d.full_tiles > 0)
        return launch_reduce_tail_nchw(ctx, st, ep.out, ep.partial, (int)(tiles - d.full_tiles), d.splits, X3_TM, X3_TN, M, N, d.mtiles, d.full_tiles, ep.bias, ep.opix, ep.relu, ep.gate);
    return launch_reduce_splits_nchw(ctx, st, ep.out, ep.partial, (size_t)M * N, d.splits, ep.bias, ep.opix, M, ep.relu, ep.gate);
}

int launch_same_x3_fwd(vdnn_ctx* ctx, hipStream_t st, StagingCarve& carve, const ConvGeo& g, const float* x, const float* w, const float* bias, float* y, int relu, bool* taken) {
    return launch_same_x3<0>(ctx, st, carve, g, x, w, StoreNCHW<float>{y, bias, g.P * g.Q, nullptr, relu, nullptr}, taken);
}
int launch_same_x3_bwd_data(vdnn_ctx* ctx, hipStream_t st, StagingCarve& carve, const ConvGeo& g, const float* dy, const float* w, float* dx, const float* gate, bool* taken) {
    return launch_same_x3<1>(ctx, st, carve, g, dy, w, StoreNCHW<float>{dx, nullptr, g.H * g.W, nullptr, 0, gate}, taken);
}

// ---- backward filter of the same layers (wgrad_same.h) --------------------------------------------------------------
static bool wgrad_same_ok(const ConvGeo& g) {
    if (!x3_layer(g) || g.C % 8 != 0 || g.K % 8 != 0) return false;
    const int WP = g.W + g.S / 2;
    return g.H > WS_SLICE / WP && (long)g.N * g.H * WP < (1l << 30); // a slice reaches at most one sample further
}
// ... and pays: the tiles count 64 channels of each operand and S/2 slots more than pixels per row; beyond three times the
// products the float engine's tiles are faster, as on small layers (4 x 64 x 30 x 31, 64 of 3x3 16.7 us there, 22.0 here; 112 x 8 x 20 x 119, 320
// of 3x3 293 and 430; 1 x 64 x 56 x 56, 128 of 3x3 33.6 and 22.5). Of 500 calls timed on both, those beyond the lines gained 19.1 ms
// together and lost 0.03.
constexpr double kWgradX3LeastOps = 6e8, kWgradX3MostWaste = 3.0;
bool wgrad_same_x3_ok(const ConvGeo& g) {
    if (!wgrad_same_ok(g)) return false;
    const double products = (double)g.C * g.K * g.W, padded = (double)((g.C + 63) / 64 * 64) * ((g.K + 63) / 64 * 64) * (g.W + g.S / 2);
    return padded <= kWgradX3MostWaste * products && 2.0 * products * g.N * g.H * g.R * g.S >= kWgradX3LeastOps;
}

// Splits of the reduction. A compute unit takes a slice of one workgroup in kAlone us, of two together in kPair (S = 3; measured on
// 64 x 128 x 112 x 112), prologue and epilogue are about four slices.
static long wgrad_same_splits(long tiles, long slices, size_t out_bytes, size_t room, int S, int num_cu) {
    constexpr double kAlone = 1.35, kPair = 2.05, kEnds = 4.0, kSum = 5.0, kBytes = 4e6;
    double best_us = 0.0;
    long best = 1;
    for (long s = 1; s <= slices / 4 || s == 1; s++) {
        if (s > 1 && (s * out_bytes > room || tiles * s > 8l * num_cu)) break;
        const long per_cu = (tiles * s + num_cu - 1) / num_cu;
        const double us = ((double)(per_cu / 2) * kPair + (double)(per_cu % 2) * kAlone) * S / 3.0 * ((double)((slices + s - 1) / s) + kEnds) +
                          (s > 1 ? kSum + 1.2 * (double)s * (double)out_bytes / kBytes : 0.0);
        if (s == 1 || us < best_us) { best = s; best_us = us; }
    }
    return best;
}

int launch_wgrad_same_x3(vdnn_ctx* ctx, hipStream_t st, const ConvGeo& g, const float* x, const float* dy, float* w, float alpha, int accumulate,
                         float* staging, size_t staging_bytes, bool* taken, BiasOut* bias) {
    *taken = false;
    if (!wgrad_same_x3_ok(g)) return VDNN_OK;
    const int S = g.S, M = g.K, N = g.C * S * S, WP = g.W + S / 2, HW = g.H * g.W;
    const int Kred = g.N * g.H * WP;
    constexpr int TM = 64;
    const int mtiles = (M + TM - 1) / TM, ntiles = S * ((g.C + WS_CH - 1) / WS_CH);
    const long tiles = (long)mtiles * ntiles;
    const long splits = wgrad_same_splits(tiles, (Kred + WS_SLICE - 1) / WS_SLICE, (size_t)M * N * sizeof(float), staging ? staging_bytes : 0, S, ctx->num_cu);
    GemmDims d = make_dims(M, N, Kred, TM, S * WS_CH, (int)splits, WS_SLICE);
    d.mtiles = mtiles; d.ntiles = ntiles;
    const long nspan = d.kchunk / (g.H * WP) + 3;
    if (nspan * g.K * HW * 4 >= (long)MAX_SUM_RANGE || nspan * g.C * HW * 4 >= (long)MAX_SUM_RANGE) return VDNN_OK; // not taken
    const long blocks = tiles * d.splits;
    if (blocks <= 0 || blocks >= (1l << 31)) return VDNN_OK;
    *taken = true;
    const bool with_bias = bias && bias->wanted() && bias_parts_fit(ctx, g.K, d.splits);
    const WgradSame geo{dy, x, g.N, g.K, g.C, g.H, g.W, w, staging, (long)M * N, alpha, accumulate, with_bias ? ctx->bias_scratch : nullptr, d.splits,
                           Kred, WS_SLICE / WP, WS_SLICE % WP};
    {
        ProfScope prof(ctx, st, S == 3 ? "conv_bwd_filter_x3_3x3" : "conv_bwd_filter_x3_5x5", 2.0 * M * (double)N * (double)g.N * HW, 0.0);
        if (S == 5) hipLaunchKernelGGL(wgrad_same_kernel<5>, dim3((unsigned)blocks), dim3(NT), 0, st, geo, d);
        else hipLaunchKernelGGL(wgrad_same_kernel<3>, dim3((unsigned)blocks), dim3(NT), 0, st, geo, d);
        VDNN_LAUNCH_CHECK();
    }
    if (with_bias) {
        const int rc = launch_bias_grad_final(ctx, st, ctx->bias_scratch, bias->out, g.K, d.splits, bias->alpha, bias->accumulate);
        if (rc != VDNN_OK) return rc;
        bias->done = true;
    }
    if (d.splits > 1) return launch_reduce_splits_tap(ctx, st, w, staging, (size_t)M * N, d.splits, alpha, accumulate, g.C, S * S);
    return VDNN_OK;
}
} // namespace vdnn
