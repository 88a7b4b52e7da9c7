// Convolution forward, backward-data and backward-filter as implicit GEMM on fp32 MFMA.
// Replaces cudnnConvolutionForward/AddTensor/BackwardData/BackwardFilter (layer.cu:539-665).
//
// GEMM views (NCHW activations, KCRS filters, cross-correlation):
//   forward      Out[k][(n,p,q)]   = sum_{(c,r,s)} w[k][(c,r,s)]   * x[n,c,p*sh-ph+r,q*sw-pw+s]
//   backward data Out[c][(n,h,w)]  = sum_{(k,r,s)} w[k,c,r,s]      * dy[n,k,(h+ph-r)/sh,(w+pw-s)/sw]
//   backward filter Out[k][(c,r,s)] = sum_{(n,p,q)} dy[n,k,p,q]    * x[n,c,p*sh-ph+r,q*sw-pw+s]
// The im2col operand is never materialised: each thread computes the addresses of its elements
// and the tiles exist only in LDS.
#include "backend_internal.h"
#include "conv_loaders.h"
#include "conv_loaders_tap.h"
#include "mfma_bf16.h"
#include "conv3x3_bf16.h"
#include "conv_launch.h"
#include "wgrad3x3_bf16.h"
#include "wgrad3x3_f32.h"
#include "wgrad3x3_split.h"
#include "conv_smallc.h"
#include "conv_smallc_mfma.h"
#include "winograd_f32.h"
#include "conv_strided.h"
#include "conv_staged.h"
#include <cmath>

namespace vdnn {

static bool geo_from_shape(const vdnn_shape_t* s, ConvGeo& g) {
    g.N = s->n; g.C = s->c; g.H = s->h; g.W = s->w; g.K = s->k; g.R = s->r; g.S = s->s;
    g.ph = s->pad_h; g.pw = s->pad_w; g.sh = s->stride_h; g.sw = s->stride_w;
    if (g.N <= 0 || g.C <= 0 || g.H <= 0 || g.W <= 0 || g.K <= 0 || g.R <= 0 || g.S <= 0) return false;
    if (g.sh <= 0 || g.sw <= 0 || g.ph < 0 || g.pw < 0) return false;
    if (g.R > 16 || g.S > 16) return false;        // tap masks are 16 bits per axis
    if (g.ph >= g.R || g.pw >= g.S) return false;  // padding of a full window or more is not supported
    g.P = vdnn_out_dim(g.H, g.ph, g.R, g.sh);
    g.Q = vdnn_out_dim(g.W, g.pw, g.S, g.sw);
    if (g.P <= 0 || g.Q <= 0) return false;
    const long x_sample = (long)g.C * g.H * g.W, y_sample = (long)g.K * g.P * g.Q;
    // one sample must fit 31 bits of elements; pixel and reduction counts must fit an int
    if (x_sample >= (1l << 29) || y_sample >= (1l << 29)) return false;
    if ((long)g.N * g.P * g.Q >= (1l << 31) || (long)g.N * g.H * g.W >= (1l << 31)) return false;
    if ((long)g.C * g.R * g.S >= (1l << 24) || (long)g.K * g.R * g.S >= (1l << 24)) return false;
    // the filter bank is addressed through one descriptor with summed offsets
    if ((long)g.K * g.C * g.R * g.S * 4 >= (long)MAX_SUM_RANGE) return false;
    return true;
}

// names of the kernel classes in the timing report: {pass}_{tile}
struct PassNames { const char* t64; const char* t128; const char* t64s = ""; };
static const PassNames kFwdNames{"conv_fwd_64x256", "conv_fwd_128x128", "conv_fwd_64x64"};
static const PassNames kBwdDataNames{"conv_bwd_data_64x256", "conv_bwd_data_128x128", "conv_bwd_data_64x64"};
static const PassNames kBwdFilterNames{"conv_bwd_filter_64x256", "conv_bwd_filter_128x128", "conv_bwd_filter_64x64"};
static const PassNames kFwdPackedNames{"conv_fwd_packed_64x256", "conv_fwd_packed_128x128", "conv_fwd_packed_64x64"};
static const PassNames kBwdDataPackedNames{"conv_bwd_data_packed_64x256", "conv_bwd_data_packed_128x128", "conv_bwd_data_packed_64x64"};
static const PassNames kFwdHalfNames{"conv_fwd_bf16mfma_64x256", "conv_fwd_bf16mfma_128x128"};
static const PassNames kBwdDataHalfNames{"conv_bwd_data_bf16mfma_64x256", "conv_bwd_data_bf16mfma_128x128"};
static const PassNames kFwdWin3Names{"conv_fwd_bf16win_64x256", "conv_fwd_bf16win_64x256"};
static const PassNames kBwdDataWin3Names{"conv_bwd_data_bf16win_64x256", "conv_bwd_data_bf16win_64x256"};
static const PassNames kFwdSplitNames{"conv_fwd_split_64x256", "conv_fwd_split_64x256"};
static const PassNames kBwdDataSplitNames{"conv_bwd_data_split_64x256", "conv_bwd_data_split_64x256"};
static const PassNames kBwdFilterHalfNames{"conv_bwd_filter_bf16mfma_64x256", "conv_bwd_filter_bf16mfma_128x128"};
static const PassNames kBwdFilterWin3Names{"conv_bwd_filter_bf16win_64x192", "conv_bwd_filter_bf16win_128x192"};
static const PassNames kBwdFilterRow3Names{"conv_bwd_filter_row_64x192", "conv_bwd_filter_row_128x192"};

// Slices on their way from memory in the float engine: two where the registers hold them without spilling to memory (168, of
// which a gather's address work takes most: dense backward filter and strided backward data keep one). Activations come
// from memory or another die's cache, and three workgroups on a compute unit do not cover that with one slice each. Same
// sums. Forward, one -> two: 32 x 448 x 71 x 71 -> 128 3x3 stride 2 390 -> 372 us, 62 x 128 x 54 x 54 -> 32 216 -> 205,
// 13 x 256 x 137 x 137 -> 640 5150 -> 4975, 16 x 22 x 87 x 208 -> 160 5x5 658 -> 640; both backward passes of the last three
// 352 -> 343, 11800 -> 11670, 1914 -> 1864. The tap by tap backward filter alone: 32 x 128 x 12 x 179 -> 208 backward 668 -> 658.
template <class BL, class EP> struct SlicesAhead { static constexpr int V = 1; };
template <class BL, class E> struct SlicesAhead<BL, StoreNCHW<E>> { static constexpr int V = FetchesAhead<BL>::V ? 2 : 1; };
template <class BL> struct SlicesAhead<BL, StoreFilterTap> { static constexpr int V = 2; };

template <int TM, int TN, class AL, class BL, class EP, bool HALF = false>
static int launch_igemm(vdnn_ctx* ctx, hipStream_t stream, const char* name, const AL& al, const BL& bl, const EP& ep, const GemmDims& d, double flops = 0.0) {
    const long all_tiles = (long)d.mtiles * d.ntiles;
    const long blocks = d.full_tiles > 0 ? d.full_tiles + (all_tiles - d.full_tiles) * d.splits : all_tiles * d.splits;
    if (blocks <= 0 || blocks >= (1l << 31)) { set_error("igemm: grid of %ld workgroups out of range", blocks); return VDNN_EINVAL; }
    // reported work is the algorithmic count where the caller gives one (backward data of a strided or
    // unpadded layer multiplies taps that fall outside the output; they are not counted)
    ProfScope prof(ctx, stream, name, flops > 0.0 ? flops : 2.0 * d.M * (double)d.N * d.K, 0.0);
    if constexpr (HALF) hipLaunchKernelGGL((igemm_bf16_kernel<TM, TN, AL, BL, EP>), dim3((unsigned)blocks), dim3(NT), 0, stream, al, bl, ep, d);
    else if constexpr (TM == 64 && TN == 64) launch_igemm64<EP::TAIL>((unsigned)blocks, stream, al, bl, ep, d); // (forward and backward data)
    else hipLaunchKernelGGL((igemm_kernel<TM, TN, AL, BL, EP, SlicesAhead<BL, EP>::V>), dim3((unsigned)blocks), dim3(NT), 0, stream, al, bl, ep, d);
    VDNN_LAUNCH_CHECK();
    return VDNN_OK;
}

// What a loader's address work costs the 64x64 and the large tile (estimates of mfma_gemm.h), against the loaders whose
// tap is a per-slice value; the others work it out for every element, a strided backward data with two divisions.
// SHORT_OPS: operations up to which a short reduction (kShortReduction) takes the 64x64 tile whatever the estimates say. A
// strided backward data fetches four times as many elements through its divisions there as in a large tile and is bound by
// that once the chip is full: 13 x 213 x 111 x 111, 13 filters of 3x3 at stride 2 216 us against 170, 16 x 600 x 75 x 75, 36 of 2x2 323
// against 251; over 2400 calls the two are even at 3e9 to 6e9 operations.
template <class BL> struct LoadCost { static constexpr double SMALL = 1.25, LARGE = 1.15, SHORT_OPS = 1e30; };
template <int MODE, class E, bool PAD> struct LoadCost<LoadIm2colPixTap<MODE, E, PAD>> { static constexpr double SMALL = 1.0, LARGE = 1.0, SHORT_OPS = 1e30; };
template <bool BIG, class E> struct LoadCost<LoadIm2colPix<2, BIG, E>> { static constexpr double SMALL = 4.0, LARGE = 2.0, SHORT_OPS = 4e9; };

// Forward / backward data. Tile shape by output-row count: 64-row tiles for narrow layers, 128
// otherwise; 64x64 where the estimates of mfma_gemm.h find it faster (float engine). A grid that cannot fill
// the chip (few output pixels: the fully connected layers written as convolutions) splits its reduction; the partial sums go to the staging area and are added in split
// order, with the bias, by a second kernel. The split count depends on the shape only.
// HALF: the bfloat16 engine (32-deep slices); partial_bytes: room behind ep.partial (the context's staging
// area unless part of it is taken by something else).
template <class AL, class BL, class E, bool HALF = false>
static int launch_by_m(vdnn_ctx* ctx, hipStream_t stream, const PassNames& names, const AL& al, const BL& bl, const StoreNCHW<E>& ep, int M, int N, int K, double flops = 0.0,
                       size_t partial_bytes = ~(size_t)0) {
    constexpr int DEPTH = HALF ? KH : KB;
    if (partial_bytes == ~(size_t)0) partial_bytes = ctx->reduce_scratch_bytes;
    const bool narrow = M <= 64;
    const int TM = narrow ? 64 : 128, TN = narrow ? 256 : 128;
    const long tiles = (long)((M + TM - 1) / TM) * ((N + TN - 1) / TN);
    const int splits = ctx->reduce_scratch && ep.partial ? pixel_product_splits(M, N, K, TM, TN, DEPTH, partial_bytes, ctx->num_cu) : 1;
    if constexpr (!HALF) {
        const SmallTilePlan plan = small_tile_plan(M, N, K, ctx->reduce_scratch && ep.partial ? partial_bytes : 0, ctx->num_cu, 4, true, LoadCost<BL>::SMALL);
        const double ops = 2.0 * M * (double)N * K;
        if ((K <= kShortReduction && ops <= LoadCost<BL>::SHORT_OPS) ||
            (ops <= kSmallTileOps && plan.us < 0.9 * large_tile_us(M, N, K, TM, TN, splits, ctx->num_cu, false, LoadCost<BL>::LARGE))) {
            GemmDims ds = make_dims(M, N, K, 64, 64, plan.splits);
            const int tail = plan.full_tiles > 0 && ds.splits > 1 ? (int)((long)ds.mtiles * ds.ntiles - plan.full_tiles) : 0;
            if (tail > 0) ds.full_tiles = (int)plan.full_tiles;
            const bool fused = fuse_split_sums(ctx, stream, ds, partial_bytes);
            const int rcs = launch_igemm<64, 64, AL, BL, StoreNCHW<E>>(ctx, stream, names.t64s, al, bl, ep, ds, flops);
            if (rcs != VDNN_OK || ds.splits == 1 || fused) return rcs;
            if (tail > 0)
                return launch_reduce_tail_nchw(ctx, stream, ep.out, ep.partial, tail, ds.splits, 64, 64, M, N, ds.mtiles, ds.full_tiles, ep.bias, ep.opix, ep.relu, ep.gate);
            return launch_reduce_splits_nchw(ctx, stream, ep.out, ep.partial, (size_t)M * N, ds.splits, ep.bias, ep.opix, M, ep.relu, ep.gate);
        }
    }
    GemmDims d = make_dims(M, N, K, TM, TN, splits, DEPTH);
    // Tail mode: when the tiles make whole rounds of resident workgroups (three per compute unit) plus a
    // small remainder, that remainder would run as a nearly empty last round as long as a full one. Its
    // tiles are split so that together they fill about one round of short workgroups instead.
    const long slots = 3l * ctx->num_cu;
    const long rem = tiles % slots;
    int tail_tiles = 0;
    if (splits == 1 && tiles > slots && rem > 0 && 2 * rem <= slots && ctx->reduce_scratch && ep.partial) {
        long s = slots / rem;
        const long by_depth = (long)K / (8 * DEPTH); // at least eight slices per split
        const long by_mem = (long)(partial_bytes / ((size_t)rem * TM * TN * sizeof(float)));
        if (s > by_depth) s = by_depth;
        if (s > by_mem) s = by_mem;
        if (s >= 2) {
            d = make_dims(M, N, K, TM, TN, (int)s, DEPTH);
            if (d.splits >= 2) { d.full_tiles = (int)(tiles - rem); tail_tiles = (int)rem; }
            else d = make_dims(M, N, K, TM, TN, 1, DEPTH);
        }
    }
    const int rc = narrow ? launch_igemm<64, 256, AL, BL, StoreNCHW<E>, HALF>(ctx, stream, names.t64, al, bl, ep, d, flops)
                          : launch_igemm<128, 128, AL, BL, StoreNCHW<E>, HALF>(ctx, stream, names.t128, al, bl, ep, d, flops);
    if (rc != VDNN_OK || d.splits == 1) return rc;
    if (tail_tiles > 0)
        return launch_reduce_tail_nchw(ctx, stream, ep.out, ep.partial, tail_tiles, d.splits, TM, TN, M, N, d.mtiles, d.full_tiles, ep.bias, ep.opix, ep.relu, ep.gate);
    return launch_reduce_splits_nchw(ctx, stream, ep.out, ep.partial, (size_t)M * N, d.splits, ep.bias, ep.opix, M, ep.relu, ep.gate);
}

// The windowed 3x3 kernel (conv3x3_bf16.h): tiles of 64 rows by 256 pixels, three workgroups resident per compute
// unit (two on float layers, where the kernel holds more registers), the reduction cut at multiples of one filter
// row of a channel block. Splits and tail mode as in launch_by_m. K counts 16-bit values of a row of the filter
// operand (float layers: two per filter element).
constexpr int kWin3SplitPerCU = 2;
template <int MODE, class E, bool PAD = false>
static int launch_win3x3(vdnn_ctx* ctx, hipStream_t stream, const PassNames& names, const LoadPackedH& al, const Win3x3T<E>& geo, const StoreNCHW<E>& ep,
                         int M, int N, int K, double flops, size_t partial_bytes) {
    constexpr bool SPLIT = sizeof(E) == 4;
    const int TM = W3_TM, TN = W3_TN;
    const long tiles = (long)((M + TM - 1) / TM) * ((N + TN - 1) / TN);
    int splits = 1;
    const size_t out_bytes = (size_t)M * N * sizeof(float);
    if (tiles < 2l * ctx->num_cu && ep.partial) {
        long cap = ((long)K + 4 * W3_DEPTH - 1) / (4 * W3_DEPTH); // at least four filter rows per split
        const long by_mem = (long)(partial_bytes / out_bytes);
        if (cap > by_mem) cap = by_mem;
        splits = choose_splits(tiles, K, cap, ctx->num_cu, out_bytes, 2.0 * TM * TN * KB);
    }
    GemmDims d = make_dims(M, N, K, TM, TN, splits, W3_DEPTH);
    const long slots = (SPLIT ? kWin3SplitPerCU : 3l) * ctx->num_cu;
    const long rem = tiles % slots;
    int tail_tiles = 0;
    if (splits == 1 && tiles > slots && rem > 0 && 2 * rem <= slots && ep.partial) {
        long s = slots / rem;
        const long by_depth = (long)K / (4 * W3_DEPTH);
        const long by_mem = (long)(partial_bytes / ((size_t)rem * TM * TN * sizeof(float)));
        if (s > by_depth) s = by_depth;
        if (s > by_mem) s = by_mem;
        if (s >= 2) {
            d = make_dims(M, N, K, TM, TN, (int)s, W3_DEPTH);
            if (d.splits >= 2) { d.full_tiles = (int)(tiles - rem); tail_tiles = (int)rem; }
            else d = make_dims(M, N, K, TM, TN, 1, W3_DEPTH);
        }
    }
    const long all_tiles = (long)d.mtiles * d.ntiles;
    const long blocks = d.full_tiles > 0 ? d.full_tiles + (all_tiles - d.full_tiles) * d.splits : all_tiles * d.splits;
    if (blocks <= 0 || blocks >= (1l << 31)) { set_error("conv3x3: grid of %ld workgroups out of range", blocks); return VDNN_EINVAL; }
    {
        ProfScope prof(ctx, stream, names.t64, flops, 0.0);
        hipLaunchKernelGGL((conv3x3_bf16_kernel<MODE, E, SPLIT ? kWin3SplitPerCU : 3, PAD>), dim3((unsigned)blocks), dim3(NT), 0, stream, al, geo, ep, d);
        VDNN_LAUNCH_CHECK();
    }
    if (d.splits == 1) return VDNN_OK;
    if (tail_tiles > 0)
        return launch_reduce_tail_nchw(ctx, stream, ep.out, ep.partial, tail_tiles, d.splits, TM, TN, M, N, d.mtiles, d.full_tiles, ep.bias, ep.opix, ep.relu, ep.gate);
    return launch_reduce_splits_nchw(ctx, stream, ep.out, ep.partial, (size_t)M * N, d.splits, ep.bias, ep.opix, M, ep.relu, ep.gate);
}

// what the windowed kernel needs: a 3x3 window at stride 1 with one pixel of padding (input and output planes of
// one extent), rows of an even number of pixels, and tiles whose samples fit one descriptor
static bool win3x3_ok(const int R, const int S, int ph, int pw, int sh, int sw, int Hs, int Ws, int OH, int OW, long sample_elems, int elem_bytes = 2) {
    return R == 3 && S == 3 && ph == 1 && pw == 1 && sh == 1 && sw == 1 && Hs == OH && Ws == OW && Ws % 2 == 0 && Ws >= 2 &&
           pixel_tile_span_ok(sample_elems, OH * OW, W3_TN, elem_bytes);
}

// forward with the given A loader (128-bit or 32-bit filter loads)
template <class AL, class E>
static int conv_fwd_with(vdnn_ctx* ctx, hipStream_t st, const ConvGeo& g, const AL& al, const E* x, const float* bias, E* y, int relu) {
    StoreNCHW<E> ep{y, bias, g.P * g.Q, ctx->reduce_scratch, relu, nullptr};
    const int M = g.K, N = g.N * g.P * g.Q, K = g.C * g.R * g.S;
    const FastDiv dRS = FastDiv::make(g.R * g.S), dS = FastDiv::make(g.S);
    if (g.R * g.S <= 32) {
        LoadIm2colPix<0, false, E> bl{x, g.H, g.W, g.P, g.Q, g.R, g.S, g.ph, g.pw, g.sh, g.sw, (long)g.C * g.H * g.W, g.N, dRS, dS};
        return launch_by_m(ctx, st, kFwdNames, al, bl, ep, M, N, K);
    }
    LoadIm2colPix<0, true, E> bl{x, g.H, g.W, g.P, g.Q, g.R, g.S, g.ph, g.pw, g.sh, g.sw, (long)g.C * g.H * g.W, g.N, dRS, dS};
    return launch_by_m(ctx, st, kFwdNames, al, bl, ep, M, N, K);
}

template <class AL, class BL>
static int conv_wgrad_with(vdnn_ctx* ctx, hipStream_t st, const AL& al, const BL& bl, const StoreDense<float>& ep, const GemmDims& d, bool narrow, bool small) {
    if (small) return launch_igemm<64, 64>(ctx, st, kBwdFilterNames.t64s, al, bl, ep, d);
    return narrow ? launch_igemm<64, 256>(ctx, st, kBwdFilterNames.t64, al, bl, ep, d)
                  : launch_igemm<128, 128>(ctx, st, kBwdFilterNames.t128, al, bl, ep, d);
}

// NTAP: taps that share a 64x64 tile's columns
template <int NTAP, class E>
static int launch_wgrad_tap_small(vdnn_ctx* ctx, hipStream_t st, const ConvGeo& g, const LoadDyRedInc<E>& al, const E* x, const StoreFilterTap& ep, const GemmDims& d, FastDiv dS) {
    const LoadIm2colRedTap<NTAP, E> bl{x, g.N, g.C, g.H, g.W, g.R, g.S, g.P, g.Q, g.ph, g.pw, g.sh, g.sw, d.N, d.kchunk, d.K, FastDiv::make(g.C), dS};
    return launch_igemm<64, 64>(ctx, st, kBwdFilterNames.t64s, al, bl, ep, d);
}

constexpr size_t kMaxWgradWorkspace = (size_t)256 << 20;

// A window that covers the whole unpadded input (the fully connected layers OverFeat writes as
// convolutions, network.cu:449-481) is a dense GEMM over (c,h,w): the implicit-GEMM backward data would
// spend R*S times the work on taps that fall outside the single output pixel.
static bool is_dense(const ConvGeo& g) { return g.P == 1 && g.Q == 1 && g.ph == 0 && g.pw == 0 && g.R == g.H && g.S == g.W; }

// Channel counts that are no whole blocks of 16 take the tap-major loaders with the last block padded where that multiplies at
// most a quarter more and the layer is large enough: the others work out a tap per element, at half the rate in large grids
// (32 x 200 x 28 x 28, 300 of 3x3 forward 356 -> 275 us; 64 x 130 x 13 x 13, 390 of 5x5 backward data 460 -> 352; 21 x 70 x 53 x 37, 130 of 3x3
// forward 151 -> 121), but need no launch for a re-laid-out filter (1 x 46 x 29 x 29, 48 of 2x2 forward 13.1 with it, 8.5 without). The
// lines, operations with the rows in whole tiles, are those of least loss over 1200 calls timed on both: 1.2 % and 0.7 %
// behind the better one in the mean.
static bool pad_pays(int channels, int M, long N, int RS, double least_ops) {
    return 4 * ((channels + KB - 1) / KB * KB) <= 5 * channels && 2.0 * ((M + 63) / 64 * 64) * (double)N * channels * RS >= least_ops;
}
// A filter re-laid-out for the tap-major loaders costs a launch and saves three of four loads of it; small layers read it as it lies (19 x 32 x 7 x 7, 13
// filters of 3x3 forward 11.1 -> 8.9 us; 15 x 16 x 17 x 17, 176 of 5x5, 3.6e8 operations, re-laid-out 14.9, else 19.4). As it lies, the elements of a tap are
// a window apart, so that the line falls with the taps. Over 5727 drawn calls timed both ways, windows of 2x2 to 5x5, the choice is 0.3 % behind the better
// way in the mean and 5 % in 44 (one line for all windows at 3e8 operations: 0.6 %, 145).
constexpr double kPackOps = 4e9;
static bool pack_pays(double ops, int taps) { return ops * taps >= kPackOps; }
constexpr double kPadFwdOps = 1.5e9, kPadBwdDataOps = 4e8;
static bool packed_fwd_ok(const ConvGeo& g) { return g.R * g.S <= 32 && g.C % KB == 0; }
static bool packed_bwd_data_ok(const ConvGeo& g) {
    return g.C > 4 && g.sh == 1 && g.sw == 1 && g.R * g.S <= 32 && g.K % KB == 0;
}

// ---- Winograd F(4x4, 3x3): the perf-optimal mode's forward / backward data of wide 3x3 layers (winograd_f32.h) -----
// Samples are processed in chunks so that the transformed input V and the transformed output M of a chunk stay
// within g_wino_chunk_bytes (512 MiB unless vdnn_conv_winograd_chunk_bytes says otherwise; and each below 2 GiB, the range of the product's descriptors). The plan depends on the shape
// alone: vdnn_conv_workspace_bytes reports it, the pass follows it.
constexpr size_t kWinoChunkBytesDefault = (size_t)512 << 20;
static size_t g_wino_chunk_bytes = kWinoChunkBytesDefault; // vdnn_conv_winograd_chunk_bytes
constexpr int kWinoMinReduced = 128;  // reduced channels from which the product's short reduction pays
struct WinoPlan {
    int rows, cred;        // output rows of the product (forward: K, backward data: C) and its reduction (C / K)
    int th, tw, per;       // tiles per column, per row, per sample
    int nc, chunks;        // samples per chunk, chunks
    long Tpad;             // columns per xi of a full chunk
    size_t u_bytes, v_bytes, m_bytes, total;
};
static bool wino_ok(const ConvGeo& g, bool bwd) {
    const int rows = bwd ? g.C : g.K, cred = bwd ? g.K : g.C;
    return g.R == 3 && g.S == 3 && g.ph == 1 && g.pw == 1 && g.sh == 1 && g.sw == 1 && g.P == g.H && g.Q == g.W &&
           cred >= kWinoMinReduced && cred % KB == 0 && rows > 64 && g.H >= 4 && g.W >= 4;
}
static WinoPlan wino_plan(const ConvGeo& g, bool bwd) {
    WinoPlan p;
    p.rows = bwd ? g.C : g.K; p.cred = bwd ? g.K : g.C;
    p.th = (g.H + 3) / 4; p.tw = (g.W + 3) / 4; p.per = p.th * p.tw;
    const size_t per_sample = (size_t)(p.rows + p.cred) * WINO_XI * p.per * sizeof(float);
    long most = (long)(g_wino_chunk_bytes / per_sample);
    if (most < 1) most = 1;
    if (most > g.N) most = g.N;
    p.chunks = (int)((g.N + most - 1) / most);
    p.nc = (g.N + p.chunks - 1) / p.chunks;
    p.Tpad = ((long)p.nc * p.per + WINO_TN - 1) / WINO_TN * WINO_TN;
    auto up = [](size_t b) { return (b + 255) / 256 * 256; };
    p.u_bytes = up((size_t)WINO_XI * p.rows * p.cred * sizeof(float));
    p.v_bytes = up((size_t)p.cred * WINO_XI * p.Tpad * sizeof(float));
    p.m_bytes = up((size_t)p.rows * WINO_XI * p.Tpad * sizeof(float));
    p.total = p.u_bytes + p.v_bytes + p.m_bytes;
    return p;
}
static bool wino_plan_ok(const WinoPlan& p) {
    return p.v_bytes < 0x7FFF0000ul && p.m_bytes < 0x7FFF0000ul && (long)WINO_XI * p.Tpad < (1l << 31) && p.rows <= 65535 && p.cred <= 65535;
}

// in: x (forward) or dy (backward data); out: y or dx. Returns VDNN_OK with *taken false when the shape or the
// workspace does not allow the variant.
static int launch_winograd(vdnn_ctx* ctx, hipStream_t st, const ConvGeo& g, bool bwd, const float* in, const float* w, const float* bias, float* out,
                           int relu, const float* gate, void* workspace, size_t workspace_bytes, bool* taken) {
    *taken = false;
    if (!wino_ok(g, bwd) || !workspace || !aligned16(workspace)) return VDNN_OK;
    const WinoPlan p = wino_plan(g, bwd);
    if (!wino_plan_ok(p) || workspace_bytes < p.total) return VDNN_OK;
    *taken = true;
    float* U = (float*)workspace;
    float* V = (float*)((char*)workspace + p.u_bytes);
    float* Mo = (float*)((char*)workspace + p.u_bytes + p.v_bytes);
    {
        const long total = (long)p.rows * p.cred;
        ProfScope prof(ctx, st, "conv_wino_filter", 0.0, (9.0 + WINO_XI) * 4.0 * (double)total);
        if (bwd) hipLaunchKernelGGL(wino_filter_kernel<true>, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, w, U, p.rows, p.cred);
        else hipLaunchKernelGGL(wino_filter_kernel<false>, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, w, U, p.rows, p.cred);
        VDNN_LAUNCH_CHECK();
    }
    const long plane = (long)g.H * g.W;
    const bool vec = g.W % 4 == 0 && aligned16(in) && aligned16(out) && (!gate || aligned16(gate));
    for (int n0 = 0; n0 < g.N; n0 += p.nc) {
        const int nc = g.N - n0 < p.nc ? g.N - n0 : p.nc;
        const int T = nc * p.per;
        const long Tpad = ((long)T + WINO_TN - 1) / WINO_TN * WINO_TN;
        const unsigned tblocks = (unsigned)((T + 255) / 256), pblocks = (unsigned)((Tpad + 255) / 256);
        {
            const WinoTiles ti{g.H, g.W, p.th, p.tw, p.cred, T, Tpad};
            ProfScope prof(ctx, st, bwd ? "conv_bwd_data_wino_in" : "conv_fwd_wino_in", 0.0, 4.0 * ((double)nc * p.cred * plane + (double)p.cred * WINO_XI * T));
            const float* src = in + (long)n0 * p.cred * plane;
            if (vec) hipLaunchKernelGGL(wino_input_kernel<true>, dim3(pblocks, (unsigned)p.cred), dim3(256), 0, st, src, V, ti);
            else hipLaunchKernelGGL(wino_input_kernel<false>, dim3(pblocks, (unsigned)p.cred), dim3(256), 0, st, src, V, ti);
            VDNN_LAUNCH_CHECK();
        }
        {
            // several column tiles per workgroup, so that all workgroups make about one round of resident ones
            const int mtiles = (p.rows + 127) / 128, tiles_per_xi = (int)(Tpad / WINO_TN);
            const long all_tiles = (long)WINO_XI * mtiles * tiles_per_xi, slots = 3l * ctx->num_cu;
            int group = (int)((all_tiles + slots - 1) / slots);
            // ... unless that round would leave more than a seventh of the places idle (few tiles: 14 x 14 planes,
            // 256 produced rows at 28 x 28): single tiles then, which the hardware hands out as places come free
            if (20 * all_tiles < 17 * (long)group * slots) group = 1;
            if (group < 1) group = 1;
            if (group > tiles_per_xi) group = tiles_per_xi;
            const int groups_per_xi = (tiles_per_xi + group - 1) / group;
            const WinoGemm gm{U, V, Mo, p.rows, p.cred, Tpad, mtiles, tiles_per_xi, group, groups_per_xi};
            // work counted in the transformed domain: 36 products per 4x4 outputs and channel pair
            ProfScope prof(ctx, st, bwd ? "conv_bwd_data_wino_gemm" : "conv_fwd_wino_gemm", 2.0 * p.rows * (double)p.cred * WINO_XI * T, 0.0);
            hipLaunchKernelGGL(wino_gemm_kernel, dim3((unsigned)(WINO_XI * mtiles * groups_per_xi)), dim3(NT), 0, st, gm);
            VDNN_LAUNCH_CHECK();
        }
        {
            const WinoTiles to{g.H, g.W, p.th, p.tw, p.rows, T, Tpad};
            ProfScope prof(ctx, st, bwd ? "conv_bwd_data_wino_out" : "conv_fwd_wino_out", 0.0,
                           4.0 * ((double)p.rows * WINO_XI * T + (double)nc * p.rows * plane * (gate ? 2.0 : 1.0)));
            const long off = (long)n0 * p.rows * plane;
            if (vec) hipLaunchKernelGGL(wino_output_kernel<true>, dim3(tblocks, (unsigned)p.rows), dim3(256), 0, st, Mo, out + off, bias, gate ? gate + off : nullptr, relu, to);
            else hipLaunchKernelGGL(wino_output_kernel<false>, dim3(tblocks, (unsigned)p.rows), dim3(256), 0, st, Mo, out + off, bias, gate ? gate + off : nullptr, relu, to);
            VDNN_LAUNCH_CHECK();
        }
    }
    return VDNN_OK;
}

// Backward filter as Winograd F(3x3, 4x4) (winograd_f32.h): per chunk of samples the transformed input V and the
// transformed output gradient D, then one launch of the tile engine for the 36 products S_xi = D_xi V_xi^t with the
// reduction over the chunk's tiles split so that the grid fills the chip; every (chunk, split) leaves one partial
// result, and a last kernel adds them in order, transforms back and applies alpha. The plan depends on the shape alone.
constexpr size_t kWinoWgradPartialBytes = (size_t)256 << 20;
struct WinoWgradPlan {
    int th, tw, per, nc, chunks, splits;
    long Tpad;
    size_t v_bytes, d_bytes, part_bytes, total;   // part_bytes: one partial result
};
static bool wino_wgrad_ok(const ConvGeo& g) {
    return g.R == 3 && g.S == 3 && g.ph == 1 && g.pw == 1 && g.sh == 1 && g.sw == 1 && g.P == g.H && g.Q == g.W &&
           g.C >= 128 && g.C % 128 == 0 && g.K > 64 && g.H >= 4 && g.W >= 4;
}
static WinoWgradPlan wino_wgrad_plan(const ConvGeo& g) {
    WinoWgradPlan p;
    p.th = (g.H + 3) / 4; p.tw = (g.W + 3) / 4; p.per = p.th * p.tw;
    const size_t per_sample = (size_t)(g.K + g.C) * WINO_XI * p.per * sizeof(float);
    long most = (long)(g_wino_chunk_bytes / per_sample);
    if (most < 1) most = 1;
    if (most > g.N) most = g.N;
    p.chunks = (int)((g.N + most - 1) / most);
    p.nc = (g.N + p.chunks - 1) / p.chunks;
    p.chunks = (g.N + p.nc - 1) / p.nc;
    p.Tpad = ((long)p.nc * p.per + WINO_TN - 1) / WINO_TN * WINO_TN;
    auto up = [](size_t b) { return (b + 255) / 256 * 256; };
    p.v_bytes = up((size_t)g.C * WINO_XI * p.Tpad * sizeof(float));
    p.d_bytes = up((size_t)g.K * WINO_XI * p.Tpad * sizeof(float));
    p.part_bytes = up((size_t)g.K * WINO_XI * g.C * sizeof(float));
    // splits of a chunk's reduction: one round of resident workgroups, at least eight slices each, partial results within their budget
    const long tiles = (long)WINO_XI * ((g.K + 127) / 128) * (g.C / 128);
    long splits = 3l * kPlanningCUs / tiles;
    const long by_len = p.Tpad / (8 * KB), by_mem = (long)(kWinoWgradPartialBytes / p.part_bytes) / p.chunks;
    if (splits > by_len) splits = by_len;
    if (splits > by_mem) splits = by_mem;
    if (splits < 1) splits = 1;
    // (the launch re-derives the split count from the chunk size through make_dims; this is its upper bound)
    p.splits = (int)splits;
    p.total = p.v_bytes + p.d_bytes + (size_t)p.chunks * p.splits * p.part_bytes;
    return p;
}
static bool wino_wgrad_plan_ok(const WinoWgradPlan& p, const ConvGeo& g) {
    return p.v_bytes < 0x7FFF0000ul && p.d_bytes < 0x7FFF0000ul && (long)WINO_XI * g.C < (1l << 24) && g.K <= 65535 && g.C <= 65535 &&
           (long)p.chunks * p.splits < 4096;
}

static int launch_winograd_wgrad(vdnn_ctx* ctx, hipStream_t st, const ConvGeo& g, const float* x, const float* dy, float* w, float alpha, int accumulate,
                                 void* workspace, size_t workspace_bytes, bool* taken, BiasOut* bias) {
    *taken = false;
    if (!wino_wgrad_ok(g) || !workspace || !aligned16(workspace)) return VDNN_OK;
    const WinoWgradPlan p = wino_wgrad_plan(g);
    if (!wino_wgrad_plan_ok(p, g) || workspace_bytes < p.total) return VDNN_OK;
    *taken = true;
    float* V = (float*)workspace;
    float* D = (float*)((char*)workspace + p.v_bytes);
    float* P = (float*)((char*)workspace + p.v_bytes + p.d_bytes);
    const long part_stride = (long)(p.part_bytes / sizeof(float));
    const long plane = (long)g.H * g.W;
    const bool vec = g.W % 4 == 0 && aligned16(x) && aligned16(dy);
    int nparts = 0;
    // the bias gradient: every workgroup of the dy transform leaves the sum of the values it read
    long bias_parts = 0;
    for (int n0 = 0; n0 < g.N; n0 += p.nc) {
        const int nc = g.N - n0 < p.nc ? g.N - n0 : p.nc;
        bias_parts += (((long)nc * p.per + WINO_TN - 1) / WINO_TN * WINO_TN + 255) / 256;
    }
    const bool with_bias = bias && bias->wanted() && bias_parts < (1 << 20) && bias_parts_fit(ctx, g.K, bias_parts);
    int bias_first = 0;
    for (int n0 = 0; n0 < g.N; n0 += p.nc) {
        const int nc = g.N - n0 < p.nc ? g.N - n0 : p.nc;
        const int T = nc * p.per;
        const long Tpad = ((long)T + WINO_TN - 1) / WINO_TN * WINO_TN;
        const unsigned pblocks = (unsigned)((Tpad + 255) / 256);
        {
            const WinoTiles ti{g.H, g.W, p.th, p.tw, g.C, T, Tpad};
            ProfScope prof(ctx, st, "conv_bwd_filter_wino_in", 0.0, 4.0 * ((double)nc * g.C * plane + (double)g.C * WINO_XI * Tpad));
            const float* src = x + (long)n0 * g.C * plane;
            if (vec) hipLaunchKernelGGL(wino_input_kernel<true>, dim3(pblocks, (unsigned)g.C), dim3(256), 0, st, src, V, ti);
            else hipLaunchKernelGGL(wino_input_kernel<false>, dim3(pblocks, (unsigned)g.C), dim3(256), 0, st, src, V, ti);
            VDNN_LAUNCH_CHECK();
        }
        {
            const WinoTiles td{g.H, g.W, p.th, p.tw, g.K, T, Tpad};
            ProfScope prof(ctx, st, "conv_bwd_filter_wino_dy", 0.0, 4.0 * ((double)nc * g.K * plane + (double)g.K * WINO_XI * Tpad));
            const float* src = dy + (long)n0 * g.K * plane;
            float* bp = with_bias ? ctx->bias_scratch : nullptr;
            if (vec && with_bias) hipLaunchKernelGGL((wino_dy_kernel<true, true>), dim3(pblocks, (unsigned)g.K), dim3(256), 0, st, src, D, td, bp, (int)bias_parts, bias_first);
            else if (vec) hipLaunchKernelGGL((wino_dy_kernel<true, false>), dim3(pblocks, (unsigned)g.K), dim3(256), 0, st, src, D, td, bp, 0, 0);
            else if (with_bias) hipLaunchKernelGGL((wino_dy_kernel<false, true>), dim3(pblocks, (unsigned)g.K), dim3(256), 0, st, src, D, td, bp, (int)bias_parts, bias_first);
            else hipLaunchKernelGGL((wino_dy_kernel<false, false>), dim3(pblocks, (unsigned)g.K), dim3(256), 0, st, src, D, td, bp, 0, 0);
            VDNN_LAUNCH_CHECK();
            bias_first += (int)pblocks;
        }
        {
            GemmDims d = make_dims(g.K, WINO_XI * g.C, (int)Tpad, 128, WINO_TN, p.splits);
            LoadWinoRed<true> al{D, Tpad, g.K, (unsigned)((size_t)g.K * WINO_XI * Tpad * sizeof(float)), g.C, d.mtiles, d.mtiles * d.ntiles, WINO_TN};
            LoadWinoRed<false> bl{V, Tpad, g.C, (unsigned)((size_t)g.C * WINO_XI * Tpad * sizeof(float)), g.C, d.mtiles, d.mtiles * d.ntiles, WINO_TN};
            float* slot = P + (long)nparts * part_stride;
            StoreDense<float> ep{slot, slot, nullptr, (long)WINO_XI * g.C, part_stride, 1.0f, 0, 0, nullptr};
            const int rc = launch_igemm<128, WINO_TN>(ctx, st, "conv_bwd_filter_wino_gemm", al, bl, ep, d, 2.0 * g.K * (double)g.C * WINO_XI * T);
            if (rc != VDNN_OK) return rc;
            nparts += d.splits;
        }
    }
    {
        const long total = (long)g.K * g.C, count = total * WINO_XI;
        ProfScope prof(ctx, st, "conv_bwd_filter_wino_out", 0.0, 4.0 * ((double)nparts * WINO_XI + 18.0) * (double)total);
        if (nparts > 2) {
            // many partial results: summed with one thread per element first
            hipLaunchKernelGGL(wino_wgrad_sum_kernel, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, st, P, part_stride, nparts, count);
            VDNN_LAUNCH_CHECK();
            nparts = 1;
        }
        hipLaunchKernelGGL(wino_wgrad_out_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, P, part_stride, nparts, w, g.K, g.C, g.C, alpha, accumulate);
        VDNN_LAUNCH_CHECK();
    }
    if (with_bias) {
        const int rc = launch_bias_grad_final(ctx, st, ctx->bias_scratch, bias->out, g.K, (int)bias_parts, bias->alpha, bias->accumulate);
        if (rc != VDNN_OK) return rc;
        bias->done = true;
    }
    return VDNN_OK;
}

// The bfloat16 engine's kernels for a geometry: the windowed one (one staged window per filter row serves the three taps of a
// 3x3 at stride 1 with padding 1), a pixel pair per lane where the pairs of an output row are contiguous in the input, or a
// pixel per lane.
enum class HalfKernel { WINDOWED, PAIRS, SINGLE };
template <int MODE>
static HalfKernel half_kernel(const LoadIm2colPix<MODE, false, bf16_t>& pix) {
    if (win3x3_ok(pix.R, pix.S, pix.ph, pix.pw, pix.sh, pix.sw, pix.Hs, pix.Ws, pix.OH, pix.OW, pix.sample_elems)) return HalfKernel::WINDOWED;
    const bool pairs = pix.OW % 2 == 0 && pix.S <= 16 && pix.Ws >= pix.S && pix.Ws > pix.pw + 1 && (MODE == 1 || pix.sw == 1);
    return pairs ? HalfKernel::PAIRS : HalfKernel::SINGLE;
}

// Channels that are no whole blocks of 32 are padded with zeros in the filter operand and not fetched in the other one: from
// twelve channels on, where the layer is large enough. This engine has tiles of 128x128 and 64x256 only; on a grid that such
// tiles leave mostly idle the float engine's 64x64 ones are faster, although it multiplies at a sixteenth of the rate (8 x 12 x 4
// x 4, 64 filters of 1x1 forward 18.8 us here, 7.8 there; 11 x 57 x 5 x 5, 45 of 2x2 backward data 35.7 and 12.4). The lines
// are those of least loss over 3200 calls of 12 to 600 channels, timed on both: operations, with few rows counting for more
// (a tile has 64 of them whatever the layer has). By them the choice is 1.2 % behind the better route's time in the mean; with
// this engine for all of them it was 15 % behind.
// 32 x 200 x 28 x 28, 300 filters of 3x3 forward 364 -> 48 us, backward data 338 -> 72; 64 x 130 x 13 x 13, 390 of 5x5 347 -> 127
// and 468 -> 147; 16 x 12 x 112 x 112, 20 of 3x3 55 -> 25 and 83 -> 24.
constexpr int kHalfMinChannels = 12;
static bool half_pad_pays(HalfKernel kernel, int rows, long N, int reduced_channels, int RS) {
    const double weighed = 2.0 * N * (double)reduced_channels * RS * std::sqrt(64.0 * rows);
    if (kernel == HalfKernel::WINDOWED) return weighed >= 1e8;
    return reduced_channels * RS > KH && weighed >= (kernel == HalfKernel::PAIRS ? 3e8 : 4e8);
}

// The bfloat16 engine's filter operand lives at the front of the staging area (rounded and re-laid-out by a
// small kernel before every use: the master copy changes every step); what is left holds partial sums.
template <int MODE>
static bool half_engine_ok(const vdnn_ctx* ctx, const LoadIm2colPix<MODE, false, bf16_t>& pix, int reduced_channels, int rows, int RS) {
    if (RS > 32 || !ctx->reduce_scratch) return false;
    const size_t elems = (size_t)rows * RS * reduced_channels, padded = (size_t)rows * RS * ((reduced_channels + KH - 1) / KH * KH);
    if (padded * 2 + (16u << 20) > ctx->reduce_scratch_bytes || padded * 2 >= 0x7FFF0000ul) return false;
    if (reduced_channels % KH == 0) return true;
    // (a filter too large for the float route's rounded copy stays refused)
    return reduced_channels >= kHalfMinChannels && elems * 4 + (8u << 20) <= ctx->reduce_scratch_bytes &&
           half_pad_pays(half_kernel(pix), rows, (long)pix.nsamples * pix.OH * pix.OW, reduced_channels, RS);
}

static int launch_pack_filter_bf16(vdnn_ctx* ctx, hipStream_t st, const float* w, unsigned short* packed, int rows, int Cred, int RS,
                                   int row_stride, int red_stride) {
    const int Cpad = (Cred + KH - 1) / KH * KH;
    const long total = (long)rows * Cpad * RS;
    ProfScope prof(ctx, st, "conv_pack_filter", 0.0, 6.0 * (double)total);
    hipLaunchKernelGGL(pack_filter_tap_bf16_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, w, packed, rows, Cred, Cpad, RS,
                       row_stride, red_stride, total);
    VDNN_LAUNCH_CHECK();
    return VDNN_OK;
}

__global__ void __launch_bounds__(256) round_filter_bf16_kernel(const float* __restrict__ w, float* __restrict__ out, long count) {
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i < count) out[i] = round_to_bf16_value(w[i]);
}

// Layers with bfloat16 activations multiply the filter rounded to bfloat16 (two bfloat16 factors per product)
// on every route. Routes outside the bfloat16 engine read a rounded float copy, made here at the front of the
// staging area. Returns null when it does not fit.
static const float* rounded_filter_copy(vdnn_ctx* ctx, hipStream_t st, StagingCarve& carve, const float* w, size_t count) {
    if (!ctx->reduce_scratch || count * sizeof(float) + (8u << 20) > ctx->reduce_scratch_bytes) return nullptr;
    float* wr = (float*)carve.take(count * sizeof(float));
    hipLaunchKernelGGL(round_filter_bf16_kernel, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, st, w, wr, (long)count);
    return wr;
}

// Forward (MODE 0) and backward data at stride 1 (MODE 1) from a copy of the source in `scratch` (conv_staged.h). al: the filter bank; K: its row.
// Where the copy fits there at once: a large source is read from memory again tap by tap (43 x 304 x 131 x 131, 64 of 3x3 forward 664 us, 837
// from a copy in nine parts; 118 x 64 x 131 x 131, 82 of 5x5 1048, 1090), and a 1x1 window reads it once anyway (6 x 64 x 105 x 105, 704 of
// 1x1 41, 44). Where the copy's trip through memory is less than what it saves of the product, rows in whole blocks of 64 and channels in
// whole blocks of 32, as both ways multiply them: much of a product that fetches single values, little of one that fetches pairs, and less the
// fewer the taps. And where the splits that the room behind the copy leaves take at most twice the rounds' time of those there would be
// without it (24 x 608 x 45 x 45, 80 of 5x5 at stride 2 forward, a hundred tiles, five splits before and one behind 59 MB: 137 us, 242). Of 260 drawn calls
// with less than half of their splits left, timed both ways, 222 take the copy: 1.1 % behind the faster way in the mean, 18 calls by more than 5 %,
// at most 1.3 times its time (by a fifth of the splits 1.4 %, 20, 1.8 times; by a third 5.5 %, 50, 1.9 times).
// Of 9494 drawn calls of 2x2 to 7x7 whose copy fits, timed both ways, 3704 took the copy by a fifth of the splits: 1.2 times as fast in the mean, 63 of
// them more than 5 % slower. By the operations alone, half of every product saved, 3668 did, 188 of them slower, by up to 1.8 times (2 x 255 x 120 x 218, 3 of
// 3x3 forward 44, 52; 27 x 347 x 78 x 78, 80 of 2x2 gated 115, 156); with a part block of channels counted as it is stored, calls that gain were left
// (93 x 16 x 38 x 38, 16 of 5x5 backward data 36, 50 without).
template <int MODE>
static int launch_staged(vdnn_ctx* ctx, hipStream_t st, const PassNames& names, const LoadPackedH& al, int K, int rows, int Cred,
                         const LoadIm2colPix<MODE, false, bf16_t>& pix, bool pairs, StoreNCHW<bf16_t> ep, double flops, char* scratch, size_t scratch_bytes, bool* taken) {
    *taken = false;
    const int blocks = (Cred + KH - 1) / KH, RS = pix.R * pix.S, opix = pix.OH * pix.OW;
    const long pixels = (long)pix.nsamples * pix.Hs * pix.Ws, N = (long)pix.nsamples * opix;
    // (the loader's descriptor starts ahead of the copy by less than the filter's rows and columns of pixels)
    const size_t lead = ((size_t)(pix.R * pix.Ws + pix.S) * blocks * 64 + 255) / 256 * 256, copy_bytes = ((size_t)pixels * blocks * 64 + 255) / 256 * 256;
    const double us = 2.0 * ((rows + 63) / 64 * 64) * (double)N * (blocks * KH) * RS / 350e6, copy_us = (double)pixels * (Cred + blocks * KH) * 2 / 3.5e6 + 4.0;
    const double saved = pairs ? (RS >= 16 ? 0.35 : RS >= 9 ? 0.1 : 0.0) : RS >= 16 ? 0.65 : RS >= 9 ? 0.5 : 0.2;
    if (RS == 1 || lead + copy_bytes > scratch_bytes || saved * us <= copy_us) return VDNN_OK;
    const int TM = rows <= 64 ? 64 : 128, TN = rows <= 64 ? 256 : 128;
    const size_t room = scratch_bytes - lead - copy_bytes;
    const long tiles = (long)((rows + TM - 1) / TM) * ((N + TN - 1) / TN);
    const int whole = pixel_product_splits(rows, (int)N, K, TM, TN, KH, scratch_bytes, ctx->num_cu), behind = pixel_product_splits(rows, (int)N, K, TM, TN, KH, room, ctx->num_cu);
    if (split_rounds_us(tiles, K, behind, ctx->num_cu, 1.0) > 2.0 * split_rounds_us(tiles, K, whole, ctx->num_cu, 1.0)) return VDNN_OK;
    *taken = true;
    unsigned short* copy = (unsigned short*)(scratch + lead);
    ep.partial = (float*)(scratch + lead + copy_bytes);
    {
        ProfScope prof(ctx, st, "conv_stage_pixels", 0.0, 4.0 * (double)pixels * Cred);
        hipLaunchKernelGGL(stage_pixels_kernel, dim3((unsigned)((pixels + 255) / 256), (unsigned)blocks), dim3(256), 0, st, pix.src, copy, Cred, pix.Hs * pix.Ws, (int)pixels, blocks);
        VDNN_LAUNCH_CHECK();
    }
    constexpr bool MIRROR = MODE == 1;
    const LoadPixStaged<MIRROR> bl{copy, pix.Hs, pix.Ws, pix.OH, pix.OW, pix.R, pix.S, MIRROR ? pix.R - 1 - pix.ph : pix.ph, MIRROR ? pix.S - 1 - pix.pw : pix.pw,
                                   MIRROR ? 1 : pix.sh, MIRROR ? 1 : pix.sw, blocks * KH, pix.nsamples, FastDiv::make(RS), FastDiv::make(pix.S)};
    return launch_by_m<LoadPackedH, LoadPixStaged<MIRROR>, bf16_t, true>(ctx, st, names, al, bl, ep, rows, (int)N, K, flops, room);
}

// forward / backward data of a bfloat16 layer on the bfloat16 matrix cores; MODE as in LoadIm2colPixTapH, PAD: Cred is no
// multiple of 32
template <int MODE, bool PAD>
static int conv_half_engine_with(vdnn_ctx* ctx, hipStream_t st, const PassNames& names, const float* w, int rows, int Cred, int RS, int row_stride, int red_stride,
                                 const LoadIm2colPix<MODE, false, bf16_t>& pix, StoreNCHW<bf16_t> ep, int N, double flops) {
    const int K = (Cred + KH - 1) / KH * KH * RS;
    const size_t filter_elems = (size_t)rows * K;
    unsigned short* packed = (unsigned short*)ctx->reduce_scratch;
    const size_t taken = (filter_elems * 2 + 255) / 256 * 256, left = ctx->reduce_scratch_bytes - taken;
    const int rc = launch_pack_filter_bf16(ctx, st, w, packed, rows, Cred, RS, row_stride, red_stride);
    if (rc != VDNN_OK) return rc;
    ep.partial = (float*)((char*)ctx->reduce_scratch + taken);
    LoadPackedH al{packed, (long)K, rows, (unsigned)(filter_elems * 2)};
    const HalfKernel kernel = half_kernel(pix);
    if (kernel == HalfKernel::WINDOWED) {
        const Win3x3 geo{pix.src, pix.Hs, pix.Ws, pix.sample_elems, pix.sample_elems * pix.nsamples, pix.nsamples, Cred};
        return launch_win3x3<MODE, bf16_t, PAD>(ctx, st, MODE == 0 ? kFwdWin3Names : kBwdDataWin3Names, al, geo, ep, rows, N, K, flops, left);
    }
    bool staged = false;
    const int rcs = launch_staged<MODE>(ctx, st, names, al, K, rows, Cred, pix, kernel == HalfKernel::PAIRS, ep, flops, (char*)ctx->reduce_scratch + taken, left, &staged);
    if (staged || rcs != VDNN_OK) return rcs;
    if (kernel == HalfKernel::PAIRS) {
        LoadIm2colPixTapH2<MODE, PAD> bl2{pix, Cred};
        return launch_by_m<LoadPackedH, LoadIm2colPixTapH2<MODE, PAD>, bf16_t, true>(ctx, st, names, al, bl2, ep, rows, N, K, flops, left);
    }
    LoadIm2colPixTapH<MODE, PAD> bl{pix, Cred};
    return launch_by_m<LoadPackedH, LoadIm2colPixTapH<MODE, PAD>, bf16_t, true>(ctx, st, names, al, bl, ep, rows, N, K, flops, left);
}
template <int MODE>
static int conv_half_engine(vdnn_ctx* ctx, hipStream_t st, const PassNames& names, const float* w, int rows, int Cred, int RS, int row_stride, int red_stride,
                            const LoadIm2colPix<MODE, false, bf16_t>& pix, const StoreNCHW<bf16_t>& ep, int N, double flops) {
    return Cred % KH == 0 ? conv_half_engine_with<MODE, false>(ctx, st, names, w, rows, Cred, RS, row_stride, red_stride, pix, ep, N, flops)
                          : conv_half_engine_with<MODE, true>(ctx, st, names, w, rows, Cred, RS, row_stride, red_stride, pix, ep, N, flops);
}

// ---- perf-optimal mode, float layers: 3x3 / stride 1 / padding 1 on the bfloat16 matrix cores ------------------
// Every float operand as two bfloat16 parts, three matrix instructions per product (conv3x3_bf16.h): forward and
// backward data through the windowed kernel, the split filter bank (as many bytes as the filter) in the workspace.
// Which variant the perf-optimal mode takes where both apply: 0 = this one, through the windowed kernel or the general
// engine (faster than Winograd on every VGG16 / AlexNet / OverFeat layer, closer to the exact result, no transformed
// tensors; backward filter of the layers it does not take stays Winograd's), 1 = Winograd. vdnn_conv_perf_variant.
static int g_perf_variant = 0;

// MODE 0: rows = output channels, reduced = input channels; MODE 1: rows = input channels, reduced = output channels
static bool split3x3_ok(const ConvGeo& g, int mode) {
    const int reduced = mode == 0 ? g.C : g.K, rows = mode == 0 ? g.K : g.C;
    const long sample = mode == 0 ? (long)g.C * g.H * g.W : (long)g.K * g.P * g.Q;
    return reduced % 16 == 0 && g.C > 4 && (long)rows * reduced * 9 * 4 < (1l << 31) &&
           win3x3_ok(g.R, g.S, g.ph, g.pw, g.sh, g.sw, g.H, g.W, g.P, g.Q, sample, 4);
}

template <int MODE>
static int launch_split3x3(vdnn_ctx* ctx, hipStream_t st, const ConvGeo& g, const float* src, const float* w, const StoreNCHW<float>& ep,
                           void* workspace, size_t workspace_bytes, bool* taken) {
    *taken = false;
    const int rows = MODE == 0 ? g.K : g.C, reduced = MODE == 0 ? g.C : g.K;
    const size_t bank = (size_t)rows * reduced * 9 * 4;
    if (!split3x3_ok(g, MODE) || !workspace || workspace_bytes < bank || !aligned16(workspace)) return VDNN_OK;
    *taken = true;
    unsigned short* packed = (unsigned short*)workspace;
    {
        const long total = (long)rows * reduced * 9;
        ProfScope prof(ctx, st, "conv_pack_filter", 0.0, 8.0 * (double)total);
        hipLaunchKernelGGL(pack_filter_split_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, w, packed, rows, reduced, 9,
                           MODE == 0 ? g.C * 9 : 9, MODE == 0 ? 9 : g.C * 9, total);
        VDNN_LAUNCH_CHECK();
    }
    const long sample = MODE == 0 ? (long)g.C * g.H * g.W : (long)g.K * g.P * g.Q;
    const LoadPackedH al{packed, (long)reduced * 18, rows, (unsigned)bank};
    const Win3x3T<float> geo{src, g.H, g.W, sample, sample * g.N, g.N};
    return launch_win3x3<MODE, float>(ctx, st, MODE == 0 ? kFwdSplitNames : kBwdDataSplitNames, al, geo, ep, rows, g.N * g.H * g.W, reduced * 18,
                                      2.0 * g.N * (double)g.K * g.C * 9 * g.P * g.Q, ctx->reduce_scratch_bytes);
}

// The same products through the general bfloat16 engine, for stride-1 layers the windowed kernel does not take (other
// windows than 3x3, no or other padding, planes with odd rows): forward (MODE 0) and backward data (MODE 1), at most 32
// taps, reduced channels a multiple of 16.
static bool split_general_ok(const ConvGeo& g, int mode) {
    const int reduced = mode == 0 ? g.C : g.K, rows = mode == 0 ? g.K : g.C;
    return g.R * g.S <= 32 && reduced % 16 == 0 && g.C > 4 && (mode == 0 || (g.sh == 1 && g.sw == 1)) &&
           (long)rows * reduced * g.R * g.S * 4 < (1l << 31);
}

static const PassNames kFwdSplitGenNames{"conv_fwd_splitgen_64x256", "conv_fwd_splitgen_128x128"};
static const PassNames kBwdDataSplitGenNames{"conv_bwd_data_splitgen_64x256", "conv_bwd_data_splitgen_128x128"};

template <int MODE>
static int launch_split_general(vdnn_ctx* ctx, hipStream_t st, const ConvGeo& g, const float* src, const float* w, const StoreNCHW<float>& ep,
                                void* workspace, size_t workspace_bytes, bool* taken) {
    *taken = false;
    const int RS = g.R * g.S;
    const int rows = MODE == 0 ? g.K : g.C, reduced = MODE == 0 ? g.C : g.K;
    const size_t bank = (size_t)rows * reduced * RS * 4;
    if (!split_general_ok(g, MODE) || !workspace || workspace_bytes < bank || !aligned16(workspace)) return VDNN_OK;
    const long sample = MODE == 0 ? (long)g.C * g.H * g.W : (long)g.K * g.P * g.Q;
    const int opix = MODE == 0 ? g.P * g.Q : g.H * g.W;
    if (!pixel_tile_span_ok(sample, opix, 256, 4)) return VDNN_OK;
    *taken = true;
    unsigned short* packed = (unsigned short*)workspace;
    {
        const long total = (long)rows * reduced * RS;
        ProfScope prof(ctx, st, "conv_pack_filter", 0.0, 8.0 * (double)total);
        hipLaunchKernelGGL(pack_filter_split_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, w, packed, rows, reduced, RS,
                           MODE == 0 ? g.C * RS : RS, MODE == 0 ? RS : g.C * RS, total);
        VDNN_LAUNCH_CHECK();
    }
    const LoadPackedH al{packed, (long)reduced * RS * 2, rows, (unsigned)bank};
    const FastDiv dRS = FastDiv::make(RS), dS = FastDiv::make(g.S);
    const double flops = 2.0 * g.N * (double)g.K * g.C * RS * g.P * g.Q;
    if (MODE == 0) {
        const LoadIm2colPixTapS<MODE> bl{{src, g.H, g.W, g.P, g.Q, g.R, g.S, g.ph, g.pw, g.sh, g.sw, sample, g.N, dRS, dS}};
        return launch_by_m<LoadPackedH, LoadIm2colPixTapS<MODE>, float, true>(ctx, st, kFwdSplitGenNames, al, bl, ep, rows, g.N * opix, reduced * RS * 2, flops);
    }
    const LoadIm2colPixTapS<MODE> bl{{src, g.P, g.Q, g.H, g.W, g.R, g.S, g.ph, g.pw, 1, 1, sample, g.N, dRS, dS}};
    return launch_by_m<LoadPackedH, LoadIm2colPixTapS<MODE>, float, true>(ctx, st, kBwdDataSplitGenNames, al, bl, ep, rows, g.N * opix, reduced * RS * 2, flops);
}

static int launch_pack_filter(vdnn_ctx* ctx, hipStream_t st, const float* w, float* packed, int rows, int Cred, int RS,
                              int row_stride, int red_stride) {
    const int Cpad = (Cred + KB - 1) / KB * KB;
    const long total = (long)rows * Cpad * RS;
    ProfScope prof(ctx, st, "conv_pack_filter", 0.0, 8.0 * (double)total);
    hipLaunchKernelGGL(pack_filter_tap_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, w, packed, rows, Cred, Cpad, RS,
                       row_stride, red_stride, total);
    VDNN_LAUNCH_CHECK();
    return VDNN_OK;
}

// Workgroups of wgrad3x3_bf16_kernel that are resident on a compute unit (its launch bounds).
constexpr int kWgrad3PerCU = 2;


static bool wgrad3x3_ok(const ConvGeo& g) {
    return g.R == 3 && g.S == 3 && g.ph == 1 && g.pw == 1 && g.sh == 1 && g.sw == 1 && g.P == g.H && g.Q == g.W &&
           g.W % 4 == 0 && g.W >= 16 && (g.H * g.W) % 8 == 0 && g.C % WG3_CH == 0; // a slice wraps at most two image rows
}

// One filter row, 64 input channels and 128 (64) output channels per workgroup; the pixel reduction is split so
// that one round of workgroups fills the chip, as far as the staging area holds the partial sums.
static int launch_wgrad3x3(vdnn_ctx* ctx, hipStream_t st, const ConvGeo& g, const bf16_t* x, const bf16_t* dy, float* w, float alpha, int accumulate,
                           float* staging, size_t staging_bytes, bool* taken, BiasOut* bias) {
    *taken = false;
    const int M = g.K, N = g.C * 9, PQ = g.H * g.W;
    const long Kred = (long)g.N * PQ;
    const bool narrow = M <= 64;
    const int TM = narrow ? 64 : 128;
    const int mtiles = (M + TM - 1) / TM, ntiles = 3 * (g.C / WG3_CH);
    const long tiles = (long)mtiles * ntiles;
    const size_t out_bytes = (size_t)M * N * sizeof(float);
    long splits = (long)kWgrad3PerCU * ctx->num_cu / tiles;
    const long by_len = Kred / (8 * KH); // at least eight slices per split
    const long by_mem = staging ? (long)(staging_bytes / out_bytes) : 1;
    if (splits > by_len) splits = by_len;
    if (splits > by_mem) splits = by_mem;
    if (splits < 1) splits = 1;
    GemmDims d = make_dims(M, N, (int)Kred, TM, 3 * WG3_CH, (int)splits, KH);
    d.mtiles = mtiles; d.ntiles = ntiles;
    const long nspan = d.kchunk / PQ + 2;
    if (nspan * g.K * PQ * 2 >= (long)MAX_SUM_RANGE || nspan * g.C * PQ * 2 >= (long)MAX_SUM_RANGE) return VDNN_OK; // not taken
    if (d.splits > 1 && !staging) return VDNN_OK;
    const long blocks = tiles * d.splits;
    if (blocks <= 0 || blocks >= (1l << 31)) return VDNN_OK;
    *taken = true;
    const bool with_bias = bias && bias->wanted() && bias_parts_fit(ctx, g.K, d.splits);
    const Wgrad3x3 geo{dy, x, g.N, g.K, g.C, g.H, g.W, w, staging, (long)M * N, alpha, accumulate, with_bias ? ctx->bias_scratch : nullptr, d.splits};
    {
        ProfScope prof(ctx, st, narrow ? kBwdFilterWin3Names.t64 : kBwdFilterWin3Names.t128, 2.0 * M * (double)N * (double)Kred, 0.0);
        const bool halfrow = g.W % 8 != 0 || g.W < KH; // the general variant: groups across two image rows, two row wraps per slice
        if (narrow && halfrow) hipLaunchKernelGGL((wgrad3x3_bf16_kernel<32, true>), dim3((unsigned)blocks), dim3(NT), 0, st, geo, d);
        else if (narrow) hipLaunchKernelGGL((wgrad3x3_bf16_kernel<32, false>), dim3((unsigned)blocks), dim3(NT), 0, st, geo, d);
        else if (halfrow) hipLaunchKernelGGL((wgrad3x3_bf16_kernel<64, true>), dim3((unsigned)blocks), dim3(NT), 0, st, geo, d);
        else hipLaunchKernelGGL((wgrad3x3_bf16_kernel<64, false>), dim3((unsigned)blocks), dim3(NT), 0, st, geo, d);
        VDNN_LAUNCH_CHECK();
    }
    if (with_bias) {
        const int rc = launch_bias_grad_final(ctx, st, ctx->bias_scratch, bias->out, g.K, d.splits, bias->alpha, bias->accumulate);
        if (rc != VDNN_OK) return rc;
        bias->done = true;
    }
    if (d.splits > 1) return launch_reduce_splits_tap(ctx, st, w, staging, (size_t)M * N, d.splits, alpha, accumulate, g.C, 9);
    return VDNN_OK;
}

// The perf-optimal float counterpart of launch_wgrad3x3 (wgrad3x3_split.h): the same tiles and splits, slices of 16 pixels.
static int launch_wgrad3x3_split(vdnn_ctx* ctx, hipStream_t st, const ConvGeo& g, const float* x, const float* dy, float* w, float alpha, int accumulate,
                                 float* staging, size_t staging_bytes, bool* taken, BiasOut* bias) {
    *taken = false;
    const int M = g.K, N = g.C * 9, PQ = g.H * g.W;
    const long Kred = (long)g.N * PQ;
    const bool narrow = M <= 64;
    const int TM = narrow ? 64 : 128;
    const int mtiles = (M + TM - 1) / TM, ntiles = 3 * (g.C / WG3_CH);
    const long tiles = (long)mtiles * ntiles;
    const size_t out_bytes = (size_t)M * N * sizeof(float);
    const long slots = (long)kWgrad3PerCU * ctx->num_cu;
    // as many rounds of workgroups as the tiles alone need, each filled by the splits
    const long rounds = (tiles + slots - 1) / slots;
    long splits = rounds * slots / tiles;
    const long by_len = Kred / (16 * WG3S_SLICE); // at least sixteen slices per split
    const long by_mem = staging ? (long)(staging_bytes / out_bytes) : 1;
    if (splits > by_len) splits = by_len;
    if (splits > by_mem) splits = by_mem;
    if (splits < 1) splits = 1;
    GemmDims d = make_dims(M, N, (int)Kred, TM, 3 * WG3_CH, (int)splits, WG3S_SLICE);
    d.mtiles = mtiles; d.ntiles = ntiles;
    const long nspan = d.kchunk / PQ + 2;
    if (nspan * g.K * PQ * 4 >= (long)MAX_SUM_RANGE || nspan * g.C * PQ * 4 >= (long)MAX_SUM_RANGE) return VDNN_OK; // not taken
    if (d.splits > 1 && !staging) return VDNN_OK;
    const long blocks = tiles * d.splits;
    if (blocks <= 0 || blocks >= (1l << 31)) return VDNN_OK;
    *taken = true;
    const bool with_bias = bias && bias->wanted() && bias_parts_fit(ctx, g.K, d.splits);
    const Wgrad3x3S geo{dy, x, g.N, g.K, g.C, g.H, g.W, w, staging, (long)M * N, alpha, accumulate, with_bias ? ctx->bias_scratch : nullptr, d.splits};
    {
        ProfScope prof(ctx, st, narrow ? "conv_bwd_filter_split_64x192" : "conv_bwd_filter_split_128x192", 2.0 * M * (double)N * (double)Kred, 0.0);
        const bool halfrow = g.W % 8 != 0; // groups of eight pixels across two image rows
        if (narrow && halfrow) hipLaunchKernelGGL((wgrad3x3_split_kernel<32, true>), dim3((unsigned)blocks), dim3(NT), 0, st, geo, d);
        else if (narrow) hipLaunchKernelGGL((wgrad3x3_split_kernel<32, false>), dim3((unsigned)blocks), dim3(NT), 0, st, geo, d);
        else if (halfrow) hipLaunchKernelGGL((wgrad3x3_split_kernel<64, true>), dim3((unsigned)blocks), dim3(NT), 0, st, geo, d);
        else hipLaunchKernelGGL((wgrad3x3_split_kernel<64, false>), dim3((unsigned)blocks), dim3(NT), 0, st, geo, d);
        VDNN_LAUNCH_CHECK();
    }
    if (with_bias) {
        const int rc = launch_bias_grad_final(ctx, st, ctx->bias_scratch, bias->out, g.K, d.splits, bias->alpha, bias->accumulate);
        if (rc != VDNN_OK) return rc;
        bias->done = true;
    }
    if (d.splits > 1) return launch_reduce_splits_tap(ctx, st, w, staging, (size_t)M * N, d.splits, alpha, accumulate, g.C, 9);
    return VDNN_OK;
}

// Workgroups of wgrad3x3_f32_kernel that are resident on a compute unit (its launch bounds; three, at 167 registers, measured 10 % slower).
constexpr int kWgrad3FPerCU = 2;

// The float counterpart of launch_wgrad3x3.
static int launch_wgrad3x3_f32(vdnn_ctx* ctx, hipStream_t st, const ConvGeo& g, const float* x, const float* dy, float* w, float alpha, int accumulate,
                               float* staging, size_t staging_bytes, bool* taken, BiasOut* bias) {
    *taken = false;
    const int M = g.K, N = g.C * 9, PQ = g.H * g.W;
    const long Kred = (long)g.N * PQ;
    const bool narrow = M <= 64;
    const int TM = narrow ? 64 : 128;
    const int mtiles = (M + TM - 1) / TM, ntiles = 3 * (g.C / WG3F_CH);
    const long tiles = (long)mtiles * ntiles;
    const size_t out_bytes = (size_t)M * N * sizeof(float);
    const long slots = (long)kWgrad3FPerCU * ctx->num_cu;
    // as many rounds of workgroups as the tiles alone need, each filled by the splits
    const long rounds = (tiles + slots - 1) / slots;
    long splits = rounds * slots / tiles;
    const long by_len = Kred / (8 * KB); // at least eight slices per split
    const long by_mem = staging ? (long)(staging_bytes / out_bytes) : 1;
    if (splits > by_len) splits = by_len;
    if (splits > by_mem) splits = by_mem;
    if (splits < 1) splits = 1;
    GemmDims d = make_dims(M, N, (int)Kred, TM, 3 * WG3F_CH, (int)splits, KB);
    d.mtiles = mtiles; d.ntiles = ntiles;
    const long nspan = d.kchunk / PQ + 2;
    if (nspan * g.K * PQ * 4 >= (long)MAX_SUM_RANGE || nspan * g.C * PQ * 4 >= (long)MAX_SUM_RANGE) return VDNN_OK; // not taken
    if (d.splits > 1 && !staging) return VDNN_OK;
    const long blocks = tiles * d.splits;
    if (blocks <= 0 || blocks >= (1l << 31)) return VDNN_OK;
    *taken = true;
    const bool with_bias = bias && bias->wanted() && bias_parts_fit(ctx, g.K, d.splits);
    const Wgrad3x3F geo{dy, x, g.N, g.K, g.C, g.H, g.W, w, staging, (long)M * N, alpha, accumulate, with_bias ? ctx->bias_scratch : nullptr, d.splits};
    {
        ProfScope prof(ctx, st, narrow ? kBwdFilterRow3Names.t64 : kBwdFilterRow3Names.t128, 2.0 * M * (double)N * (double)Kred, 0.0);
        const bool halfrow = g.W % 4 != 0 || g.W < KB; // the general variant: groups across two image rows, two row wraps per slice
        if (narrow && halfrow) hipLaunchKernelGGL((wgrad3x3_f32_kernel<32, true>), dim3((unsigned)blocks), dim3(NT), 0, st, geo, d);
        else if (narrow) hipLaunchKernelGGL((wgrad3x3_f32_kernel<32, false>), dim3((unsigned)blocks), dim3(NT), 0, st, geo, d);
        else if (halfrow) hipLaunchKernelGGL((wgrad3x3_f32_kernel<64, true>), dim3((unsigned)blocks), dim3(NT), 0, st, geo, d);
        else hipLaunchKernelGGL((wgrad3x3_f32_kernel<64, false>), dim3((unsigned)blocks), dim3(NT), 0, st, geo, d);
        VDNN_LAUNCH_CHECK();
    }
    if (with_bias) {
        const int rc = launch_bias_grad_final(ctx, st, ctx->bias_scratch, bias->out, g.K, d.splits, bias->alpha, bias->accumulate);
        if (rc != VDNN_OK) return rc;
        bias->done = true;
    }
    if (d.splits > 1) return launch_reduce_splits_tap(ctx, st, w, staging, (size_t)M * N, d.splits, alpha, accumulate, g.C, 9);
    return VDNN_OK;
}

// Forward of a 3x3 / stride 1 / padding 1 layer with at most four input and 64 output channels: wavefronts stream over
// the pixels, three workgroups per compute unit.
static bool fwd_smallc3x3_ok(const ConvGeo& g, size_t elem_bytes) {
    return g.C <= 4 && g.K <= 64 && g.R == 3 && g.S == 3 && g.ph == 1 && g.pw == 1 && g.sh == 1 && g.sw == 1 && g.P == g.H && g.Q == g.W &&
           (long)g.N * g.C * g.H * g.W * (long)elem_bytes < (1l << 31) && (long)g.N * g.K * g.H * g.W * (long)elem_bytes < (1l << 31);
}
template <class E>
static int launch_fwd_smallc3x3(vdnn_ctx* ctx, hipStream_t st, const ConvGeo& g, const E* x, const float* w, const float* bias, E* y, int relu) {
    // two blocks of 32 pixels per unit where that makes a store a whole 128-byte line (two-byte elements: 0.47 -> 0.38 ms
    // for VGG16's first layer at batch 128); with floats a block's 32 pixels are a line already and two measured the same
    const int up = sizeof(E) == 2 ? 2 : 1;
    const long units = ((long)g.N * g.H * g.W + 32 * up - 1) / (32 * up);
    long blocks = (units + 3) / 4;
    // bound by its stores from two workgroups per unit on (four measured 20 % slower); with two blocks per unit the
    // registers allow two
    const long resident = (up == 2 ? 2l : 3l) * ctx->num_cu;
    if (blocks > resident) blocks = resident;
    ProfScope prof(ctx, st, "conv_fwd_smallc", 2.0 * g.K * 9.0 * g.C * (double)g.N * g.H * g.W, 0.0);
#define VDNN_FWD_SMALLC_UP(CC, RB, UP) hipLaunchKernelGGL((conv_fwd_smallc3x3_kernel<CC, RB, UP, E>), dim3((unsigned)blocks), dim3(256), 0, st, x, w, bias, y, g.N, g.K, g.H, g.W, relu)
#define VDNN_FWD_SMALLC(CC)                                                                         \
    do {                                                                                            \
        if (g.K <= 32) { if (up == 2) VDNN_FWD_SMALLC_UP(CC, 1, 2); else VDNN_FWD_SMALLC_UP(CC, 1, 1); } \
        else { if (up == 2) VDNN_FWD_SMALLC_UP(CC, 2, 2); else VDNN_FWD_SMALLC_UP(CC, 2, 1); }           \
    } while (0)
    switch (g.C) {
    case 1: VDNN_FWD_SMALLC(1); break;
    case 2: VDNN_FWD_SMALLC(2); break;
    case 3: VDNN_FWD_SMALLC(3); break;
    default: VDNN_FWD_SMALLC(4); break;
    }
#undef VDNN_FWD_SMALLC_UP
#undef VDNN_FWD_SMALLC
    VDNN_LAUNCH_CHECK();
    return VDNN_OK;
}

// Backward data by residue classes saves matrix work and pays with float results in the staging area, read again by the
// merge: it loses where a pixel of dx has few products (32 x 128 x 94 x 94, 2 filters of 3x3 at stride 3x1: 106 us in one
// product, 282 by classes; 57 x 121 x 89 x 89 bfloat16, 7 of 1x1 at stride 2: 103 and 232). Both times are estimated, from 4900
// calls timed on both routes: launches, matrix work (by classes at 105 TFLOP/s; in one product, with a tap to work out per
// element, at 50 up to 4 GFLOP, on the 64x64 tile, and 85 beyond, on the large ones; a bfloat16 layer's filter is rounded first),
// and what moving the elements of dx adds, with the gate and beyond what the caches hold. The choice is 0.4 % (floats) and 0.7 %
// (bfloat16) behind the better route in the mean.
static bool classes_pay(const ConvGeo& g, int elem_bytes, bool gated) {
    const bool half = elem_bytes == 2;
    const double reduction = (double)g.K * g.R * g.S, pixels = (double)g.N * g.H * g.W, elems = 1e-6 * pixels * g.C;
    const double rows = (g.C + 63) / 64 * 64, padded = (double)((g.K + KB - 1) / KB * KB) * g.R * g.S;
    const double classes_ops = 2e-8 * padded * rows * pixels / (g.sh * g.sw), one_ops = 2e-8 * reduction * rows * pixels;
    const double small = one_ops < 40.0 ? one_ops : 40.0, uncached = elems > 12.0 ? elems - 12.0 : 0.0;
    const double classes_us = 14.2 + 0.95 * classes_ops + (gated ? 4.55 : 4.05) * elems + (!gated ? 0.15 : half ? 0.75 : 1.75) * uncached;
    const double one_us = half ? 10.5 + 0.23 * std::sqrt(reduction) + 2.0 * small + 1.2 * (one_ops - small) + (gated ? 2.1 : 1.2) * elems
                               : 8.8 + 0.09 * std::sqrt(reduction) + 2.0 * small + 1.17 * (one_ops - small) + (gated ? 1.45 : 1.05) * elems;
    return classes_us < one_us;
}

// Backward data of a strided layer by residue classes (conv_strided.h): as many samples at a time as the staging area
// holds results of, 64x64 tiles, the reductions cut so that the workgroups of all classes together fill the chip.
template <class E>
static int launch_strided_bwd_data(vdnn_ctx* ctx, hipStream_t st, const ConvGeo& g, const E* dy, const float* w, E* dx, const E* gate, bool* taken) {
    *taken = false;
    const int classes = g.sh * g.sw;
    // (samples that the one product's tiles could not address stay refused by the caller)
    if (classes > kStridedClasses || !classes_pay(g, (int)sizeof(E), gate != nullptr) || !ctx->reduce_scratch || !pixel_tile_span_ok((long)g.K * g.P * g.Q, g.H * g.W, 256, (int)sizeof(E))) return VDNN_OK;
    StridedGeo q{};
    q.sh = g.sh; q.sw = g.sw; q.ph = g.ph; q.pw = g.pw;
    q.C = g.C; q.H = g.H; q.W = g.W; q.R = g.R; q.S = g.S; q.K = g.K; q.Kpad = (g.K + KB - 1) / KB * KB;
    long filter_elems = 0, most_slices = 0;
    const long sample = (long)g.K * g.P * g.Q;
    for (int a = 0; a < g.sh; a++)
        for (int b = 0; b < g.sw; b++) {
            StridedClassGeo& c = q.c[a * g.sw + b];
            c.rows = a < g.R ? (g.R - a + g.sh - 1) / g.sh : 0;
            c.cols = b < g.S ? (g.S - b + g.sw - 1) / g.sw : 0;
            c.taps = c.rows * c.cols;
            c.u0 = g.ph > a ? (g.ph - a + g.sh - 1) / g.sh : 0;
            c.v0 = g.pw > b ? (g.pw - b + g.sw - 1) / g.sw : 0;
            c.opix_h = g.H - 1 + g.ph >= a ? (g.H - 1 + g.ph - a) / g.sh - c.u0 + 1 : 0;
            c.opix_w = g.W - 1 + g.pw >= b ? (g.W - 1 + g.pw - b) / g.sw - c.v0 + 1 : 0;
            c.filter_first = filter_elems;
            filter_elems += (long)g.C * q.Kpad * c.taps;
            if (c.taps > 32) return VDNN_OK;
            if (c.opix_h <= 0 || c.opix_w <= 0) { c.opix_h = c.opix_w = 0; continue; }
            if (!pixel_tile_span_ok(sample, c.opix_h * c.opix_w, 64, (int)sizeof(E))) return VDNN_OK;
            const long slices = (long)(q.Kpad / KB) * c.taps;
            if (slices > most_slices) most_slices = slices;
        }
    if (most_slices == 0 || filter_elems * 4 >= 0x7FFF0000l) return VDNN_OK;
    StagingCarve carve(ctx);
    float* packed = packed_filter_place(ctx, carve, (size_t)filter_elems * sizeof(float));
    if (!packed) return VDNN_OK;
    const long per_sample = (long)g.C * g.H * g.W, room = (long)(ctx->reduce_scratch_bytes / sizeof(float));
    const long nb = room / per_sample < g.N ? room / per_sample : g.N;
    if (nb < 1 || nb * per_sample >= (1l << 31)) return VDNN_OK;
    *taken = true;
    {
        ProfScope prof(ctx, st, "conv_pack_filter", 0.0, 8.0 * (double)filter_elems);
        const dim3 grid((unsigned)((filter_elems + 255) / 256));
        if (sizeof(E) == 2) hipLaunchKernelGGL(pack_filter_classes_kernel<true>, grid, dim3(256), 0, st, w, packed, q, filter_elems);
        else hipLaunchKernelGGL(pack_filter_classes_kernel<false>, grid, dim3(256), 0, st, w, packed, q, filter_elems);
        VDNN_LAUNCH_CHECK();
    }
    // slices per workgroup: the estimate of small_tile_plan over the tiles of all classes of the first (largest) chunk
    auto class_splits = [&](const StridedClassGeo& c, long per) { return ((long)(q.Kpad / KB) * c.taps + per - 1) / per; };
    auto tiles_of = [&](const StridedClassGeo& c, long n) { return (g.C + 63) / 64 * ((n * c.opix_h * c.opix_w + 63) / 64); };
    long per = most_slices;
    double best = 0.0;
    for (long s = 1; s <= 32; s++) {
        const long len = (most_slices + s - 1) / s;
        if (s > 1 && len < 4) break;
        long blocks = 0, elems = 0, work = 0;
        for (int c = 0; c < classes; c++) {
            if (q.c[c].opix_h == 0 || q.c[c].taps == 0) continue;
            const long splits = class_splits(q.c[c], len), tiles = tiles_of(q.c[c], nb), slices = (long)(q.Kpad / KB) * q.c[c].taps;
            blocks += tiles * splits;
            work += tiles * (slices + 8 * splits);
            elems += splits * nb * g.C * q.c[c].opix_h * q.c[c].opix_w;
        }
        if (elems > room) break;
        // a round of workgroups lasts as long as its longest; beyond that the units share the work evenly
        double us = 0.27 * (double)((work + ctx->num_cu - 1) / ctx->num_cu);
        const double floor_us = 0.27 * (double)(len + 8) * (blocks <= ctx->num_cu ? 1.5 : 1.2);
        if (us < floor_us) us = floor_us;
        us += (double)elems * 2.4 / 4e6;
        if (best == 0.0 || us < best) { best = us; per = len; }
    }
    const FastDiv one = FastDiv::make(1);
    for (int n0 = 0; n0 < g.N; n0 += (int)nb) {
        const int nc = g.N - n0 < nb ? g.N - n0 : (int)nb;
        StridedLaunch<E> launch{};
        long first = 0, blocks = 0;
        for (int c = 0; c < classes; c++) {
            StridedClassGeo& cg = q.c[c];
            cg.result_first = first;
            cg.splits = 0;
            if (cg.opix_h == 0 || cg.taps == 0) continue;
            const int opix = cg.opix_h * cg.opix_w, K = q.Kpad * cg.taps;
            const GemmDims d = make_dims(g.C, nc * opix, K, 64, 64, (int)class_splits(cg, per));
            cg.splits = d.splits;
            float* out = ctx->reduce_scratch + first;
            StridedClass<E> k{};
            k.al = LoadDenseRed<true>{packed + cg.filter_first, (long)K, g.C, (unsigned)((long)g.C * K * 4)};
            k.bl.base = LoadIm2colPix<1, false, E>{dy + (long)n0 * sample, g.P, g.Q, cg.opix_h, cg.opix_w, cg.rows, cg.cols, cg.u0, cg.v0, 1, 1, sample, nc, one, one};
            k.bl.base.divRS = FastDiv::make(cg.taps); k.bl.base.divS = FastDiv::make(cg.cols);
            k.bl.channels = g.K;
            k.ep = StoreNCHW<float>{out, nullptr, opix, out, 0, nullptr};
            k.d = d;
            k.blocks = d.mtiles * d.ntiles * d.splits;
            blocks += k.blocks;
            first += (long)d.splits * nc * g.C * opix;
            // the classes of most taps first
            int at = launch.count++;
            for (; at > 0 && launch.c[at - 1].d.kchunk < d.kchunk; at--) launch.c[at] = launch.c[at - 1];
            launch.c[at] = k;
        }
        VDNN_REQUIRE(blocks < (1l << 31), "grid too large");
        {
            ProfScope prof(ctx, st, "conv_bwd_data_classes_64x64", 2.0 * nc * (double)g.K * g.C * g.R * g.S * g.P * g.Q, 0.0);
            if (small_tile_ahead(launch.c[launch.count - 1].d, blocks)) hipLaunchKernelGGL((igemm_classes_kernel<E, kSmallTileAhead>), dim3((unsigned)blocks), dim3(NT), 0, st, launch);
            else hipLaunchKernelGGL((igemm_classes_kernel<E, 1>), dim3((unsigned)blocks), dim3(NT), 0, st, launch);
            VDNN_LAUNCH_CHECK();
        }
        const long total = (long)nc * per_sample;
        ProfScope prof(ctx, st, "conv_bwd_data_merge", 0.0, (double)first * 4.0 + (double)total * sizeof(E) * (gate ? 2.0 : 1.0));
        hipLaunchKernelGGL(merge_classes_kernel<E>, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, ctx->reduce_scratch, dx + (long)n0 * per_sample,
                           gate ? gate + (long)n0 * per_sample : nullptr, q, nc, (unsigned)total);
        VDNN_LAUNCH_CHECK();
    }
    return VDNN_OK;
}

// Backward filter of a bfloat16 3x3 / stride 1 / padding 1 layer with the vector loaders: picks the instantiation
// for the number of taps per tile and the pixel group (combinations whose loads would mix taps do not exist).
template <int TM, int TN, int NTAP, int G>
static int launch_wgrad_vec_one(vdnn_ctx* ctx, hipStream_t st, const char* name, const LoadDyRedVecH<8>& al, const LoadIm2colRedTapVecH<1, 4>& geo,
                                const StoreFilterTap& ep, const GemmDims& d) {
    if constexpr ((TN / NTAP) % (NT / (KH / G)) != 0) {
        set_error("backward filter: %d taps per %d-column tile with groups of %d pixels", NTAP, TN, G);
        return VDNN_EINVAL;
    } else {
        LoadIm2colRedTapVecH<NTAP, G> bl{geo.x, geo.N, geo.C, geo.H, geo.W, geo.ncols, geo.kchunk, geo.Ktot, geo.divC};
        return launch_igemm<TM, TN, LoadDyRedVecH<8>, LoadIm2colRedTapVecH<NTAP, G>, StoreFilterTap, true>(ctx, st, name, al, bl, ep, d);
    }
}
template <int TM, int TN>
static int launch_wgrad_vec(vdnn_ctx* ctx, hipStream_t st, const char* name, const LoadDyRedVecH<8>& al, const LoadIm2colRedTapVecH<1, 4>& geo,
                            const StoreFilterTap& ep, const GemmDims& d, int ntap, int group) {
    if (group != 4) { set_error("backward filter: groups of %d pixels", group); return VDNN_EINVAL; }
    if (ntap == 1) return launch_wgrad_vec_one<TM, TN, 1, 4>(ctx, st, name, al, geo, ep, d);
    if (ntap == 2) return launch_wgrad_vec_one<TM, TN, 2, 4>(ctx, st, name, al, geo, ep, d);
    return launch_wgrad_vec_one<TM, TN, 4, 4>(ctx, st, name, al, geo, ep, d);
}

} // namespace vdnn

using namespace vdnn;

template <class E>
static int conv_fwd_impl(vdnn_ctx* ctx, vdnn_stream_t stream, const vdnn_shape_t* shape, int algo_mode,
                         const E* x, const float* w, const float* bias, E* y,
                         void* workspace, size_t workspace_bytes, int relu) {
    VDNN_KERNEL_PROLOGUE(ctx);
    ConvGeo g;
    VDNN_REQUIRE(shape && geo_from_shape(shape, g), "unsupported convolution geometry");
    VDNN_REQUIRE(x && w && y, "null tensor");
    if (is_dense(g))
        return relu ? vdnn_fc_fwd_relu(ctx, stream, g.N, g.C * g.H * g.W, g.K, x, w, bias, y)
                    : vdnn_fc_fwd(ctx, stream, g.N, g.C * g.H * g.W, g.K, x, w, bias, y);
    VDNN_REQUIRE(pixel_tile_span_ok((long)g.C * g.H * g.W, g.P * g.Q, 256, (int)sizeof(E)), "input samples too large for one tile's descriptor");
    hipStream_t st = stream_of(ctx, stream);
    const int K = g.C * g.R * g.S;
    const unsigned wbytes = (unsigned)((long)g.K * K * 4);
    if constexpr (sizeof(E) == 2) {
        const int RS = g.R * g.S;
        const LoadIm2colPix<0, false, bf16_t> pix{x, g.H, g.W, g.P, g.Q, g.R, g.S, g.ph, g.pw, g.sh, g.sw, (long)g.C * g.H * g.W, g.N,
                                                 FastDiv::make(RS), FastDiv::make(g.S)};
        if (half_engine_ok(ctx, pix, g.C, g.K, RS)) {
            StoreNCHW<bf16_t> ep{y, bias, g.P * g.Q, nullptr, relu, nullptr};
            return conv_half_engine<0>(ctx, st, kFwdHalfNames, w, g.K, g.C, RS, g.C * RS, RS, pix, ep, g.N * g.P * g.Q,
                                       2.0 * g.N * (double)g.K * K * g.P * g.Q);
        }
    }
    StagingCarve carve(ctx);
    if constexpr (sizeof(E) == 2) {
        w = rounded_filter_copy(ctx, st, carve, w, (size_t)g.K * K);
        VDNN_REQUIRE(w != nullptr, "filter too large for the staging area (bfloat16 layer outside the bfloat16 engine)");
        VDNN_LAUNCH_CHECK();
    }
    if (fwd_smallc3x3_ok(g, sizeof(E))) return launch_fwd_smallc3x3<E>(ctx, st, g, x, w, bias, y, relu);
    if constexpr (sizeof(E) == 4) {
        if (algo_mode == 1) {
            // perf-optimal: 3x3 layers on the bfloat16 matrix cores, or as Winograd F(4x4, 3x3), through the workspace
            bool taken = false;
            if (g_perf_variant == 0) {
                const StoreNCHW<float> eps{y, bias, g.P * g.Q, ctx->reduce_scratch, relu, nullptr};
                const int rc = launch_split3x3<0>(ctx, st, g, x, w, eps, workspace, workspace_bytes, &taken);
                if (taken || rc != VDNN_OK) return rc;
                const int rcg = launch_split_general<0>(ctx, st, g, x, w, eps, workspace, workspace_bytes, &taken);
                if (taken || rcg != VDNN_OK) return rcg;
            }
            const int rc = launch_winograd(ctx, st, g, false, x, w, bias, y, relu, nullptr, workspace, workspace_bytes, &taken);
            if (taken || rc != VDNN_OK) return rc;
        }
    }
    if constexpr (sizeof(E) == 4) {
        bool taken = false;
        const int rc = launch_same_x3_fwd(ctx, st, carve, g, x, w, bias, y, relu, &taken);
        if (taken || rc != VDNN_OK) return rc;
    }
    if (g.R * g.S <= 32 && g.C % KB != 0 && pad_pays(g.C, g.K, (long)g.N * g.P * g.Q, g.R * g.S, kPadFwdOps)) {
        // the same with the last block of channels filled up by zeros
        const int RS = g.R * g.S, Kpad = (g.C + KB - 1) / KB * KB * RS;
        const size_t bytes = (size_t)g.K * Kpad * 4;
        if (float* packed = packed_filter_place(ctx, carve, bytes)) {
            const int rc = launch_pack_filter(ctx, st, w, packed, g.K, g.C, RS, g.C * RS, RS);
            if (rc != VDNN_OK) return rc;
            LoadDenseRed<true> alp{packed, (long)Kpad, g.K, (unsigned)bytes};
            LoadIm2colPixTap<0, E, true> bl{{x, g.H, g.W, g.P, g.Q, g.R, g.S, g.ph, g.pw, g.sh, g.sw, (long)g.C * g.H * g.W, g.N, FastDiv::make(RS), FastDiv::make(g.S)}, g.C};
            StoreNCHW<E> ep{y, bias, g.P * g.Q, ctx->reduce_scratch, relu, nullptr};
            return launch_by_m(ctx, st, kFwdNames, alp, bl, ep, g.K, g.N * g.P * g.Q, Kpad, 2.0 * g.K * (double)g.N * g.P * g.Q * K);
        }
    }
    if (g.R * g.S <= 32 && g.C % KB == 0) {
        // blocked tap-major reduction: one slice = one tap x 16 input channels
        const int RS = g.R * g.S;
        LoadIm2colPixTap<0, E> bl{{x, g.H, g.W, g.P, g.Q, g.R, g.S, g.ph, g.pw, g.sh, g.sw, (long)g.C * g.H * g.W, g.N,
                                FastDiv::make(RS), FastDiv::make(g.S)}};
        // The filter bank re-laid-out in the blocked tap-major order is a dense operand read with 128-bit loads (in the
        // master copy's order a slice's sixteen channels of one tap lie R*S floats apart). Perf-optimal: in the
        // workspace. Memory-optimal: at the front of the context's staging area, where it leaves room for the partial sums.
        const bool in_workspace = algo_mode == 1 && workspace && workspace_bytes >= wbytes && aligned16(workspace);
        if (RS == 1 && aligned16(w)) { // one tap: the filter is laid out as it is packed
            StoreNCHW<E> ep{y, bias, g.P * g.Q, ctx->reduce_scratch, relu, nullptr};
            LoadDenseRed<true> al{w, (long)K, g.K, wbytes};
            return launch_by_m(ctx, st, in_workspace ? kFwdPackedNames : kFwdNames, al, bl, ep, g.K, g.N * g.P * g.Q, K);
        }
        float* packed = pack_pays(2.0 * g.K * (double)g.N * g.P * g.Q * K, RS) ? (in_workspace ? (float*)workspace : packed_filter_place(ctx, carve, wbytes)) : nullptr;
        StoreNCHW<E> ep{y, bias, g.P * g.Q, ctx->reduce_scratch, relu, nullptr};
        if (packed) {
            const int rc = launch_pack_filter(ctx, st, w, packed, g.K, g.C, RS, g.C * RS, RS);
            if (rc != VDNN_OK) return rc;
            LoadDenseRed<true> alp{packed, (long)K, g.K, wbytes};
            return launch_by_m(ctx, st, in_workspace ? kFwdPackedNames : kFwdNames, alp, bl, ep, g.K, g.N * g.P * g.Q, K);
        }
        LoadFilterTap<false> al{w, g.C * RS, RS, g.K, RS, wbytes, FastDiv::make(RS)};
        return launch_by_m(ctx, st, kFwdNames, al, bl, ep, g.K, g.N * g.P * g.Q, K);
    }
    if (K % 4 == 0 && aligned16(w)) {
        LoadDenseRed<true> al{w, (long)K, g.K, wbytes};
        return conv_fwd_with(ctx, st, g, al, x, bias, y, relu);
    }
    LoadDenseRed<false> al{w, (long)K, g.K, wbytes};
    return conv_fwd_with(ctx, st, g, al, x, bias, y, relu);
}

// The kernels that a stride-1 layer with more than four input channels takes store through StoreNCHW or one of the
// split reductions: a lane reads the gate's element before it writes the gradient's, and no kernel reads the layer's
// input otherwise. (Layers that are one dense product are left out: their filter gradient is as large as the filter.)
static bool conv_bwd_data_in_place_ok(const ConvGeo& g) {
    return g.sh == 1 && g.sw == 1 && g.C > 4 && !is_dense(g);
}

// The row kernel of 3x3 layers of up to three channels (conv_smallc_mfma.h): about three workgroups per compute unit, strips of at least eight image rows
struct RowStrips { int rows, strips, cblocks; };
static RowStrips row_strips(const ConvGeo& g, int num_cu) {
    RowStrips r;
    r.cblocks = (g.W + BDS_EMIT - 1) / BDS_EMIT;
    const long per_row = (long)g.N * r.cblocks;
    r.strips = (int)((3l * num_cu + per_row - 1) / per_row);
    r.rows = (g.H + r.strips - 1) / r.strips;
    // a strip forms the products of two rows beyond its own, so eight or more of its own - unless that leaves units idle:
    // then the walk down a strip is the kernel's whole time (4 x 3 x 20 x 20, 8 filters: 20.8 -> 10.1 us with strips of two rows)
    const int fill = (int)((per_row * g.H + num_cu - 1) / num_cu);
    const int least = fill >= 8 ? 8 : fill < 2 ? 2 : fill;
    if (r.rows < least) r.rows = least;
    if (r.rows > g.H) r.rows = g.H;
    r.strips = (g.H + r.rows - 1) / r.rows;
    return r;
}

// Samples whose products of all taps the staging area holds at a time (32-bit indexes in the kernel that gathers them)
static int gather_samples(const vdnn_ctx* ctx, const ConvGeo& g) {
    const long fit = (long)(ctx->reduce_scratch_bytes / ((size_t)g.C * g.R * g.S * g.P * g.Q * sizeof(float))), indexes = (1l << 31) / ((long)g.C * g.H * g.W);
    const long n = fit < indexes ? fit : indexes;
    return (int)(n < g.N ? n : g.N);
}

// Gated backward data of up to four input channels: whether the products of all taps once and a gather (rows3: the row kernel) are faster than the
// product of C rows over every (filter, tap), which wastes 61 of a tile's 64 rows but reads little when there are few filters. Estimates in us, by
// that product's own (one) and least squares over 5174 drawn calls of 1 to 256 filters of 2x2 to 11x11, strides 1 to 4, timed both ways; the gather waits
// for the taps that reach a pixel one after the other, 0.3 us each. Of 1422 calls at stride 1, 524 take the products, 2.7 times as fast as the
// product of C rows in the mean (one more than 5 % slower; 753 where all of them took the products); of 258 for the row kernel 55, 2.2 times (none;
// 146); of 3494 strided ones 3200, 3.5 times (21; 175). The choice is 1.1 %, 2.1 % and 0.4 % behind the faster route. Up to eight filters at
// stride 1 never gained: 87 x 3 x 190 x 190, 2 of 11x11 1054 us, 5875 by the products; 75 x 2 x 138 x 5, 4 of 3x3 11.7, 88.6 by the row kernel.
static bool gated_products_pay(const vdnn_ctx* ctx, const ConvGeo& g, bool rows3) {
    const int RS = g.R * g.S, PQ = g.P * g.Q;
    const bool s1 = g.sh == 1 && g.sw == 1;
    if (s1 && g.K <= 8) return false;
    const double one = pixel_product_us(g.C, g.N * g.H * g.W, g.K * RS, ctx->reduce_scratch_bytes, ctx->num_cu, s1 ? 1.25 : 4.0, s1 ? 1.15 : 2.0);
    const double one_us = s1 ? 1.8 + 0.785 * one : RS < 9 ? 4.0 + 0.24 * one : RS <= 32 ? 2.7 + 0.36 * one : 0.67 * one;
    if (rows3) {
        const RowStrips r = row_strips(g, ctx->num_cu);
        const long rounds = ((long)g.N * r.strips * r.cblocks + 3l * ctx->num_cu - 1) / (3l * ctx->num_cu);
        return 2.55 * (double)rounds * (r.rows + 2) < 0.8 * one_us;
    }
    const int nb = gather_samples(ctx, g), chunks = (g.N + nb - 1) / nb;
    const double products = pixel_product_us(g.C * RS, nb * PQ, g.K, 0, ctx->num_cu, 1.25, 1.15) * g.N / nb;
    const double reach = (double)((g.R + g.sh - 1) / g.sh) * ((g.S + g.sw - 1) / g.sw), mb = 4e-6 * g.N * (double)g.C * RS * PQ;
    return 0.575 * products + 0.05 * mb + chunks * (5.3 + 0.3 * reach) < (s1 ? 0.9 : 1.0) * one_us;
}

template <class E>
static int conv_bwd_data_impl(vdnn_ctx* ctx, vdnn_stream_t stream, const vdnn_shape_t* shape, int algo_mode,
                              const E* dy, const float* w, E* dx,
                              void* workspace, size_t workspace_bytes, const E* gate) {
    VDNN_KERNEL_PROLOGUE(ctx);
    ConvGeo g;
    VDNN_REQUIRE(shape && geo_from_shape(shape, g), "unsupported convolution geometry");
    VDNN_REQUIRE(dy && w && dx, "null tensor");
    VDNN_REQUIRE((const void*)dx != (const void*)dy, "the input gradient cannot be written over the output gradient");
    VDNN_REQUIRE((const void*)dx != (const void*)gate || conv_bwd_data_in_place_ok(g),
                 "the input gradient may be written over the gating input only where vdnn_conv_bwd_data_in_place_ok says so");
    if (is_dense(g))
        return gate ? vdnn_fc_bwd_data_relu(ctx, stream, g.N, g.C * g.H * g.W, g.K, dy, w, gate, dx)
                    : vdnn_fc_bwd_data(ctx, stream, g.N, g.C * g.H * g.W, g.K, dy, w, dx);
    hipStream_t st = stream_of(ctx, stream);
    StagingCarve carve(ctx);
    // Up to four input channels. As a product of C rows the reduction over (k, r, s) fills 3 of a tile's 64 rows (and of a strided layer 16 of
    // 121 taps); the products w * dy of all taps as rows of a 1x1 convolution fill C*R*S of them, each computed once, and a second kernel adds
    // them up and gates. Whole gated backward passes of 3 channels, product of C rows -> here: 23 x 176 x 176, 160 filters of 11x11 at stride 4 27.7 ms ->
    // 0.19; 14 x 128 x 128, 594 of 5x5 3.69 -> 0.81; 25 x 86 x 86, 64 of 3x3 222 us -> 140; bfloat16 8 x 87 x 87, 323 of 11x11 at stride 4 5.5 ms -> 0.06.
    // Gated layers that keep the product of C rows: 1x1 windows (nothing to save: 108 x 20 x 20, 512 filters 73 us, 97 here) and bfloat16 at
    // stride 1, where that product runs on the bfloat16 matrix cores (10 x 132 x 132, 26 of 3x3 57 us, 66 here; 28 x 141 x 141, 128 373, 317).
    const bool rows3 = g.C <= 3 && g.K <= 64 && g.R == 3 && g.S == 3 && g.ph == 1 && g.pw == 1 && g.sh == 1 && g.sw == 1 && (long)g.K * g.P * g.Q * (long)sizeof(E) < (long)MAX_SUM_RANGE;
    // (the rounded filter of a bfloat16 layer lies in the staging area too; a gated layer whose filter does not fit keeps the other route)
    const size_t filter_bytes = (size_t)g.K * g.C * g.R * g.S * sizeof(float), rounded_bytes = sizeof(E) == 2 ? (filter_bytes + 255) / 256 * 256 : 0;
    const bool products = g.C <= 4 && g.R * g.S <= SMALLC_MAXTAPS && ctx->reduce_scratch &&
                          ctx->reduce_scratch_bytes >= rounded_bytes + (size_t)g.C * g.R * g.S * g.P * g.Q * sizeof(float) &&
                          (!gate || !rounded_bytes || filter_bytes + (8u << 20) <= ctx->reduce_scratch_bytes) &&
                          pixel_tile_span_ok((long)g.K * g.P * g.Q, g.P * g.Q, 256, (int)sizeof(E));
    const bool few_channels = g.C <= 4 && g.R * g.S <= SMALLC_MAXTAPS &&
                              (!gate || (g.R * g.S > 1 && (sizeof(E) == 4 || g.sh > 1 || g.sw > 1) && (rows3 || products) && gated_products_pay(ctx, g, rows3)));
    if (!few_channels && (g.sh != 1 || g.sw != 1)) {
        bool taken = false;
        const int rc = launch_strided_bwd_data<E>(ctx, st, g, dy, w, dx, gate, &taken);
        if (taken || rc != VDNN_OK) return rc;
    }
    bool half_engine = false;
    const LoadIm2colPix<1, false, E> pix{dy, g.P, g.Q, g.H, g.W, g.R, g.S, g.ph, g.pw, 1, 1, (long)g.K * g.P * g.Q, g.N, FastDiv::make(g.R * g.S), FastDiv::make(g.S)};
    if constexpr (sizeof(E) == 2) {
        half_engine = !few_channels && g.sh == 1 && g.sw == 1 && half_engine_ok(ctx, pix, g.K, g.C, g.R * g.S);
        if (!half_engine) {
            w = rounded_filter_copy(ctx, st, carve, w, (size_t)g.K * g.C * g.R * g.S);
            VDNN_REQUIRE(w != nullptr, "filter too large for the staging area (bfloat16 layer outside the bfloat16 engine)");
            VDNN_LAUNCH_CHECK();
        }
    }
    if (few_channels) {
        const bool s1 = g.sh == 1 && g.sw == 1;
        if (products && (s1 ? gate && !rows3 : true)) {
            // The products once, into the staging area, gathered into dx by a second kernel; as many samples at a time as the
            // staging area holds.
            const int RS = g.R * g.S, CRS = g.C * RS, PQ = g.P * g.Q;
            const size_t per_sample = (size_t)CRS * PQ * sizeof(float);
            const int nb = gather_samples(ctx, g);
            float* T = ctx->reduce_scratch;
            LoadFilterT alt{w, CRS, 1, (unsigned)((long)g.K * CRS * 4), FastDiv::make(1)};
            for (int n0 = 0; n0 < g.N; n0 += nb) {
                const int nc = g.N - n0 < nb ? g.N - n0 : nb;
                LoadIm2colPix<0, false, E> bl{dy + (long)n0 * g.K * PQ, g.P, g.Q, g.P, g.Q, 1, 1, 0, 0, 1, 1, (long)g.K * PQ, nc,
                                              FastDiv::make(1), FastDiv::make(1)};
                StoreNCHW<float> ept{T, nullptr, PQ, nullptr, 0, nullptr};
                const int rc = launch_by_m(ctx, st, kBwdDataNames, alt, bl, ept, CRS, nc * PQ, g.K, 2.0 * nc * (double)g.K * CRS * PQ);
                if (rc != VDNN_OK) return rc;
                ConvGeo gc = g; gc.N = nc;
                const long total = (long)nc * g.C * g.H * g.W, first = (long)n0 * g.C * g.H * g.W;
                ProfScope gather(ctx, st, "conv_bwd_data_gather", 0.0, (double)per_sample * nc + (double)total * sizeof(E) * (gate ? 2.0 : 1.0));
                hipLaunchKernelGGL(conv_bwd_data_gather_taps_kernel<E>, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st,
                                   T, dx + first, gate ? gate + first : nullptr, gc, (unsigned)total);
                VDNN_LAUNCH_CHECK();
            }
            return VDNN_OK;
        }
        const long total = (long)g.N * g.H * g.W;
        const long blocks = (total + 255) / 256;
        VDNN_REQUIRE(blocks < (1l << 31), "grid too large");
        ProfScope prof(ctx, st, "conv_bwd_data_smallc", 2.0 * g.C * (double)g.N * g.P * g.Q * g.K * g.R * g.S, 0.0);
        const bool s1_3x3 = g.sh == 1 && g.sw == 1 && g.R == 3 && g.S == 3;
        // 3x3, padding 1, at most three input and 64 output channels: the products once, on the matrix cores, row by row
        if (rows3) {
            const RowStrips strip = row_strips(g, ctx->num_cu);
            const int rows = strip.rows;
            const dim3 grid((unsigned)(g.N * strip.strips * strip.cblocks));
            if (g.C == 1) hipLaunchKernelGGL((conv_bwd_data_smallc3x3_mfma_kernel<1, E>), grid, dim3(256), 0, st, dy, w, dx, gate, g.N, g.K, g.H, g.W, rows);
            else if (g.C == 2) hipLaunchKernelGGL((conv_bwd_data_smallc3x3_mfma_kernel<2, E>), grid, dim3(256), 0, st, dy, w, dx, gate, g.N, g.K, g.H, g.W, rows);
            else hipLaunchKernelGGL((conv_bwd_data_smallc3x3_mfma_kernel<3, E>), grid, dim3(256), 0, st, dy, w, dx, gate, g.N, g.K, g.H, g.W, rows);
            VDNN_LAUNCH_CHECK();
            return VDNN_OK;
        }
        if (s1_3x3 && g.C == 3) hipLaunchKernelGGL((conv_bwd_data_smallc_s1_kernel<3, 3, 3, E>), dim3((unsigned)blocks), dim3(256), 0, st, dy, w, dx, g);
        else if (s1_3x3 && g.C == 4) hipLaunchKernelGGL((conv_bwd_data_smallc_s1_kernel<3, 3, 4, E>), dim3((unsigned)blocks), dim3(256), 0, st, dy, w, dx, g);
        else if (g.sh == 1 && g.sw == 1) hipLaunchKernelGGL(conv_bwd_data_smallc_kernel<E>, dim3((unsigned)blocks), dim3(256), 0, st, dy, w, dx, g);
        else {
            // one workgroup per 256 pixels of one (sample, residue class modulo the stride)
            const int Ht = (g.H + g.ph + g.sh - 1) / g.sh, Wt = (g.W + g.pw + g.sw - 1) / g.sw;
            const long per_class = ((long)Ht * Wt + 255) / 256;
            const long sblocks = per_class * g.sh * g.sw * g.N;
            VDNN_REQUIRE(sblocks < (1l << 31), "grid too large");
            hipLaunchKernelGGL(conv_bwd_data_smallc_strided_kernel<E>, dim3((unsigned)sblocks), dim3(256), 0, st, dy, w, dx, g, Ht, Wt, (int)per_class);
        }
        VDNN_LAUNCH_CHECK();
        return VDNN_OK;
    }
    VDNN_REQUIRE(pixel_tile_span_ok((long)g.K * g.P * g.Q, g.H * g.W, 256, (int)sizeof(E)), "output-gradient samples too large for one tile's descriptor");
    if constexpr (sizeof(E) == 4) {
        if (algo_mode == 1) {
            bool taken = false;
            if (g_perf_variant == 0) {
                const StoreNCHW<float> eps{dx, nullptr, g.H * g.W, ctx->reduce_scratch, 0, gate};
                const int rc = launch_split3x3<1>(ctx, st, g, dy, w, eps, workspace, workspace_bytes, &taken);
                if (taken || rc != VDNN_OK) return rc;
                const int rcg = launch_split_general<1>(ctx, st, g, dy, w, eps, workspace, workspace_bytes, &taken);
                if (taken || rcg != VDNN_OK) return rcg;
            }
            const int rc = launch_winograd(ctx, st, g, true, dy, w, nullptr, dx, 0, gate, workspace, workspace_bytes, &taken);
            if (taken || rc != VDNN_OK) return rc;
        }
    }
    if constexpr (sizeof(E) == 4) {
        bool taken = false;
        const int rc = launch_same_x3_bwd_data(ctx, st, carve, g, dy, w, dx, gate, &taken);
        if (taken || rc != VDNN_OK) return rc;
    }
    const int RS = g.R * g.S;
    LoadFilterT al{w, g.C, RS, (unsigned)((long)g.K * g.C * RS * 4), FastDiv::make(RS)};
    StoreNCHW<E> ep{dx, nullptr, g.H * g.W, ctx->reduce_scratch, 0, gate};
    const int M = g.C, N = g.N * g.H * g.W, K = g.K * RS;
    const FastDiv dRS = FastDiv::make(RS), dS = FastDiv::make(g.S);
    const long sample = (long)g.K * g.P * g.Q;
    const double flops = 2.0 * g.N * (double)g.K * g.C * RS * g.P * g.Q;
    if constexpr (sizeof(E) == 2) {
        if (half_engine) {
            return conv_half_engine<1>(ctx, st, kBwdDataHalfNames, w, g.C, g.K, RS, RS, g.C * RS, pix, ep, N, flops);
        }
    }
    if (g.sh == 1 && g.sw == 1) {
        if (RS <= 32 && g.K % KB == 0) {
            // blocked tap-major reduction: one slice = one tap x 16 output channels
            const unsigned wbytes = (unsigned)((long)g.K * g.C * RS * 4);
            LoadIm2colPixTap<1, E> bl{{dy, g.P, g.Q, g.H, g.W, g.R, g.S, g.ph, g.pw, 1, 1, sample, g.N, dRS, dS}};
            const bool in_workspace = algo_mode == 1 && workspace && workspace_bytes >= wbytes && aligned16(workspace);
            if (RS == 1) { // one tap: the filter read as it lies, lanes along the input channels
                LoadDenseRow<float> alr{w, (long)g.C, g.C, wbytes};
                return launch_by_m(ctx, st, in_workspace ? kBwdDataPackedNames : kBwdDataNames, alr, bl, ep, M, N, K, flops);
            }
            float* packed = pack_pays(2.0 * M * (double)N * K, RS) ? (in_workspace ? (float*)workspace : packed_filter_place(ctx, carve, wbytes)) : nullptr; // [c][(kb*RS + tap)*16 + l]
            if (packed) {
                ep.partial = ctx->reduce_scratch; // (behind the filter bank, if that lies in the staging area)
                const int rc = launch_pack_filter(ctx, st, w, packed, g.C, g.K, RS, RS, g.C * RS);
                if (rc != VDNN_OK) return rc;
                LoadDenseRed<true> alp{packed, (long)K, g.C, wbytes};
                return launch_by_m(ctx, st, in_workspace ? kBwdDataPackedNames : kBwdDataNames, alp, bl, ep, M, N, K, flops);
            }
            LoadFilterTap<true> alt{w, RS, g.C * RS, g.C, RS, wbytes, dRS};
            return launch_by_m(ctx, st, kBwdDataNames, alt, bl, ep, M, N, K, flops);
        }
        if (RS <= 32 && g.K % KB != 0 && pad_pays(g.K, M, N, RS, kPadBwdDataOps)) {
            const int Kpad = (g.K + KB - 1) / KB * KB * RS;
            const size_t bytes = (size_t)g.C * Kpad * 4;
            if (float* packed = packed_filter_place(ctx, carve, bytes)) {
                ep.partial = ctx->reduce_scratch;
                const int rc = launch_pack_filter(ctx, st, w, packed, g.C, g.K, RS, RS, g.C * RS);
                if (rc != VDNN_OK) return rc;
                LoadDenseRed<true> alp{packed, (long)Kpad, g.C, (unsigned)bytes};
                LoadIm2colPixTap<1, E, true> bl{{dy, g.P, g.Q, g.H, g.W, g.R, g.S, g.ph, g.pw, 1, 1, sample, g.N, dRS, dS}, g.K};
                return launch_by_m(ctx, st, kBwdDataNames, alp, bl, ep, M, N, Kpad, flops);
            }
        }
        if (RS <= 32) {
            LoadIm2colPix<1, false, E> bl{dy, g.P, g.Q, g.H, g.W, g.R, g.S, g.ph, g.pw, 1, 1, sample, g.N, dRS, dS};
            return launch_by_m(ctx, st, kBwdDataNames, al, bl, ep, M, N, K, flops);
        }
        LoadIm2colPix<1, true, E> bl{dy, g.P, g.Q, g.H, g.W, g.R, g.S, g.ph, g.pw, 1, 1, sample, g.N, dRS, dS};
        return launch_by_m(ctx, st, kBwdDataNames, al, bl, ep, M, N, K, flops);
    }
    LoadIm2colPix<2, true, E> bl{dy, g.P, g.Q, g.H, g.W, g.R, g.S, g.ph, g.pw, g.sh, g.sw, sample, g.N, dRS, dS};
    return launch_by_m(ctx, st, kBwdDataNames, al, bl, ep, M, N, K, flops);
}

// out = (accumulate ? out : 0) + alpha * dW; the bias gradient too where the chosen kernel can (bias->done)
template <class E>
static int conv_bwd_filter_core(vdnn_ctx* ctx, vdnn_stream_t stream, const vdnn_shape_t* shape, int algo_mode,
                                const E* x, const E* dy, float* w, float alpha, int accumulate,
                                void* workspace, size_t workspace_bytes, BiasOut* bias) {
    VDNN_KERNEL_PROLOGUE(ctx);
    ConvGeo g;
    VDNN_REQUIRE(shape && geo_from_shape(shape, g), "unsupported convolution geometry");
    VDNN_REQUIRE(x && dy && w, "null tensor");
    if (is_dense(g))
        return accumulate ? vdnn_fc_bwd_weight_sgd(ctx, stream, g.N, g.C * g.H * g.W, g.K, x, dy, w, alpha)
                          : vdnn_fc_bwd_weight(ctx, stream, g.N, g.C * g.H * g.W, g.K, x, dy, w);
    hipStream_t st = stream_of(ctx, stream);
    const int M = g.K, N = g.C * g.R * g.S, PQ = g.P * g.Q, RS = g.R * g.S;
    const long Kred = (long)g.N * PQ;
    VDNN_REQUIRE(Kred < (1l << 31), "reduction too long");
    VDNN_REQUIRE((long)(PQ + KB) * PQ < (1l << 32), "output plane too large for the pixel cursor's exact division");
    if constexpr (sizeof(E) == 4) {
        if (algo_mode == 1) {
            // perf-optimal: 3x3 layers on the bfloat16 matrix cores (partial sums in the staging area, or in the workspace
            // if that is larger), or as Winograd F(3x3, 4x4) through the workspace
            bool taken = false;
            if (g_perf_variant == 0 && wgrad3x3_ok(g)) {
                float* staging = ctx->reduce_scratch;
                size_t staging_bytes = ctx->reduce_scratch_bytes;
                if (workspace && workspace_bytes > staging_bytes && aligned16(workspace)) { staging = (float*)workspace; staging_bytes = workspace_bytes; }
                const int rcs = launch_wgrad3x3_split(ctx, st, g, x, dy, w, alpha, accumulate, staging, staging_bytes, &taken, bias);
                if (taken || rcs != VDNN_OK) return rcs;
            }
            const int rc = launch_winograd_wgrad(ctx, st, g, x, dy, w, alpha, accumulate, workspace, workspace_bytes, &taken, bias);
            if (taken || rc != VDNN_OK) return rc;
        }
    }
    if (g.C <= 3 && g.R == 3 && g.S == 3 && g.ph == 1 && g.pw == 1 && g.sh == 1 && g.sw == 1 && g.P == g.H && g.Q == g.W && g.W % 4 == 0 && g.W >= KB &&
        ctx->reduce_scratch) {
        // few input channels, rows of whole groups of four pixels: dy streamed once through the matrix cores, then the ordered split sum
        const int mtiles = (g.K + 63) / 64;
        const size_t out_bytes = (size_t)M * N * sizeof(float);
        long splits = 3l * ctx->num_cu / mtiles;
        // four slices per split or more, unless that leaves units idle (4 x 3 x 20 x 20, 8 filters: 14.8 -> 9.2 us)
        long by_len = Kred / (4 * WSC_SLICE);
        const long by_mem = (long)(ctx->reduce_scratch_bytes / out_bytes), one_round = ctx->num_cu / mtiles;
        if (by_len < one_round) by_len = Kred / WSC_SLICE < one_round ? Kred / WSC_SLICE : one_round;
        if (splits > by_len) splits = by_len;
        if (splits > by_mem) splits = by_mem;
        if (splits < 1) splits = 1;
        long kchunk = (Kred + splits - 1) / splits;
        kchunk = (kchunk + WSC_SLICE - 1) / WSC_SLICE * WSC_SLICE;
        splits = (Kred + kchunk - 1) / kchunk;
        const long nspan = kchunk / PQ + 2;
        if (PQ >= WSC_SLICE && nspan * g.K * PQ * (long)sizeof(E) < (long)MAX_SUM_RANGE && nspan * g.C * PQ * (long)sizeof(E) < (long)MAX_SUM_RANGE) {
            const bool with_bias = bias && bias->wanted() && bias_parts_fit(ctx, g.K, splits);
            const WgradSmallC geo{dy, x, g.N, g.K, g.H, g.W, ctx->reduce_scratch, (int)kchunk, with_bias ? ctx->bias_scratch : nullptr, (int)splits};
            {
                ProfScope prof(ctx, st, "conv_bwd_filter_smallc", 2.0 * (double)M * N * (double)Kred, 0.0);
                const dim3 grid((unsigned)(mtiles * splits));
                switch (g.C) {
                case 1: hipLaunchKernelGGL((wgrad_smallc3x3_mfma_kernel<1, E>), grid, dim3(NT), 0, st, geo); break;
                case 2: hipLaunchKernelGGL((wgrad_smallc3x3_mfma_kernel<2, E>), grid, dim3(NT), 0, st, geo); break;
                default: hipLaunchKernelGGL((wgrad_smallc3x3_mfma_kernel<3, E>), grid, dim3(NT), 0, st, geo); break;
                }
                VDNN_LAUNCH_CHECK();
            }
            if (with_bias) {
                const int rcb = launch_bias_grad_final(ctx, st, ctx->bias_scratch, bias->out, g.K, (int)splits, bias->alpha, bias->accumulate);
                if (rcb != VDNN_OK) return rcb;
                bias->done = true;
            }
            return launch_reduce_splits(ctx, st, w, ctx->reduce_scratch, (size_t)M * N, (int)splits, alpha, accumulate, nullptr, 0);
        }
    }
    if (g.C <= 4 && g.R == 3 && g.S == 3 && g.K % 4 == 0 && ctx->reduce_scratch) {
        // few input channels: vector-ALU kernel over chunks of output pixels, then the ordered chunk sum
        const long total = Kred;
        const size_t out_bytes = (size_t)M * N * sizeof(float);
        long chunks = (total + 256 * 96 - 1) / (256 * 96);
        // a thread walks its share of a chunk pixel by pixel: on a chip that few chunks leave idle that walk is the whole time
        // (backward 26 x 3 x 50 x 50, 128 of 3x3, no padding: 177 us with the chunks of large layers, 73 with these), down to four pixels a thread
        const long fill = (2l * ctx->num_cu + g.K / 4 - 1) / (g.K / 4), shortest = (total + 4 * 256 - 1) / (4 * 256);
        if (chunks < fill) chunks = fill < shortest ? fill : shortest;
        const long by_mem = (long)(ctx->reduce_scratch_bytes / out_bytes);
        if (chunks > by_mem) chunks = by_mem;
        if (chunks < 1) chunks = 1;
        long per = (total + chunks - 1) / chunks;
        per = (per + 255) / 256 * 256;
        chunks = (total + per - 1) / per;
        const long blocks = chunks * (g.K / 4);
        VDNN_REQUIRE(blocks < (1l << 31), "grid too large");
        const PixelStep step{256 / PQ, (256 % PQ) / g.Q, (256 % PQ) % g.Q};
        float* staging = ctx->reduce_scratch;
        {
            ProfScope prof(ctx, st, "conv_bwd_filter_smallc", 2.0 * (double)M * N * (double)Kred, 0.0);
            switch (g.C) {
            case 1: hipLaunchKernelGGL((conv_bwd_filter_smallc3x3_kernel<1, 4, E>), dim3((unsigned)blocks), dim3(256), 0, st, dy, x, staging, g, per, step); break;
            case 2: hipLaunchKernelGGL((conv_bwd_filter_smallc3x3_kernel<2, 4, E>), dim3((unsigned)blocks), dim3(256), 0, st, dy, x, staging, g, per, step); break;
            case 3: hipLaunchKernelGGL((conv_bwd_filter_smallc3x3_kernel<3, 4, E>), dim3((unsigned)blocks), dim3(256), 0, st, dy, x, staging, g, per, step); break;
            default: hipLaunchKernelGGL((conv_bwd_filter_smallc3x3_kernel<4, 4, E>), dim3((unsigned)blocks), dim3(256), 0, st, dy, x, staging, g, per, step); break;
            }
            VDNN_LAUNCH_CHECK();
        }
        return launch_reduce_splits(ctx, st, w, staging, (size_t)M * N, (int)chunks, alpha, accumulate, nullptr, 0);
    }
    // Split the (n,p,q) reduction so the grid fills the chip; partial sums go to a staging area and
    // are added in split order by a second kernel (no floating-point atomics).
    const bool narrow = M <= 64;
    const int TM = narrow ? 64 : 128, TN = narrow ? 256 : 128;
    const long tiles = (long)((M + TM - 1) / TM) * ((N + TN - 1) / TN);
    float* staging = ctx->reduce_scratch;
    size_t staging_bytes = ctx->reduce_scratch_bytes;
    if (workspace && workspace_bytes > staging_bytes) { staging = (float*)workspace; staging_bytes = workspace_bytes; }
    const size_t out_bytes = (size_t)M * N * sizeof(float);
    const long by_mem = staging ? (long)(staging_bytes / out_bytes) : 1;
    const FilterTilePlan tile_plan = filter_tile_plan(g, staging ? staging_bytes : 0, ctx->num_cu);
    const int want = tile_plan.want;
    const SmallTilePlan& plan = tile_plan.small;
    const bool vec = PQ % 4 == 0 && aligned16(dy); // bf16: four elements are 8 bytes, covered by the same test
    const bool tap_planes = vec && PQ >= KB && 2 * g.Q >= KB; // planes the tap-major loaders take
    // the 64x64 tile; its loaders have a column's tap to work out per element unless a tile's columns share it. Tile and
    // splits go by the shape alone (an aligned dy, filter_tile_plan): they decide the order of the sums, which is not to change with an address
    const bool small_tap = tap_planes && g.C % 32 == 0;
    // one split's samples of dy and of x are addressed through one descriptor with summed offsets
    auto span_ok = [&](int kchunk) {
        const long nspan = kchunk / PQ + 2;
        return nspan * g.K * PQ * (long)sizeof(E) < (long)MAX_SUM_RANGE && nspan * g.C * g.H * g.W * (long)sizeof(E) < (long)MAX_SUM_RANGE;
    };
    const GemmDims d_small = make_dims(M, N, (int)Kred, 64, 64, plan.splits);
    // Rows that end in the first half of a 128-row tile leave a 64-row tile less to multiply for nothing than the estimates see
    // (21 x 70 x 53 x 37, 130 of 3x3 at stride 2 54 -> 50 us, 16 x 100 x 40 x 40 51 -> 46, 10 x 33 x 60 x 60, 150 of 5x5 62 -> 57). Of 900 drawn calls of 65 to 704
    // filters some 290 change their tile for it, by 12 % faster in the mean and 4 % slower at most; up to 1.12 of the estimate and 3e10 operations 210 do, some slower (14 x 10 x 56 x 56, 294
    // of 7x7 at stride 2 56 -> 61, 79 x 128 x 14 x 14, 565 of 3x3 150 -> 169). Small products go by the estimates, which are right there (2 x 16 x 8 x 8,
    // 275 of 3x3 10.7 us, 12.5 in the other tile).
    const double half_ops = 2.0 * M * (double)N * (double)Kred;
    const bool half_tile = !narrow && M % TM != 0 && M % TM <= 64 && half_ops >= 5e8 && half_ops <= 1e10;
    const bool small = (Kred <= kShortReduction || (2.0 * M * (double)N * (double)Kred <= kSmallTileOps &&
                                                    plan.us < (half_tile ? 1.07 : 0.9) * tile_plan.large_us)) &&
                       span_ok(d_small.kchunk);
    const GemmDims d = small ? d_small : make_dims(M, N, (int)Kred, TM, TN, want);
    VDNN_REQUIRE(span_ok(d.kchunk), "samples of one reduction split too large for one descriptor");
    StoreDense<float> ep{w, staging, nullptr, (long)N, (long)M * N, alpha, accumulate};
    const FastDiv dRS = FastDiv::make(RS), dS = FastDiv::make(g.S), dQ = FastDiv::make(g.Q), dPQ = FastDiv::make(PQ);
    // tap-major column order when the tile's columns fall into whole groups of channels with one tap each
    const int tile_n = narrow ? 256 : 128;
    const int ntap = g.C % tile_n == 0 ? 1 : (g.C % (tile_n / 2) == 0 ? 2 : (g.C % (tile_n / 4) == 0 ? 4 : 0));
    if constexpr (sizeof(E) == 2) {
        // bfloat16 activations: both factors of every product are bfloat16 already
        if (wgrad3x3_ok(g)) { // loads of eight pixels take any alignment of the tensors
            bool taken = false;
            const int rcw = launch_wgrad3x3(ctx, st, g, x, dy, w, alpha, accumulate, staging, staging_bytes, &taken, bias);
            if (taken || rcw != VDNN_OK) return rcw;
        }
        if (vec && ntap != 0 && PQ >= KH && 3 * g.Q >= KH && g.Q % 2 == 0 && ((uintptr_t)x & 3) == 0 && staging) {
            long caph = (Kred + 4 * KH - 1) / (4 * KH);
            if (caph > by_mem) caph = by_mem;
            const int wanth = choose_splits(tiles, Kred, caph, ctx->num_cu, out_bytes, 2.0 * TM * TN * KB);
            GemmDims dh = make_dims(M, N, (int)Kred, TM, TN, wanth, KH);
            const long nspanh = dh.kchunk / PQ + 2;
            if (nspanh * g.K * PQ * 2 < (long)MAX_SUM_RANGE && nspanh * g.C * g.H * g.W * 2 < (long)MAX_SUM_RANGE) {
                const FastDiv dC = FastDiv::make(g.C);
                StoreFilterTap ept{w, staging, g.C, RS, (long)M * N, alpha, accumulate, dC};
                LoadDyRedIncH al{dy, g.N, g.K, PQ, dh.kchunk, dh.K};
                int rch;
                // 3x3, stride 1, padding 1, channel counts the kernel above does not take: a tap's im2col operand is the plane
                // shifted by a constant, fetched in groups of four pixels when the image rows are whole groups
                const int vg = g.W % 4 == 0 ? 4 : 0;
                const int tap_cols = tile_n / ntap; // columns of the tile that share a tap
                if (g.R == 3 && g.S == 3 && g.ph == 1 && g.pw == 1 && g.sh == 1 && g.sw == 1 && g.P == g.H && g.Q == g.W && PQ % 8 == 0 &&
                    vg != 0 && tap_cols % (8 * vg) == 0 && (long)g.C * g.H * g.W * 2 < (long)MAX_SUM_RANGE) {
                    LoadDyRedVecH<8> alv{dy, g.N, g.K, PQ, dh.kchunk, dh.K};
                    LoadIm2colRedTapVecH<1, 4> geo{x, g.N, g.C, g.H, g.W, N, dh.kchunk, dh.K, dC};
                    rch = narrow ? launch_wgrad_vec<64, 256>(ctx, st, kBwdFilterHalfNames.t64, alv, geo, ept, dh, ntap, vg)
                                 : launch_wgrad_vec<128, 128>(ctx, st, kBwdFilterHalfNames.t128, alv, geo, ept, dh, ntap, vg);
                    if (rch != VDNN_OK) return rch;
                    if (dh.splits > 1) return launch_reduce_splits_tap(ctx, st, w, staging, (size_t)M * N, dh.splits, alpha, accumulate, g.C, RS);
                    return VDNN_OK;
                }
#define VDNN_WGRAD_TAP_H(NTAP)                                                                                              \
                do {                                                                                                        \
                    if (g.sw == 1 && g.W >= 2) {                                                                                      \
                        LoadIm2colRedTapH<NTAP, true> bl{x, g.N, g.C, g.H, g.W, g.R, g.S, g.P, g.Q, g.ph, g.pw, g.sh, g.sw, N, dh.kchunk, dh.K, dC, dS}; \
                        rch = narrow ? launch_igemm<64, 256, LoadDyRedIncH, LoadIm2colRedTapH<NTAP, true>, StoreFilterTap, true>(ctx, st, kBwdFilterHalfNames.t64, al, bl, ept, dh) \
                                     : launch_igemm<128, 128, LoadDyRedIncH, LoadIm2colRedTapH<NTAP, true>, StoreFilterTap, true>(ctx, st, kBwdFilterHalfNames.t128, al, bl, ept, dh); \
                        break;                                                                                              \
                    }                                                                                                       \
                    LoadIm2colRedTapH<NTAP> bl{x, g.N, g.C, g.H, g.W, g.R, g.S, g.P, g.Q, g.ph, g.pw, g.sh, g.sw, N, dh.kchunk, dh.K, dC, dS}; \
                    rch = narrow ? launch_igemm<64, 256, LoadDyRedIncH, LoadIm2colRedTapH<NTAP>, StoreFilterTap, true>(ctx, st, kBwdFilterHalfNames.t64, al, bl, ept, dh) \
                                 : launch_igemm<128, 128, LoadDyRedIncH, LoadIm2colRedTapH<NTAP>, StoreFilterTap, true>(ctx, st, kBwdFilterHalfNames.t128, al, bl, ept, dh); \
                } while (0)
                if (ntap == 1) VDNN_WGRAD_TAP_H(1);
                else if (ntap == 2) VDNN_WGRAD_TAP_H(2);
                else VDNN_WGRAD_TAP_H(4);
#undef VDNN_WGRAD_TAP_H
                if (rch != VDNN_OK) return rch;
                if (dh.splits > 1) return launch_reduce_splits_tap(ctx, st, w, staging, (size_t)M * N, dh.splits, alpha, accumulate, g.C, RS);
                return VDNN_OK;
            }
        }
    }
    if constexpr (sizeof(E) == 2) {
        // Every other plane of at least four pixels a row: output rows padded to groups of four pixels. Layers too small for
        // this engine's 128x128 and 64x256 tiles stay on the float engine, whose 64x64 tiles fill the chip with them (5 x 26 x 32
        // x 32, 5 filters of 3x3 at stride 2: 20.0 us here, 8.0 there). The lines, operations with less than a tile's 64 filters counting
        // for more, are those of least loss over 2060 calls timed on both: 0.6 % behind the better route in the mean, 24 % with
        // this one for all.
        const PixelGroupStep step = PixelGroupStep::make(g.P, g.Q);
        const long Kpad = (long)g.N * g.P * step.QG * 4, per = 4l * g.P * step.QG;
        const bool unit = g.sw == 1 && g.W >= 4;
        const bool pays = 2.0 * M * (double)N * (double)Kred * (narrow ? std::sqrt(64.0 / M) : 1.0) >= (unit ? 2e8 : 3e8);
        if (pays && g.Q >= 4 && Kpad < (1l << 31) - 4 * KH) {
            long caph = (Kpad + 4 * KH - 1) / (4 * KH); // at least four slices per split
            if (caph > by_mem) caph = by_mem;
            const int wanth = choose_splits(tiles, Kpad, caph, ctx->num_cu, out_bytes, 2.0 * TM * TN * KB);
            const GemmDims dh = make_dims(M, N, (int)Kpad, TM, TN, wanth, KH);
            const long nspanh = dh.kchunk / per + 2 + KH / per; // a slice past the end of a range is fetched and not used
            if (nspanh * g.K * PQ * 2 < (long)MAX_SUM_RANGE && nspanh * g.C * g.H * g.W * 2 < (long)MAX_SUM_RANGE) {
                const LoadDyRowH al{dy, g.N, g.K, g.P, g.Q, dh.kchunk, dh.K, step};
                int rch;
#define VDNN_WGRAD_ROW_H(UNIT)                                                                                              \
                do {                                                                                                        \
                    const LoadIm2colRowH<UNIT> bl{x, g.N, g.C, g.H, g.W, g.R, g.S, g.P, g.Q, g.ph, g.pw, g.sh, g.sw, N, dh.kchunk, dh.K, dRS, dS, step}; \
                    rch = narrow ? launch_igemm<64, 256, LoadDyRowH, LoadIm2colRowH<UNIT>, StoreDense<float>, true>(ctx, st, kBwdFilterHalfNames.t64, al, bl, ep, dh) \
                                 : launch_igemm<128, 128, LoadDyRowH, LoadIm2colRowH<UNIT>, StoreDense<float>, true>(ctx, st, kBwdFilterHalfNames.t128, al, bl, ep, dh); \
                } while (0)
                if (unit) VDNN_WGRAD_ROW_H(true);
                else VDNN_WGRAD_ROW_H(false);
#undef VDNN_WGRAD_ROW_H
                if (rch != VDNN_OK) return rch;
                if (dh.splits > 1) return launch_reduce_splits(ctx, st, w, staging, (size_t)M * N, dh.splits, alpha, accumulate, nullptr, 0);
                return VDNN_OK;
            }
        }
    }
    if constexpr (sizeof(E) == 4) {
        bool taken = false;
        const int rcs = launch_wgrad_same_x3(ctx, st, g, x, dy, w, alpha, accumulate, staging, staging_bytes, &taken, bias);
        if (taken || rcs != VDNN_OK) return rcs;
    }
    if constexpr (sizeof(E) == 4) {
        // 3x3, stride 1, padding 1: one filter row and 64 input channels per workgroup, one fetch for three taps
        if (wgrad3x3_f32_ok(g)) { // loads of four pixels take any alignment of the tensors
            bool taken = false;
            const int rcw = launch_wgrad3x3_f32(ctx, st, g, x, dy, w, alpha, accumulate, staging, staging_bytes, &taken, bias);
            if (taken || rcw != VDNN_OK) return rcw;
        }
    }
    if (small ? small_tap : tap_planes && ntap != 0) {
        const FastDiv dC = FastDiv::make(g.C);
        StoreFilterTap ept{w, staging, g.C, RS, (long)M * N, alpha, accumulate, dC};
        LoadDyRedInc<E> al{dy, g.N, g.K, PQ, d.kchunk, d.K};
        int rc2;
#define VDNN_WGRAD_TAP(NTAP)                                                                                                \
        do {                                                                                                                \
            LoadIm2colRedTap<NTAP, E> bl{x, g.N, g.C, g.H, g.W, g.R, g.S, g.P, g.Q, g.ph, g.pw, g.sh, g.sw, N, d.kchunk, d.K, dC, dS}; \
            rc2 = narrow ? launch_igemm<64, 256>(ctx, st, kBwdFilterNames.t64, al, bl, ept, d)                               \
                         : launch_igemm<128, 128>(ctx, st, kBwdFilterNames.t128, al, bl, ept, d);                            \
        } while (0)
        if (small) {
            if (g.C % 64 == 0) rc2 = launch_wgrad_tap_small<1, E>(ctx, st, g, al, x, ept, d, dS);
            else rc2 = launch_wgrad_tap_small<2, E>(ctx, st, g, al, x, ept, d, dS);
        }
        else if (ntap == 1) VDNN_WGRAD_TAP(1);
        else if (ntap == 2) VDNN_WGRAD_TAP(2);
        else VDNN_WGRAD_TAP(4);
#undef VDNN_WGRAD_TAP
        if (rc2 != VDNN_OK) return rc2;
        if (d.splits > 1) return launch_reduce_splits_tap(ctx, st, w, staging, (size_t)M * N, d.splits, alpha, accumulate, g.C, RS);
        return VDNN_OK;
    }
    const bool big = RS > 32;
    int rc;
#define VDNN_WGRAD(VEC, BIG)                                                                                              \
    do {                                                                                                                  \
        LoadDyRed<VEC, E> al{dy, g.N, g.K, PQ, d.kchunk, d.K, dPQ};                                                               \
        LoadIm2colRed<BIG, E> bl{x, g.N, g.C, g.H, g.W, g.R, g.S, g.P, g.Q, g.ph, g.pw, g.sh, g.sw, N, d.kchunk, d.K, dRS, dS, dQ, dPQ}; \
        rc = conv_wgrad_with(ctx, st, al, bl, ep, d, narrow, small);                                                             \
    } while (0)
    if (vec && !big) VDNN_WGRAD(true, false);
    else if (vec && big) VDNN_WGRAD(true, true);
    else if (!vec && !big) VDNN_WGRAD(false, false);
    else VDNN_WGRAD(false, true);
#undef VDNN_WGRAD
    if (rc != VDNN_OK) return rc;
    if (d.splits > 1) return launch_reduce_splits(ctx, st, w, staging, (size_t)M * N, d.splits, alpha, accumulate, nullptr, 0);
    return VDNN_OK;
}

// Backward filter, and with `bias` the bias gradient as well: inside the filter-gradient kernel where the shape's kernel
// can, otherwise by the kernels of vdnn_conv_bwd_bias[_sgd] behind it on the same stream.
template <class E>
static int conv_bwd_filter_impl(vdnn_ctx* ctx, vdnn_stream_t stream, const vdnn_shape_t* shape, int algo_mode,
                                const E* x, const E* dy, float* w, float alpha, int accumulate,
                                void* workspace, size_t workspace_bytes, BiasOut* bias = nullptr) {
    const int rc = conv_bwd_filter_core<E>(ctx, stream, shape, algo_mode, x, dy, w, alpha, accumulate, workspace, workspace_bytes, bias);
    if (rc != VDNN_OK || !bias || !bias->wanted() || bias->done || ctx->plan_only) return rc;
    return bias->accumulate ? vdnn_conv_bwd_bias_sgd(ctx, stream, shape, dy, bias->out, bias->alpha)
                            : vdnn_conv_bwd_bias(ctx, stream, shape, dy, bias->out);
}

// Does backward filter of this shape add up the bias gradient inside its own kernel? (The shapes' dispatch above: the
// Winograd variant - float activations only -, the first-layer kernel, the filter-row kernels and wgrad_same.h's.)
static bool bwd_filter_sums_bias(const ConvGeo& g, int algo_mode, int dtype) {
    if (is_dense(g)) return false;
    const bool f32 = dtype == VDNN_DTYPE_F32;
    if (f32 && algo_mode == 1 && wino_wgrad_ok(g) && wino_wgrad_plan_ok(wino_wgrad_plan(g), g)) return true;
    if (g.C <= 3 && g.R == 3 && g.S == 3 && g.ph == 1 && g.pw == 1 && g.sh == 1 && g.sw == 1 && g.P == g.H && g.Q == g.W && g.W % 4 == 0 && g.W >= KB &&
        g.P * g.Q >= WSC_SLICE)
        return true;
    return g.C > 4 && (f32 ? wgrad3x3_f32_ok(g) || wgrad_same_x3_ok(g) : wgrad3x3_ok(g));
}

extern "C" {

int vdnn_conv_bwd_filter_sums_bias(const vdnn_shape_t* shape, int algo_mode, int dtype) {
    ConvGeo g;
    return shape && geo_from_shape(shape, g) && bwd_filter_sums_bias(g, algo_mode, dtype);
}

int vdnn_conv_bwd_filter_bias_sgd(vdnn_ctx* ctx, vdnn_stream_t stream, const vdnn_shape_t* shape, int algo_mode,
                                  const void* x, const void* dy, float* w, float* bias, float alpha,
                                  void* workspace, size_t workspace_bytes) {
    VDNN_REQUIRE(bias != nullptr, "null bias");
    BiasOut b; b.out = bias; b.alpha = alpha; b.accumulate = 1;
    return VDNN_BY_ACT(ctx, conv_bwd_filter_impl<float>(ctx, stream, shape, algo_mode, (const float*)x, (const float*)dy, w, alpha, 1, workspace, workspace_bytes, &b),
                       conv_bwd_filter_impl<bf16_t>(ctx, stream, shape, algo_mode, (const bf16_t*)x, (const bf16_t*)dy, w, alpha, 1, workspace, workspace_bytes, &b));
}

int vdnn_conv_bwd_filter_bias(vdnn_ctx* ctx, vdnn_stream_t stream, const vdnn_shape_t* shape, int algo_mode,
                              const void* x, const void* dy, float* dw, float* db, void* workspace, size_t workspace_bytes) {
    VDNN_REQUIRE(db != nullptr, "null bias gradient");
    BiasOut b; b.out = db; b.alpha = 1.0f; b.accumulate = 0;
    return VDNN_BY_ACT(ctx, conv_bwd_filter_impl<float>(ctx, stream, shape, algo_mode, (const float*)x, (const float*)dy, dw, 1.0f, 0, workspace, workspace_bytes, &b),
                       conv_bwd_filter_impl<bf16_t>(ctx, stream, shape, algo_mode, (const bf16_t*)x, (const bf16_t*)dy, dw, 1.0f, 0, workspace, workspace_bytes, &b));
}

int vdnn_conv_bwd_filter_then_bias_sgd(vdnn_ctx* ctx, vdnn_stream_t stream, const vdnn_shape_t* shape, int algo_mode,
                                       const void* x, const void* dy, float* dw, float* bias, float alpha,
                                       void* workspace, size_t workspace_bytes) {
    VDNN_REQUIRE(bias != nullptr, "null bias");
    BiasOut b; b.out = bias; b.alpha = alpha; b.accumulate = 1;
    return VDNN_BY_ACT(ctx, conv_bwd_filter_impl<float>(ctx, stream, shape, algo_mode, (const float*)x, (const float*)dy, dw, 1.0f, 0, workspace, workspace_bytes, &b),
                       conv_bwd_filter_impl<bf16_t>(ctx, stream, shape, algo_mode, (const bf16_t*)x, (const bf16_t*)dy, dw, 1.0f, 0, workspace, workspace_bytes, &b));
}

size_t vdnn_conv_winograd_chunk_bytes(size_t bytes) {
    const size_t before = g_wino_chunk_bytes;
    g_wino_chunk_bytes = bytes ? bytes : kWinoChunkBytesDefault;
    return before;
}

int vdnn_conv_perf_variant(int variant) {
    const int before = g_perf_variant;
    if (variant == 0 || variant == 1) g_perf_variant = variant;
    return before;
}

size_t vdnn_conv_workspace_bytes(const vdnn_shape_t* shape, int algo_mode, int pass) {
    return vdnn_conv_workspace_bytes_dtype(shape, algo_mode, pass, VDNN_DTYPE_F32);
}

size_t vdnn_conv_workspace_bytes_dtype(const vdnn_shape_t* shape, int algo_mode, int pass, int dtype) {
    ConvGeo g;
    if (!shape || !geo_from_shape(shape, g)) return 0;
    if (algo_mode == 0 /* VDNN_MEMORY_OPT_ALGO */ || is_dense(g)) return 0;
    // Perf-optimal mode, float activations: forward and backward data on the bfloat16 matrix cores take the filter bank
    // split into bfloat16 parts (the filter's bytes); under the Winograd variant, and for backward filter where the default
    // has no kernel, wide 3x3 layers take the transformed filter, input and output of a chunk of samples; other layers
    // re-lay the filter bank out for 128-bit operand loads; backward filter otherwise takes a staging area large enough
    // for the split count that fills the chip.
    const int RS = g.R * g.S;
    const size_t filter_bytes = (size_t)g.K * g.C * RS * sizeof(float);
    if (dtype == VDNN_DTYPE_F32 && pass != 2 && g_perf_variant == 0 && (split3x3_ok(g, pass) || split_general_ok(g, pass))) return filter_bytes;
    if (dtype == VDNN_DTYPE_F32 && pass != 2 && wino_ok(g, pass == 1)) {
        const WinoPlan p = wino_plan(g, pass == 1);
        if (wino_plan_ok(p)) return p.total;
    }
    const bool split_wgrad = dtype == VDNN_DTYPE_F32 && pass == 2 && g_perf_variant == 0 && wgrad3x3_ok(g);
    if (dtype == VDNN_DTYPE_F32 && pass == 2 && !split_wgrad && wino_wgrad_ok(g)) {
        const WinoWgradPlan p = wino_wgrad_plan(g);
        if (wino_wgrad_plan_ok(p, g)) return p.total;
    }
    if (pass == 0) return packed_fwd_ok(g) ? filter_bytes : 0;
    if (pass == 1) return packed_bwd_data_ok(g) ? filter_bytes : 0;
    const int M = g.K, N = g.C * RS;
    const bool narrow = M <= 64;
    const int TM = narrow ? 64 : 128, TN = narrow ? 256 : 128;
    const long tiles = (long)((M + TM - 1) / TM) * ((N + TN - 1) / TN);
    long cap = ((long)g.N * g.P * g.Q + 4 * KB - 1) / (4 * KB);
    const long by_mem = (long)(kMaxWgradWorkspace / filter_bytes);
    if (cap > by_mem) cap = by_mem;
    const int want = choose_splits(tiles, (long)g.N * g.P * g.Q, cap, kPlanningCUs, filter_bytes, 2.0 * TM * TN * KB);
    if (want <= 1) return 0;
    const size_t need = (size_t)want * filter_bytes;
    if (need <= kDefaultStagingBytes) return 0; // the context's own staging area already holds it
    return need;
}

int vdnn_conv_fwd(vdnn_ctx* ctx, vdnn_stream_t stream, const vdnn_shape_t* shape, int algo_mode,
                  const void* x, const float* w, const float* bias, void* y,
                  void* workspace, size_t workspace_bytes) {
    return VDNN_BY_ACT(ctx, conv_fwd_impl<float>(ctx, stream, shape, algo_mode, (const float*)x, w, bias, (float*)y, workspace, workspace_bytes, 0),
                       conv_fwd_impl<bf16_t>(ctx, stream, shape, algo_mode, (const bf16_t*)x, w, bias, (bf16_t*)y, workspace, workspace_bytes, 0));
}

int vdnn_conv_fwd_relu(vdnn_ctx* ctx, vdnn_stream_t stream, const vdnn_shape_t* shape, int algo_mode,
                       const void* x, const float* w, const float* bias, void* y,
                       void* workspace, size_t workspace_bytes) {
    return VDNN_BY_ACT(ctx, conv_fwd_impl<float>(ctx, stream, shape, algo_mode, (const float*)x, w, bias, (float*)y, workspace, workspace_bytes, 1),
                       conv_fwd_impl<bf16_t>(ctx, stream, shape, algo_mode, (const bf16_t*)x, w, bias, (bf16_t*)y, workspace, workspace_bytes, 1));
}

int vdnn_conv_bwd_data(vdnn_ctx* ctx, vdnn_stream_t stream, const vdnn_shape_t* shape, int algo_mode,
                       const void* dy, const float* w, void* dx,
                       void* workspace, size_t workspace_bytes) {
    return VDNN_BY_ACT(ctx, conv_bwd_data_impl<float>(ctx, stream, shape, algo_mode, (const float*)dy, w, (float*)dx, workspace, workspace_bytes, nullptr),
                       conv_bwd_data_impl<bf16_t>(ctx, stream, shape, algo_mode, (const bf16_t*)dy, w, (bf16_t*)dx, workspace, workspace_bytes, nullptr));
}

int vdnn_conv_bwd_data_in_place_ok(const vdnn_shape_t* shape) {
    ConvGeo g;
    return shape && geo_from_shape(shape, g) && conv_bwd_data_in_place_ok(g);
}

int vdnn_conv_bwd_data_relu(vdnn_ctx* ctx, vdnn_stream_t stream, const vdnn_shape_t* shape, int algo_mode,
                            const void* dy, const float* w, const void* x, void* dx,
                            void* workspace, size_t workspace_bytes) {
    VDNN_REQUIRE(x != nullptr, "null input tensor");
    return VDNN_BY_ACT(ctx, conv_bwd_data_impl<float>(ctx, stream, shape, algo_mode, (const float*)dy, w, (float*)dx, workspace, workspace_bytes, (const float*)x),
                       conv_bwd_data_impl<bf16_t>(ctx, stream, shape, algo_mode, (const bf16_t*)dy, w, (bf16_t*)dx, workspace, workspace_bytes, (const bf16_t*)x));
}

int vdnn_conv_bwd_filter_sgd(vdnn_ctx* ctx, vdnn_stream_t stream, const vdnn_shape_t* shape, int algo_mode,
                             const void* x, const void* dy, float* w, float alpha,
                             void* workspace, size_t workspace_bytes) {
    return VDNN_BY_ACT(ctx, conv_bwd_filter_impl<float>(ctx, stream, shape, algo_mode, (const float*)x, (const float*)dy, w, alpha, 1, workspace, workspace_bytes),
                       conv_bwd_filter_impl<bf16_t>(ctx, stream, shape, algo_mode, (const bf16_t*)x, (const bf16_t*)dy, w, alpha, 1, workspace, workspace_bytes));
}

int vdnn_conv_bwd_filter(vdnn_ctx* ctx, vdnn_stream_t stream, const vdnn_shape_t* shape, int algo_mode,
                         const void* x, const void* dy, float* dw, void* workspace, size_t workspace_bytes) {
    return VDNN_BY_ACT(ctx, conv_bwd_filter_impl<float>(ctx, stream, shape, algo_mode, (const float*)x, (const float*)dy, dw, 1.0f, 0, workspace, workspace_bytes),
                       conv_bwd_filter_impl<bf16_t>(ctx, stream, shape, algo_mode, (const bf16_t*)x, (const bf16_t*)dy, dw, 1.0f, 0, workspace, workspace_bytes));
}

} // extern "C"
