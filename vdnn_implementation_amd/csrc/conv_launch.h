// What the launchers of the convolution kernels share (conv.hip, conv_same.hip).
#pragma once
#include "backend_internal.h"
#include "conv_loaders.h"

namespace vdnn {

// samples one tile of `tile` pixels can touch, times the sample size: must stay below 2 GiB so that
// per-lane byte offsets are positive ints and the exhausted-range scalar offset is out of range
static inline bool pixel_tile_span_ok(long sample_elems, int opix, int tile, int elem_bytes) {
    const long span = (long)(tile / opix + 2) * sample_elems * elem_bytes;
    return span < 0x7FFF0000l;
}

static inline GemmDims make_dims(int M, int N, int K, int TM, int TN, int splits, int depth = KB) {
    GemmDims d;
    d.M = M; d.N = N; d.K = K;
    d.mtiles = (M + TM - 1) / TM;
    d.ntiles = (N + TN - 1) / TN;
    if (splits < 1) splits = 1;
    int kchunk = (K + splits - 1) / splits;
    kchunk = (kchunk + depth - 1) / depth * depth;
    d.kchunk = kchunk;
    d.splits = (K + kchunk - 1) / kchunk;
    d.full_tiles = 0;
    return d;
}

// Split tiles of the 64x64 kernel added up by the workgroup that ends last (sum_splits), where their sums fit the staging area tile by tile.
// Up to six splits: one workgroup reads them all, and with many that takes longer than a second kernel on the whole chip (sixteen
// splits, forward 3 x 141 x 14 x 14, 320 of 3x3 at stride 2: 13.0 us with the second kernel, 15.4 without). 9549 drawn calls that fall
// under the rule, timed both ways, gain 4.1 % (two to five splits 3 to 5 %, six 2.5 %), 10740 fully connected ones 8.1 % (six splits 1.6 %). Not for
// backward filter, whose products fill the chip by their splits: 5 x 144 x 16 x 16, 128 of 3x3 backward 33.1 -> 35.2.
constexpr int kFusedSplits = 6;
static inline bool fuse_split_sums(vdnn_ctx* ctx, hipStream_t stream, GemmDims& d, size_t partial_bytes) {
    const long tiles = (long)d.mtiles * d.ntiles - d.full_tiles;
    if (d.splits < 2 || d.splits > kFusedSplits || tiles > kTileCounters || (size_t)tiles * d.splits * 64 * 64 * sizeof(float) > partial_bytes) return false;
    d.counters = tile_counters_of(ctx, stream);
    return d.counters != nullptr;
}

// What is planned without a context at hand assumes the 256 compute units of the target part and the staging area as it is made.
constexpr int kPlanningCUs = 256;
constexpr size_t kDefaultStagingBytes = (size_t)64 << 20;

// Splits of a forward / backward data product in large tiles (launch_by_m): where the tiles do not fill the chip
static inline int pixel_product_splits(int M, int N, int K, int TM, int TN, int depth, size_t partial_bytes, int num_cu) {
    const long tiles = (long)((M + TM - 1) / TM) * ((N + TN - 1) / TN);
    const size_t out_bytes = (size_t)M * N * sizeof(float);
    if (tiles >= 2l * num_cu) return 1;
    long cap = ((long)K + 8 * depth - 1) / (8 * depth); // at least eight slices per split
    const long by_mem = (long)(partial_bytes / out_bytes);
    if (cap > by_mem) cap = by_mem;
    return choose_splits(tiles, K, cap, num_cu, out_bytes, 2.0 * TM * TN * KB);
}
// ... and what the tile engine takes for it in the tile it would choose (small_cost, large_cost: the loaders' work, LoadCost in conv.hip; 1: the
// filter re-laid out tap-major)
static inline double pixel_product_us(int M, int N, int K, size_t partial_bytes, int num_cu, double small_cost = 1.0, double large_cost = 1.0) {
    const int TM = M <= 64 ? 64 : 128, TN = M <= 64 ? 256 : 128;
    const double small = small_tile_plan(M, N, K, partial_bytes, num_cu, 4, true, small_cost).us;
    const double large = large_tile_us(M, N, K, TM, TN, pixel_product_splits(M, N, K, TM, TN, KB, partial_bytes, num_cu), num_cu, false, large_cost);
    return K <= kShortReduction || small < 0.9 * large ? small : large;
}

// Backward filter on the tile engine: the splits of large tiles, the 64x64 tile's plan, both estimates
struct FilterTilePlan { int want; SmallTilePlan small; double large_us; };
static inline FilterTilePlan filter_tile_plan(const ConvGeo& g, size_t staging_bytes, int num_cu) {
    const int M = g.K, N = g.C * g.R * g.S, PQ = g.P * g.Q, TM = M <= 64 ? 64 : 128, TN = M <= 64 ? 256 : 128;
    const long Kred = (long)g.N * PQ, tiles = (long)((M + TM - 1) / TM) * ((N + TN - 1) / TN);
    const size_t out_bytes = (size_t)M * N * sizeof(float);
    const bool taps = PQ % 4 == 0 && PQ >= KB && 2 * g.Q >= KB; // planes the tap-major loaders take
    long cap = (Kred + 4 * KB - 1) / (4 * KB); // at least four slices per split
    const long by_mem = (long)(staging_bytes / out_bytes);
    if (cap > by_mem) cap = by_mem;
    FilterTilePlan p;
    p.want = choose_splits(tiles, Kred, cap, num_cu, out_bytes, 2.0 * TM * TN * KB);
    p.small = small_tile_plan(M, N, Kred, staging_bytes, num_cu, 2, false, taps && g.C % 64 == 0 ? 1.05 : 1.9);
    p.large_us = large_tile_us(M, N, Kred, TM, TN, p.want, num_cu, true, taps && g.C % 32 == 0 ? 1.0 : 1.15);
    return p;
}

int launch_reduce_tail_nchw(vdnn_ctx* ctx, hipStream_t stream, float* out, const float* partial, int tail_tiles, int splits, int TM, int TN,
                            int M, int N, int mtiles, int full_tiles, const float* bias, int opix, int relu, const float* gate);
int launch_reduce_tail_nchw(vdnn_ctx* ctx, hipStream_t stream, bf16_t* out, const float* partial, int tail_tiles, int splits, int TM, int TN,
                            int M, int N, int mtiles, int full_tiles, const float* bias, int opix, int relu, const bf16_t* gate);
int launch_reduce_splits_tap(vdnn_ctx* ctx, hipStream_t stream, float* out, const float* partial, size_t count, int splits,
                             float alpha, int accumulate, int C, int RS);
int launch_reduce_splits_nchw(vdnn_ctx* ctx, hipStream_t stream, float* out, const float* partial, size_t count, int splits,
                              const float* bias, int opix, int channels, int relu, const float* gate);
int launch_reduce_splits_nchw(vdnn_ctx* ctx, hipStream_t stream, bf16_t* out, const float* partial, size_t count, int splits,
                              const float* bias, int opix, int channels, int relu, const bf16_t* gate);

int launch_reduce_splits(vdnn_ctx* ctx, hipStream_t stream, float* out, const float* partial, size_t count,
                         int splits, float alpha, int accumulate, const float* bias_j, int ncols, int relu = 0, const float* gate = nullptr);

static inline bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }


int launch_bias_grad_final(vdnn_ctx* ctx, hipStream_t st, const float* partial, float* bias, int K, int splits, float alpha, int accumulate, bool in_double = false);

// The bias gradient as a by-product of backward filter (cudnnConvolutionBackwardBias, layer.cu:631-637, reads the same dy
// as cudnnConvolutionBackwardFilter, :651-660): where the filter-gradient kernel of a shape can add up the dy values it
// streams, it leaves per-channel partial sums in the context's bias staging area and `done` is set; the caller runs the
// ordered final sum. out = (accumulate ? out : 0) + alpha * sum over n, p, q of dy.
struct BiasOut {
    float* out = nullptr;
    float alpha = 1.0f;
    int accumulate = 0;
    bool done = false;
    bool wanted() const { return out != nullptr; }
};
// room for K x parts partial sums in the bias staging area?
static inline bool bias_parts_fit(const vdnn_ctx* ctx, int K, long parts) {
    return ctx->bias_scratch && parts > 0 && (size_t)K * (size_t)parts * sizeof(float) <= ctx->bias_scratch_bytes;
}

// Takes bytes from the front of the context's staging area for as long as the object lives; everything that
// uses the staging area meanwhile (partial sums, intermediate products) sees the remainder.
struct StagingCarve {
    vdnn_ctx* ctx;
    float* base = nullptr;
    size_t total = 0;
    bool taken = false;
    explicit StagingCarve(vdnn_ctx* c) : ctx(c) {}
    void* take(size_t bytes) {
        base = ctx->reduce_scratch; total = ctx->reduce_scratch_bytes; taken = true;
        const size_t t = (bytes + 255) / 256 * 256;
        ctx->reduce_scratch = (float*)((char*)base + t);
        ctx->reduce_scratch_bytes = total - t;
        return base;
    }
    ~StagingCarve() { if (taken) { ctx->reduce_scratch = base; ctx->reduce_scratch_bytes = total; } }
};

// Room for a re-laid-out filter bank at the front of the staging area: only if nothing was taken from it yet and at
// least half of it stays for the partial sums of split reductions (the largest need of a layer is a round of partial
// tiles: 768 x 64 KB). Null otherwise.
static inline float* packed_filter_place(vdnn_ctx* ctx, StagingCarve& carve, size_t bytes) {
    if (carve.taken || !ctx->reduce_scratch || 2 * ((bytes + 255) / 256 * 256) > ctx->reduce_scratch_bytes) return nullptr;
    return (float*)carve.take(bytes);
}

// what the filter-row kernel of float layers needs (wgrad3x3_f32.h): a slice wraps at most two image rows
static inline bool wgrad3x3_f32_ok(const ConvGeo& g) {
    return g.R == 3 && g.S == 3 && g.ph == 1 && g.pw == 1 && g.sh == 1 && g.sw == 1 && g.P == g.H && g.Q == g.W &&
           g.W % 2 == 0 && g.W >= 14 && (g.H * g.W) % 4 == 0 && g.C % 64 == 0;
}

// conv_same.hip: the float layers that conv_same_f32x3.h takes; *taken false where it does not
int launch_same_x3_fwd(vdnn_ctx* ctx, hipStream_t st, StagingCarve& carve, const ConvGeo& g, const float* x, const float* w, const float* bias, float* y, int relu, bool* taken);
int launch_same_x3_bwd_data(vdnn_ctx* ctx, hipStream_t st, StagingCarve& carve, const ConvGeo& g, const float* dy, const float* w, float* dx, const float* gate, bool* taken);

bool wgrad_same_x3_ok(const ConvGeo& g);
int launch_wgrad_same_x3(vdnn_ctx* ctx, hipStream_t st, const ConvGeo& g, const float* x, const float* dy, float* w, float alpha, int accumulate,
                         float* staging, size_t staging_bytes, bool* taken, BiasOut* bias);

} // namespace vdnn
