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


int launch_bias_grad_final(vdnn_ctx* ctx, hipStream_t st, const float* partial, float* bias, int K, int splits, float alpha, int accumulate);

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
