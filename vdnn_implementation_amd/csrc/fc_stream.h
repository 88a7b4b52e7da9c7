// Forward and backward data of fully connected layers with float activations and up to 32 rows:
//   forward        out[n][o] = sum_i x[n][i]  * w[o][i]     (both operands run along the reduction)
//   backward data  out[n][i] = sum_o dy[n][o] * w[o][i]     (the filter runs along the columns)
//
// The filter's trip through memory is the floor: 25 us for the 151 MB of a 9216 -> 4096 layer at 6 TB/s. The tile engine took 48: its 64
// rows double the matrix work of a batch of 32, and its wavefronts wait for each other at a barrier in every slice. Here a wavefront owns
// 32 rows x 64 columns and fetches its own fragments: a lane's four values of a slice's half are one 128-bit load along the reduction (the
// filter's in forward, the rows' in both) or four 32-bit ones of 128-byte runs (the filter's in backward data). No LDS, no barrier. Two slices are
// fetched at a time, a whole line of every row, and two such fetches are in flight; 133 registers, three workgroups per compute unit.
// Slices, splits and the order inside a slice are the tile engine's (fc_gemm, mfma_gemm.h): the same sums, the same bits.
// One call, tile engine -> here: 32 rows, 9216 -> 4096 forward 47.7 -> 41.2 us, backward data 50.1 -> 38.6; 7 rows 45.2 -> 33.4 and 46.8 ->
// 32.4; one row, 25088 -> 4096 114 -> 100 and 118 -> 77. With two blocks of rows per wavefront (64 rows) the loads through L1, twice
// as many per matrix instruction as out of LDS, cost more than the barriers: 127 -> 160 us.
#pragma once
#include "mfma_gemm.h"

namespace vdnn {

struct FcStream {
    const float* rows; // [M][K]
    const float* w;    // forward [N][K], backward data [K][N]
    unsigned row_bytes, w_bytes;
};

// A workgroup has 32 rows and 256 columns. d.K a multiple of sixteen.
template <bool BWD>
__global__ void __launch_bounds__(NT, 3) fc_stream_kernel(const FcStream g, const StoreDense<float> ep, const GemmDims d) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l32 = lane & 31, lk = lane >> 5;
    const int bid = xcd_remap(blockIdx.x, gridDim.x);
    const int tile = bid % d.ntiles, ks = bid / d.ntiles;
    const int j0 = (tile * 4 + wave) * 64;
    const int k_begin = ks * d.kchunk, k_end = min(d.K, k_begin + d.kchunk);
    if (j0 >= d.N) return;

    const __amdgpu_buffer_rsrc_t rsA = make_rsrc(g.rows, g.row_bytes), rsB = make_rsrc(g.w, g.w_bytes);
    const int va = l32 < d.M ? (int)(((long)l32 * d.K + 4 * lk) * 4) : OOB;
    int vb[2];
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int col = j0 + 32 * j + l32;
        vb[j] = col >= d.N ? OOB : BWD ? (int)(((long)4 * lk * d.N + col) * 4) : (int)(((long)col * d.K + 4 * lk) * 4);
    }
    struct Slice { floatx4 a[2], b[2][2]; }; // [half of the slice][block of columns]
    struct Two { Slice s[2]; };
    // the four pieces of a row's line one after the other: L1 has let go of it a few rows on
    auto load = [&](int k0, Two& t) {
        if (k0 >= k_end) return; // uniform
        const int k1 = k0 + 16 < k_end ? k0 + 16 : k0; // (the second slice of the last two may be missing: fetched and not used)
#pragma unroll
        for (int p = 0; p < 4; p++) t.s[p / 2].a[p % 2] = buf_load4(rsA, va, ((p / 2 ? k1 : k0) + 8 * (p % 2)) * 4);
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int p = 0; p < 4; p++) {
                const int k = (p / 2 ? k1 : k0) + 8 * (p % 2);
                if constexpr (BWD) {
#pragma unroll
                    for (int e = 0; e < 4; e++) t.s[p / 2].b[p % 2][j][e] = buf_load(rsB, vb[j], (int)((long)(k + e) * d.N * 4));
                } else t.s[p / 2].b[p % 2][j] = buf_load4(rsB, vb[j], k * 4);
            }
    };
    floatx16 acc[1][2];
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc[0][j][v] = 0.0f;
    auto multiply = [&](int k0, const Two& t) {
#pragma unroll
        for (int u = 0; u < 2; u++) {
            if (k0 + 16 * u >= k_end) return; // uniform
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int e = 0; e < 4; e++)
#pragma unroll
                    for (int j = 0; j < 2; j++) acc[0][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(t.s[u].a[h][e], t.s[u].b[h][j][e], acc[0][j], 0, 0, 0);
        }
    };
    Two t0, t1;
    load(k_begin, t0);
    load(k_begin + 32, t1);
    for (int k0 = k_begin; k0 < k_end; k0 += 64) {
        multiply(k0, t0);
        load(k0 + 64, t0);
        multiply(k0 + 32, t1);
        load(k0 + 96, t1);
    }
    ep.store(acc, 0, j0, lane, ks, d, d.splits > 1);
}

} // namespace vdnn
