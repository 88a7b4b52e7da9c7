// Filter update of a fully connected layer with float activations and few rows: out[o][i] = (accumulate ? out : 0) + alpha * sum_n dy[n][o] * x[n][i].
//
// With a batch of 64 the product is 13 GFLOP over a filter of 411 MB that is read and written: 90 us on the float matrix cores and 150 at the
// rate of a plain copy, so the stream has to run while the products do. The tile engine's workgroups fetch, multiply, then read and write
// their outputs, each phase waiting for the one before: 3.05 TB/s. Here a wavefront owns 32 rows x 128 columns and nothing is
// shared, so nothing waits at a barrier: the operands come straight from L2 (dy and x are 1 and 6 MB; a workgroup's four wavefronts
// read the same x) a slice ahead, the old values arrive in 64 registers while the last two slices are multiplied, and the eight
// wavefronts of a compute unit are at different points of this. 64 rows, 25088 -> 4096 244 -> 186 us (4.4 TB/s); 128 rows 337 -> 267;
// 32 rows, 9216 -> 4096 62.5 -> 50.2 (6.0 TB/s). A lane owns four consecutive columns (block jt of the product is column 4 l + jt), so that x, the old
// values and the results move 128 bits at a time, 512 bytes of a row per instruction.
// The matrix instructions take the reduction in the tile engine's order (mfma_gemm.h: index 8g + 4 (lane / 32) + e of a slice of sixteen):
// the same sums, the same multiply-add, the same bits.
#pragma once
#include "mfma_gemm.h"

namespace vdnn {

constexpr int FCU_TM = 128, FCU_TN = 128;

struct FcUpdate {
    const float* dy; // [n][rows]
    const float* x;  // [n][cols], cols a multiple of four
    float* out;      // [rows][cols], FCU_TM rows below 2 GiB
    int n, rows, cols;
    float alpha;
    int accumulate;
};

__global__ void __launch_bounds__(NT, 2) fc_update_kernel(const FcUpdate g, int jtiles) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l32 = lane & 31, lk = lane >> 5;
    const int tile = xcd_remap(blockIdx.x, gridDim.x);
    const int mt = tile / jtiles, jt0 = tile - mt * jtiles; // column tiles fastest: the workgroups at work together write runs of rows
    const int m0 = mt * FCU_TM + 32 * wave, j0 = jt0 * FCU_TN;
    if (m0 >= g.rows) return;

    const __amdgpu_buffer_rsrc_t rsY = make_rsrc(g.dy, clamp_range((long)g.n * g.rows * 4));
    const __amdgpu_buffer_rsrc_t rsX = make_rsrc(g.x, clamp_range((long)g.n * g.cols * 4));
    // the descriptor ends with the last row: rows beyond are neither read nor written
    const int here = g.rows - m0 < 32 ? g.rows - m0 : 32;
    const __amdgpu_buffer_rsrc_t rsO = make_rsrc(g.out + (long)m0 * g.cols, clamp_range((long)here * g.cols * 4));
    const int j = j0 + 4 * l32;
    const bool inside = j < g.cols;
    const int row_bytes = g.cols * 4;

    // old values: register group v holds row 8 (v / 4) + 4 lk + v % 4, four columns
    const int vo = inside ? 4 * lk * row_bytes + j * 4 : OOB;
    floatx4 old[16];
    auto load_old = [&] {
        if (g.accumulate) {
#pragma unroll
            for (int v = 0; v < 16; v++) old[v] = buf_load4(rsO, vo, (8 * (v / 4) + v % 4) * row_bytes);
        }
    };

    const int vy = m0 + l32 < g.rows ? (4 * lk * g.rows + m0 + l32) * 4 : OOB;
    const int vx = inside ? (4 * lk * g.cols + j) * 4 : OOB;
    struct Slice { float a[8]; floatx4 b[8]; };
    auto load = [&](int k0, Slice& s) { // rows of dy and x past the last read as zero
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int k = k0 + 8 * (i / 4) + i % 4;
            s.a[i] = buf_load(rsY, vy, k * g.rows * 4);
            s.b[i] = buf_load4(rsX, vx, k * g.cols * 4);
        }
    };
    floatx16 acc[4];
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc[t][v] = 0.0f;
    auto multiply = [&](const Slice& s) {
#pragma unroll
        for (int i = 0; i < 8; i++)
#pragma unroll
            for (int t = 0; t < 4; t++) acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(s.a[i], s.b[i][t], acc[t], 0, 0, 0);
    };
    // Loads return in the order of their issue: the old values are requested behind the last operands, two slices of products
    // before they are needed (requested first, every product waited for them: 64 rows, 25088 -> 4096 220 us instead of 186).
    Slice s0, s1;
    load(0, s0);
    load(KB, s1);
    const int slices = (g.n + KB - 1) / KB;
    for (int s = 0; s < slices; s += 2) {
        if (s + 2 >= slices) load_old();
        __builtin_amdgcn_sched_barrier(0);
        multiply(s0);
        if (s + 2 < slices) load((s + 2) * KB, s0);
        if (s + 1 < slices) multiply(s1);
        if (s + 3 < slices) load((s + 3) * KB, s1);
        __builtin_amdgcn_sched_barrier(0);
    }

#pragma unroll
    for (int v = 0; v < 16; v++) {
        floatx4 r;
#pragma unroll
        for (int t = 0; t < 4; t++) r[t] = g.accumulate ? __fmaf_rn(g.alpha, acc[t][v], old[v][t]) : g.alpha * acc[t][v];
        typedef unsigned uint4v __attribute__((ext_vector_type(4)));
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(uint4v, r), rsO, vo, (8 * (v / 4) + v % 4) * row_bytes, 0);
    }
}

} // namespace vdnn
