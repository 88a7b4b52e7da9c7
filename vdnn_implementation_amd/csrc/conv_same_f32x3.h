// Stride-1 float convolutions whose output plane is as large as their input plane (3x3 with padding 1, 5x5 with padding 2) -
// forward and backward data - with float precision on the bfloat16 matrix cores.
//
// A float has 24 significant bits and a bfloat16 eight, so every finite float is the exact sum of three bfloat16 values,
//   v = v0 + v1 + v2,  v0 = bf16(v), v1 = bf16(v - v0), v2 = v - v0 - v1   (|v1| <= 2^-8 |v|, |v2| <= 2^-17 |v|),
// and a product of two floats is the sum of nine products of bfloat16 values, each exact in float. The six of at least 2^-17
// of the product (a0 b0; a0 b1, a1 b0; a1 b1, a0 b2, a2 b0) are accumulated in float by v_mfma_f32_32x32x16_bf16; the other
// three are below 2^-24 of the product together, less than the rounding of one float addition to a sum of the product's own
// size. The instruction rounds its accumulator once per eight products (measured), the float one once or more per two; the five
// small products have accumulators of their own, so a sum meets two roundings per sixteen channels instead of eight or
// more: against 64 bits the error by 2-norm was 0.43 of the float instruction's in the median of 541 passes of drawn layers and
// 0.82 at most (with one set of accumulators 0.7 to 1.3). Six instructions of the 16x faster kind replace one.
// One pass, float engine -> here: 32 x 256 x 13 x 13, 384 filters of 3x3 forward 97.6 -> 75.4 us, backward data 97.0 -> 74.8; 32 x 96 x 27 x 27,
// 256 of 5x5 246 -> 159 and 309 -> 184; where the grid is large 220-228 TFLOP/s against 135-140, 1350 as issued: the matrix pipes at
// the clock the part delivers under them.
//
// Values that this does not hold for: infinities, NaN and the 2^-9 of floats next to the largest one (v0 rounds to an infinity)
// all give NaN in some part. A wavefront whose block of results holds any value that is not finite computes the block
// again with the float instruction from the unsplit operands, so what leaves is what the float engine gives.
//
// The scheme of conv3x3_bf16.h: 64 rows (channels) x 256 pixels per workgroup, 64 x 64 per wavefront; the taps of a filter row
// share one window of 256 + S - 1 positions, staged for 16 channels, and tap s reads the window s positions on; a tap outside
// the image's columns reads a row of zeros. An LDS row is [v0 of 16 channels | v1 | v2] and 16 bytes: 28 words, so eight
// lanes on consecutive rows - a fragment read - tile the 32 banks. Two workgroups per compute unit (72 KB of LDS, 72.8 for 5x5).
#pragma once
#include <type_traits>
#include "mfma_bf16.h"

namespace vdnn {

constexpr int X3_TM = 64;     // output rows (channels) per tile
constexpr int X3_TN = 256;    // pixels per tile
constexpr int X3_CH = 16;     // reduced channels of a step
constexpr int X3_ROW = 56;    // LDS row, 16-bit units: three parts of sixteen channels, padding

// three parts of two floats, each pair packed into one word (first value in the low half)
__device__ __forceinline__ void split3_pair(float a, float b, unsigned& p0, unsigned& p1, unsigned& p2) {
    p0 = pack2_bf16(a, b);
    const float a1 = a - __builtin_bit_cast(float, p0 << 16), b1 = b - __builtin_bit_cast(float, p0 & 0xFFFF0000u);
    p1 = pack2_bf16(a1, b1);
    p2 = pack2_bf16(a1 - __builtin_bit_cast(float, p1 << 16), b1 - __builtin_bit_cast(float, p1 & 0xFFFF0000u));
}

// Filter bank in three parts, blocked tap-major: packed[row][((cb*RS + tap)*3 + part)*16 + l] = part of
// w[row*row_stride + (cb*16 + l)*red_stride + tap] (row_stride / red_stride as in pack_filter_tap_bf16_kernel).
// One thread per filter element, reduced channels a multiple of 16.
static __global__ void __launch_bounds__(256) pack_filter_split3_kernel(const float* __restrict__ w, unsigned short* __restrict__ packed, int Cred, int RS,
                                                                 int row_stride, int red_stride, long total) {
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i >= total) return;
    const int per_row = Cred * RS;
    const int row = (int)(i / per_row), kk = (int)(i - (long)row * per_row);
    const int l = kk & 15, slice = kk >> 4;
    const int cb = slice / RS, tap = slice - cb * RS;
    unsigned p0, p1, p2;
    split3_pair(w[(long)row * row_stride + (long)(cb * 16 + l) * red_stride + tap], 0.0f, p0, p1, p2);
    unsigned short* at = packed + ((long)row * per_row + (long)slice * 16) * 3 + l;
    at[0] = (unsigned short)p0; at[16] = (unsigned short)p1; at[32] = (unsigned short)p2;
}

struct ConvSameX3 {
    const float* src;             // x (forward) or dy (backward data)
    const unsigned short* packed; // pack_filter_split3_kernel
    const float* w;               // the filter itself, for blocks with values that are not finite
    unsigned packed_bytes;        // below 2 GiB
    int row_stride, red_stride;   // of w
    int H, W;                     // extent of a plane (input and output planes agree)
    int reduced;                  // reduced channels, a multiple of 16
    long sample_elems;            // reduced * H * W
    int nsamples;
};

// MODE 0: forward, filter row r lies r - S/2 rows below the pixel and tap s reads s - S/2 columns to its right. MODE 1: backward
// data, both mirrored. PAIRS: rows of an even number of pixels (a pair never straddles two rows: one 64-bit load, one test).
// d.K = reduced * S * S, split at multiples of 16 * S (one filter row of sixteen channels).
template <int MODE, int S, bool PAIRS>
__global__ void __launch_bounds__(NT, 2) conv_same_f32x3_kernel(const ConvSameX3 geo, const StoreNCHW<float> ep, const GemmDims d) {
    constexpr int PAD = S / 2, ROWS = X3_TN + S - 1, TM = X3_TM;
    __shared__ __attribute__((aligned(16))) unsigned short As[2][TM * X3_ROW];
    __shared__ __attribute__((aligned(16))) unsigned short Bw[2][(ROWS + 1) * X3_ROW]; // the window and a row of zeros

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int ntiles_all = d.mtiles * d.ntiles;
    int tile, ks;
    bool whole;
    if ((int)blockIdx.x < d.full_tiles) {
        tile = xcd_remap(blockIdx.x, d.full_tiles); ks = 0; whole = true;
    } else if (d.full_tiles > 0) {
        const int r = blockIdx.x - d.full_tiles, tl = ntiles_all - d.full_tiles;
        tile = d.full_tiles + r % tl; ks = r / tl; whole = false;
    } else {
        const int bid = xcd_remap(blockIdx.x, gridDim.x);
        tile = bid % ntiles_all; ks = bid / ntiles_all; whole = d.splits == 1;
    }
    const int mt = tile % d.mtiles, nt = tile / d.mtiles;
    const int m0 = mt * TM, j0 = nt * X3_TN;
    const int k_begin = whole ? 0 : ks * d.kchunk;
    const int k_end = whole ? d.K : min(d.K, k_begin + d.kchunk);
    const int row_begin = k_begin / (X3_CH * S), row_end = (k_end + X3_CH * S - 1) / (X3_CH * S); // (channel block, filter row) steps

    const int W = geo.W, plane = geo.H * geo.W;
    const int n_first = j0 / plane;
    int n_last = (j0 + X3_TN - 1) / plane;
    if (n_last > geo.nsamples - 1) n_last = geo.nsamples - 1;
    // the descriptor starts `lead` elements ahead of the first sample, so that every offset below is non-negative (what
    // lies before the sample is never fetched), and ends with the last sample the tile touches
    const int lead = PAD * (W + 1);
    const __amdgpu_buffer_rsrc_t rsrc = make_rsrc(geo.src + (long)n_first * geo.sample_elems - lead, clamp_range(((long)(n_last - n_first + 1) * geo.sample_elems + lead) * 4));

    // ---- filter operand: 64 rows of 96 bytes a step, parts 0 and 1 by all threads, part 2 by wavefronts 0 and 1 ----
    const __amdgpu_buffer_rsrc_t rsw = make_rsrc(geo.packed, geo.packed_bytes);
    struct FilterRegs { uintx4 v01, v2; };
    FilterRegs ra[2]; // of the step after next, about to be written to LDS, and of the one behind it
    const int row4 = rows_by_four_lanes(tid), row2 = rows_by_two_lanes(tid) & 63; // (no LDS bank conflicts in the stores)
    const int ld = d.K * 6;                                                        // bytes of a row of the bank
    const int vrow4 = m0 + row4 < d.M ? (int)((long)(m0 + row4) * ld) + 16 * (tid & 3) : OOB;
    const int vrow2 = m0 + row2 < d.M ? (int)((long)(m0 + row2) * ld) + 64 + 16 * (tid & 1) : OOB;
    auto load_filter = [&](int step, FilterRegs& r) {
        const int soff = step * (X3_CH * 6);
        r.v01 = __builtin_bit_cast(uintx4, __builtin_amdgcn_raw_buffer_load_b128(rsw, vrow4, soff, 0));
        if (wave < 2) r.v2 = __builtin_bit_cast(uintx4, __builtin_amdgcn_raw_buffer_load_b128(rsw, vrow2, soff, 0));
    };
    auto store_filter = [&](unsigned short* lds, const FilterRegs& r) {
        *(uintx4*)(lds + row4 * X3_ROW + 8 * (tid & 3)) = r.v01;
        if (wave < 2) *(uintx4*)(lds + row2 * X3_ROW + 32 + 8 * (tid & 1)) = r.v2;
    };

    // ---- window: thread = (pixel pair tid % 128, channels 8 (tid / 128) .. + 7) ------------------------------------
    int voff[PAIRS ? 1 : 2];        // byte offset of the pixel (pair) in its sample's first plane, or out of range
    unsigned rowinv[PAIRS ? 1 : 2]; // bit r: filter row r of its image row lies outside the image
#pragma unroll
    for (int e = 0; e < (PAIRS ? 1 : 2); e++) {
        const int j = j0 + 2 * (tid & 127) + e;
        const bool valid = j < d.N;
        const int jj = valid ? j : j0;
        const int n = jj / plane, pix = jj - n * plane;
        const int p = pix / W;
        voff[e] = valid ? (int)(((long)(n - n_first) * geo.sample_elems + pix) * 4) : OOB;
        rowinv[e] = 0;
#pragma unroll
        for (int r = 0; r < S; r++) {
            const int ih = MODE == 0 ? p + r - PAD : p + PAD - r;
            if (!((unsigned)ih < (unsigned)geo.H)) rowinv[e] |= 1u << r;
        }
    }
    // the S - 1 positions beside the tile (PAD to the left, then PAD to the right), sixteen channels each: lanes of wavefront 0.
    // Needed where they lie in the image row of the tile's first (last) pixel.
    int hoff = OOB;
    unsigned hrowinv = 0;
    const bool halo_lane = wave == 0 && lane < (S - 1) * X3_CH;
    const int hside = lane / X3_CH, hch = lane % X3_CH;
    if (halo_lane) {
        const bool right = hside >= PAD;
        const int j = right ? j0 + X3_TN - 1 : j0, dx = right ? hside - PAD + 1 : hside - PAD;
        if (j < d.N) {
            const int n = j / plane, pix = j - n * plane;
            const int p = pix / W, q = pix - p * W;
            if ((unsigned)(q + dx) < (unsigned)W) hoff = (int)(((long)(n - n_first) * geo.sample_elems + (long)hch * plane + pix + dx) * 4);
#pragma unroll
            for (int r = 0; r < S; r++) {
                const int ih = MODE == 0 ? p + r - PAD : p + PAD - r;
                if (!((unsigned)ih < (unsigned)geo.H)) hrowinv |= 1u << r;
            }
        }
    }
    const int hrow = (hside < PAD ? hside : X3_TN + hside) * X3_ROW + hch;
    // where this lane's fragment of column block jt lies in a window buffer when the tap reads the window `shift` positions on:
    // that position, or the row of zeros where the tap's column lies outside the image
    const int wn0 = wave * 64;
    const int l32 = lane & 31, lk = lane >> 5;
    int frag[2][S];
#pragma unroll
    for (int jt = 0; jt < 2; jt++) {
        const int j = j0 + wn0 + jt * 32 + l32;
        const int q = j % plane % W;
#pragma unroll
        for (int shift = 0; shift < S; shift++) {
            const bool outside = !((unsigned)(q + shift - PAD) < (unsigned)W);
            frag[jt][shift] = (outside ? ROWS : wn0 + jt * 32 + l32 + shift) * X3_ROW + 8 * lk;
        }
    }
    if (tid < X3_ROW) { Bw[0][ROWS * X3_ROW + tid] = 0; Bw[1][ROWS * X3_ROW + tid] = 0; }

    // the window of the next row step, in flight for a whole row step
    struct Fetched { floatx2 raw[8]; float hr; };
    Fetched f;
    f.hr = 0.0f;
    const int g0 = __builtin_amdgcn_readfirstlane(tid >> 7);
    const int swapped = (tid >> 2) & 1; // this lane stores its second pixel first: eight lanes then tile the banks (see conv3x3_bf16.h)
    auto load_window = [&](int row_step) {
        const int cb = row_step / S, r = row_step - cb * S;
        const int rowoff = (MODE == 0 ? r - PAD : PAD - r) * W + lead;
        const int soff = ((cb * X3_CH + 8 * g0) * plane + rowoff) * 4, step = plane * 4;
        const int v0 = voff[0] | bit_to_all_ones(rowinv[0], r);
        if constexpr (PAIRS) {
#pragma unroll
            for (int e = 0; e < 8; e++) f.raw[e] = __builtin_bit_cast(floatx2, __builtin_amdgcn_raw_buffer_load_b64(rsrc, v0, soff + e * step, 0));
        } else {
            const int v1 = voff[1] | bit_to_all_ones(rowinv[1], r);
#pragma unroll
            for (int e = 0; e < 8; e++) {
                f.raw[e].x = buf_load(rsrc, v0, soff + e * step);
                f.raw[e].y = buf_load(rsrc, v1, soff + e * step);
            }
        }
        if (halo_lane) f.hr = buf_load(rsrc, hoff | bit_to_all_ones(hrowinv, r), (cb * X3_CH * plane + rowoff) * 4);
    };
    auto store_window = [&](unsigned short* lds) {
#pragma unroll
        for (int e = 0; e < 2; e++) {
            uintx4 p[3];
            unsigned q0[4], q1[4], q2[4];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const float a = (e ^ swapped) ? f.raw[2 * k].y : f.raw[2 * k].x, b = (e ^ swapped) ? f.raw[2 * k + 1].y : f.raw[2 * k + 1].x;
                split3_pair(a, b, q0[k], q1[k], q2[k]);
            }
            p[0].x = q0[0]; p[0].y = q0[1]; p[0].z = q0[2]; p[0].w = q0[3];
            p[1].x = q1[0]; p[1].y = q1[1]; p[1].z = q1[2]; p[1].w = q1[3];
            p[2].x = q2[0]; p[2].y = q2[1]; p[2].z = q2[2]; p[2].w = q2[3];
            unsigned short* at = lds + (PAD + 2 * (tid & 127) + (e ^ swapped)) * X3_ROW + 8 * (tid >> 7);
#pragma unroll
            for (int k = 0; k < 3; k++) *(uintx4*)(at + 16 * k) = p[k];
        }
        if (halo_lane) {
            unsigned p0, p1, p2;
            split3_pair(f.hr, 0.0f, p0, p1, p2);
            unsigned short* at = lds + hrow;
            at[0] = (unsigned short)p0; at[16] = (unsigned short)p1; at[32] = (unsigned short)p2;
        }
    };

    // [row block][column block]: the products 0 x 0, and the five small ones apart - 2^-8 of the sum at most, so that their
    // roundings do not count: a sum then meets one rounding per sixteen channels
    floatx16 acc[2][2], low[2][2];
    auto clear = [](floatx16 (&a)[2][2]) {
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int v = 0; v < 16; v++) a[i][j][v] = 0.0f;
    };
    clear(acc);
    clear(low);

    auto read_a = [&](const unsigned short* buf, int part, bf16x8 (&a)[2]) {
        const unsigned short* ap = buf + l32 * X3_ROW + 8 * lk + 16 * part;
#pragma unroll
        for (int i = 0; i < 2; i++) a[i] = *(const bf16x8*)(ap + i * 32 * X3_ROW);
    };
    auto read_b = [&](const unsigned short* win, int s, int part, bf16x8 (&b)[2]) {
        const int shift = MODE == 0 ? s : S - 1 - s;
#pragma unroll
        for (int jt = 0; jt < 2; jt++) b[jt] = *(const bf16x8*)(win + frag[jt][shift] + 16 * part);
    };
    auto multiply = [](floatx16 (&to)[2][2], const bf16x8 (&a)[2], const bf16x8 (&b)[2]) {
#pragma unroll
        for (int jt = 0; jt < 2; jt++)
#pragma unroll
            for (int i = 0; i < 2; i++) to[i][jt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[jt], to[i][jt], 0, 0, 0);
    };

    // Pipeline. Step g = (row step, tap s) multiplies from As[g % 2] and the window buffer row_step % 2, 24 matrix instructions
    // a wavefront with one barrier between them:
    //   first half:   read parts 1 and 2 of step g, multiply 0 x 0 (fragments already in registers), 0 x 1, 1 x 0; write the
    //                 filter of step g + 1 to the other As buffer and, at the last tap, the next row step's window;
    //   barrier;
    //   second half:  fetch the filter of step g + 3 (at the last tap also the window of the row step after the next), read part 0
    //                 of step g + 1 from the buffers just completed, multiply 1 x 1, 0 x 2, 2 x 0.
    // All reads of a buffer precede the barrier after which it is overwritten. Fetches past the end of the range are never used.
    const int step0 = row_begin * S;
    load_filter(step0, ra[0]);
    load_window(row_begin);
    store_filter(As[0], ra[0]);
    store_window(Bw[0]);
    load_filter(step0 + 1, ra[1]);
    load_filter(step0 + 2, ra[0]);
    load_window(row_begin + 1);
    __syncthreads();
    bf16x8 a0[2][2], b0[2][2], a1[2], b1[2], a2[2], b2[2];
    read_a(As[0], 0, a0[0]);
    read_b(Bw[0], 0, 0, b0[0]);
    auto row_step_body = [&](int row_step, auto odd) {
        constexpr int ODD = decltype(odd)::value;
#pragma unroll
        for (int s = 0; s < S; s++) {
            const int g = (row_step - row_begin) * S + s;
            const int cur = (S * ODD + s) & 1, nxt = cur ^ 1; // = g & 1
            read_a(As[cur], 1, a1);
            read_b(Bw[ODD], s, 1, b1);
            read_a(As[cur], 2, a2);
            read_b(Bw[ODD], s, 2, b2);
            multiply(acc, a0[cur], b0[cur]);
            multiply(low, a0[cur], b1);
            multiply(low, a1, b0[cur]);
            store_filter(As[nxt], ra[nxt]);
            if (s == S - 1) store_window(Bw[ODD ^ 1]);
            // an LDS access behind every matrix instruction
#pragma unroll
            for (int i = 0; i < 12; i++) { __builtin_amdgcn_sched_group_barrier(0x008, 1, 0); __builtin_amdgcn_sched_group_barrier(0x300, 1, 0); }
            __syncthreads();
            load_filter(step0 + g + 3, ra[nxt]);
            if (s == S - 1) load_window(row_step + 2);
            read_a(As[nxt], 0, a0[nxt]);
            read_b(s == S - 1 ? Bw[ODD ^ 1] : Bw[ODD], s == S - 1 ? 0 : s + 1, 0, b0[nxt]);
            multiply(low, a1, b1);
            multiply(low, a0[cur], b2);
            multiply(low, a2, b0[cur]);
            // a memory instruction and an LDS read behind every matrix instruction
#pragma unroll
            for (int i = 0; i < 12; i++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            }
        }
    };
    for (int row_step = row_begin; row_step < row_end; row_step += 2) {
        row_step_body(row_step, std::integral_constant<int, 0>{});
        if (row_step + 1 < row_end) row_step_body(row_step + 1, std::integral_constant<int, 1>{});
    }

    // a result that is not finite: the wavefront's block again, with the float instruction
    float bad = 0.0f;
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) {
                acc[i][j][v] += low[i][j][v];
                bad = __fmaf_rn(acc[i][j][v], 0.0f, bad);
            }
    if (__any(bad != 0.0f)) {
        clear(acc);
        int pbase[2], prow[2], pcol[2];
#pragma unroll
        for (int jt = 0; jt < 2; jt++) {
            const int j = j0 + wn0 + jt * 32 + l32;
            const int n = j / plane, pix = j - n * plane;
            prow[jt] = j < d.N ? pix / W : -S; // (no tap of such a pixel lies inside the image)
            pcol[jt] = pix % W;
            pbase[jt] = (int)(((long)(n - n_first) * geo.sample_elems + pix + lead) * 4);
        }
#pragma unroll 1
        for (int step = row_begin * S; step < row_end * S; step++) {
            const int cb = step / (S * S), tap = step - cb * (S * S), r = tap / S, s = tap - r * S;
            const int dh = MODE == 0 ? r - PAD : PAD - r, dw = MODE == 0 ? s - PAD : PAD - s;
            int at[2];
#pragma unroll
            for (int jt = 0; jt < 2; jt++) {
                const bool inside = (unsigned)(prow[jt] + dh) < (unsigned)geo.H && (unsigned)(pcol[jt] + dw) < (unsigned)W;
                at[jt] = inside ? pbase[jt] + ((cb * X3_CH + lk) * plane + dh * W + dw) * 4 : OOB;
            }
#pragma unroll 1
            for (int c = 0; c < X3_CH; c += 2) {
                float a[2], b[2];
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    const int m = m0 + i * 32 + l32;
                    a[i] = m < d.M ? geo.w[(long)m * geo.row_stride + (long)(cb * X3_CH + c + lk) * geo.red_stride + tap] : 0.0f;
                    b[i] = buf_load(rsrc, at[i], c * plane * 4);
                }
#pragma unroll
                for (int jt = 0; jt < 2; jt++)
#pragma unroll
                    for (int i = 0; i < 2; i++) acc[i][jt] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[jt], acc[i][jt], 0, 0, 0);
            }
        }
    }

    if (StoreNCHW<float>::TAIL && d.full_tiles > 0 && !whole)
        ep.store_tail(acc, 0, wn0, lane, (long)(tile - d.full_tiles) * d.splits + ks, TM, X3_TN);
    else
        ep.store(acc, m0, j0 + wn0, lane, ks, d, !whole);
}

} // namespace vdnn
