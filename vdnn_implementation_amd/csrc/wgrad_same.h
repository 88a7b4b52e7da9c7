// Backward filter of stride-1 convolutions whose output plane is as large as their input plane (3x3 with padding 1, 5x5 with
// padding 2), planes of any extent, on the bfloat16 matrix cores.
//
//   dW[k][c][r][s] = sum over (n,p,q) of dy[n,k,p,q] * x[n,c,p+r-PAD,q+s-PAD]
//
// A workgroup owns one filter row r, 64 input channels and 64 output channels. The reduction runs over *slots*: the image rows one
// after the other, each followed by PAD slots that hold zero in both operands. Then tap s of a dy slot t meets x slot t + s - PAD
// whatever t is: the zeros behind a row are the padding to its right and to the left of the next one, so no tap needs
// a mask, at the price of W + PAD slots for W pixels (an eighth on 7 x 7 planes, 4 % on 28 x 28).
//
// LDS holds both operands slot-major, [slot][part][channel]: a lane fetches its slot from eight channel planes (a wavefront's
// load: 32 consecutive pixels of two planes, the channel's offset is uniform), and stores eight channels at once. The matrix
// instruction wants eight consecutive slots of a channel per lane; the transposing LDS read (ds_read_b64_tr_b16) delivers
// four per lane and instruction. A tap is then a constant row offset of the read: no shifting of registers (in the earlier
// filter-row kernel, which kept rows of pixels per channel, shifting and masking the fragments was a third of the vector
// work).
//
// Every float in three bfloat16 parts, which are the value exactly, and six products of parts added up, as in conv_same_f32x3.h, which
// explains the error; the five small products have accumulators of their own, which leaves two roundings per sixteen slots.
// That takes a wavefront's registers to one block of 32 rows: with two (and one set of accumulators) large layers run a tenth
// faster, 220 TFLOP/s instead of 198, at 1.1 to 2.5 times the float instruction's error; as it is the error by 2-norm was 0.63 of
// that in the median of 300 drawn layers and 0.99 at most.
// One pass, float engine -> here: 32 x 256 x 13 x 13, 384 filters of 3x3 109 -> 67.5 us; 32 x 96 x 27 x 27, 256 of 5x5 277 -> 203.
#pragma once
#include "conv_same_f32x3.h"

namespace vdnn {

constexpr int WS_CH = 64;    // input channels of a workgroup's tile
constexpr int WS_SLICE = 32; // slots of a slice

struct WgradSame {
    const float* dy;
    const float* x;
    int N, K, C, H, W;   // K and C multiples of 8
    float* out;          // filter gradient target [K][C][S][S]
    float* partial;      // staging area: [split][K][S*S*C], column = tap*C + c
    long partial_stride; // K*S*S*C
    float alpha;
    int accumulate;
    float* bias_partial; // optional: [K][bias_splits], written by the workgroups of the centre filter row and the first channel block
    int bias_splits;
    int slots, step_rows, step_cols; // of the whole reduction; a slice's 32 slots as whole rows and a rest
};

typedef short short4v __attribute__((ext_vector_type(4)));

// d.M = K, d.K = N * H * (W + S/2) slots; d.mtiles tiles of 64 output channels, d.ntiles = S * ceil(C / 64) (filter row fastest),
// d.splits reduction splits of d.kchunk slots (a multiple of 32).
template <int S>
__global__ void __launch_bounds__(NT, 2) wgrad_same_kernel(const WgradSame g, const GemmDims d) {
    constexpr int PAD = S / 2, TM = 64, SL = WS_SLICE;
    // rows of whole groups of eight words and an odd number of them: the four slots of a transposing read fall on different banks
    constexpr int AROW = 3 * TM + 16, BROW = 3 * WS_CH + 16, BSLOTS = SL + S - 1; // 16-bit units
    static_assert((AROW / 2) % 16 == 8 && (BROW / 2) % 16 == 8, "bank spread");
    __shared__ __attribute__((aligned(16))) unsigned short As[2][SL * AROW];
    __shared__ __attribute__((aligned(16))) unsigned short Bs[2][BSLOTS * BROW]; // x slots PAD before the slice to PAD behind it

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ntiles_all = d.mtiles * d.ntiles;
    const int bid = xcd_remap(blockIdx.x, gridDim.x);
    const int tile = bid % ntiles_all, ks = bid / ntiles_all;
    const int mt = tile % d.mtiles, nt = tile / d.mtiles;
    const int r = nt % S, c0 = (nt / S) * WS_CH;
    const int m0 = mt * TM;
    const int k_begin = ks * d.kchunk;
    const int k_end = min(d.K, k_begin + d.kchunk);
    const int H = g.H, W = g.W, WP = W + PAD, HW = H * W;

    const int n_first = k_begin / (H * WP);
    int n_last = (k_end + PAD - 1) / (H * WP);
    if (n_last > g.N - 1) n_last = g.N - 1;
    const __amdgpu_buffer_rsrc_t rsA = make_rsrc(g.dy + (long)n_first * g.K * HW, clamp_range((long)(n_last - n_first + 1) * g.K * HW * 4));
    const __amdgpu_buffer_rsrc_t rsB = make_rsrc(g.x + (long)n_first * g.C * HW, clamp_range((long)(n_last - n_first + 1) * g.C * HW * 4));

    // This lane's slot of a slice and its group of eight channels among the wavefront's sixteen: four slots of one group beside
    // four of the other in every eight lanes, whose 128-bit stores then tile the banks.
    const int slot = (lane & 3) | ((lane >> 3) << 2), grp = (lane >> 2) & 1;
    // a slot's position: image row, column, byte offset of its sample behind the first (dy counts K planes a sample, x C)
    struct Pos { int t, n, p, q; };
    auto at_slot = [&](int t) {
        Pos s;
        s.t = t;
        const int row = t / WP;
        s.q = t - row * WP;
        s.n = row / H;
        s.p = row - s.n * H;
        s.n -= n_first;
        return s;
    };
    auto advance = [&](Pos& s) {
        s.t += SL; s.q += g.step_cols; s.p += g.step_rows;
        const bool wrap = s.q >= WP;
        s.q -= wrap ? WP : 0; s.p += wrap ? 1 : 0;
        const bool next = s.p >= H; // (at most one sample: the launcher asks for planes of more rows than a slice spans)
        s.p -= next ? H : 0; s.n += next ? 1 : 0;
    };
    Pos pa = at_slot(k_begin + slot), pb = at_slot(k_begin + PAD + slot);
    // byte offsets of a lane's channel group, or out of range where the operand has no such channels; the wavefront's own
    // sixteen channels ride in the scalar offset
    const int grpA = m0 + 16 * wave + 8 * grp < g.K ? 8 * grp * HW * 4 : OOB;
    const int grpB = c0 + 16 * wave + 8 * grp < g.C ? 8 * grp * HW * 4 : OOB;

    float fa[8], fb[8]; // what a slice's fetch leaves in registers: eight channels of a slot, of dy and of x
    auto fetch = [&] {
        {
            const bool ok = pa.t < k_end && pa.q < W;
            const int at = pa.n * (g.K * HW * 4) + (pa.p * W + pa.q) * 4;
            const int voff = ok && grpA != OOB ? at + grpA : OOB;
            const int soff = (m0 + 16 * wave) * HW * 4;
#pragma unroll
            for (int e = 0; e < 8; e++) fa[e] = buf_load(rsA, voff, soff + e * HW * 4);
            advance(pa);
        }
        {
            const int row = pb.p + r - PAD;
            const bool ok = (unsigned)row < (unsigned)H && pb.q < W && grpB != OOB;
            const int voff = ok ? pb.n * (g.C * HW * 4) + (row * W + pb.q) * 4 + grpB : OOB;
            const int soff = (c0 + 16 * wave) * HW * 4;
#pragma unroll
            for (int e = 0; e < 8; e++) fb[e] = buf_load(rsB, voff, soff + e * HW * 4);
            advance(pb);
        }
    };
    // eight channels of a slot to LDS, one 128-bit store per part
    auto store8 = [](unsigned short* at, int part_stride, const float (&v)[8]) {
        uintx4 p[3];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            unsigned q0, q1, q2;
            split3_pair(v[2 * k], v[2 * k + 1], q0, q1, q2);
            p[0][k] = q0; p[1][k] = q1; p[2][k] = q2;
        }
#pragma unroll
        for (int k = 0; k < 3; k++) *(uintx4*)(at + k * part_stride) = p[k];
    };
    // of this lane's slots, per channel: sixteen slices at a time, so that no chain of additions grows long
    float bias_sum[8], bias_part[8];
#pragma unroll
    for (int e = 0; e < 8; e++) bias_sum[e] = bias_part[e] = 0.0f;
    auto flush_bias = [&] {
#pragma unroll
        for (int e = 0; e < 8; e++) { bias_sum[e] += bias_part[e]; bias_part[e] = 0.0f; }
    };
    auto stash = [&](int buf, auto with_bias) {
        store8(As[buf] + slot * AROW + 16 * wave + 8 * grp, TM, fa);
        if constexpr (decltype(with_bias)::value) {
#pragma unroll
            for (int e = 0; e < 8; e++) bias_part[e] += fa[e];
        }
        store8(Bs[buf] + (S - 1 + slot) * BROW + 16 * wave + 8 * grp, WS_CH, fb);
    };
    // the last S - 1 x slots of a buffer are the first of the next one
    auto carry = [&](int from, int to) {
        constexpr int PIECES = 3 * WS_CH / 8;
        if (tid < (S - 1) * PIECES) {
            const int row = tid / PIECES, col = 8 * (tid - row * PIECES);
            *(uintx4*)(Bs[to] + row * BROW + col) = *(const uintx4*)(Bs[from] + (SL + row) * BROW + col);
        }
    };

    floatx16 acc[S], low[S]; // the products 0 x 0, and the small ones
#pragma unroll
    for (int s = 0; s < S; s++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc[s][v] = low[s][v] = 0.0f;

    // The transposing read: sixteen lanes read four slots of sixteen channels (lane i slot i/4, channels 4 (i%4) .. + 3) and
    // get, each, one channel's four slots. Lane l of a fragment holds channel l % 32, slots 8 (l / 32) .. + 7: two reads.
    const int l32 = lane & 31, lk = lane >> 5, l16 = lane & 15;
    const int wm0 = (wave & 1) * 32, wc0 = (wave >> 1) * 32;
    const int frow = 8 * lk + (l16 >> 2), fcol = 16 * ((lane >> 4) & 1) + 4 * (l16 & 3);
    typedef __attribute__((address_space(3))) short4v LdsV4;
    auto read_frag = [](const unsigned short* at, int row_stride) {
        const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsV4*)at);
        const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsV4*)(at + 4 * row_stride));
        typedef short short8v __attribute__((ext_vector_type(8)));
        return __builtin_bit_cast(bf16x8, (short8v)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    };
    auto multiply = [&](int buf, int h) {
        const unsigned short* ap = As[buf] + (16 * h + frow) * AROW + wm0 + fcol;
        const unsigned short* bp = Bs[buf] + (16 * h + frow) * BROW + wc0 + fcol;
        bf16x8 a[3];
#pragma unroll
        for (int k = 0; k < 3; k++) a[k] = read_frag(ap + k * TM, AROW);
#pragma unroll
        for (int s = 0; s < S; s++) {
            bf16x8 b[3];
#pragma unroll
            for (int k = 0; k < 3; k++) b[k] = read_frag(bp + s * BROW + k * WS_CH, BROW);
            auto product = [&](floatx16& to, int ka, int kb) { to = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[ka], b[kb], to, 0, 0, 0); };
            product(acc[s], 0, 0);
            product(low[s], 0, 1); product(low[s], 1, 0);
            product(low[s], 1, 1); product(low[s], 0, 2); product(low[s], 2, 0);
        }
    };

    const int nslices = (k_end - k_begin + SL - 1) / SL;
    // Slice i (LDS buffers i % 2): multiply its first half; write slice i + 1, fetched a slice ago, to the other buffers; fetch
    // slice i + 2; multiply the second half; barrier. Fetches past the end of the range give zeros that are never used.
    auto run = [&](auto with_bias) {
        fetch();
        stash(0, with_bias);
        // the S - 1 x slots ahead of the first slice: one channel per lane, wavefront = slot
        if (wave < S - 1) {
            const int t = k_begin - PAD + wave;
            const Pos s = at_slot(t < 0 ? 0 : t);
            const int row = s.p + r - PAD, c = c0 + lane;
            // (a slot of the sample before the descriptor's first one is the zero behind its last row)
            const bool ok = t >= 0 && s.n >= 0 && (unsigned)row < (unsigned)H && s.q < W && c < g.C;
            unsigned p0, p1, p2;
            split3_pair(buf_load(rsB, ok ? s.n * (g.C * HW * 4) + (c * HW + row * W + s.q) * 4 : OOB, 0), 0.0f, p0, p1, p2);
            unsigned short* at = Bs[0] + wave * BROW + lane;
            at[0] = (unsigned short)p0; at[WS_CH] = (unsigned short)p1; at[2 * WS_CH] = (unsigned short)p2;
        }
        fetch();
        __syncthreads();
        auto slice = [&](auto parity) {
            constexpr int cur = decltype(parity)::value;
            multiply(cur, 0);
            stash(cur ^ 1, with_bias);
            carry(cur, cur ^ 1);
            fetch();
            multiply(cur, 1);
            __syncthreads();
        };
        for (int i = 0; i < nslices; i += 2) {
            slice(std::integral_constant<int, 0>{});
            if (i + 1 < nslices) slice(std::integral_constant<int, 1>{});
            if constexpr (decltype(with_bias)::value) {
                if ((i & 15) == 14) flush_bias();
            }
        }
        if constexpr (decltype(with_bias)::value) flush_bias();
    };
    if (g.bias_partial) run(std::true_type{});
    else run(std::false_type{});
    if (g.bias_partial && nt == PAD) {
        // the 32 slots of a channel: lanes that differ in bits 0, 1, 3, 4, 5
#pragma unroll
        for (int e = 0; e < 8; e++) {
            float v = bias_sum[e];
            v += __shfl_xor(v, 1); v += __shfl_xor(v, 2); v += __shfl_xor(v, 8); v += __shfl_xor(v, 16); v += __shfl_xor(v, 32);
            const int m = m0 + 16 * wave + 8 * grp + e;
            if (slot == 0 && m < g.K) g.bias_partial[(long)m * g.bias_splits + ks] = v;
        }
    }

    // a result that is not finite: the wavefront's block again, with the float instruction (see conv_same_f32x3.h)
    float bad = 0.0f;
#pragma unroll
    for (int s = 0; s < S; s++)
#pragma unroll
        for (int v = 0; v < 16; v++) {
            acc[s][v] += low[s][v];
            bad = __fmaf_rn(acc[s][v], 0.0f, bad);
        }
    if (__any(bad != 0.0f)) {
#pragma unroll
        for (int s = 0; s < S; s++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[s][v] = 0.0f;
#pragma unroll 1
        for (int t = k_begin; t < k_end; t += 2) {
            const Pos s0 = at_slot(t + lk);
            const bool okA = t + lk < k_end && s0.q < W;
            const int row = s0.p + r - PAD, m = m0 + wm0 + l32, c = c0 + wc0 + l32;
            const float a = buf_load(rsA, okA && m < g.K ? s0.n * (g.K * HW * 4) + (m * HW + s0.p * W + s0.q) * 4 : OOB, 0);
#pragma unroll
            for (int s = 0; s < S; s++) {
                const int col = s0.q + s - PAD;
                const bool ok = okA && (unsigned)row < (unsigned)H && (unsigned)col < (unsigned)W && c < g.C;
                const float b = buf_load(rsB, ok ? s0.n * (g.C * HW * 4) + (c * HW + row * W + col) * 4 : OOB, 0);
                acc[s] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc[s], 0, 0, 0);
            }
        }
    }

    // acc[s][v]: output channel m0 + wm0 + 8*(v/4) + 4*lk + v%4, input channel c0 + wc0 + l32, tap (r, s)
    const int c = c0 + wc0 + l32;
    const int ncols = S * S * g.C;
    const bool to_partial = d.splits > 1;
#pragma unroll
    for (int s = 0; s < S; s++) {
        const int tap = S * r + s;
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const int m = m0 + wm0 + 8 * (v / 4) + 4 * lk + (v % 4);
            if (m >= g.K || c >= g.C) continue;
            const float a = acc[s][v];
            if (to_partial) g.partial[(long)ks * g.partial_stride + (long)m * ncols + (long)tap * g.C + c] = a;
            else {
                const long idx = (long)m * ncols + (long)c * (S * S) + tap;
                g.out[idx] = g.accumulate ? __fmaf_rn(g.alpha, a, g.out[idx]) : g.alpha * a;
            }
        }
    }
}

} // namespace vdnn
