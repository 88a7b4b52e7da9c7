// Forward and backward data of bfloat16 layers on the bfloat16 engine (igemm_bf16_kernel) from a copy of the source tensor with the
// channels of a pixel side by side.
//
// In the tensors' own order (NCHW) a slice's 32 channels of a pixel lie a plane apart: a thread fetches sixteen 16-bit values per slice
// (eight 32-bit ones where pixels come in pairs), and every tap fetches them again. A kernel of its own lays the samples out as
// [sample][pixel][block of channels][32 values] in the staging area, zeros behind the last channel, and a thread of the product
// then fetches its part of a slice with one 128-bit load per pixel. The same products in the same order, the same bits.
// The product itself is bound by LDS: a slice of a 128x128 tile is 32 KB of fragments read and 16 KB written for 256 cycles of matrix
// instructions, at 128 bytes a cycle.
// One call: forward 30 x 359 x 18 x 18, 704 filters of 5x5 at stride 2 129 -> 85 us; 57 x 179 x 40 x 25, 13 of 5x5 126 -> 71; 73 x 220 x 29 x 29, 96 of 3x3
// 72 -> 60; backward 64 x 96 x 27 x 27, 256 of 5x5 295 -> 257.
#pragma once
#include "mfma_bf16.h"

namespace vdnn {

// One thread per pixel and block of channels. Bound by the memory it moves.
__global__ void __launch_bounds__(256) stage_pixels_kernel(const bf16_t* __restrict__ src, unsigned short* __restrict__ out, int C, int plane, int total, int blocks) {
    const int j = blockIdx.x * 256 + threadIdx.x, cb = blockIdx.y;
    if (j >= total) return;
    const int n = j / plane, pix = j - n * plane, c0 = cb * KH;
    const bf16_t* p = src + ((long)n * C + c0) * plane + pix;
    unsigned v[KH];
#pragma unroll
    for (int c = 0; c < KH; c++) {
        v[c] = p[(long)min(c, C - 1 - c0) * plane].bits;
        if (c0 + c >= C) v[c] = 0;
    }
    uintx4* o = (uintx4*)(out + ((long)j * blocks + cb) * KH);
#pragma unroll
    for (int q = 0; q < 4; q++) {
        uintx4 w;
#pragma unroll
        for (int e = 0; e < 4; e++) w[e] = v[8 * q + 2 * e] | v[8 * q + 2 * e + 1] << 16;
        o[q] = w;
    }
}

// The im2col operand from the copy: a pixel's 32 values of a tap and block. thread t: values 8*(t%4) .. +7 of pixels rows_by_four_lanes(t) + 64*i.
// MIRROR (backward data at stride 1): the filter's taps run backwards over the window, whose padding is then R - 1 - pad.
template <bool MIRROR>
struct LoadPixStaged {
    const unsigned short* src;
    int Hs, Ws, OH, OW, R, S, ph, pw, sh, sw; // of the window over the source
    int row;                                  // 16-bit values of a pixel
    int nsamples;                             // (the copy is no larger than the staging area)
    FastDiv divRS, divS;
    template <int T> struct Regs { uintx4 v[T / 64]; };
    template <int T> struct State { int vbase[T / 64]; unsigned inv[T / 64]; __amdgpu_buffer_rsrc_t rsrc; };
    template <int T>
    __device__ __forceinline__ void init(State<T>& st, int j0, int tid, int ncols, int) const {
        // the descriptor starts `lead` values ahead of the copy, so that every offset below is non-negative (what lies there is never fetched)
        const int opix = OH * OW, lead = (ph * Ws + pw) * row;
        st.rsrc = make_rsrc(src - lead, (unsigned)((nsamples * Hs * Ws * row + lead) * 2));
#pragma unroll
        for (int i = 0; i < T / 64; i++) {
            const int j = j0 + rows_by_four_lanes(tid) + 64 * i;
            const bool valid = j < ncols;
            const int jj = valid ? j : j0, n = jj / opix, pix = jj - n * opix, oh = pix / OW, ow = pix - oh * OW;
            st.vbase[i] = ((n * Hs + oh * sh) * Ws + ow * sw) * row * 2 + 16 * (tid & 3);
            const unsigned vrow = valid ? valid_window_bits(oh * sh - ph, R, Hs) : 0u, vcol = valid_window_bits(ow * sw - pw, S, Ws);
            unsigned v = 0;
            for (int r = 0; r < R; r++) if ((vrow >> r) & 1u) v |= vcol << (r * S);
            st.inv[i] = ~v;
        }
    }
    template <int T>
    __device__ __forceinline__ void load(State<T>& st, int kk0, int, int, Regs<T>& r) const {
        const int slice = kk0 / KH, cb = divRS.div(slice), at = slice - cb * (R * S);
        const int tap = MIRROR ? R * S - 1 - at : at, tr = divS.div(tap), ts = tap - tr * S;
        const int soff = ((tr * Ws + ts) * row + cb * KH) * 2;
#pragma unroll
        for (int i = 0; i < T / 64; i++) r.v[i] = __builtin_bit_cast(uintx4, __builtin_amdgcn_raw_buffer_load_b128(st.rsrc, st.vbase[i] | bit_to_all_ones(st.inv[i], tap), soff, 0));
    }
    template <int T>
    __device__ static __forceinline__ void store(unsigned short* lds, int tid, const Regs<T>& r) {
#pragma unroll
        for (int i = 0; i < T / 64; i++) *(uintx4*)(lds + (rows_by_four_lanes(tid) + 64 * i) * HSTRIDE + 8 * (tid & 3)) = r.v[i];
    }
};
} // namespace vdnn
