// Backward data of strided layers by residue classes.
//
// A pixel (h, w) of dx takes part only in the taps r = (h + ph) mod sh, + sh, + 2 sh, ... (and columns alike): the pixels
// of one residue class (a, b) = ((h + ph) mod sh, (w + pw) mod sw) are the result of a backward data at stride 1 whose
// window is every sh-th row and sw-th column of the filter, starting at (a, b). Through one product over all R*S taps
// (a gather with two divisions per element, three quarters of its elements zero at stride 2) the matrix cores did sh*sw
// times the work at a third of their rate; here each class is a product of its own over its own taps:
//   pack_filter_classes_kernel  the filter bank per class, blocked tap-major, output channels padded to whole slices with
//                               zeros (so that odd channel counts take the loaders whose tap is a per-slice value)
//   igemm_classes_kernel        all classes in one launch, the longest reductions first; each writes its own compact
//                               [n][c][pixels of the class], split reductions one such block per split
//   merge_classes_kernel        dx from them: ordered sum of the splits, gate, whole rows of dx per store
// One call, before -> after (floats): 21 x 70 x 53 x 37, 130 filters of 3x3, stride 2: 197 -> 64 us; 32 x 256 x 28 x 28, 512
// of 3x3: 937 -> 187; 128 x 64 x 112 x 112, 64 of 3x3: 1955 -> 919; 1 x 64 x 56 x 56, 128 of 3x3: 41 -> 17; 64 x 128 x 56 x 56,
// 128 of 1x1 (a quarter of the pixels have a tap): 141 -> 134. Layers of short reductions stay with the one product (classes_pay
// in conv.hip).
#pragma once
#include "conv_loaders_tap.h"

namespace vdnn {

constexpr int kStridedClasses = 4; // residue classes of a launch: strides with sh * sw up to this

template <class E>
struct StridedClass {
    LoadDenseRed<true> al;
    LoadIm2colPixTap<1, E, true> bl;
    StoreNCHW<float> ep;
    GemmDims d;
    int blocks;
};
template <class E>
struct StridedLaunch {
    StridedClass<E> c[kStridedClasses];
    int count;
};

template <class E, int AHEAD>
__global__ void __launch_bounds__(NT) igemm_classes_kernel(const StridedLaunch<E> s) {
    int c = 0, bid = blockIdx.x;
    while (c + 1 < s.count && bid >= s.c[c].blocks) bid -= s.c[c++].blocks;
    igemm_small_tile<AHEAD, false>(s.c[c].al, s.c[c].bl, s.c[c].ep, s.c[c].d, bid, s.c[c].blocks);
}

// where a class's filter taps, pixels and partial sums lie
struct StridedClassGeo {
    int rows, cols, taps;       // window
    int u0, v0;                 // first source row / column of the class's first pixel's tap 0
    int opix_h, opix_w;         // pixels of the class
    long filter_first;          // elements before its filter bank
    long result_first;          // elements before its result
    int splits;                 // 0: no tap reaches the class, dx is zero there
};
struct StridedGeo {
    StridedClassGeo c[kStridedClasses]; // class a * sw + b
    int sh, sw, ph, pw;
    int C, H, W, R, S, K, Kpad;
};

// packed[class][row][(kb * taps + tap) * 16 + l] = w[kb * 16 + l][row][tap of the class], zero behind the last channel
template <bool ROUND>
__global__ void __launch_bounds__(256) pack_filter_classes_kernel(const float* __restrict__ w, float* __restrict__ packed, StridedGeo g, long total) {
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i >= total) return;
    int cls = 0;
    for (int c = 1; c < g.sh * g.sw; c++) if (g.c[c].taps > 0 && i >= g.c[c].filter_first) cls = c;
    const StridedClassGeo& q = g.c[cls];
    const long j = i - q.filter_first;
    const int per_row = g.Kpad * q.taps;
    const int row = (int)(j / per_row), kk = (int)(j - (long)row * per_row);
    const int l = kk & 15, slice = kk >> 4;
    const int kb = slice / q.taps, tap = slice - kb * q.taps;
    const int r = cls / g.sw + g.sh * (tap / q.cols), s = cls % g.sw + g.sw * (tap % q.cols);
    const int k = kb * 16 + l;
    float v = 0.0f;
    if (k < g.K) v = w[(((long)k * g.C + row) * g.R + r) * g.S + s];
    packed[i] = ROUND ? round_to_bf16_value(v) : v;
}

// Bound by the memory it moves: neighbouring threads read neighbouring elements of sw classes. A launch covers no more
// elements than the staging area holds (2^24), so that 32-bit indexes and divisions do.
template <class E>
__global__ void __launch_bounds__(256) merge_classes_kernel(const float* __restrict__ part, E* dx, const E* gate, StridedGeo g, int N, unsigned total) {
    const unsigned i = blockIdx.x * 256 + threadIdx.x;
    if (i >= total) return;
    const unsigned row = i / (unsigned)g.W, w = i - row * (unsigned)g.W;
    const unsigned plane = row / (unsigned)g.H, h = row - plane * (unsigned)g.H; // n * C + c
    const unsigned hq = (h + g.ph) / (unsigned)g.sh, wq = (w + g.pw) / (unsigned)g.sw;
    const unsigned a = h + g.ph - hq * g.sh, b = w + g.pw - wq * g.sw;
    const StridedClassGeo& q = g.c[a * g.sw + b];
    float v = 0.0f;
    if (q.splits > 0) {
        const long opix = (long)q.opix_h * q.opix_w, stride = (long)N * g.C * opix;
        const float* p = part + q.result_first + (long)plane * opix + (long)(hq - q.u0) * q.opix_w + (wq - q.v0);
        for (int s = 0; s < q.splits; s++) v += p[s * stride];
    }
    if (gate) v = load_elem(gate + i) > 0.0f ? v : 0.0f;
    store_elem(dx + i, v);
}

} // namespace vdnn
