// fp32 MFMA tile engine shared by the convolution and fully-connected kernels.
//
// One workgroup of 256 threads (4 wavefronts of 64) produces a TM x TN tile of
//     Out[m][j] = sum_kk A[m][kk] * B[kk][j]
// from KB-deep slices staged in LDS. In the large tiles (igemm_tile) each wavefront owns a 64x64 sub-tile = 2x2 MFMA tiles of
// v_mfma_f32_32x32x2_f32 (64 accumulator registers per lane), in the 64x64 tile (igemm_small_tile) one MFMA tile. Operands come from "loader" policies:
// a loader says how element (row, kk) of its operand is fetched from global memory (a dense matrix,
// a filter bank, or an im2col view of an NCHW tensor computed on the fly - the im2col matrix only
// ever exists as LDS tiles). Global loads run AHEAD slices ahead in registers beside the one in
// LDS (one, two or four), LDS is double-buffered, and the loop has one barrier per slice and no branch but, with AHEAD > 1, those of
// the slices that are left behind whole rounds of AHEAD.
//
// The matrix pipe and the vector ALU of a SIMD do not overlap well, so every vector instruction in
// the loop costs MFMA time. The loaders therefore fetch through buffer descriptors: an element that
// must read as zero (outside the matrix, a padding tap, beyond the reduction range) is given an
// out-of-range offset and the hardware returns 0 - no branch, no select, and nothing depends on the
// loaded value until it is written to LDS. Uniform parts of an address go into the scalar offset.
//
// LDS layouts:
//   reduction-major operand (a thread's load runs along kk): lds[row * (KB+4) + kk], moved as
//       128-bit chunks of four consecutive kk where the source allows
//   row-major operand (lanes run along the row/column index): lds[kk * T + row]
// MFMA operand mapping for 32x32x2: lane l supplies A[i = l%32][k = l/32] and B[k = l/32][j = l%32];
// result register v of lane l is D[8*(v/4) + 4*(l/32) + v%4][l%32]. The order in which the KB
// reduction indices of a slice are consumed is free as long as A and B agree: step (g, i) uses
// k = 8g + 4*(l/32) + i, so a lane's four values of a reduction-major operand are one 128-bit read.
#pragma once
#include <hip/hip_runtime.h>

namespace vdnn {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int KB = 16;              // reduction depth of one LDS slice
constexpr int NT = 256;             // threads per workgroup
constexpr int RED_STRIDE = KB + 4;  // row stride of a reduction-major LDS tile (80 bytes: 128-bit reads of 8 consecutive rows hit 8 different bank groups)
constexpr int OOB = -1;             // byte offset that is out of range for every descriptor
constexpr int SENT = 0x40000000;    // out-of-range marker that survives one addition of a second offset below 1 GiB
constexpr unsigned MAX_SUM_RANGE = 0x40000000u; // descriptors addressed with summed offsets must be smaller than this

// MI355X has 8 XCDs, each with its own L2; consecutive workgroup ids are dealt round-robin to the
// XCDs. Remap so that consecutive *logical* tiles (which share operand tiles) land on one XCD.
__device__ __forceinline__ int xcd_remap(int bid, int nblocks) {
    constexpr int XCD = 8;
    const int per = nblocks / XCD, rem = nblocks % XCD;
    const int xcd = bid % XCD, idx = bid / XCD;
    // XCD x holds logical ids [start_x, start_x + per + (x < rem))
    const int start = xcd * per + (xcd < rem ? xcd : rem);
    return start + idx;
}

// Division of a small non-negative integer by a loop-invariant divisor as a multiply-high with the
// 33-bit constant ceil(2^32 / d), kept as (hi, lo) so that d == 1 needs no branch.
// Exact while x * d < 2^32 (callers bound x below 2^24 and d by 256).
struct FastDiv {
    unsigned lo, hi;
    __host__ __device__ static FastDiv make(int divisor) {
        const unsigned long long m = (0x100000000ull + (unsigned)divisor - 1) / (unsigned)divisor;
        FastDiv f;
        f.lo = (unsigned)m;
        f.hi = (unsigned)(m >> 32);
        return f;
    }
    __device__ __forceinline__ int div(int x) const { return (int)(__umulhi((unsigned)x, lo) + (unsigned)x * hi); }
};

// ---- buffer descriptors: loads that return 0 outside [0, bytes) ----------------------------------
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* p, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000);
}
// voff: per-lane byte offset; soff: wave-uniform byte offset. Out of range if voff + soff >= bytes
// (no 32-bit wrap-around: OOB + anything stays out of range).
__device__ __forceinline__ float buf_load(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}
__device__ __forceinline__ floatx4 buf_load4(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    return __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}
// Descriptor range for `bytes` remaining after the base, clamped to what a descriptor can hold.
__device__ __forceinline__ unsigned clamp_range(long bytes) {
    return bytes <= 0 ? 0u : (bytes > 0xFFFFFFF0l ? 0xFFFFFFF0u : (unsigned)bytes);
}

// ---- element types of activation tensors -------------------------------------------------------------
// Activations are float or bfloat16 in memory; every kernel computes in float. A bf16 value is the
// upper half of the float with the same value; storing rounds to nearest, ties to even, NaN stays NaN.
struct bf16_t { unsigned short bits; };
template <class E> struct ElemBytes { static constexpr int V = (int)sizeof(E); };

__host__ __device__ __forceinline__ float bf16_bits_to_float(unsigned bits) {
    return __builtin_bit_cast(float, bits << 16);
}
// On the device the conversion is one instruction (v_cvt_pk_bf16_f32, two values at a time); it gives the bits of
// the arithmetic below for every one of the 2^32 inputs, NaN payloads and denormals included.
__host__ __device__ __forceinline__ unsigned short float_to_bf16_bits(float f) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_bit_cast(unsigned short, (__bf16)f);
#else
    unsigned u = __builtin_bit_cast(unsigned, f);
    if ((u & 0x7FFFFFFFu) > 0x7F800000u) return (unsigned short)((u >> 16) | 0x40u);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (unsigned short)(u >> 16);
#endif
}
// two values in one word, the first in the lower half
__device__ __forceinline__ unsigned pack2_bf16(float lo, float hi) {
    typedef float float_x2 __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16_x2 __attribute__((ext_vector_type(2)));
    float_x2 f; f.x = lo; f.y = hi;
    return __builtin_bit_cast(unsigned, __builtin_convertvector(f, bf16_x2));
}
__device__ __forceinline__ float load_elem(const float* p) { return *p; }
__device__ __forceinline__ float load_elem(const bf16_t* p) { return bf16_bits_to_float(p->bits); }
__device__ __forceinline__ void store_elem(float* p, float v) { *p = v; }
__device__ __forceinline__ void store_elem(bf16_t* p, float v) { p->bits = float_to_bf16_bits(v); }

// one element / four consecutive elements through a descriptor, as float (offsets in bytes)
// max(v, 0) that lets NaN through
__device__ __forceinline__ float relu_value(float v) { return v > 0.0f ? v : (v != v ? v : 0.0f); }

template <class E> __device__ __forceinline__ float buf_load_e(__amdgpu_buffer_rsrc_t r, int voff, int soff);
template <> __device__ __forceinline__ float buf_load_e<float>(__amdgpu_buffer_rsrc_t r, int voff, int soff) { return buf_load(r, voff, soff); }
template <> __device__ __forceinline__ float buf_load_e<bf16_t>(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    return bf16_bits_to_float((unsigned)(unsigned short)__builtin_amdgcn_raw_buffer_load_b16(r, voff, soff, 0));
}
template <class E> __device__ __forceinline__ floatx4 buf_load4_e(__amdgpu_buffer_rsrc_t r, int voff, int soff);
template <> __device__ __forceinline__ floatx4 buf_load4_e<float>(__amdgpu_buffer_rsrc_t r, int voff, int soff) { return buf_load4(r, voff, soff); }
template <> __device__ __forceinline__ floatx4 buf_load4_e<bf16_t>(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    typedef unsigned uintx2 __attribute__((ext_vector_type(2)));
    const uintx2 w = __builtin_bit_cast(uintx2, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
    floatx4 v;
    v.x = __builtin_bit_cast(float, w.x << 16); v.y = __builtin_bit_cast(float, w.x & 0xFFFF0000u);
    v.z = __builtin_bit_cast(float, w.y << 16); v.w = __builtin_bit_cast(float, w.y & 0xFFFF0000u);
    return v;
}

// ---- LDS tile geometry ------------------------------------------------------------------------------
template <int T, bool RED_MAJOR>
struct LdsTile {
    static constexpr int SIZE = RED_MAJOR ? T * RED_STRIDE : KB * T;
    static constexpr int ROW_STRIDE = RED_MAJOR ? RED_STRIDE : 1;
};

// Four reduction values (k = 8g + 4*lk + i, i = 0..3) of row l32 of a 32-row tile at `tile`.
template <int T, bool RED_MAJOR>
__device__ __forceinline__ floatx4 read_frag(const float* tile, int l32, int lk, int g) {
    if (RED_MAJOR) {
        return *(const floatx4*)(tile + l32 * RED_STRIDE + 8 * g + 4 * lk);
    } else {
        const float* p = tile + (8 * g + 4 * lk) * T + l32;
        floatx4 v;
        v.x = p[0]; v.y = p[T]; v.z = p[2 * T]; v.w = p[3 * T];
        return v;
    }
}

// row of a 32x32 result tile that register v of a lane holds (l >> 5 = lk)
__device__ __forceinline__ int result_row(int v, int lk) { return 8 * (v / 4) + 4 * lk + v % 4; }

// Launch geometry of one igemm call. Split s covers reduction indices [s*kchunk, min(K, (s+1)*kchunk)).
// full_tiles > 0 (tail mode): the first full_tiles tiles are computed whole by one workgroup each, only the
// remaining tiles - the ones that would start a nearly empty last round - are split.
struct GemmDims {
    int M, N, K;
    int mtiles, ntiles, splits, kchunk;
    int full_tiles;
    unsigned* counters = nullptr; // the 64x64 tile: splits are added up by the workgroup that ends last (sum_splits), one counter a split tile
};

// The rounds' part of the estimate of choose_splits: s splits of a reduction of K for `tiles` output tiles; *splits: how many that makes.
static inline double split_rounds_us(long tiles, long K, long s, int num_cu, double us_per_slice, long* splits = nullptr) {
    long kchunk = (K + s - 1) / s;
    kchunk = (kchunk + KB - 1) / KB * KB;
    const long made = (K + kchunk - 1) / kchunk;
    const long rounds = (tiles * made + num_cu - 1) / num_cu;
    const double eff = rounds == 1 ? 0.72 : rounds == 2 ? 0.92 : rounds == 4 ? 0.93 : rounds % 3 == 0 ? 1.0 : 0.97;
    if (splits) *splits = made;
    return (double)rounds * (double)(kchunk / KB + 6) * us_per_slice / eff;
}

// Number of reduction splits for a grid of `tiles` output tiles over a reduction of K, at most
// max_splits. Measured on the part: workgroups are resident three to a compute unit, so a grid runs
// fastest when it is a little under a multiple of the unit count, best a multiple of three units'
// worth; one more workgroup than that starts a nearly empty round. The estimate below counts, per
// compute unit, rounds x (slices per split + a fixed prologue/epilogue) with the measured efficiency
// of a round count, plus the traffic of writing and re-reading one partial result per split.
static inline int choose_splits(long tiles, long K, long max_splits, int num_cu, size_t out_bytes, double tile_flops_per_slice) {
    if (max_splits < 1) max_splits = 1;
    const long useful = 12l * num_cu / tiles + 1; // beyond twelve rounds the estimate only grows
    if (max_splits > useful) max_splits = useful;
    const double us_per_slice = tile_flops_per_slice / (118e6 / num_cu); // one unit at ~118 TFLOP/s / units
    const double us_per_split = (double)out_bytes * 2.0 / 4e6;           // partials at ~4 TB/s
    double best = 0.0;
    int best_s = 1;
    for (long s = 1; s <= max_splits; s++) {
        long splits;
        const double rounds_us = split_rounds_us(tiles, K, s, num_cu, us_per_slice, &splits);
        const double cost = rounds_us + (splits > 1 ? (double)splits * us_per_split : 0.0);
        if (s == 1 || cost < best) { best = cost; best_s = (int)s; }
    }
    return best_s;
}

// The 64x64 tile (wavefront tiles of 32x32): a quarter of the large tile's work per workgroup. A grid that leaves compute
// units idle, or ends in a nearly empty round, is cut four times finer, and a workgroup's prologue and epilogue (address
// set-up, the first slices' trip through memory, 16 stores per lane instead of 64, a kernel text a quarter as long to
// fetch) are that much shorter, which is most of a small layer's time. Twice the operand loads and LDS reads per matrix
// instruction make it 5-8 % slower where the grid fills the chip many times over.
// One call, floats, before -> after: 1x64x56x56 with 128 filters of 3x3 forward 24.6 -> 17.7 us; 4x8x10x10, 12 filters of
// 5x5 19.3 -> 8.9 us; 32x256x28x28, 256 filters of 3x3 304 -> 249 us (392 large tiles for 256 units); fully connected
// 25088 -> 4096 at 64 rows, filter update (four slices a tile) 311 -> 241 us.
// Which tile: the times of both are estimated, from 290 measured calls of 1 to 128 samples, 8 to 1024 channels, 1x1 to
// 5x5, planes of 7 to 56 pixels a side; the choice is within 3 % of the better one in all but a few of them.
// Products of more than kSmallTileOps operations keep the large tile whatever the estimates say: their grids seldom gain (the
// 64x64 tile is 5-8 % slower on a full chip), and large training steps keep the order of their sums. Reductions of up to
// kShortReduction are the exception: they take the 64x64 tile at any size, because a large tile is mostly prologue and
// epilogue there (strided backward data up to 4e9 operations, LoadCost in conv.hip). Their splits are this plan's,
// so a remainder behind whole rounds may be summed in another order than the large tile's; fully connected layers, whose rule
// is in fc.hip, keep the large tile's splits and with them its bits.
struct SmallTilePlan {
    int splits = 0;      // Splits of every tile, or (full_tiles > 0) of the tiles behind the first full_tiles
    long full_tiles = 0;
    double us = 0.0;
};
constexpr double kSmallTileOps = 3e10;
constexpr long kShortReduction = 192; // up to here a large tile is mostly prologue and epilogue: 1.3-2.5x on every grid measured
// load_cost: work of the loaders against those of the blocked tap-major order (1)
static inline SmallTilePlan small_tile_plan(long M, long N, long K, size_t partial_bytes, int num_cu, long min_slices, bool tail_mode, double load_cost) {
    constexpr double kSum = 4.0;                             // the second kernel of a split reduction, us
    constexpr long kPrologue = 8;                            // prologue and epilogue, in slices
    const double slice_us = 0.27 * load_cost;                // a unit's share of a 64x64x16 slice
    // a workgroup has one wavefront per SIMD: one or two of them do not cover the latency of their loads
    auto filled = [](long per_cu) { return per_cu <= 1 ? 0.66 : per_cu == 2 ? 0.86 : per_cu == 3 ? 0.97 : 1.0; };
    const long tiles = ((M + 63) / 64) * ((N + 63) / 64), slices = (K + KB - 1) / KB;
    const size_t out_bytes = (size_t)M * N * sizeof(float), tile_bytes = 64 * 64 * sizeof(float);
    const long by_depth = slices / min_slices > 1 ? slices / min_slices : 1, full = tiles / num_cu * num_cu, rem = tiles - full;
    SmallTilePlan best;
    // every tile split
    long cap = 8l * num_cu / tiles + 1;
    if (cap > by_depth) cap = by_depth;
    if (cap > (long)(partial_bytes / out_bytes)) cap = (long)(partial_bytes / out_bytes);
    if (cap < 1) cap = 1;
    for (long s = 1; s <= cap; s++) {
        const long rounds = (tiles * s + num_cu - 1) / num_cu;
        const double us = (double)rounds * (double)((slices + s - 1) / s + kPrologue) * slice_us / filled(rounds) +
                          (s > 1 ? kSum + (double)s * (double)out_bytes * 0.6 / 4e6 : 0.0);
        if (best.splits == 0 || us < best.us) { best.splits = (int)s; best.us = us; }
    }
    // only the tiles behind whole rounds split
    if (tail_mode && full > 0 && rem > 0) {
        long most = 4l * num_cu / rem + 1;
        if (most > by_depth) most = by_depth;
        if (most > (long)(partial_bytes / (rem * tile_bytes))) most = (long)(partial_bytes / (rem * tile_bytes));
        for (long s = 2; s <= most; s++) {
            const long f = full / num_cu, r = (rem * s + num_cu - 1) / num_cu;
            const double us = ((double)f * (double)(slices + 2) / filled(f) + (double)r * (double)((slices + s - 1) / s + kPrologue)) * slice_us +
                              kSum + (double)(s * rem) * (double)tile_bytes * 0.6 / 4e6;
            if (us < best.us) { best.splits = (int)s; best.full_tiles = full; best.us = us; }
        }
    }
    return best;
}
// The large tile's time on the same scale. whole_grids: the reduction is split whatever the number of tiles (backward
// filter, fully connected layers); otherwise only a grid below two workgroups a unit is, and a remainder behind rounds of
// three workgroups a unit runs in tail mode.
static inline double large_tile_us(long M, long N, long K, int TM, int TN, int splits, int num_cu, bool whole_grids, double load_cost) {
    constexpr double kSum = 4.0;
    const double slice_us = 2.0 * TM * TN * KB / (118e6 / num_cu);
    auto eff = [](long rounds) { return rounds == 1 ? 0.72 : rounds == 2 ? 0.92 : rounds == 4 ? 0.93 : rounds % 3 == 0 ? 1.0 : 0.97; };
    const long tiles = ((M + TM - 1) / TM) * ((N + TN - 1) / TN), slices = (K + KB - 1) / KB;
    if (whole_grids || tiles < 2l * num_cu) {
        const long rounds = (tiles * splits + num_cu - 1) / num_cu;
        return ((double)rounds * (double)((slices + splits - 1) / splits + 6) * slice_us / eff(rounds) + (splits > 1 ? (double)splits * (double)(M * N) * 8.0 / 4e6 : 0.0)) * 0.85 * load_cost +
               (splits > 1 ? kSum : 0.0);
    }
    const long slots = 3l * num_cu, rem = tiles % slots;
    const double us = (double)((tiles - rem) / num_cu) * (double)(slices + 2) * slice_us;
    if (tiles > slots && rem > 0 && 2 * rem <= slots)
        return (us + 3.0 * ((double)slices / (double)(slots / rem) + 6.0) * slice_us) * 0.88 * load_cost + kSum;
    const long last = (rem + num_cu - 1) / num_cu;
    return (us + (double)last * (double)(slices + 2) * slice_us / (last == 1 ? 0.72 : last == 2 ? 0.92 : 1.0)) * 0.88 * load_cost;
}

// The tile and the part of the reduction that a workgroup computes.
struct TilePlace {
    int tile, ks, m0, j0, k_begin, k_end;
    bool whole; // the whole reduction
};
__device__ __forceinline__ TilePlace tile_place(const GemmDims& d, int block, int blocks, int TM, int TN) {
    // m-tile fastest: workgroups that share a B tile (the large operand) are neighbours
    const int ntiles_all = d.mtiles * d.ntiles;
    TilePlace p;
    if (block < d.full_tiles) {
        p.tile = xcd_remap(block, d.full_tiles); p.ks = 0; p.whole = true;
    } else if (d.full_tiles > 0) {
        const int r = block - d.full_tiles, tl = ntiles_all - d.full_tiles;
        p.tile = d.full_tiles + r % tl; p.ks = r / tl; p.whole = false;
    } else {
        const int bid = xcd_remap(block, blocks);
        p.tile = bid % ntiles_all; p.ks = bid / ntiles_all; p.whole = d.splits == 1;
    }
    p.m0 = p.tile % d.mtiles * TM;
    p.j0 = p.tile / d.mtiles * TN;
    p.k_begin = p.whole ? 0 : p.ks * d.kchunk;
    p.k_end = p.whole ? d.K : min(d.K, p.k_begin + d.kchunk);
    return p;
}

// AHEAD: slices on their way from memory beside the one in LDS and the one that is being multiplied.
template <int TM, int TN, int AHEAD, class AL, class BL, class EP>
__device__ __forceinline__ void igemm_tile(const AL& al, const BL& bl, const EP& ep, const GemmDims& d, int block, int blocks) {
    constexpr int MI = 2, NJ = 2; // MFMA tiles of a wavefront
    constexpr int WAVES_M = TM / (32 * MI);
    static_assert(TM % (32 * MI) == 0 && TN % (32 * NJ) == 0 && WAVES_M * (TN / (32 * NJ)) == 4, "four wave tiles");
    using LA = LdsTile<TM, AL::RED_MAJOR>;
    using LB = LdsTile<TN, BL::RED_MAJOR>;
    __shared__ __attribute__((aligned(16))) float As[2][LA::SIZE];
    __shared__ __attribute__((aligned(16))) float Bs[2][LB::SIZE];

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const TilePlace at = tile_place(d, block, blocks, TM, TN);
    const int tile = at.tile, ks = at.ks, m0 = at.m0, j0 = at.j0, k_begin = at.k_begin, k_end = at.k_end;
    const bool whole = at.whole;

    typename AL::template State<TM> sa;
    typename BL::template State<TN> sb;
    al.template init<TM>(sa, m0, tid, d.M, k_begin);
    bl.template init<TN>(sb, j0, tid, d.N, k_begin);

    floatx16 acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[i][j][v] = 0.0f;

    const int wm0 = (wave % WAVES_M) * 32 * MI, wn0 = (wave / WAVES_M) * 32 * NJ;
    typename AL::template Regs<TM> ra[AHEAD];
    typename BL::template Regs<TN> rb[AHEAD];

    // Software pipeline, one barrier per slice - in the middle of it - and no branch within a slice.
    // A slice's 32 MFMAs per wavefront run as two groups of 16 (reduction indices 0-7 and 8-15).
    //   first half of slice s:  read the fragments of (s, group 1) from LDS buffer s%2, multiply group 0
    //                           (fragments already in registers), write the registers holding slice s+1
    //                           (fetched during slice s-AHEAD) to the other LDS buffer;
    //   barrier;
    //   second half:            issue the fetch of slice s+1+AHEAD into the same registers, read the fragments
    //                           of (s+1, group 0) from the buffer just completed, multiply group 1.
    // Each group's fragments are thus read while the previous group is multiplied, across the barrier as
    // well, so no wavefront waits for LDS; a global load has AHEAD slices of MFMA time to return. All
    // reads of a buffer precede the barrier after which it may be overwritten. Fetches past the end of
    // the range read as zero or are never used: buffer loads cannot fault, the last rounds need no guard.
    const int nslices = (k_end - k_begin + KB - 1) / KB;
    const int l32 = lane & 31, lk = lane >> 5;
    constexpr int A_TILE = 32 * LA::ROW_STRIDE, B_TILE = 32 * LB::ROW_STRIDE;
    const int a_off = wm0 * LA::ROW_STRIDE, b_off = wn0 * LB::ROW_STRIDE;
    {
        typename AL::template Regs<TM> fa;
        typename BL::template Regs<TN> fb;
        al.template load<TM>(sa, k_begin, k_end, tid, fa);
        bl.template load<TN>(sb, k_begin, k_end, tid, fb);
        if constexpr (AHEAD == 1) {
            AL::template store<TM>(As[0], tid, fa);
            BL::template store<TN>(Bs[0], tid, fb);
        }
#pragma unroll
        for (int u = 0; u < AHEAD; u++) {
            al.template load<TM>(sa, k_begin + (u + 1) * KB, k_end, tid, ra[u]);
            bl.template load<TN>(sb, k_begin + (u + 1) * KB, k_end, tid, rb[u]);
        }
        if constexpr (AHEAD > 1) {
            AL::template store<TM>(As[0], tid, fa);
            BL::template store<TN>(Bs[0], tid, fb);
        }
    }
    __syncthreads();
    floatx4 a0[MI], b0[NJ], a1[MI], b1[NJ];
#pragma unroll
    for (int i = 0; i < MI; i++) a0[i] = read_frag<TM, AL::RED_MAJOR>(As[0] + a_off + i * A_TILE, l32, lk, 0);
#pragma unroll
    for (int j = 0; j < NJ; j++) b0[j] = read_frag<TN, BL::RED_MAJOR>(Bs[0] + b_off + j * B_TILE, l32, lk, 0);
    auto slice = [&](int s, int cur, typename AL::template Regs<TM>& na, typename BL::template Regs<TN>& nb) {
        const int nxt = cur ^ 1;
#pragma unroll
        for (int i = 0; i < MI; i++) a1[i] = read_frag<TM, AL::RED_MAJOR>(As[cur] + a_off + i * A_TILE, l32, lk, 1);
#pragma unroll
        for (int j = 0; j < NJ; j++) b1[j] = read_frag<TN, BL::RED_MAJOR>(Bs[cur] + b_off + j * B_TILE, l32, lk, 1);
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
            for (int i = 0; i < MI; i++)
#pragma unroll
                for (int j = 0; j < NJ; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0[i][e], b0[j][e], acc[i][j], 0, 0, 0);
        AL::template store<TM>(As[nxt], tid, na);
        BL::template store<TN>(Bs[nxt], tid, nb);
        // issue order of the first half: every MFMA is followed by one LDS access
#pragma unroll
        for (int i = 0; i < 4 * MI * NJ; i++) { __builtin_amdgcn_sched_group_barrier(0x008, 1, 0); __builtin_amdgcn_sched_group_barrier(0x300, 2, 0); }
        __syncthreads();
        const int kk0 = k_begin + (s + 1 + AHEAD) * KB;
        al.template load<TM>(sa, kk0, k_end, tid, na);
        bl.template load<TN>(sb, kk0, k_end, tid, nb);
#pragma unroll
        for (int i = 0; i < MI; i++) a0[i] = read_frag<TM, AL::RED_MAJOR>(As[nxt] + a_off + i * A_TILE, l32, lk, 0);
#pragma unroll
        for (int j = 0; j < NJ; j++) b0[j] = read_frag<TN, BL::RED_MAJOR>(Bs[nxt] + b_off + j * B_TILE, l32, lk, 0);
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
            for (int i = 0; i < MI; i++)
#pragma unroll
                for (int j = 0; j < NJ; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1[i][e], b1[j][e], acc[i][j], 0, 0, 0);
        // second half: every MFMA is followed by a global load and an LDS read
#pragma unroll
        for (int i = 0; i < 4 * MI * NJ; i++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
    };
    if constexpr (AHEAD == 1) {
        for (int s = 0; s < nslices; s++) slice(s, s & 1, ra[0], rb[0]);
    } else {
        static_assert(AHEAD % 2 == 0, "a round of slices ends in the LDS buffer it began with");
        int s = 0;
        for (; s + AHEAD <= nslices; s += AHEAD) {
#pragma unroll
            for (int u = 0; u < AHEAD; u++) slice(s + u, u & 1, ra[u], rb[u]);
        }
#pragma unroll
        for (int u = 0; u + 1 < AHEAD; u++) {
            if (s + u >= nslices) break;
            slice(s + u, u & 1, ra[u], rb[u]);
        }
    }

    if (EP::TAIL && d.full_tiles > 0 && !whole)
        ep.store_tail(acc, wm0, wn0, lane, (long)(tile - d.full_tiles) * d.splits + ks, TM, TN);
    else
        ep.store(acc, m0 + wm0, j0 + wn0, lane, ks, d, !whole);
}

// Workgroups of the large tiles that share a compute unit: three, for which 168 registers are left - two where a loader's address work takes more
// (column operands of 256 with a window beyond 32 taps: 16 registers spilled in the loop at three, backward filter 4 x 49 x 138 x 138, 58 of
// 7x7 at stride 3 72 us, 50 at two; 42 x 436 x 57 x 57, 16 of 7x7 479, 358).
template <int TN, class BL> struct LargeTileResident { static constexpr int V = 3; };

template <int TM, int TN, class AL, class BL, class EP, int AHEAD = 1>
__global__ void __launch_bounds__(NT, (LargeTileResident<TN, BL>::V)) igemm_kernel(const AL al, const BL bl, const EP ep, const GemmDims d) {
    igemm_tile<TM, TN, AHEAD>(al, bl, ep, d, blockIdx.x, gridDim.x);
}

// Split reductions of the 64x64 tile without a second kernel. Every workgroup of a tile leaves its sums in the staging area and counts
// itself; the one that counts last adds them up in split order - the sums a second kernel would form - and writes the result. The
// counters are zero between launches: the last workgroup puts its tile's back.
// The eight L2s are not coherent with each other. The sums are therefore stored and loaded at device scope (sc1: through the L2, as
// relaxed atomics at that scope are), and a workgroup counts only when every wavefront has waited for its stores to complete. A
// release and an acquire of everything would write back and invalidate the whole L2, per workgroup: with them a layer of 10 x 192 x 13 x 13,
// 256 filters of 3x3 at stride 2 took 23 us, with a second kernel 18.
typedef unsigned word4 __attribute__((ext_vector_type(4)));
constexpr int kDeviceScope = 16; // cache policy of a buffer access: sc1
// live: the eights of rows of the wavefront's block that begin inside the matrix; the others lie out of the descriptor's range, where nothing moves (a layer of
// few rows would move its tile's 64: 3 rows, 5893 <- 753 backward data in bfloat16 14.6 us with the second kernel, 16.9 so, 15.4 now).
__device__ __forceinline__ bool sum_splits(floatx16& acc, float* staging, const GemmDims& d, int slot_tile, int ks, int tid, int live) {
    __shared__ int last;
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(staging + (long)slot_tile * d.splits * (64 * 64), (unsigned)d.splits * (64 * 64 * 4));
    int place[4];
#pragma unroll
    for (int q = 0; q < 4; q++) place[q] = q < live ? tid * 16 + q * (NT * 16) : OOB;
#pragma unroll
    for (int q = 0; q < 4; q++)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(word4, floatx4{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]}), rs, place[q],
                                               ks * (64 * 64 * 4), kDeviceScope);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) {
        const unsigned before = __hip_atomic_fetch_add(d.counters + slot_tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        last = before == (unsigned)d.splits - 1;
        if (last) __hip_atomic_store(d.counters + slot_tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!last) return false;
    auto load = [&](int q, int s) { return __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(rs, place[q], s * (64 * 64 * 4), kDeviceScope)); };
    floatx4 sum[4];
#pragma unroll
    for (int q = 0; q < 4; q++) sum[q] = load(q, 0);
    // two splits on their way at once: with more, these registers would be the kernel's most
    int s = 1;
    for (; s + 2 <= d.splits; s += 2) {
        floatx4 v[2][4];
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int q = 0; q < 4; q++) v[u][q] = load(q, s + u);
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int q = 0; q < 4; q++) sum[q] += v[u][q];
    }
    for (; s < d.splits; s++)
#pragma unroll
        for (int q = 0; q < 4; q++) sum[q] += load(q, s);
#pragma unroll
    for (int v = 0; v < 16; v++) acc[v] = sum[v / 4][v % 4];
    return true;
}

// The 64x64 tile. A workgroup has one wavefront per SIMD and a few to some tens of slices, and where it is taken most of the chip
// has one or two workgroups a unit: what counts is the latency of every step (1 x 64 x 112 x 112, 64 filters of 3x3, 36 slices on 196
// lone workgroups, clocked inside the kernel). Against igemm_tile's pipeline:
// - AHEAD slices are on their way from memory (four, or one where there are few), so that a slice's values are there when they are
//   written to LDS: operands that another kernel has just written 0.37 -> 0.33 us a slice. (0.21 are the matrix instructions; with
//   one wavefront per SIMD the rest is the issue of some hundred instructions and the barrier.)
// - What the result is combined with (bias, gate, old values) is read before the loop (behind it in the instances that fill the chip), and the epilogue branches on what is
//   uniform only, once per tile: 2.7 -> 0.9 us.
// One call: forward 1 x 64 x 56 x 56, 128 of 3x3 17.7 -> 16.4 us; 49 x 38 x 8 x 8, 224 of 3x3 17.3 -> 14.1; fully connected 79 rows, 1473 -> 108, all
// four passes 30.0 -> 23.6; backward 21 x 70 x 53 x 37, 130 of 3x3 at stride 2 108.9 -> 104.6.
template <int AHEAD, bool SUMS, class AL, class BL, class EP>
__device__ __forceinline__ void igemm_small_tile(const AL& al, const BL& bl, const EP& ep, const GemmDims& d, int block, int blocks) {
    constexpr int T = 64;
    using LA = LdsTile<T, AL::RED_MAJOR>;
    using LB = LdsTile<T, BL::RED_MAJOR>;
    __shared__ __attribute__((aligned(16))) float As[2][LA::SIZE];
    __shared__ __attribute__((aligned(16))) float Bs[2][LB::SIZE];

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const TilePlace at = tile_place(d, block, blocks, T, T);
    const int k_begin = at.k_begin, k_end = at.k_end;

    typename AL::template State<T> sa;
    typename BL::template State<T> sb;
    al.template init<T>(sa, at.m0, tid, d.M, k_begin);
    bl.template init<T>(sb, at.j0, tid, d.N, k_begin);

    typename AL::template Regs<T> fa, ra[AHEAD];
    typename BL::template Regs<T> fb, rb[AHEAD];
    al.template load<T>(sa, k_begin, k_end, tid, fa);
    bl.template load<T>(sb, k_begin, k_end, tid, fb);
#pragma unroll
    for (int u = 0; u < AHEAD; u++) {
        al.template load<T>(sa, k_begin + (u + 1) * KB, k_end, tid, ra[u]);
        bl.template load<T>(sb, k_begin + (u + 1) * KB, k_end, tid, rb[u]);
    }

    const int nslices = (k_end - k_begin + KB - 1) / KB;
    const int l32 = lane & 31, lk = lane >> 5;
    const int wm0 = (wave & 1) * 32, wn0 = (wave >> 1) * 32;
    constexpr bool AUX_FIRST = AHEAD > 1 || SUMS; // (where the registers are there anyway; the others fill the chip, or are over at once)
    float aux[16] = {};
    if constexpr (AUX_FIRST) ep.read_aux(aux, at.m0 + wm0, at.j0 + wn0, lane, d, !at.whole);
    floatx16 acc;
#pragma unroll
    for (int v = 0; v < 16; v++) acc[v] = 0.0f;

    const int a_off = wm0 * LA::ROW_STRIDE, b_off = wn0 * LB::ROW_STRIDE;
    AL::template store<T>(As[0], tid, fa);
    BL::template store<T>(Bs[0], tid, fb);
    __syncthreads();
    floatx4 a0 = read_frag<T, AL::RED_MAJOR>(As[0] + a_off, l32, lk, 0), b0 = read_frag<T, BL::RED_MAJOR>(Bs[0] + b_off, l32, lk, 0);
    // Slice s: write slice s+1 to the other LDS buffer, read the second group's fragments, multiply the first group; barrier; fetch
    // slice s+1+AHEAD into the registers just written, read the first group's fragments of s+1, multiply the second group.
    // All reads of a buffer precede the barrier after which it is overwritten. Fetches past the end of the range read as zero or
    // are never used: buffer loads cannot fault.
    auto slice = [&](int s, int cur, typename AL::template Regs<T>& na, typename BL::template Regs<T>& nb) {
        const int nxt = cur ^ 1;
        const floatx4 a1 = read_frag<T, AL::RED_MAJOR>(As[cur] + a_off, l32, lk, 1), b1 = read_frag<T, BL::RED_MAJOR>(Bs[cur] + b_off, l32, lk, 1);
        AL::template store<T>(As[nxt], tid, na);
        BL::template store<T>(Bs[nxt], tid, nb);
#pragma unroll
        for (int e = 0; e < 4; e++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a0[e], b0[e], acc, 0, 0, 0);
        if constexpr (AHEAD > 1) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x300, 16, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 3, 0);
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++) { __builtin_amdgcn_sched_group_barrier(0x008, 1, 0); __builtin_amdgcn_sched_group_barrier(0x300, 2, 0); }
        }
        __syncthreads();
        const int kk0 = k_begin + (s + 1 + AHEAD) * KB;
        al.template load<T>(sa, kk0, k_end, tid, na);
        bl.template load<T>(sb, kk0, k_end, tid, nb);
        a0 = read_frag<T, AL::RED_MAJOR>(As[nxt] + a_off, l32, lk, 0);
        b0 = read_frag<T, BL::RED_MAJOR>(Bs[nxt] + b_off, l32, lk, 0);
#pragma unroll
        for (int e = 0; e < 4; e++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a1[e], b1[e], acc, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x020, 2, 0);
        }
    };
    if constexpr (AHEAD == 1) {
        for (int s = 0; s < nslices; s++) slice(s, s & 1, ra[0], rb[0]);
    } else {
        static_assert(AHEAD % 2 == 0, "a round of slices ends in the LDS buffer it began with");
        int s = 0;
        for (; s + AHEAD <= nslices; s += AHEAD) {
#pragma unroll
            for (int u = 0; u < AHEAD; u++) slice(s + u, u & 1, ra[u], rb[u]);
        }
#pragma unroll
        for (int u = 0; u + 1 < AHEAD; u++) {
            if (s + u >= nslices) break;
            slice(s + u, u & 1, ra[u], rb[u]);
        }
    }

    if (SUMS && !at.whole && d.counters) {
        const int live = (__builtin_amdgcn_readfirstlane(d.M - at.m0 - wm0) + 7) >> 3;
        if (!sum_splits(acc, ep.partial, d, at.tile - d.full_tiles, at.ks, tid, live)) return;
        ep.read_aux(aux, at.m0 + wm0, at.j0 + wn0, lane, d, false);
        ep.store32(acc, aux, at.m0 + wm0, at.j0 + wn0, lane, 0, d, false);
    } else if (EP::TAIL && d.full_tiles > 0 && !at.whole) {
        const floatx16 tail[1][1] = {{acc}};
        ep.store_tail(tail, wm0, wn0, lane, (long)(at.tile - d.full_tiles) * d.splits + at.ks, T, T);
    } else {
        if constexpr (!AUX_FIRST) ep.read_aux(aux, at.m0 + wm0, at.j0 + wn0, lane, d, !at.whole);
        ep.store32(acc, aux, at.m0 + wm0, at.j0 + wn0, lane, at.ks, d, !at.whole);
    }
}
// Slices ahead: four where the shortest reduction of a workgroup is long enough for them
constexpr int kSmallTileAhead = 4;
// Workgroups up to which they are: four on each unit is what that variant's registers leave room for. (256 units, the target part: callers that plan
// have no context at hand.) 4294 drawn float calls below the line, timed with four and with one: four are 1.2 % faster in the mean, more than 5 % in 473
// and slower in 29; up to 2048 workgroups 1.1 % (68, 12), beyond nothing (59, 38).
constexpr long kSmallTileLone = 1024;
static inline bool small_tile_ahead(const GemmDims& d, long blocks) { return d.kchunk >= (kSmallTileAhead + 2) * KB && blocks <= kSmallTileLone; }
// ... and where the loader's address work does not count for more than the latency (LoadIm2colPix<2>: two divisions per element)
template <class L> struct FetchesAhead { static constexpr bool V = true; };

// SUMS: whether the instance can add up splits itself. That takes half of its registers (with one slice ahead eight wavefronts a SIMD become
// four) and stands in the text that a lone workgroup fetches, so calls without take another.
template <class AL, class BL, class EP, int AHEAD, bool SUMS>
__global__ void __launch_bounds__(NT) igemm64_kernel(const AL al, const BL bl, const EP ep, const GemmDims d) {
    igemm_small_tile<AHEAD, SUMS>(al, bl, ep, d, blockIdx.x, gridDim.x);
}
template <bool SUMS, class AL, class BL, class EP>
static inline void launch_igemm64(unsigned blocks, hipStream_t stream, const AL& al, const BL& bl, const EP& ep, const GemmDims& d) {
    if constexpr (SUMS) {
        if (!d.counters) {
            launch_igemm64<false>(blocks, stream, al, bl, ep, d);
            return;
        }
    }
    if constexpr (FetchesAhead<BL>::V) {
        if (small_tile_ahead(d, blocks)) {
            hipLaunchKernelGGL((igemm64_kernel<AL, BL, EP, kSmallTileAhead, SUMS>), dim3(blocks), dim3(NT), 0, stream, al, bl, ep, d);
            return;
        }
    }
    hipLaunchKernelGGL((igemm64_kernel<AL, BL, EP, 1, SUMS>), dim3(blocks), dim3(NT), 0, stream, al, bl, ep, d);
}

// ---- dense reduction-major operand: element (row, kk) at base[row*ld + kk] -------------------------
// VEC4: rows are 16-byte aligned and the reduction range is a multiple of four, so a thread moves
// 128-bit chunks (thread t: chunk t%4 of rows t/4 + 64*i). Otherwise 32-bit elements
// (thread t: kk t%16 of rows t/16 + 16*i).
template <bool VEC4, class E = float>
struct LoadDenseRed {
    static constexpr bool RED_MAJOR = true;
    static constexpr int ES = ElemBytes<E>::V;
    const E* base;
    long ld;          // elements between rows
    int rows;         // valid rows
    unsigned bytes;   // extent of the matrix in bytes (below 2 GiB)
    template <int T> struct Regs { floatx4 v[T / 64]; float s[VEC4 ? 1 : T / 16]; };
    template <int T> struct State { int vrow[VEC4 ? T / 64 : T / 16]; __amdgpu_buffer_rsrc_t rsrc; };
    template <int T>
    __device__ __forceinline__ void init(State<T>& st, int row0, int tid, int, int) const {
        st.rsrc = make_rsrc(base, bytes);
        if (VEC4) {
#pragma unroll
            for (int i = 0; i < T / 64; i++) {
                const int row = row0 + (tid >> 2) + 64 * i;
                st.vrow[i] = row < rows ? (int)(((long)row * ld + 4 * (tid & 3)) * ES) : OOB;
            }
        } else {
#pragma unroll
            for (int i = 0; i < T / 16; i++) {
                const int row = row0 + (tid >> 4) + 16 * i;
                st.vrow[i] = row < rows ? (int)(((long)row * ld + (tid & 15)) * ES) : OOB;
            }
        }
    }
    template <int T>
    __device__ __forceinline__ void load(State<T>& st, int kk0, int kend, int tid, Regs<T>& r) const {
        const int soff = kk0 * ES;
        // only the last slice of a range can be partial; there a thread past the end reads out of range
        const bool tail = kk0 + KB > kend;
        if (VEC4) {
            const bool dead = tail && (kk0 + 4 * (tid & 3) >= kend);
#pragma unroll
            for (int i = 0; i < T / 64; i++) r.v[i] = buf_load4_e<E>(st.rsrc, dead ? OOB : st.vrow[i], soff);
        } else {
            const bool dead = tail && (kk0 + (tid & 15) >= kend);
#pragma unroll
            for (int i = 0; i < T / 16; i++) r.s[i] = buf_load_e<E>(st.rsrc, dead ? OOB : st.vrow[i], soff);
        }
    }
    template <int T>
    __device__ static __forceinline__ void store(float* lds, int tid, const Regs<T>& r) {
        if (VEC4) {
#pragma unroll
            for (int i = 0; i < T / 64; i++) *(floatx4*)(lds + ((tid >> 2) + 64 * i) * RED_STRIDE + 4 * (tid & 3)) = r.v[i];
        } else {
#pragma unroll
            for (int i = 0; i < T / 16; i++) lds[((tid >> 4) + 16 * i) * RED_STRIDE + (tid & 15)] = r.s[i];
        }
    }
};

// ---- dense row-major operand: element (row, kk) at base[kk*ld_k + row] ------------------------------
// lanes run along rows (coalesced); the reduction index is wave-uniform and lives in the scalar offset
template <class E = float>
struct LoadDenseRow {
    static constexpr bool RED_MAJOR = false;
    static constexpr int ES = ElemBytes<E>::V;
    const E* base;
    long ld_k;        // elements between consecutive kk
    int rows;
    unsigned bytes;   // extent in bytes (below 2 GiB)
    template <int T> struct Regs { float s[T * KB / NT]; };
    template <int T> struct State { int vrow; __amdgpu_buffer_rsrc_t rsrc; };
    template <int T>
    __device__ __forceinline__ void init(State<T>& st, int row0, int tid, int, int) const {
        st.rsrc = make_rsrc(base, bytes);
        const int row = row0 + tid % T;
        st.vrow = row < rows ? row * ES : OOB;
    }
    template <int T>
    __device__ __forceinline__ void load(State<T>& st, int kk0, int kend, int tid, Regs<T>& r) const {
        const int kbase = __builtin_amdgcn_readfirstlane(kk0 + tid / T);
#pragma unroll
        for (int i = 0; i < T * KB / NT; i++) {
            const int kk = kbase + (NT / T) * i;
            const int soff = kk < kend ? (int)((long)kk * ld_k * ES) : 0x7FFFFFF0;
            r.s[i] = buf_load_e<E>(st.rsrc, st.vrow, soff);
        }
    }
    template <int T>
    __device__ static __forceinline__ void store(float* lds, int tid, const Regs<T>& r) {
#pragma unroll
        for (int i = 0; i < T * KB / NT; i++) lds[(tid / T + (NT / T) * i) * T + tid % T] = r.s[i];
    }
};

// the float nearest to v among those exactly representable in bfloat16 (ties to even, NaN stays NaN)
__device__ __forceinline__ float round_to_bf16_value(float v) { return bf16_bits_to_float(float_to_bf16_bits(v)); }

// An operand whose values are rounded to bfloat16 on their way into LDS: the filter operands of layers whose
// activations are stored as bfloat16 (the filter itself stays a float master copy in memory).
template <class L>
struct RoundedToBf16 : L {
    template <int T>
    __device__ static __forceinline__ void store(float* lds, int tid, const typename L::template Regs<T>& r) {
        typename L::template Regs<T> q = r;
        float* f = (float*)&q;
#pragma unroll
        for (int i = 0; i < (int)(sizeof(q) / sizeof(float)); i++) f[i] = round_to_bf16_value(f[i]);
        L::template store<T>(lds, tid, q);
    }
};

// The first of the eight rows from which a lane's registers 4 q .. 4 q + 3 are, past the last row or not; the same for the whole wavefront.
__device__ __forceinline__ bool rows_behind(int m0, int q, int M) { return __builtin_amdgcn_readfirstlane(m0) + 8 * q >= M; }

// An element as it lies in memory, in a float's place, and its value. What a block is combined with is read behind a branch for each eight of its
// rows: with the conversion of a two-byte element in there every branch waits for its loads (7 x 160 x 170 x 170, 32 of 1x1
// gated backward data in bfloat16 45 us, 59 so; 334 of 3290 drawn gated calls more than 5 % slower).
__device__ __forceinline__ float load_raw(const float* p) { return *p; }
__device__ __forceinline__ float load_raw(const bf16_t* p) { return __builtin_bit_cast(float, (unsigned)p->bits); }
template <class E>
__device__ __forceinline__ float raw_value(float raw) {
    if constexpr (sizeof(E) == 2) {
        asm("" : "+v"(raw)); // (the compiler would move the conversion up to the load)
        return bf16_bits_to_float(__builtin_bit_cast(unsigned, raw));
    } else return raw;
}

// A lane's sixteen results of a 32x32 block, `to` at row m0 + 4 lk, rows from M on left out. The test per row is for the blocks at the
// lower edge only, and there for the rows of the eights that begin inside: with a branch on each of a tile's 64 rows, and one each on bias,
// gate and rectifier, a tile's epilogue took 2.7 us per 32x32 block of a wavefront, most of it the fetch of its text. Forward 9 x 448 x 189 x 189, 576 of 1x1 in bfloat16 631 -> 418 us; 29 x 32 x 30 x 30, 289
// of 3x3 30 -> 22; backward 11 x 486 x 71 x 71, 64 of 3x3 246 -> 184; floats at two bfloat16 parts, 122 x 80 x 23 x 23, 528 of 3x3 216 -> 198.
template <class E, class L>
__device__ __forceinline__ void store_rows(E* to, const floatx16& acc, L stride, int m0, int lk, int M) {
    if (m0 + 32 <= M) {
#pragma unroll
        for (int v = 0; v < 16; v++) store_elem(to + (long)(8 * (v / 4) + v % 4) * stride, acc[v]);
    } else {
#pragma unroll
        for (int q = 0; q < 4; q++) {
            if (rows_behind(m0, q, M)) break;
#pragma unroll
            for (int v = 4 * q; v < 4 * q + 4; v++)
                if (m0 + result_row(v, lk) < M) store_elem(to + (long)(8 * q + v % 4) * stride, acc[v]);
        }
    }
}

// ---- dense result: out[m*ld_m + j] = alpha*acc (+ old if accumulate) (+ bias[j]); or a split's
//      partial sums to scratch[ks][m*ld_m + j] ------------------------------------------------------
template <class E = float>
struct StoreDense {
    E* out;
    float* partial;     // used when splits > 1
    const float* bias_j; // optional, indexed by column
    long ld_m;
    long partial_stride; // elements per split
    float alpha;
    int accumulate;
    int relu;      // rectify the result (after the bias)
    const E* gate; // optional, same layout as out: the result is kept where gate > 0 and zero elsewhere
    // The old values or the gate, as they lie (load_raw; a call asks for one of the two at most), of a lane's sixteen results of a 32x32 block; columns past the
    // end, and rows past it in the eight that begins inside, read some element inside. What else is past it is not read (nor stored).
    __device__ __forceinline__ void read_aux(float (&aux)[16], int m0, int j0, int lane, const GemmDims& d, bool to_partial) const {
        if (to_partial || !(accumulate || gate)) return;
        const int j = min(j0 + (lane & 31), d.N - 1), lk = lane >> 5;
        const E* from = accumulate ? out : gate;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            if (rows_behind(m0, q, d.M)) break;
#pragma unroll
            for (int v = 4 * q; v < 4 * q + 4; v++) aux[v] = load_raw(from + (long)min(m0 + result_row(v, lk), d.M - 1) * ld_m + j);
        }
    }
    __device__ __forceinline__ void store32(floatx16 acc, const float (&aux)[16], int m0, int j0, int lane, int ks, const GemmDims& d, bool to_partial) const {
        const int j = j0 + (lane & 31), lk = lane >> 5;
        if (j >= d.N) return;
        const long first = (long)(m0 + 4 * lk) * ld_m + j;
        if (to_partial) {
            store_rows(partial + (long)ks * partial_stride + first, acc, ld_m, m0, lk, d.M);
            return;
        }
        float with[16]; // (converted behind one branch, not one for each row)
#pragma unroll
        for (int v = 0; v < 16; v++) with[v] = aux[v];
        if (sizeof(E) == 2 && (accumulate || gate)) {
#pragma unroll
            for (int v = 0; v < 16; v++) with[v] = raw_value<E>(aux[v]);
        }
#pragma unroll
        for (int v = 0; v < 16; v++) acc[v] = accumulate ? __fmaf_rn(alpha, acc[v], with[v]) : alpha * acc[v];
        if (bias_j) {
            const float bj = bias_j[j];
#pragma unroll
            for (int v = 0; v < 16; v++) acc[v] += bj;
        }
        if (relu) {
#pragma unroll
            for (int v = 0; v < 16; v++) acc[v] = relu_value(acc[v]);
        }
        if (gate) {
#pragma unroll
            for (int v = 0; v < 16; v++) acc[v] = with[v] > 0.0f ? acc[v] : 0.0f;
        }
        store_rows(out + first, acc, ld_m, m0, lk, d.M);
    }
    static constexpr bool TAIL = false;
    template <int MI, int NJ>
    __device__ __forceinline__ void store_tail(const floatx16 (&)[MI][NJ], int, int, int, long, int, int) const {}
    // What a block is combined with is read sixteen elements ahead of its stores: a load issued after a store
    // through the same pointer would have to wait for it (the compiler cannot know that the rows differ), and
    // sixty-four round trips to memory in a row are the kernel's whole time when the output is large (the filter of
    // a fully connected layer, updated in place). Sixteen, not more: the registers they wait in count against the
    // workgroups a compute unit holds.
    template <int MI, int NJ>
    __device__ __forceinline__ void store(const floatx16 (&acc)[MI][NJ], int m0, int j0, int lane, int ks, const GemmDims& d, bool to_partial) const {
#pragma unroll
        for (int jt = 0; jt < NJ; jt++)
#pragma unroll
            for (int it = 0; it < MI; it++) {
                if (rows_behind(m0, 4 * it, d.M)) break;
                float aux[16] = {};
                read_aux(aux, m0 + it * 32, j0 + jt * 32, lane, d, to_partial);
                store32(acc[it][jt], aux, m0 + it * 32, j0 + jt * 32, lane, ks, d, to_partial);
            }
    }
};

} // namespace vdnn
