// Zero-value compression of offloaded tensors. The reference moves every offloaded tensor whole
// (cudaMemcpyAsync in offloadSrcData / prefetchPreviousSrcData, layer.cu:969-987). A rectified tensor is
// about half zeros, and the link to host memory is more than a hundred times slower than HBM, so here the
// tensor crosses the link without its zero elements. The code is lossless: every element comes back with
// the bits it had (an element is dropped only when all its bits are zero).
//
// Packed stream. The tensor is cut into chunks of kZvcChunk elements. The stream starts with a table of one
// 32-bit word per chunk (padded to 16 bytes): the offset of the chunk's record in units of 16 bytes. A record
// is a map of 64 little-endian 64-bit words followed by the kept elements in the order of the map's bits, zero
// filled to a multiple of 16 bytes. The map follows the way a wave reads memory: a lane holds V = 16 / (bytes per
// element) consecutive elements, one 128-bit load, so 64 lanes cover a block of 64 V elements and the block's map
// is V words - bit l of word j of block b (word b V + j of the chunk) is set when element 64 V b + V l + j of the
// chunk is kept. Records follow the table
// without gaps, in the order in which the packing teams claimed their place (an atomic cursor), so the
// stream is as long as its content and its length is known on the device only.
//
// Offload. The packing kernel reads the tensor at HBM speed (zvc_pack_rows_kernel; without a staging buffer
// zvc_pack_kernel stores everything into host memory). Bytes of the stream below `staging_bytes` go to
// a staging buffer in device memory, which the copy engine then moves to the pinned host buffer like any
// other offload; bytes beyond it are stored by the kernel straight into the host buffer through the device's
// mapping of pinned memory. The caller sizes the staging buffer from the length the same tensor had the step
// before (the kernel reports it in a host word); any size is correct. Stores from a kernel to host memory
// hold up the stores of the kernels on the other streams (a convolution forward ran at 0.6 of its rate
// beside a kernel that wrote the whole stream that way), loads from host memory do not: so the way out
// goes through the copy engine, and the way back is a kernel that reads the host buffer and expands as it goes.
#include "backend_internal.h"

#include <algorithm>

namespace vdnn {

static constexpr int kZvcChunk = 4096;      // elements per record
static constexpr int kZvcMapBytes = kZvcChunk / 8;
static constexpr int kZvcGroups = kZvcChunk / 64;          // 64-bit words of the map
static constexpr int kZvcGroupsPerWave = kZvcGroups / 4;   // a team is 256 threads = 4 waves
static constexpr int kZvcPad = 8;           // elements of zero fill behind the last kept element
// A workgroup is kZvcTeams teams of 256 threads, each team on a chunk of its own. The expanding kernel spends
// its life waiting for the link, so what matters there is bytes in flight per resident workgroup; a resident
// workgroup costs the convolutions of the other streams a place on its compute unit, and few large
// workgroups cost few places.
static constexpr int kZvcTeams = 4;
static constexpr int kZvcThreads = 256 * kZvcTeams;
// Workgroups per compute unit of zvc_pack_rows_kernel. One leaves the convolution beside it alone but takes twice as long by itself
// (a pooling layer has no matrix work to hide it behind); beyond two, a step gains nothing (six steps of VGG16 at batch 128 in bfloat16
// 129.1 ms with two, 129.4 with three) and the kernel alone loses (400 MB of bfloat16 167 us with two, 182 with three and four, 186 with six).
static constexpr int kZvcPackPerCu = 2;
static constexpr int kZvcCursors = 64;      // cursors of a block

__host__ __device__ inline size_t zvc_table_bytes(size_t chunks) { return (chunks * 4 + 15) / 16 * 16; }
__host__ __device__ inline size_t zvc_record_bytes_max(int elem_bytes) { return size_t(kZvcMapBytes) + size_t(kZvcChunk) * elem_bytes; }

typedef unsigned v4u __attribute__((ext_vector_type(4)));

// One record as it lies in the stream: the map, then the kept elements.
template <class E>
struct alignas(16) ZvcRecord {
    unsigned long long words[kZvcGroups];
    E kept[kZvcChunk + kZvcPad];
};

// Where an offload's claims stand: the bytes of records claimed so far, and the workgroups that are done. Both words are zero
// between the offloads of a stream: the workgroup that is done last puts them back, so no launch before the packing kernel clears them and
// none behind it reads them (they were two launches of 5 us each, one after the other with the packing kernel, per tensor).
struct ZvcCursor {
    unsigned long long claimed;
    unsigned long long done;
};

// The end of a packing workgroup, by one of its threads, whose claims have all returned.
// total: length of the stream. link: bytes that cross the link for it (the copy engine moves `staging_bytes`
// whatever the stream's length; with keep the block stays on the device and only what did not fit crosses the link).
__device__ __forceinline__ void zvc_finish(ZvcCursor* cursor, unsigned long long table_bytes, unsigned long long staging_bytes, bool keep,
                                           unsigned long long* total_host, unsigned long long* link_bytes) {
    if (atomicAdd(&cursor->done, 1ull) != gridDim.x - 1) return;
    const unsigned long long total = table_bytes + atomicExch(&cursor->claimed, 0ull);
    atomicExch(&cursor->done, 0ull);
    if (total_host) *total_host = total;
    if (keep) atomicAdd(link_bytes, total > staging_bytes ? total - staging_bytes : 0ull);
    else atomicAdd(link_bytes, total > staging_bytes ? total : staging_bytes);
}

struct ZvcReport {
    unsigned long long* total_host;
    unsigned long long* link_bytes;
    int keep;
};

// Packing into a staging buffer in device memory. A wavefront has a chunk to itself: it holds the chunk's 4096 elements in registers (a lane
// a map word as well), a workgroup of four claims the place of its records together (a claim is an atomic on one word for the
// whole device, 3.5 ns apiece), and every row of 64 elements leaves with one masked store of its kept elements, which lie one
// behind the other. No element goes through LDS and a wavefront meets the others of its workgroup twice per chunk.
// Alone it is bound by memory on large tensors and by the chain load, claim, store on those of one or two trips. With its launch, half of the
// elements zero, against a kernel through LDS with one launch before and one behind it: 400 MB of floats 132 -> 122 us, of bfloat16 194 ->
// 167; 6 MB 11 -> 11; 50 MB 24 -> 29 and 31 -> 34 (that kernel had four wavefronts on a chunk). What does not fit the staging buffer goes to
// the host in rows as well, at the link's rate: half of 27 MB 254 -> 259 us. In a training step it runs beside a convolution, and
// what counts is the room it takes there: workgroups of sixteen wavefronts with 35 to 68 KB of LDS waited for a place
// until the convolution's first round was over and ended behind it (64 channels of 112 x 112, batch 128, bfloat16: 715 us beside a
// convolution of 536); this one starts at once, 52 (bfloat16) or 86 registers a wavefront, and takes 254 to 316 us there.
template <class E>
__global__ __launch_bounds__(256) void zvc_pack_rows_kernel(const E* __restrict__ src, size_t count, size_t chunks,
                                                            unsigned char* __restrict__ staging, size_t staging_bytes,
                                                            unsigned char* __restrict__ host, ZvcCursor* __restrict__ cursor, ZvcReport report) {
    constexpr int V = 16 / int(sizeof(E));   // elements per 128-bit load
    constexpr int kBlocks = kZvcChunk / (64 * V);
    __shared__ unsigned wave_bytes[4];
    __shared__ unsigned long long place;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool aligned = (reinterpret_cast<uintptr_t>(src) & 15) == 0;   // (chunks start at multiples of 16 bytes)
    const size_t table_bytes = zvc_table_bytes(chunks);
    // every wavefront of a workgroup makes the same number of trips, so that the barriers meet
    for (size_t first_chunk = size_t(blockIdx.x) * 4; first_chunk < chunks; first_chunk += size_t(gridDim.x) * 4) {
        const size_t chunk = first_chunk + wave;
        const bool live = chunk < chunks;
        const size_t base = chunk * kZvcChunk + size_t(lane) * V;
        v4u q[kBlocks];   // q[b]: this lane's V elements of block b
        if (live && aligned && (chunk + 1) * kZvcChunk <= count) {
#pragma unroll
            for (int b = 0; b < kBlocks; ++b) q[b] = *reinterpret_cast<const v4u*>(src + base + size_t(b) * 64 * V);
        } else {
#pragma unroll
            for (int b = 0; b < kBlocks; ++b) {
                const size_t idx = base + size_t(b) * 64 * V;
                unsigned w[4] = {0, 0, 0, 0};
#pragma unroll
                for (int j = 0; j < V; ++j)
                    if (live && idx + j < count) w[j * int(sizeof(E)) / 4] |= unsigned(src[idx + j]) << (j * int(sizeof(E)) % 4 * 8);
#pragma unroll
                for (int j = 0; j < 4; ++j) q[b][j] = w[j];
            }
        }
        auto element = [&](int b, int j) -> E { return E(q[b][j * int(sizeof(E)) / 4] >> (j * int(sizeof(E)) % 4 * 8)); };
        unsigned word_lo = 0, word_hi = 0;   // word `lane` of the map
        unsigned kept = 0;
#pragma unroll
        for (int b = 0; b < kBlocks; ++b)
#pragma unroll
            for (int j = 0; j < V; ++j) {
                const unsigned long long m = __ballot(element(b, j) != 0);
                // lane b V + j = m (two wait states after the comparison that wrote the mask)
                asm("s_nop 1\n\tv_writelane_b32 %0, %2, %4\n\tv_writelane_b32 %1, %3, %4" : "+v"(word_lo), "+v"(word_hi) : "s"(unsigned(m)), "s"(unsigned(m >> 32)), "n"(b * V + j));
                kept += __popcll(m);
            }
        const unsigned long long word = (unsigned long long)word_hi << 32 | word_lo;
        // (the stores below compare again: the masks of 64 rows kept from here would not fit the scalar registers)
#pragma unroll
        for (int b = 0; b < kBlocks; ++b) asm volatile("" : "+v"(q[b]));
        const unsigned bytes = live ? kZvcMapBytes + (kept * unsigned(sizeof(E)) + 15u) / 16u * 16u : 0u;
        if (lane == 0) wave_bytes[wave] = bytes;
        __syncthreads();
        if (threadIdx.x == 0) place = atomicAdd(&cursor->claimed, (unsigned long long)(wave_bytes[0] + wave_bytes[1] + wave_bytes[2] + wave_bytes[3]));
        unsigned ahead = 0;   // (read between the barriers: behind the second one the next trip's sizes may come in)
#pragma unroll
        for (int w = 0; w < 3; ++w) ahead += w < wave ? wave_bytes[w] : 0u;
        __syncthreads();
        size_t at = table_bytes + place + ahead;
        if (!live) continue;   // (in the last trip only)
        at = (size_t)__builtin_amdgcn_readfirstlane(unsigned(at)) | (size_t)__builtin_amdgcn_readfirstlane(unsigned(at >> 32)) << 32;
        if (lane == 0) {
            const size_t entry = chunk * 4;
            *reinterpret_cast<unsigned*>((entry < staging_bytes ? staging : host) + entry) = unsigned(at / 16);
        }
        const unsigned fill = (bytes - kZvcMapBytes) / unsigned(sizeof(E)) - kept;   // elements of zero fill
        if (at + bytes <= staging_bytes) {
            unsigned char* p = staging + at;
            reinterpret_cast<unsigned long long*>(p)[lane] = word;
            p += kZvcMapBytes;
#pragma unroll
            for (int b = 0; b < kBlocks; ++b)
#pragma unroll
                for (int j = 0; j < V; ++j) {
                    const E e = element(b, j);
                    const unsigned long long m = __ballot(e != 0);
                    const unsigned to = __builtin_amdgcn_mbcnt_hi(unsigned(m >> 32), __builtin_amdgcn_mbcnt_lo(unsigned(m), 0u));
                    if (e != 0) reinterpret_cast<E*>(p)[to] = e;
                    p += size_t(__popcll(m)) * sizeof(E);
                }
            if (unsigned(lane) < fill) reinterpret_cast<E*>(p)[lane] = E(0);
        } else {
            // the record ends behind the staging buffer: each piece goes where its place lies
            auto target = [&](size_t o) { return (o < staging_bytes ? staging : host) + o; };
            *reinterpret_cast<unsigned long long*>(target(at + size_t(lane) * 8)) = word;
            size_t o = at + kZvcMapBytes;
#pragma unroll
            for (int b = 0; b < kBlocks; ++b)
#pragma unroll
                for (int j = 0; j < V; ++j) {
                    const E e = element(b, j);
                    const unsigned long long m = __ballot(e != 0);
                    const unsigned to = __builtin_amdgcn_mbcnt_hi(unsigned(m >> 32), __builtin_amdgcn_mbcnt_lo(unsigned(m), 0u));
                    if (e != 0) *reinterpret_cast<E*>(target(o + to * sizeof(E))) = e;
                    o += size_t(__popcll(m)) * sizeof(E);
                }
            if (unsigned(lane) < fill) *reinterpret_cast<E*>(target(o + lane * sizeof(E))) = E(0);
            // a wavefront has one record on its way to host memory at a time: stores that pile up ahead of the link
            // hold up the stores of the kernels on the other streams behind them
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
    }
    if (threadIdx.x == 0) zvc_finish(cursor, table_bytes, staging_bytes, report.keep != 0, report.total_host, report.link_bytes);
}

// Packing straight into host memory. The records go through LDS, so that what crosses the link are whole 16-byte pieces side by
// side, and few workgroups share the link. E is the element as raw bits (uint32_t for float, uint16_t for bfloat16).
template <class E>
__global__ __launch_bounds__(kZvcThreads) void zvc_pack_kernel(const E* __restrict__ src, size_t count, size_t chunks,
                                                               unsigned char* __restrict__ host, ZvcCursor* __restrict__ cursor, ZvcReport report) {
    __shared__ ZvcRecord<E> rec[kZvcTeams];
    __shared__ unsigned wave_total[kZvcTeams][4];
    __shared__ unsigned long long place[kZvcTeams];
    const int team = threadIdx.x >> 8, tid = threadIdx.x & 255;
    const int lane = tid & 63, wave = tid >> 6;
    const unsigned long long below = (1ull << lane) - 1ull;
    const size_t stride = size_t(gridDim.x) * kZvcTeams, table_bytes = zvc_table_bytes(chunks);
    const bool aligned = (reinterpret_cast<uintptr_t>(src) & 15) == 0;   // (chunks start at multiples of 16 bytes)
    // every team makes the same number of trips, so that the barriers meet; a team past the end idles through them
    for (size_t first_chunk = size_t(blockIdx.x) * kZvcTeams; first_chunk < chunks; first_chunk += stride) {
        const size_t chunk = first_chunk + team;
        const bool live = chunk < chunks;
        // this wave's 16 words are kZvcGroupsPerWave / V blocks; v[b V + j] is this lane's element j of block b
        constexpr int V = 16 / int(sizeof(E));
        const size_t base = chunk * kZvcChunk + size_t(wave) * kZvcGroupsPerWave * 64 + size_t(lane) * V;
        E v[kZvcGroupsPerWave];
        unsigned long long m[kZvcGroupsPerWave];
        unsigned kept = 0;
#pragma unroll
        for (int b = 0; b < kZvcGroupsPerWave / V; ++b) {
            const size_t idx = base + size_t(b) * 64 * V;
            if (live && aligned && idx + V <= count) {
                const v4u q = *reinterpret_cast<const v4u*>(src + idx);
                const E* e = reinterpret_cast<const E*>(&q);
#pragma unroll
                for (int j = 0; j < V; ++j) v[b * V + j] = e[j];
            } else {
#pragma unroll
                for (int j = 0; j < V; ++j) v[b * V + j] = live && idx + j < count ? src[idx + j] : E(0);
            }
        }
#pragma unroll
        for (int i = 0; i < kZvcGroupsPerWave; ++i) {
            m[i] = __ballot(v[i] != 0);
            kept += __popcll(m[i]);
            if (lane == i) rec[team].words[wave * kZvcGroupsPerWave + i] = m[i];
        }
        if (lane == 0) wave_total[team][wave] = kept;
        __syncthreads();
        unsigned pos = 0, total = 0;
#pragma unroll
        for (int w = 0; w < 4; ++w) { const unsigned t = wave_total[team][w]; pos += w < wave ? t : 0u; total += t; }
        const unsigned units = kZvcMapBytes / 16 + (total * unsigned(sizeof(E)) + 15u) / 16u;   // 16-byte units of the record
        if (threadIdx.x == 0) {
            // one claim for the workgroup's records: every claim is an atomic on the same word
            unsigned bytes[kZvcTeams], all = 0;
#pragma unroll
            for (int t = 0; t < kZvcTeams; ++t) {
                unsigned n = 0;
#pragma unroll
                for (int w = 0; w < 4; ++w) n += wave_total[t][w];
                bytes[t] = first_chunk + t < chunks ? kZvcMapBytes + (n * unsigned(sizeof(E)) + 15u) / 16u * 16u : 0u;
                all += bytes[t];
            }
            unsigned long long at = table_bytes + atomicAdd(&cursor->claimed, (unsigned long long)all);
#pragma unroll
            for (int t = 0; t < kZvcTeams; ++t) { place[t] = at; at += bytes[t]; }
        }
#pragma unroll
        for (int i = 0; i < kZvcGroupsPerWave; ++i) {
            if (v[i] != 0) rec[team].kept[pos + __popcll(m[i] & below)] = v[i];
            pos += __popcll(m[i]);
        }
        if (tid < kZvcPad) rec[team].kept[total + tid] = E(0);
        __syncthreads();
        if (live) {
            const size_t at = place[team];
            if (tid == 0) *reinterpret_cast<unsigned*>(host + chunk * 4) = unsigned(at / 16);
            const v4u* in = reinterpret_cast<const v4u*>(&rec[team]);
            for (unsigned u = tid; u < units; u += 256) *reinterpret_cast<v4u*>(host + at + size_t(u) * 16) = in[u];
            // a team has one record on its way to host memory at a time: stores that pile up ahead of the link
            // hold up the stores of the kernels on the other streams behind them
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) zvc_finish(cursor, table_bytes, 0, report.keep != 0, report.total_host, report.link_bytes);
}

// The stream's bytes below `device_bytes` are read from `device` (a staging block that was kept), the rest from `host`.
template <class E>
__global__ __launch_bounds__(kZvcThreads) void zvc_unpack_kernel(const unsigned char* __restrict__ device, size_t device_bytes,
                                                                 const unsigned char* __restrict__ host, E* __restrict__ dst,
                                                                 size_t count, size_t chunks) {
    __shared__ unsigned long long words[kZvcTeams][kZvcGroups];
    __shared__ unsigned first[kZvcTeams][kZvcGroups + 1];   // kept elements ahead of each group, and their number overall
    __shared__ unsigned long long place[kZvcTeams];
    __shared__ __attribute__((aligned(16))) E kept[kZvcTeams][kZvcChunk + kZvcPad];
    const int team = threadIdx.x >> 8, tid = threadIdx.x & 255;
    const int lane = tid & 63, wave = tid >> 6;
    const unsigned long long below = (1ull << lane) - 1ull;
    const size_t stride = size_t(gridDim.x) * kZvcTeams;
    const bool aligned = (reinterpret_cast<uintptr_t>(dst) & 15) == 0;
    for (size_t first_chunk = size_t(blockIdx.x) * kZvcTeams; first_chunk < chunks; first_chunk += stride) {
        const size_t chunk = first_chunk + team;
        const bool live = chunk < chunks;
        if (wave == 0) {
            const size_t entry = chunk * 4;
            const size_t at = live ? size_t(*reinterpret_cast<const unsigned*>((entry < device_bytes ? device : host) + entry)) * 16 : 0;
            const size_t mine = at + size_t(lane) * 8;
            const unsigned long long w = live ? *reinterpret_cast<const unsigned long long*>((mine < device_bytes ? device : host) + mine) : 0ull;
            words[team][lane] = w;
            unsigned sum = __popcll(w);
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const unsigned up = __shfl_up(sum, d, 64);
                sum += lane >= d ? up : 0u;
            }
            first[team][lane + 1] = sum;
            if (lane == 0) { first[team][0] = 0; place[team] = at; }
        }
        __syncthreads();
        const unsigned total = first[team][kZvcGroups];
        const unsigned n16 = (total * unsigned(sizeof(E)) + 15u) / 16u;
        const size_t values = place[team] + kZvcMapBytes;
        v4u* st = reinterpret_cast<v4u*>(kept[team]);
        for (unsigned u = tid; u < n16; u += 256) {
            const size_t o = values + size_t(u) * 16;
            st[u] = *reinterpret_cast<const v4u*>((o < device_bytes ? device : host) + o);
        }
        __syncthreads();
        constexpr int V = 16 / int(sizeof(E));
        const size_t base = chunk * kZvcChunk + size_t(wave) * kZvcGroupsPerWave * 64 + size_t(lane) * V;
#pragma unroll
        for (int b = 0; b < kZvcGroupsPerWave / V; ++b) {
            v4u q;
            E* e = reinterpret_cast<E*>(&q);
#pragma unroll
            for (int j = 0; j < V; ++j) {
                const int g = wave * kZvcGroupsPerWave + b * V + j;
                const unsigned long long w = words[team][g];
                e[j] = (w >> lane) & 1ull ? kept[team][first[team][g] + __popcll(w & below)] : E(0);
            }
            const size_t idx = base + size_t(b) * 64 * V;
            if (live && aligned && idx + V <= count) {
                *reinterpret_cast<v4u*>(dst + idx) = q;
            } else {
#pragma unroll
                for (int j = 0; j < V; ++j) if (live && idx + j < count) dst[idx + j] = e[j];
            }
        }
        __syncthreads();
    }
}

static int zvc_ensure_counters(vdnn_ctx* ctx) {
    if (!ctx->zvc_counters) ctx->zvc_counters = (unsigned long long*)zeroed_device_memory(sizeof(unsigned long long));
    if (!ctx->zvc_counters) { set_error("no device memory for the offload's counter"); return VDNN_EDEVICE; }
    return VDNN_OK;
}

// The cursor of a packing kernel on `stream`. A stream's kernels run one behind the other and each leaves its cursor at zero, so one per
// stream does for any number of offloads in flight; two that ran on one cursor at once would write into each other's records and past
// the stream's end. A captured call, whose graph may run beside anything, has a cursor of its own.
static ZvcCursor* zvc_cursor(vdnn_ctx* ctx, hipStream_t stream) {
    auto& owners = ctx->zvc_cursor_streams;
    const bool captured = stream_is_captured(stream);
    size_t i = captured ? owners.size() : size_t(std::find(owners.begin(), owners.end(), stream) - owners.begin());
    if (i == owners.size()) {
        if (i == ctx->zvc_cursor_blocks.size() * kZvcCursors) {
            void* block = zeroed_device_memory(sizeof(ZvcCursor) * kZvcCursors);
            if (!block) return nullptr;
            ctx->zvc_cursor_blocks.push_back(block);
        }
        owners.push_back(captured ? nullptr : stream);
    }
    return (ZvcCursor*)ctx->zvc_cursor_blocks[i / kZvcCursors] + i % kZvcCursors;
}

static int zvc_offload(vdnn_ctx* ctx, void* dst_host, void* staging_dev, size_t staging_bytes, const void* src_dev, size_t count,
                       int elem_bytes, unsigned long long* total_host, vdnn_stream_t pack_stream, vdnn_stream_t copy_stream, vdnn_event_t packed,
                       bool keep_on_device) {
    VDNN_REQUIRE(ctx, "null context");
    VDNN_REQUIRE(elem_bytes == 2 || elem_bytes == 4, "elements are two or four bytes");
    if (ctx->plan_only) return VDNN_OK;
    hipStream_t cs = copy_stream ? (hipStream_t)copy_stream : ctx->d2h;
    // without an event to order the two streams the kernels run on the copy stream
    hipStream_t ps = !packed ? cs : pack_stream ? (hipStream_t)pack_stream : ctx->pack;
    if (count == 0) {
        if (packed) { VDNN_HIP(hipEventRecord((hipEvent_t)packed, ps)); VDNN_HIP(hipStreamWaitEvent(cs, (hipEvent_t)packed, 0)); }
        return VDNN_OK;
    }
    VDNN_REQUIRE(dst_host && src_dev, "null pointer");
    VDNN_REQUIRE(((uintptr_t)dst_host & 15) == 0 && ((uintptr_t)src_dev & (elem_bytes - 1)) == 0, "misaligned buffer");
    VDNN_REQUIRE(staging_bytes == 0 || (staging_dev && ((uintptr_t)staging_dev & 15) == 0 && staging_bytes % 16 == 0),
                 "staging buffer: 16-byte aligned, a multiple of 16 bytes");
    VDNN_REQUIRE(staging_bytes <= vdnn_zvc_buffer_bytes(count, elem_bytes), "staging buffer longer than the longest stream");
    if (int rc = zvc_ensure_counters(ctx)) return rc;
    const size_t chunks = (count + kZvcChunk - 1) / kZvcChunk;
    ZvcCursor* cursor = zvc_cursor(ctx, ps);
    if (!cursor) { set_error("no device memory for the offload's cursor"); return VDNN_EDEVICE; }
    const ZvcReport report{total_host, ctx->zvc_counters, keep_on_device};
    auto grid = [&](size_t per_workgroup, size_t cap) { return int(std::min((chunks + per_workgroup - 1) / per_workgroup, cap)); };
    {
        ProfScope prof(ctx, ps, staging_bytes ? "offload_zvc_pack" : "offload_zvc", 0.0, (double)(count * elem_bytes));
        auto pack = [&](auto element) {
            using E = decltype(element);
            if (staging_bytes)
                zvc_pack_rows_kernel<E><<<grid(4, size_t(ctx->num_cu) * kZvcPackPerCu), 256, 0, ps>>>((const E*)src_dev, count, chunks, (unsigned char*)staging_dev,
                                                                                          staging_bytes, (unsigned char*)dst_host, cursor, report);
            else   // bound by the link and by how many stores it may have in flight
                zvc_pack_kernel<E><<<grid(kZvcTeams, size_t(ctx->num_cu) / 8), kZvcThreads, 0, ps>>>((const E*)src_dev, count, chunks, (unsigned char*)dst_host,
                                                                                               cursor, report);
        };
        if (elem_bytes == 4) pack(uint32_t(0));
        else pack(uint16_t(0));
        VDNN_HIP(hipGetLastError());
    }
    if (packed) {
        VDNN_HIP(hipEventRecord((hipEvent_t)packed, ps));
        VDNN_HIP(hipStreamWaitEvent(cs, (hipEvent_t)packed, 0));
    }
    if (staging_bytes && !keep_on_device) {
        ProfScope prof(ctx, cs, "offload_zvc_copy", 0.0, (double)(count * elem_bytes));
        VDNN_HIP(hipMemcpyAsync(dst_host, staging_dev, staging_bytes, hipMemcpyDeviceToHost, cs));
    }
    ctx->zvc_raw_bytes += (unsigned long long)count * elem_bytes;
    return VDNN_OK;
}

} // namespace vdnn

using namespace vdnn;

size_t vdnn_zvc_buffer_bytes(size_t count, int elem_bytes) {
    if (elem_bytes != 2 && elem_bytes != 4) return 0;
    const size_t chunks = (count + kZvcChunk - 1) / kZvcChunk;
    return zvc_table_bytes(chunks) + chunks * zvc_record_bytes_max(elem_bytes);
}

int vdnn_zvc_offload_async(vdnn_ctx* ctx, void* dst_host, const void* src_dev, size_t count, int elem_bytes, vdnn_stream_t stream) {
    return zvc_offload(ctx, dst_host, nullptr, 0, src_dev, count, elem_bytes, nullptr, nullptr, stream, nullptr, false);
}

int vdnn_zvc_offload_staged_async(vdnn_ctx* ctx, void* dst_host, void* staging_dev, size_t staging_bytes, const void* src_dev, size_t count,
                                  int elem_bytes, unsigned long long* total_host, vdnn_stream_t pack_stream, vdnn_stream_t copy_stream,
                                  vdnn_event_t packed, int keep_on_device) {
    return zvc_offload(ctx, dst_host, staging_dev, staging_bytes, src_dev, count, elem_bytes, total_host, pack_stream, copy_stream, packed,
                       keep_on_device != 0);
}

static int zvc_prefetch(vdnn_ctx* ctx, void* dst_dev, const void* staging_dev, size_t staging_bytes, const void* src_host, size_t count,
                        int elem_bytes, vdnn_stream_t stream) {
    VDNN_REQUIRE(ctx, "null context");
    VDNN_REQUIRE(elem_bytes == 2 || elem_bytes == 4, "elements are two or four bytes");
    if (ctx->plan_only || count == 0) return VDNN_OK;
    VDNN_REQUIRE(dst_dev && src_host, "null pointer");
    VDNN_REQUIRE(((uintptr_t)src_host & 15) == 0 && ((uintptr_t)dst_dev & (elem_bytes - 1)) == 0, "misaligned buffer");
    VDNN_REQUIRE(staging_bytes == 0 || (staging_dev && ((uintptr_t)staging_dev & 15) == 0 && staging_bytes % 16 == 0),
                 "staging buffer: 16-byte aligned, a multiple of 16 bytes");
    hipStream_t s = stream ? (hipStream_t)stream : ctx->h2d;
    const size_t chunks = (count + kZvcChunk - 1) / kZvcChunk;
    // from host memory: enough records in flight to keep the link busy across their round trips, on an eighth of
    // the compute units; from a block on the device: the whole device, briefly
    const size_t need = (chunks + kZvcTeams - 1) / kZvcTeams;
    const size_t cap = staging_bytes ? size_t(ctx->num_cu) * 2 : size_t(ctx->num_cu) / 8;
    const int grid = int(need < cap ? need : cap);
    ProfScope prof(ctx, s, staging_bytes ? "prefetch_zvc_device" : "prefetch_zvc", 0.0, (double)(count * elem_bytes));
    if (elem_bytes == 4)
        zvc_unpack_kernel<uint32_t><<<grid, kZvcThreads, 0, s>>>((const unsigned char*)staging_dev, staging_bytes, (const unsigned char*)src_host,
                                                                  (uint32_t*)dst_dev, count, chunks);
    else
        zvc_unpack_kernel<uint16_t><<<grid, kZvcThreads, 0, s>>>((const unsigned char*)staging_dev, staging_bytes, (const unsigned char*)src_host,
                                                                  (uint16_t*)dst_dev, count, chunks);
    VDNN_HIP(hipGetLastError());
    return VDNN_OK;
}

int vdnn_zvc_prefetch_async(vdnn_ctx* ctx, void* dst_dev, const void* src_host, size_t count, int elem_bytes, vdnn_stream_t stream) {
    return zvc_prefetch(ctx, dst_dev, nullptr, 0, src_host, count, elem_bytes, stream);
}

int vdnn_zvc_prefetch_staged_async(vdnn_ctx* ctx, void* dst_dev, const void* staging_dev, size_t staging_bytes, const void* src_host,
                                   size_t count, int elem_bytes, vdnn_stream_t stream) {
    return zvc_prefetch(ctx, dst_dev, staging_dev, staging_bytes, src_host, count, elem_bytes, stream);
}

int vdnn_zvc_traffic(vdnn_ctx* ctx, unsigned long long* tensor_bytes, unsigned long long* link_bytes) {
    VDNN_REQUIRE(ctx && tensor_bytes && link_bytes, "null argument");
    *tensor_bytes = ctx->zvc_raw_bytes;
    *link_bytes = 0;
    if (ctx->plan_only || !ctx->zvc_counters) return VDNN_OK;
    VDNN_HIP(hipDeviceSynchronize());
    VDNN_HIP(hipMemcpy(link_bytes, ctx->zvc_counters, sizeof(unsigned long long), hipMemcpyDeviceToHost));
    return VDNN_OK;
}
