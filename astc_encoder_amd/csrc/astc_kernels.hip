// astc_kernels.hip -- gfx950 kernels of the ASTC encoder.
//
// encode_plain_kernel: the per-texture launch that replaces MainCS
// (ASTC_Encode.hlsl:553-582).  One lane encodes one block: with ~1-2.5k
// floating-point operations per block and hundreds of thousands of blocks per
// texture, keeping each block in one lane avoids cross-lane reductions and
// replicated serial work (the 16-step power iteration), so every lane issues
// useful VALU work.  A workgroup of 256 lanes takes steps of 256 consecutive
// blocks in row-major block order (plain_grid shares them out): in a step that
// begins at block s, lane t encodes block s + t, so the lanes of a wave read
// adjacent blocks of the texture and write 16-byte blocks to consecutive
// addresses.  By default a lane issues its next block's loads as soon as the
// current block is converted (tiled RGB8 sources: after the store); the 6x6
// encoder holds 144 texel floats per lane and runs two waves per SIMD.  encode_plain_pair_kernel is the
// two-lanes-per-block 6x6 form (astc_plain_tuning.lanes_per_block = 2), and
// encode_plain_packed_kernel the form that holds the fetched bytes instead of
// floats (astc_plain_tuning.packed_texels = 1).
#include <cstring>

#include "astc_internal.h"

namespace astc {

struct PlainArgs {
    FetchArgs f;
    int nblocks;
    uint32_t* dst;
    const DeviceTables* tables;
    // steps of a workgroup, the first `longer` workgroups having one more, or 0 for
    // every gridDim-th step (plain_grid)
    int steps, longer;
};

// The workgroup's share of the image: blocks from `first` on, below `first + count`, in
// steps of `step` blocks that begin `stride` apart.
struct PlainShare { int first, count, stride; };
__device__ __forceinline__ PlainShare plain_share(const PlainArgs& a, int step) {
    const int b = blockIdx.x;
    if (a.steps == 0) return PlainShare{b * step, a.nblocks - b * step, int(gridDim.x) * step};
    const int first = (b * a.steps + min(b, a.longer)) * step;
    return PlainShare{first, min((a.steps + (b < a.longer ? 1 : 0)) * step, a.nblocks - first), step};
}

// LDS tables: lut[0..255] sRGB -> float(linear) * 255, lut[256..511] UNORM8 ->
// float * 255 as the hardware converts it (binary32 c * (1/255), then x255; 126
// values land one ulp off the integer), and the trit groups' code bits for both
// weight quantisations.
// In two parts, one table entry a thread, so that a kernel can have the reads in
// flight before it knows its work.  srgb: whether lut[0..255] is the sRGB table
// (else the UNORM one again).
struct TableEntry {
    float srgb;
    uint32_t trit;
};
__device__ __forceinline__ TableEntry fetch_table_entry(const DeviceTables* t) {
    static_assert(kPlainThreads == 256, "one entry a thread");
    return TableEntry{t->srgb[threadIdx.x], t->trit[threadIdx.x]};
}
__device__ __forceinline__ void stage_table_entry(const TableEntry& e, float* lut, PackTables* pack, bool srgb = true) {
    const int i = threadIdx.x;
    const float unorm = (float(i) * (1.0f / 255.0f)) * 255.0f;
    lut[i] = srgb ? e.srgb : unorm;
    lut[256 + i] = unorm;
    pack->spread[0][i] = trit_group_spread(e.trit, kSplitQ6.bits);
    pack->spread[1][i] = trit_group_spread(e.trit, kSplitQ12.bits);
}
__device__ __forceinline__ void stage_tables(const DeviceTables* t, float* lut, PackTables* pack) {
    stage_table_entry(fetch_table_entry(t), lut, pack);
}

template <int DIM, int CH, int ROWS = ROWS_BOTH, bool AHEAD = false>
__device__ __forceinline__ void load_block_id(const FetchArgs& f, int id, uint32_t p[Layout<DIM, CH>::WORDS]) {
    const int by = block_row_of(f, id);
    load_block<DIM, CH, DIM, ROWS, AHEAD>(f, id - by * f.xblocks, by, p);
}

__host__ __device__ inline int channel_class(int fmt, uint32_t flags, int width, int height, int dim) {
    if (flags & FLAG_NORMAL) return CH_NORMAL;
    return (fmt == FMT_RGB8 && width % dim == 0 && height % dim == 0) ? CH_RGB8 : CH_ALL;
}

// SRGB: 1 / 0 fixes the fetch at compile time, -1 is the batch kernels', which
// stage the work item's colour table in lut[0..255].  Either way the table's
// place is fixed, so that a lookup's address is one instruction.  The channel class CH is the number of active
// channels the encoder works on.  OVERRIDE applies the normal-map override
// (blue = alpha = 255) to the texel words.  Only an encoder that reads blue or
// alpha of a normal map needs it: the principal component encoders take every
// normal map through the two-channel class, which reads red and green only, and
// the mask is zero for every other image, so only the four-channel
// max-accumulation search sets it.
template <int DIM, int SRGB, int CH, bool OVERRIDE = false, int NR = DIM>
__device__ __forceinline__ void unpack_texels(const uint32_t p[NR * Layout<DIM, CH>::WPR], const FetchArgs& f,
                                              const float* lut, float x[NR * DIM][4]) {
    const float* colour = SRGB == 0 ? lut + 256 : lut;
    unpack_block<DIM, CH, NR>(p, OVERRIDE ? f.or_mask : 0u, colour, lut + 256, x);
}

__device__ __forceinline__ void store_block(uint32_t* dst, int id, const Block128& b) {
    reinterpret_cast<uint4*>(dst)[id] = make_uint4(b.w[0], b.w[1], b.w[2], b.w[3]);
}

// Encode blocks of one image with the workgroup's threads: step k, thread t takes
// block first + k * stride + t, for as long as that is below first + count.  `cur`
// holds the packed texels of the thread's first block (the caller issues those
// loads).  With prefetch the next step's texels are loaded as soon as the
// current ones are converted (into the same registers), so the loads are in
// flight while the block is encoded; without, after the block is stored.
// From the store of one block to the end of the next block's conversion (and,
// with prefetch, the issue of the following block's loads) the wave runs at
// issue priority 2 (issue_priority): that phase is a chain of dependent memory
// and LDS operations with little arithmetic, and giving it precedence over the
// other wave's encode keeps the two waves of a SIMD out of phase.
// FLAT: a wave whose blocks all have a flat alpha (flat_alpha) is encoded by
// the three-channel path (same bytes); a separately compiled kernel, which the
// default plain tuning uses for four-channel encodes (the batch kernels do not
// test for flat alpha).
template <int DIM, bool ALPHA, int SRGB, int CH, int METHOD = METHOD_PCA, bool FLAT = false>
__device__ __forceinline__ void encode_loaded(const FetchArgs& f, uint32_t* dst, int first, int count, int stride,
                                              bool prefetch, const float* lut, const PackTables* trit,
                                              uint32_t cur[Layout<DIM, CH>::WORDS]) {
#pragma unroll 1
    for (int o = threadIdx.x;; o += stride) {
        const bool has_next = uint32_t(o) + uint32_t(stride) < uint32_t(count);  // the sum can pass 2^31
        constexpr bool kFlat = FLAT && CH == CH_ALL && METHOD == METHOD_PCA;
        const bool flat = kFlat && __all(flat_alpha<DIM * DIM>(cur, lut + 256));
        float x[DIM * DIM][4];
        unpack_texels<DIM, SRGB, CH, METHOD == METHOD_MAX_ACCUMULATION>(cur, f, lut, x);
        // the packed words are dead once converted: the next block's loads reuse them
        if (has_next && prefetch) load_block_id<DIM, CH, ROWS_BOTH, true>(f, first + o + stride, cur);
        issue_priority(0);
        Block128 b;
        if (kFlat && flat) {
            // keeps the two encoders' code apart: merged, their live values exceed the register file
            __builtin_amdgcn_sched_barrier(0);
            b = encode_block<DIM, ALPHA, CH_RGB8, METHOD>(x, trit, x[0][3]);
        } else {
            b = encode_block<DIM, ALPHA, CH, METHOD>(x, trit);
        }
        issue_priority(2);
        store_block(dst, first + o, b);
        if (!has_next) break;
        if (!prefetch) load_block_id<DIM, CH, ROWS_BOTH, true>(f, first + o + stride, cur);
    }
    issue_priority(0);
}

template <int DIM, bool ALPHA, int SRGB, int CH, int METHOD = METHOD_PCA, bool FLAT = false>
__device__ __forceinline__ void encode_chunk(const FetchArgs& f, uint32_t* dst, int first, int count, int stride,
                                             bool prefetch, const float* lut, const PackTables* trit) {
    if (int(threadIdx.x) >= count) return;
    uint32_t cur[Layout<DIM, CH>::WORDS];
    issue_priority(2);  // the first block's fetch, like every later one (encode_loaded)
    load_block_id<DIM, CH>(f, first + threadIdx.x, cur);
    wait_for_loads();  // the loop's first use is of all of them
    encode_loaded<DIM, ALPHA, SRGB, CH, METHOD, FLAT>(f, dst, first, count, stride, prefetch, lut, trit, cur);
}

// Minimum waves per SIMD the register budget must allow: 4x4 encoders fit in
// 128 VGPRs (the reduced-channel ones use 68-90 and run at five to seven waves);
// 6x6 blocks hold 144 texel floats and run at two.
template <int DIM>
struct PlainWaves { static constexpr int value = DIM == 4 ? 4 : 2; };

template <int DIM, bool ALPHA, bool SRGB, int CH, int METHOD, bool FLAT = false>
__global__ void __launch_bounds__(kPlainThreads)
__attribute__((amdgpu_waves_per_eu(PlainWaves<DIM>::value))) encode_plain_kernel(PlainArgs a, int prefetch) {
    __shared__ float lut[512];
    __shared__ PackTables trit;
    stage_tables(a.tables, lut, &trit);
    __syncthreads();
    const PlainShare s = plain_share(a, kPlainThreads);
    encode_chunk<DIM, ALPHA, SRGB ? 1 : 0, CH, METHOD, FLAT>(a.f, a.dst, s.first, s.count, s.stride, prefetch != 0, lut,
                                                             &trit);
}

// ---------------------------------------------------------------------------
// One lane per block with the texels held as the fetched words (PackedTexels,
// astc_plain_tuning.packed_texels = 1): each pass of the encode converts them
// again through the LDS tables, which trades VALU and LDS instructions for
// registers: a 6x6 four-channel block needs ~170 VGPRs instead of 218 (three
// waves per SIMD instead of two), a 4x4 one ~96 (five instead of four).  The
// words are live through the encode, so the next block is loaded after the
// store (no prefetch).  Principal component encodes only.
// ---------------------------------------------------------------------------
template <int DIM>
struct PackedWaves { static constexpr int value = DIM == 4 ? 5 : 3; };

// ROWS: one of the two row loads each (with both in one kernel it spills more, or has
// fewer table reads in flight: RGBA 6x6 opaque 4096x4096 60 us, so 53; RGB8 6x6
// 1500x1500 8.2, so 7.3).
template <int DIM, bool ALPHA, bool SRGB, int CH, int ROWS>
__global__ void __launch_bounds__(kPlainThreads) __attribute__((amdgpu_waves_per_eu(PackedWaves<DIM>::value)))
encode_plain_packed_kernel(PlainArgs a) {
    __shared__ float lut[512];
    __shared__ PackTables trit;
    stage_tables(a.tables, lut, &trit);
    __syncthreads();
    const PlainShare s = plain_share(a, kPlainThreads);
    if (int(threadIdx.x) >= s.count) return;
    PackedTexels<DIM, CH> x;
    x.colour = SRGB ? lut : lut + 256;
    x.unorm = lut + 256;
    load_block_id<DIM, CH, ROWS>(a.f, s.first + threadIdx.x, x.p);
#pragma unroll 1
    for (int o = threadIdx.x;; o += s.stride) {
        const bool has_next = uint32_t(o) + uint32_t(s.stride) < uint32_t(s.count);
        store_block(a.dst, s.first + o, encode_block<DIM, ALPHA, CH, METHOD_PCA>(x, &trit));
        if (!has_next) break;
        load_block_id<DIM, CH, ROWS>(a.f, s.first + o + s.stride, x.p);
    }
}

// ---------------------------------------------------------------------------
// Two lanes per 6x6 block (encode_block_pair): lanes 2j and 2j+1 load, convert
// and encode rows 0-2 and 3-5 of one block and each store 8 of its 16 bytes.
// A workgroup of 256 lanes covers 128 blocks per step: in step k, lane pair j
// encodes block first + 128 k + j.  Half the texels per lane lowers the
// register budget (a third wave per SIMD) and halves the work of one wave
// iteration (finer balance over the SIMDs); the serial part of the encode runs
// on both lanes.
// ---------------------------------------------------------------------------
template <int CH>
__device__ __forceinline__ void load_half_block(const FetchArgs& f, int id, int half,
                                                uint32_t p[3 * Layout<6, CH>::WPR]) {
    const int by = block_row_of(f, id);
    load_block<6, CH, 3>(f, id - by * f.xblocks, by, p, 3 * half);
}

__device__ __forceinline__ void store_half_block(uint32_t* dst, int id, int half, const Block128& b) {
    reinterpret_cast<uint2*>(dst)[2 * id + half] = half ? make_uint2(b.w[2], b.w[3]) : make_uint2(b.w[0], b.w[1]);
}

template <bool ALPHA, int SRGB, int CH>
__device__ __forceinline__ void encode_chunk_pair(const FetchArgs& f, uint32_t* dst, int first, int count,
                                                  int stride, bool prefetch, const float* lut, const PackTables* trit) {
    const int half = threadIdx.x & 1;
    int o = threadIdx.x >> 1;
    if (o >= count) return;
    uint32_t cur[3 * Layout<6, CH>::WPR];
    load_half_block<CH>(f, first + o, half, cur);
#pragma unroll 1
    for (;; o += stride) {
        const bool has_next = uint32_t(o) + uint32_t(stride) < uint32_t(count);  // the sum can pass 2^31
        float x[18][4];
        unpack_texels<6, SRGB, CH, false, 3>(cur, f, lut, x);
        issue_priority(0);
        if (has_next && prefetch) load_half_block<CH>(f, first + o + stride, half, cur);
        const Block128 b = encode_block_pair<ALPHA, CH>(x, half, trit);
        issue_priority(2);  // as in encode_loaded
        store_half_block(dst, first + o, half, b);
        if (!has_next) break;
        if (!prefetch) load_half_block<CH>(f, first + o + stride, half, cur);
    }
    issue_priority(0);
}

template <bool ALPHA, bool SRGB, int CH>
__global__ void __launch_bounds__(kPlainThreads) __attribute__((amdgpu_waves_per_eu(3)))
encode_plain_pair_kernel(PlainArgs a, int prefetch) {
    __shared__ float lut[512];
    __shared__ PackTables trit;
    stage_tables(a.tables, lut, &trit);
    __syncthreads();
    const PlainShare s = plain_share(a, kPlainThreads / 2);
    encode_chunk_pair<ALPHA, SRGB ? 1 : 0, CH>(a.f, a.dst, s.first, s.count, s.stride, prefetch != 0, lut, &trit);
}

// ---------------------------------------------------------------------------
// Batch kernels: a workgroup takes one work item of the device work list.  An
// item is either a chunk of one image (up to 256 x bpl blocks) or a pack of up to
// kMaxSegs small images (at most one block per thread).  Items are uniform in
// mode (block size x alpha x colour table x channel class), so each workgroup
// runs one encoder specialisation.
//
// The launch has a workgroup for every item and the hardware's dispatcher hands
// them out as others finish.  (A persistent grid that claimed items from one queue
// head paid 13 ns a claim, one workgroup after the other, and a launch to clear
// the head: one 4096x4096 RGB8 texture took 89 us, now 21, and 20 by its plain
// launch; 347 images of all sizes 207, now 111; the 512-texture set, best tuning
// each, 2.05 ms, now 1.66.)
// ---------------------------------------------------------------------------
// The image and block of a pack's lane: lane o of the item's blocks, counted
// through its images in order; level -1 past the last block.  Each lane of a wave
// reads one segment (kMaxSegs at most) and all of them are then compared from
// there, so the lanes of different images meet again before the blocks are
// loaded and the whole wave encodes at once.  (One image after the other, a wave
// ran up to sixteen encodes: 217 images under 4096 texels took 147 us, now 14.)
// Both lane reads stand outside the comparison: inside it the segment's load could
// be moved there too, and the lane that holds the segment need not be active.
struct PackBlock { int level, id; };
__device__ __forceinline__ PackBlock pack_block_of(const BatchArgs& a, const BatchItem& item, int o) {
    static_assert(kMaxSegs <= 64, "one segment a lane");
    const int lane = threadIdx.x & 63;
    BatchSeg sg{0, 0};
    if (lane < item.nseg()) sg = a.segs[item.at + lane];
    PackBlock b{-1, 0};
    for (int s = 0; s < item.nseg(); ++s) {
        const int count = __builtin_amdgcn_readlane(sg.count, s), level = __builtin_amdgcn_readlane(sg.level, s);
        const bool here = o >= 0 && o < count;
        b.level = here ? level : b.level;
        b.id = here ? o : b.id;
        o -= count;
    }
    return b;
}

// LPB = 2: 6x6 items with two lanes per block (encode_block_pair): a chunk
// runs encode_chunk_pair; a pack of small images (at most 256 blocks) takes
// two rounds of 128 lane pairs.
template <int DIM, bool ALPHA, int CH, int LPB = 1>
__device__ __forceinline__ void process_item(const BatchArgs& a, const BatchItem& item, const BatchLevel& chunk,
                                             const float* lut, const PackTables* trit) {
    if (DIM == 6 && LPB == 2) {
        if (item.nseg() == 1) {
            encode_chunk_pair<ALPHA, -1, CH>(chunk.f, chunk.dst, item.first_block, item.count, kPlainThreads / 2,
                                             a.prefetch != 0, lut, trit);
            return;
        }
        const int half = threadIdx.x & 1, pairs = blockDim.x >> 1;
#pragma unroll 1
        for (int r = 0; r < 2; ++r) {
            const PackBlock pb = pack_block_of(a, item, r * pairs + (threadIdx.x >> 1));
            if (pb.level < 0) continue;
            const BatchLevel& L = a.levels[pb.level];
            uint32_t p[3 * Layout<6, CH>::WPR];
            load_half_block<CH>(L.f, pb.id, half, p);
            float x[18][4];
            unpack_texels<6, -1, CH, false, 3>(p, L.f, lut, x);
            store_half_block(L.dst, pb.id, half, encode_block_pair<ALPHA, CH>(x, half, trit));
        }
        return;
    }
    if (item.nseg() == 1) {
        encode_chunk<DIM, ALPHA, -1, CH>(chunk.f, chunk.dst, item.first_block, item.count, kPlainThreads,
                                         a.prefetch != 0, lut, trit);
        return;
    }
    const PackBlock pb = pack_block_of(a, item, threadIdx.x);
    if (pb.level < 0) return;
    const BatchLevel& L = a.levels[pb.level];
    uint4* out = reinterpret_cast<uint4*>(L.dst) + pb.id;
    uint32_t p[Layout<DIM, CH>::WORDS];
    issue_priority(2);  // fetch and conversion, as in encode_loaded
    load_block_id<DIM, CH>(L.f, pb.id, p);
    float x[DIM * DIM][4];
    unpack_texels<DIM, -1, CH>(p, L.f, lut, x);
    issue_priority(0);
    store_block(reinterpret_cast<uint32_t*>(out), 0,
                encode_block<DIM, ALPHA, CH, METHOD_PCA>(x, trit));
}

template <int DIM, bool ALPHA, int LPB>
__device__ __forceinline__ void process_item_ch(const BatchArgs& a, const BatchItem& item, const BatchLevel& chunk,
                                                const float* lut, const PackTables* trit) {
    switch (item.mode() & MODE_CH_MASK) {
    case MODE_CH_NORMAL: process_item<DIM, ALPHA, CH_NORMAL, LPB>(a, item, chunk, lut, trit); break;
    case MODE_CH_RGB8: process_item<DIM, ALPHA, CH_RGB8, LPB>(a, item, chunk, lut, trit); break;
    default: process_item<DIM, ALPHA, CH_ALL, LPB>(a, item, chunk, lut, trit); break;
    }
}

// The list's three runs of items and their kernels, each with its own register
// budget: 6x6 items (two waves per SIMD, or three with LPB = 2, two lanes per
// block), four-channel 4x4 items (four waves) and 4x4 items of the reduced
// channel classes (RGB8 tiles and normal maps, five waves).
template <int RUN, int LPB>
struct BatchWaves { static constexpr int value = RUN == RUN_LIGHT ? 5 : RUN == RUN_4x4 ? 4 : LPB == 2 ? 3 : 2; };

template <int RUN, bool ALPHA>
__device__ __forceinline__ void process_item_4x4(const BatchArgs& a, const BatchItem& item, const BatchLevel& chunk,
                                                 const float* lut, const PackTables* trit) {
    if (RUN == RUN_4x4) {
        process_item<4, ALPHA, CH_ALL>(a, item, chunk, lut, trit);
    } else if ((item.mode() & MODE_CH_MASK) == MODE_CH_NORMAL) {
        process_item<4, ALPHA, CH_NORMAL>(a, item, chunk, lut, trit);
    } else {
        process_item<4, ALPHA, CH_RGB8>(a, item, chunk, lut, trit);
    }
}

// The grid is the run's item count as planned; the count in the list also lets a
// launch over an empty list (a server's first, at its creation) end at once.
template <int RUN, int LPB = 1>
__global__ void __launch_bounds__(kPlainThreads) __attribute__((amdgpu_waves_per_eu(BatchWaves<RUN, LPB>::value)))
encode_batch_kernel(BatchArgs a) {
    __shared__ float lut[512];
    __shared__ PackTables trit;
    const TableEntry entry = fetch_table_entry(a.tables);
    const int it = (RUN == 0 ? 0 : a.scalars[RUN - 1]) + int(blockIdx.x);
    if (it >= a.scalars[RUN]) return;
    const BatchItem item = a.items[it];
    // a chunk's image, read beside the tables: one after the other (tables, image,
    // texels) each workgroup waited 1-2 us longer for its first texels, 142 us
    // against 123 for the 347 images
    BatchLevel chunk;
    if (item.nseg() == 1) chunk = a.levels[item.at];
    stage_table_entry(entry, lut, &trit, (item.mode() & MODE_SRGB) != 0);
    __syncthreads();
    const bool alpha = item.mode() & 1;
    if (RUN == RUN_6x6) {
        if (alpha) process_item_ch<6, true, LPB>(a, item, chunk, lut, &trit);
        else process_item_ch<6, false, LPB>(a, item, chunk, lut, &trit);
    } else {
        if (alpha) process_item_4x4<RUN, true>(a, item, chunk, lut, &trit);
        else process_item_4x4<RUN, false>(a, item, chunk, lut, &trit);
    }
}

// The runs' kernels one after the other.  Beside each other on two streams they
// took as long for the largest batches (512 mip-chained textures, 1.99 ms either
// way) and the fork and join cost 20 us of the smallest.
// one_per_cu: LDS that the kernels do not use, half of a compute unit's 160 KB beside
// their tables' 4, so that two workgroups of a kernel do not fit one (nine 4096x4096
// images, three for each kernel: 388 us against 280).
constexpr size_t kHalfOfLds = 80 << 10;
hipError_t launch_encode_batch(const BatchArgs& a, const BatchLaunch& l, hipStream_t stream) {
    (void)hipGetLastError();  // report this launch's errors only, not an earlier call's
    const dim3 n6(unsigned(l.end[RUN_6x6])), n4(unsigned(l.end[RUN_4x4] - l.end[RUN_6x6])),
        nlight(unsigned(l.end[RUN_LIGHT] - l.end[RUN_4x4])), threads(kPlainThreads);
    const size_t lds = l.one_per_cu ? kHalfOfLds : 0;
    if (n6.x && l.lanes == 2) hipLaunchKernelGGL((encode_batch_kernel<RUN_6x6, 2>), n6, threads, lds, stream, a);
    else if (n6.x) hipLaunchKernelGGL((encode_batch_kernel<RUN_6x6, 1>), n6, threads, lds, stream, a);
    if (n4.x) hipLaunchKernelGGL(encode_batch_kernel<RUN_4x4>, n4, threads, lds, stream, a);
    if (nlight.x) hipLaunchKernelGGL(encode_batch_kernel<RUN_LIGHT>, nlight, threads, lds, stream, a);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Mip generation: levels of a tightly packed 8-bit image.  A side of at least 8
// halves (rounding down) and a shorter side is kept, so every tap is inside the
// source.  2x2 box filter in stored space, (a+b+c+d+2)>>2, or (a+b+1)>>1 along
// the one axis that halves.
//
// One launch makes up to kMipLevels levels: a workgroup takes a 64x64 tile of the
// source, which holds every tap of its 32x32 texels of the first level, 16x16 of
// the second and so on (an axis that is kept has one tile), so each level after
// the first is filtered from the previous one in LDS and the source is read once.
// The first level is 4x1 texels a lane from two 8-texel rows (16-byte loads and
// stores for RGBA8); all four bytes of a texel are filtered at once, two to a
// 32-bit sum.  The chain of a 4096x4096 RGBA8 texture takes two launches of 16.5
// and 4 us (89 MB, 4.4 TB/s; the second works on one 64x64 tile and is a chain of
// latencies); one launch a level and a lane an output byte took ten, 56 us the
// first.
// ---------------------------------------------------------------------------
constexpr int kMipTile = 64, kMipPitch = kMipTile / 2;

struct MipArgs {
    const uint8_t* src;
    int w, h, levels, tiles_x;
    uint8_t* dst[kMipLevels];  // the levels after the source
};

__device__ __forceinline__ uint32_t average4(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    constexpr uint32_t m = 0x00FF00FFu;
    const uint32_t even = (a & m) + (b & m) + (c & m) + (d & m) + 0x00020002u;
    const uint32_t odd = (a >> 8 & m) + (b >> 8 & m) + (c >> 8 & m) + (d >> 8 & m) + 0x00020002u;
    return (even >> 2 & m) | (odd >> 2 & m) << 8;
}
__device__ __forceinline__ uint32_t average2(uint32_t a, uint32_t b) { return (a | b) - ((a ^ b) >> 1 & 0x7F7F7F7Fu); }

template <int BPP>
__device__ __forceinline__ uint32_t mip_load(const uint8_t* p) {
    uint32_t t = 0;
#pragma unroll
    for (int c = 0; c < BPP; ++c) t |= uint32_t(p[c]) << (8 * c);
    return t;
}
template <int BPP>
__device__ __forceinline__ void mip_store(uint8_t* p, uint32_t t) {
#pragma unroll
    for (int c = 0; c < BPP; ++c) p[c] = uint8_t(t >> (8 * c));
}

// N texels at any byte address, as whole words.
template <int BPP, int N>
__device__ __forceinline__ void mip_load_row(const uint8_t* p, uint32_t t[N]) {
    uint32_t w[N * BPP / 4 + 1];
    __builtin_memcpy(w, p, N * BPP);
    w[N * BPP / 4] = 0;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int j = i * BPP;
        t[i] = BPP == 4 ? w[i] : __builtin_amdgcn_alignbyte(w[(j >> 2) + 1], w[j >> 2], j & 3) & ((1u << 8 * (BPP & 3)) - 1u);
    }
}
template <int BPP>
__device__ __forceinline__ void mip_store_row4(uint8_t* p, const uint32_t t[4]) {
    uint32_t w[BPP];
    if (BPP == 4) {
#pragma unroll
        for (int i = 0; i < 4; ++i) w[i & (BPP - 1)] = t[i];
    } else if (BPP == 3) {
        w[0] = t[0] | t[1] << 24;
        w[1] = t[1] >> 8 | t[2] << 16;
        w[BPP - 1] = t[2] >> 16 | t[3] << 8;
    } else {
        w[0] = t[0] | t[1] << 16;
        w[1] = t[2] | t[3] << 16;
    }
    __builtin_memcpy(p, w, 4 * BPP);
}

template <int BPP>
__global__ void __launch_bounds__(256) mip_kernel(MipArgs a) {
    __shared__ uint32_t tile[2][kMipPitch * kMipPitch];
    const int t = threadIdx.x;
    const int ty = int(blockIdx.x) / a.tiles_x, tx = int(blockIdx.x) - ty * a.tiles_x;
    int w = a.w, h = a.h;  // the level being filtered
    bool hx = w >= 8, hy = h >= 8;
    int ow = hx ? w >> 1 : w, oh = hy ? h >> 1 : h;
    int tw = hx ? kMipPitch : 8, th = hy ? kMipPitch : 8;  // the tile's texels in the level made
    if (hx && hy) {
        const int x = 4 * (t & 7), y = t >> 3;
        const int ox = tx * tw + x, oy = ty * th + y;
        if (ox < ow && oy < oh) {
            const uint8_t* r0 = a.src + (int64_t(2 * oy) * w + 2 * ox) * BPP;
            const uint8_t* r1 = r0 + int64_t(w) * BPP;
            uint8_t* out = a.dst[0] + (int64_t(oy) * ow + ox) * BPP;
            uint32_t v[4] = {0, 0, 0, 0};
            if (ox + 4 <= ow) {
                uint32_t s0[8], s1[8];
                mip_load_row<BPP, 8>(r0, s0);
                mip_load_row<BPP, 8>(r1, s1);
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = average4(s0[2 * i], s0[2 * i + 1], s1[2 * i], s1[2 * i + 1]);
                mip_store_row4<BPP>(out, v);
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (ox + i >= ow) break;
                    const int j = 2 * i * BPP;
                    v[i] = average4(mip_load<BPP>(r0 + j), mip_load<BPP>(r0 + j + BPP), mip_load<BPP>(r1 + j),
                                    mip_load<BPP>(r1 + j + BPP));
                    mip_store<BPP>(out + i * BPP, v[i]);
                }
            }
            // texels past the level's edge are not read again
#pragma unroll
            for (int i = 0; i < 4; ++i) tile[0][y * kMipPitch + x + i] = v[i];
        }
    } else {  // one axis is kept: 8 x 32 or 32 x 8 texels, one a lane
        const int x = hx ? t & 31 : t & 7, y = hx ? t >> 5 : t >> 3;
        const int ox = tx * tw + x, oy = ty * th + y;
        if (ox < ow && oy < oh) {
            const uint8_t* s = a.src + (int64_t(hy ? 2 * oy : oy) * w + (hx ? 2 * ox : ox)) * BPP;
            const uint32_t v = average2(mip_load<BPP>(s), mip_load<BPP>(s + (hx ? BPP : int64_t(w) * BPP)));
            mip_store<BPP>(a.dst[0] + (int64_t(oy) * ow + ox) * BPP, v);
            tile[0][y * kMipPitch + x] = v;
        }
    }
    for (int l = 1; l < a.levels; ++l) {
        __syncthreads();
        const uint32_t* in = tile[(l - 1) & 1];
        uint32_t* made = tile[l & 1];
        w = ow;
        h = oh;
        hx = w >= 8;
        hy = h >= 8;
        if (hx) { ow = w >> 1; tw >>= 1; }
        if (hy) { oh = h >> 1; th >>= 1; }
        const int shift = 31 - __builtin_clz(tw);
        for (int i = t; i < tw * th; i += 256) {
            const int x = i & (tw - 1), y = i >> shift;
            const int ox = tx * tw + x, oy = ty * th + y;
            if (ox >= ow || oy >= oh) continue;
            const uint32_t* p = in + (hy ? 2 * y : y) * kMipPitch + (hx ? 2 * x : x);
            const uint32_t v = hx && hy ? average4(p[0], p[1], p[kMipPitch], p[kMipPitch + 1])
                                        : average2(p[0], p[hx ? 1 : kMipPitch]);
            made[y * kMipPitch + x] = v;
            mip_store<BPP>(a.dst[l] + (int64_t(oy) * ow + ox) * BPP, v);
        }
    }
}

// Copies of the server's and the allocation-free entry point's: sources into the
// ring, blocks out of it, work lists from pinned staging.  A kernel of the
// library's own keeps them on the compute queue of the caller's stream, and one
// launch takes up to kMaxCopies of them: one a launch took 4 us each, one after the
// other, a batch of 48 requests about 100 of them.
// A workgroup copies one kCopyChunk piece of one range (found by comparing the
// ranges' first pieces, one in each lane), four 16-byte vectors a lane in flight;
// sources may be at any byte address, a destination that is not 16-byte aligned
// is written byte by byte.  300 MB of 48 requests' sources take 94 us and 65 MB of
// their blocks 27 (6.4 and 4.8 TB/s read and written); a work list of six pieces, read
// from host memory, 13.
constexpr int kCopyChunk = 256 * 16 * 8;
struct CopyList {
    CopyRange range[kMaxCopies];
    int first[kMaxCopies];  // each range's first piece
    int count;
};
static_assert(sizeof(CopyList) <= 4096 && kMaxCopies == 64, "a kernel argument; one range a lane");

__global__ void __launch_bounds__(256) copy_kernel(CopyList a) {
    const int piece = blockIdx.x, lane = threadIdx.x & 63;
    const int r = __popcll(__ballot(lane < a.count && a.first[lane] <= piece)) - 1;
    const int64_t at = int64_t(piece - a.first[r]) * kCopyChunk;
    uint8_t* dst = static_cast<uint8_t*>(a.range[r].dst) + at;
    const uint8_t* src = static_cast<const uint8_t*>(a.range[r].src) + at;
    const int bytes = int(min(int64_t(kCopyChunk), a.range[r].bytes - at));
    const int vectors = (reinterpret_cast<uintptr_t>(dst) & 15u) == 0 ? bytes >> 4 : 0;
    uint4* d = reinterpret_cast<uint4*>(dst);
    for (int i = threadIdx.x; i < vectors; i += 4 * 256) {
        uint4 v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (i + 256 * k < vectors) __builtin_memcpy(&v[k], src + 16 * (i + 256 * k), 16);
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (i + 256 * k < vectors) d[i + 256 * k] = v[k];
    }
    for (int i = 16 * vectors + threadIdx.x; i < bytes; i += 256) dst[i] = src[i];
}

hipError_t launch_copies(const CopyRange* ranges, int count, hipStream_t stream) {
    (void)hipGetLastError();  // report this launch's errors only, not an earlier call's
    for (int next = 0; next < count;) {
        CopyList a;
        int64_t pieces = 0;
        a.count = 0;
        for (; next < count && a.count < kMaxCopies; ++next) {
            if (ranges[next].bytes <= 0) continue;
            a.range[a.count] = ranges[next];
            a.first[a.count++] = int(pieces);
            pieces += (ranges[next].bytes + kCopyChunk - 1) / kCopyChunk;
        }
        if (!pieces) break;
        hipLaunchKernelGGL(copy_kernel, dim3(unsigned(pieces)), dim3(256), 0, stream, a);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// Words that travel as a kernel argument, so that a graph which captures the launch
// holds them itself.  4 KB a launch: a list of 100 images takes two or three.
constexpr int kInlineWords = 1008;
struct InlineWords {
    uint32_t* dst;
    int count;
    uint32_t word[kInlineWords];
};
static_assert(sizeof(InlineWords) <= 4096, "a kernel argument");

__global__ void __launch_bounds__(256) inline_words_kernel(InlineWords a) {
    for (int i = threadIdx.x; i < a.count; i += 256) a.dst[i] = a.word[i];
}

hipError_t launch_inline_words(void* dst, const void* src, size_t bytes, hipStream_t stream) {
    (void)hipGetLastError();  // report this launch's errors only, not an earlier call's
    for (size_t at = 0; at < bytes; at += 4 * kInlineWords) {
        InlineWords a;
        a.dst = reinterpret_cast<uint32_t*>(static_cast<uint8_t*>(dst) + at);
        a.count = int(std::min<size_t>(bytes - at, 4 * kInlineWords) / 4);
        std::memcpy(a.word, static_cast<const uint8_t*>(src) + at, 4 * size_t(a.count));
        hipLaunchKernelGGL(inline_words_kernel, dim3(1), dim3(256), 0, stream, a);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t launch_mips(const uint8_t* src, int w, int h, int bpp, void* const* dst, int levels, hipStream_t stream) {
    (void)hipGetLastError();  // report this launch's errors only, not an earlier call's
    for (int first = 0; first < levels; first += kMipLevels) {
        MipArgs a{};
        a.src = src;
        a.w = w;
        a.h = h;
        a.levels = std::min(levels - first, kMipLevels);
        a.tiles_x = (w + kMipTile - 1) / kMipTile;
        for (int l = 0; l < a.levels; ++l) {
            a.dst[l] = static_cast<uint8_t*>(dst[first + l]);
            w = w >= 8 ? w >> 1 : w;
            h = h >= 8 ? h >> 1 : h;
        }
        src = a.dst[a.levels - 1];
        const int64_t tiles = int64_t(a.tiles_x) * ((a.h + kMipTile - 1) / kMipTile);
        const dim3 grid{unsigned(tiles)}, threads(256);
        if (bpp == 4) hipLaunchKernelGGL(mip_kernel<4>, grid, threads, 0, stream, a);
        else if (bpp == 3) hipLaunchKernelGGL(mip_kernel<3>, grid, threads, 0, stream, a);
        else hipLaunchKernelGGL(mip_kernel<2>, grid, threads, 0, stream, a);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// Workgroups of a plain launch's kernels resident on a compute unit: one-lane 6x6,
// two of four waves; two-lane or packed-texel 6x6, three; 4x4 four, packed five.
static int plain_resident(int dim, int lanes_per_block, bool packed) {
    return dim == 4 ? (packed ? PackedWaves<4>::value : PlainWaves<4>::value)
                    : (lanes_per_block == 2 ? 3 : packed ? PackedWaves<6>::value : PlainWaves<6>::value);
}

// Workgroups of a plain launch, and how its steps (one block a lane) are shared out:
// enough workgroups that none has more than blocks_per_lane steps, and as many as are
// resident at once if there are steps for them, shared evenly.  (Workgroups of the
// same power of two left up to half of the compute units with one workgroup while
// the others ran two.)  Up to four steps are consecutive, which keeps a workgroup's
// texel rows close together; more are taken every grid-th, which keeps all of the
// workgroups' rows together.  RGBA 6x6, us a launch among others, by chunks of the same
// power of two / now, the other order of steps in brackets:
//   3001x2003  15.8 / 12.1 (12.4)    4000x3000 opaque  22.4 / 18.4 (19.2)
//   4096x4096  26.0 / 24.1 (24.1)    4608x4608  39.1 / 25.6 (26.1)
//   8192x4096  42.5 / 39.7 (41.4)    8192x8192  83.9 / 80.7 (80.4)
// Where such chunks all but fill the chip they were as good (4092x4092 22.4 / 22.9,
// opaque 20.0 / 20.4); as many workgroups as have the most steps of all alike are 2-14%
// slower between such sizes (3300x3300 16.4, so 17.7).
constexpr int64_t kConsecutiveSteps = 4;
static unsigned plain_grid(int64_t nblocks, int dim, const PlainTuning& t, int num_cus, PlainArgs* a) {
    const int64_t per_step = kPlainThreads / t.lanes_per_block;
    const int64_t steps = (nblocks + per_step - 1) / per_step;
    const int64_t slots = int64_t(num_cus) * plain_resident(dim, t.lanes_per_block, t.packed_texels != 0);
    const int64_t grid = std::max((steps + t.blocks_per_lane - 1) / t.blocks_per_lane, std::min(steps, slots));
    a->steps = steps <= kConsecutiveSteps * grid ? int(steps / grid) : 0;
    a->longer = int(steps % grid);
    return unsigned(grid);
}

template <int DIM, bool ALPHA, int CH, int METHOD = METHOD_PCA>
static void launch_plain_ch(PlainArgs a, int64_t nblocks, const PlainTuning& t, int num_cus, hipStream_t stream) {
    const bool srgb = a.f.flags & FLAG_SRGB;
    if (DIM == 6 && METHOD == METHOD_PCA && t.lanes_per_block == 2) {
        const dim3 grid(plain_grid(nblocks, DIM, t, num_cus, &a));
        if (srgb)
            hipLaunchKernelGGL((encode_plain_pair_kernel<ALPHA, true, CH>), grid, dim3(kPlainThreads), 0, stream, a, t.prefetch);
        else
            hipLaunchKernelGGL((encode_plain_pair_kernel<ALPHA, false, CH>), grid, dim3(kPlainThreads), 0, stream, a, t.prefetch);
        return;
    }
    const dim3 grid(plain_grid(nblocks, DIM, t, num_cus, &a));
    if (METHOD == METHOD_PCA && t.packed_texels) {
        const dim3 threads(kPlainThreads);
        const bool as_they_are = rows_as_they_are(a.f, CH);
        if (srgb && as_they_are)
            hipLaunchKernelGGL((encode_plain_packed_kernel<DIM, ALPHA, true, CH, ROWS_AS_THEY_ARE>), grid, threads, 0, stream, a);
        else if (srgb)
            hipLaunchKernelGGL((encode_plain_packed_kernel<DIM, ALPHA, true, CH, ROWS_ANY>), grid, threads, 0, stream, a);
        else if (as_they_are)
            hipLaunchKernelGGL((encode_plain_packed_kernel<DIM, ALPHA, false, CH, ROWS_AS_THEY_ARE>), grid, threads, 0, stream, a);
        else
            hipLaunchKernelGGL((encode_plain_packed_kernel<DIM, ALPHA, false, CH, ROWS_ANY>), grid, threads, 0, stream, a);
        return;
    }
    constexpr bool kFlatCapable = CH == CH_ALL && METHOD == METHOD_PCA;
    if (kFlatCapable && t.flat_alpha) {
        if (srgb)
            hipLaunchKernelGGL((encode_plain_kernel<DIM, ALPHA, true, CH, METHOD, kFlatCapable>), grid,
                               dim3(kPlainThreads), 0, stream, a, t.prefetch);
        else
            hipLaunchKernelGGL((encode_plain_kernel<DIM, ALPHA, false, CH, METHOD, kFlatCapable>), grid,
                               dim3(kPlainThreads), 0, stream, a, t.prefetch);
        return;
    }
    if (srgb)
        hipLaunchKernelGGL((encode_plain_kernel<DIM, ALPHA, true, CH, METHOD>), grid, dim3(kPlainThreads), 0, stream, a, t.prefetch);
    else
        hipLaunchKernelGGL((encode_plain_kernel<DIM, ALPHA, false, CH, METHOD>), grid, dim3(kPlainThreads), 0, stream,
                           a, t.prefetch);
}

template <int DIM, bool ALPHA>
static void launch_plain_t(const PlainArgs& a, int64_t nblocks, const PlainTuning& t, int num_cus,
                           hipStream_t stream) {
    if (a.f.flags & FLAG_MAX_ACCUMULATION) {  // optional search: four-channel, one-lane, unpacked encoder only
        PlainTuning one = t;
        one.lanes_per_block = 1;
        one.packed_texels = 0;
        launch_plain_ch<DIM, ALPHA, CH_ALL, METHOD_MAX_ACCUMULATION>(a, nblocks, one, num_cus, stream);
        return;
    }
    switch (channel_class(a.f.fmt, a.f.flags, a.f.width, a.f.height, DIM)) {
    case CH_NORMAL: launch_plain_ch<DIM, ALPHA, CH_NORMAL>(a, nblocks, t, num_cus, stream); break;
    case CH_RGB8: launch_plain_ch<DIM, ALPHA, CH_RGB8>(a, nblocks, t, num_cus, stream); break;
    default: launch_plain_ch<DIM, ALPHA, CH_ALL>(a, nblocks, t, num_cus, stream); break;
    }
}

// Blocks per lane for a plain launch: the fewest (1, 2, 4 or 8) that let every
// workgroup be resident at once, so that no second round of workgroup starts (table
// staging, first fetch) trails the first.
int plain_blocks_per_lane(int64_t nblocks, int dim, int lanes_per_block, int num_cus, bool packed) {
    // 4x4 one-lane encodes: one block per lane, whatever the count; the
    // workgroups that do not fit at first start as others finish, which
    // balances the end of the launch (4096x4096 RGBA8: 21.4 us against 23.0 us
    // at the resident-workgroup rule below)
    if (dim == 4 && !packed) return 1;
    const int64_t slots = int64_t(num_cus) * plain_resident(dim, lanes_per_block, packed);
    const int64_t per_step = kPlainThreads / lanes_per_block;
    int bpl = 1;
    while (bpl < 8 && (nblocks + per_step * bpl - 1) / (per_step * bpl) > slots) bpl *= 2;
    return bpl;
}

// Default plain tuning: one lane per block; the next block's loads issued
// before the current block is encoded except for tiled RGB8 sources (measured
// with the issue priorities: 1-4% faster on RGBA8 and normal maps, 4% slower on
// 4096x4096 RGB8 6x6); the flat-alpha test for four-channel principal component
// encodes (with prefetch: 3% faster on the 4096x4096 noise RGBA8 6x6 texture,
// 5-9% on opaque textures, within 1% slower on 4x4 noise).
PlainTuning default_plain_tuning(const astc_image_desc& d, int64_t nblocks, int num_cus) {
    PlainTuning t;
    t.lanes_per_block = 1;
    const int ch = channel_class(d.src_format, d.flags, d.width, d.height, d.block_dim);
    t.prefetch = ch == CH_RGB8 ? 0 : 1;
    t.flat_alpha = (ch == CH_ALL && !(d.flags & FLAG_MAX_ACCUMULATION)) ? 1 : 0;
    t.packed_texels = 0;
    t.blocks_per_lane = plain_blocks_per_lane(nblocks, d.block_dim, t.lanes_per_block, num_cus);
    return t;
}

hipError_t launch_encode_plain(const DeviceTables* d_tables, const astc_image_desc& d, const ImageGeom& g,
                               const void* src, void* dst, hipStream_t stream, int num_cus, const PlainTuning* tuning) {
    PlainArgs a;
    a.f.src = static_cast<const uint8_t*>(src);
    a.f.width = d.width;
    a.f.height = d.height;
    a.f.row_pitch = d.row_pitch;
    a.f.fmt = d.src_format;
    a.f.flags = d.flags;
    a.f.aligned = ((reinterpret_cast<uintptr_t>(src) & 3u) == 0) && ((d.row_pitch & 3) == 0);
    a.f.or_mask = normal_or_mask(d.flags);
    set_block_row(&a.f, g.xblocks);
    a.nblocks = int(g.nblocks);
    a.dst = static_cast<uint32_t*>(dst);
    a.tables = d_tables;
    PlainTuning t = tuning ? *tuning : default_plain_tuning(d, g.nblocks, num_cus);
    (void)hipGetLastError();  // report this launch's errors only, not an earlier call's
    if (d.block_dim != 6) t.lanes_per_block = 1;
    if (t.blocks_per_lane == 0)
        t.blocks_per_lane = plain_blocks_per_lane(g.nblocks, d.block_dim, t.lanes_per_block, num_cus,
                                                  t.packed_texels && !(d.flags & FLAG_MAX_ACCUMULATION));
    const bool alpha = d.flags & FLAG_ALPHA;
    if (d.block_dim == 4) {
        if (alpha) launch_plain_t<4, true>(a, g.nblocks, t, num_cus, stream);
        else launch_plain_t<4, false>(a, g.nblocks, t, num_cus, stream);
    } else {
        if (alpha) launch_plain_t<6, true>(a, g.nblocks, t, num_cus, stream);
        else launch_plain_t<6, false>(a, g.nblocks, t, num_cus, stream);
    }
    return hipGetLastError();
}

}  // namespace astc
