// astc_batch.cpp -- batched encoding: work-list planning, hipGraph
// capture and the autotuner (include/astc_mi355x.h, astc_batch_*).
#include <algorithm>
#include <array>
#include <cstdint>
#include <cstring>
#include <new>
#include <stdexcept>
#include <vector>

#include "astc_internal.h"

using namespace astc;

struct astc_batch {
    astc_ctx* ctx = nullptr;
    int device = 0;
    int num_cus = 0;
    std::vector<BatchLevel> levels;  // host copies
    std::vector<int> modes;          // kNoMode for images encoded by plain launches
    // images with the max-accumulation search: one plain launch each, captured in
    // the same graph after the batch kernels (the work list has no such mode)
    struct PlainImage {
        astc_image_desc desc;
        ImageGeom geom;
        const void* src;
        void* dst;
    };
    std::vector<PlainImage> plain;
    int64_t blocks = 0, texels = 0;
    astc_tuning tuning{4, 2, 1, 1, 1};
    // device work list
    BatchLevel* d_levels = nullptr;
    BatchSeg* d_segs = nullptr;
    BatchItem* d_items = nullptr;
    int* d_scalars = nullptr;  // end of each run of items
    int nitems = 0;
    // the batch kernels' launch; a batch with plain images replays it and theirs
    // as one graph, any other launches its kernels (three at most) itself: 9 us
    // less than the graph's replay of one kernel
    BatchArgs args{};
    BatchLaunch launch{};
    bool built = false;
    hipStream_t capture_stream = nullptr;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
};

namespace astc {

// Mode code of an image that is not in the work list (no code the planner visits).
constexpr int kNoMode = -1;

// Image index bits of a planner sort key.
constexpr int kKeyIndexBits = 27;

// Sort n unsigned keys (distinct, so the result is one order) in place with a
// least-significant-digit radix sort over 8-bit digits; tmp holds n keys.  A
// digit that is the same in every key is skipped.
void radix_sort_keys(uint64_t* keys, uint64_t* tmp, int n) {
    uint64_t* src = keys;
    uint64_t* dst = tmp;
    for (int shift = 0; shift < 64; shift += 8) {
        int count[257] = {0};
        for (int i = 0; i < n; ++i) ++count[((src[i] >> shift) & 0xFF) + 1];
        if (n == 0 || count[((src[0] >> shift) & 0xFF) + 1] == n) continue;
        for (int d = 0; d < 256; ++d) count[d + 1] += count[d];
        for (int i = 0; i < n; ++i) dst[count[(src[i] >> shift) & 0xFF]++] = src[i];
        std::swap(src, dst);
    }
    if (src != keys) std::memcpy(keys, src, size_t(n) * sizeof(uint64_t));
}

// The run a mode's items belong to.
int run_of(int mode) {
    if (mode & 2) return RUN_6x6;
    return (mode & MODE_CH_MASK) == MODE_CH_ALL ? RUN_4x4 : RUN_LIGHT;
}

// Position of each mode code in the planner's visiting order: most expensive
// first (block size, then active channels, alpha, sRGB), ties by code.
int mode_position(int mode) {
    int pos = 0;
    for (int m = 0; m < MODE_COUNT; ++m)
        pos += mode_cost_rank(m) > mode_cost_rank(mode) || (mode_cost_rank(m) == mode_cost_rank(mode) && m < mode);
    return pos;
}

// Blocks per lane of each run's chunks: the fewest, up to the tuning's, that let
// the run's workgroups all be resident at once (the kernels' waves per SIMD are
// workgroups per compute unit), as for a plain launch.  Chunks of the tuning's size
// leave most of the chip idle on small batches: mixed textures of 8 M texels took
// 43 us at 4 blocks per lane and 74 at 8, 25 so; 64 M texels 118, 105 so; the
// 512-texture set (1.7 G) is the same.  (Cutting smaller chunks only towards the
// end of a run was no faster, and 10-30% slower on one large 6x6 texture.)
RunSteps run_steps(const BatchLevel* levels, const int* modes, int nlevels, const astc_tuning& t, int num_cus) {
    int64_t blocks[RUN_COUNT] = {};
    for (int i = 0; i < nlevels; ++i)
        if (modes[i] >= 0 && modes[i] < MODE_COUNT) blocks[run_of(modes[i])] += levels[i].nblocks;
    const int waves[RUN_COUNT] = {batch_lanes(t) == 2 ? 3 : 2, 4, 5};  // BatchWaves
    RunSteps s;
    for (int r = 0; r < RUN_COUNT; ++r) {
        const int64_t step = int64_t(num_cus) * (batch_one_per_cu(t) ? 1 : waves[r]) * kPlainThreads;
        s.steps[r] = int(std::max<int64_t>(1, std::min<int64_t>(t.blocks_per_lane, (blocks[r] + step - 1) / step)));
    }
    return s;
}

// Work list for a tuning.  Modes are ordered by cost (6x6 RGBA first) so the
// longest items start first; within a mode, images by size (large first, then
// by index), large ones split into chunks of 256 x the run's steps blocks,
// images under 256 blocks packed up to kMaxSegs per item (one block per
// thread).  That order holds the three runs one after the other: every 6x6 mode
// costs more than every 4x4 one, and of those the four-channel ones more than
// the RGB8 and normal-map ones.  Codes with both class bits set are not
// modes (no image has them); images with a mode outside 0..MODE_COUNT-1 are
// left out.  Writes into the caller's arrays (keys: 2 nlevels of room) and
// allocates nothing; returns false if segs or items would exceed their capacity
// or nlevels is 2^27 or more.
bool plan_work_into(const BatchLevel* levels, const int* modes, int nlevels, const RunSteps& steps, uint64_t* keys,
                    BatchSeg* segs, int seg_cap, BatchItem* items, int item_cap, int* nseg, int end[RUN_COUNT]) {
    if (nlevels < 0 || nlevels >= (1 << kKeyIndexBits)) return false;
    int pos[MODE_COUNT];
    for (int m = 0; m < MODE_COUNT; ++m) pos[m] = mode_position(m);
    // visiting order: mode position, then blocks (large first), then index, as
    // one unsigned key per image (position | complement of the block count |
    // index), sorted by a least-significant-digit radix sort
    int n = 0;
    for (int i = 0; i < nlevels; ++i)
        if (modes[i] >= 0 && modes[i] < MODE_COUNT)
            keys[n++] = uint64_t(pos[modes[i]]) << (kKeyIndexBits + 31) |
                        uint64_t(0x7FFFFFFF - std::max(0, levels[i].nblocks)) << kKeyIndexBits | uint64_t(i);
    radix_sort_keys(keys, keys + n, n);
    const uint64_t index_mask = (uint64_t(1) << kKeyIndexBits) - 1;
    int ns = 0, ni = 0;
    for (int r = 0; r < RUN_COUNT; ++r) end[r] = 0;
    int pack_begin = 0, pack_nseg = 0, pack_blocks = 0, cur_mode = -1;
    auto flush = [&]() -> bool {
        if (pack_nseg) {
            if (ni >= item_cap) return false;
            if (pack_nseg == 1) {  // an image by itself is a chunk
                items[ni++] = BatchItem{cur_mode | 1 << 8, segs[pack_begin].level, 0, pack_blocks};
                ns = pack_begin;
            } else {
                items[ni++] = BatchItem{cur_mode | pack_nseg << 8, pack_begin, 0, pack_blocks};
            }
            end[run_of(cur_mode)] = ni;
        }
        pack_begin = ns;
        pack_nseg = pack_blocks = 0;
        return true;
    };
    for (int k = 0; k < n; ++k) {
        const int li = int(keys[k] & index_mask), mode = modes[li];
        if (mode != cur_mode) {
            if (!flush()) return false;
            cur_mode = mode;
        }
        const int nb = levels[li].nblocks;
        if (nb >= kPlainThreads) {
            const int chunk = kPlainThreads * steps.steps[run_of(mode)];
            for (int64_t first = 0; first < nb; first += chunk) {  // past 2^31 for the largest images
                if (ni >= item_cap) return false;
                items[ni++] = BatchItem{mode | 1 << 8, li, int(first), int(std::min<int64_t>(chunk, nb - first))};
            }
            end[run_of(mode)] = ni;
            continue;
        }
        if (pack_blocks + nb > kPlainThreads || pack_nseg == kMaxSegs) {
            if (!flush()) return false;  // packs stay contiguous in the segment array
        }
        if (ns >= seg_cap) return false;
        segs[ns++] = BatchSeg{li, nb};
        ++pack_nseg;
        pack_blocks += nb;
    }
    if (!flush()) return false;
    for (int r = 1; r < RUN_COUNT; ++r) end[r] = std::max(end[r], end[r - 1]);  // empty runs
    *nseg = ns;
    return true;
}

void plan_work(const std::vector<BatchLevel>& levels, const std::vector<int>& modes, const RunSteps& steps,
               std::vector<BatchSeg>* segs, std::vector<BatchItem>* items, int end[RUN_COUNT]) {
    // every image yields at most max(1, ceil(nblocks / chunk)) items, and at most
    // one segment
    int64_t cap = 1;
    for (size_t i = 0; i < levels.size(); ++i)
        if (modes[i] >= 0 && modes[i] < MODE_COUNT)
            cap += levels[i].nblocks / (int64_t(kPlainThreads) * steps.steps[run_of(modes[i])]) + 1;
    std::vector<uint64_t> keys(2 * levels.size());
    segs->resize(levels.size() + 1);
    items->resize(size_t(cap));
    int ns = 0;
    if (!plan_work_into(levels.data(), modes.data(), (int)levels.size(), steps, keys.data(), segs->data(),
                        (int)segs->size(), items->data(), (int)cap, &ns, end))
        throw std::length_error("work list: too many images");
    segs->resize(size_t(ns));
    items->resize(size_t(end[RUN_COUNT - 1]));
}

}  // namespace astc

namespace {

void free_worklist(astc_batch* b) {
    if (b->exec) (void)hipGraphExecDestroy(b->exec);
    if (b->graph) (void)hipGraphDestroy(b->graph);
    b->exec = nullptr;
    b->graph = nullptr;
    b->built = false;
    for (void* p : {(void*)b->d_segs, (void*)b->d_items})
        if (p) (void)hipFree(p);
    b->d_segs = nullptr;
    b->d_items = nullptr;
}

// Queue the batch on `stream`: the batch kernels, then the plain images' launches.
hipError_t queue(astc_batch* b, hipStream_t stream) {
    hipError_t e = launch_encode_batch(b->args, b->launch, stream);
    for (const astc_batch::PlainImage& p : b->plain) {
        if (e != hipSuccess) break;
        e = launch_encode_plain(b->ctx->d_tables, p.desc, p.geom, p.src, p.dst, stream, b->num_cus);
    }
    return e;
}

int build(astc_batch* b) {
    free_worklist(b);
    std::vector<BatchSeg> segs;
    std::vector<BatchItem> items;
    BatchLaunch& l = b->launch;
    const RunSteps steps =
        run_steps(b->levels.data(), b->modes.data(), (int)b->levels.size(), b->tuning, b->num_cus);
    plan_work(b->levels, b->modes, steps, &segs, &items, l.end);
    hipError_t e;
    if ((e = hipMalloc(&b->d_segs, std::max<size_t>(1, segs.size()) * sizeof(BatchSeg))) != hipSuccess)
        return hip_fail(e, "hipMalloc(segs)");
    if ((e = hipMalloc(&b->d_items, std::max<size_t>(1, items.size()) * sizeof(BatchItem))) != hipSuccess)
        return hip_fail(e, "hipMalloc(items)");
    if (!segs.empty() &&
        (e = hipMemcpy(b->d_segs, segs.data(), segs.size() * sizeof(BatchSeg), hipMemcpyHostToDevice)) != hipSuccess)
        return hip_fail(e, "hipMemcpy(segs)");
    if (!items.empty() && (e = hipMemcpy(b->d_items, items.data(), items.size() * sizeof(BatchItem),
                                         hipMemcpyHostToDevice)) != hipSuccess)
        return hip_fail(e, "hipMemcpy(items)");
    b->nitems = (int)items.size();
    if ((e = hipMemcpy(b->d_scalars, l.end, sizeof(l.end), hipMemcpyHostToDevice)) != hipSuccess)
        return hip_fail(e, "hipMemcpy(scalars)");

    BatchArgs& a = b->args;
    a.levels = b->d_levels;
    a.segs = b->d_segs;
    a.items = b->d_items;
    a.scalars = b->d_scalars;
    a.tables = b->ctx->d_tables;
    a.prefetch = b->tuning.prefetch;
    l.lanes = batch_lanes(b->tuning);
    l.one_per_cu = batch_one_per_cu(b->tuning);
    if (b->plain.empty()) {
        b->built = true;
        return ASTC_OK;
    }
    if ((e = hipStreamBeginCapture(b->capture_stream, hipStreamCaptureModeThreadLocal)) != hipSuccess)
        return hip_fail(e, "hipStreamBeginCapture");
    const hipError_t le = queue(b, b->capture_stream);
    e = hipStreamEndCapture(b->capture_stream, &b->graph);
    if (le != hipSuccess) return hip_fail(le, "batch launch capture");
    if (e != hipSuccess) return hip_fail(e, "hipStreamEndCapture");
    if ((e = hipGraphInstantiate(&b->exec, b->graph, nullptr, nullptr, 0)) != hipSuccess)
        return hip_fail(e, "hipGraphInstantiate");
    b->built = true;
    return ASTC_OK;
}

bool valid_tuning(const astc_tuning* t) { return valid_batch_tuning(*t); }

}  // namespace

extern "C" {

int astc_batch_create(astc_ctx* ctx, const astc_image_desc* descs, const void* const* srcs, void* const* dsts,
                      int count, astc_batch** out) {
    return guarded([&]() -> int {
        if (!out) return fail(ASTC_ERR_INVALID_ARG, "out is NULL");
        *out = nullptr;
        if (!ctx || !descs || !srcs || !dsts || count < 1) return fail(ASTC_ERR_INVALID_ARG, "empty or NULL batch");
        hipError_t e = hipSetDevice(ctx->device);
        if (e != hipSuccess) return hip_fail(e, "hipSetDevice");
        astc_batch* b = new (std::nothrow) astc_batch();
        if (!b) return fail(ASTC_ERR_NO_MEMORY, "host allocation failed");
        b->ctx = ctx;
        b->device = ctx->device;
        b->levels.resize(count);
        b->modes.resize(count);
        for (int i = 0; i < count; ++i) {
            ImageGeom g;
            int rc = check_desc(&descs[i], &g);
            if (rc != ASTC_OK || !srcs[i] || !dsts[i] || (reinterpret_cast<uintptr_t>(dsts[i]) & 15u)) {
                delete b;
                if (rc == ASTC_OK) rc = fail(ASTC_ERR_INVALID_ARG, "image " + std::to_string(i) + ": bad src/dst pointer");
                else set_error("image " + std::to_string(i) + ": " + astc_last_error());
                return rc;
            }
            BatchLevel& L = b->levels[i];
            L.f.src = static_cast<const uint8_t*>(srcs[i]);
            L.f.width = descs[i].width;
            L.f.height = descs[i].height;
            L.f.row_pitch = descs[i].row_pitch;
            L.f.fmt = descs[i].src_format;
            L.f.flags = descs[i].flags;
            L.f.aligned = ((reinterpret_cast<uintptr_t>(srcs[i]) & 3u) == 0) && ((descs[i].row_pitch & 3) == 0);
            L.f.or_mask = normal_or_mask(descs[i].flags);
            set_block_row(&L.f, g.xblocks);
            L.dst = static_cast<uint32_t*>(dsts[i]);
            L.nblocks = (int)g.nblocks;
            b->modes[i] = mode_of(descs[i].block_dim, descs[i].src_format, descs[i].flags, descs[i].width, descs[i].height);
            if (descs[i].flags & ASTC_FLAG_MAX_ACCUMULATION) {
                b->modes[i] = kNoMode;
                b->plain.push_back(astc_batch::PlainImage{descs[i], g, srcs[i], dsts[i]});
            }
            b->blocks += g.nblocks;
            b->texels += (int64_t)descs[i].width * descs[i].height;
        }
        int rc = ASTC_OK;
        if ((e = hipDeviceGetAttribute(&b->num_cus, hipDeviceAttributeMultiprocessorCount, ctx->device)) != hipSuccess)
            rc = hip_fail(e, "hipDeviceGetAttribute");
        else if ((e = hipMalloc(&b->d_levels, count * sizeof(BatchLevel))) != hipSuccess)
            rc = hip_fail(e, "hipMalloc(levels)");
        else if ((e = hipMemcpy(b->d_levels, b->levels.data(), count * sizeof(BatchLevel), hipMemcpyHostToDevice)) !=
                 hipSuccess)
            rc = hip_fail(e, "hipMemcpy(levels)");
        else if ((e = hipMalloc(&b->d_scalars, 4 * sizeof(int))) != hipSuccess)
            rc = hip_fail(e, "hipMalloc(scalars)");
        else if (!b->plain.empty() &&
                 (e = hipStreamCreateWithFlags(&b->capture_stream, hipStreamNonBlocking)) != hipSuccess)
            rc = hip_fail(e, "stream creation");
        else
            rc = build(b);
        if (rc != ASTC_OK) {
            astc_batch_destroy(b);
            return rc;
        }
        *out = b;
        return ASTC_OK;
    });
}

int astc_batch_set_tuning(astc_batch* b, const astc_tuning* t) {
    return guarded([&]() -> int {
        if (!b || !t) return fail(ASTC_ERR_INVALID_ARG, "NULL argument");
        if (!valid_tuning(t)) return fail(ASTC_ERR_INVALID_ARG, "tuning out of range");
        hipError_t e = hipSetDevice(b->device);
        if (e != hipSuccess) return hip_fail(e, "hipSetDevice");
        b->tuning = *t;
        return build(b);
    });
}

int astc_batch_get_tuning(const astc_batch* b, astc_tuning* t) {
    if (!b || !t) return fail(ASTC_ERR_INVALID_ARG, "NULL argument");
    *t = b->tuning;
    return ASTC_OK;
}

int astc_batch_launch(astc_batch* b, void* stream) {
    if (!b || !b->built) return fail(ASTC_ERR_INVALID_ARG, "batch is NULL or not built");
    hipError_t e = hipSetDevice(b->device);
    if (e != hipSuccess) return hip_fail(e, "hipSetDevice");
    hipStream_t s = static_cast<hipStream_t>(stream);
    // a graph's launch leaves nothing in a stream's capture: the kernels are queued
    // there one by one
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (b->exec && s && (e = hipStreamIsCapturing(s, &capture)) != hipSuccess) return hip_fail(e, "hipStreamIsCapturing");
    if (!b->exec || capture != hipStreamCaptureStatusNone) {
        if ((e = queue(b, s)) != hipSuccess) return hip_fail(e, "batch launch");
    } else if ((e = hipGraphLaunch(b->exec, s)) != hipSuccess) {
        return hip_fail(e, "hipGraphLaunch");
    }
    return ASTC_OK;
}

int astc_batch_autotune(astc_batch* b, void* stream, int reps, astc_tuning* best_out) {
    return guarded([&]() -> int {
        if (!b) return fail(ASTC_ERR_INVALID_ARG, "batch is NULL");
        if (reps < 1) reps = 1;
        hipStream_t s = static_cast<hipStream_t>(stream);
        hipEvent_t t0, t1;
        hipError_t e;
        if ((e = hipEventCreate(&t0)) != hipSuccess) return hip_fail(e, "hipEventCreate");
        if ((e = hipEventCreate(&t1)) != hipSuccess) {
            (void)hipEventDestroy(t0);
            return hip_fail(e, "hipEventCreate");
        }
        astc_tuning best = b->tuning;
        float best_ms = 1e30f;
        std::vector<astc_tuning> candidates;
        // workgroups_per_cu and split_modes only limit what a batch takes of the chip:
        // the batch's own stay.  Of tunings that launch the same (the same steps in
        // every run; lanes count where there are 6x6 blocks, prefetch where a run has
        // several steps) the first is timed.
        bool any6 = false;
        for (int m : b->modes) any6 = any6 || (m >= 0 && run_of(m) == RUN_6x6);
        std::vector<std::array<int, RUN_COUNT + 2>> plans;
        for (int lanes : {1, 2})
            for (int bpl : {1, 2, 4, 8})
                for (int pf : {0, 1}) {
                    const astc_tuning t{bpl, b->tuning.workgroups_per_cu, pf, b->tuning.split_modes, lanes};
                    const RunSteps steps = run_steps(b->levels.data(), b->modes.data(), (int)b->levels.size(), t, b->num_cus);
                    std::array<int, RUN_COUNT + 2> plan{};
                    std::copy(steps.steps, steps.steps + RUN_COUNT, plan.begin());
                    plan[RUN_COUNT] = any6 ? lanes : 1;
                    plan[RUN_COUNT + 1] = *std::max_element(steps.steps, steps.steps + RUN_COUNT) > 1 ? pf : 0;
                    if (std::find(plans.begin(), plans.end(), plan) != plans.end()) continue;
                    plans.push_back(plan);
                    candidates.push_back(t);
                }
        int rc = ASTC_OK;
        for (const astc_tuning& t : candidates) {
            if ((rc = astc_batch_set_tuning(b, &t)) != ASTC_OK) break;
            if ((rc = astc_batch_launch(b, stream)) != ASTC_OK) break;  // warm-up
            if ((e = hipEventRecord(t0, s)) != hipSuccess) {
                rc = hip_fail(e, "hipEventRecord");
                break;
            }
            for (int r = 0; r < reps && rc == ASTC_OK; ++r) rc = astc_batch_launch(b, stream);
            if (rc != ASTC_OK) break;
            if ((e = hipEventRecord(t1, s)) != hipSuccess || (e = hipEventSynchronize(t1)) != hipSuccess) {
                rc = hip_fail(e, "timing event");
                break;
            }
            float ms = 0.f;
            (void)hipEventElapsedTime(&ms, t0, t1);
            if (ms < best_ms) {
                best_ms = ms;
                best = t;
            }
        }
        (void)hipEventDestroy(t0);
        (void)hipEventDestroy(t1);
        if (rc != ASTC_OK) return rc;
        if ((rc = astc_batch_set_tuning(b, &best)) != ASTC_OK) return rc;
        if (best_out) *best_out = best;
        return ASTC_OK;
    });
}

int astc_batch_info(const astc_batch* b, int64_t* blocks, int64_t* texels, int32_t* items) {
    if (!b) return fail(ASTC_ERR_INVALID_ARG, "batch is NULL");
    if (blocks) *blocks = b->blocks;
    if (texels) *texels = b->texels;
    if (items) *items = b->nitems;
    return ASTC_OK;
}

int astc_batch_destroy(astc_batch* b) {
    if (!b) return ASTC_OK;
    (void)hipSetDevice(b->device);
    free_worklist(b);
    if (b->d_levels) (void)hipFree(b->d_levels);
    if (b->d_scalars) (void)hipFree(b->d_scalars);
    if (b->capture_stream) (void)hipStreamDestroy(b->capture_stream);
    delete b;
    return ASTC_OK;
}

}  // extern "C"
