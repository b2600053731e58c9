// astc_noalloc.hip -- astc_encode_batch_noalloc: the batched encode
// with its work list in a fixed device array, for callers that cannot allocate
// device memory (code under graph capture, tight serving loops, harnesses that
// forbid hipMalloc).
//
// The batch kernels read a work list (image descriptions, packs' images, items):
// device memory beyond the inputs and outputs.
// astc_batch_create allocates it per batch; this entry point instead keeps it
// in `scratch`, a file-scope device array of kNoAllocScratchBytes that every
// GPU the library runs on holds until the process ends.  Its address on each
// device is taken once, in astc_ctx_create (noalloc_setup, with the device
// current), and only that address is used on the host.  The plan is written
// into pinned host staging that the context allocated at creation, copied into
// scratch on the caller's stream by the library's copy kernel (which reads the
// staging through its device address), and the staging is reused only after
// that copy has completed (an event).
//
// A call under stream capture is replayed after other calls have refilled the
// staging, with launches made for its own list.  Its list is therefore planned in
// host memory of its own and written to scratch from kernel arguments, which the
// graph keeps: a replay encodes the captured call's images.
//
// Every call on one GPU uses that GPU's scratch: calls on one stream follow
// each other, but calls that overlap on the device (different streams, or other
// threads' streams) race on it.
#include <cstdlib>

#include "astc_internal.h"

namespace astc {

static __device__ __align__(256) uint8_t scratch[kNoAllocScratchBytes];

int noalloc_setup(astc_ctx* ctx) {
    hipError_t e = hipGetSymbolAddress(&ctx->noalloc.scratch, HIP_SYMBOL(scratch));
    if (e != hipSuccess) {
        ctx->noalloc.scratch = nullptr;
        return hip_fail(e, "hipGetSymbolAddress(scratch)");
    }
    if ((e = hipHostMalloc(reinterpret_cast<void**>(&ctx->noalloc.staging), sizeof(NoAllocPlan), 0)) != hipSuccess) {
        ctx->noalloc.staging = nullptr;
        return hip_fail(e, "hipHostMalloc(no-alloc staging)");
    }
    if ((e = hipHostGetDevicePointer(const_cast<void**>(&ctx->noalloc.staging_dev), ctx->noalloc.staging, 0)) !=
        hipSuccess) {
        ctx->noalloc.staging_dev = nullptr;
        return hip_fail(e, "hipHostGetDevicePointer(no-alloc staging)");
    }
    if ((e = hipEventCreateWithFlags(&ctx->noalloc.staged, hipEventDisableTiming)) != hipSuccess) {
        ctx->noalloc.staged = nullptr;
        return hip_fail(e, "hipEventCreate(no-alloc staging)");
    }
    ctx->noalloc.captured = static_cast<NoAllocPlan*>(std::malloc(sizeof(NoAllocPlan)));
    if (!ctx->noalloc.captured) return fail(ASTC_ERR_NO_MEMORY, "host allocation failed");
    return ASTC_OK;
}

void noalloc_teardown(astc_ctx* ctx) {
    if (ctx->noalloc.staged) {
        (void)hipEventSynchronize(ctx->noalloc.staged);
        (void)hipEventDestroy(ctx->noalloc.staged);
    }
    if (ctx->noalloc.staging) (void)hipHostFree(ctx->noalloc.staging);
    std::free(ctx->noalloc.captured);
    ctx->noalloc.captured = nullptr;
    ctx->noalloc.staged = nullptr;
    ctx->noalloc.staging = nullptr;
    ctx->noalloc.staging_dev = nullptr;
    ctx->noalloc.scratch = nullptr;
}

}  // namespace astc

using namespace astc;

extern "C" int astc_encode_batch_noalloc(astc_ctx* ctx, const astc_image_desc* descs, const void* const* srcs,
                                         void* const* dsts, int count, const astc_tuning* tuning, void* stream) {
    return guarded([&]() -> int {
        if (!ctx || !descs || !srcs || !dsts || count < 1) return fail(ASTC_ERR_INVALID_ARG, "empty or NULL batch");
        if (!ctx->noalloc.scratch || !ctx->noalloc.staging || !ctx->noalloc.staging_dev || !ctx->noalloc.staged ||
            !ctx->noalloc.captured)
            return fail(ASTC_ERR_INVALID_ARG, "context has no no-alloc scratch");
        if (count > kNoAllocMaxImages) return fail(ASTC_ERR_INVALID_ARG, "more images than the no-alloc maximum (8192)");
        const astc_tuning t = tuning ? *tuning : astc_tuning{4, 2, 1, 0, 1};
        const int bpl = t.blocks_per_lane;
        if (!valid_batch_tuning(t) || t.split_modes != 0)
            return fail(ASTC_ERR_INVALID_ARG, "tuning out of range (the no-alloc form takes split_modes 0 only)");
        hipError_t e = hipSetDevice(ctx->device);
        if (e != hipSuccess) return hip_fail(e, "hipSetDevice");
        hipStream_t s = static_cast<hipStream_t>(stream);

        hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
        if (s && (e = hipStreamIsCapturing(s, &capture)) != hipSuccess) return hip_fail(e, "hipStreamIsCapturing");
        const bool capturing = capture != hipStreamCaptureStatusNone;

        std::lock_guard<std::mutex> lock(ctx->noalloc.mu);
        // the previous call's upload has been read out of the staging
        if (!capturing && (e = hipEventSynchronize(ctx->noalloc.staged)) != hipSuccess)
            return hip_fail(e, "no-alloc staging event");
        NoAllocPlan& P = capturing ? *ctx->noalloc.captured : *ctx->noalloc.staging;
        int* modes = ctx->noalloc.modes;
        int nplain = 0;
        for (int i = 0; i < count; ++i) {
            ImageGeom g;
            if (check_desc(&descs[i], &g) != ASTC_OK) return ASTC_ERR_INVALID_ARG;  // message set by check_desc
            if (!srcs[i] || !dsts[i] || (reinterpret_cast<uintptr_t>(dsts[i]) & 15u))
                return fail(ASTC_ERR_INVALID_ARG, "bad src/dst pointer (dst must be 16-byte aligned)");
            BatchLevel& L = P.levels[i];
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
            L.pad = 0;
            modes[i] = mode_of(descs[i].block_dim, descs[i].src_format, descs[i].flags, descs[i].width,
                               descs[i].height);
            if (descs[i].flags & ASTC_FLAG_MAX_ACCUMULATION) {
                modes[i] = -1;  // one plain launch after the batch kernels
                ++nplain;
            }
        }
        int nseg = 0;
        BatchLaunch l{};
        // a list that only fits in chunks of the tuning's size is planned with those
        const RunSteps whole{{bpl, bpl, bpl}};
        if (!plan_work_into(P.levels, modes, count, run_steps(P.levels, modes, count, t, ctx->num_cus),
                            ctx->noalloc.keys, P.segs, kNoAllocMaxImages, P.items, kNoAllocMaxItems, &nseg, l.end) &&
            !plan_work_into(P.levels, modes, count, whole, ctx->noalloc.keys, P.segs, kNoAllocMaxImages, P.items,
                            kNoAllocMaxItems, &nseg, l.end))
            return fail(ASTC_ERR_INVALID_ARG, "the batch needs more work items than the no-alloc maximum (131072)");
        for (int r = 0; r < RUN_COUNT; ++r) P.scalars[r] = l.end[r];

        uint8_t* base = static_cast<uint8_t*>(ctx->noalloc.scratch);
        BatchArgs a;
        a.levels = reinterpret_cast<const BatchLevel*>(base + offsetof(NoAllocPlan, levels));
        a.segs = reinterpret_cast<const BatchSeg*>(base + offsetof(NoAllocPlan, segs));
        a.items = reinterpret_cast<const BatchItem*>(base + offsetof(NoAllocPlan, items));
        a.scalars = reinterpret_cast<const int*>(base + offsetof(NoAllocPlan, scalars));
        a.tables = ctx->d_tables;
        a.prefetch = t.prefetch;
        const struct { size_t off, bytes; } parts[4] = {
            {offsetof(NoAllocPlan, levels), size_t(count) * sizeof(BatchLevel)},
            {offsetof(NoAllocPlan, segs), size_t(nseg) * sizeof(BatchSeg)},
            {offsetof(NoAllocPlan, items), size_t(l.end[RUN_COUNT - 1]) * sizeof(BatchItem)},
            {offsetof(NoAllocPlan, scalars), sizeof(P.scalars)}};
        if (capturing) {
            for (const auto& part : parts)
                if ((e = launch_inline_words(base + part.off, reinterpret_cast<const uint8_t*>(&P) + part.off, part.bytes,
                                             s)) != hipSuccess)
                    return hip_fail(e, "no-alloc work-list upload");
        } else {
            // fetched by the library's copy kernel through the staging's device address
            // (no DMA-engine copy: those stalled the host for milliseconds now and then)
            const uint8_t* staged_dev = static_cast<const uint8_t*>(ctx->noalloc.staging_dev);
            CopyRange ranges[4];
            for (int i = 0; i < 4; ++i)
                ranges[i] = CopyRange{base + parts[i].off, staged_dev + parts[i].off, int64_t(parts[i].bytes)};
            if ((e = launch_copies(ranges, 4, s)) != hipSuccess) return hip_fail(e, "no-alloc work-list upload");
            if ((e = hipEventRecord(ctx->noalloc.staged, s)) != hipSuccess)
                return hip_fail(e, "no-alloc staging event");
        }
        l.lanes = batch_lanes(t);
        l.one_per_cu = batch_one_per_cu(t);
        if ((e = launch_encode_batch(a, l, s)) != hipSuccess) return hip_fail(e, "no-alloc batch launch");
        for (int i = 0; i < count && nplain; ++i) {
            if (!(descs[i].flags & ASTC_FLAG_MAX_ACCUMULATION)) continue;
            ImageGeom g;
            (void)check_desc(&descs[i], &g);
            if ((e = launch_encode_plain(ctx->d_tables, descs[i], g, srcs[i], dsts[i], s, ctx->num_cus)) != hipSuccess)
                return hip_fail(e, "no-alloc plain launch");
        }
        return ASTC_OK;
    });
}
