// Path pool and device work-queue loop of the regenerating wavefront
// renderers (batch.hip: the batch and fixed-spp path tracing; lt.hip:
// light tracing): a fixed pool of path slots whose free slots take the next
// work items, an iteration of regenerate -> extend -> shade -> connect
// kernels, enqueued in pairs until every item is done.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <functional>
#include <vector>

#include "lmgpu_internal.h"
#include "pt_device.h"

// Path pool of a fixed-spp render: slots per pixel and at most (1080p, 1.32M
// triangles, 16 spp: 1 per pixel 69.7 ms, 2: 56.6, 4: 51.2, 8: 47.6, before
// samples were resolved at the end of a run; 2^24 slots take 3.6 GB).
#ifndef LMGPU_REGEN_SLOTS_PER_PIXEL
#define LMGPU_REGEN_SLOTS_PER_PIXEL 8
#endif
#ifndef LMGPU_REGEN_MAX_SLOTS
#define LMGPU_REGEN_MAX_SLOTS (1 << 24)
#endif
// Samples a render keeps before they go to the film together: 16 B each, 2 GB
// at most (64 per pixel at 1080p). The buffer is allocated last, from what memory
// is left, outlives the render, and is given back when a later call of the
// scene has no memory for buffers of its own or renders far fewer samples
// (wavefront_give_back).
#ifndef LMGPU_REGEN_SAMPLES
#define LMGPU_REGEN_SAMPLES (1 << 27)
#endif
// Path pool of a guided render, whose slots also hold training records
// (record_depth x 96 B each): 4 slots per pixel, at most 2^23. With fewer
// paths in flight an iteration finishes about half a sample per pixel's
// worth of paths, so the guide can train after every such sample.
#ifndef LMGPU_REGEN_GUIDED_SLOTS_PER_PIXEL
#define LMGPU_REGEN_GUIDED_SLOTS_PER_PIXEL 4
#endif
#ifndef LMGPU_REGEN_GUIDED_MAX_SLOTS
#define LMGPU_REGEN_GUIDED_MAX_SLOTS (1 << 23)
#endif

namespace lmgpu {

struct JobDev {
    SceneDev sc;          // job-local pointers into the shading arenas
    int root;             // root of the job's BVH in the node arena
    int npix, spp, max_verts, mode, rr_depth;
    uint32_t seed_lo, seed_hi;
    int64_t film_off;     // first double of the job's film (3 per pixel)
};

// A run of consecutive work items: the pixels 0.. of one sample of one job,
// starting at queue position `start`.
struct WorkSeg {
    int64_t start;
    int32_t job, sample;
};

// Slot states, in the low bits; a finishing path's slot holds the vertex
// count at which it ended above them.
constexpr int32_t kFree = 0, kActive = 1, kFinishing = 2;
constexpr int kStateShift = 8;
constexpr int32_t kStateMask = (1 << kStateShift) - 1;

// Path slots: what outlives one iteration of a path. L.w holds the sample
// index's bits.
struct PoolDev {
    int32_t *job, *pixel, *state;
    float4* L;
};

// Vertex count and flags (PathRegs::info.x, .z) of a path in one word.
LMGPU_HD int32_t pack_info(int nv, int flags) { return nv | (flags << 8); }
LMGPU_HD int info_verts(int32_t w) { return w & 0xff; }
LMGPU_HD int info_flags(int32_t w) { return w >> 8; }

// Extension queues: entry i of a queue is a path's next ray with its state,
// written by the vertex that sampled it and read once by the next.
struct BatchQ {
    lmgpu_ray* ext[2];    // tmin holds the slot's bits, tmax the pdf of the direction (projected SA)
    float4* thr[2];       // throughput, w = pack_info bits
    float4* prev[2];      // shading normal of the previous vertex, w = pixel bits
    lmgpu_hit* hit;
    lmgpu_ray* sh;
    float4* sh_contrib;   // xyz contribution, w = path slot bits
    int32_t* counts;      // see ext_count, shadow_count; [5] stack overflow flag
};

struct BatchCtl {
    // the two counters that every block of the regenerate kernel updates sit
    // in cache lines of their own
    alignas(128) unsigned long long work_next;   // next work item to hand out
    alignas(128) unsigned long long remaining;   // work items not yet accumulated
    alignas(128) unsigned long long ext_rays;
    unsigned long long shadow_rays;
    unsigned long long t_start;     // device clock at the start of the run
    unsigned long long iterations;  // iterations that found work left
};


// Grid of a regenerate kernel over a pool of `cap` slots: at most
// kRegenStrides strides of the pool per block (its LDS table), and otherwise
// kRegenMinStrides, as each block updates the shared counters once (12 ns an
// update; 1, 4 and 8 strides: 9.6, 8.2 and 8.1 ms for a guided 540p frame);
// at most 4096 blocks.
constexpr int kRegenStrides = 32;
constexpr int kRegenMinStrides = 8;
inline unsigned regen_grid(int64_t cap, int block) {
    auto blocks = [&](int64_t per) { return (cap + per * block - 1) / (per * block); };
    return unsigned(std::max(std::max<int64_t>(1, std::min<int64_t>(blocks(kRegenMinStrides), 4096)), blocks(kRegenStrides)));
}

struct Guide;

// Guided path tracing in the regenerating loop: the guide, its options and
// the scene the inference reads hit points from.
struct RegenGuide {
    Guide* g = nullptr;
    SceneDev sc{};
    GBox box{};
    float alpha = 0.5f, lr = 1e-3f, wclamp = 50.f;
    int batch = 0, steps = 0, rec_depth = 0;
    int npix = 0;   // the guide trains after every npix finished paths
};

// Path pool, work queue and the loop that drains it (regenerate -> extend ->
// shade -> connect, pairs of iterations one ahead of the device), shared by the batch
// and by lmgpu_pt_render's regenerating path.
struct Wavefront {
    int cap = 0;
    DevBuf<int32_t> pjob, ppix, pstate, counts;
    DevBuf<float4> pL, thr0, thr1, prev0, prev1;
    DevBuf<lmgpu_ray> ext0, ext1, sh;
    DevBuf<lmgpu_hit> hit;
    DevBuf<float4> shc;
    DevBuf<float4> psample;   // finished samples of a single scene's run, by work item
    DevBuf<BatchCtl> ctl;
    // pinned host copies of the control block and the queue counts, one per
    // parity of the pairs of iterations, with the pairs' events
    struct HostMirror {
        BatchCtl ctl;
        int32_t counts[16];
    };
    HostMirror* mirror = nullptr;
    HostMirror last{};                // the copy that ended the last run
    hipEvent_t pair_ev[2] = {nullptr, nullptr}, ev[2] = {nullptr, nullptr};
    DevBuf<unsigned long long> next;
    // per-run tables: jobs, work segments, per-job completion counters and clocks
    DevBuf<JobDev> djobs;
    DevBuf<WorkSeg> dsegs;
    DevBuf<unsigned long long> job_done, job_time;
    // guided runs: training records per (vertex, slot), decoded mixtures per
    // extension-queue entry, the record slot of each shadow-queue entry, the
    // training buffer with its counters ([0] appended, [1] released to the
    // training steps, [2] paths finished since the last release) and the
    // count of training records
    DevBuf<GRec> grec;
    DevBuf<float> gmix, gtrain;
    DevBuf<int32_t> gshrec, gcnt;
    DevBuf<unsigned long long> grecorded;
    Wavefront() = default;
    Wavefront(const Wavefront&) = delete;
    Wavefront& operator=(const Wavefront&) = delete;
    ~Wavefront();
    int ensure_host();
    int ensure_pool(int cap);
    // Guided buffers for the current pool (records zeroed when allocated).
    int ensure_guided(int rec_depth, int64_t train_cap);
    // Uploads the jobs and the work segments (queue order) of one run, on s; the
    // vectors live until the run has ended.
    int set_work(const std::vector<JobDev>& jobs, const std::vector<WorkSeg>& segs, hipStream_t s);
    // Renders every work item of the tables set last into film_sum / film_sq
    // (film_sq may be null) and waits for the end.
    // With a guide, the directions at diffuse and glossy vertices come from
    // the one-sample mixture of guide and BSDF, and the guide trains online
    // on the records of finished paths.
    // single: one job, whose work segment 0 starts at its first sample
    // (kernels specialised for it, at their own block size). resolve: its
    // samples are left in psample, which holds `total`, not added to the film.
    int run(const void* trav_nodes, const TriV* tris, int width, int block, bool single, int64_t total, int max_verts,
            double* film_sum, double* film_sq, double* elapsed, int64_t* iters, hipStream_t s,
            const RegenGuide* guide = nullptr, bool resolve = false);
    // The loop itself: frees the pool, sets the run's counters for `total`
    // items and enqueues pairs of iteration(stream, 0) and iteration(stream, 1)
    // (the kernels of one iteration on queue parity 0 / 1), captured as one
    // graph if `graph`, until every item is done; max_verts bounds the
    // iterations. `last` holds the final counters.
    int loop(const std::function<void(hipStream_t, int)>& iteration, int64_t total, int max_verts, bool graph,
             double* elapsed, int64_t* iters, hipStream_t s);
    // Slot count for `total` items over `npix` pixels: per_pixel slots per
    // pixel, a power of two in [4096, max_slots].
    static int pool_size(int64_t total, int npix, int per_pixel = LMGPU_REGEN_SLOTS_PER_PIXEL,
                         int max_slots = LMGPU_REGEN_MAX_SLOTS) {
        const int64_t want = std::min<int64_t>(total, int64_t(per_pixel) * npix);
        int c = 4096;
        while (c < want && c < max_slots) c <<= 1;
        return c;
    }
};

}  // namespace lmgpu


