// Host launch interface of the wavefront path-tracing stages.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "dev_guide.h"
#include "pt_types.h"

// Path state, indexed by path id (tile pixel).  A path's first shading starts
// it (generation writes only the random-number state), and a bounce reads and
// writes what the path needs: absorb only inside an absorbing medium, texc
// only in scenes with texture maps, the next-event arrays only for the terms a
// vertex has.
struct PathBufs {
    float4* rad;     // radiance, state word (material, pending next-event terms, absorb stored)
    float4* thr;     // throughput, previous BSDF pdf
    float4* absorb;  // Beer-Lambert absorption coefficient
    uint4* rng;      // pcg4d state
    float2* texc;    // last surface's texture coordinate
    float4* nee;     // 3 arrays: env term, light term (w = 1 while unoccluded), throughput
    int* job;        // job id per path (multi-job passes only)
    int64_t stride;  // paths per array of nee
};

// Learned-guide hook of a pass.
//   enabled  the shade stage draws from the guide (lobes of the current hit
//            queue, kGuideLobeF4 float4 per entry) mixed with the BSDF
//   train    training records are written for paths p with p % stride == phase:
//            4 float4 per (recorded path, depth) = (pos, continued),
//            (n, lum throughput before the vertex), (wo, lum radiance before
//            the next vertex), (wi, 0)
namespace lfhd {
struct GuideHook {
    int enabled = 0;
    int sample = 1;   // 0: the guide is queried and trained but directions come from the BSDF alone
    int train = 0;
    int max_depth = 0;
    int stride = 1;
    int phase = 0;
    float4* rec = nullptr;
    // processed lobes of hit-queue entry i: float4 k at lobes[k * lobe_stride + i]
    // (structure of arrays, so each of a wave's ten loads is one contiguous run)
    const float4* lobes = nullptr;
    int lobe_stride = 0;
};
}  // namespace lfhd
using lfhd::GuideHook;


// Queues and counters of a wavefront.  counts: the (extension, shadow) rays
// that each of kQueueSets traversals in turn takes, 8-byte aligned pairs;
// work: their fetch counters and the running ray totals.
struct PtQueues {
    float4* rayq[2];      // extension rays of even and odd depths, 2 float4 each
    float4* hitq;         // 2 float4 per extension ray
    float4* shadowq;      // 2 float4 per shadow ray, two per path
    uint32_t* counts;
    unsigned long long* work;
    uint32_t* spill;      // traversal stacks of grid_blocks blocks
    int* err;             // set when a stack overflows
    int maxq;             // path capacity
    int grid_blocks;
    float cull;
};

// Starts a wavefront: adds the ray counts the last one left to the totals and
// clears the counters.
hipError_t pt_reset(uint32_t* counters, unsigned long long* work, hipStream_t s);
// max_depth: the depth of the bounces that follow
hipError_t pt_generate(const lfhd::CamParams& cam, int max_depth, const PathBufs& pb, float4* rayq, uint32_t* count,
                       hipStream_t s);
hipError_t pt_generate_rays(const float* rays6, const uint4* seeds, int n, int max_depth, const PathBufs& pb, float4* rayq,
                            uint32_t* count, hipStream_t s);
// All the bounces of a wavefront (gh.enabled: guided with gd's weights).
hipError_t pt_bounces(const lfhd::ShadeScene& sc, int max_depth, const PtQueues& q, const PathBufs& pb,
                      const GuideHook& gh, const lfhd::GuideDev* gd, hipStream_t s);
// Multi-job pass (serving): every job renders its full frame once; rays of all
// jobs share the queues.  jobs: device table of njobs entries.
hipError_t pt_generate_multi(const lfhd::JobDev* jobs, int njobs, int total, int max_depth, const PathBufs& pb, float4* rayq,
                             uint32_t* count, hipStream_t s);
// gh.enabled: a guided wavefront, all of whose jobs render guide_sc's scene.
hipError_t pt_bounces_multi(const lfhd::JobDev* jobs, int max_depth, const PtQueues& q, const PathBufs& pb,
                            const GuideHook& gh, const lfhd::GuideDev* gd, const lfhd::ShadeScene* guide_sc,
                            hipStream_t s);
// keep_radiance: the paths' final radiance stays in pb.rad (guide training)
hipError_t pt_accumulate_multi(const lfhd::JobDev* jobs, int total, const PathBufs& pb, bool keep_radiance,
                               hipStream_t s);
hipError_t pt_accumulate(const PathBufs& pb, const lfhd::CamParams& cam, float4* accum, float4* comp, int kahan,
                         bool keep_radiance, hipStream_t s);
hipError_t pt_collect(const PathBufs& pb, int n, float* out, hipStream_t s);
hipError_t pt_output(const float4* accum, const float4* comp, int64_t npix, float inv, float* out, hipStream_t s);
hipError_t pt_clear4(float4* a, int64_t n, hipStream_t s);
hipError_t pt_clear_flag(int* flag, hipStream_t s);
int pt_trace_grid_blocks();

hipError_t stage_eval_bsdf(const lfhd::ShadeScene& sc, const float* fr, const float* L, int n, float* f, float* pdf,
                           hipStream_t s);
hipError_t stage_sample_bsdf(const lfhd::ShadeScene& sc, const float* fr, uint4* seeds, int n, float* L, float* f,
                             float* pdf, hipStream_t s);
hipError_t stage_sample_light(const lfhd::ShadeScene& sc, const float* pos, uint4* seeds, int n, float* dir,
                              float* nrm, float* em, float* dist, float* pdf, hipStream_t s);
hipError_t stage_sample_env(const lfhd::ShadeScene& sc, uint4* seeds, int n, float* dir, float* pdf, float* col,
                            hipStream_t s);
hipError_t stage_env_pdf(const lfhd::ShadeScene& sc, const float* dir, int n, float* pdf, hipStream_t s);
