/* Thin C-ABI launch layer of the hip path tracer (libospray_module_hip.so).
 *
 * Replaces the reference's device-runtime seam: devicert::Device::
 * launchRendererKernel / launchFrameOpKernel (ospray/common/DeviceRT.h:170-195)
 * and the ISPC/SYCL launch templates DEFINE_RENDERER_KERNEL_LAUNCHER /
 * DEFINE_FRAMEOP_KERNEL_LAUNCHER (modules/cpu/common/DeviceRT.ih:12-115).
 * Every function enqueues on the given stream, never throws, never
 * allocates, and returns the hipError_t of the launch.  Arguments are plain
 * structs of device pointers and sizes whose layout is defined in
 * ospray_amd/csrc/hip/pt_types.h (HptScene = hpt::DScene,
 * HptFrame = hpt::DFrame, HptPaths = hpt::DPaths).
 */
#pragma once

#include <hip/hip_runtime_api.h>
#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

typedef struct HptScene HptScene; /* committed world: BVH, primitives, materials, lights */
typedef struct HptFrame HptFrame; /* camera, renderer parameters, pass range, fb buffers */
typedef struct HptPaths HptPaths; /* wavefront path state, queues and counters */

#ifndef HPT_API
#define HPT_API __attribute__((visibility("default")))
#endif

/* Counters of the queues, in one of two ways.
 *
 * A block for each bounce, cleared at once: P->pass points to
 * hpt_counter_bytes(bounces) bytes of device memory.  hpt_begin_pass clears
 * them for a pass of `bounces` bounces and polls the frame's cancellation,
 * whose latch firstPass != 0 clears before.  hpt_at_bounce (host only) points
 * P at the counters of bounce b (from 0) for the calls that follow, and leaves
 * P as it is where P->pass is null or b is negative.  Stages of bounce b may
 * run on a second stream beside the extension of bounce b+1: they share no
 * counter. */
HPT_API size_t hpt_counter_bytes(int bounces);
HPT_API hipError_t hpt_begin_pass(const HptPaths *P, int bounces, int firstPass, hipStream_t s);
HPT_API void hpt_at_bounce(HptPaths *P, int bounce);
/* The same counters for every bounce: P->pass is null and P->counters points
 * to kNumCounters words; the calls below clear them between the bounces, and
 * fail with hipErrorInvalidValue where P->pass is set.
 * keepIndex -1: sets every counter to 0.  keepIndex 0 or 1: sets the
 * per-bounce queue counters to 0 except the two words of extension queue
 * `keepIndex` (its entry count and the NEE samples appended with it; the
 * radiance-cache counters of the pass are kept).  A cancelled frame (the
 * host wrote the frame's generation into the paths' cancellation word)
 * also empties the kept queue and latches the cancellation. */
HPT_API hipError_t hpt_reset_counters(const HptPaths *P, int keepIndex, hipStream_t s);
/* The parts of the per-bounce reset, for a frame whose shadow-ray stages
 * (hpt_nee .. hpt_resolve) of bounce b run on a second stream beside the
 * extension of bounce b+1: before the extension, its work fetch and the
 * near-tie queue (with the cancellation check); after bounce b's resolve
 * (which still reads the queue it shaded), the two words of the queue the
 * shading of bounce b+1 appends to (extension queue keepIndex ^ 1); on the
 * second stream before bounce b+1's NEE, the shadow records, the
 * transparency queue and their work fetch. */
HPT_API hipError_t hpt_reset_extension_counters(const HptPaths *P, int keepIndex, hipStream_t s);
HPT_API hipError_t hpt_reset_append_counters(const HptPaths *P, int keepIndex, hipStream_t s);
HPT_API hipError_t hpt_reset_shadow_counters(const HptPaths *P, hipStream_t s);
HPT_API hipError_t hpt_fill_u32(uint32_t *ptr, size_t n, uint32_t value, hipStream_t s);
/* dst <- src, bytes a multiple of 16: a plain streaming copy that calibrates
 * bandwidth figures and HBM counters (no reference counterpart). */
HPT_API hipError_t hpt_copy(void *dst, const void *src, size_t bytes, hipStream_t s);

/* Camera rays of the pass's samples (PathTracer.ispc:75-170). */
HPT_API hipError_t hpt_generate(const HptFrame *F, const HptPaths *P, hipStream_t s);
/* Closest hit of every ray in extension queue `queue` (World.ih:247-286). */
HPT_API hipError_t hpt_extend(const HptScene *S, const HptPaths *P, int queue, int residentBlocks, int stats, hipStream_t s);
/* FP64 re-resolution of the extension hits hpt_extend found within a
 * near-tie window of another hit (the FP64 intersection check on near-tie
 * rays; no counterpart in the reference, which trusts Embree's float hit):
 * every hit in the window gets its distance in double precision and the
 * smallest (FP64 t, key) is kept.  residentBlocks: at most the grid the
 * traversal scratch rows are sized for.  stats != 0 adds node visits and
 * primitive tests to P->stats[0..1]. */
HPT_API hipError_t hpt_ties(const HptScene *S, const HptPaths *P, int residentBlocks, int stats, hipStream_t s);
/* volumeSampleFreePath (volumes/VolumeSampler.ispc:96-199) of every ray of
 * extension queue `queue` after hpt_extend: delta tracking up to the
 * surface hit; a collision turns the hit record into a volume vertex.
 * Launched only for worlds with volumes.  stats != 0 adds voxel samples,
 * macrocell intervals and tracked segments to P->stats[9..11]. */
HPT_API hipError_t hpt_volume(const HptScene *S, const HptPaths *P, int queue, int blocks, int stats, hipStream_t s);
/* One samplePath bounce (PathSampler.ispc:143-407) for queue `queue`; the
 * NEE light samples of its smooth vertices are queued for hpt_nee.  With
 * F->nrcBounce >= 0 the vertices of that depth become radiance-cache
 * queries or training records (no reference counterpart). */
HPT_API hipError_t hpt_shade(const HptScene *S, const HptFrame *F, const HptPaths *P, int queue, int blocks, hipStream_t s);
/* One NEE light sample per thread for the vertices shaded from extension
 * queue `queue`: light selection and sampling, BSDF evaluation, shadow-ray
 * record (NextEventEstimation.ispc:54-146). */
HPT_API hipError_t hpt_nee(const HptScene *S, const HptFrame *F, const HptPaths *P, int queue, int blocks, hipStream_t s);
/* transparentShadow of every NEE record (TransparentShadow.ispc:18-85),
 * first pass: occlusion with early exit on an opaque primitive; records
 * that hit only non-opaque surfaces are queued for hpt_shadow_trans.
 * stats != 0 adds node visits, primitive tests and traversals to
 * P->stats[3..5]. */
HPT_API hipError_t hpt_shadow(
    const HptScene *S, const HptFrame *F, const HptPaths *P, int residentBlocks, int stats, hipStream_t s);
/* transparentShadow, second pass: the closest-hit loop through non-opaque
 * surfaces (TransparentShadow.ispc:36-84) for the queued records. */
HPT_API hipError_t hpt_shadow_trans(
    const HptScene *S, const HptFrame *F, const HptPaths *P, int residentBlocks, int stats, hipStream_t s);
/* Radiance cache (no reference counterpart): the raw inputs (position,
 * direction, normal, albedo) of the n queued query (which = 0) or training
 * (which = 1) records; contribution += throughput * max(prediction, 0) for
 * the n queries; the n training targets (radiance gathered after the
 * vertex / throughput at the vertex, clamped to [0, 1e4]). */
HPT_API hipError_t hpt_nrc_gather(const HptPaths *P, int which, int n, float *raw12, hipStream_t s);
HPT_API hipError_t hpt_nrc_apply(const HptPaths *P, int n, const float *pred3, hipStream_t s);
HPT_API hipError_t hpt_nrc_targets(const HptPaths *P, int n, float *target3, hipStream_t s);
/* Ordered sum of the NEE samples of every vertex shaded from extension
 * queue `queue` (NextEventEstimation.ispc:150-159); with volumes, each
 * visible sample's transmittance estimates (NextEventEstimation.ispc:126-149). */
HPT_API hipError_t hpt_resolve(
    const HptScene *S, const HptFrame *F, const HptPaths *P, int queue, int blocks, hipStream_t s);
/* ScreenSample_accumulate over the pass (PathTracer.ispc:170-197). */
HPT_API hipError_t hpt_finish_pass(const HptFrame *F, const HptPaths *P, hipStream_t s);
/* LocalFB_accumulateSample (fb/LocalFB.ispc:14-78). */
HPT_API hipError_t hpt_fb_accumulate(const HptFrame *F, hipStream_t s);
/* A frame's last pass in one kernel: hpt_finish_pass, hpt_fb_accumulate and,
 * where F->fbConverted is set, hpt_color_convert to F->fbFormat. */
HPT_API hipError_t hpt_finish_frame(const HptFrame *F, const HptPaths *P, hipStream_t s);
/* Variance_kernel (fb/frame_ops/Variance.ispc:11-59). */
HPT_API hipError_t hpt_variance(const HptFrame *F, hipStream_t s);
/* getAvgError (fb/frame_ops/Variance.cpp:32-46), FP64 sum, one float out.
 * frameState (optional): the device-resident frame index of a captured
 * batch frame; the reduction then runs only when it is odd. */
HPT_API hipError_t hpt_variance_reduce(const float *taskVariance, int n, float threshold, float *out,
    const uint32_t *frameState, hipStream_t s);
/* ColorConversion_kernel (fb/frame_ops/ColorConversion.ispc:11-36);
 * format is an OSPFrameBufferFormat. */
HPT_API hipError_t hpt_color_convert(const float *color, int npix, int format, void *out, hipStream_t s);
/* Closest hits of an explicit ray list: rays8 = org.xyz, dir.xyz, t0, t1;
 * outTUV = t,u,v; outIDs = instance, model, primitive (0xffffffff on miss);
 * stats (optional) += node visits, primitive tests. */
HPT_API hipError_t hpt_trace_rays(const HptScene *S, const float *rays8, int n, float *outTUV, uint32_t *outIDs,
    uint32_t *overflow, int residentBlocks, unsigned long long *stats, hipStream_t s);

/* hpt_trace_rays without a scratch argument, for callers that cannot
 * allocate device memory (code under HIP graph capture, tight serving
 * loops, harnesses that forbid hipMalloc).  No counterpart in the
 * reference.  The traversal scratch rows come from a fixed device array of
 * the module (66 MiB per GPU, held until the process ends), so
 * residentBlocks must be in [1, hpt_trace_noalloc_max_blocks()]; anything
 * else returns hipErrorInvalidValue before launching.  Allocates nothing
 * (no hipMalloc, hipFree or allocating library call).  All calls on one GPU
 * share that GPU's array: calls that overlap in time on one GPU (on
 * different streams or from different threads) race and must be
 * serialised by the caller.  Results equal hpt_trace_rays's. */
HPT_API hipError_t hpt_trace_rays_noalloc(const HptScene *S, const float *rays8, int n, float *outTUV,
    uint32_t *outIDs, int residentBlocks, unsigned long long *stats, hipStream_t s);
/* the largest residentBlocks hpt_trace_rays_noalloc accepts */
HPT_API int hpt_trace_noalloc_max_blocks(void);

/* threads per block of the traversal kernels */
HPT_API int hpt_trace_block_size(void);
/* 32-bit words of the scratch row each resident traversal thread needs in
 * `overflow` (HptPaths and hpt_trace_rays): the traversal-stack overflow,
 * then the transparent hits an occlusion traversal records and their
 * count.  The rows must be zero when first used (hpt_shadow keeps each
 * row's count at zero between rays). */
HPT_API int hpt_overflow_depth(void);
/* traversal stack entries per ray (LDS + overflow) */
HPT_API int hpt_stack_capacity(void);
/* transparent hits the occlusion pass records per shadow ray for the
 * transparency pass (HptPaths.transHits holds this many per queue slot) */
HPT_API int hpt_trans_record_hits(void);

#ifdef __cplusplus
}
#endif
