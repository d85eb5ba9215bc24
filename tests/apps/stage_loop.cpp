// A caller of the stage kernels' C ABI (include/ospray_hip/hip_pt.h) other
// than the device: one frame of a committed world without volumes and without
// the radiance cache, 64-slot tiles of 8x8 pixels, point filter, the camera
// looking along +z with y up.  Built as a shared library by the test.
#include <hip/hip_runtime_api.h>

#include <cmath>
#include <cstring>
#include <vector>

#include "ospray_hip/hip_pt.h"
#include "pt_types.h"

namespace {
struct Buffers
{
  std::vector<void *> all;
  hipError_t err = hipSuccess;
  ~Buffers()
  {
    for (void *p : all)
      (void)hipFree(p);
  }
  template <typename T = float>
  T *words(size_t n) // cleared
  {
    void *p = nullptr;
    if (err == hipSuccess)
      err = hipMalloc(&p, 4 * n);
    if (err == hipSuccess) {
      all.push_back(p);
      err = hipMemset(p, 0, 4 * n);
    }
    return (T *)p;
  }
};
} // namespace

#define TRY(x)                                                                                                     \
  do {                                                                                                             \
    const hipError_t e_ = (x);                                                                                     \
    if (e_ != hipSuccess)                                                                                          \
      return (int)e_;                                                                                              \
  } while (0)

// counters: 0 a block for each bounce, the last pass in one kernel; 1 the same
// counters for every bounce, cleared between them; 2 cleared in their parts.
// outColor: w * h float4; outBytes: w * h sRGB words.
extern "C" int stage_loop(const HptScene *S, int w, int h, int spp, int perPass, int maxDepth, float fovy,
    const float *camPos, int counters, int blocks, float *outColor, uint32_t *outBytes)
{
  const hpt::DScene &scene = *reinterpret_cast<const hpt::DScene *>(S);
  Buffers B;
  hpt::DFrame F;
  std::memset(&F, 0, sizeof(F));
  F.width = w;
  F.height = h;
  F.tilesX = F.slotTilesX = (w + 7) / 8;
  F.tilesY = (h + 7) / 8;
  F.slotShift = 3;
  F.numPixPadded = F.tilesX * F.tilesY * 64;
  F.spp = spp;
  F.channels = 1;
  F.maxDepth = maxDepth;
  F.rouletteDepth = 5;
  F.maxScatteringEvents = 20;
  F.numFirstLightSamples = (uint32_t)scene.numLights;
  F.numIndirectLightSamples = 1;
  F.minContribution = 0.001f;
  F.maxRadiance = INFINITY;
  F.idxMask = F.idxMaskLight = 0xffff0000u;
  F.maxRec = scene.numLights;
  F.nrcBounce = -1;
  const float size = 2.f * std::tan(0.5f * fovy * 0.01745329251994329577f);
  const float sx = size * ((float)w / (float)h);
  std::memcpy(F.camOrg, camPos, 12);
  F.camDu[0] = -1.f * sx;
  F.camDv[1] = size;
  F.camDir00[0] = 0.f - 0.5f * F.camDu[0];
  F.camDir00[1] = 0.f - 0.5f * F.camDv[1];
  F.camDir00[2] = 1.f;
  F.camDirection[2] = 1.f;
  const size_t npix = (size_t)w * h, slots = (size_t)perPass * F.numPixPadded, recs = slots * F.maxRec;
  F.accRGBA = B.words(4 * npix);
  F.accZ = B.words(npix);
  F.accIDs = B.words<uint32_t>(3 * npix);
  F.fbColor = B.words(4 * npix);
  uint32_t *bytes = B.words<uint32_t>(npix);
  F.fbFormat = 2; // OSP_FB_SRGBA
  if (counters == 0)
    F.fbConverted = bytes;

  hpt::DPaths p{};
  for (float **a : {&p.org, &p.dir, &p.thr, &p.contrib, &p.lastP, &p.lastNs, &p.hitA, &p.hitB, &p.vtxP, &p.vtxNg, &p.vtxNs,
           &p.vtxThr, &p.vtxWo})
    *a = B.words(4 * slots);
  for (uint32_t **a : {&p.ld, &p.ids, &p.rng, &p.vtxLd})
    *a = B.words<uint32_t>(4 * slots);
  for (uint32_t **a : {&p.hitPrim, &p.neeN, &p.queue[0], &p.queue[1], &p.tieQueue})
    *a = B.words<uint32_t>(slots);
  for (float **a : {&p.recOrg, &p.recDir, &p.recContrib, &p.recResult, &p.recVol})
    *a = B.words(4 * recs);
  for (uint32_t **a : {&p.shadowQueue, &p.transQueue, &p.neeSampleQueue, &p.transCount})
    *a = B.words<uint32_t>(recs);
  p.transCap = (int32_t)recs;
  p.transHits = B.words(4 * hpt_trans_record_hits() * recs);
  p.overflow = B.words<uint32_t>((size_t)blocks * hpt_trace_block_size() * hpt_overflow_depth());
  p.stats = B.words<unsigned long long>(32);
  if (counters == 0)
    p.pass = B.words<int32_t>(hpt_counter_bytes(maxDepth + 1) / 4);
  else
    p.counters = B.words<int32_t>(hpt::kNumCounters);
  TRY(B.err);
  TRY(hipDeviceSynchronize());

  HptPaths *P = reinterpret_cast<HptPaths *>(&p);
  const HptFrame *Fp = reinterpret_cast<const HptFrame *>(&F);
  for (F.passS0 = 0; F.passS0 < spp; F.passS0 += perPass) {
    F.passCount = spp - F.passS0 < perPass ? spp - F.passS0 : perPass;
    if (counters == 0) {
      TRY(hpt_begin_pass(P, maxDepth + 1, F.passS0 == 0, nullptr));
      hpt_at_bounce(P, 0);
    } else {
      TRY(hpt_reset_counters(P, -1, nullptr));
    }
    TRY(hpt_generate(Fp, P, nullptr));
    for (int b = 0, q = 0; b <= maxDepth; b++, q ^= 1) {
      if (counters == 0)
        hpt_at_bounce(P, b);
      else if (counters == 1)
        TRY(hpt_reset_counters(P, q, nullptr));
      else
        TRY(hpt_reset_extension_counters(P, q, nullptr));
      TRY(hpt_extend(S, P, q, blocks, 0, nullptr));
      TRY(hpt_ties(S, P, blocks, 0, nullptr));
      if (counters == 2)
        TRY(hpt_reset_append_counters(P, q, nullptr));
      TRY(hpt_shade(S, Fp, P, q, blocks, nullptr));
      if (counters == 2)
        TRY(hpt_reset_shadow_counters(P, nullptr));
      TRY(hpt_nee(S, Fp, P, q, blocks, nullptr));
      TRY(hpt_shadow(S, Fp, P, blocks, 0, nullptr));
      TRY(hpt_shadow_trans(S, Fp, P, blocks, 0, nullptr));
      TRY(hpt_resolve(S, Fp, P, q, blocks, nullptr));
    }
    const bool last = F.passS0 + F.passCount >= spp;
    TRY(counters == 0 && last ? hpt_finish_frame(Fp, P, nullptr) : hpt_finish_pass(Fp, P, nullptr));
  }
  if (counters != 0) {
    TRY(hpt_fb_accumulate(Fp, nullptr));
    TRY(hpt_color_convert(F.fbColor, w * h, F.fbFormat, bytes, nullptr));
  }
  TRY(hipMemcpy(outColor, F.fbColor, 16 * npix, hipMemcpyDeviceToHost));
  TRY(hipMemcpy(outBytes, bytes, 4 * npix, hipMemcpyDeviceToHost));
  return 0;
}

// the counters at `pass` as a pass of `bounces` bounces finds them
extern "C" int begin_pass(int32_t *pass, int bounces)
{
  hpt::DPaths p{};
  p.pass = pass;
  return (int)hpt_begin_pass(reinterpret_cast<const HptPaths *>(&p), bounces, 1, nullptr);
}
