// Volume sampling of the hip path tracer: structured-regular grids,
// piecewise-linear transfer function, macrocell majorants, delta tracking
// and the Henyey-Greenstein phase function, following
//   render/pathtracer/volumes/VolumeSampler.ispc:13-279 (delta_tracking,
//     volumeSampleFreePath, volumeTransmittance)
//   volume/transferFunction/LinearTransferFunction.ispc:11-60
//   render/pathtracer/volumes/HenyeyGreenstein.ih:14-77
//   math/random.ih:116-154 (the per-path PCG32 RandomSampler)
// The reference leaves grid sampling and interval iteration to OpenVKL; here
// a sample is the trilinear interpolation of the vertex-centred voxels
// (NaN outside the box) and the intervals of a ray are its runs through
// the macrocells of kMacro^3 cells, each with the macrocell's (min, max)
// voxel value as value range (its majorant precomputed per model).
#pragma once

#include "pt_shade.h"
#include "pt_types.h"

namespace hpt {

// ---- PCG32 RandomSampler (math/random.ih:116-154) ---------------------------------

struct RandomSampler
{
  uint64_t state;
  uint32_t stream;
};

HPT_HD uint32_t murmur3Mix(uint32_t hash, uint32_t k)
{
  k *= 0xcc9e2d51u;
  k = (k << 15) | (k >> 17);
  k *= 0x1b873593u;
  hash ^= k;
  return ((hash << 13) | (hash >> 19)) * 5u + 0xe6546b64u;
}

HPT_HD uint32_t murmur3Finalize(uint32_t h)
{
  h ^= h >> 16;
  h *= 0x85ebca6bu;
  h ^= h >> 13;
  h *= 0xc2b2ae35u;
  h ^= h >> 16;
  return h;
}

HPT_HD uint32_t pcg32(RandomSampler &r)
{
  const uint64_t old = r.state;
  r.state = old * 6364136223846793005ULL + (uint64_t)(r.stream | 1u);
  const uint32_t xorshifted = (uint32_t)(((old >> 18u) ^ old) >> 27u);
  const uint32_t rot = (uint32_t)(old >> 59u);
  return (xorshifted >> rot) | (xorshifted << ((0u - rot) & 31u));
}

HPT_HD void randomSamplerInit(RandomSampler &r, uint32_t seed, uint32_t stream)
{
  r.stream = (stream << 1u) | 1u;
  r.state = murmur3Finalize(murmur3Mix(0u, seed));
  pcg32(r);
  r.state += seed;
  pcg32(r);
}

HPT_HD float randomFloat(RandomSampler &r) { return to_float_unorm(pcg32(r)); }

// ---- grid and transfer function ------------------------------------------------------

HPT_HD float lerpf(float t, float a, float b) { return (1.f - t) * a + t * b; }

HPT_HD float safeRcp(float d) // |d| >= 1e-18
{
  const float ad = fabsf(d);
  return 1.0f / (ad < 1e-18f ? copysignf(1e-18f, d) : d);
}

// trilinear sample at volume-space p; NaN outside the grid's box
HPT_HD float volumeSample(const DVolume &v, vec3f p)
{
  const float lx = (p.x - v.origin[0]) / v.spacing[0];
  const float ly = (p.y - v.origin[1]) / v.spacing[1];
  const float lz = (p.z - v.origin[2]) / v.spacing[2];
  if (!(lx >= 0.f && ly >= 0.f && lz >= 0.f && lx <= (float)(v.dims[0] - 1) && ly <= (float)(v.dims[1] - 1)
          && lz <= (float)(v.dims[2] - 1)))
    return __builtin_nanf("");
  const int ix = (int)lx < v.dims[0] - 2 ? (int)lx : v.dims[0] - 2;
  const int iy = (int)ly < v.dims[1] - 2 ? (int)ly : v.dims[1] - 2;
  const int iz = (int)lz < v.dims[2] - 2 ? (int)lz : v.dims[2] - 2;
  const float fx = lx - (float)ix, fy = ly - (float)iy, fz = lz - (float)iz;
  const size_t sy = (size_t)v.dims[0], sz = (size_t)v.dims[0] * (size_t)v.dims[1];
  const float *b = v.voxels + (size_t)iz * sz + (size_t)iy * sy + (size_t)ix;
  const float c00 = lerpf(fx, b[0], b[1]);
  const float c10 = lerpf(fx, b[sy], b[sy + 1]);
  const float c01 = lerpf(fx, b[sz], b[sz + 1]);
  const float c11 = lerpf(fx, b[sz + sy], b[sz + sy + 1]);
  const float c0 = lerpf(fy, c00, c10);
  const float c1 = lerpf(fy, c01, c11);
  return lerpf(fz, c0, c1);
}

// LinearTransferFunction_get (LinearTransferFunction.ispc:11-43), split in
// the opacity (every tentative collision) and the colour (real collisions)
// scale: rcp(tfUpper - tfLower)
HPT_HD float tfUnit(const DVolume &v, float value, float scale)
{
  value = (value - v.tfLower) * scale;
  const float nextBefore1 = 0.999999940395355224609375f; // 0x1.fffffep-1
  return !(value > 0.f) ? 0.f : (value > nextBefore1 ? nextBefore1 : value); // NaN -> 0
}

HPT_HD float tfOpacity(const DVolume &v, float u)
{
  const int maxIdx = v.numOpacities - 1;
  const float idxf = u * (float)maxIdx;
  const float frac = idxf - floorf(idxf);
  const int idx = (int)idxf;
  return lerpf(frac, v.tfOpacity[idx], v.tfOpacity[idx + 1 < maxIdx ? idx + 1 : maxIdx]);
}

HPT_HD vec3f tfColor(const DVolume &v, float u)
{
  const int maxIdx = v.numColors - 1;
  const float idxf = u * (float)maxIdx;
  const float frac = idxf - floorf(idxf);
  const int idx = (int)idxf;
  const int idx1 = idx + 1 < maxIdx ? idx + 1 : maxIdx;
  const float *c0 = v.tfColor + 3 * idx, *c1 = v.tfColor + 3 * idx1;
  return v3(lerpf(frac, c0[0], c1[0]), lerpf(frac, c0[1], c1[1]), lerpf(frac, c0[2], c1[2]));
}

// LinearTransferFunction_getMaxOpacity (LinearTransferFunction.ispc:45-58)
// over a kTfSubranges^2 table (used on the host to build the majorant grid)
HPT_HD float tfMaxOpacity(const float *maxOpacity, float tfLower, float tfUpper, float lower, float upper)
{
  const int maxDim = kTfSubranges - 1;
  const float denom = tfUpper - tfLower;
  const float a = (lower - tfLower) / denom, b = (upper - tfLower) / denom;
  const int i = (int)floorf((!(a > 0.f) ? 0.f : (a > 1.f ? 1.f : a)) * (float)maxDim); // NaN -> 0
  const int j = (int)ceilf((!(b > 0.f) ? 0.f : (b > 1.f ? 1.f : b)) * (float)maxDim);
  return maxOpacity[(i < maxDim ? i : maxDim) * kTfSubranges + (j < maxDim ? j : maxDim)];
}

// the ray's parameter range inside the volume's box, clipped to [t0, t1]
// (intersectBox, common/Intersect.ih:195-222; Volume_intersect_kernel,
// volume/Volume.ispc:22-75)
HPT_HD bool volumeBox(const DVolume &v, vec3f o, vec3f d, float t0, float t1, float &lo, float &hi)
{
  const vec3f inv = v3(safeRcp(d.x), safeRcp(d.y), safeRcp(d.z));
  const vec3f mins = (ld3(v.origin) - o) * inv, maxs = (ld3(v.upper) - o) * inv;
  const float nx = minf(mins.x, maxs.x), ny = minf(mins.y, maxs.y), nz = minf(mins.z, maxs.z);
  const float fx = maxf(mins.x, maxs.x), fy = maxf(mins.y, maxs.y), fz = maxf(mins.z, maxs.z);
  const float entry = maxf(maxf(nx, ny), nz);
  const float exit = minf(minf(fx, fy), fz);
  lo = maxf(t0, entry);
  hi = minf(t1, exit);
  return lo < hi;
}

template <typename T>
__device__ __forceinline__ T pick(int a, T x, T y, T z)
{
  return a == 0 ? x : (a == 1 ? y : z);
}

// tentative collisions per track before delta tracking gives up (the
// track then counts as passed)
constexpr int kMaxDeltaSteps = 1 << 16;

// work counters of delta tracking: voxel samples (tentative collisions),
// macrocell intervals entered, tracked segments
struct VolCount
{
  uint32_t samples = 0, cells = 0, tracks = 0;
};

// delta_tracking (VolumeSampler.ispc:13-92) over [t0, t1] (inside the box),
// walking the macrocells with a 3D DDA: the distance of the first real
// collision (inf if none) and its albedo.  The optical depth to the next
// tentative collision, tau ~ Exp(1), is drawn once per track and after each
// tentative collision, and carried across macrocell intervals: an interval
// of majorant mu and length l uses up mu * l of it.  The exponential is
// memoryless, so the collision distances have the distribution of a fresh
// draw per interval, with one logarithm per collision instead of one per
// interval.
//
// A macrocell step is short and waits on one load, a tentative collision is
// some ten times as long and rare (a few a track), so a lane that reaches
// one holds it until as many lanes hold as walk, and the load of the next
// interval's majorant is issued before the present interval is looked at
// (its cell does not depend on it).  Colliding as it came and loading on
// arrival, the 720p cloud frame's free paths took 1.69 ms and its shadow
// transmittances 2.55; now 1.14 and 1.96 (collisions at two, four and eight
// walkers a holder: 1.19, 1.26, 1.35 and 2.02, 2.16, 2.32; at half a walker
// 1.20 and 2.00).
__device__ __forceinline__ float deltaTracking(
    const DVolume &v, vec3f o, vec3f d, float t0, float t1, RandomSampler &rs, vec3f &albedo, VolCount &cnt)
{
  if (!(t0 < t1))
    return kInf;
  cnt.tracks++;
  const DVolume vc = v; // loaded once a track
  const float oo[3] = {o.x, o.y, o.z}, dd[3] = {d.x, d.y, d.z};
  const float ii[3] = {safeRcp(d.x), safeRcp(d.y), safeRcp(d.z)};
  const float tfScale = rcp(vc.tfUpper - vc.tfLower);
  float msz[3], tnext[3];
  int m[3], step[3];
  for (int k = 0; k < 3; k++) {
    msz[k] = vc.spacing[k] * (float)kMacro;
    const float p = oo[k] + t0 * dd[k];
    const float cf = floorf((p - vc.origin[k]) / msz[k]);
    const int c = !(cf > 0.f) ? 0 : (cf >= (float)vc.mdims[k] ? vc.mdims[k] - 1 : (int)cf);
    m[k] = c;
    step[k] = dd[k] > 0.f ? 1 : (dd[k] < 0.f ? -1 : 0);
    tnext[k] = step[k] == 0 ? kInf : (vc.origin[k] + (float)(c + (step[k] > 0 ? 1 : 0)) * msz[k] - oo[k]) * ii[k];
  }
  // the interval ahead: [t, tb] up to its macrocell's exit through axis a,
  // of majorant mu (on its way from memory); ahead: there is one
  float t = t0, tb = 0.f, mu = 0.f;
  int a = 0, guard = vc.mdims[0] + vc.mdims[1] + vc.mdims[2];
  bool ahead = false;
  const auto look = [&] {
    ahead = t < t1 && guard > 0;
    if (ahead) {
      a = tnext[0] < tnext[1] ? (tnext[0] < tnext[2] ? 0 : 2) : (tnext[1] < tnext[2] ? 1 : 2);
      tb = minf(pick(a, tnext[0], tnext[1], tnext[2]), t1);
      if (tb > t)
        mu = vc.majorant[((size_t)m[2] * (size_t)vc.mdims[1] + (size_t)m[1]) * (size_t)vc.mdims[0] + (size_t)m[0]];
    }
  };
  look();
  float tau = -flog(1.f - randomFloat(rs));
  float ct = 0.f, cb = 0.f, cmu = 0.f; // the interval of a tentative collision
  bool held = false;
  int steps = 0;
  float dist = kInf;
  for (;;) {
    const bool walks = ahead && !held;
    const unsigned long long w = __builtin_amdgcn_ballot_w64(walks), h = __builtin_amdgcn_ballot_w64(held);
    if ((w | h) == 0ull)
      break;
    if (__popcll(w) > __popcll(h)) {
      if (walks) {
        const float it = t, ib = tb, imu = mu;
        if (tb > t) {
          t = tb;
          cnt.cells++;
        }
        const int sa = pick(a, step[0], step[1], step[2]);
        const int ma = pick(a, m[0], m[1], m[2]) + sa;
        if (ma < 0 || ma >= pick(a, vc.mdims[0], vc.mdims[1], vc.mdims[2]))
          ahead = false;
        else {
          const float tn = (pick(a, vc.origin[0], vc.origin[1], vc.origin[2])
              + (float)(ma + (sa > 0 ? 1 : 0)) * pick(a, msz[0], msz[1], msz[2]) - pick(a, oo[0], oo[1], oo[2]))
              * pick(a, ii[0], ii[1], ii[2]);
          for (int k = 0; k < 3; k++) {
            m[k] = a == k ? ma : m[k];
            tnext[k] = a == k ? tn : tnext[k];
          }
          guard--;
          look();
        }
        if (ib > it && imu > 0.f) {
          const float seg = imu * (ib - it);
          if (tau > seg)
            tau -= seg; // the track leaves the interval
          else {
            held = true;
            ct = it;
            cb = ib;
            cmu = imu;
          }
        }
      }
    } else if (held) {
      ct += tau / cmu; // tentative collision
      const float xi = randomFloat(rs);
      cnt.samples++;
      const vec3f p = o + ct * d;
      const float smp = volumeSample(vc, p);
      bool real = false;
      if (smp == smp) {
        const float u = tfUnit(vc, smp, tfScale);
        const float mu_t = vc.densityScale * tfOpacity(vc, u);
        real = xi < mu_t / cmu;
        if (real)
          albedo = tfColor(vc, u);
      }
      if (real) {
        dist = ct;
        held = ahead = false;
      } else if (++steps >= kMaxDeltaSteps)
        held = ahead = false;
      else {
        tau = -flog(1.f - randomFloat(rs));
        const float seg = cmu * (cb - ct);
        if (tau > seg) {
          tau -= seg;
          held = false;
        }
      }
    }
  }
  return dist;
}

HPT_HD void toVolumeSpace(const DInstance &I, vec3f worg, vec3f wdir, vec3f &o, vec3f &d)
{
  const linear3f rl = {{I.rcp[0], I.rcp[1], I.rcp[2]}, {I.rcp[3], I.rcp[4], I.rcp[5]}, {I.rcp[6], I.rcp[7], I.rcp[8]}};
  o = mul(rl, worg) + v3(I.rcp[9], I.rcp[10], I.rcp[11]);
  d = mul(rl, wdir);
}

// volumeSampleFreePath (VolumeSampler.ispc:96-199) for a ray [t0, tTrace]
// whose surface hit (if any) is at tTrace; [r0, r1] is the clipping
// pass's ray range.  The nearest collision wins and clips the later
// intervals.  Returns its distance (inf: none), pair index and albedo.
__device__ __forceinline__ float volumeFreePath(const DScene &S, vec3f org, vec3f dir, float t0, float tTrace, bool surfaceHit, float r0,
    float r1, RandomSampler &rs, int &pair, vec3f &albedo, VolCount &cnt)
{
  float minDist = kInf;
  float tClip = tTrace;
  bool clipped = surfaceHit;
  pair = -1;
  for (int j = 0; j < S.numVolInsts; j++) {
    const DVolInst vi = S.volInsts[j];
    const DVolume &v = S.volumes[vi.vol];
    vec3f o, d;
    toVolumeSpace(S.instances[vi.inst], org, dir, o, d);
    float lo, hi;
    if (!volumeBox(v, o, d, t0, tTrace, lo, hi))
      continue;
    lo = maxf(0.f, lo);
    if (clipped)
      hi = minf(hi, tClip);
    if (hi < lo)
      continue;
    if (hi < r0 || r1 < lo)
      continue;
    vec3f alb;
    const float dist = deltaTracking(v, o, d, maxf(r0, lo), minf(r1, hi), rs, alb, cnt);
    if (dist < kInf && dist < minDist) {
      minDist = dist;
      pair = j;
      albedo = alb;
      tClip = dist;
      clipped = true;
    }
  }
  return minDist;
}

// volumeTransmittance (VolumeSampler.ispc:201-277): 1 if delta tracking
// passes every volume interval of [t0, t1] (within [r0, r1]), else 0
__device__ __forceinline__ float volumeTransmittance(
    const DScene &S, vec3f org, vec3f dir, float t0, float t1, float r0, float r1, RandomSampler &rs, VolCount &cnt)
{
  float T = 1.f;
  for (int j = 0; j < S.numVolInsts && T > 0.f; j++) {
    const DVolInst vi = S.volInsts[j];
    const DVolume &v = S.volumes[vi.vol];
    vec3f o, d;
    toVolumeSpace(S.instances[vi.inst], org, dir, o, d);
    float lo, hi;
    if (!volumeBox(v, o, d, t0, t1, lo, hi))
      continue;
    if (hi < r0 || r1 < lo)
      continue;
    const float b = minf(r1, hi);
    vec3f alb;
    const float dist = deltaTracking(v, o, d, maxf(r0, lo), b, rs, alb, cnt);
    T = T * (dist < b ? 0.f : 1.f);
  }
  return T;
}

// ---- Henyey-Greenstein (volumes/HenyeyGreenstein.ih:14-77) -------------------------

HPT_HD float hgPhase(float cosTheta, float g)
{
  const float denom = 1.f + g * g - 2.f * g * cosTheta;
  return rcp(4.f * kPi) * (1.f - g * g) * rcp(denom * sqrtf(denom));
}

HPT_HD bool hgIsSmooth(float g) { return !(fabsf(g) > 1.f - 1e-3f); }

// the eval's pdf is the phase function whatever the anisotropy
HPT_HD EvalRes hgEval(float g, vec3f wo, vec3f wi)
{
  const float p = hgPhase(dot(neg(wo), wi), g);
  EvalRes r;
  r.value = v3(p);
  r.pdf = p;
  return r;
}

HPT_HD SampleRes hgSample(float g, vec3f wo, vec2f s)
{
  SampleRes res;
  res.weight = v3(1.f);
  if (!hgIsSmooth(g)) { // a delta function
    res.wi = g > 0 ? neg(wo) : wo;
    res.pdf = kInf;
    res.type = g > 0 ? SPEC_TRANS : SPEC_REFL;
    return res;
  }
  float cosTheta;
  if (fabsf(g) < 1e-3f)
    cosTheta = 1.f - 2.f * s.x;
  else {
    const float sqrTerm = (1.f - g * g) * rcp(1.f - g + 2.f * g * s.x);
    cosTheta = (1.f + g * g - sqrTerm * sqrTerm) * rcp(2.f * g);
  }
  res.type = S_SMOOTH;
  const float sinTheta = sqrtf(maxf(0.f, 1.f - cosTheta * cosTheta));
  const float phi = kTwoPi * s.y;
  res.wi = mul(frame(neg(wo)), cartesian(phi, sinTheta, cosTheta));
  res.pdf = hgPhase(cosTheta, g);
  return res;
}

} // namespace hpt
