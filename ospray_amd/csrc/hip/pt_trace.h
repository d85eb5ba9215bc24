// BVH traversal and ray/primitive tests of the hip path tracer (device).
//
// The reference hands these to Embree (rtcIntersectV,
// modules/cpu/common/World.ih:29-52, 247-286).  Here:
//   * two-level 4-wide BVH (TLAS over instances, one BLAS per group) in
//     64-byte nodes holding four child boxes; one lane per ray, children
//     visited nearest first, speculative while-while order (Aila and Laine,
//     "Understanding the efficiency of ray traversal on GPUs", 2009): a
//     lane holds a leaf it reaches and goes on with inner nodes until no
//     more lanes of the wave look for one than hold one;
//   * the traversal stack lives in LDS (LDS_DEPTH entries per lane, laid out
//     [depth][lane] so lanes hit distinct banks) and spills to a per-thread
//     global overflow row beyond that;
//   * triangles: watertight test (Woop, Benthin, Wald 2013) in float: an
//     edge function depends on the edge's two vertices only and is exactly
//     antisymmetric between the two triangles sharing the edge, so a ray
//     never passes between them; quads as two triangles (v0,v1,v3) and
//     (v2,v3,v1); spheres: Intersect.ih:29-80;
//   * closest hit = smallest t in (t0, tfar]; exact ties resolved by the
//     smallest (instance, model, primitive, half), so results do not depend
//     on BVH layout;
//   * near-ties of extension rays (TIES): when another hit's float t lies
//     within kTieEps (relative) of the closest one, a second traversal over
//     that window re-resolves the hit in FP64: every hit in the window gets
//     its distance recomputed in double precision from the world ray
//     (object ray formed in double from the instance's inverse transform)
//     and the float vertices, and the smallest (FP64 t, key) wins.  The
//     flag that triggers it is independent of traversal order: a hit is
//     compared with the current closest on arrival, hits up to kTieEps
//     beyond it are still tested, and the flag clears only when a hit
//     closer than the window's lower end arrives;
//   * node boxes only cull, conservatively (nodeNear).
#pragma once

#include "pt_math.h"
#include "pt_types.h"

namespace hpt {

constexpr int kTraceBlock = 128;
constexpr int kLdsDepth = 24;
constexpr int kOverflowDepth = 112;
// Entries a world may need by the builders' count: one less than its children
// for each node on the way down, and the two of an instance's entry.  The rows
// hold more: a ray that enters an unused slot of a node (k_place) pushes
// that too, up to three entries beyond the count in the BLAS and in the TLAS
// each, since only a node without inner children has unused slots; and one row
// holds the sentinel.  (A multiple of four, so that the recorded hits stay
// 16-byte aligned.)
constexpr int kStackCapacity = 128;
constexpr int kUnusedSlots = 6;
static_assert(kStackCapacity + kUnusedSlots + 1 <= kLdsDepth + kOverflowDepth && kOverflowDepth % 4 == 0, "stack rows");
// transparent hits an occlusion traversal records for the transparency pass
constexpr int kTransRecHits = 4;
// words of scratch per resident traversal thread: the stack overflow, then
// kTransRecHits recorded hits of 4 words (one float4, 16-byte aligned),
// then their count (padded to 4 words)
constexpr int kThreadRow = kOverflowDepth + 4 * kTransRecHits + 4;
constexpr int32_t kMarker = 0x7fffffff;

struct Hit
{
  float t, u, v;
  vec3f Ng;
  uint32_t inst, model, prim, half;
  bool hit;
};

HPT_HD bool keyLess(uint32_t i0, uint32_t m0, uint32_t p0, uint32_t h0, const Hit &b)
{
  if (i0 != b.inst)
    return i0 < b.inst;
  if (m0 != b.model)
    return m0 < b.model;
  if (p0 != b.prim)
    return p0 < b.prim;
  return h0 < b.half;
}

HPT_HD bool better(float t, uint32_t i, uint32_t m, uint32_t p, uint32_t h, const Hit &b)
{
  return !b.hit || t < b.t || (t == b.t && keyLess(i, m, p, h, b));
}

// reciprocal of a direction component for the box tests, good to 1 ulp
__device__ __forceinline__ float boxInv(float d)
{
  const float ad = fabsf(d);
  return __builtin_amdgcn_rcpf(ad < 1e-18f ? copysignf(1e-18f, d) : d);
}

// The shear of the watertight test along the ray's largest axis kz, with
// the other two axes in cyclic order.  (Exchanging them for a negative
// direction, as the paper does, negates U, V, W and their sum exactly and
// with them nothing of t, u, v: the sign tests are symmetric.)
struct TriPre
{
  int kz;
  float Sx, Sy, Sz;
};

// component kz of a and the two after it
HPT_HD void rotateTo(int kz, vec3f a, float &x, float &y, float &z)
{
  x = kz == 0 ? a.y : (kz == 1 ? a.z : a.x);
  y = kz == 0 ? a.z : (kz == 1 ? a.x : a.y);
  z = kz == 0 ? a.x : (kz == 1 ? a.y : a.z);
}

HPT_HD TriPre triPrecompute(vec3f dir)
{
  TriPre p;
  const vec3f ad = vabs(dir);
  p.kz = ad.x > ad.y ? (ad.x > ad.z ? 0 : 2) : (ad.y > ad.z ? 1 : 2);
  float dx, dy, dz;
  rotateTo(p.kz, dir, dx, dy, dz);
  p.Sx = dx / dz;
  p.Sy = dy / dz;
  p.Sz = 1.0f / dz;
  return p;
}

HPT_HD bool intersectTriangle(vec3f org, float t0, const TriPre &pc, vec3f v0, vec3f v1, vec3f v2, float tmax,
    float &t, float &u, float &v)
{
  float Ax_, Ay_, Az_, Bx_, By_, Bz_, Cx_, Cy_, Cz_;
  rotateTo(pc.kz, v0 - org, Ax_, Ay_, Az_);
  rotateTo(pc.kz, v1 - org, Bx_, By_, Bz_);
  rotateTo(pc.kz, v2 - org, Cx_, Cy_, Cz_);
  const float Ax = Ax_ - pc.Sx * Az_;
  const float Ay = Ay_ - pc.Sy * Az_;
  const float Bx = Bx_ - pc.Sx * Bz_;
  const float By = By_ - pc.Sy * Bz_;
  const float Cx = Cx_ - pc.Sx * Cz_;
  const float Cy = Cy_ - pc.Sy * Cz_;
  const float U = Cx * By - Cy * Bx;
  const float V = Ax * Cy - Ay * Cx;
  const float W = Bx * Ay - By * Ax;
  if ((U < 0.0f || V < 0.0f || W < 0.0f) && (U > 0.0f || V > 0.0f || W > 0.0f))
    return false;
  const float det = U + V + W;
  if (det == 0.0f)
    return false;
  const float Az = pc.Sz * Az_;
  const float Bz = pc.Sz * Bz_;
  const float Cz = pc.Sz * Cz_;
  const float T = U * Az + V * Bz + W * Cz;
  const float rcpDet = 1.0f / det;
  const float tt = T * rcpDet;
  if (!(tt > t0) || !(tt <= tmax))
    return false;
  t = tt;
  u = V * rcpDet;
  v = W * rcpDet;
  return true;
}

// both roots of the ray/sphere test, with the arithmetic of
// intersectSphere: bit 0 = entry (tE, NE) in (t0, tmax], bit 1 = exit
HPT_HD int sphereRoots(vec3f org, vec3f d, float t0, vec3f center, float radius, float tmax, float &tE, vec3f &NE,
    float &tX, vec3f &NX)
{
  const float rd2 = 1.0f / dot(d, d);
  const vec3f CO = center - org;
  const float projCO = dot(CO, d) * rd2;
  const vec3f perp = CO - projCO * d;
  const float l2 = dot(perp, perp);
  const float r2 = radius * radius;
  if (l2 > r2)
    return 0;
  const float td = sqrtf((r2 - l2) * rd2);
  tE = projCO - td;
  tX = projCO + td;
  NE = (-td) * d - perp;
  NX = td * d - perp;
  return (tE > t0 && tE <= tmax ? 1 : 0) | (tX > t0 && tX <= tmax ? 2 : 0);
}

HPT_HD bool intersectSphere(vec3f org, vec3f d, float t0, vec3f center, float radius, float tmax, float &t, vec3f &N)
{
  const float rd2 = 1.0f / dot(d, d);
  const vec3f CO = center - org;
  const float projCO = dot(CO, d) * rd2;
  const vec3f perp = CO - projCO * d;
  const float l2 = dot(perp, perp);
  const float r2 = radius * radius;
  if (l2 > r2)
    return false;
  const float td = sqrtf((r2 - l2) * rd2);
  const float tEntry = projCO - td;
  const float tExit = projCO + td;
  if (tEntry > t0 && tEntry <= tmax) {
    t = tEntry;
    N = (-td) * d - perp;
    return true;
  }
  if (tExit > t0 && tExit <= tmax) {
    t = tExit;
    N = td * d - perp;
    return true;
  }
  return false;
}

struct TraceStats
{
  uint32_t nodes, prims;
};

// relative window of float distances within which two extension-ray hits
// count as a near-tie (64 ulp at 1.0 is 7.6e-6; the float t of the
// watertight test is good to a few ulp away from grazing incidence)
constexpr float kTieEps = 1.0e-5f;
// lower end of the boxes the FP64 re-resolution opens, relative to the
// float closest hit
constexpr float kTieBoxLow = 0.9f;

HPT_HD bool nearTie(float t, float tBest) { return fabsf(t - tBest) <= kTieEps * tBest; }

// FP64 distance along the world ray (worg + t wdir) to the plane of
// triangle (a, b, c) of instance rcp (inverse transform, columns vx, vy,
// vz, p): the object ray is formed in double from the float world ray and
// the float transform, the plane from the float vertices
HPT_HD void fp64ObjectRay(const float *rcp, vec3f worg, vec3f wdir, double o[3], double d[3])
{
  const double wo[3] = {worg.x, worg.y, worg.z}, wd[3] = {wdir.x, wdir.y, wdir.z};
  for (int r = 0; r < 3; r++) {
    o[r] = (double)rcp[r] * wo[0] + (double)rcp[3 + r] * wo[1] + (double)rcp[6 + r] * wo[2] + (double)rcp[9 + r];
    d[r] = (double)rcp[r] * wd[0] + (double)rcp[3 + r] * wd[1] + (double)rcp[6 + r] * wd[2];
  }
}

HPT_HD double fp64TriangleT(const double o[3], const double d[3], vec3f a, vec3f b, vec3f c)
{
  const double e1[3] = {(double)b.x - a.x, (double)b.y - a.y, (double)b.z - a.z};
  const double e2[3] = {(double)c.x - a.x, (double)c.y - a.y, (double)c.z - a.z};
  const double n[3] = {e1[1] * e2[2] - e1[2] * e2[1], e1[2] * e2[0] - e1[0] * e2[2], e1[0] * e2[1] - e1[1] * e2[0]};
  const double ao[3] = {(double)a.x - o[0], (double)a.y - o[1], (double)a.z - o[2]};
  const double num = ao[0] * n[0] + ao[1] * n[1] + ao[2] * n[2];
  const double den = d[0] * n[0] + d[1] * n[1] + d[2] * n[2];
  return num / den;
}

// FP64 entry (exitRoot 0) or exit (1) distance of a sphere
HPT_HD double fp64SphereT(const double o[3], const double d[3], vec3f center, float radius, int exitRoot)
{
  const double oc[3] = {o[0] - center.x, o[1] - center.y, o[2] - center.z};
  const double A = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
  const double B = oc[0] * d[0] + oc[1] * d[1] + oc[2] * d[2];
  const double C = oc[0] * oc[0] + oc[1] * oc[1] + oc[2] * oc[2] - (double)radius * (double)radius;
  const double disc = B * B - A * C;
  const double sq = disc > 0.0 ? sqrt(disc) : 0.0;
  return (exitRoot ? (-B + sq) : (-B - sq)) / A;
}

// one 4-wide node as its four 16-byte loads (DNode4)
struct Node4
{
  float4 a, b; // p, s.x | s.y, s.z, lox, hix
  uint4 c;     // loy, hiy, loz, hiz
  int4 child;
};

// What the box test needs of a ray: its origin and 1 / d per axis
struct BoxRay
{
  vec3f o, inv;
};

__device__ __forceinline__ BoxRay boxRay(vec3f o, vec3f d) { return {o, v3(boxInv(d.x), boxInv(d.y), boxInv(d.z))}; }

// 12 u, u = 2^-24, of the distance to a node's first plane (see nodeNear)
constexpr float kBoxPad = 7.15255737e-7f;

__device__ __forceinline__ Node4 loadNode(const DNode4 *nodes, int idx)
{
  const float4 *np = reinterpret_cast<const float4 *>(nodes + idx);
  Node4 n;
  n.a = np[0];
  n.b = np[1];
  n.c = reinterpret_cast<const uint4 *>(np)[2];
  n.child = reinterpret_cast<const int4 *>(np)[3];
  return n;
}

// order (t, child) pairs by t
__device__ __forceinline__ void cswap(float &ta, int &ca, float &tb, int &cb)
{
  const bool sw = tb < ta;
  const float t = sw ? tb : ta;
  const int c = sw ? cb : ca;
  tb = sw ? ta : tb;
  cb = sw ? ca : cb;
  ta = t;
  ca = c;
}

// one axis of a node for a ray: plane q is entered at q * a + near (from
// the byte of `first`) and left at q * a + far (`last`)
struct NodeAxis
{
  float a, near, far;
  uint32_t first, last;
};

__device__ __forceinline__ NodeAxis nodeAxis(float p, float s, uint32_t lo, uint32_t hi, float o, float inv)
{
  NodeAxis x;
  const float m = (p - o) * inv;
  x.a = s * inv;
  x.near = fmaf(-kBoxPad, fabsf(m), m);
  x.far = fmaf(kBoxPad, fabsf(m), m);
  const bool back = inv < 0.f;
  x.first = back ? hi : lo;
  x.last = back ? lo : hi;
  return x;
}

// Entry distances t[c] of the four children's boxes over [t0, tb], +inf for
// a box the ray misses.
//
// Conservative: with u = 2^-24, M = (p - o) / d and Q = q s / d, the distance
// M + Q of plane q comes out off by at most 6 u |M| + 4 u |Q|: p - o, 1 / d (1
// ulp, 2 u), their product, the padding's and the last sum on M, 1 / d, s / d
// and the last sum on Q.  The near planes are moved down and the far ones up
// by 12 u |M| here and by 10 u of the node's size over |d| in the grid itself
// (k_place), which leaves 6 u of both for a primitive's own hit distance,
// so the closest hit does not depend on the tree.  Neither padding looks
// further than the node and the ray's origin: culling next to an object does
// not depend on what else is in the tree, nor on where the origin of the
// coordinates lies.  (Padded by the tree's largest coordinate, one instance at
// 1e6 widened every box of the world by 0.6.)  A NaN (overflow) leaves the
// axis out of the test.  The near plane of an axis is picked once for the four
// children, a word at a time: a minimum or maximum costs 4.3 cycles of a SIMD,
// a select or FMA 2.6 (measured).
__device__ __forceinline__ void nodeNear(const Node4 &n, const BoxRay &r, float t0, float tb, float t[4])
{
  const NodeAxis x = nodeAxis(n.a.x, n.a.w, __float_as_uint(n.b.z), __float_as_uint(n.b.w), r.o.x, r.inv.x);
  const NodeAxis y = nodeAxis(n.a.y, n.b.x, n.c.x, n.c.y, r.o.y, r.inv.y);
  const NodeAxis z = nodeAxis(n.a.z, n.b.y, n.c.z, n.c.w, r.o.z, r.inv.z);
#pragma unroll
  for (int c = 0; c < 4; c++) {
    auto q = [c](uint32_t w) { return (float)((w >> (8 * c)) & 0xffu); };
    const float tn = fmaxf(fmaxf(fmaf(q(x.first), x.a, x.near), fmaf(q(y.first), y.a, y.near)),
        fmaxf(fmaf(q(z.first), z.a, z.near), t0));
    const float tf = fminf(fminf(fmaf(q(x.last), x.a, x.far), fmaf(q(y.last), y.a, y.far)),
        fminf(fmaf(q(z.last), z.a, z.far), tb));
    t[c] = tn <= tf ? tn : kInf;
  }
}

// Traversal modes: MODE_CLOSEST returns the closest hit; MODE_OCCLUSION
// returns as soon as a primitive of an opaque model is hit and otherwise
// reports in `sawTransparent` whether any (non-opaque) primitive was hit.
// With RECORD, an occlusion traversal also records every hit of a
// non-opaque primitive in (t0, tfar] (both roots of a sphere) in the
// thread's scratch row after the stack overflow (recordedHits): one float4
// (t, instance, index into S.prims, root: 1 = a sphere's exit) per hit, up
// to kTransRecHits, and in the word after them the count of all of them,
// also those beyond the capacity (0 when the traversal starts: the caller
// resets it after each ray that recorded hits; it lives in memory rather
// than a register since transparent hits are rare).
// hitFromRecord rebuilds the closest-hit record of one of them.

__device__ __forceinline__ float4 *recordedHits(uint32_t *ovf)
{
  return reinterpret_cast<float4 *>(ovf + kOverflowDepth);
}

__device__ __forceinline__ uint32_t *recordedCount(uint32_t *ovf)
{
  return ovf + kOverflowDepth + 4 * kTransRecHits;
}

__device__ __forceinline__ void recordHit(uint32_t *ovf, float t, uint32_t inst, uint32_t primIndex, uint32_t exitRoot)
{
  uint32_t *cnt = recordedCount(ovf);
  const uint32_t c = *cnt;
  if (c < (uint32_t)kTransRecHits)
    recordedHits(ovf)[c] = make_float4(t, __uint_as_float(inst), __uint_as_float(primIndex), __uint_as_float(exitRoot));
  *cnt = c + 1;
}
enum TraceMode
{
  MODE_CLOSEST = 0,
  MODE_OCCLUSION = 1
};

// Second traversal of a ray whose closest hit `best` has a near-tie: every
// hit whose float t is a near-tie of best.t gets its FP64 distance, and the
// smallest (FP64 t, key) becomes `best` (with its float hit record).  A
// plain stack traversal: the result is a minimum over a set, so the visit
// order does not matter.  Boxes are opened over [tLo, tHi]: every hit of
// the set has a float t within 1e-5 of tF, and tLo = 0.9 tF leaves a
// margin far above the float error of a hit distance, so only the boxes
// around the hit point are visited (the descent to it, not every box the
// ray crosses before it).
template <bool STATS>
__device__ void resolveNearTie(const DScene &S, vec3f worg, vec3f wdir, float t0, float tfar, Hit &best,
    uint32_t *lds, uint32_t *ovf, TraceStats &st)
{
  const int lane = threadIdx.x;
  const float tF = best.t;
  const float tHi = fminf(tF + kTieEps * tF, tfar);
  const float tLo = fmaxf(t0, kTieBoxLow * tF);
  const BoxRay wbox = boxRay(worg, wdir);
  Hit w = best;
  double wD = 0.0;
  bool have = false;
  int sp = 0;
  auto push = [&](int v) {
    if (sp < kLdsDepth)
      lds[sp * kTraceBlock + lane] = (uint32_t)v;
    else
      ovf[sp - kLdsDepth] = (uint32_t)v;
    sp++;
  };
  auto pop = [&]() -> int {
    sp--;
    if (sp < kLdsDepth)
      return (int)lds[sp * kTraceBlock + lane];
    return (int)ovf[sp - kLdsDepth];
  };
  // children of node `cur` whose boxes the ray enters in (t0, tHi]
  auto expand = [&](int cur, const BoxRay &r) -> bool {
    const Node4 nd = loadNode(S.nodes, cur);
    if (STATS)
      st.nodes++;
    float tc[4];
    nodeNear(nd, r, tLo, tHi, tc);
    const int ch[4] = {nd.child.x, nd.child.y, nd.child.z, nd.child.w};
    for (int c = 0; c < 4; c++)
      if (tc[c] != kInf) {
        if (sp >= kLdsDepth + kOverflowDepth) // cannot happen: the world commit checks the stack need (kStackCapacity)
          return false;
        push(ch[c]);
      }
    return true;
  };
  push(S.tlasRoot);
  while (sp > 0) {
    const int cur = pop();
    if (cur >= 0) {
      if (!expand(cur, wbox))
        return;
      continue;
    }
    const uint32_t inst = ~(uint32_t)cur >> 3; // world leaf: one instance
    const DInstance &I = S.instances[inst];
    const linear3f rl = {{I.rcp[0], I.rcp[1], I.rcp[2]}, {I.rcp[3], I.rcp[4], I.rcp[5]}, {I.rcp[6], I.rcp[7], I.rcp[8]}};
    const vec3f o = mul(rl, worg) + v3(I.rcp[9], I.rcp[10], I.rcp[11]);
    const vec3f d = mul(rl, wdir);
    const BoxRay box = boxRay(o, d);
    const TriPre pc = triPrecompute(d);
    double od[3], dd[3];
    fp64ObjectRay(I.rcp, worg, wdir, od, dd);
    const int base = sp;
    push(I.blasRoot);
    while (sp > base) {
      const int c = pop();
      if (c >= 0) {
        if (!expand(c, box))
          return;
        continue;
      }
      const uint32_t enc = ~(uint32_t)c;
      const uint32_t first = enc >> 3, count = (enc & 7u) + 1u;
      for (uint32_t k = 0; k < count; k++) {
        const DPrim &P = S.prims[first + k];
        const float4 pa = reinterpret_cast<const float4 *>(&P)[0];
        const float4 pb = reinterpret_cast<const float4 *>(&P)[1];
        const float4 pcv = reinterpret_cast<const float4 *>(&P)[2];
        const uint32_t primID = __float_as_uint(pa.w);
        const uint32_t mk = __float_as_uint(pb.w);
        const uint32_t model = mk & 0x0fffffffu, kind = mk >> 28;
        if (STATS)
          st.prims++;
        float t, u = 0.f, v = 0.f;
        vec3f Ng;
        uint32_t half = 0;
        double tD;
        if (kind == PRIM_SPHERE) {
          float tE, tX;
          vec3f NE, NX;
          const int roots = sphereRoots(o, d, t0, v3(pa.x, pa.y, pa.z), pb.x, tHi, tE, NE, tX, NX);
          if (!roots)
            continue;
          const int exitRoot = (roots & 1) ? 0 : 1;
          t = exitRoot ? tX : tE;
          Ng = exitRoot ? NX : NE;
          if (!nearTie(t, tF))
            continue;
          tD = fp64SphereT(od, dd, v3(pa.x, pa.y, pa.z), pb.x, exitRoot);
        } else {
          const vec3f A = v3(pa.x, pa.y, pa.z), B = v3(pb.x, pb.y, pb.z), C = v3(pcv.x, pcv.y, pcv.z);
          if (!intersectTriangle(o, t0, pc, A, B, C, tHi, t, u, v) || !nearTie(t, tF))
            continue;
          Ng = cross(B - A, C - A);
          if (kind == PRIM_QUAD1) {
            half = 1;
            u = 1.0f - u;
            v = 1.0f - v;
          }
          tD = fp64TriangleT(od, dd, A, B, C);
        }
        if (!have || tD < wD || (tD == wD && keyLess(inst, model, primID, half, w))) {
          have = true;
          wD = tD;
          w.hit = true;
          w.t = t;
          w.u = u;
          w.v = v;
          w.Ng = Ng;
          w.inst = inst;
          w.model = model;
          w.prim = primID;
          w.half = half;
        }
      }
    }
  }
  if (have)
    best = w;
}

// near-tie handling of a closest-hit traversal (see the header comment):
// off; re-resolved in FP64 at the end of the traversal; or only reported
// (in sawTransparent, unused by closest-hit traversals otherwise) for a
// later pass to re-resolve with resolveNearTie, which keeps the FP64 code
// and its registers out of the traversal kernel
constexpr int TIES_OFF = 0, TIES_RESOLVE = 1, TIES_REPORT = 2;

// The closest hit as a traversal keeps it: what depends on the primitive
// alone (model, ids, normal) is read again from its record once the ray has
// ended (hitFromTrace), so an update in the leaf loop is five moves.
struct TraceHit
{
  float t, u, v;  // u, v of the record's own triangle
  uint32_t inst;
  uint32_t prim; // index into DScene::prims, kInvalidID: no hit
};

// Per-lane state of one traversal.  A traversal runs as rounds of
// traceDescend (inner nodes, speculative while-while) and traceLeaf (the
// leaf the lane holds); traceRay runs one ray to its end, traceQueue (in
// the kernels) keeps the lanes of a wave busy with rays from a queue.
struct TraceState
{
  vec3f worg, wdir; // the world ray
  BoxRay box;       // of the current (world or object) ray
  TriPre pc;
  float t0, tfar;
  float tb; // hits beyond it are of no interest: the closest one (with TIES, a near-tie beyond it)
  int inst, cur, post;
  int modelOffset;     // MODE_OCCLUSION: the instance's first model, -1 if all are opaque
  int sp; // see stackAt
  bool tie;            // a near-tie of the current closest hit has been seen (TIES != TIES_OFF)
  bool sawTransparent; // MODE_OCCLUSION: a non-opaque primitive was hit
};

// `cur` of a lane whose traversal has no node left
constexpr int kTraceDone = 0x7ffffffe;

__device__ __forceinline__ void traceBegin(
    TraceState &s, const DScene &S, vec3f worg, vec3f wdir, float t0, float tfar, TraceHit &best, uint32_t *lds)
{
  best.t = tfar;
  best.u = best.v = 0.f;
  best.inst = best.prim = kInvalidID;
  s.worg = worg;
  s.wdir = wdir;
  s.box = boxRay(worg, wdir);
  s.pc = {0, 0.f, 0.f, 0.f};
  s.t0 = t0;
  s.tfar = tfar;
  s.tb = tfar;
  s.inst = -1;
  s.modelOffset = -1;
  lds[threadIdx.x] = (uint32_t)kTraceDone;
  s.sp = 4 * ((int)threadIdx.x + kTraceBlock); // entry 1 (kStackRow)
  s.cur = S.tlasRoot;
  s.post = 0;
  s.tie = false;
  s.sawTransparent = false;
}

// The stack of a lane: s.sp is the byte offset in the block's LDS rows of
// the next free entry (row d of lane l at d * kStackRow + 4 l), entries from
// row kLdsDepth on live in the overflow row.  Entry 0 is kTraceDone, so a
// pop needs no test for an empty stack.
constexpr int kStackRow = 4 * kTraceBlock;
constexpr int kStackLds = kLdsDepth * kStackRow;

__device__ __forceinline__ uint32_t *stackAt(uint32_t *lds, int sp)
{
  return reinterpret_cast<uint32_t *>(reinterpret_cast<char *>(lds) + sp);
}

// the entry's word in the overflow row (sp >= kStackLds)
__device__ __forceinline__ uint32_t *overflowAt(uint32_t *ovf, int sp) { return ovf + (sp / kStackRow - kLdsDepth); }

// callers check that the stack holds another entry
__device__ __forceinline__ void tracePush(TraceState &s, uint32_t *lds, uint32_t *ovf, int v)
{
  if (s.sp < kStackLds)
    *stackAt(lds, s.sp) = (uint32_t)v;
  else
    *overflowAt(ovf, s.sp) = (uint32_t)v;
  s.sp += kStackRow;
}

// the LDS read is unconditional (a clamped row), the overflow row is read
// only by the rare lanes whose stack is deeper than kLdsDepth (a volatile
// read, so the compiler keeps the two reads apart instead of merging them
// into one generic-address load)
__device__ __forceinline__ int tracePop(TraceState &s, uint32_t *lds, uint32_t *ovf)
{
  s.sp -= kStackRow;
  int v = (int)*stackAt(lds, s.sp < kStackLds ? s.sp : 4 * (int)threadIdx.x);
  if (s.sp >= kStackLds)
    v = (int)*reinterpret_cast<const volatile uint32_t *>(overflowAt(ovf, s.sp));
  return v;
}

// the lanes of the wave for which x holds (__ballot takes an int, which
// costs two more vector instructions)
__device__ __forceinline__ unsigned long long waveMask(bool x) { return __builtin_amdgcn_ballot_w64(x); }

// a lane that needs traceLeaf: it holds a leaf or stands at the exit of an
// instance
__device__ __forceinline__ bool traceHolds(const TraceState &s) { return s.post != 0 || s.cur == kMarker; }

// Inner nodes of the speculative while-while traversal: a lane that reaches
// a leaf keeps it aside (post) and goes on with inner nodes until at most
// as many lanes still look for a leaf as hold one.  Waiting for the last
// lane ran 10.8 node steps per call with 18.5 of 64 lanes active on the
// 1080p terrain (88 % of the traversal's instructions), since a lane that
// meets its second leaf stands still; leaving as soon as half have one
// trades some fuller leaf rounds for that.  1920x1080, 4 spp, whole frames:
// 26.4 -> 23.9 ms.  (Ratios of searching to holding lanes 1/4, 1/2, 2/3, 1,
// 3/2, 2, 4, without the maps: 25.2, 24.7, 24.7, 24.8, 25.1, 25.4, 26.6.)
// Never later than that, so a wave with few rays goes on as before.  The exit
// of an instance (its marker) stops a lane too: traceLeaf gives it the world
// ray back.  A held instance leaf is entered from the world level, with the
// next world node pushed below the marker.  Lanes with cur == kTraceDone and
// no held leaf (finished or idle) only take part in the wave vote.
template <int MODE, bool STATS>
__device__ __forceinline__ void traceDescend(
    TraceState &s, const DScene &S, uint32_t *lds, uint32_t *ovf, TraceStats &st)
{
  for (;;) {
    if ((uint32_t)s.cur < (uint32_t)kTraceDone) {
      const Node4 nd = loadNode(S.nodes, s.cur);
      if (STATS)
        st.nodes++;
      float tc[4];
      nodeNear(nd, s.box, MODE == MODE_OCCLUSION ? 0.f : s.t0, s.tb, tc); // shadow rays start at 0
      float t0c = tc[0], t1c = tc[1], t2c = tc[2], t3c = tc[3];
      int c0 = nd.child.x, c1 = nd.child.y, c2 = nd.child.z, c3 = nd.child.w;
      cswap(t0c, c0, t1c, c1);
      cswap(t2c, c2, t3c, c3);
      cswap(t0c, c0, t2c, c2);
      cswap(t1c, c1, t3c, c3);
      cswap(t1c, c1, t2c, c2);
      if (t0c == kInf) {
        s.cur = tracePop(s, lds, ovf);
      } else {
        const bool h1 = t1c != kInf, h2 = t2c != kInf, h3 = t3c != kInf;
        const int grow = h3 ? 3 * kStackRow : (h2 ? 2 * kStackRow : (h1 ? kStackRow : 0));
        if (s.sp < kStackLds - 2 * kStackRow) {
          // the children after the nearest, farthest first: the sorted
          // boxes that were hit are a prefix, so the entries pushed are the
          // last child hit .. c1; the rows above them get don't-care copies
          uint32_t *top = stackAt(lds, s.sp);
          top[0] = (uint32_t)(h3 ? c3 : (h2 ? c2 : c1));
          top[kTraceBlock] = (uint32_t)(h3 ? c2 : c1);
          top[2 * kTraceBlock] = (uint32_t)c1;
          s.sp += grow;
          s.cur = c0;
        } else if (s.sp + grow >= (kLdsDepth + kOverflowDepth + 1) * kStackRow) { // cannot happen, as above
          s.cur = kTraceDone;
        } else {
          if (h3)
            tracePush(s, lds, ovf, c3);
          if (h2)
            tracePush(s, lds, ovf, c2);
          if (h1)
            tracePush(s, lds, ovf, c1);
          s.cur = c0;
        }
      }
    }
    if (s.cur < 0 && s.post == 0) { // hold the leaf, go on
      s.post = s.cur;
      s.cur = tracePop(s, lds, ovf);
    }
    const unsigned long long holding = waveMask(s.post != 0) | waveMask(s.cur == kMarker);
    const unsigned long long stepping = waveMask((uint32_t)s.cur < (uint32_t)kTraceDone);
    if (__builtin_popcountll(stepping & ~holding) <= __builtin_popcountll(holding))
      break;
  }
}

__device__ __forceinline__ void objectRay(const DInstance &I, vec3f worg, vec3f wdir, vec3f &o, vec3f &d)
{
  const linear3f rl = {{I.rcp[0], I.rcp[1], I.rcp[2]}, {I.rcp[3], I.rcp[4], I.rcp[5]}, {I.rcp[6], I.rcp[7], I.rcp[8]}};
  o = mul(rl, worg) + v3(I.rcp[9], I.rcp[10], I.rcp[11]);
  d = mul(rl, wdir);
}

// model, primitive and half of a record
__device__ __forceinline__ void primKey(const DScene &S, uint32_t index, uint32_t &model, uint32_t &prim, uint32_t &half)
{
  const DPrim &P = S.prims[index];
  model = P.modelKind & 0x0fffffffu;
  prim = P.primID;
  half = (P.modelKind >> 28) == PRIM_QUAD1 ? 1u : 0u;
}

// the order of two hits at the same distance (rare: kept out of line)
__device__ __forceinline__ bool primLess(const DScene &S, uint32_t inst, uint32_t prim, const TraceHit &best)
{
  Hit b;
  uint32_t m, p, h;
  primKey(S, prim, m, p, h);
  primKey(S, best.prim, b.model, b.prim, b.half);
  b.inst = best.inst;
  return keyLess(inst, m, p, h, b);
}

// the hit record of a traversal's result: the same primitive test on the
// same object ray gives a sphere's normal bit for bit
__device__ __forceinline__ Hit hitFromTrace(const DScene &S, vec3f worg, vec3f wdir, float t0, const TraceHit &b)
{
  Hit h;
  h.hit = b.prim != kInvalidID;
  h.t = b.t;
  h.u = b.u;
  h.v = b.v;
  h.Ng = v3(0.f);
  h.inst = h.model = h.prim = kInvalidID;
  h.half = 0;
  if (h.hit) {
    const float4 *P = reinterpret_cast<const float4 *>(S.prims + b.prim);
    const float4 pa = P[0], pb = P[1], pc = P[2];
    const uint32_t mk = __float_as_uint(pb.w), kind = mk >> 28;
    const vec3f A = v3(pa.x, pa.y, pa.z);
    h.inst = b.inst;
    h.model = mk & 0x0fffffffu;
    h.prim = __float_as_uint(pa.w);
    if (kind == PRIM_SPHERE) {
      vec3f o, d;
      objectRay(S.instances[b.inst], worg, wdir, o, d);
      intersectSphere(o, d, t0, A, pb.x, b.t, h.t, h.Ng);
    } else {
      h.Ng = cross(v3(pb.x, pb.y, pb.z) - A, v3(pc.x, pc.y, pc.z) - A);
      if (kind == PRIM_QUAD1) {
        h.half = 1;
        h.u = 1.0f - h.u;
        h.v = 1.0f - h.v;
      }
    }
  }
  return h;
}

// The words of a primitive record the test needs, each a register of its
// own (held as the loaded quads they would be allocated, and spilled, four
// at a time).
struct PrimWords
{
  vec3f A, B, C;
  uint32_t mk;
};

__device__ __forceinline__ PrimWords primWords(float4 a, float4 b, float4 c)
{
  return {v3(a.x, a.y, a.z), v3(b.x, b.y, b.z), v3(c.x, c.y, c.z), __float_as_uint(b.w)};
}

// One primitive record (index k) of the current instance.
// Returns true for an opaque occluder (MODE_OCCLUSION).
template <int MODE, bool RECORD, int TIES>
__device__ __forceinline__ bool tracePrim(
    TraceState &s, const DScene &S, TraceHit &best, const PrimWords &w, uint32_t k, uint32_t *ovf)
{
  const uint32_t mk = w.mk;
  float t, u = 0.f, v = 0.f, tX = 0.f;
  int roots = 1;
  if (mk >> 28 != PRIM_SPHERE) {
    if (!intersectTriangle(s.box.o, MODE == MODE_OCCLUSION ? 0.f : s.t0, s.pc, w.A, w.B, w.C, s.tb, t, u, v))
      return false;
  } else {
    // the object direction again, rather than three registers held for it
    vec3f o, d, NE, NX;
    objectRay(S.instances[s.inst], s.worg, s.wdir, o, d);
    roots = sphereRoots(o, d, MODE == MODE_OCCLUSION ? 0.f : s.t0, w.A, w.B.x, s.tb, t, NE, tX, NX);
    if (roots == 0)
      return false;
    if (MODE == MODE_CLOSEST && !(roots & 1))
      t = tX;
  }
  if (MODE == MODE_OCCLUSION) {
    if (s.modelOffset < 0 || S.models[s.modelOffset + (int)(mk & 0x0fffffffu)].opaque)
      return true;
    s.sawTransparent = true;
    if (RECORD) {
      if (roots & 1)
        recordHit(ovf, t, (uint32_t)s.inst, k, 0);
      if (roots & 2)
        recordHit(ovf, tX, (uint32_t)s.inst, k, 1);
    }
    return false;
  }
  const bool any = best.prim != kInvalidID;
  const bool nt = TIES != TIES_OFF && any && nearTie(t, best.t);
  // t <= tfar: without a hit yet every hit is the closest
  if (!any || t < best.t || (t == best.t && primLess(S, (uint32_t)s.inst, k, best))) {
    if (TIES != TIES_OFF)
      s.tie = nt; // a hit below the window of the previous closest one clears the flag
    // (the reporting traversal's rays have no far end)
    s.tb = TIES == TIES_OFF ? t : (TIES == TIES_REPORT ? t + kTieEps * t : fminf(t + kTieEps * t, s.tfar));
    best.t = t;
    best.u = u;
    best.v = v;
    best.inst = (uint32_t)s.inst;
    best.prim = k;
  } else if (nt) {
    s.tie = true;
  }
  return false;
}

// What a lane holds (traceHolds): an instance leaf enters the instance's
// BLAS with the object ray; a BLAS leaf tests its primitives; the marker
// leaves the instance.  Returns true when the lane's traversal has ended: no node left, an
// opaque occluder (MODE_OCCLUSION, `occluded` set) or a full stack.
template <int MODE, bool STATS, bool RECORD, int TIES>
__device__ __forceinline__ bool traceLeaf(TraceState &s, const DScene &S, TraceHit &best, uint32_t *lds, uint32_t *ovf,
    TraceStats &st, bool &occluded)
{
  if (s.post != 0) {
    const uint32_t enc = ~(uint32_t)s.post;
    s.post = 0;
    const uint32_t first = enc >> 3;
    // An instance's transform and a primitive record are both three 16-byte
    // words, and a BLAS leaf holds at most two records as a rule: six loads
    // fetch what either kind of leaf needs, so a round waits for memory once
    // and not for the instances, the first and the second records in turn.
    // (Once the node loop leaves early, leaf rounds are half of the work;
    // 1080p terrain at 4 spp, streams serialised, with the lean hit update
    // below: k_extend 6.43 -> 5.71 ms, k_shadow 7.65 -> 6.97 ms.)
    const bool enter = s.inst < 0;
    const float4 *P = enter ? reinterpret_cast<const float4 *>(S.instances + first)
                            : reinterpret_cast<const float4 *>(S.prims + first);
    const float4 r0 = P[0], r1 = P[1], r2 = P[2], r3 = P[3], r4 = P[4], r5 = P[5];
    if (enter) {
      // world leaf: one instance; continue in its BLAS with the object ray
      s.inst = (int)first;
      const linear3f rl = {{r0.x, r0.y, r0.z}, {r0.w, r1.x, r1.y}, {r1.z, r1.w, r2.x}};
      const vec3f d = mul(rl, s.wdir);
      s.box = boxRay(mul(rl, s.worg) + v3(r2.y, r2.z, r2.w), d);
      s.pc = triPrecompute(d);
      if (MODE == MODE_OCCLUSION)
        s.modelOffset = __float_as_int(r3.z) ? -1 : __float_as_int(r3.y);
      if (s.sp + kStackRow >= (kLdsDepth + kOverflowDepth) * kStackRow) // cannot happen, as above
        return true;
      tracePush(s, lds, ovf, s.cur); // kTraceDone too: it goes back where it came from
      tracePush(s, lds, ovf, kMarker);
      s.cur = __float_as_int(r3.x);
      return false;
    }
    const uint32_t end = first + (enc & 7u) + 1u;
    PrimWords w = primWords(r0, r1, r2), next = primWords(r3, r4, r5);
    for (uint32_t k = first;;) {
      if (STATS)
        st.prims++;
      if (tracePrim<MODE, RECORD, TIES>(s, S, best, w, k, ovf)) {
        occluded = true;
        return true;
      }
      if (++k == end)
        break;
      if (k != first + 1) {
        const float4 *N = reinterpret_cast<const float4 *>(S.prims + k);
        next = primWords(N[0], N[1], N[2]);
      }
      w = next;
    }
  }
  if (s.cur == kMarker) {
    s.box = boxRay(s.worg, s.wdir);
    s.inst = -1;
    s.cur = tracePop(s, lds, ovf);
  }
  return s.cur == kTraceDone;
}

template <int MODE, bool STATS, bool RECORD = false, int TIES = TIES_OFF>
__device__ bool traceRay(const DScene &S, vec3f worg, vec3f wdir, float t0, float tfar, Hit &best,
    uint32_t *lds, uint32_t *ovf, bool &sawTransparent, TraceStats &st)
{
  TraceState s;
  TraceHit hit;
  traceBegin(s, S, worg, wdir, t0, tfar, hit, lds);
  bool occluded = false;
  for (;;) {
    traceDescend<MODE, STATS>(s, S, lds, ovf, st);
    if (!traceHolds(s)) {
      if (s.cur == kTraceDone) // no node left
        break;
      continue; // other lanes hold leaves
    }
    if (traceLeaf<MODE, STATS, RECORD, TIES>(s, S, hit, lds, ovf, st, occluded))
      break;
  }
  sawTransparent = s.sawTransparent;
  if (MODE == MODE_OCCLUSION)
    return occluded;
  best = hitFromTrace(S, worg, wdir, t0, hit);
  if (TIES == TIES_RESOLVE && s.tie)
    resolveNearTie<STATS>(S, worg, wdir, t0, tfar, best, lds, ovf, st);
  if (TIES == TIES_REPORT)
    sawTransparent = s.tie;
  return best.hit;
}

// The hit record the closest-hit traversal of (worg, wdir) returns for a
// hit recorded by the occlusion traversal: the same object ray (instance
// transform, triPrecompute) and the same primitive test give the same
// t, u, v and Ng bit for bit.
__device__ __forceinline__ void hitFromRecord(const DScene &S, vec3f worg, vec3f wdir, float4 r, Hit &h)
{
  const uint32_t inst = __float_as_uint(r.y);
  vec3f o, d;
  objectRay(S.instances[inst], worg, wdir, o, d);
  const DPrim &P = S.prims[__float_as_uint(r.z)];
  const float4 pa = reinterpret_cast<const float4 *>(&P)[0];
  const float4 pb = reinterpret_cast<const float4 *>(&P)[1];
  const float4 pcv = reinterpret_cast<const float4 *>(&P)[2];
  const uint32_t mk = __float_as_uint(pb.w);
  const uint32_t kind = mk >> 28;
  h.hit = true;
  h.t = r.x;
  h.inst = inst;
  h.model = mk & 0x0fffffffu;
  h.prim = __float_as_uint(pa.w);
  h.half = 0;
  h.u = h.v = 0.f;
  if (kind == PRIM_SPHERE) {
    float tE, tX;
    vec3f NE, NX;
    sphereRoots(o, d, -kInf, v3(pa.x, pa.y, pa.z), pb.x, kInf, tE, NE, tX, NX);
    h.Ng = __float_as_uint(r.w) ? NX : NE;
  } else {
    const vec3f A = v3(pa.x, pa.y, pa.z), B = v3(pb.x, pb.y, pb.z), C = v3(pcv.x, pcv.y, pcv.z);
    float t, u = 0.f, v = 0.f;
    intersectTriangle(o, -kInf, triPrecompute(d), A, B, C, kInf, t, u, v);
    h.Ng = cross(B - A, C - A);
    h.u = u;
    h.v = v;
    if (kind == PRIM_QUAD1) {
      h.half = 1;
      h.u = 1.0f - u;
      h.v = 1.0f - v;
    }
  }
}

} // namespace hpt
