// Traversal of one ray by a whole wave (device), for queues with fewer rays
// than the chip has waves.
//
// A lane that traverses alone takes its 20 to 150 node steps one after
// another, and a launch over a few rays lasts as long as the longest of
// them.  Here sixteen nodes are stepped at a time, four lanes to a node (one
// to a child), and up to 32 BLAS leaves are tested at a time, two lanes to a
// leaf, so a ray takes about as many steps as the tree has levels.  It opens
// some nodes a nearest-first traversal would have skipped, on a chip that
// would have idled.
//
// A ray runs in phases over lists in the wave's part of the LDS rows:
//   world     nodes of the TLAS until its instances fill a list or none are
//             left;
//   instances up to kWideSlots - 1 of the listed instances are entered, each
//             with a slot that holds its object ray (slot 0: the world ray);
//   BLAS      nodes and leaves above the world's part of the stack until
//             none are left; then the slots are free again.
// The result is the one of the traversal by lanes: the set of primitives
// whose boxes a ray enters contains every hit either way, and the closest of
// them is chosen by the same (t, key).
#pragma once

#include "pt_trace.h"

namespace hpt {

constexpr int kWideSlots = 24, kWideSlotWords = 13; // (odd: slots on distinct banks)
constexpr int kWideStack = 320; // entries
constexpr int kWideList = 96; // entries of the leaf and of the instance list
constexpr int kWideBatch = 32; // listed leaves that are worth a test, instances that end the world phase
// Nodes popped at a time may push four times as many: several are popped
// only while the stack stays this low, then one at a time as a lane would
// (a world's stack need, TLAS and BLAS together, is at most kStackCapacity).
constexpr int kWideWorldMax = 48, kWideBlasMax = kWideStack - kStackCapacity;
static_assert(kWideWorldMax + kWideSlots + kStackCapacity <= kWideStack, "wide stack");
static_assert(4 * (kWideSlots * kWideSlotWords + 2 * kWideStack + 4 * kWideList) <= kLdsDepth * 64 * 4, "wide LDS");
static_assert(kWideBatch + 64 <= kWideList, "wide lists");

// A stack or list entry: a reference and the distance at which its box is
// entered, whose lowest 5 bits (rounded towards the ray's origin for t >= 0)
// hold the slot of its ray.
struct WideEntry
{
  uint32_t ref, ts;
};

__device__ __forceinline__ uint32_t widePack(float t, uint32_t slot) { return (__float_as_uint(t) & ~31u) | slot; }
__device__ __forceinline__ float wideT(uint32_t ts) { return __uint_as_float(ts & ~31u); }

struct WideLds
{
  float slots[kWideSlots * kWideSlotWords]; // o, 1 / d, Sx, Sy, Sz, kz, instance, first model
  WideEntry stack[kWideStack];
  WideEntry leaves[kWideList], insts[kWideList];
};

__device__ __forceinline__ void wideStoreBox(float *w, const BoxRay &b)
{
  w[0] = b.o.x, w[1] = b.o.y, w[2] = b.o.z;
  w[3] = b.inv.x, w[4] = b.inv.y, w[5] = b.inv.z;
}

// x of the lane `mask` away within the group of four (1, 2 or 3)
template <int MASK>
__device__ __forceinline__ float quadXor(float x)
{
  constexpr int ctrl = MASK == 1 ? 0xB1 : (MASK == 2 ? 0x4E : 0x1B); // quad_perm
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), ctrl, 0xf, 0xf, false));
}

__device__ __forceinline__ int bits(unsigned long long m) { return __builtin_popcountll(m); }
__device__ __forceinline__ float laneF(float x, int lane)
{
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), lane));
}

// The ray (worg, wdir, [t0, tfar]), the same in every lane of the wave.
// best, tie and sawTransparent as the traversal by lanes leaves them; RECORD
// writes the recorded hits of lane 0's row.  Returns whether an opaque
// occluder was hit (MODE_OCCLUSION).  The whole wave calls it.
template <int MODE, bool STATS, bool RECORD, int TIES>
__device__ __forceinline__ bool traceWide(const DScene &S, vec3f worg, vec3f wdir, float t0, float tfar,
    TraceHit &best, bool &tie, bool &sawTransparent, WideLds &W, uint32_t *row0, TraceStats &st)
{
  const int lane = (int)__lane_id(), group = lane >> 2, c = lane & 3;
  const unsigned long long below = (1ull << lane) - 1ull; // lanes below this one
  const unsigned long long belowGroup = (1ull << (lane & ~3)) - 1ull;
  best.t = tfar;
  best.u = best.v = 0.f;
  best.inst = best.prim = kInvalidID;
  tie = sawTransparent = false;
  float tb = tfar;
  uint32_t recorded = 0; // hits of non-opaque primitives
  if (lane == 0) {
    wideStoreBox(W.slots, boxRay(worg, wdir));
    W.stack[0] = {(uint32_t)S.tlasRoot, 0u};
  }
  // wave-uniform: entries of the stack, of the world's part of it, of the lists
  int sp = 1, base = 0, nLeaves = 0, nInsts = 0;
  bool world = true;
  for (;;) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); // the last round's LDS writes before this one's reads
    if (nLeaves >= kWideBatch || (nLeaves > 0 && sp == base)) {
      // ---- BLAS leaves: two lanes each
      const int L = min(nLeaves, kWideBatch);
      const int li = nLeaves - 1 - (lane >> 1);
      uint32_t k = 0, end = 0;
      const float *w = W.slots;
      if ((lane >> 1) < L) {
        const WideEntry e = W.leaves[li];
        const uint32_t enc = ~e.ref;
        if (wideT(e.ts) <= tb) {
          k = (enc >> 3) + (uint32_t)(lane & 1);
          end = (enc >> 3) + (enc & 7u) + 1u;
        }
        w = W.slots + (e.ts & 31u) * kWideSlotWords;
      }
      nLeaves -= L;
      while (waveMask(k < end) != 0ull) { // once, for leaves of two
        float t = kInf, u = 0.f, v = 0.f, tX = 0.f;
        int roots = 0;
        uint32_t mk = 0;
        const uint32_t inst = __float_as_uint(w[10]);
        if (k < end) {
          const float4 *P = reinterpret_cast<const float4 *>(S.prims + k);
          const PrimWords q = primWords(P[0], P[1], P[2]);
          mk = q.mk;
          if (STATS)
            st.prims++;
          if (mk >> 28 != PRIM_SPHERE) {
            const TriPre pc = {__float_as_int(w[9]), w[6], w[7], w[8]};
            float tt;
            if (intersectTriangle(v3(w[0], w[1], w[2]), t0, pc, q.A, q.B, q.C, tb, tt, u, v)) {
              roots = 1;
              t = tt;
            }
          } else {
            vec3f o, d, NE, NX;
            objectRay(S.instances[inst], worg, wdir, o, d);
            float tE;
            roots = sphereRoots(o, d, t0, q.A, q.B.x, tb, tE, NE, tX, NX);
            if (roots)
              t = (roots & 1) ? tE : tX;
          }
        }
        const unsigned long long hits = waveMask(roots != 0);
        if (hits != 0ull) {
          if (MODE == MODE_OCCLUSION) {
            const int offset = __float_as_int(w[11]);
            const bool opaque = roots != 0 && (offset < 0 || S.models[offset + (int)(mk & 0x0fffffffu)].opaque);
            if (waveMask(opaque) != 0ull)
              return true; // sawTransparent of no matter, and no count written
            sawTransparent = true;
            if (RECORD) { // as recordHit, the count in a register until the end
              for (unsigned long long m = hits; m != 0ull; m &= m - 1ull) {
                const int l = __builtin_ctzll(m);
                const int rl = __builtin_amdgcn_readlane(roots, l);
                if (lane == l) {
                  uint32_t at = recorded;
                  if ((roots & 1) && at < (uint32_t)kTransRecHits)
                    recordedHits(row0)[at] = make_float4(t, __uint_as_float(inst), __uint_as_float(k), __uint_as_float(0u));
                  at += roots & 1;
                  if ((roots & 2) && at < (uint32_t)kTransRecHits)
                    recordedHits(row0)[at] = make_float4(tX, __uint_as_float(inst), __uint_as_float(k), __uint_as_float(1u));
                }
                recorded += (uint32_t)((rl & 1) + (rl >> 1));
              }
            }
          } else {
            float tm = t;
            for (int o = 32; o > 0; o >>= 1)
              tm = fminf(tm, __shfl_xor(tm, o));
            tm = laneF(tm, 0);
            const float before = best.prim != kInvalidID ? best.t : kInf;
            if (TIES != TIES_OFF && tm < before && !(before - tm <= kTieEps * before))
              tie = false; // below the window of the previous closest hit
            // the closest hits of the round, in any order
            for (unsigned long long m = waveMask(t == tm && roots != 0); m != 0ull; m &= m - 1ull) {
              const int l = __builtin_ctzll(m);
              const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)inst, l),
                             hk = (uint32_t)__builtin_amdgcn_readlane((int)k, l);
              const bool any = best.prim != kInvalidID;
              if (!any || tm < best.t || (tm == best.t && primLess(S, hi, hk, best))) {
                best.t = tm;
                best.u = laneF(u, l);
                best.v = laneF(v, l);
                best.inst = hi;
                best.prim = hk;
              }
            }
            if (TIES != TIES_OFF) {
              // another hit, in this batch of leaves or before it, within the window
              // of the closest one (the wider of the two hits' windows)
              const int near = bits(waveMask(roots != 0 && t - best.t <= kTieEps * t));
              if (near > 1 || (near == 1 && before < kInf && fabsf(before - tm) <= kTieEps * fmaxf(before, tm)))
                tie = true;
            }
            tb = TIES == TIES_OFF ? best.t
                                  : (TIES == TIES_REPORT ? best.t + kTieEps * best.t
                                                         : fminf(best.t + kTieEps * best.t, tfar));
          }
        }
        k += 2;
      }
      continue;
    }
    if (sp > base) {
      // ---- nodes: four lanes each, the nearest of the top node ends on top
      const int room = ((world ? kWideWorldMax : kWideBlasMax) - sp) / 3;
      const int m = min(min(16, sp - base), max(1, room));
      bool hit = false;
      float tn = kInf;
      uint32_t slot = 0;
      int32_t child = 0;
      if (group < m) {
        const WideEntry e = W.stack[sp - 1 - group];
        slot = e.ts & 31u;
        if (wideT(e.ts) <= tb) {
          const float4 *np = reinterpret_cast<const float4 *>(S.nodes + e.ref);
          const float4 a = np[0], b = np[1];
          const uint4 q = reinterpret_cast<const uint4 *>(np)[2];
          child = reinterpret_cast<const int32_t *>(np + 3)[c];
          const float *w = W.slots + slot * kWideSlotWords;
          if (STATS && c == 0)
            st.nodes++;
          const NodeAxis x = nodeAxis(a.x, a.w, __float_as_uint(b.z), __float_as_uint(b.w), w[0], w[3]);
          const NodeAxis y = nodeAxis(a.y, b.x, q.x, q.y, w[1], w[4]);
          const NodeAxis z = nodeAxis(a.z, b.y, q.z, q.w, w[2], w[5]);
          const int sh = 8 * c;
          auto plane = [sh](uint32_t words) { return (float)((words >> sh) & 0xffu); };
          const float n = fmaxf(fmaxf(fmaf(plane(x.first), x.a, x.near), fmaf(plane(y.first), y.a, y.near)),
              fmaxf(fmaf(plane(z.first), z.a, z.near), t0));
          const float f = fminf(fminf(fmaf(plane(x.last), x.a, x.far), fmaf(plane(y.last), y.a, y.far)),
              fminf(fmaf(plane(z.last), z.a, z.far), tb));
          hit = n <= f && n < kInf;
          tn = hit ? (n >= 0.f ? n : -kInf) : kInf; // (t0 may be negative)
        }
      }
      sp -= m;
      const bool inner = hit && child >= 0;
      // rank of an inner child among its group's, by distance
      const float ti = inner ? tn : kInf;
      const float t1 = quadXor<1>(ti), t2 = quadXor<2>(ti), t3 = quadXor<3>(ti);
      const int rank = (t1 < ti || (t1 == ti && (c & 1))) + (t2 < ti || (t2 == ti && (c & 2)))
          + (t3 < ti || (t3 == ti && (c & 2)));
      const unsigned long long im = waveMask(inner), lm = waveMask(hit && child < 0);
      const int total = bits(im);
      if (inner && sp + total <= kWideStack) // always (kWideBlasMax)
        W.stack[sp + total - 1 - (bits(im & belowGroup) + rank)] = {(uint32_t)child, widePack(tn, slot)};
      sp = min(sp + total, kWideStack);
      WideEntry *list = world ? W.insts : W.leaves;
      const int at = (world ? nInsts : nLeaves) + bits(lm & below);
      if (hit && child < 0)
        list[at] = {(uint32_t)child, widePack(tn, slot)};
      if (world)
        nInsts += bits(lm);
      else
        nLeaves += bits(lm);
      if (!world || (sp > 0 && nInsts < kWideBatch))
        continue;
    }
    // ---- the phase has ended: no node left of it, or enough instances
    if (nInsts > 0) {
      const int n = min(nInsts, kWideSlots - 1);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      bool enter = false, leaf = false;
      uint32_t ts = 0;
      int root = 0;
      float4 r0, r1, r2, r3;
      uint32_t inst = 0;
      if (lane < n) {
        const WideEntry e = W.insts[nInsts - n + lane];
        ts = e.ts;
        inst = ~e.ref >> 3;
        if (wideT(ts) <= tb) {
          const float4 *I = reinterpret_cast<const float4 *>(S.instances + inst);
          r0 = I[0], r1 = I[1], r2 = I[2], r3 = I[3];
          root = __float_as_int(r3.x);
          enter = root >= 0;
          leaf = root < 0;
        }
      }
      nInsts -= n;
      const unsigned long long em = waveMask(enter), lm = waveMask(leaf);
      base = sp;
      if (enter || leaf) {
        const uint32_t slot = 1u + (uint32_t)bits((em | lm) & below);
        const linear3f rl = {{r0.x, r0.y, r0.z}, {r0.w, r1.x, r1.y}, {r1.z, r1.w, r2.x}};
        const vec3f o = mul(rl, worg) + v3(r2.y, r2.z, r2.w);
        const vec3f d = mul(rl, wdir);
        const TriPre pc = triPrecompute(d);
        float *w = W.slots + slot * kWideSlotWords;
        wideStoreBox(w, boxRay(o, d));
        w[6] = pc.Sx, w[7] = pc.Sy, w[8] = pc.Sz;
        w[9] = __int_as_float(pc.kz);
        w[10] = __uint_as_float(inst);
        w[11] = __int_as_float(__float_as_int(r3.z) ? -1 : __float_as_int(r3.y));
        const WideEntry e = {(uint32_t)root, (ts & ~31u) | slot};
        if (enter) // the first listed on top
          W.stack[sp + bits(em) - 1 - bits(em & below)] = e;
        else // a BLAS that is one leaf
          W.leaves[bits(lm & below)] = e;
      }
      sp += bits(em);
      nLeaves = bits(lm);
      world = false;
      if (sp > base || nLeaves > 0)
        continue;
    }
    if (nInsts > 0)
      continue; // the listed ones lay beyond the closest hit
    // the BLAS phase has ended: on with the world's nodes
    base = 0;
    world = true;
    if (sp == 0) {
      if (RECORD && recorded > 0) {
        if (lane == 0)
          *recordedCount(row0) = recorded;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup"); // lane 0 reads the other lanes' records
      }
      return false;
    }
  }
}

} // namespace hpt
