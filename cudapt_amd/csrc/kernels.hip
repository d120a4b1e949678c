// gfx950 kernels of the streaming-BDPT hot path.
//
//  trace8         closest/any hit of a wave's rays over 8-wide nodes with FP16
//                 boxes: a node a lane per step, then the wave's leaf triangles
//                 as one list, one (ray, triangle) pair per lane.  Replaces
//                 TracePrimitive (src/cudaRTCommon.cu:66-127).
//  traverse4      the same over 128-byte FP32 4-wide nodes, one ray a thread,
//                 ordered near-first, stack top in LDS, deeper entries private.
//  traverse_bin   the same query over the reference's binary CompactBVH
//                 layout (src/cudaRTCommon.cu:527-541), kept as the baseline.
//  k_light_pass   light-vertex cache: pt_genLightPathQueue_kernel +
//                 pt_traceLight_kernel loop (src/cudaRTBDPTStream.cu:180-363,
//                 545-617, 875-906) in one workgroup; stream order of the
//                 reference's stable compaction from a workgroup prefix sum.
//  k_gen_eye      pt_genPathQueue_kernel (src/cudaRTBDPTStream.cu:619-640).
//  k_extend       closest hit of every live path (SoA queue).
//  k_shade        pt_traceSample_kernel body + connection set-up of
//                 pt_connectEyeLightPath_kernel + pt_applyPathQueueResult_kernel
//                 for terminated paths (src/cudaRTBDPTStream.cu:365-543,
//                 665-778); survivors and shadow rays compacted with a wave64
//                 ballot + per-workgroup prefix, one atomic per workgroup.
//  k_shadow       occlusion of the connection segment and the N += 4 update.
//
// Hit semantics: the closest hit is the minimum of (t, original triangle id)
// over all triangles with 0 <= t < maxDist, each tested with IntersectTri's
// exact arithmetic (src/cudaRTCommon.cu:42-64).  Over the 8-wide nodes culling is
// conservative, so the answer does not depend on the visiting order.  Over
// the FP32 4-wide nodes (Ize 2013 slab widening + a slack for IntersectTri's eps
// origin shift) a ray that touches a triangle's edge within rounding may miss its
// box: see kQueryFp32 for how often.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "devmath.h"
#include "kernels.h"

namespace cpt {

// Stack entries per thread in total; the top STK live in LDS, the rest in
// private memory.  A 4-wide level pushes at most 3 entries and the depth is
// <= 31 (checked at build), so 96 entries never overflow.
#define CPT_STACK_TOTAL 96
#define CPT_LDS_STACK 16   // default LDS share (k_light_pass, shadow)

// Smallest float >= 1e-9: float |det| < it  <=>  (double)|det| < M_EPSILON.
__device__ constexpr float kDetEps = 0x1.12e0c0p-30f;
__device__ constexpr float kPiF = 3.14159265358979323846f;
constexpr double kPiD = 3.14159265358979323846;

struct TraceHit {
  float t, u, v;
  uint32_t leaf, orig;
};

// splitmix64 finaliser (Steele, Lea, Flood 2014) keyed by (seed, frame, domain,
// sample): the per-path PCG32 initstate that takes the place of
// curand_init(WangHash(frameN) + index, 0, 0) (src/cudaRTBDPTStream.cu:552,633).
// Domains: 1 eye paths, 2 light paths.
__device__ __forceinline__ uint64_t stream_key(uint64_t seed, uint32_t frame, uint32_t domain, uint32_t sample) {
  uint64_t z = seed + 0x9E3779B97F4A7C15ULL * (uint64_t)(frame + 1) + ((uint64_t)sample << 32) + ((uint64_t)domain << 60);
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ULL;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebULL;
  return z ^ (z >> 31);
}


__device__ __forceinline__ float escape_zero(float v) {
  const float e = 1e-9f;
  if (fabsf(v) < e) v = (v > 0.f) ? v + e : v - e;
  return v;
}
__device__ __forceinline__ float cull_slack(float best, float eps) { return eps + best * 1e-4f + 1e-5f; }

// CURay::IntersectTri (src/cudaRTCommon.cu:42-64); o2 = orig + eps * dir.
__device__ __forceinline__ float isect_tri(f3 o2, f3 d, f3 p0, f3 e0, f3 e1, bool cull, float& u, float& v) {
  if (cull && dot(cross(e0, e1), d) > 0.f) return kInfF;
  f3 de2 = cross(d, e1);
  float div = dot(de2, e0);
  if (fabsf(div) < kDetEps) return kInfF;
  div = 1.0f / div;
  f3 t = o2 - p0;
  f3 te1 = cross(t, e0);
  float rT = dot(te1, e1) * div;
  if (rT < 0.f) return kInfF;
  u = dot(de2, t) * div;
  if (u < 0.f || u > 1.f) return kInfF;
  v = dot(te1, d) * div;
  if (v < 0.f || (u + v) > 1.f) return kInfF;
  return rT;
}

__device__ __forceinline__ bool better(float t, uint32_t oid, const TraceHit& h) {
  return t < h.t || (t == h.t && h.leaf != kInvalid && oid < h.orig);
}

__device__ __forceinline__ void test_leaf(const float4* __restrict__ tris, uint32_t first, uint32_t count, f3 o2, f3 d,
                                          bool cull, TraceHit& h, uint32_t& nt) {
  for (uint32_t i = first; i < first + count; i++) {
    float4 a = tris[3 * i], b = tris[3 * i + 1], c = tris[3 * i + 2];
    float u = 0.f, v = 0.f;
    float t = isect_tri(o2, d, ld3(a), ld3(b), ld3(c), cull, u, v);
    uint32_t oid = __float_as_uint(a.w);
    if (t >= 0.f && better(t, oid, h)) { h.t = t; h.u = u; h.v = v; h.leaf = i; h.orig = oid; }
  }
  nt += count;
}

__device__ __forceinline__ void cswap(uint64_t& a, uint64_t& b) {
  uint64_t lo = a < b ? a : b, hi = a < b ? b : a;
  a = lo; b = hi;
}

// Child boxes and links of a 4-wide node (128 bytes, FP32).
struct NodeView {
  float lx[4], hx[4], ly[4], hy[4], lz[4], hz[4];
  uint32_t ch[4], cn[4];
};
__device__ __forceinline__ void load_node(const DevScene& sc, uint32_t node, NodeView& v) {
  const Node4* N = sc.nodes4 + node;
  const float4 lx = *(const float4*)N->lox, hx = *(const float4*)N->hix;
  const float4 ly = *(const float4*)N->loy, hy = *(const float4*)N->hiy;
  const float4 lz = *(const float4*)N->loz, hz = *(const float4*)N->hiz;
  const uint4 ch = *(const uint4*)N->child, cn = *(const uint4*)N->count;
  v.lx[0] = lx.x; v.lx[1] = lx.y; v.lx[2] = lx.z; v.lx[3] = lx.w;
  v.hx[0] = hx.x; v.hx[1] = hx.y; v.hx[2] = hx.z; v.hx[3] = hx.w;
  v.ly[0] = ly.x; v.ly[1] = ly.y; v.ly[2] = ly.z; v.ly[3] = ly.w;
  v.hy[0] = hy.x; v.hy[1] = hy.y; v.hy[2] = hy.z; v.hy[3] = hy.w;
  v.lz[0] = lz.x; v.lz[1] = lz.y; v.lz[2] = lz.z; v.lz[3] = lz.w;
  v.hz[0] = hz.x; v.hz[1] = hz.y; v.hz[2] = hz.z; v.hz[3] = hz.w;
  v.ch[0] = ch.x; v.ch[1] = ch.y; v.ch[2] = ch.z; v.ch[3] = ch.w;
  v.cn[0] = cn.x; v.cn[1] = cn.y; v.cn[2] = cn.z; v.cn[3] = cn.w;
}

// Instantiates launch macro M(stack entries, min waves per SIMD) for the
// traversal variant v (traversal_variant_ok); other values return an error.
#define CPT_VARIANT_SWITCH(v, M)            \
  switch (v) {                              \
    case 8: M(8, 0); break;                 \
    case 16: M(16, 0); break;               \
    case 24: M(24, 0); break;               \
    case 806: M(8, 6); break;               \
    case 807: M(8, 7); break;               \
    case 808: M(8, 8); break;               \
    case 1606: M(16, 6); break;             \
    default: return hipErrorInvalidValue;   \
  }

// The top of a thread's traversal stack: its column of a [entries][kBlock] u64
// array in LDS, typed as LDS so that the pop (LDS or private, by depth) stays
// two plain accesses instead of one generic one.
typedef __attribute__((address_space(3))) uint64_t LdsU64;
__device__ __forceinline__ LdsU64* lds_column(uint64_t* shared_base) {
  return (LdsU64*)(shared_base + threadIdx.x);
}

// ---- 4-wide traversal ------------------------------------------------------
// The state of one ray's traversal, advanced one node at a time by ray_step, so
// that a lane whose ray has finished can start another while the rest of its
// wave is still traversing (k_trace_dyn) or simply loop (traverse4).
struct RayState {
  f3 o, d, idir, o2;
  float eps;
  TraceHit h;
  uint32_t node;
  int sp;
};
__device__ __forceinline__ void ray_begin(RayState& R, f3 o, f3 d, float maxd, float eps) {
  R.o = o;
  R.d = d;
  R.idir = mk3(1.f / escape_zero(d.x), 1.f / escape_zero(d.y), 1.f / escape_zero(d.z));
  R.o2 = o + d * eps;
  R.eps = eps;
  R.h.t = maxd; R.h.u = R.h.v = 0.f; R.h.leaf = kInvalid; R.h.orig = kInvalid;
  R.node = 0;
  R.sp = 0;
}
// The four child boxes of node R.node: entry / exit distances (entry clamped
// at 0), children and leaf counts.
__device__ __forceinline__ void child_boxes(const DevScene& sc, const RayState& R, float tn[4], float tf[4],
                                            uint32_t ch[4], uint32_t cn[4]) {
  NodeView nv;
  load_node(sc, R.node, nv);
#pragma unroll
  for (int c = 0; c < 4; c++) {
    float t0x = (nv.lx[c] - R.o.x) * R.idir.x, t1x = (nv.hx[c] - R.o.x) * R.idir.x;
    float t0y = (nv.ly[c] - R.o.y) * R.idir.y, t1y = (nv.hy[c] - R.o.y) * R.idir.y;
    float t0z = (nv.lz[c] - R.o.z) * R.idir.z, t1z = (nv.hz[c] - R.o.z) * R.idir.z;
    tn[c] = fmaxf(fmaxf(fminf(t0x, t1x), fminf(t0y, t1y)), fmaxf(fminf(t0z, t1z), 0.f));
    tf[c] = fminf(fminf(fmaxf(t0x, t1x), fmaxf(t0y, t1y)), fmaxf(t0z, t1z)) * 1.0000004f;
    ch[c] = nv.ch[c];
    cn[c] = nv.cn[c];
  }
}

// The leaf children's triangles as one run (child order, triangle order):
// child c contributes ln[c] triangles from lf[c] on.  Run position k lies in
// child c when p_c <= k < p_(c+1) (prefix sums of the counts); its triangle is
// k + (first_c - p_c): selects, no branches.  Returns true when an occlusion
// ray (ANY) found a hit.
template <bool ANY>
__device__ __forceinline__ bool test_run(const DevScene& sc, RayState& R, bool cull, const uint32_t lf[4],
                                         const uint32_t ln[4], uint32_t& nt) {
  const uint32_t p1 = ln[0], p2 = p1 + ln[1], p3 = p2 + ln[2];
  const uint32_t ntri = p3 + ln[3];
  nt += ntri;
  const uint32_t d0 = lf[0], d1 = lf[1] - p1, d2 = lf[2] - p2, d3 = lf[3] - p3;
  // All of a triangle's 48 bytes are fetched at once (the empty asm needs the
  // vertex before the determinant test, which would otherwise delay its load
  // to a second round trip); one triangle per round trip for both ray kinds:
  // fetching two for occlusion rays spilled five registers of the shadow
  // kernel and ran it 2 % slower end to end.
  for (uint32_t k = 0; k < ntri; k++) {
    const uint32_t i = k + (k < p1 ? d0 : k < p2 ? d1 : k < p3 ? d2 : d3);
    const float4 a = sc.tris[3 * i], b = sc.tris[3 * i + 1], cc = sc.tris[3 * i + 2];
    asm volatile("" : : "v"(a.x), "v"(a.y), "v"(a.z));
    float u = 0.f, v = 0.f;
    const float t = isect_tri(R.o2, R.d, ld3(a), ld3(b), ld3(cc), cull, u, v);
    const uint32_t oid = __float_as_uint(a.w);
    if (t >= 0.f && better(t, oid, R.h)) { R.h.t = t; R.h.u = u; R.h.v = v; R.h.leaf = i; R.h.orig = oid; }
    if (ANY && R.h.leaf != kInvalid) return true;
  }
  return false;
}

// Pops the nearest pending node still in front of the best hit into R.node;
// false when the stack runs out (the ray is finished).
template <int STK>
__device__ __forceinline__ bool pop_node(RayState& R, const LdsU64* lstk, const uint64_t* pstk) {
  while (R.sp > 0) {
    R.sp--;
    uint64_t e = R.sp < STK ? lstk[R.sp * kBlock] : pstk[R.sp - STK];
    float tn = __uint_as_float((uint32_t)(e >> 32));
    if (tn <= R.h.t + cull_slack(R.h.t, R.eps)) { R.node = (uint32_t)e; return true; }
  }
  return false;
}

// One node: the four child boxes against the ray (culled beyond the best hit
// plus slack); the leaf children hit are then tested as one run of triangles
// (test_run), so that lanes whose leaves sit under different children test
// them in the same loop; interior children are culled again with the updated
// best hit, sorted near-first, the nearest taken next and the rest pushed
// (LDS stack top, private stack below it).  The closest hit is the
// (t, original id) minimum, which neither the test order nor the conservative
// culling changes.  Returns true when the ray is finished.
// lstk points at this thread's column of a [STK][kBlock] u64 array in LDS.
// spill (an LDS word of the wave, or null) counts pushes that land below the
// LDS top, in the private (scratch) stack: an LDS atomic on that rare event
// instead of a counter register in the loop.
template <bool ANY, int STK>
__device__ __forceinline__ bool ray_step(const DevScene& sc, RayState& R, bool cull, LdsU64* lstk, uint64_t* pstk,
                                         uint32_t& nn, uint32_t& nt, uint32_t* spill) {
  float tn[4], tf[4];
  uint32_t ch[4], cn[4];
  child_boxes(sc, R, tn, tf, ch, cn);
  nn++;
  const float lim = R.h.t + cull_slack(R.h.t, R.eps);
  uint64_t key[4];
  uint32_t lf[4], ln[4];
#pragma unroll
  for (int c = 0; c < 4; c++) {
    const float tnear = tn[c];
    bool hit = ch[c] != kInvalid && tnear <= tf[c] && tnear <= lim;
    const bool leaf = cn[c] > 0;
    lf[c] = ch[c];
    ln[c] = hit && leaf ? cn[c] : 0u;
    // 0 marks no interior child (a child link is never the root, 0)
    key[c] = hit && !leaf ? ((uint64_t)__float_as_uint(tnear) << 32) | ch[c] : 0ull;
  }
  if (ln[0] + ln[1] + ln[2] + ln[3]) {
    if (test_run<ANY>(sc, R, cull, lf, ln, nt)) return true;
    const float lim2 = R.h.t + cull_slack(R.h.t, R.eps);
#pragma unroll
    for (int q = 0; q < 4; q++)
      if (__uint_as_float((uint32_t)(key[q] >> 32)) > lim2) key[q] = 0ull;
  }
  // Near-first for both ray kinds: occlusion rays taken in node order visit
  // 15 % fewer nodes but test 23 % more triangles and run 1 % slower on the
  // sphere grid.  Sorted ascending, the n interior children hit are the last n
  // keys: key[4 - n] is taken next and key[3], key[2], key[1] (those of them
  // past it) are pushed farthest first.  Slots from sp on are free, so when
  // all three fit the LDS top they are written unconditionally and sp moves
  // by n - 1.
  // With one interior child hit there is nothing to sort or push: its key is
  // the OR of the four (the others are 0).
  const int n = ((uint32_t)key[0] != 0u) + ((uint32_t)key[1] != 0u) + ((uint32_t)key[2] != 0u) +
                ((uint32_t)key[3] != 0u);
  if (n == 1) {
    R.node = (uint32_t)(key[0] | key[1] | key[2] | key[3]);
    return false;
  }
  if (n) {
    cswap(key[0], key[1]); cswap(key[2], key[3]); cswap(key[0], key[2]); cswap(key[1], key[3]); cswap(key[1], key[2]);
    R.node = n >= 3 ? (uint32_t)(n >= 4 ? key[0] : key[1]) : (uint32_t)key[2];
    if (R.sp + 3 <= STK) {
      lstk[R.sp * kBlock] = key[3];
      lstk[(R.sp + 1) * kBlock] = key[2];
      lstk[(R.sp + 2) * kBlock] = key[1];
      R.sp += n - 1;
    } else {
#pragma unroll
      for (int c = 3; c >= 1; c--) {
        if (c + n > 4 && R.sp < CPT_STACK_TOTAL) {
          if (R.sp < STK) {
            lstk[R.sp * kBlock] = key[c];
          } else {
            pstk[R.sp - STK] = key[c];
            if (spill) atomicAdd(spill, 1u);
          }
          R.sp++;
        }
      }
    }
    return false;
  }
  return !pop_node<STK>(R, lstk, pstk);
}

// Closest (ANY: any) hit of one ray, the loop of ray_step.  pstk:
// CPT_STACK_TOTAL - STK private entries.
template <bool ANY, int STK>
__device__ __forceinline__ bool traverse4(const DevScene& sc, f3 o, f3 d, float maxd, float eps, bool cull,
                                          LdsU64* lstk, uint64_t* pstk, TraceHit& h, uint32_t& nn, uint32_t& nt) {
  RayState R;
  ray_begin(R, o, d, maxd, eps);
  while (!ray_step<ANY, STK>(sc, R, cull, lstk, pstk, nn, nt, nullptr)) {
  }
  h = R.h;
  return h.leaf != kInvalid;
}
template <bool ANY, int STK = CPT_LDS_STACK>
__device__ bool traverse4(const DevScene& sc, f3 o, f3 d, float maxd, float eps, bool cull, LdsU64* lstk,
                          TraceHit& h, uint32_t& nn, uint32_t& nt) {
  uint64_t pstk[CPT_STACK_TOTAL - STK];
  return traverse4<ANY, STK>(sc, o, d, maxd, eps, cull, lstk, pstk, h, nn, nt);
}

// Whether traverse4 is sure to test the triangle of device leaf index `leaf`,
// which the ray hits at t: whether the triangle's own box passes child_boxes'
// test with t as the best hit.  FP32 subtraction, multiplication, minimum and
// maximum are monotone, so every box round it passes then too.
// idir: v_rcp's, within 2 u (u = 2^-24) of 1 / d where child_boxes' is within u;
// the distances here are then within 5 u of the ones there.  Per axis the entry
// never lies past the exit; across axes the factor 1 + 2^-21 covers
// both distances' 5 u (child_boxes multiplies the exit by 1 + 6 u).  Exits
// and reciprocals near the denormals, where no relative bound holds, fail.
__device__ __forceinline__ bool reached4(const DevScene& sc, uint32_t leaf, f3 o, f3 idir, float t, float eps) {
  const float4 lo = sc.tri_box[2 * (size_t)leaf], hi = sc.tri_box[2 * (size_t)leaf + 1];
  const float k = 1.f + 0x1p-21f;
  const float x0 = (lo.x - o.x) * idir.x, x1 = (hi.x - o.x) * idir.x;
  const float y0 = (lo.y - o.y) * idir.y, y1 = (hi.y - o.y) * idir.y;
  const float z0 = (lo.z - o.z) * idir.z, z1 = (hi.z - o.z) * idir.z;
  const float ex = fminf(x0, x1) * k, fx = fmaxf(x0, x1);
  const float ey = fminf(y0, y1) * k, fy = fmaxf(y0, y1);
  const float ez = fminf(z0, z1) * k, fz = fmaxf(z0, z1);
  return ex <= fminf(fy, fz) && ey <= fminf(fx, fz) && ez <= fminf(fx, fy) &&
         fmaxf(fmaxf(ex, ey), fmaxf(ez, 0.f)) <= t + cull_slack(t, eps) &&
         fminf(fx, fminf(fy, fz)) >= 0x1p-100f &&
         fminf(fabsf(idir.x), fminf(fabsf(idir.y), fabsf(idir.z))) >= 0x1p-100f;
}

// ---- 8-wide traversal -------------------------------------------------------
// A wave traces its lanes' rays together.  Every step each lane visits one
// 8-wide quantized node; then all the leaf triangles that the wave's lanes hit
// in that step are tested as one list, one (ray, triangle) pair per lane
// whoever's ray it is.  A lane that walks its own triangles makes the wave wait
// for the longest run (three or four tests a step at a tenth of the lanes), and
// makes each test's load wait for the one before; the list takes one test
// and one round trip to memory for up to 64 pairs.  The ray a tester needs (o +
// eps d, d) and the best hit it competes for live in LDS, one column per lane.
//
// What bounds it: VALU instructions where the launch is large (the vector units
// issue all the time), the chain of node and triangle round trips of the
// longest ray where it is small; eight children a node shorten both.  FP16
// fractions cost no conversion (8-bit ones took one per plane: 205 against 150
// VALU instructions a node).  Over 4-wide 64-byte nodes with each lane walking
// its own triangles (sphere grid, 1280 x 720, 64 frames): 9.9 -> 6.3 nodes per
// extension ray, 14.7 -> 8.9 per shadow ray, lane use 37 -> 56 % and more;
// extension after the first bounce 8.65 -> 7.17 ms, first bounce 3.36 -> 3.24,
// shadow 13.6 -> 10.4 ms; a frame of 480,000 paths 1.77 -> 1.46 ms.  A node
// visited again for each child in plain octant order, without the nearest
// child first and the second nearest's distance to cull the rest by, takes 14 %
// more visits.
//
// The closest hit is the (t, original id) minimum: the order of the tests, the
// visiting order and the conservative culling do not change it.
template <int STK>
struct Wave8 {
  float ray[6][64];         // o + eps d, d
  uint64_t best[64];        // t bits << 32 | original id + 1 of the closest hit; low word 0: none
  uint32_t rec[4][64];      // that hit's t, u, v, device leaf index
  uint64_t list[64];        // the round's tests: triangle | lane << 32
  uint64_t stk[STK][64];    // top of the group stacks
};
// One ray's traversal: the node to visit next; sx, sy, sz: 16 where the
// direction is negative (the byte offset of an axis's near plane in a node); pn,
// pf: -o * idir moved out by the box test's slack, per axis.  A stack entry is a
// group, the other interior children that the ray hit under one node: the first
// child's node in the low word, above it the children still to visit (bit slot
// ^ octant, so that lower bits come first along the ray), the node's interior
// mask << 8, and the upper half of the bits of a lower bound on their entry
// distances << 16.
struct Ray8 {
  f3 idir, pn, pf;
  float eps, ht;
  uint32_t node;
  int sp;
};

// LDS accesses of one wave execute in issue order; this keeps the compiler
// from moving them across the point.
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}
template <int STK>
__device__ __forceinline__ void ray8_begin(Ray8& R, Wave8<STK>& W, int lane, f3 o, f3 d, float maxd, float eps,
                                           float qmag) {
  // within an ulp of 1 / d: the box test's slack covers it
  R.idir = mk3(__builtin_amdgcn_rcpf(escape_zero(d.x)), __builtin_amdgcn_rcpf(escape_zero(d.y)),
               __builtin_amdgcn_rcpf(escape_zero(d.z)));
  // Slack of the quantized box test (box8): 2^-20 = 16 u per unit of
  // |idir| (qmag + |o|), twice the rounding bound of that test's distances.
  const float k = 0x1p-20f;
  const float sx = (fabsf(R.idir.x) * (qmag + fabsf(o.x))) * k;
  const float sy = (fabsf(R.idir.y) * (qmag + fabsf(o.y))) * k;
  const float sz = (fabsf(R.idir.z) * (qmag + fabsf(o.z))) * k;
  const f3 oi = mk3(-(o.x * R.idir.x), -(o.y * R.idir.y), -(o.z * R.idir.z));
  R.pn = mk3(oi.x - sx, oi.y - sy, oi.z - sz);
  R.pf = mk3(oi.x + sx, oi.y + sy, oi.z + sz);
  // No triangle is hit from an origin that is infinite or NaN, or along a NaN (the
  // test's determinant or distance is one): such a ray meets no box, where NaN
  // distances would pass every box of the tree.
  constexpr int kNotFinite = 0x207;                  // v_cmp_class: NaN, -inf, +inf
  if (__builtin_amdgcn_classf(o.x, kNotFinite) || __builtin_amdgcn_classf(o.y, kNotFinite) ||
      __builtin_amdgcn_classf(o.z, kNotFinite) || __builtin_isunordered(d.x, d.y) ||
      __builtin_isunordered(d.z, eps)) {
    R.idir.x = 0.f;
    R.pn.x = __builtin_huge_valf();
    R.pf.x = -__builtin_huge_valf();
  }
  R.eps = eps;
  // no hit lies at t >= 0 below a maximum that is negative or NaN
  R.ht = maxd > 0.f ? maxd : 0.f;
  R.node = 0u;
  R.sp = 0;
  const f3 o2 = o + d * eps;
  W.ray[0][lane] = o2.x; W.ray[1][lane] = o2.y; W.ray[2][lane] = o2.z;
  W.ray[3][lane] = d.x; W.ray[4][lane] = d.y; W.ray[5][lane] = d.z;
  W.best[lane] = (uint64_t)__float_as_uint(R.ht) << 32;
}
// The lane's result once its ray has finished.
template <int STK>
__device__ __forceinline__ bool ray8_hit(const Wave8<STK>& W, int lane, TraceHit& h) {
  const uint32_t id = (uint32_t)W.best[lane];
  if (id == 0u) {
    h.t = kInfF; h.u = h.v = 0.f; h.leaf = h.orig = kInvalid;
    return false;
  }
  h.t = __uint_as_float(W.rec[0][lane]);
  h.u = __uint_as_float(W.rec[1][lane]);
  h.v = __uint_as_float(W.rec[2][lane]);
  h.leaf = W.rec[3][lane];
  h.orig = id - 1u;
  return true;
}

// The eight child boxes of a node against the ray: entry distances tn (clamped
// at 0) and the mask of the boxes the ray meets at or before lim.  A slab plane
// is o_a + h e_a with h the stored FP16 fraction and e_a a power of two, so its
// distance (o_a + h e_a - ray.o_a) idir_a is fma(h, e_a idir_a, c_a) with
// c_a = fma(o_a, idir_a, -ray.o_a idir_a) per node (e_a idir_a is exact); the
// near plane of each axis (by the sign of idir_a) gives the entry and the far
// plane the exit, so no per-axis min / max is needed.  With M = sc.qmag,
// u = 2^-24 and slack = 16 u |idir_a| (M + |ray.o_a|), the distance differs
// from the exact one to the host's plane by at most seven roundings (two for
// idir, within an ulp of 1 / d, the plane's own, -ray.o_a idir_a, the slack's
// addition and the two fmas), each within u (|idir_a| (M + |ray.o_a|) + slack):
// under half the slack, which is subtracted from entries (R.pn) and added to exits
// (R.pf), so no box that the ray meets in exact arithmetic is culled.
// Only the loads are masked by `active`: the vector caches serve one line a
// cycle (unmasked, 80 % of their cycles busy in the sphere grid's secondary rays), so the
// lines of idle lanes cost as much as the others', while idle lanes in the arithmetic
// cost nothing.  Masked / not: still of 64 1280 x 720 frames 18.4 / 19.2 ms, 8 views of
// the heightfield 11.2 / 12.3 ms, 1,000,003 occlusion rays there 146 / 163 us.
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
__device__ __forceinline__ uint32_t box8(const char* __restrict__ nodes, uint32_t node, const Ray8& R, float lim,
                                         float tn[8], uint4& A, uint4& B, bool active) {
  const uint32_t at = node * 128u;
  const uint32_t ox = R.idir.x >= 0.f ? 0u : 16u, oy = R.idir.y >= 0.f ? 0u : 16u, oz = R.idir.z >= 0.f ? 0u : 16u;
  h8 nx, fx, ny, fy, nz, fz;
  if (active) {
    A = *(const uint4*)(nodes + at);
    nx = *(const h8*)(nodes + (at | ox) + 32), fx = *(const h8*)(nodes + ((at | ox) ^ 16u) + 32);
    ny = *(const h8*)(nodes + (at | oy) + 64), fy = *(const h8*)(nodes + ((at | oy) ^ 16u) + 64);
    nz = *(const h8*)(nodes + (at | oz) + 96), fz = *(const h8*)(nodes + ((at | oz) ^ 16u) + 96);
    B = *(const uint4*)(nodes + at + 16);
  }
  const float ex = __uint_as_float((A.w & 0xFFu) << 23) * R.idir.x;
  const float ey = __uint_as_float(((A.w >> 8) & 0xFFu) << 23) * R.idir.y;
  const float ez = __uint_as_float(((A.w >> 16) & 0xFFu) << 23) * R.idir.z;
  const float qx = __uint_as_float(A.x), qy = __uint_as_float(A.y), qz = __uint_as_float(A.z);
  const float cnx = __builtin_fmaf(qx, R.idir.x, R.pn.x), cfx = __builtin_fmaf(qx, R.idir.x, R.pf.x);
  const float cny = __builtin_fmaf(qy, R.idir.y, R.pn.y), cfy = __builtin_fmaf(qy, R.idir.y, R.pf.y);
  const float cnz = __builtin_fmaf(qz, R.idir.z, R.pn.z), cfz = __builtin_fmaf(qz, R.idir.z, R.pf.z);
  uint32_t hits = 0;
#pragma unroll
  for (int c = 0; c < 8; c++) {
    const float ax = __builtin_fmaf((float)nx[c], ex, cnx), bx = __builtin_fmaf((float)fx[c], ex, cfx);
    const float ay = __builtin_fmaf((float)ny[c], ey, cny), by = __builtin_fmaf((float)fy[c], ey, cfy);
    const float az = __builtin_fmaf((float)nz[c], ez, cnz), bz = __builtin_fmaf((float)fz[c], ez, cfz);
    tn[c] = fmaxf(fmaxf(ax, ay), fmaxf(az, 0.f));
    const float tf = fminf(fminf(bx, by), fminf(bz, lim));
    hits |= tn[c] <= tf ? 1u << c : 0u;
  }
  return hits;
}

// The wave's pending leaf triangles (tmask: bits of `valid`, the node's first
// triangle tbase), tested against their lanes' rays, up to 64 a round.  Called
// by the whole wave.
template <int STK>
__device__ __forceinline__ void test_pairs(const DevScene& sc, Wave8<STK>& W, int lane, uint32_t tmask,
                                           uint32_t valid, uint32_t tbase, bool cull) {
  uint32_t n = 0;                                   // pairs listed (uniform)
  for (;;) {
    const uint64_t more = __ballot(tmask != 0u);
    const uint32_t m = (uint32_t)__popcll(more);
    if (m != 0u && n + m <= 64u) {                  // every lane with triangles left lists its next one
      if (tmask) {
        const uint32_t pos =
            n + __builtin_amdgcn_mbcnt_hi((uint32_t)(more >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)more, 0u));
        const uint32_t low = tmask - 1u, below = low & ~tmask;
        W.list[pos] = (uint64_t)(tbase + (uint32_t)__popc(valid & below)) | ((uint64_t)(uint32_t)lane << 32);
        tmask &= low;
      }
      n += m;
      continue;
    }
    wave_lds_order();
    if ((uint32_t)lane < n) {
      const uint64_t e = W.list[lane];
      const uint32_t i = (uint32_t)e, own = (uint32_t)(e >> 32);
      const float4* T = sc.tris8 + 3 * (size_t)i;
      const float4 a = T[0], b = T[1], c = T[2];
      const f3 o2 = mk3(W.ray[0][own], W.ray[1][own], W.ray[2][own]);
      const f3 d = mk3(W.ray[3][own], W.ray[4][own], W.ray[5][own]);
      // all of the triangle in one round trip, not its vertex in a second one
      asm volatile("" : : "v"(a.x), "v"(a.y), "v"(a.z));
      float u = 0.f, v = 0.f;
      const float t = isect_tri(o2, d, ld3(a), ld3(b), ld3(c), cull, u, v);
      if (t >= 0.f && t != kInfF) {                 // kInfF: missed
        // t + 0: a hit at -0 orders as 0
        const uint64_t key = ((uint64_t)__float_as_uint(t + 0.f) << 32) | (__float_as_uint(a.w) + 1u);
        __hip_atomic_fetch_min(&W.best[own], key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
        wave_lds_order();
        if (W.best[own] == key) {                   // each triangle is tested once per ray: one winner
          W.rec[0][own] = __float_as_uint(t);
          W.rec[1][own] = __float_as_uint(u);
          W.rec[2][own] = __float_as_uint(v);
          W.rec[3][own] = __float_as_uint(b.w);
        }
      }
    }
    wave_lds_order();
    if (m == 0u) break;
    n = 0;
  }
}

// One step of the wave's active rays: a node visit each, the wave's triangle
// tests, and each ray's next node: the nearest interior child hit, the others
// pushed as one group (with the second nearest's distance), or else the first
// child left of the top group that is still in front of the best hit.  Lanes
// without a ray run the box tests on nothing (a branch round them
// costs two dozen moves of their results) and take part in the triangle tests.
// Clears `active` of the rays that finish.  spill (an LDS word of the wave, or
// null) counts group pushes below the LDS top, into the private (scratch)
// stack.
template <bool ANY, int STK>
__device__ __forceinline__ void ray8_step(const DevScene& sc, Ray8& R, bool& active, bool cull, Wave8<STK>& W,
                                          LdsU64* stk, uint64_t* pstk, int lane, uint32_t& nn, uint32_t& nt,
                                          uint32_t* spill) {
  float tn[8];
  uint4 A, B;
  const uint32_t hits =
      box8((const char*)sc.nodes8, R.node, R, R.ht + cull_slack(R.ht, R.eps), tn, A, B, active);
  const uint32_t imask = A.w >> 24;
  // the four triangle bits of each slot hit
  uint32_t x = active ? hits : 0u;
  x = (x | (x << 12)) & 0x000F000Fu;
  x = (x | (x << 6)) & 0x03030303u;
  x = (x | (x << 3)) & 0x11111111u;
  const uint32_t tmask = ((x << 4) - x) & B.z;
  nn += active ? 1u : 0u;
  nt += (uint32_t)__popc(tmask);
  if (__ballot(tmask != 0u)) {
    test_pairs(sc, W, lane, tmask, B.z, B.y, cull);
    const uint64_t best = W.best[lane];
    if (ANY) {
      if ((uint32_t)best != 0u) active = false;
    } else if (active) {
      R.ht = __uint_as_float((uint32_t)(best >> 32));
    }
  }
  if (active) {
    const uint32_t inner = hits & imask;
    if (inner) {
      // the two smallest entry distances, the child's slot in the low three bits
      uint32_t k[8];
#pragma unroll
      for (int c = 0; c < 8; c++)
        k[c] = ((__float_as_uint(tn[c]) & ~7u) | (uint32_t)c) |
               (uint32_t)((int32_t)(~inner << (31 - c)) >> 31);
      uint32_t m1 = min(k[0], k[1]), m2 = max(k[0], k[1]);
#pragma unroll
      for (int c = 2; c < 8; c += 2) {
        const uint32_t lo = min(k[c], k[c + 1]), hi = max(k[c], k[c + 1]);
        m2 = min(m2, max(min(m1, hi), lo));         // the median of m1, lo <= hi
        m1 = min(m1, lo);
      }
      const uint32_t s = m1 & 7u;
      R.node = B.x + (uint32_t)__popc(imask & ((1u << s) - 1u));
      uint32_t rest = inner & ~(1u << s);
      if (rest) {
        if (!(R.idir.x >= 0.f)) rest = ((rest & 0x55u) << 1) | ((rest >> 1) & 0x55u);
        if (!(R.idir.y >= 0.f)) rest = ((rest & 0x33u) << 2) | ((rest >> 2) & 0x33u);
        if (!(R.idir.z >= 0.f)) rest = ((rest & 0x0Fu) << 4) | (rest >> 4);
        const uint64_t e = (uint64_t)B.x | ((uint64_t)((m2 & 0xFFFF0000u) | (imask << 8) | rest) << 32);
        if (R.sp < STK) {
          stk[R.sp * 64] = e;
        } else {
          pstk[R.sp - STK] = e;
          if (spill) atomicAdd(spill, 1u);
        }
        R.sp++;
      }
    } else {
      const float lim = R.ht + cull_slack(R.ht, R.eps);
      for (;;) {
        if (R.sp == 0) { active = false; break; }
        uint64_t e;
        if (R.sp <= STK) e = stk[(R.sp - 1) * 64]; else e = pstk[R.sp - 1 - STK];
        const uint32_t w = (uint32_t)(e >> 32);
        if (__uint_as_float(w & 0xFFFF0000u) > lim) { R.sp--; continue; }
        const uint32_t oct = (R.idir.x >= 0.f ? 0u : 1u) | (R.idir.y >= 0.f ? 0u : 2u) | (R.idir.z >= 0.f ? 0u : 4u);
        const uint32_t s = (uint32_t)__builtin_ctz(w) ^ oct;
        R.node = (uint32_t)e + (uint32_t)__popc((w >> 8) & 0xFFu & ((1u << s) - 1u));
        const uint32_t left = w & (w - 1u);
        if (left & 0xFFu) {
          if (R.sp <= STK) stk[(R.sp - 1) * 64] = (uint64_t)(uint32_t)e | ((uint64_t)left << 32);
          else pstk[R.sp - 1 - STK] = (uint64_t)(uint32_t)e | ((uint64_t)left << 32);
        } else {
          R.sp--;
        }
        break;
      }
    }
  }
}

// Private stack entries below an STK-entry LDS top.
template <int STK>
constexpr int kPriv8 = (int)kMaxDepth8 - STK;

// Closest (ANY: any) hit of the wave's rays, one per active lane.  Called by
// the whole wave.
template <bool ANY, int STK>
__device__ bool trace8(const DevScene& sc, Wave8<STK>& W, bool active, f3 o, f3 d, float maxd, float eps, bool cull,
                       TraceHit& h, uint32_t& nn, uint32_t& nt) {
  const int lane = threadIdx.x & 63;
  uint64_t pstk[kPriv8<STK>];
  Ray8 R = {};                                      // lanes without a ray visit the root
  const bool traced = active;
  if (active) ray8_begin(R, W, lane, o, d, maxd, eps, sc.qmag);
  while (__ballot(active))
    ray8_step<ANY, STK>(sc, R, active, cull, W, (LdsU64*)&W.stk[0][lane], pstk, lane, nn, nt, nullptr);
  return traced && ray8_hit(W, lane, h);
}

// LDS of a workgroup's traversals: 8-wide (Q) or 4-wide nodes.  STK is the
// traversal variant's stack entries; a group entry stands for up to seven
// nodes, so the 8-wide top takes fewer (six: six workgroups fit a compute
// unit's LDS).
template <int STK>
constexpr int kStk8 = STK == 8 ? 6 : STK == 16 ? 10 : 14;
template <int STK, bool Q>
struct TravLds;
template <int STK>
struct TravLds<STK, true> {
  Wave8<kStk8<STK>> w[kBlock / 64];
};
template <int STK>
struct TravLds<STK, false> {
  uint64_t stk[STK * kBlock];
};
// Closest (ANY: any) hit of every active thread's ray.  Called by whole waves.
template <bool ANY, int STK, bool Q>
__device__ __forceinline__ bool trace_rays(const DevScene& sc, TravLds<STK, Q>& L, bool active, f3 o, f3 d,
                                           float maxd, float eps, bool cull, TraceHit& h, uint32_t& nn,
                                           uint32_t& nt) {
  if constexpr (Q)
    return trace8<ANY>(sc, L.w[__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)], active, o, d, maxd, eps, cull, h,
                       nn, nt);
  else
    return active && traverse4<ANY, STK>(sc, o, d, maxd, eps, cull, lds_column(L.stk), h, nn, nt);
}

// Same query over the reference's binary layout (right child popped first).
template <bool ANY>
__device__ bool traverse_bin(const DevScene& sc, f3 o, f3 d, float maxd, float eps, bool cull, TraceHit& h,
                             uint32_t& nn, uint32_t& nt) {
  const f3 idir = mk3(1.f / escape_zero(d.x), 1.f / escape_zero(d.y), 1.f / escape_zero(d.z));
  const f3 o2 = o + d * eps;
  h.t = maxd; h.u = h.v = 0.f; h.leaf = kInvalid; h.orig = kInvalid;
  uint32_t stk[64];
  int sp = 0;
  stk[0] = 0;
  while (sp >= 0) {
    uint32_t n = stk[sp--];
    float4 mn = sc.bnodes[2 * n], mx = sc.bnodes[2 * n + 1];
    uint2 off = sc.boff[n];
    nn++;
    float t0x = (mn.x - o.x) * idir.x, t1x = (mx.x - o.x) * idir.x;
    float t0y = (mn.y - o.y) * idir.y, t1y = (mx.y - o.y) * idir.y;
    float t0z = (mn.z - o.z) * idir.z, t1z = (mx.z - o.z) * idir.z;
    float tnear = fmaxf(fmaxf(fminf(t0x, t1x), fminf(t0y, t1y)), fmaxf(fminf(t0z, t1z), 0.f));
    float tfar = fminf(fminf(fmaxf(t0x, t1x), fmaxf(t0y, t1y)), fmaxf(t0z, t1z)) * 1.0000004f;
    if (!(tnear <= tfar && tnear <= h.t + cull_slack(h.t, eps))) continue;
    if (off.y == 0) {
      if (mn.x > mx.x) continue;                     // empty leaf of a degenerate split
      if (sp < 62) { stk[++sp] = n + 1; stk[++sp] = n + off.x; }
    } else {
      test_leaf(sc.tris_bin, off.x, off.y, o2, d, cull, h, nt);
      if (ANY && h.leaf != kInvalid) return true;
    }
  }
  return h.leaf != kInvalid;
}

// ---- the BVH debug renderer's depth queries ---------------------------------
// CURay::IntersectAABB (src/cudaRTCommon.cu:24-40) as written: the entry
// distance (0 within M_EPSILON of the origin), kInfF on a miss.
__device__ __forceinline__ float ref_aabb(f3 o, f3 rcp, float4 mn, float4 mx) {
  const float t0x = (mn.x - o.x) * rcp.x, t1x = (mx.x - o.x) * rcp.x;
  const float t0y = (mn.y - o.y) * rcp.y, t1y = (mx.y - o.y) * rcp.y;
  const float t0z = (mn.z - o.z) * rcp.z, t1z = (mx.z - o.z) * rcp.z;
  const float minmax = fminf(fminf(fmaxf(t0x, t1x), fmaxf(t0y, t1y)), fmaxf(t0z, t1z));
  const float maxmin = fmaxf(fmaxf(fminf(t0x, t1x), fminf(t0y, t1y)), fminf(t0z, t1z));
  if (minmax >= maxmin && (minmax > 0.f || maxmin > 0.f)) return ((double)maxmin > 1e-9) ? maxmin : 0.f;
  return kInfF;
}
// TraceDepth / TraceDepthParent (src/cudaRTCommon.cu:129-231) as written, over
// the reference's binary tree: right child popped first, a 32-entry command
// stack, at most 2048 pops.  spec == 0xFFFFFFFF: TraceDepth, out = {hit,
// depth, leaf}; otherwise TraceDepthParent(spec), out = {hit, depth
// (0xFFFFFFFF for -1), parent node}.
__global__ __launch_bounds__(kBlock) void k_bvh_depth(DevScene sc, const float4* __restrict__ rays, uint32_t n,
                                                      uint32_t spec, uint32_t* __restrict__ out) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const float4 a = rays[2 * i], b = rays[2 * i + 1];
  const f3 o = ld3(a), d = ld3(b);
  const f3 rcp = mk3(1.f / escape_zero(d.x), 1.f / escape_zero(d.y), 1.f / escape_zero(d.z));
  float minI = a.w;
  uint32_t cmd[32], par[32], dep[32];
  cmd[0] = 0; par[0] = 0; dep[0] = 0;
  int sp = 0;
  uint32_t traced = 0;
  uint32_t r0 = 0, r1 = 0, r2 = 0;
  if (spec == 0xFFFFFFFFu) {
    uint32_t depth = 0;
    bool leaf = false;
    while (sp >= 0 && traced++ < 2048u) {
      const uint32_t nd = cmd[sp--];
      const float tb = ref_aabb(o, rcp, sc.bnodes[2 * nd], sc.bnodes[2 * nd + 1]);
      if (tb >= 0.f && tb < minI) {
        const uint2 off = sc.boff[nd];
        if (off.y == 0) {
          if (sp < 30) { cmd[++sp] = nd + 1; cmd[++sp] = nd + off.x; }
        } else {
          leaf = true; minI = tb; depth = (uint32_t)(sp + 2);
        }
      } else {
        depth = max(depth, (uint32_t)(sp + 1));
      }
    }
    r0 = depth != 0; r1 = depth; r2 = leaf;
  } else {
    int depth = -1;
    uint32_t parent = 0;
    bool any = false;
    while (sp >= 0 && traced++ < 2048u) {
      const int cp = sp--;
      const uint32_t nd = cmd[cp];
      const float tb = ref_aabb(o, rcp, sc.bnodes[2 * nd], sc.bnodes[2 * nd + 1]);
      if (tb >= 0.f && tb < minI) {
        any = true;
        const uint32_t cd = dep[cp];
        if (spec == cd) { minI = tb; depth = (int)cd; parent = par[cp]; break; }
        const uint2 off = sc.boff[nd];
        if (off.y == 0 && sp < 30) {
          ++sp; cmd[sp] = nd + 1; par[sp] = nd; dep[sp] = cd + 1;
          ++sp; cmd[sp] = nd + off.x; par[sp] = nd; dep[sp] = cd + 1;
        }
      }
    }
    r0 = any; r1 = any ? (uint32_t)depth : 0xFFFFFFFFu; r2 = any ? parent : 0u;
  }
  out[3 * i] = r0;
  out[3 * i + 1] = r1;
  out[3 * i + 2] = r2;
}
hipError_t launch_bvh_depth(const DevScene& sc, const float4* rays, uint32_t n, uint32_t spec, uint32_t* out,
                            hipStream_t st) {
  if (n == 0) return hipSuccess;
  if (!rays || !out || !sc.bnodes || !sc.boff) return hipErrorInvalidValue;
  k_bvh_depth<<<(n + kBlock - 1) / kBlock, kBlock, 0, st>>>(sc, rays, n, spec, out);
  return hipGetLastError();
}

__device__ __forceinline__ DevStats* stat_slot(DevStats* stats) { return stats + blockIdx.x % kStatSlots; }
__device__ __forceinline__ uint32_t wave_sum(uint32_t v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Host-side guards: a launch never receives a null buffer it will index.
static bool pathbuf_ok(const PathBuf& b) {
  return b.ray_o && b.ray_d && b.pix && b.sid && b.depth && b.mul && b.smp && b.acc && b.rng;
}
static bool nodes_ok(const DevScene& sc, int quant) { return quant ? sc.nodes8 && sc.tris8 : sc.nodes4 != nullptr; }
static bool rec_ok(const SampleRec& r) { return r.acc && r.gpos && r.gnrm && r.gdif; }

// ---------------------------------------------------------------- scene records
// Filled here: the host would gather 48 and 36 bytes a triangle and send 80 over the
// bus (heightfield of 1,050,976 triangles: upload 129 ms so, 105 here).
__global__ __launch_bounds__(kBlock) void k_tri_records(const float4* __restrict__ tris,
                                                        const uint4* __restrict__ tri_verts,
                                                        const float4* __restrict__ vpos, uint32_t n,
                                                        const uint32_t* __restrict__ order8, uint32_t n8,
                                                        float4* __restrict__ tris8, float4* __restrict__ tri_box) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) {
    const uint4 v = tri_verts[i];
    const f3 a = ld3(vpos[v.x]), b = ld3(vpos[v.y]), c = ld3(vpos[v.z]);
    tri_box[2 * (size_t)i] =
        make_float4(fminf(c.x, fminf(b.x, a.x)), fminf(c.y, fminf(b.y, a.y)), fminf(c.z, fminf(b.z, a.z)), 0.f);
    tri_box[2 * (size_t)i + 1] =
        make_float4(fmaxf(c.x, fmaxf(b.x, a.x)), fmaxf(c.y, fmaxf(b.y, a.y)), fmaxf(c.z, fmaxf(b.z, a.z)), 0.f);
  }
  if (i < n8) {
    const uint32_t leaf = order8[i];
    const float4* T = tris + 3 * (size_t)leaf;
    float4 e0 = T[1];
    e0.w = __uint_as_float(leaf);
    tris8[3 * (size_t)i] = T[0];
    tris8[3 * (size_t)i + 1] = e0;
    tris8[3 * (size_t)i + 2] = T[2];
  }
}
hipError_t launch_tri_records(const float4* tris, const uint4* tri_verts, const float4* vpos, uint32_t n,
                              const uint32_t* order8, uint32_t n8, float4* tris8, float4* tri_box, hipStream_t st) {
  if (n == 0) return hipSuccess;
  if (!tris || !tri_verts || !vpos || !tri_box || n8 > n || (n8 && (!order8 || !tris8))) return hipErrorInvalidValue;
  k_tri_records<<<(n + kBlock - 1) / kBlock, kBlock, 0, st>>>(tris, tri_verts, vpos, n, order8, n8, tris8, tri_box);
  return hipGetLastError();
}

// ---------------------------------------------------------------- trace API
// out mode 0: cpt_hit {orig id, t, u, v}; 1: {t, leaf bits, u, v}; 2: occluded flag.
// MINW: minimum resident waves per SIMD requested from the register allocator
// (0 = compiler default).
template <int LAYOUT, bool ANY, int OUT, int STK = CPT_LDS_STACK, int MINW = 0>
__global__ __launch_bounds__(kBlock, MINW) void k_trace(DevScene sc, const float4* __restrict__ ro,
                                                  const float4* __restrict__ rd, uint32_t stride,
                                                  const uint32_t* __restrict__ countp, uint32_t n, uint32_t cull,
                                                  float4* __restrict__ out, DevStats* __restrict__ stats) {
  __shared__ TravLds<STK, LAYOUT == 2> lds;
  uint32_t count = countp ? *countp : n;
  uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  uint32_t nn = 0, nt = 0;
  float4 a = make_float4(0.f, 0.f, 0.f, 0.f), b = a;
  if (i < count) {
    a = ro[(size_t)i * stride];
    b = rd[(size_t)i * stride];
  }
  TraceHit h;
  bool hit = false;
  if constexpr (LAYOUT == 1) {
    if (i < count) hit = traverse_bin<ANY>(sc, ld3(a), ld3(b), a.w, b.w, cull != 0, h, nn, nt);
  } else {
    hit = trace_rays<ANY, STK, LAYOUT == 2>(sc, lds, i < count, ld3(a), ld3(b), a.w, b.w, cull != 0, h, nn, nt);
  }
  if (i < count) {
    if (OUT == 0) {
      float4 r;
      r.x = __uint_as_float(hit ? h.orig : kInvalid);
      r.y = hit ? h.t : kInfF;
      r.z = hit ? h.u : 0.f;
      r.w = hit ? h.v : 0.f;
      out[i] = r;
    } else if (OUT == 1) {
      float4 r;
      r.x = hit ? h.t : kInfF;
      r.y = __uint_as_float(hit ? h.leaf : kInvalid);
      r.z = hit ? h.u : 0.f;
      r.w = hit ? h.v : 0.f;
      out[i] = r;
    } else if (OUT == 2) {
      ((uint32_t*)out)[i] = hit ? 1u : 0u;
    } else {
      ((uint2*)out)[i] = make_uint2(nn, nt);      // this ray's node visits and triangle tests
    }
  }
  if (stats) {
    stats = stat_slot(stats);
    uint32_t sn = wave_sum(nn), st = wave_sum(nt);
    if ((threadIdx.x & 63) == 0 && (sn | st)) {
      atomicAdd(&stats->ext_nodes, (unsigned long long)sn);
      atomicAdd(&stats->ext_tris, (unsigned long long)st);
    }
  }
}

hipError_t launch_trace(const DevScene& sc, const float4* rays, uint32_t n, uint32_t cull, float4* out, int any_hit,
                        uint32_t layout, int cost, DevStats* stats, hipStream_t st) {
  if (n == 0) return hipSuccess;
  dim3 grid((n + kBlock - 1) / kBlock), block(kBlock);
  if (layout == 2 && !sc.nodes8) layout = 0;       // not every scene has 8-wide nodes (collapse_bvh8)
  if (layout > 2 || (layout == 2 && !sc.tris8) || (layout == 0 && !sc.nodes4)) return hipErrorInvalidValue;
  // hits and flags over the 8-wide nodes are launch_trace_rays', flags over binary ones nobody's
  if (!cost && (any_hit ? layout != 0 : layout == 2)) return hipErrorInvalidValue;
#define CPT_TR(L, A, O) k_trace<L, A, O><<<grid, block, 0, st>>>(sc, rays, rays + 1, 2, nullptr, n, cull, out, stats)
  if (cost) {
    if (layout == 0) CPT_TR(0, false, 3); else if (layout == 2) CPT_TR(2, false, 3); else CPT_TR(1, false, 3);
  } else if (any_hit) {
    CPT_TR(0, true, 2);
  } else {
    if (layout == 0) CPT_TR(0, false, 0); else CPT_TR(1, false, 0);
  }
#undef CPT_TR
  return hipGetLastError();
}

// ---------------------------------------------------------------- shading
// src/cudaRTCommon.cu:284-365 with the reference's mixed float/double
// expressions (M_PI and the bias epsilons are double literals there).
__device__ __forceinline__ bool prob_rand(uint64_t& st, uint64_t inc, float prob) {
  if ((double)prob < kBiasEps) return false;
  if ((double)prob + kBiasEps > 1.0) return true;
  return uniform01(st, inc) < prob;
}
__device__ __forceinline__ float vis_smith(float r, float nov, float nol) {
  float k = (r * r) / 2.f;
  return (nov / (nov * (1.f - k) + k)) * (nol / (nol * (1.f - k) + k));
}
__device__ __forceinline__ float d_ggx(float r, float noh) {
  float m = r * r, m2 = m * m;
  float d = (noh * m2 - noh) * noh + 1.f;
  return (float)((double)m2 / (kPiD * (double)d * (double)d));
}
// x^5 of Schlick's term: the power in double (x^2 exact, x^4 and x^5 rounded
// at 2^-53) rounded once to float, the correctly rounded x^5 except within
// ~2^-51 of a rounding boundary (the reference's powf is within an ulp of it);
// a few instructions where a general powf takes dozens.
__device__ __forceinline__ float pow5f(float x) {
  const double d = (double)x, d2 = d * d;
  return (float)(d2 * d2 * d);
}
__device__ __forceinline__ f3 f_schlick(f3 s, float voh) {
  float fc = pow5f(1.f - voh);
  double z = 50.0 * (double)s.z;
  float first = (float)(z < 0.0 ? 0.0 : (z > 1.0 ? 1.0 : z)) * fc;
  return mk3(first, first, first) + s * (1.f - fc);
}
__device__ __forceinline__ void basis(f3 w, f3& u, f3& v) {
  f3 a = (double)fabsf(w.x) > 0.1 ? mk3(0.f, 1.f, 0.f) : mk3(1.f, 0.f, 0.f);
  u = normalize(cross(a, w));
  v = cross(w, u);
  u = cross(v, w);
}
// (u, v, n): the tangent frame basis(n) gives.
__device__ __forceinline__ f3 sample_ggx(float xi0, float xi1, float rough, f3 n, f3 u, f3 v) {
  float a = rough * rough;
  float phi = (float)(2.0 * kPiD * (double)xi0);
  float ct = sqrtf((1.f - xi1) / (1.f + (a * a - 1.f) * xi1));
  float st = sqrtf(1.f - ct * ct);
  float sp, cp;
  sincos_def(phi, sp, cp);
  f3 h = mk3(st * cp, st * sp, ct);
  return (u * h.x + v * h.y) + n * h.z;
}
__device__ __forceinline__ f3 lambert(f3 diff) { return diff * (float)(1.0 / kPiD); }
// GetShadingResult (src/cudaRTBDPTStream.cu:642-663)
__device__ __forceinline__ f3 shading(f3 outDir, f3 inDir, f3 irrad, f3 n, f3 diff, float metal, float rough,
                                      float spec, float dw, float sw) {
  if (dot(n, inDir) <= 0.f) return mk3(0.f, 0.f, 0.f);
  f3 h = normalize(outDir + inDir);
  float voh = dot(outDir, h), nov = dot(n, outDir), noh = dot(n, h), nol = dot(n, inDir);
  f3 f0 = vlerp(mk3(1.f, 1.f, 1.f) * (0.08f * spec), diff, metal);
  f3 F = f_schlick(f0, voh);
  float dd = d_ggx(rough, noh), vv = vis_smith(rough, nov, nol);
  f3 specI = F * (dd * vv);
  f3 diffI = vmul(mk3(1.f, 1.f, 1.f) - F, lambert(diff));
  return vmul(irrad * nol, specI * sw + diffI * dw);
}

struct Surf {
  f3 norm, pos, diff, emissive;
  float trans, spec, metal, rough;
};
// tex2D of a float4 texture with normalized coordinates, wrap addressing and
// linear filtering (the reference's texture objects, src/cudaRTCommon.cu:416-441):
// the coordinate wraps to [0, 1), scales to texels, and the four texels around
// x - 0.5, y - 0.5 (indices wrapped) are blended in x, then in y.
__device__ __forceinline__ float4 tex_sample(const DevScene& sc, uint32_t id, float u, float v) {
  const uint4 d = sc.tex_desc[id];
  const int W = (int)d.y, H = (int)d.z;
  if (!(fabsf(u) < 1e30f)) u = 0.f;                 // NaN and infinities sample texel (0, 0)
  if (!(fabsf(v) < 1e30f)) v = 0.f;
  const float fu = u - floorf(u), fv = v - floorf(v);
  const float x = fu * (float)W - 0.5f, y = fv * (float)H - 0.5f;
  const float fx = floorf(x), fy = floorf(y);
  const float a = x - fx, b = y - fy;
  int i0 = min(max((int)fx, -1), W - 1), j0 = min(max((int)fy, -1), H - 1);
  if (i0 < 0) i0 += W;
  if (j0 < 0) j0 += H;
  const int i1 = i0 + 1 == W ? 0 : i0 + 1, j1 = j0 + 1 == H ? 0 : j0 + 1;
  const float4 t00 = sc.tex[d.x + (uint32_t)(j0 * W + i0)], t10 = sc.tex[d.x + (uint32_t)(j0 * W + i1)];
  const float4 t01 = sc.tex[d.x + (uint32_t)(j1 * W + i0)], t11 = sc.tex[d.x + (uint32_t)(j1 * W + i1)];
  const float ia = 1.f - a, ib = 1.f - b;
  float4 r;
  r.x = (t00.x * ia + t10.x * a) * ib + (t01.x * ia + t11.x * a) * b;
  r.y = (t00.y * ia + t10.y * a) * ib + (t01.y * ia + t11.y * a) * b;
  r.z = (t00.z * ia + t10.z * a) * ib + (t01.z * ia + t11.z * a) * b;
  r.w = (t00.w * ia + t10.w * a) * ib + (t01.w * ia + t11.w * a) * b;
  return r;
}

// Shading inputs at a hit: interpolated normal (and position), material, and
// GetMaterialColors' textures (src/cudaRTCommon.cu:369-406): a diffuse texture
// gives the colour and scales transparency by its alpha, an emissive texture
// gives the emission; texture ids outside the scene's textures mean none.
// The hit's surface from its triangle's 128-byte shading record: normals and
// material in one round trip after the hit; texture u and the vertex positions
// only for textured materials and first-hit G-buffers.
// Radiance the environment sends along direction d (no reference counterpart:
// the reference lights scenes with emissive triangles only).  Latitude-longitude
// map: u = atan2(d.z, d.x) / 2pi + 1/2, v = acos(d.y) / pi, texel centres at
// half-integers, bilinear between the four around (u W - 1/2, v H - 1/2), u
// wrapping and v clamped to the first and last rows.  A non-finite d sees 0.
__device__ __forceinline__ f3 env_radiance(const DevScene& sc, f3 d) {
  const int W = (int)sc.env_w, H = (int)sc.env_h;
  const float u = atan2_def(d.z, d.x) * (float)(0.5 / kPiD) + 0.5f;
  const float v = acos_def(fminf(fmaxf(d.y, -1.f), 1.f)) * (float)(1.0 / kPiD);
  const float x = u * (float)W - 0.5f, y = v * (float)H - 0.5f;
  if (!(fabsf(x) < 1e30f) || !(fabsf(y) < 1e30f)) return mk3(0.f, 0.f, 0.f);
  const float fx = floorf(x), fy = floorf(y);
  const float a = x - fx, b = y - fy;
  int i0 = (int)fx % W;
  if (i0 < 0) i0 += W;
  const int i1 = i0 + 1 == W ? 0 : i0 + 1;
  const int j0 = min(max((int)fy, 0), H - 1), j1 = min(max((int)fy + 1, 0), H - 1);
  const float4 t00 = sc.env[j0 * W + i0], t10 = sc.env[j0 * W + i1];
  const float4 t01 = sc.env[j1 * W + i0], t11 = sc.env[j1 * W + i1];
  const float ia = 1.f - a, ib = 1.f - b;
  return mk3((t00.x * ia + t10.x * a) * ib + (t01.x * ia + t11.x * a) * b,
             (t00.y * ia + t10.y * a) * ib + (t01.y * ia + t11.y * a) * b,
             (t00.z * ia + t10.z * a) * ib + (t01.z * ia + t11.z * a) * b);
}

__device__ __forceinline__ Surf fetch_surf(const DevScene& sc, uint32_t leaf, float w, float u, float v, bool want_pos) {
  Surf s;
  const float4* R = sc.surf + 8 * (size_t)leaf;
  const float4 r0 = R[0], r1 = R[1], r2 = R[2], md = R[3], me = R[4], mx = R[5];
  f3 n0 = ld3(r0), n1 = ld3(r1), n2 = ld3(r2);
  s.norm = (n0 * w + n1 * u) + n2 * v;
  const uint32_t dtid = __float_as_uint(mx.z), etid = __float_as_uint(mx.w);
  const bool dtex = dtid < sc.n_tex, etex = etid < sc.n_tex;
  s.diff = ld3(md);
  s.trans = md.w;
  s.emissive = ld3(me);
  if (want_pos) {
    const float4 ix = R[7];
    const float4 p0 = sc.vpos[__float_as_uint(ix.x)], p1 = sc.vpos[__float_as_uint(ix.y)],
                 p2 = sc.vpos[__float_as_uint(ix.z)];
    s.pos = (ld3(p0) * w + ld3(p1) * u) + ld3(p2) * v;
  } else {
    s.pos = mk3(0.f, 0.f, 0.f);
  }
  if (dtex || etex) {
    // uv = uv0 * w + uv1 * u + uv2 * v (cudaRTBDPTStream.cu:379-382)
    const float4 tu4 = R[6];
    const float tu = (tu4.x * w + tu4.y * u) + tu4.z * v, tvv = (r0.w * w + r1.w * u) + r2.w * v;
    if (dtex) {
      const float4 t = tex_sample(sc, dtid, tu, tvv);
      s.diff = mk3(t.x, t.y, t.z);
      s.trans = t.w * md.w;
    }
    if (etex) {
      const float4 t = tex_sample(sc, etid, tu, tvv);
      s.emissive = mk3(t.x, t.y, t.z);
    }
  }
  s.spec = me.w; s.metal = mx.x; s.rough = mx.y;
  return s;
}

enum { RT_EYE = 0, RT_DIFF = 1, RT_SPEC = 2, RT_LIGHT = 3 };
struct Bounce {
  f3 orig, dir, mul;
  int type;
};
// BRDF sample of one bounce (src/cudaRTBDPTStream.cu:228-329 and :402-502).
// tir_reflect: a refraction past the critical angle turns into a reflection
// (the path tracers, cudaRTPTStream.cu:152-160); the BDPT files take the
// refracted direction as computed.
__device__ Bounce sample_bounce(uint64_t& st, uint64_t inc, f3 ro, f3 rd, float t, const Surf& s, f3 nl, int cur,
                                bool refl_offset = false, bool tir_reflect = false) {
  float x0 = uniform01(st, inc), x1 = uniform01(st, inc);
  f3 u, v;                                           // one tangent frame for both samplers
  basis(nl, u, v);
  f3 hDir = sample_ggx(x0, x1, s.rough, nl, u, v);
  f3 ndir = rd * -1.f;
  float voH = dot(ndir, hDir);
  f3 f0 = vlerp(mk3(0.08f * s.spec, 0.08f * s.spec, 0.08f * s.spec), s.diff, s.metal);
  f3 F = f_schlick(f0, voH);
  float reflProb = lerpf(length(F), 1.f, s.metal);
  float refrProb = s.trans;
  f3 reflDir = mk3(0.f, 0.f, 0.f), refrDir = mk3(0.f, 0.f, 0.f);
  Bounce b;
  b.orig = ro; b.dir = rd; b.type = cur; b.mul = mk3(0.f, 0.f, 0.f);
  if (refrProb > 0.f) {
    bool into = dot(nl, s.norm) > 0.f;
    float nt = s.spec * 0.8f + 1.f, nc = 1.f;
    float nnt = into ? nc / nt : nt / nc;
    float ddn = dot(hDir, rd);
    float cos2t = 1.f - nnt * nnt * (1.f - ddn * ddn);
    if (tir_reflect && cos2t < 0.f) reflProb = 1.f;
    else refrDir = normalize(rd * nnt - hDir * (ddn * nnt + sqrtf(cos2t)));
  }
  if (reflProb > 0.f) {
    reflDir = normalize(rd - (hDir * 2.f) * dot(hDir, rd));
    if (dot(reflDir, nl) < 0.f) reflProb = 0.f;
  }
  if (prob_rand(st, inc, reflProb)) {
    b.orig = ro + rd * (float)((double)t - kBiasEps);
    // the adaptive files also step off along the reflection (AdapBilatAtomic.cu:584)
    if (refl_offset) b.orig = b.orig + reflDir * (float)kBiasEps;
    b.dir = reflDir;
    float VoH = dot(ndir, hDir), NoV = dot(nl, ndir), NoH = dot(nl, hDir), NoL = dot(nl, reflDir);
    float G = vis_smith(s.rough, NoV, NoL);
    b.mul = (F * G * VoH) / (NoV * NoH * reflProb);
    b.type = RT_SPEC;
  } else if (prob_rand(st, inc, refrProb)) {
    b.orig = (ro + rd * (float)((double)t + kBiasEps)) + refrDir * (float)kBiasEps;
    b.dir = refrDir;
    float cosine = dot(nl * -1.f, refrDir);
    b.mul = s.diff * cosine / (refrProb * (1.f - reflProb));
    b.type = RT_SPEC;
  } else {
    float r1 = (float)(2.0 * kPiD * (double)uniform01(st, inc));
    float r2cos = sqrtf(uniform01(st, inc));
    float r2sin = 1.f - r2cos * r2cos;
    float s1, c1;
    sincos_def(r1, s1, c1);
    f3 dd = normalize((nl * r2cos + (u * r2sin) * c1) + (v * r2sin) * s1);
    b.orig = (ro + rd * t) + dd * (float)kBiasEps;
    b.dir = dd;
    b.mul = lambert(s.diff) * (float)kPiD / ((1.f - refrProb) * (1.f - reflProb));
    b.type = RT_DIFF;
  }
  return b;
}

__device__ __forceinline__ double shadow_max(double dist, uint32_t flags) {
  return (flags & 1u) ? dist - kBiasEps : dist - 2.0 * kBiasEps;
}

// First frame of the batch: the argument, or the device counter of a replayed graph.
__device__ __forceinline__ uint32_t frame_base(const FrameArgs& fa) {
  return fa.frame_dev ? *fa.frame_dev : fa.frame0;
}

// View of a batch-global pixel (0 without a view table).
__device__ __forceinline__ uint32_t view_of(const FrameArgs& fa, uint32_t pix) {
  uint32_t lo = 0, hi = fa.n_views;
  while (hi - lo > 1) {
    uint32_t mid = (lo + hi) >> 1;
    if (fa.views[mid].offset <= pix) lo = mid; else hi = mid;
  }
  return lo;
}
// The pixel's index within its view: the PCG32 stream of an eye path is keyed
// by it, so every view of a batch traces the samples a one-view renderer would.
__device__ __forceinline__ uint32_t local_pixel(const FrameArgs& fa, uint32_t pix) {
  return fa.views ? pix - fa.views[view_of(fa, pix)].offset : pix;
}

// ---------------------------------------------------------------- frame
__global__ void k_fill_u32(uint32_t* p, uint32_t v) { *p = v; }
__global__ void k_fill_n_u32(uint32_t* p, uint32_t n, uint32_t v) {
  for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) p[i] = v;
}
__global__ void k_queues_clear(uint32_t* queue) {
  queue[threadIdx.x * kDealStride] = 0u;
}
hipError_t launch_queues_clear(uint32_t* queue, hipStream_t st) {
  k_queues_clear<<<1, kQueues * kDealers, 0, st>>>(queue);
  return hipGetLastError();
}
__global__ void k_frame_begin(FrameCounters* fc, uint32_t n_paths) {
  uint32_t i = threadIdx.x;
  if (i < 16) { fc->active[i] = i == 0 ? n_paths : 0u; fc->shadow[i] = 0u; }
}
hipError_t launch_frame_begin(FrameCounters* fc, uint32_t n_paths, hipStream_t st) {
  k_frame_begin<<<1, 64, 0, st>>>(fc, n_paths);
  return hipGetLastError();
}
__global__ void k_frame_begin_dev(FrameCounters* fc, const uint32_t* total, uint32_t cap) {
  uint32_t i = threadIdx.x;
  uint32_t t = *total;
  if (i < 16) { fc->active[i] = i == 0 ? (t < cap ? t : cap) : 0u; fc->shadow[i] = 0u; }
}
hipError_t launch_frame_begin_dev(FrameCounters* fc, const uint32_t* total, uint32_t cap, hipStream_t st) {
  k_frame_begin_dev<<<1, 64, 0, st>>>(fc, total, cap);
  return hipGetLastError();
}

// n_whole > 0: every one of the frame's n_whole paths was carried whole and no
// frame_begin ran: the counters are set here, from the parts alone.
__global__ void k_frame_end(FrameCounters* fc, DevStats* stats, uint32_t nframes, uint32_t depth, int parts,
                            uint32_t n_whole) {
  const uint32_t c = threadIdx.x & 31u, half = threadIdx.x >> 5;   // 32 counters, two threads each
  uint32_t v = 0;
  if (parts) {
#pragma unroll 8
    for (uint32_t s = half; s < kPartSlots; s += 2) {
      v += fc->part[s][c];
      fc->part[s][c] = 0u;
    }
    v += __shfl_xor(v, 32, 64);
  }
  uint32_t* at = c < 16 ? &fc->active[c] : &fc->shadow[c - 16];
  const uint32_t f = v + (n_whole ? (c == 0 ? n_whole : 0u) : *at);
  if (half == 0) *at = f;
  const bool counts = half == 0 && (c & 15u) < depth;
  const auto sum = [](uint32_t x) {                 // 64 bits: the bounces' counts together may pass 32
    return (unsigned long long)wave_sum(x & 0xFFFFu) + ((unsigned long long)wave_sum(x >> 16) << 16);
  };
  const unsigned long long e = sum(counts && c < 16 ? f : 0u), s = sum(counts && c >= 16 ? f : 0u);
  if (threadIdx.x == 0) {
    stats->ext_rays += e;
    stats->shadow_rays += s;
    stats->eye_paths += f;
    stats->frames += nframes;
  }
}
hipError_t launch_frame_end(FrameCounters* fc, DevStats* stats, uint32_t nframes, uint32_t depth, int parts,
                            uint32_t n_whole, hipStream_t st) {
  k_frame_end<<<1, 64, 0, st>>>(fc, stats, nframes, depth, parts, n_whole);
  return hipGetLastError();
}
__global__ void k_frame_advance(uint32_t* frame_dev, uint32_t k) {
  if (threadIdx.x == 0) *frame_dev += k;
}
hipError_t launch_frame_advance(uint32_t* frame_dev, uint32_t k, hipStream_t st) {
  if (!frame_dev) return hipErrorInvalidValue;
  k_frame_advance<<<1, 64, 0, st>>>(frame_dev, k);
  return hipGetLastError();
}

__device__ __forceinline__ void store_lv(LightVert& V, f3 pos, f3 norm, f3 irrad, f3 irradDir, const Surf& s) {
  V.pos[0] = pos.x; V.pos[1] = pos.y; V.pos[2] = pos.z;
  V.norm[0] = norm.x; V.norm[1] = norm.y; V.norm[2] = norm.z;
  V.irrad[0] = irrad.x; V.irrad[1] = irrad.y; V.irrad[2] = irrad.z;
  V.irradDir[0] = irradDir.x; V.irradDir[1] = irradDir.y; V.irradDir[2] = irradDir.z;
  V.diff[0] = s.diff.x; V.diff[1] = s.diff.y; V.diff[2] = s.diff.z;
  V.emissive[0] = s.emissive.x; V.emissive[1] = s.emissive.y; V.emissive[2] = s.emissive.z;
  V.specular = s.spec; V.metallic = s.metal; V.roughness = s.rough;
  V.pad[0] = V.pad[1] = V.pad[2] = 0.f;
}

// Light-vertex caches, one workgroup per cache slot to build (light_paths <= kBlock).
template <bool Q>
__global__ __launch_bounds__(kBlock) void k_light_pass(DevScene sc, FrameArgs fa, LightJobs jobs,
                                                       LightVert* __restrict__ lv_all,
                                                       FrameCounters* __restrict__ fc) {
  __shared__ TravLds<8, Q> lds;
  __shared__ uint32_t wcnt[kBlock / 64];
  const uint32_t x = threadIdx.x, L = fa.light_paths;
  uint32_t slot, job_frame;
  if (jobs.dev_groups) {                       // groups of the device-counted batch
    const uint32_t f0 = frame_base(fa), g = f0 / 3u + blockIdx.x;
    if (g > (f0 + fa.nframes - 1u) / 3u) return;
    slot = g % (uint32_t)kLightSlots;
    job_frame = 3u * g;
  } else {
    slot = jobs.slot[blockIdx.x];
    job_frame = jobs.frame[blockIdx.x];
  }
  LightVert* __restrict__ lv = lv_all + (size_t)slot * fa.lv_stride;
  const uint64_t light_key = stream_key(fa.seed, job_frame, 2u, 0u);
  const uint64_t inc = ((uint64_t)x << 1) | 1u;
  uint64_t st = 0;
  bool live = false;
  f3 orig = mk3(0.f, 0.f, 0.f), dir = orig, smp = orig, mul = mk3(1.f, 1.f, 1.f);
  int type = RT_LIGHT;
  uint32_t depth = 0;
  if (sc.n_light_tris == 0) {
    if (x == 0) fc->light_n[slot] = 0;
    return;
  }
  if (x < L) {
    pcg32_seed(st, inc, light_key);
    uint32_t id = (uint32_t)(uniform01(st, inc) * (float)sc.n_light_tris);
    if (id >= sc.n_light_tris) id = sc.n_light_tris - 1;
    float lw = uniform01(st, inc), lu = uniform01(st, inc);
    if (lw + lu > 1.f) { lw = 1.f - lw; lu = 1.f - lu; }
    float lvv = (1.f - lw) - lu;
    Surf s = fetch_surf(sc, sc.light_tris[id], lw, lu, lvv, true);
    f3 u, v;
    basis(s.norm, u, v);
    float r1 = (float)(2.0 * kPiD * (double)uniform01(st, inc));
    float r2cos = sqrtf(uniform01(st, inc));
    float r2sin = 1.f - r2cos * r2cos;
    float s1, c1;
    sincos_def(r1, s1, c1);
    f3 dd = normalize((s.norm * r2cos + (u * r2sin) * c1) + (v * r2sin) * s1);
    orig = s.pos + s.norm * (float)kBiasEps;
    dir = dd;
    smp = s.emissive;
    live = true;
    store_lv(lv[x], s.pos, s.norm, s.emissive, mk3(0.f, 0.f, 0.f), s);
  }
  __syncthreads();
  uint32_t cur = L;
  const int lane = x & 63, wid = x >> 6;
  for (;;) {
    unsigned long long m = __ballot(live);
    uint32_t below = __popcll(m & ((1ull << lane) - 1ull));
    if (lane == 0) wcnt[wid] = __popcll(m);
    __syncthreads();
    uint32_t pre = 0, total = 0;
    for (int w = 0; w < kBlock / 64; w++) { if (w < wid) pre += wcnt[w]; total += wcnt[w]; }
    __syncthreads();
    if (total == 0) break;
    TraceHit h;
    uint32_t nn = 0, nt = 0;
    const bool hit = trace_rays<false, 8, Q>(sc, lds, live, orig, dir, kInfF, (float)kBiasEps, false, h, nn, nt);
    if (live) {
      uint32_t slot = cur + pre + below;
      if (!hit) {
        lv[slot] = lv[x];
        live = false;
      } else {
        float w = (1.f - h.u) - h.v;
        Surf s = fetch_surf(sc, h.leaf, w, h.u, h.v, true);
        f3 nl = dot(s.norm, dir) < 0.f ? s.norm : s.norm * -1.f;
        Bounce b = sample_bounce(st, inc, orig, dir, h.t, s, nl, type);
        f3 irr = b.type != RT_DIFF ? mk3(0.f, 0.f, 0.f) : smp;
        f3 vn = dot(b.dir, nl) < 0.f ? nl * -1.f : nl;
        store_lv(lv[slot], s.pos, vn, irr, dir * -1.f, s);
        smp = s.emissive + vmul(smp, b.mul);
        float contrib = length(mul) * length(b.mul);
        if (length(s.emissive) > 0.f) contrib = 0.f;
        if (uniform01(st, inc) > contrib || depth + 1 >= fa.light_depth) {
          live = false;
        } else {
          mul = vmul(mul, b.mul);
          dir = b.dir;
          orig = b.orig;
          type = b.type;
          depth++;
        }
      }
    }
    cur += total;
    __syncthreads();
  }
  if (x == 0) fc->light_n[slot] = cur;
}
hipError_t launch_light_pass(const DevScene& sc, const FrameArgs& fa, const LightJobs& jobs, LightVert* lv,
                             FrameCounters* fc, int quant, hipStream_t st) {
  if (jobs.n == 0 && jobs.dev_groups == 0) return hipSuccess;
  if (!lv || !sc.tris || !nodes_ok(sc, quant) || !fc || fa.light_paths > (uint32_t)kBlock || (sc.n_light_tris && !sc.light_tris) ||
      jobs.n > (uint32_t)kLightSlots || jobs.dev_groups > (uint32_t)kLightSlots ||
      (jobs.dev_groups && !fa.frame_dev))
    return hipErrorInvalidValue;
  for (uint32_t j = 0; j < jobs.n; j++)
    if (jobs.slot[j] >= (uint32_t)kLightSlots) return hipErrorInvalidValue;
  const uint32_t grid = jobs.dev_groups ? jobs.dev_groups : jobs.n;
  if (quant) k_light_pass<true><<<grid, kBlock, 0, st>>>(sc, fa, jobs, lv, fc);
  else k_light_pass<false><<<grid, kBlock, 0, st>>>(sc, fa, jobs, lv, fc);
  return hipGetLastError();
}

// Running-mean update of pt_applyPathQueueResult_kernel
// (src/cudaRTBDPTStream.cu:754-776); one path per pixel per frame.
__device__ __forceinline__ void apply_pixel(float* result, uint32_t* sample_n, uint32_t pix, uint32_t frame, f3 acc,
                                            uint32_t n) {
  uint32_t nold = frame == 0 ? 0u : sample_n[pix];
  if (frame == 0) sample_n[pix] = 0u;
  uint32_t nn = nold + n;
  if (!(nn > nold) || isinf3(acc)) return;
  float ri = 1.f / (float)nn, oi = (float)nold * ri;
  float* r = result + (size_t)pix * 3;
  r[0] = fmaxf(ri * acc.x + oi * r[0], 0.f);
  r[1] = fmaxf(ri * acc.y + oi * r[1], 0.f);
  r[2] = fmaxf(ri * acc.z + oi * r[2], 0.f);
  sample_n[pix] = nn;
}

// One eye path in registers: the ray (o, max distance; d, epsilon), pixel,
// sample slot, depth, frame offset in the batch, throughput, emission gathered
// so far, the accumulated radiance with its sample count (acc.w, as bits) and
// the RNG state.  PathBuf holds the same fields as columns.
struct PathState {
  float4 ro, rd, mul, smp, acc;
  uint32_t pix, sid, depth, fk;
  uint32_t lim;    // depth bound of this path (0: the frame's eye depth)
  uint32_t type;   // type of the ray being traced (RT_EYE, RT_DIFF, RT_SPEC)
  uint64_t rng;
};
// PathBuf::depth packs depth (bits 0-7), frame offset (8-15), depth bound
// (16-23), ray type (24-25) and kFreshPath: a path k_gen_eye started, whose
// mul / smp / acc columns were not written (throughput 1, nothing gathered).
constexpr uint32_t kFreshPath = 1u << 26;
__device__ __forceinline__ uint32_t pack_dk(const PathState& p) {
  return p.depth | (p.fk << 8) | (p.lim << 16) | (p.type << 24);
}
__device__ __forceinline__ void unpack_dk(PathState& p, uint32_t dk) {
  p.depth = dk & 0xFFu;
  p.fk = (dk >> 8) & 0xFFu;
  p.lim = (dk >> 16) & 0xFFu;
  p.type = (dk >> 24) & 3u;
}
// The connection's shadow ray: origin and max distance, direction and epsilon,
// contribution added to the path's accumulator when nothing occludes it.
// A shadow ray's target slot with this bit set adds its contribution without
// the connection's N += 4 (the Disney mode's light samples are part of their
// path's one sample).  Slots stay below 2^31.
constexpr uint32_t kShadowNoCount = 1u << 31;
struct ShadowRay {
  float4 o, d, c;
};

// Eye ray of pixel (x, y) drawn from PCG32 stream `key`, pixel as sequence
// (pt_genPathQueue_kernel, src/cudaRTBDPTStream.cu:619-640; the adaptive queue
// of AdapBilatAtomic.cu:826-840 uses the same pinhole).  In a multi-view batch
// `pix` is the batch-global pixel: the camera and the pixel's position come
// from its view, the RNG stream stays keyed by the global pixel.
// st: the path's PCG32 state, positioned where the jitter draws start.
__device__ __forceinline__ PathState eye_path_at(const FrameArgs& fa, uint32_t pix, uint32_t sid, uint64_t st) {
  uint32_t lp = pix, vw = fa.width, vh = fa.height;
  const float *cpos = fa.cam_pos, *cdir = fa.cam_dir, *cup = fa.cam_up, *cright = fa.cam_right;
  float tf = fa.tan_half;
  if (fa.views) {
    const ViewDesc& V = fa.views[view_of(fa, pix)];
    lp = pix - V.offset;
    vw = V.width;
    vh = V.height;
    cpos = V.cam_pos; cdir = V.cam_dir; cup = V.cam_up; cright = V.cam_right;
    tf = V.tan_half;
  }
  uint32_t y = lp / vw, x = lp - y * vw;
  float W = (float)vw, H = (float)vh;
  float u = ((((2.f * ((float)x + 0.5f)) / W - 1.f) * tf) * W) / H;
  float v = ((2.f * ((float)y + 0.5f)) / H - 1.f) * tf;
  const uint64_t inc = ((uint64_t)lp << 1) | 1u;
  float au = u + ((uniform01(st, inc) - 0.5f) / H) * tf;
  float av = v + ((uniform01(st, inc) - 0.5f) / H) * tf;
  f3 right = mk3(cright[0], cright[1], cright[2]);
  f3 up = mk3(cup[0], cup[1], cup[2]);
  f3 cd = mk3(cdir[0], cdir[1], cdir[2]);
  f3 d = normalize((right * au + up * av) + cd);
  PathState p;
  p.ro = make_float4(cpos[0], cpos[1], cpos[2], kInfF);
  p.rd = make_float4(d.x, d.y, d.z, (float)kBiasEps);
  p.pix = pix;
  p.sid = sid;
  p.depth = 0;
  p.fk = 0;
  p.lim = 0;
  p.type = RT_EYE;
  p.mul = make_float4(1.f, 1.f, 1.f, 0.f);
  p.smp = make_float4(0.f, 0.f, 0.f, 0.f);
  p.acc = make_float4(0.f, 0.f, 0.f, 0.f);
  p.rng = st;
  return p;
}
__device__ __forceinline__ PathState eye_path(const FrameArgs& fa, uint32_t pix, uint32_t sid, uint64_t key) {
  const uint64_t inc = ((uint64_t)local_pixel(fa, pix) << 1) | 1u;
  uint64_t st;
  pcg32_seed(st, inc, key);
  return eye_path_at(fa, pix, sid, st);
}
__device__ __forceinline__ void write_eye_path(const FrameArgs& fa, PathBuf& pb, uint32_t slot, uint32_t pix,
                                               uint32_t sid, uint64_t key) {
  const PathState p = eye_path(fa, pix, sid, key);
  pb.ray_o[slot] = p.ro;
  pb.ray_d[slot] = p.rd;
  pb.pix[slot] = p.pix;
  pb.sid[slot] = p.sid;
  pb.depth[slot] = 0;
  pb.mul[slot] = p.mul;
  pb.smp[slot] = p.smp;
  pb.acc[slot] = p.acc;
  pb.rng[slot] = p.rng;
}

__device__ __forceinline__ void zero_rec(SampleRec& rec, uint32_t q) {
  const float4 z = make_float4(0.f, 0.f, 0.f, 0.f);
  rec.acc[q] = z; rec.gpos[q] = z; rec.gnrm[q] = z; rec.gdif[q] = z;
}

// One path per pixel and frame of the batch.  Path slots are pixel-major
// (slot = pixel * frames + frame offset): a wave's first rays are one pixel's
// jittered rays of consecutive frames, which visit the same nodes, where
// frame-major slots give it 64 neighbouring pixels (extension 21 % faster on
// the 262k-triangle grid at 64 frames).  The sample record stays
// frame-major (sid = frame offset * W*H + pixel) for k_apply_frames.
// The eye path of slot i and its packed depth word.  The first extension and
// shading of a batch can call this in place of reading what k_gen_eye wrote.
__device__ __forceinline__ PathState eye_slot(const FrameArgs& fa, uint32_t i, uint32_t& dk) {
  const uint32_t wh = fa.width * fa.height, K = fa.nframes, pix = i / K, k = i - pix * K;
  dk = (k << 8) | kFreshPath;
  return eye_path(fa, pix, k * wh + pix, stream_key(fa.seed, frame_base(fa) + k, 1u, 0u));
}
__global__ __launch_bounds__(kBlock) void k_gen_eye(FrameArgs fa, PathBuf pb, SampleRec rec) {
  uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= fa.width * fa.height * fa.nframes) return;
  uint32_t dk;
  const PathState p = eye_slot(fa, i, dk);
  pb.ray_o[i] = p.ro;
  pb.ray_d[i] = p.rd;
  pb.pix[i] = p.pix;
  pb.sid[i] = p.sid;
  pb.depth[i] = dk;
  pb.rng[i] = p.rng;
  if (rec.acc) zero_rec(rec, p.sid);
}
hipError_t launch_gen_eye(const FrameArgs& fa, PathBuf pb, hipStream_t st) {
  if (!pathbuf_ok(pb)) return hipErrorInvalidValue;
  uint32_t n = fa.width * fa.height * fa.nframes;
  SampleRec none = {nullptr, nullptr, nullptr, nullptr};
  k_gen_eye<<<(n + kBlock - 1) / kBlock, kBlock, 0, st>>>(fa, pb, none);
  return hipGetLastError();
}
hipError_t launch_gen_eye_rec(const FrameArgs& fa, PathBuf pb, SampleRec rec, hipStream_t st) {
  if (!pathbuf_ok(pb) || !rec_ok(rec)) return hipErrorInvalidValue;
  uint32_t n = fa.width * fa.height * fa.nframes;
  k_gen_eye<<<(n + kBlock - 1) / kBlock, kBlock, 0, st>>>(fa, pb, rec);
  return hipGetLastError();
}

// The path tracers' running mean (pt_applyPathQueueResult_kernel,
// src/cudaRTPTStream.cu:303-325): the frame's per-pixel mean acc / n weighted
// 1 / (frame + 1), whatever the number of samples the pixel took.
__device__ __forceinline__ void apply_pixel_pt(float* result, uint32_t* sample_n, uint32_t pix, uint32_t frame, f3 acc,
                                               uint32_t n) {
  const uint32_t nold = frame == 0 ? 0u : sample_n[pix];
  if (n > 0) {
    const float fn = (float)n;
    const f3 sr = mk3(acc.x / fn, acc.y / fn, acc.z / fn);
    const float ri = 1.f / (float)(frame + 1), oi = 1.f - ri;
    float* r = result + (size_t)pix * 3;
    r[0] = fmaxf(ri * sr.x + oi * r[0], 0.f);
    r[1] = fmaxf(ri * sr.y + oi * r[1], 0.f);
    r[2] = fmaxf(ri * sr.z + oi * r[2], 0.f);
  }
  sample_n[pix] = nold + n;
}

// Frames of the batch applied in order: pt_applyPathQueueResult_kernel's
// running mean (src/cudaRTBDPTStream.cu:741-778) once per frame (pt: the path
// tracers' mean).
__global__ __launch_bounds__(kBlock) void k_apply_frames(FrameArgs fa, const float4* __restrict__ rec_acc,
                                                         float* __restrict__ result, uint32_t* __restrict__ sample_n,
                                                         int pt) {
  const uint32_t wh = fa.width * fa.height;
  const uint32_t pix = blockIdx.x * kBlock + threadIdx.x;
  if (pix >= wh) return;
  const uint32_t f0 = frame_base(fa);
  for (uint32_t k = 0; k < fa.nframes; k++) {
    float4 a = rec_acc[(size_t)k * wh + pix];
    if (pt) apply_pixel_pt(result, sample_n, pix, f0 + k, ld3(a), __float_as_uint(a.w));
    else apply_pixel(result, sample_n, pix, f0 + k, ld3(a), __float_as_uint(a.w));
  }
}
hipError_t launch_apply_frames(const FrameArgs& fa, const float4* rec_acc, float* result, uint32_t* sample_n,
                               int pt, hipStream_t st) {
  if (!rec_acc || !result || !sample_n) return hipErrorInvalidValue;
  uint32_t wh = fa.width * fa.height;
  k_apply_frames<<<(wh + kBlock - 1) / kBlock, kBlock, 0, st>>>(fa, rec_acc, result, sample_n, pt);
  return hipGetLastError();
}

hipError_t launch_extend(const DevScene& sc, PathBuf pb, const FrameCounters* fc, int bounce, uint32_t max_n,
                         float4* hits, DevStats* stats, int lds_stack, int quant, hipStream_t st) {
  if (max_n == 0) return hipSuccess;
  if (!pathbuf_ok(pb) || !fc || !hits || !sc.tris || !nodes_ok(sc, quant))
    return hipErrorInvalidValue;
  dim3 grid((max_n + kBlock - 1) / kBlock), block(kBlock);
  const uint32_t* cnt = &fc->active[bounce];
#define CPT_EXT(L, S, W) k_trace<L, false, 1, S, W><<<grid, block, 0, st>>>(sc, pb.ray_o, pb.ray_d, 1, cnt, max_n, 0, hits, stats)
  if (quant) {
#define CPT_EXT_Q(S, W) CPT_EXT(2, S, W)
#define CPT_EXT_F(S, W) CPT_EXT(0, S, W)
    CPT_VARIANT_SWITCH(lds_stack, CPT_EXT_Q)
  } else {
    CPT_VARIANT_SWITCH(lds_stack, CPT_EXT_F)
  }
#undef CPT_EXT_Q
#undef CPT_EXT_F
#undef CPT_EXT
  return hipGetLastError();
}

// Persistent closest-hit grid over a global queue of the bounce's live rays.
template <int STK, int MINW, bool Q>
__global__ __launch_bounds__(kBlock, MINW) void k_extend_persist(DevScene sc, const float4* __restrict__ ro,
                                                                 const float4* __restrict__ rd,
                                                                 const uint32_t* __restrict__ countp, uint32_t chunk,
                                                                 uint32_t* __restrict__ queue,
                                                                 float4* __restrict__ out,
                                                                 DevStats* __restrict__ stats) {
  __shared__ TravLds<STK, Q> lds;
  __shared__ uint32_t base_s;
  const uint32_t count = *countp;
  uint32_t nn = 0, nt = 0;
  for (;;) {
    if (threadIdx.x == 0) base_s = atomicAdd(queue, chunk);
    __syncthreads();
    const uint32_t base = base_s;
    __syncthreads();
    if (base >= count) break;
    const uint32_t end = min(base + chunk, count);
    for (uint32_t b0 = base; b0 < end; b0 += kBlock) {       // workgroup-uniform
      const uint32_t i = b0 + threadIdx.x;
      float4 a = make_float4(0.f, 0.f, 0.f, 0.f), b = a;
      if (i < end) { a = ro[i]; b = rd[i]; }
      TraceHit h;
      const bool hit = trace_rays<false, STK, Q>(sc, lds, i < end, ld3(a), ld3(b), a.w, b.w, false, h, nn, nt);
      if (i < end) {
        float4 r;
        r.x = hit ? h.t : kInfF;
        r.y = __uint_as_float(hit ? h.leaf : kInvalid);
        r.z = hit ? h.u : 0.f;
        r.w = hit ? h.v : 0.f;
        out[i] = r;
      }
    }
  }
  if (stats) {
    stats = stat_slot(stats);
    uint32_t sn = wave_sum(nn), st = wave_sum(nt);
    if ((threadIdx.x & 63) == 0 && (sn | st)) {
      atomicAdd(&stats->ext_nodes, (unsigned long long)sn);
      atomicAdd(&stats->ext_tris, (unsigned long long)st);
    }
  }
}
hipError_t launch_extend_persist(const DevScene& sc, PathBuf pb, const FrameCounters* fc, int bounce, float4* hits,
                                 DevStats* stats, int lds_stack, int quant, uint32_t chunk, uint32_t grid,
                                 uint32_t* queue, hipStream_t st) {
  if (!pathbuf_ok(pb) || !fc || !hits || !sc.tris || !queue || chunk == 0 || grid == 0 ||
      !nodes_ok(sc, quant))
    return hipErrorInvalidValue;
  k_fill_u32<<<1, 1, 0, st>>>(queue, 0u);
  const uint32_t* cnt = &fc->active[bounce];
#define CPT_EXTP(S, W, Q) k_extend_persist<S, W, Q><<<grid, kBlock, 0, st>>>(sc, pb.ray_o, pb.ray_d, cnt, chunk, queue, hits, stats)
#define CPT_EXTP_Q(S, W) CPT_EXTP(S, W, true)
#define CPT_EXTP_F(S, W) CPT_EXTP(S, W, false)
  if (quant) {
    CPT_VARIANT_SWITCH(lds_stack, CPT_EXTP_Q)
  } else {
    CPT_VARIANT_SWITCH(lds_stack, CPT_EXTP_F)
  }
#undef CPT_EXTP_Q
#undef CPT_EXTP_F
#undef CPT_EXTP
  return hipGetLastError();
}

// The rays [0, count) of a launch dealt to the waves of a persistent grid.
// Workgroups go to the chip's eight dies (each with its own L2) in turn, so the
// rays are cut into kDealers contiguous shares, one a die: neighbouring rays, which meet
// the same nodes, stay within one L2.  Of its die's share each wave first
// takes a quarter of an even part with no atomic; further chunks come from the
// share's counter, half an even part of what the wave knows to be left, so
// that they shrink towards the end (64 rays at the least).  A wave whose share is
// dealt out goes on with the next, whose counter it reads before adding to it (atomics on one
// address are served one after the other).  Launches of up to 64 rays a wave
// are dealt once, evenly over the waves (kDealLow rays at the least: fewer rays
// a wave end sooner, 16 / 64 take 25.3 / 25.8 ms in the learned frames).
// queue: kDealers counters, kDealStride words apart, zero when the launch starts.
// One share instead of eight takes 28.1 ms in the learned frames against 26.0 and the
// same elsewhere; one counter with chunks of 256 and no first chunk, as before, 30.5
// there and 20.2 against 19.2 ms for a still of 64 1280 x 720 frames.
struct Deal {
  uint32_t share, len, start, fixed, waves;   // of the share being drawn from (all uniform across the wave)
  uint32_t left;                              // shares left to visit, this one included
  uint32_t known;                             // rays of the share known to be dealt
};
__device__ __forceinline__ uint32_t deal_clamp(uint32_t v) {
  v &= ~63u;
  return v < 64u ? 64u : v > kDealMax ? kDealMax : v;
}
__device__ __forceinline__ void deal_share(Deal& D, uint32_t share, uint32_t count) {
  const uint32_t part = ((count - 1u) / kDealers / 64u + 1u) * 64u;      // count > 0
  D.share = share;
  D.start = min((uint64_t)share * part, (uint64_t)count);
  D.len = min(part, count - D.start);
  D.waves = gridDim.x > share ? (gridDim.x - share + kDealers - 1u) / kDealers * (kBlock / 64) : 0u;
  D.fixed = deal_clamp(D.len / (4u * max(D.waves, 1u)));
}
__device__ __forceinline__ void deal_first(Deal& D, uint32_t count, uint32_t wave, uint32_t& at, uint32_t& end) {
  D.left = count ? kDealers : 0u;
  at = end = 0u;
  if (!count) return;
  const uint32_t waves = gridDim.x * (kBlock / 64), k = blockIdx.x * (kBlock / 64) + wave;
  if (count <= waves * 64u) {
    D.left = 0u;
    const uint32_t per = min(64u, max(kDealLow, (count + waves - 1u) / waves));
    if (k * per < count) {
      at = k * per;
      end = min(at + per, count);
    }
    return;
  }
  deal_share(D, blockIdx.x % kDealers, count);
  const uint64_t off = (uint64_t)(blockIdx.x / kDealers * (kBlock / 64) + wave) * D.fixed;
  D.known = D.waves * D.fixed;
  if (off < D.len) {
    at = D.start + (uint32_t)off;
    end = D.start + min((uint32_t)off + D.fixed, D.len);
  }
}
// The wave's next chunk; false when none is left.
__device__ __forceinline__ bool deal_next(Deal& D, uint32_t count, uint32_t* __restrict__ queue, int lane, uint32_t& at,
                                          uint32_t& end) {
  while (D.left) {
    const uint32_t given = D.waves * D.fixed;
    uint32_t* ctr = queue + D.share * kDealStride;
    if (given < D.len && D.known < D.len) {
      const uint32_t step = deal_clamp((D.len - D.known) / (2u * max(D.waves, 1u)));
      uint32_t q = 0;
      if (lane == 0) q = atomicAdd(ctr, step);
      q = __builtin_amdgcn_readfirstlane(q);
      D.known = given + q;
      if (D.known < D.len) {
        at = D.start + D.known;
        end = D.start + min(D.known + step, D.len);
        return true;
      }
    }
    if (--D.left == 0) break;
    deal_share(D, (D.share + 1u) % kDealers, count);
    const uint32_t g = D.waves * D.fixed;
    uint32_t q = 0;
    if (g < D.len) {
      if (lane == 0) q = __hip_atomic_load(queue + D.share * kDealStride, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      q = __builtin_amdgcn_readfirstlane(q);
    }
    D.known = g + q;
  }
  return false;
}

// Dynamic refill: a persistent grid whose lanes each trace one ray at a time
// and take the next as soon as theirs is finished; lanes refill once at least
// `refill` (1..64) are idle, from a chunk of rays that the wave holds (Deal).
// A finished lane writes its result at the wave's next refill point, together
// with the other finished lanes, not in the traversal loop: the shadow
// epilogue's read-modify-write would otherwise stall the whole wave on its load
// every time one lane finishes.
// OUT 1: closest hit (t, leaf, u, v) into out[ray]; OUT 3: the connection's
// visibility (k_shadow's epilogue).
// Query flags: the back-face test; the answers of the FP32 4-wide nodes.  The
// two layouts' box tests differ where a ray touches a triangle's edge within
// rounding: the 8-wide one is conservative, so its hit is the (t, id) minimum over
// all triangles, while child_boxes may cull the box (2 of 126 M rays spread over
// the sphere grid, a few in 10^5 of those aimed at its edges, one in 10^3 on the
// Cornell box).  What the 4-wide nodes find the 8-wide ones find too, so a miss
// stands, and a hit stands if they are sure to test its triangle (reached4); the
// other rays are traced again by traverse4.  So are, with either layout's answers, rays
// with no hit within 1e20 but a longer reach: IntersectTri's 1e20 for a missed triangle is then a hit
// of the first one tested.  And rays whose boxes say little of their triangles: of
// negative eps (culled by distances behind the best hit's), or short (under 1e-2)
// with a component that escape_zero moves (by 1e-9, far off at their distances): their
// answer is that of the tree's order and leaves.  2,097,143 closest hits on the sphere
// grid 203 -> 219 us, 1,000,003 occlusion rays on the heightfield 131 -> 142 (box
// gathered from the vertices 229 / 148, with child_boxes' divisions 223 / 145).
constexpr uint32_t kQueryCull = 1u, kQueryFp32 = 2u;
constexpr uint32_t kQueryAgain = 0xFFFFFFFEu;        // written for such a ray until the wave's others are done
// EYE (closest hit, quantized nodes): ray i is the eye ray of path slot i of
// the batch fa describes, computed in place of reading ro / rd.  A separate
// instantiation, so that the plain kernels' code is not touched by it.
template <int OUT, int STK, int MINW, bool Q, bool EYE = false>
__global__ __launch_bounds__(kBlock, MINW) void k_trace_dyn(DevScene sc, const float4* __restrict__ ro,
                                                            const float4* __restrict__ rd,
                                                            const uint32_t* __restrict__ countp,
                                                            uint32_t* __restrict__ queue, float4* __restrict__ out,
                                                            const float4* __restrict__ contrib, PathBuf nxt,
                                                            DevStats* __restrict__ stats, uint32_t refill,
                                                            FrameArgs fa) {
  constexpr bool API = OUT == 0 || OUT == 2;        // fa.width rays as cpt_ray records, fa.flags: kQuery*
  constexpr bool ANY = OUT == 2 || OUT == 3;
  constexpr bool SH = OUT == 3;                     // counted as shadow rays; queries of either kind are not
  constexpr int S8 = kStk8<STK>;
  __shared__ TravLds<STK, Q> lds;
  static_assert(kPriv8<S8> <= CPT_STACK_TOTAL, "API: the stack of traverse4 too, once the wave's rays have finished");
  uint64_t pstk[API ? CPT_STACK_TOTAL : Q ? kPriv8<S8> : CPT_STACK_TOTAL - STK];
  const uint32_t count = API ? fa.width : *countp;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint64_t below = (1ull << lane) - 1ull;
  // Queries of the trace entry points have no counters (calls on several streams
  // would share them): wave w takes chunks of 64 w, w + waves, ...
  const uint32_t waves = gridDim.x * (kBlock / 64);
  uint32_t cnext, cend;                    // the wave's chunk (uniform across the wave)
  uint32_t base = 0;                       // where it began (API)
  Deal deal;
  if constexpr (API) {
    cnext = base = min((blockIdx.x * (kBlock / 64) + wid) * 64u, count);
    cend = min(cnext + 64u, count);
  } else {
    deal_first(deal, count, wid, cnext, cend);
  }
  bool exhausted = false;                  // uniform
  bool active = false;
  bool pending = false;                    // finished, result not yet written
  bool redo = false;                       // API: wrote kQueryAgain
  uint32_t ray = 0;
  std::conditional_t<Q, Ray8, RayState> R = {};   // 8-wide: lanes without a ray visit the root
  uint32_t nn = 0, nt = 0;
  __shared__ uint32_t spill_all[kBlock / 64];
  uint32_t* spill = spill_all + wid;
  if (lane == 0) *spill = 0u;
  for (;;) {
    const uint64_t idle = __ballot(!active);
    const uint32_t n_idle = (uint32_t)__popcll(idle);
    if (n_idle >= refill && pending) {
      pending = false;
      TraceHit h;
      bool hit;
      if constexpr (Q) {
        hit = ray8_hit(lds.w[wid], lane, h);
      } else {
        h = R.h;
        hit = h.leaf != kInvalid;
      }
      bool again = false;
      if constexpr (API) {
        again = R.ht > kInfF && !(ANY && hit);
        if (fa.flags & kQueryFp32) {
          const float lo = fminf(fabsf(R.idir.x), fminf(fabsf(R.idir.y), fabsf(R.idir.z)));
          const float hi = fmaxf(fabsf(R.idir.x), fmaxf(fabsf(R.idir.y), fabsf(R.idir.z)));
          again = again || R.eps < 0.f || (lo > 100.f && hi > 4e8f);
          if (hit && !again) again = !reached4(sc, h.leaf, ld3(ro[2 * (size_t)ray]), R.idir, h.t, R.eps);
        }
        redo = redo || again;
      }
      if (OUT == 1) {
        float4 r;
        r.x = hit ? h.t : kInfF;
        r.y = __uint_as_float(hit ? h.leaf : kInvalid);
        r.z = hit ? h.u : 0.f;
        r.w = hit ? h.v : 0.f;
        out[ray] = r;
      } else if (OUT == 0) {
        out[ray] = make_float4(__uint_as_float(again ? kQueryAgain : h.orig), h.t, h.u, h.v);
      } else if (OUT == 2) {
        ((uint32_t*)out)[ray] = again ? kQueryAgain : hit ? 1u : 0u;
      } else if (!hit) {
        const float4 c = contrib[ray];
        const uint32_t bits = __float_as_uint(c.w), slot = bits & ~kShadowNoCount;
        float4 acc = nxt.acc[slot];
        acc.x = acc.x + c.x;
        acc.y = acc.y + c.y;
        acc.z = acc.z + c.z;
        acc.w = __uint_as_float(__float_as_uint(acc.w) + ((bits & kShadowNoCount) ? 0u : 4u));
        nxt.acc[slot] = acc;
      }
    }
    if (!exhausted && n_idle >= refill) {
      const uint32_t rank = (uint32_t)__popcll(idle & below);
      uint32_t given = 0;
      while (given < n_idle) {
        if (cnext >= cend) {
          if constexpr (API) {
            const uint64_t b = (uint64_t)base + (uint64_t)waves * 64u;
            if (b >= count) { exhausted = true; break; }
            base = cnext = (uint32_t)b;
            cend = (uint32_t)min<uint64_t>(b + 64u, count);
          } else if (!deal_next(deal, count, queue, lane, cnext, cend)) {
            exhausted = true;
            break;
          }
        }
        const uint32_t take = min(n_idle - given, cend - cnext);
        if (!active && rank >= given && rank < given + take) {
          ray = cnext + (rank - given);
          float4 a, b4;
          if (EYE) {
            uint32_t dk;
            const PathState e = eye_slot(fa, ray, dk);
            a = e.ro;
            b4 = e.rd;
          } else if (API) {
            a = ro[2 * (size_t)ray];
            b4 = ro[2 * (size_t)ray + 1];
          } else {
            a = ro[ray];
            b4 = rd[ray];
          }
          if constexpr (Q) ray8_begin(R, lds.w[wid], lane, ld3(a), ld3(b4), a.w, b4.w, sc.qmag);
          else ray_begin(R, ld3(a), ld3(b4), a.w, b4.w);
          active = true;
        }
        cnext += take;
        given += take;
      }
    }
    // every lane idle with nothing left to take: the results were written above
    if (__ballot(active) == 0ull) break;
    if constexpr (Q) {
      const bool was = active;
      ray8_step<ANY, S8>(sc, R, active, API && (fa.flags & kQueryCull), lds.w[wid], (LdsU64*)&lds.w[wid].stk[0][lane],
                         pstk, lane, nn, nt, spill);
      if (was && !active) pending = true;
    } else if (active && ray_step<ANY, STK>(sc, R, false, lds_column(lds.stk), pstk, nn, nt, spill)) {
      active = false;
      pending = true;
    }
  }
  if constexpr (API) {
    if (__ballot(redo)) {                    // behind the loop, whose registers traverse4 would take
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
      const uint32_t* flag = (const uint32_t*)out;
      for (uint64_t b = (uint64_t)(blockIdx.x * (kBlock / 64) + wid) * 64u; b < count; b += (uint64_t)waves * 64u) {
        const uint64_t i = b + lane;
        if (i >= count || flag[ANY ? i : 4 * i] != kQueryAgain) continue;
        const float4 a = ro[2 * i], b4 = ro[2 * i + 1];
        TraceHit h;
        const bool hit =
            traverse4<ANY, 0>(sc, ld3(a), ld3(b4), a.w, b4.w, fa.flags & kQueryCull, nullptr, pstk, h, nn, nt);
        if (ANY) ((uint32_t*)out)[i] = hit ? 1u : 0u;
        else out[i] = hit ? make_float4(__uint_as_float(h.orig), h.t, h.u, h.v)
                          : make_float4(__uint_as_float(kInvalid), kInfF, 0.f, 0.f);
      }
    }
  }
  if (stats) {
    stats = stat_slot(stats);
    uint32_t sn = wave_sum(nn), st = wave_sum(nt);
    const uint32_t ss = *spill;         // the wave's own word, after its last atomic
    if (lane == 0 && (sn | st)) {
      atomicAdd(SH ? &stats->sh_nodes : &stats->ext_nodes, (unsigned long long)sn);
      atomicAdd(SH ? &stats->sh_tris : &stats->ext_tris, (unsigned long long)st);
      if (ss) atomicAdd(SH ? &stats->sh_spill : &stats->ext_spill, (unsigned long long)ss);
    }
  }
}
// Workgroups of a kernel that a compute unit holds at once.  A persistent grid
// is no larger: workgroups past it start only when others have ended, and would keep the
// chunks they begin with until then (8 a compute unit asked for, 6 resident, 8 / 6
// launched: 26.7 / 26.1 ms for the learned frames, 19.6 / 19.2 the 64-frame still).
uint32_t resident_groups(const void* kernel) {
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, kBlock, 0) != hipSuccess || n < 1) return 32;
  return (uint32_t)n;
}
hipError_t launch_trace_dyn(const DevScene& sc, const float4* ro, const float4* rd, const uint32_t* count,
                            float4* out, const float4* contrib, PathBuf nxt, DevStats* stats, int lds_stack,
                            int quant, int shadow, uint32_t groups, uint32_t cus, uint32_t refill, uint32_t* queue,
                            hipStream_t st, const FrameArgs* eye) {
  if (!ro || !rd || !count || !queue || groups == 0 || cus == 0 || refill < 1 || refill > 64 || !sc.tris ||
      !nodes_ok(sc, quant))
    return hipErrorInvalidValue;
  if (shadow ? (!contrib || !pathbuf_ok(nxt) || eye) : !out) return hipErrorInvalidValue;
  const FrameArgs fa = eye ? *eye : FrameArgs{};
#define CPT_DYN_E(O, S, W, Qb, Eb)                                                                              \
  {                                                                                                             \
    static const uint32_t resident = resident_groups((const void*)k_trace_dyn<O, S, W, Qb, Eb>);                \
    const uint32_t grid = (groups < resident ? groups : resident) * cus;                                        \
    k_trace_dyn<O, S, W, Qb, Eb><<<grid, kBlock, 0, st>>>(sc, ro, rd, count, queue, out, contrib, nxt, stats,   \
                                                          refill, fa);                                          \
  }
#define CPT_DYN(O, S, W, Qb) CPT_DYN_E(O, S, W, Qb, false)
#define CPT_DYN_1E(S, W) CPT_DYN_E(1, S, W, true, true)
#define CPT_DYN_3Q(S, W) CPT_DYN(3, S, W, true)
#define CPT_DYN_3F(S, W) CPT_DYN(3, S, W, false)
#define CPT_DYN_1Q(S, W) CPT_DYN(1, S, W, true)
#define CPT_DYN_1F(S, W) CPT_DYN(1, S, W, false)
  if (shadow) {
    if (quant) { CPT_VARIANT_SWITCH(lds_stack, CPT_DYN_3Q) } else { CPT_VARIANT_SWITCH(lds_stack, CPT_DYN_3F) }
  } else if (eye) {
    if (!quant) return hipErrorInvalidValue;
    CPT_VARIANT_SWITCH(lds_stack, CPT_DYN_1E)
  } else {
    if (quant) { CPT_VARIANT_SWITCH(lds_stack, CPT_DYN_1Q) } else { CPT_VARIANT_SWITCH(lds_stack, CPT_DYN_1F) }
  }
#undef CPT_DYN_3Q
#undef CPT_DYN_3F
#undef CPT_DYN_1Q
#undef CPT_DYN_1F
#undef CPT_DYN_1E
#undef CPT_DYN
#undef CPT_DYN_E
  return hipGetLastError();
}

// Rays of the trace entry points: the persistent grid's workgroups (six a compute
// unit are resident: more would start after the first have drained; 3, 4, 5, 6
// and 8 take 415, 365, 339, 335 and 403 us for 2,097,143 closest-hit rays on the
// heightfield), lanes refilled once 16 are idle (64, 48, 32, 16: 457, 347, 335,
// 328 us there; 327, 278, 281, 266 on the sphere grid).  Up to one chunk of 64
// rays a wave the grid is no larger than the rays and nothing is refilled.
// One thread per ray over 128-byte 4-wide nodes took 920 us on the sphere grid,
// and 1,000,003 occlusion rays on the heightfield 255.
constexpr uint32_t kTraceGroups = 6, kTraceRefill = 16;
hipError_t launch_trace_rays(const DevScene& sc, const float4* rays, uint32_t n, uint32_t cull, float4* out, int any,
                             int fp32, DevStats* stats, uint32_t cus, hipStream_t st) {
  if (n == 0) return hipSuccess;
  if (!sc.nodes8) return launch_trace(sc, rays, n, cull, out, any, 0, 0, stats, st);
  if (!rays || !out || !sc.tris8 || cus == 0) return hipErrorInvalidValue;
  FrameArgs fa = {};
  fa.width = n;
  fa.flags = (cull ? kQueryCull : 0u) | (fp32 ? kQueryFp32 : 0u);
  const uint32_t blocks = (n + kBlock - 1) / kBlock;
  const uint32_t grid = blocks < kTraceGroups * cus ? blocks : kTraceGroups * cus;
  if (any)
    k_trace_dyn<2, 8, 6, true><<<grid, kBlock, 0, st>>>(sc, rays, nullptr, nullptr, nullptr, out, nullptr, PathBuf{},
                                                        stats, kTraceRefill, fa);
  else
    k_trace_dyn<0, 8, 6, true><<<grid, kBlock, 0, st>>>(sc, rays, nullptr, nullptr, nullptr, out, nullptr, PathBuf{},
                                                        stats, kTraceRefill, fa);
  return hipGetLastError();
}

// Same plus the count-weighted first-hit G-buffer running means of the
// adaptive file (src/cudaRTBDPTStreamAdapBilatAtomic.cu:999-1036).
__device__ __forceinline__ void apply_pixel_gbuf(const Accum& ac, uint32_t pix, uint32_t frame, f3 acc, uint32_t n,
                                                 uint32_t sid) {
  uint32_t nold = frame == 0 ? 0u : ac.sample_n[pix];
  if (frame == 0) ac.sample_n[pix] = 0u;
  uint32_t nn = nold + n;
  if (!(nn > nold) || isinf3(acc)) return;
  float ri = 1.f / (float)nn, oi = (float)nold * ri;
  float* r = ac.result + (size_t)pix * 3;
  r[0] = fmaxf(ri * acc.x + oi * r[0], 0.f);
  r[1] = fmaxf(ri * acc.y + oi * r[1], 0.f);
  r[2] = fmaxf(ri * acc.z + oi * r[2], 0.f);
  ac.sample_n[pix] = nn;
  const float nf = (float)n;
  float4 g[3] = {ac.rec.gpos[sid], ac.rec.gnrm[sid], ac.rec.gdif[sid]};
  float* dst[3] = {ac.gpos + (size_t)pix * 3, ac.gnrm + (size_t)pix * 3, ac.gdif + (size_t)pix * 3};
#pragma unroll
  for (int k = 0; k < 3; k++) {
    f3 w = ld3(g[k]) * nf;
    dst[k][0] = ri * w.x + oi * dst[k][0];
    dst[k][1] = ri * w.y + oi * dst[k][1];
    dst[k][2] = ri * w.z + oi * dst[k][2];
  }
  if (ac.sq) {                                     // squareResult (AdapEmp.cu:927-944)
    float* q = ac.sq + (size_t)pix * 3;
    q[0] = fmaxf(ri * (acc.x * acc.x) + oi * q[0], 0.f);
    q[1] = fmaxf(ri * (acc.y * acc.y) + oi * q[1], 0.f);
    q[2] = fmaxf(ri * (acc.z * acc.z) + oi * q[2], 0.f);
  }
}

// Append with one atomic per workgroup of B threads, grouped by a 3-bit key
// (the ray direction's octant): within the workgroup's share of each queue the
// lanes come key by key, so that a wave of the next traversal holds rays of few
// octants.  k0 / k1: the key of a lane appending to queue 0 / 1.
template <int B>
__device__ __forceinline__ void block_append2_oct(bool p0, uint32_t k0, bool p1, uint32_t k1, uint32_t* ctr0,
                                                  uint32_t* ctr1, uint32_t& s0, uint32_t& s1) {
  constexpr int W = B / 64;
  __shared__ uint32_t c0[8][W], c1[8][W], base0, base1;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const unsigned long long below = (1ull << lane) - 1ull;
  uint32_t r0 = 0, r1 = 0;
#pragma unroll
  for (uint32_t b = 0; b < 8; b++) {
    const unsigned long long m0 = __ballot(p0 && k0 == b), m1 = __ballot(p1 && k1 == b);
    if (lane == 0) { c0[b][wid] = (uint32_t)__popcll(m0); c1[b][wid] = (uint32_t)__popcll(m1); }
    if (k0 == b) r0 = (uint32_t)__popcll(m0 & below);
    if (k1 == b) r1 = (uint32_t)__popcll(m1 & below);
  }
  __syncthreads();
  if (threadIdx.x == 0) {                  // exclusive prefix over (key, wave), then one atomic per queue
    uint32_t t0 = 0, t1 = 0;
    for (int b = 0; b < 8; b++)
      for (int w = 0; w < W; w++) {
        const uint32_t a = c0[b][w], c = c1[b][w];
        c0[b][w] = t0; c1[b][w] = t1;
        t0 += a; t1 += c;
      }
    base0 = t0 ? atomicAdd(ctr0, t0) : 0u;
    base1 = t1 ? atomicAdd(ctr1, t1) : 0u;
  }
  __syncthreads();
  s0 = p0 ? base0 + c0[k0 & 7u][wid] + r0 : 0u;
  s1 = p1 ? base1 + c1[k1 & 7u][wid] + r1 : 0u;
}
__device__ __forceinline__ uint32_t octant(float4 d) {
  return (d.x < 0.f ? 1u : 0u) | (d.y < 0.f ? 2u : 0u) | (d.z < 0.f ? 4u : 0u);
}

// One eye-path vertex (pt_traceSample_kernel, src/cudaRTBDPTStream.cu:365-543,
// and the connection set-up of pt_connectEyeLightPath_kernel, :665-723):
// emission, BRDF sample, Russian roulette, termination into the accumulators,
// and for a surviving diffuse bounce the light-vertex connection's shadow ray.
// p holds the path before the bounce and, when `survive`, after it.
__device__ __forceinline__ void shade_path(const DevScene& sc, const FrameArgs& fa, const FrameCounters* fc,
                                           const LightVert* __restrict__ lv, const Accum& ac, PathState& p, float4 h,
                                           bool& survive, bool& emit, ShadowRay& sr) {
  const uint32_t pix = p.pix, sid = p.sid;
  uint32_t depth = p.depth;
  const uint32_t frame = frame_base(fa) + p.fk;
  const uint32_t slot = (frame / 3u) % (uint32_t)kLightSlots;
  const uint32_t lvN = fc->light_n[slot];
  const LightVert* __restrict__ lvb = lv + (size_t)slot * fa.lv_stride;
  uint64_t st = p.rng;
  const float4 ro = p.ro, rd = p.rd, m4 = p.mul, s4 = p.smp, a4 = p.acc;
  float4 o_out, d_out, mul_out, smp_out, acc_out;
  float4& so = sr.o;
  float4& sd = sr.d;
  float4& sc4 = sr.c;
  const uint64_t inc = ((uint64_t)local_pixel(fa, pix) << 1) | 1u;
  f3 orig = ld3(ro), dir = ld3(rd), mul = ld3(m4), psample = ld3(s4), acc = ld3(a4);
  uint32_t N = __float_as_uint(a4.w);
  uint32_t leaf = __float_as_uint(h.y);
  bool term = false;
  if (leaf == kInvalid) {
    // an escaping eye path gathers the environment's radiance through its throughput
    if (sc.env_w) psample = psample + vmul(env_radiance(sc, dir), mul);
    acc = acc + psample; N++; term = true;
  } else {
    float w = (1.f - h.z) - h.w;
    const bool gbuf = (ac.variant & kVariantGbuf) && depth == 0;
    Surf s = fetch_surf(sc, leaf, w, h.z, h.w, gbuf);
    f3 nl = dot(s.norm, dir) < 0.f ? s.norm : s.norm * -1.f;
    if (gbuf) {                                          // AdapBilatAtomic.cu:650-655
      ac.rec.gpos[sid] = make_float4(s.pos.x, s.pos.y, s.pos.z, 0.f);
      ac.rec.gnrm[sid] = make_float4(nl.x, nl.y, nl.z, 0.f);
      ac.rec.gdif[sid] = make_float4(s.diff.x, s.diff.y, s.diff.z, 0.f);
    }
    const bool pt = (ac.variant & kVariantPT) != 0;
    Bounce b = sample_bounce(st, inc, orig, dir, h.x, s, nl, RT_EYE, (ac.variant & kVariantReflOffset) != 0, pt);
    psample = psample + vmul(s.emissive, mul);
    f3 inMul = mul, inDir = dir * -1.f;
    float contrib = length(mul) * length(b.mul);
    if (length(s.emissive) > 0.f) contrib = 0.f;
    // the regenerating path tracer also ends a diffuse-to-specular step
    // (cudaRTPTStreamRegen.cu:241)
    if ((ac.variant & kVariantPTRegen) && p.type == RT_DIFF && b.type == RT_SPEC) contrib = 0.f;
    const uint32_t lim = p.lim ? p.lim : fa.eye_depth;
    if (uniform01(st, inc) > contrib || depth + 1 >= lim) {
      acc = acc + psample; N++; term = true;
    } else {
      mul = vmul(mul, b.mul);
      dir = b.dir;
      depth++;
      orig = b.orig;
      p.type = b.type;
      if (!pt && b.type == RT_DIFF && lvN > 0) {
        f3 pos = orig + nl * (float)kBiasEps;
        uint32_t li = (uint32_t)(uniform01(st, inc) * (float)lvN);
        if (li >= lvN) li = lvN - 1;
        const LightVert& L = lvb[li];
        f3 lpos = mk3(L.pos[0], L.pos[1], L.pos[2]);
        f3 lirr = mk3(L.irrad[0], L.irrad[1], L.irrad[2]);
        f3 toL = normalize(lpos - pos);
        float dist = length(lpos - pos);
        if (length(lirr) > 0.f && dot(nl, toL) > 0.f) {
          f3 irrad, irradDir;
          if ((double)dist > kFltEps) {
            irrad = shading(toL * -1.f, mk3(L.irradDir[0], L.irradDir[1], L.irradDir[2]), lirr,
                            mk3(L.norm[0], L.norm[1], L.norm[2]), mk3(L.diff[0], L.diff[1], L.diff[2]), L.metallic,
                            L.roughness, L.specular, 1.f, 1.f) +
                    mk3(L.emissive[0], L.emissive[1], L.emissive[2]);
            irradDir = toL;
          } else {
            irrad = lirr;
            irradDir = mk3(L.irradDir[0], L.irradDir[1], L.irradDir[2]) * -1.f;
          }
          f3 c = vmax0(shading(inDir, irradDir, irrad, nl, s.diff, s.metal, s.rough, s.spec, 1.f - s.trans, 1.f));
          if (length(c) > 0.f) {
            f3 pay = vmul(c, inMul);
            emit = true;
            so = make_float4(pos.x, pos.y, pos.z, (float)shadow_max((double)dist, fa.flags));
            sd = make_float4(toL.x, toL.y, toL.z, (float)kBiasEps);
            sc4 = make_float4(pay.x, pay.y, pay.z, 0.f);
          }
        }
      }
    }
  }
  if (term) {
    if (ac.term_bounce) {                                 // regeneration: where and in which state it ended
      ac.term_bounce[sid] = depth;
      ac.term_rng[sid] = st;
    }
    if (ac.apply == 0) apply_pixel(ac.result, ac.sample_n, pix, frame, acc, N);
    else if (ac.apply == 1) apply_pixel_gbuf(ac, pix, frame, acc, N, sid);
    else ac.rec.acc[sid] = make_float4(acc.x, acc.y, acc.z, __uint_as_float(N));
  } else {
    survive = true;
    o_out = make_float4(orig.x, orig.y, orig.z, kInfF);
    d_out = make_float4(dir.x, dir.y, dir.z, (float)kBiasEps);
    mul_out = make_float4(mul.x, mul.y, mul.z, 0.f);
    smp_out = make_float4(psample.x, psample.y, psample.z, 0.f);
    acc_out = make_float4(acc.x, acc.y, acc.z, __uint_as_float(N));
  }
  if (survive) {
    p.ro = o_out;
    p.rd = d_out;
    p.mul = mul_out;
    p.smp = smp_out;
    p.acc = acc_out;
    p.depth = depth;
  }
  p.rng = st;
}

// ---- Disney-BRDF path tracer (extension; no reference counterpart) ----------
// The principled BRDF of Burley (SIGGRAPH 2012 course notes and brdf.txt),
// isotropic, specular tint 0, opaque, with next-event estimation to the
// emissive triangles and power-heuristic MIS against the BRDF samples.  The
// same operations, in the same order and drawing the same uniforms, as the
// oracle's FP64 restatement (disney_path).
struct DisneyMat {
  f3 base;
  float metallic, subsurface, specular, roughness, sheen, sheenTint, clearcoat, clearcoatGloss;
};
__device__ __forceinline__ float schlick_w(float c) {
  float m = fminf(fmaxf(1.f - c, 0.f), 1.f);
  return (m * m) * (m * m) * m;
}
__device__ __forceinline__ float gtr1(float nh, float a) {
  if (a >= 1.f) return (float)(1.0 / kPiD);
  const float a2 = a * a, t = 1.f + (a2 - 1.f) * nh * nh;
  return (a2 - 1.f) / (kPiF * logf(a2) * t);
}
__device__ __forceinline__ float gtr2(float nh, float a) {
  const float a2 = a * a, t = 1.f + (a2 - 1.f) * nh * nh;
  return a2 / (kPiF * t * t);
}
__device__ __forceinline__ float smith_g(float n, float a) {
  const float a2 = a * a, b = n * n;
  return 1.f / (n + sqrtf(a2 + b - a2 * b));
}
__device__ __forceinline__ float disney_alpha(const DisneyMat& m) { return fmaxf(m.roughness * m.roughness, 1e-3f); }
__device__ __forceinline__ float disney_cc_alpha(const DisneyMat& m) {
  return 0.1f + (0.001f - 0.1f) * m.clearcoatGloss;
}
__device__ __forceinline__ void disney_lobes(const DisneyMat& m, float& pd, float& ps, float& pc) {
  const float wd = 1.f - m.metallic, ws = 1.f, wc = 0.25f * m.clearcoat, t = (wd + ws) + wc;
  pd = wd / t; ps = ws / t; pc = wc / t;
}
__device__ f3 disney_f(const DisneyMat& m, f3 n, f3 wo, f3 wi) {
  const float nl = dot(n, wi), nv = dot(n, wo);
  if (nl <= 0.f || nv <= 0.f) return mk3(0.f, 0.f, 0.f);
  const f3 hv = wi + wo;
  const float hl = length(hv);
  if (!(hl > 0.f)) return mk3(0.f, 0.f, 0.f);
  const f3 h = hv / hl;
  const float nh = dot(n, h), lh = dot(wi, h);
  const float lum = 0.3f * m.base.x + 0.6f * m.base.y + 0.1f * m.base.z;
  const f3 tint = lum > 0.f ? m.base / lum : mk3(1.f, 1.f, 1.f);
  const f3 one = mk3(1.f, 1.f, 1.f);
  const f3 cspec0 = one * (0.08f * m.specular) + (m.base - one * (0.08f * m.specular)) * m.metallic;
  const f3 csheen = one + (tint - one) * m.sheenTint;
  const float fl = schlick_w(nl), fv = schlick_w(nv), fh = schlick_w(lh);
  const float fd90 = 0.5f + 2.f * lh * lh * m.roughness;
  const float fd = (1.f + (fd90 - 1.f) * fl) * (1.f + (fd90 - 1.f) * fv);
  const float fss90 = lh * lh * m.roughness;
  const float fss = (1.f + (fss90 - 1.f) * fl) * (1.f + (fss90 - 1.f) * fv);
  const float ss = 1.25f * (fss * (1.f / (nl + nv) - 0.5f) + 0.5f);
  const float a = disney_alpha(m);
  const float ds = gtr2(nh, a);
  const f3 fs = cspec0 + (one - cspec0) * fh;
  const float gs = smith_g(nl, a) * smith_g(nv, a);
  const f3 fsheen = csheen * (fh * m.sheen);
  const float dr = gtr1(nh, disney_cc_alpha(m));
  const float fr = 0.04f + (1.f - 0.04f) * fh;
  const float gr = smith_g(nl, 0.25f) * smith_g(nv, 0.25f);
  const f3 diffuse = (m.base * ((float)(1.0 / kPiD) * (fd + (ss - fd) * m.subsurface)) + fsheen) * (1.f - m.metallic);
  return (diffuse + fs * (gs * ds)) + one * (0.25f * m.clearcoat * gr * fr * dr);
}
__device__ float disney_pdf(const DisneyMat& m, f3 n, f3 wo, f3 wi) {
  const float nl = dot(n, wi), nv = dot(n, wo);
  if (nl <= 0.f || nv <= 0.f) return 0.f;
  const f3 hv = wi + wo;
  const float hl = length(hv);
  if (!(hl > 0.f)) return 0.f;
  const f3 h = hv / hl;
  const float nh = dot(n, h), vh = dot(wo, h);
  if (vh <= 0.f) return 0.f;
  float pd, ps, pc;
  disney_lobes(m, pd, ps, pc);
  float pdf = pd * nl * (float)(1.0 / kPiD);
  pdf = pdf + ps * gtr2(nh, disney_alpha(m)) * nh / (4.f * vh);
  pdf = pdf + pc * gtr1(nh, disney_cc_alpha(m)) * nh / (4.f * vh);
  return pdf;
}
__device__ bool disney_sample(const DisneyMat& m, f3 n, f3 wo, float u0, float u1, float u2, f3& wi) {
  float pd, ps, pc;
  disney_lobes(m, pd, ps, pc);
  f3 u, v;
  basis(n, u, v);
  const float phi = (float)(2.0 * kPiD * (double)u1);
  if (u0 < pd) {
    const float ct = sqrtf(u2), st = sqrtf(1.f - u2);
    float sp, cp;
    sincos_def(phi, sp, cp);
    wi = normalize((n * ct + (u * st) * cp) + (v * st) * sp);
  } else {
    const bool spec = u0 < pd + ps;
    const float a = spec ? disney_alpha(m) : disney_cc_alpha(m);
    float ct;
    if (spec) ct = sqrtf((1.f - u2) / (1.f + (a * a - 1.f) * u2));
    else ct = a >= 1.f ? sqrtf(1.f - u2) : sqrtf((1.f - powf(a * a, 1.f - u2)) / (1.f - a * a));
    const float st = sqrtf(fmaxf(0.f, 1.f - ct * ct));
    float sp, cp;
    sincos_def(phi, sp, cp);
    const f3 h = (n * ct + (u * st) * cp) + (v * st) * sp;
    wi = normalize(h * (2.f * dot(wo, h)) - wo);
  }
  return dot(n, wi) > 0.f;
}
__device__ __forceinline__ DisneyMat disney_of(const DevScene& sc, uint32_t leaf, const Surf& s) {
  DisneyMat m;
  m.base = s.diff; m.metallic = s.metal; m.specular = s.spec; m.roughness = s.rough;
  const uint32_t mi = __float_as_uint(sc.surf[8 * (size_t)leaf + 7].w);
  const DevMaterial& d = sc.mats[mi];
  m.subsurface = d.subsurface; m.sheen = d.sheen; m.sheenTint = d.sheenTint;
  m.clearcoat = d.clearcoat; m.clearcoatGloss = d.clearcoatGloss;
  return m;
}
// Solid-angle density of the light sampler at the point at distance t along
// unit d on leaf triangle `leaf`: 1 / n_lights, uniform by area, two faces.
__device__ __forceinline__ float light_pdf(const DevScene& sc, uint32_t leaf, float t, f3 d) {
  const f3 ng = cross(ld3(sc.tris[3 * (size_t)leaf + 1]), ld3(sc.tris[3 * (size_t)leaf + 2]));
  const float a2 = length(ng);
  const float c = fabsf(dot(ng, d)) / a2;
  if (!(c > 0.f) || !(a2 > 0.f)) return 0.f;
  return t * t / (c * (a2 * 0.5f) * (float)sc.n_light_tris);
}
// One bounce of the Disney path tracer: emission (MIS-weighted against the
// previous bounce's light sample), the depth bound, Russian roulette, the light
// sample (a shadow ray adding to the path's accumulator without a count) and
// the BRDF sample.  smp.w carries the BRDF density of the ray being traced.
__device__ __forceinline__ void shade_disney(const DevScene& sc, const FrameArgs& fa, const Accum& ac, PathState& p,
                                             float4 h, bool& survive, bool& emit, ShadowRay& sr) {
  const uint32_t pix = p.pix, sid = p.sid;
  uint32_t depth = p.depth;
  const uint32_t frame = frame_base(fa) + p.fk;
  uint64_t st = p.rng;
  const uint64_t inc = ((uint64_t)local_pixel(fa, pix) << 1) | 1u;
  f3 orig = ld3(p.ro), dir = ld3(p.rd), T = ld3(p.mul), L = ld3(p.smp), acc = ld3(p.acc);
  const float prev_pdf = p.smp.w;
  uint32_t N = __float_as_uint(p.acc.w);
  const uint32_t leaf = __float_as_uint(h.y);
  bool term = false, dead = false;
  float next_pdf = 0.f;
  if (leaf == kInvalid) {
    if (sc.env_w) L = L + vmul(T, env_radiance(sc, dir));
    term = true;
  } else {
    const float w = (1.f - h.z) - h.w;
    const Surf s = fetch_surf(sc, leaf, w, h.z, h.w, false);
    if (length(s.emissive) > 0.f) {
      float wt = 1.f;
      if (depth > 0) {
        const float pl = light_pdf(sc, leaf, h.x, dir);
        wt = prev_pdf * prev_pdf / (prev_pdf * prev_pdf + pl * pl);
      }
      L = L + vmul(T, s.emissive) * wt;
    }
    const uint32_t lim = p.lim ? p.lim : fa.eye_depth;
    if (depth + 1 >= lim) term = true;
    if (!term && depth >= 3) {
      const float q = fminf(0.95f, fmaxf(T.x, fmaxf(T.y, T.z)));
      if (uniform01(st, inc) >= q) term = true;
      else T = T / q;
    }
    if (!term) {
      const f3 nl = dot(s.norm, dir) < 0.f ? s.norm : s.norm * -1.f;
      const f3 pos = orig + dir * h.x, wo = dir * -1.f;
      const DisneyMat m = disney_of(sc, leaf, s);
      const uint32_t nL = sc.n_light_tris;
      if (nL > 0) {
        const float l0 = uniform01(st, inc);
        float l1 = uniform01(st, inc), l2 = uniform01(st, inc);
        uint32_t li = (uint32_t)(l0 * (float)nL);
        if (li >= nL) li = nL - 1;
        if (l1 + l2 > 1.f) { l1 = 1.f - l1; l2 = 1.f - l2; }
        const uint32_t lt = sc.light_tris[li];
        const float4 q0 = sc.tris[3 * (size_t)lt], q1 = sc.tris[3 * (size_t)lt + 1], q2 = sc.tris[3 * (size_t)lt + 2];
        const f3 lp = (ld3(q0) + ld3(q1) * l1) + ld3(q2) * l2;
        const f3 so = pos + nl * (float)kBiasEps;
        const f3 toL = lp - so;
        const float dist = length(toL);
        if ((double)dist > kFltEps) {
          const f3 wi = toL / dist;
          const float cs = dot(nl, wi);
          const float pl = light_pdf(sc, lt, dist, wi);
          if (cs > 0.f && pl > 0.f) {
            const f3 f = disney_f(m, nl, wo, wi);
            const float pb = disney_pdf(m, nl, wo, wi);
            const float wt = pl * pl / (pl * pl + pb * pb);
            const f3 le = ld3(sc.surf[8 * (size_t)lt + 4]);
            const f3 c = vmul(vmul(T, f), le) * (cs * wt / pl);
            if (length(c) > 0.f) {
              emit = true;
              sr.o = make_float4(so.x, so.y, so.z, (float)((double)dist - 2.0 * kBiasEps));
              sr.d = make_float4(wi.x, wi.y, wi.z, (float)kBiasEps);
              sr.c = make_float4(c.x, c.y, c.z, 0.f);
            }
          }
        }
      }
      const float b0 = uniform01(st, inc), b1 = uniform01(st, inc), b2 = uniform01(st, inc);
      f3 wi;
      const bool ok = disney_sample(m, nl, wo, b0, b1, b2, wi);
      const float pdf = ok ? disney_pdf(m, nl, wo, wi) : 0.f;
      if (!(pdf > 0.f)) {
        // no continuation; a pending light sample still needs the slot: the
        // path lives one more, empty segment (maximum distance 0, throughput 0)
        if (emit) dead = true;
        else term = true;
      } else {
        T = vmul(T, disney_f(m, nl, wo, wi)) * (dot(nl, wi) / pdf);
        next_pdf = pdf;
        orig = pos + wi * (float)kBiasEps;
        dir = wi;
      }
    }
  }
  if (term) {
    acc = acc + L;
    N++;
    if (ac.apply == 0) apply_pixel(ac.result, ac.sample_n, pix, frame, acc, N);
    else ac.rec.acc[sid] = make_float4(acc.x, acc.y, acc.z, __uint_as_float(N));
  } else {
    survive = true;
    if (dead) T = mk3(0.f, 0.f, 0.f);
    p.ro = make_float4(orig.x, orig.y, orig.z, dead ? 0.f : kInfF);
    p.rd = make_float4(dir.x, dir.y, dir.z, (float)kBiasEps);
    p.mul = make_float4(T.x, T.y, T.z, 0.f);
    p.smp = make_float4(L.x, L.y, L.z, next_pdf);
    p.acc = make_float4(acc.x, acc.y, acc.z, __uint_as_float(N));
    p.depth = depth + 1;
    p.type = RT_DIFF;
  }
  p.rng = st;
}

// The shading pass of one bounce over the live paths: survivors compacted into
// nxt, connection shadow rays into sb (contribution .w = the survivor's slot).
// Workgroup of the shading pass: its compaction takes one atomic per counter
// per workgroup.
constexpr int kShadeBlock = 256;
// Five waves per SIMD: 96 VGPRs without spills; left to itself the compiler
// takes 97 and four waves, and the pass is then 5-7 % slower.
// DISNEY: the Disney path tracer's bounce (shade_disney) in an instance of its
// own, so that its larger live set does not spill the BDPT instance's.
template <bool DISNEY>
__global__ __launch_bounds__(kShadeBlock, DISNEY ? 4 : 5) void k_shade(DevScene sc, FrameArgs fa, PathBuf cur,
                                                                       PathBuf nxt,
                                                  const float4* __restrict__ hits, FrameCounters* __restrict__ fc,
                                                  int bounce, ShadowBuf sb, const LightVert* __restrict__ lv,
                                                  Accum ac, int eye) {
  const uint32_t i = blockIdx.x * kShadeBlock + threadIdx.x;
  const uint32_t count = fc->active[bounce];
  if (blockIdx.x * kShadeBlock >= count) return;               // whole workgroup idle
  bool survive = false, emit = false;
  PathState p;
  ShadowRay sr;
  sr.o = sr.d = sr.c = make_float4(0.f, 0.f, 0.f, 0.f);
  if (i < count) {
    uint32_t dk;
    if (eye) {
      p = eye_slot(fa, i, dk);
    } else {
      p.ro = cur.ray_o[i];
      p.rd = cur.ray_d[i];
      p.pix = cur.pix[i];
      p.sid = cur.sid[i];
      dk = cur.depth[i];
      p.rng = cur.rng[i];
    }
    unpack_dk(p, dk);
    if (dk & kFreshPath) {
      p.mul = make_float4(1.f, 1.f, 1.f, 0.f);
      p.smp = make_float4(0.f, 0.f, 0.f, 0.f);
      p.acc = p.smp;
    } else {
      p.mul = cur.mul[i];
      p.smp = cur.smp[i];
      p.acc = cur.acc[i];
    }
    if constexpr (DISNEY) shade_disney(sc, fa, ac, p, hits[i], survive, emit, sr);
    else shade_path(sc, fa, fc, lv, ac, p, hits[i], survive, emit, sr);
  }
  uint32_t slot = 0, sslot = 0;
  block_append2_oct<kShadeBlock>(survive, survive ? octant(p.rd) : 8u, emit, emit ? octant(sr.d) : 8u,
                                 &fc->active[bounce + 1], &fc->shadow[bounce], slot, sslot);
  if (survive) {
    nxt.ray_o[slot] = p.ro;
    nxt.ray_d[slot] = p.rd;
    nxt.pix[slot] = p.pix;
    nxt.sid[slot] = p.sid;
    nxt.depth[slot] = pack_dk(p);
    nxt.mul[slot] = p.mul;
    nxt.smp[slot] = p.smp;
    nxt.acc[slot] = p.acc;
    nxt.rng[slot] = p.rng;
  }
  if (emit) {
    sr.c.w = __uint_as_float(slot | (DISNEY ? kShadowNoCount : 0u));
    sb.ray_o[sslot] = sr.o;
    sb.ray_d[sslot] = sr.d;
    sb.contrib[sslot] = sr.c;
  }
}
hipError_t launch_shade(const DevScene& sc, const FrameArgs& fa, PathBuf cur, PathBuf nxt, const float4* hits,
                        FrameCounters* fc, int bounce, uint32_t max_n, ShadowBuf sb, const LightVert* lv,
                        const Accum& ac, hipStream_t st, int eye) {
  if (max_n == 0) return hipSuccess;
  if (!pathbuf_ok(cur) || !pathbuf_ok(nxt) || !hits || !fc || !lv || !sb.ray_o || !sb.ray_d || !sb.contrib ||
      !ac.result || !ac.sample_n)
    return hipErrorInvalidValue;
  if (ac.apply == 1 && (!rec_ok(ac.rec) || !ac.gpos || !ac.gnrm || !ac.gdif)) return hipErrorInvalidValue;
  if (ac.apply == 2 && !ac.rec.acc) return hipErrorInvalidValue;
  if ((ac.variant & kVariantGbuf) && !rec_ok(ac.rec)) return hipErrorInvalidValue;
  const uint32_t grid = (max_n + kShadeBlock - 1) / kShadeBlock;
  if (ac.variant & kVariantDisney)
    k_shade<true><<<grid, kShadeBlock, 0, st>>>(sc, fa, cur, nxt, hits, fc, bounce, sb, lv, ac, eye);
  else
    k_shade<false><<<grid, kShadeBlock, 0, st>>>(sc, fa, cur, nxt, hits, fc, bounce, sb, lv, ac, eye);
  return hipGetLastError();
}

template <int STK, int MINW = 0, bool Q = false>
__global__ __launch_bounds__(kBlock, MINW) void k_shadow(DevScene sc, ShadowBuf sb, PathBuf nxt,
                                                   const FrameCounters* __restrict__ fc, int bounce,
                                                   DevStats* __restrict__ stats) {
  __shared__ TravLds<STK, Q> lds;
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  const uint32_t count = fc->shadow[bounce];
  uint32_t nn = 0, nt = 0;
  float4 a = make_float4(0.f, 0.f, 0.f, 0.f), b = a;
  if (i < count) {
    a = sb.ray_o[i];
    b = sb.ray_d[i];
  }
  TraceHit h;
  const bool hit = trace_rays<true, STK, Q>(sc, lds, i < count, ld3(a), ld3(b), a.w, b.w, false, h, nn, nt);
  if (i < count) {
    if (!hit) {
      const float4 c = sb.contrib[i];
      const uint32_t bits = __float_as_uint(c.w), slot = bits & ~kShadowNoCount;
      float4 acc = nxt.acc[slot];
      acc.x = acc.x + c.x;
      acc.y = acc.y + c.y;
      acc.z = acc.z + c.z;
      acc.w = __uint_as_float(__float_as_uint(acc.w) + ((bits & kShadowNoCount) ? 0u : 4u));
      nxt.acc[slot] = acc;
    }
  }
  if (stats) {
    stats = stat_slot(stats);
    uint32_t sn = wave_sum(nn), st = wave_sum(nt);
    if ((threadIdx.x & 63) == 0 && (sn | st)) {
      atomicAdd(&stats->sh_nodes, (unsigned long long)sn);
      atomicAdd(&stats->sh_tris, (unsigned long long)st);
    }
  }
}
hipError_t launch_shadow(const DevScene& sc, ShadowBuf sb, PathBuf nxt, const FrameCounters* fc, int bounce,
                         uint32_t max_n, int lds_stack, int quant, DevStats* stats, hipStream_t st) {
  if (max_n == 0) return hipSuccess;
  if (!pathbuf_ok(nxt) || !sb.ray_o || !sb.ray_d || !sb.contrib || !fc || !sc.tris ||
      !nodes_ok(sc, quant))
    return hipErrorInvalidValue;
  dim3 grid((max_n + kBlock - 1) / kBlock), block(kBlock);
#define CPT_SH(S, W, Q) k_shadow<S, W, Q><<<grid, block, 0, st>>>(sc, sb, nxt, fc, bounce, stats)
  if (quant) {
#define CPT_SH_Q(S, W) CPT_SH(S, W, true)
#define CPT_SH_F(S, W) CPT_SH(S, W, false)
    CPT_VARIANT_SWITCH(lds_stack, CPT_SH_Q)
  } else {
    CPT_VARIANT_SWITCH(lds_stack, CPT_SH_F)
  }
#undef CPT_SH_Q
#undef CPT_SH_F
#undef CPT_SH
  return hipGetLastError();
}

// ---------------------------------------------------------------- path regeneration
// cudaRTPTStreamRegen (src/cudaRTPTStreamRegen.cu:300-478): a slot whose path
// ends while other paths of the frame are still being traced restarts once,
// for the same pixel with its RNG state continuing (pt_reinitRegenPathStream_kernel),
// and the frame stops when its last first-generation path ends; a restarted
// path still running then adds what it gathered (pt_applyPathQueueResult_kernel).
// While the stream holds the whole frame (W*H <= 640,000 there), a path that
// ended at bounce b runs bounces b+1 .. T of the restart, T the frame's last
// first-generation bounce, which no other path influences.  So the restarts
// are traced as a second wavefront after the first: tend[k] = T of frame k,
// and the restart's depth bound is min(eye depth, T - b).

// tend[k] = max over the frame's slots of the bounce its path ended at.
__global__ __launch_bounds__(kBlock) void k_term_max(const uint32_t* __restrict__ tb, uint32_t wh,
                                                     uint32_t* __restrict__ tend) {
  __shared__ uint32_t wmax[kBlock / 64];
  const uint32_t k = blockIdx.y;
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  uint32_t v = i < wh ? tb[(size_t)k * wh + i] : 0u;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v = max(v, (uint32_t)__shfl_xor(v, o, 64));
  if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t m = 0;
    for (int w = 0; w < kBlock / 64; w++) m = max(m, wmax[w]);
    if (m) atomicMax(&tend[k], m);
  }
}

// The restarts: sample slot sid of frame k when its path ended before tend[k],
// visited pixel-major as k_gen_eye lays out first paths; workgroups of 1024 so
// that the append takes a quarter of the atomics on the one counter (the
// restart pass took 3.9 ms at 1280 x 720 x 64 frames with 256).
constexpr int kRegenBlock = 1024;
__global__ __launch_bounds__(kRegenBlock) void k_gen_regen(FrameArgs fa, PathBuf pb, const uint32_t* __restrict__ tb,
                                                      const uint64_t* __restrict__ trng,
                                                      const uint32_t* __restrict__ tend,
                                                      const float4* __restrict__ rec_acc,
                                                      FrameCounters* __restrict__ fc) {
  __shared__ uint32_t wc[kRegenBlock / 64], base;
  const uint32_t wh = fa.width * fa.height;
  const uint32_t i = blockIdx.x * kRegenBlock + threadIdx.x;
  bool take = false;
  PathState p;
  if (i < wh * fa.nframes) {
    const uint32_t K = fa.nframes, pix = i / K, k = i - pix * K, sid = k * wh + pix;
    const uint32_t b = tb[sid], T = tend[k];
    if (b < T) {
      take = true;
      p = eye_path_at(fa, pix, sid, trng[sid]);
      p.fk = k;
      p.lim = min(T - b, fa.eye_depth);
      p.acc = rec_acc[sid];
    }
  }
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const unsigned long long m = __ballot(take);
  if (lane == 0) wc[wid] = (uint32_t)__popcll(m);
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t t = 0;
    for (int w = 0; w < kRegenBlock / 64; w++) t += wc[w];
    base = t ? atomicAdd(&fc->active[0], t) : 0u;
  }
  __syncthreads();
  if (take) {
    uint32_t slot = base + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
    for (int w = 0; w < wid; w++) slot += wc[w];
    pb.ray_o[slot] = p.ro;
    pb.ray_d[slot] = p.rd;
    pb.pix[slot] = p.pix;
    pb.sid[slot] = p.sid;
    pb.depth[slot] = pack_dk(p);
    pb.mul[slot] = p.mul;
    pb.smp[slot] = p.smp;
    pb.acc[slot] = p.acc;
    pb.rng[slot] = p.rng;
  }
}
hipError_t launch_regen(const FrameArgs& fa, PathBuf pb, const Accum& ac, FrameCounters* fc, hipStream_t st) {
  const uint32_t wh = fa.width * fa.height;
  const uint64_t n = (uint64_t)wh * fa.nframes;
  if (n == 0) return hipSuccess;
  if (!pathbuf_ok(pb) || !fc || !ac.term_bounce || !ac.term_rng || !ac.tend || !ac.rec.acc || fa.nframes > 255 ||
      fa.views)
    return hipErrorInvalidValue;
  k_fill_n_u32<<<1, kBlock, 0, st>>>(ac.tend, fa.nframes, 0u);
  k_term_max<<<dim3((wh + kBlock - 1) / kBlock, fa.nframes), kBlock, 0, st>>>(ac.term_bounce, wh, ac.tend);
  k_frame_begin<<<1, 64, 0, st>>>(fc, 0u);
  k_gen_regen<<<(uint32_t)((n + kRegenBlock - 1) / kRegenBlock), kRegenBlock, 0, st>>>(fa, pb, ac.term_bounce, ac.term_rng, ac.tend,
                                                                         ac.rec.acc, fc);
  return hipGetLastError();
}

// ---------------------------------------------------------------- "Path Regen" BDPT
// The reference's megakernel BDPT renderer (src/cudaRTBDPTRegen.cu, the
// "Path Regen" baseline), one thread per pixel.
//  - k_regen_light, every third frame: 128 light paths of 5 vertices each fill
//    a 640-vertex cache (bdpt_light_kernel :314-330, bdpt_light_ray
//    :80-309).  A path starts on a random emissive triangle (vertex: irrad =
//    emissive, no direction) and then carries the throughput (1, 1, 1), not
//    the emission (:179, :307); later vertices store the throughput they
//    arrived with and the hit's interpolated normal; a miss stores an empty
//    vertex, and the next vertex starts a new path, as does a throughput
//    below 1e-4.
//  - k_regen_eye: pt0_normalRay's recursion (:433-625) as a loop over at most
//    eye_depth levels with the per-level factors kept in registers: the BRDF
//    bounce (refraction past the critical angle reflects, :501-505), Russian
//    roulette on the pixel weight, whose failure restarts a camera path for
//    the same pixel (:562-571) and whose success connects a diffuse bounce to a
//    uniformly chosen cache vertex; then the radiance summed back up the
//    levels, r = f * r' + emission + connection, banked where a camera path
//    starts (:598-606), and the pixel's running mean over the count of camera
//    paths plus 4 per contributing connection (:655-664).
constexpr uint32_t kRegenLightN = kRegenLightVerts, kRegenLightDepth = 5, kRegenMaxLevels = 8;
constexpr uint32_t kDomainRegenLight = 4u, kDomainRegenEye = 5u;

template <bool Q>
__global__ __launch_bounds__(kRegenLightN / kRegenLightDepth) void k_regen_light(DevScene sc, FrameArgs fa,
                                                                                  LightVert* __restrict__ lv) {
  __shared__ TravLds<8, Q> lds;
  const uint32_t x = threadIdx.x;
  const uint64_t inc = ((uint64_t)x << 1) | 1u;
  uint64_t st;
  pcg32_seed(st, inc, stream_key(fa.seed, fa.frame0, kDomainRegenLight, 0u));
  bool valid = false;
  f3 o = mk3(0.f, 0.f, 0.f), d = o, irr = o;
  const Surf none = {o, o, o, o, 0.f, 0.f, 0.f, 0.f};
  for (uint32_t k = 0; k < kRegenLightDepth; k++) {
    f3 mulT = mk3(1.f, 1.f, 1.f), no = o, nd = d;
    bool nvalid = false;
    LightVert& V = lv[x * kRegenLightDepth + k];
    store_lv(V, o * 0.f, o * 0.f, o * 0.f, o * 0.f, none);
    const bool start = !valid || length(irr) < (float)kBiasEps;
    TraceHit h;
    uint32_t nn = 0, nt = 0;
    const bool hit = trace_rays<false, 8, Q>(sc, lds, !start, o, d, kInfF, (float)kBiasEps, false, h, nn, nt);
    if (start) {
      if (sc.n_light_tris > 0) {                         // a new path on an emitter (:94-158)
        uint32_t id = (uint32_t)(uniform01(st, inc) * (float)sc.n_light_tris);
        if (id >= sc.n_light_tris) id = sc.n_light_tris - 1;
        float lw = uniform01(st, inc), lu = uniform01(st, inc);
        if (lw + lu > 1.f) { lw = 1.f - lw; lu = 1.f - lu; }
        const float lvv = (1.f - lw) - lu;
        const Surf s = fetch_surf(sc, sc.light_tris[id], lw, lu, lvv, true);
        f3 u, v;
        basis(s.norm, u, v);
        const float r1 = (float)(2.0 * kPiD * (double)uniform01(st, inc));
        const float r2cos = sqrtf(uniform01(st, inc));
        const float r2sin = 1.f - r2cos * r2cos;
        float s1, c1;
        sincos_def(r1, s1, c1);
        nd = normalize((s.norm * r2cos + (u * r2sin) * c1) + (v * r2sin) * s1);
        no = s.pos + s.norm * (float)kBiasEps;
        nvalid = true;
        store_lv(V, s.pos, s.norm, s.emissive, mk3(0.f, 0.f, 0.f), s);
      }
    } else {
      if (hit) {                                         // :159-299
        const float w = (1.f - h.u) - h.v;
        const Surf s = fetch_surf(sc, h.leaf, w, h.u, h.v, true);
        const f3 nl = dot(s.norm, d) < 0.f ? s.norm : s.norm * -1.f;
        const Bounce b = sample_bounce(st, inc, o, d, h.t, s, nl, RT_LIGHT, false, true);
        no = b.orig;
        nd = b.dir;
        nvalid = true;
        mulT = vmul(b.mul, irr);
        store_lv(V, s.pos, s.norm, irr, d * -1.f, s);
      }
    }
    valid = nvalid;
    o = no;
    d = nd;
    irr = mulT;
  }
}

template <int STK, bool Q>
__global__ __launch_bounds__(kBlock) void k_regen_eye(DevScene sc, FrameArgs fa, const LightVert* __restrict__ lv,
                                                      float* __restrict__ result, uint32_t* __restrict__ sample_n,
                                                      DevStats* __restrict__ stats) {
  __shared__ TravLds<STK, Q> lds;
  const uint32_t W = fa.width, H = fa.height, pix = blockIdx.x * kBlock + threadIdx.x;
  const int lane = threadIdx.x & 63;
  uint32_t ext = 0, shr = 0, paths = 0, en = 0, et = 0, sn = 0, stc = 0;
  {                                                      // whole waves: lanes past the image carry no path
    bool live = pix < W * H;
    const uint32_t levels = fa.eye_depth < kRegenMaxLevels ? fa.eye_depth : kRegenMaxLevels;
    const uint32_t y = pix / W, x = pix - y * W;
    const uint64_t inc = ((uint64_t)pix << 1) | 1u;
    uint64_t st;
    pcg32_seed(st, inc, stream_key(fa.seed, fa.frame0, kDomainRegenEye, 0u));
    const f3 cpos = mk3(fa.cam_pos[0], fa.cam_pos[1], fa.cam_pos[2]);
    const f3 cright = mk3(fa.cam_right[0], fa.cam_right[1], fa.cam_right[2]);
    const f3 cup = mk3(fa.cam_up[0], fa.cam_up[1], fa.cam_up[2]);
    const f3 cdir = mk3(fa.cam_dir[0], fa.cam_dir[1], fa.cam_dir[2]);
    const float Wf = (float)W, Hf = (float)H, tf = fa.tan_half;
    const float pu = ((((2.f * ((float)x + 0.5f)) / Wf - 1.f) * tf) * Wf) / Hf;   // pt0_kernel :646-647
    const float pv = ((2.f * ((float)y + 0.5f)) / Hf - 1.f) * tf;
    auto camera_ray = [&]() {
      const float au = pu + ((uniform01(st, inc) - 0.5f) / Hf) * tf;
      const float av = pv + ((uniform01(st, inc) - 0.5f) / Hf) * tf;
      return normalize((cright * au + cup * av) + cdir);
    };
    f3 o = cpos, d = camera_ray();
    float weight = 1.f;
    uint32_t depth = 0, count = 0, D = levels;
    f3 mul[kRegenMaxLevels], em[kRegenMaxLevels], con[kRegenMaxLevels];   // per level: f, emission, connection
    uint32_t bank = 0;                                     // levels where a camera path starts
    paths = live;
    for (uint32_t L = 0; L < levels; L++) {
      if (__ballot(live) == 0ull) break;                 // wave-uniform
      TraceHit h;
      ext += live;
      const bool hit = trace_rays<false, STK, Q>(sc, lds, live, o, d, kInfF, (float)kBiasEps, false, h, en, et);
      if (live && !hit) {                                // :620-623
        D = L;
        live = false;
      }
      // the level's bounce; a connection waits for its occlusion test below
      Surf s;
      Bounce b;
      f3 nl, P = o, toL = d, no = o, nd = d;
      float dist = 0.f;
      bool diffuse = false, lit = false;
      uint32_t li = 0;
      if (live) {
      const float w = (1.f - h.u) - h.v;
      s = fetch_surf(sc, h.leaf, w, h.u, h.v, true);
      nl = dot(s.norm, d) < 0.f ? s.norm : s.norm * -1.f;
      b = sample_bounce(st, inc, o, d, h.t, s, nl, RT_EYE, false, true);
      weight = weight * length(b.mul);
      if (length(s.emissive) > 0.f) weight = 0.f;
      if (depth == 0) bank |= 1u << L;
      no = b.orig;
      nd = b.dir;
      if (!prob_rand(st, inc, weight)) {                 // a new camera path for the pixel (:562-571)
        weight = 1.f;
        depth = 0;
        count++;
        no = cpos;
        nd = camera_ray();
        paths++;
      } else {
        depth++;
        if (b.type == RT_DIFF) {                          // GetLightFromRandLightVertices (:400-431)
          diffuse = true;
          P = s.pos + nl * (float)kBiasEps;
          li = (uint32_t)(uniform01(st, inc) * (float)kRegenLightN);
          if (li >= kRegenLightN) li = kRegenLightN - 1;
          const LightVert& LV = lv[li];
          const f3 lpos = mk3(LV.pos[0], LV.pos[1], LV.pos[2]), lirr = mk3(LV.irrad[0], LV.irrad[1], LV.irrad[2]);
          toL = normalize(lpos - P);
          dist = length(lpos - P);
          lit = length(lirr) > 0.f && dot(nl, toL) > 0.f;
        }
      }
      }
      bool occluded = false;
      if (__ballot(lit)) {
        TraceHit hs;
        shr += lit;
        occluded = trace_rays<true, STK, Q>(sc, lds, lit, P, toL, (float)shadow_max((double)dist, fa.flags),
                                            (float)kBiasEps, false, hs, sn, stc);
      }
      if (!live) continue;
      f3 c = mk3(0.f, 0.f, 0.f);
      if (diffuse) {
        const LightVert& LV = lv[li];
        f3 irrad = c, irradDir = c;
        if (lit) {
          const f3 lirr = mk3(LV.irrad[0], LV.irrad[1], LV.irrad[2]);
          const f3 ldir = mk3(LV.irradDir[0], LV.irradDir[1], LV.irradDir[2]);
          if (!occluded) {
            if (length(ldir) > (float)kFltEps)
              irrad = shading(toL * -1.f, ldir, lirr, mk3(LV.norm[0], LV.norm[1], LV.norm[2]),
                              mk3(LV.diff[0], LV.diff[1], LV.diff[2]), LV.metallic, LV.roughness, LV.specular,
                              1.f, 1.f) +
                      mk3(LV.emissive[0], LV.emissive[1], LV.emissive[2]);
            else
              irrad = lirr;
            irradDir = toL;
          }
        }
        c = vmax0(shading(d * -1.f, irradDir, irrad, nl, s.diff, s.metal, s.rough, s.spec, 1.f - s.trans, 1.f));
        if (length(c) > 0.f) count += 4;
      }
      mul[L] = b.mul;
      em[L] = s.emissive;
      con[L] = c;
      o = no;
      d = nd;
    }
    count++;                                               // the miss or the level bound (:620-630)
    f3 r = mk3(0.f, 0.f, 0.f), accum = r;
    for (uint32_t k = D; k-- > 0;) {
      r = (vmul(mul[k], r) + em[k]) + con[k];
      if ((bank >> k) & 1u) {
        accum = accum + r;
        r = mk3(0.f, 0.f, 0.f);
      }
    }
    if (pix < W * H) {
    const uint32_t nold = fa.frame0 == 0 ? 0u : sample_n[pix], nn = nold + count;
    const float ri = 1.f / (float)nn, oi = (float)nold * ri;
    float* res = result + (size_t)pix * 3;
    res[0] = fmaxf(ri * accum.x + oi * res[0], 0.f);
    res[1] = fmaxf(ri * accum.y + oi * res[1], 0.f);
    res[2] = fmaxf(ri * accum.z + oi * res[2], 0.f);
    sample_n[pix] = nn;
    }
  }
  if (stats) {
    stats = stat_slot(stats);
    if (blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(&stats->frames, 1ull);
    const uint32_t a0 = wave_sum(ext), a1 = wave_sum(shr), a2 = wave_sum(paths);
    const uint32_t b0 = wave_sum(en), b1 = wave_sum(et), b2 = wave_sum(sn), b3 = wave_sum(stc);
    if (lane == 0 && (a0 | a2)) {
      atomicAdd(&stats->ext_rays, (unsigned long long)a0);
      atomicAdd(&stats->shadow_rays, (unsigned long long)a1);
      atomicAdd(&stats->eye_paths, (unsigned long long)a2);
      atomicAdd(&stats->ext_nodes, (unsigned long long)b0);
      atomicAdd(&stats->ext_tris, (unsigned long long)b1);
      atomicAdd(&stats->sh_nodes, (unsigned long long)b2);
      atomicAdd(&stats->sh_tris, (unsigned long long)b3);
    }
  }
}

hipError_t launch_regen_light(const DevScene& sc, const FrameArgs& fa, LightVert* lv, int quant, hipStream_t st) {
  if (!lv || !sc.tris || !nodes_ok(sc, quant) || (sc.n_light_tris && !sc.light_tris)) return hipErrorInvalidValue;
  if (quant) k_regen_light<true><<<1, kRegenLightN / kRegenLightDepth, 0, st>>>(sc, fa, lv);
  else k_regen_light<false><<<1, kRegenLightN / kRegenLightDepth, 0, st>>>(sc, fa, lv);
  return hipGetLastError();
}
hipError_t launch_regen_eye(const DevScene& sc, const FrameArgs& fa, const LightVert* lv, float* result,
                            uint32_t* sample_n, int lds_stack, int quant, DevStats* stats, hipStream_t st) {
  const uint64_t n = (uint64_t)fa.width * fa.height;
  if (n == 0) return hipSuccess;
  if (!lv || !result || !sample_n || n > 0xFFFFFFFFull - kBlock || fa.eye_depth < 1 ||
      fa.eye_depth > kRegenMaxLevels || !sc.tris || !nodes_ok(sc, quant))
    return hipErrorInvalidValue;
  const uint32_t grid = (uint32_t)((n + kBlock - 1) / kBlock);
#define CPT_RG(S, W, Q) k_regen_eye<S, Q><<<grid, kBlock, 0, st>>>(sc, fa, lv, result, sample_n, stats)
#define CPT_RG_Q(S, W) CPT_RG(S, W, true)
#define CPT_RG_F(S, W) CPT_RG(S, W, false)
  if (quant) {
    CPT_VARIANT_SWITCH(lds_stack, CPT_RG_Q)
  } else {
    CPT_VARIANT_SWITCH(lds_stack, CPT_RG_F)
  }
#undef CPT_RG_Q
#undef CPT_RG_F
#undef CPT_RG
  return hipGetLastError();
}

// ---------------------------------------------------------------- megakernel
// The reference's regeneration baseline (cudaRTBDPTRegen: one thread carries
// its sample through every bounce, src/cudaRTBDPTRegen.cu) over this library's
// functions: one thread per sample slot of the batch generates the eye path
// (eye_path), and per bounce traces the closest hit (traverse4), shades it
// (shade_path) and traces the connection's occlusion ray, adding the
// contribution when nothing occludes it.  The per-path arithmetic and its order
// are those of the wavefront passes (k_gen_eye, k_trace_dyn, k_shade,
// k_shadow), so the image is the same bit for bit; only the schedule differs:
// no path buffers, no compaction, and lanes of a wave idle once their paths
// end.  The frame counters receive the same per-bounce counts.  Bound by the latency of its
// chain of node visits: four waves a SIMD (128 VGPRs, 14 of them spilled outside
// the traversal) take 936 us for an 800 x 600 frame on the sphere grid, three (143) 977.
// One bounce of a path that one thread carries (k_mega, k_tail): the closest
// hit, shade_path, and the occlusion ray of the connection it sets up, whose
// contribution is added when nothing occludes it.
// Called by whole waves; `live` lanes carry a path.
template <int STK, bool Q>
__device__ __forceinline__ void carry_bounce(const DevScene& sc, const FrameArgs& fa, FrameCounters* fc,
                                             const LightVert* lv, const Accum& ac, PathState& p,
                                             TravLds<STK, Q>& lds, bool live, bool& survive, bool& emit, uint32_t& en,
                                             uint32_t& et, uint32_t& sn, uint32_t& st) {
  TraceHit h;
  const bool hit = trace_rays<false, STK, Q>(sc, lds, live, ld3(p.ro), ld3(p.rd), p.ro.w, p.rd.w, false, h, en, et);
  ShadowRay sr;
  sr.o = sr.d = sr.c = make_float4(0.f, 0.f, 0.f, 0.f);
  if (live) {
    const float4 hv = make_float4(hit ? h.t : kInfF, __uint_as_float(hit ? h.leaf : kInvalid), hit ? h.u : 0.f,
                                  hit ? h.v : 0.f);
    shade_path(sc, fa, fc, lv, ac, p, hv, survive, emit, sr);
  }
  if (__ballot(emit) == 0ull) return;                       // wave-uniform
  TraceHit hs;
  const bool occluded =
      trace_rays<true, STK, Q>(sc, lds, emit, ld3(sr.o), ld3(sr.d), sr.o.w, sr.d.w, false, hs, sn, st);
  if (emit && !occluded) {
    p.acc.x = p.acc.x + sr.c.x;
    p.acc.y = p.acc.y + sr.c.y;
    p.acc.z = p.acc.z + sr.c.z;
    p.acc.w = __uint_as_float(__float_as_uint(p.acc.w) + 4u);
  }
}

// A workgroup's counts: live and shadow rays per bounce; nodes and triangles of
// the extension and the shadow rays, then the tail's nodes, triangles and rays.
struct CarryCounts {
  uint32_t live[16], shadow[16], trav[8];
};
__device__ __forceinline__ void carry_counts_clear(CarryCounts& C) {
  static_assert(sizeof(CarryCounts) == 40 * 4, "one word a thread");
  if (threadIdx.x < 40) ((uint32_t*)&C)[threadIdx.x] = 0u;
  __syncthreads();
}
// Adds one bounce of a wave.  Called by the whole wave.
__device__ __forceinline__ void carry_count(CarryCounts& C, uint32_t b, bool tail, uint32_t rays, bool survive,
                                            bool emit, uint32_t en, uint32_t et, uint32_t sn, uint32_t st) {
  const uint32_t cs = (uint32_t)__popcll(__ballot(survive)), ce = (uint32_t)__popcll(__ballot(emit));
  const uint32_t a0 = wave_sum(en), a1 = wave_sum(et), a2 = wave_sum(sn), a3 = wave_sum(st);
  if ((threadIdx.x & 63) == 0) {
    atomicAdd(&C.live[b], cs);
    atomicAdd(&C.shadow[b], ce);
    atomicAdd(&C.trav[tail ? 4 : 0], tail ? a0 + a2 : a0);
    atomicAdd(&C.trav[tail ? 5 : 1], tail ? a1 + a3 : a1);
    atomicAdd(&C.trav[tail ? 6 : 2], tail ? rays : a2);
    if (!tail) atomicAdd(&C.trav[3], a3);
  }
}
// Into the frame counters and the statistics.
__device__ __forceinline__ void carry_flush(FrameCounters* fc, DevStats* stats, const CarryCounts& C, uint32_t depth) {
  __syncthreads();
  const uint32_t t = threadIdx.x;
  if (t < depth) {
    uint32_t* part = fc->part[blockIdx.x % kPartSlots];
    if (t + 1 < 16 && C.live[t]) atomicAdd(&part[t + 1], C.live[t]);
    if (C.shadow[t]) atomicAdd(&part[16 + t], C.shadow[t]);
  }
  if (stats && t < 7 && C.trav[t]) {
    stats = stat_slot(stats);
    unsigned long long* to[7] = {&stats->ext_nodes, &stats->ext_tris, &stats->sh_nodes, &stats->sh_tris,
                                 &stats->tail_nodes, &stats->tail_tris, &stats->tail_rays};
    atomicAdd(to[t], (unsigned long long)C.trav[t]);
  }
}

// Paths a wave carries: 64, but no more than spread a launch over half the waves
// resident at once (`waves`), down to 16: a step of fewer rays tests its
// triangles in fewer rounds and waits for fewer paths, while more waves a SIMD
// wait for each other.  Frames of 128 x 128 and 256 x 256 paths on the sphere grid,
// us: 64 a wave 303 / 386, over all resident waves (16) 246 / 354, over half of them
// (16 / 32) 248 / 360; of 256 x 256 on the Cornell box 179 / 203 / 180.
__host__ __device__ __forceinline__ uint32_t carry_paths(uint32_t n, uint32_t waves) {
  const uint32_t w2 = waves / 2u, per = n / w2 + (n % w2 ? 1u : 0u);
  return per < 16u ? 16u : per > 64u ? 64u : per;
}

template <int STK, bool Q>
__global__ __launch_bounds__(kBlock, 4) void k_mega(DevScene sc, FrameArgs fa, FrameCounters* __restrict__ fc,
                                                 const LightVert* __restrict__ lv, Accum ac,
                                                 DevStats* __restrict__ stats, uint32_t per) {
  __shared__ TravLds<STK, Q> lds;
  __shared__ CarryCounts counts;
  carry_counts_clear(counts);
  const int lane = threadIdx.x & 63;
  const uint32_t i = (blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6)) * per + lane;
  bool live = lane < (int)per && i < fa.width * fa.height * fa.nframes;
  PathState p;
  if (live) {                                               // pixel-major, as k_gen_eye
    uint32_t dk;
    p = eye_slot(fa, i, dk);
    unpack_dk(p, dk);
    if (ac.variant & kVariantGbuf) zero_rec(ac.rec, p.sid); // a miss leaves the G-buffer record at zero
  }
  const uint32_t depth = fa.eye_depth < 16u ? fa.eye_depth : 16u;
  for (uint32_t b = 0; b < depth; b++) {
    if (__ballot(live) == 0ull) break;                    // wave-uniform
    bool survive = false, emit = false;
    uint32_t en = 0, et = 0, sn = 0, st = 0;
    carry_bounce<STK, Q>(sc, fa, fc, lv, ac, p, lds, live, survive, emit, en, et, sn, st);
    live = survive;
    carry_count(counts, b, false, 0u, survive, emit, en, et, sn, st);
  }
  carry_flush(fc, stats, counts, depth);
}

// The last bounces of the wavefront in one launch.  Once few paths are left,
// a bounce's refilling grid runs partly empty and each of its three launches
// (extension, shading, occlusion) waits for its slowest ray; from bounce
// `bounce0` on, each wave instead takes live slots of `cur` (strided over a
// persistent grid) and carries each path through the remaining bounces as
// k_mega does, with the same per-path arithmetic: the image does not change.
// Traversal of bounces before `tail0` counts as extension and shadow work, of
// the others as the tail's.  waves: those resident at once (carry_paths).
template <int STK, bool Q>
__global__ __launch_bounds__(kBlock, 4) void k_tail(DevScene sc, FrameArgs fa, PathBuf cur,
                                                 FrameCounters* __restrict__ fc, uint32_t bounce0, uint32_t tail0,
                                                 const LightVert* __restrict__ lv, Accum ac,
                                                 DevStats* __restrict__ stats, uint32_t waves) {
  __shared__ TravLds<STK, Q> lds;
  __shared__ CarryCounts counts;
  carry_counts_clear(counts);
  const uint32_t count = fc->active[bounce0];
  const uint32_t per = carry_paths(count, waves);
  const int lane = threadIdx.x & 63;
  const uint32_t depth = fa.eye_depth < 16u ? fa.eye_depth : 16u;
  const uint32_t wave = blockIdx.x * (kBlock / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (uint32_t base = wave * per; base < count; base += gridDim.x * (kBlock / 64) * per) {   // wave-uniform
    const uint32_t i = base + lane;
    bool live = lane < (int)per && i < count;
    PathState p;
    if (live) {
      p.ro = cur.ray_o[i];
      p.rd = cur.ray_d[i];
      p.pix = cur.pix[i];
      p.sid = cur.sid[i];
      p.rng = cur.rng[i];
      const uint32_t dk = cur.depth[i];
      unpack_dk(p, dk);
      if (dk & kFreshPath) {
        p.mul = make_float4(1.f, 1.f, 1.f, 0.f);
        p.smp = make_float4(0.f, 0.f, 0.f, 0.f);
        p.acc = p.smp;
      } else {
        p.mul = cur.mul[i];
        p.smp = cur.smp[i];
        p.acc = cur.acc[i];
      }
    }
    for (uint32_t b = bounce0; b < depth; b++) {
      if (__ballot(live) == 0ull) break;                  // wave-uniform
      bool survive = false, emit = false;
      uint32_t en = 0, et = 0, sn = 0, st = 0;
      const uint32_t rays = (uint32_t)__popcll(__ballot(live));
      carry_bounce<STK, Q>(sc, fa, fc, lv, ac, p, lds, live, survive, emit, en, et, sn, st);
      live = survive;
      carry_count(counts, b, b >= tail0, rays, survive, emit, en, et, sn, st);
    }
  }
  carry_flush(fc, stats, counts, depth);
}
hipError_t launch_tail(const DevScene& sc, const FrameArgs& fa, PathBuf cur, FrameCounters* fc, uint32_t bounce0,
                       uint32_t tail0, uint32_t groups, uint32_t cus, const LightVert* lv, const Accum& ac,
                       int lds_stack, int quant, DevStats* stats, hipStream_t st) {
  if (!fc || !lv || !ac.rec.acc || fa.eye_depth > 16 ||
      bounce0 >= fa.eye_depth || groups == 0 || cus == 0 || !pathbuf_ok(cur) || !sc.tris || !nodes_ok(sc, quant))
    return hipErrorInvalidValue;
#define CPT_TL(S, W, Q)                                                                                           \
  {                                                                                                               \
    static const uint32_t resident = resident_groups((const void*)k_tail<S, Q>);                                  \
    k_tail<S, Q><<<groups * cus, kBlock, 0, st>>>(sc, fa, cur, fc, bounce0, tail0, lv, ac, stats,                 \
                                                  resident * cus * (kBlock / 64));                                \
  }
#define CPT_TL_Q(S, W) CPT_TL(S, W, true)
#define CPT_TL_F(S, W) CPT_TL(S, W, false)
  if (quant) {
    CPT_VARIANT_SWITCH(lds_stack, CPT_TL_Q)
  } else {
    CPT_VARIANT_SWITCH(lds_stack, CPT_TL_F)
  }
#undef CPT_TL_Q
#undef CPT_TL_F
#undef CPT_TL
  return hipGetLastError();
}
hipError_t launch_mega(const DevScene& sc, const FrameArgs& fa, FrameCounters* fc, const LightVert* lv,
                       const Accum& ac, int lds_stack, int quant, uint32_t cus, DevStats* stats, hipStream_t st) {
  const uint64_t n = (uint64_t)fa.width * fa.height * fa.nframes;
  if (n == 0) return hipSuccess;
  if (n > 0xFFFFFFFFull - 4 * kBlock || !fc || !lv || !ac.rec.acc || fa.eye_depth > 16 || cus == 0 || !sc.tris ||
      !nodes_ok(sc, quant) || ((ac.variant & kVariantGbuf) && !rec_ok(ac.rec)))
    return hipErrorInvalidValue;
#define CPT_MG(S, W, Q)                                                                                           \
  {                                                                                                               \
    static const uint32_t resident = resident_groups((const void*)k_mega<S, Q>);                                  \
    const uint32_t per = carry_paths((uint32_t)n, resident * cus * (kBlock / 64)), wg = per * (kBlock / 64);      \
    k_mega<S, Q><<<(uint32_t)((n + wg - 1) / wg), kBlock, 0, st>>>(sc, fa, fc, lv, ac, stats, per);               \
  }
  if (quant) {
#define CPT_MG_Q(S, W) CPT_MG(S, W, true)
#define CPT_MG_F(S, W) CPT_MG(S, W, false)
    CPT_VARIANT_SWITCH(lds_stack, CPT_MG_Q)
  } else {
    CPT_VARIANT_SWITCH(lds_stack, CPT_MG_F)
  }
#undef CPT_MG_Q
#undef CPT_MG_F
#undef CPT_MG
  return hipGetLastError();
}

// ---------------------------------------------------------------- adaptive sampling
// e^-a for a that is 0 or more, or NaN (0 past 103): Cody-Waite reduction +
// degree-7 Taylor polynomial, 2^k by ldexp (Cody & Waite 1980).  The host oracle
// evaluates the identical fma sequence.
__device__ __forceinline__ float cpt_exp_neg(float a) {
  const float k = rintf(-a * 1.44269504f);
  float r = fmaf(k, -0.693145751953125f, -a);
  r = fmaf(k, -1.42860676533018e-06f, r);
  float p = 1.f / 5040.f;
  p = fmaf(p, r, 1.f / 720.f);
  p = fmaf(p, r, 1.f / 120.f);
  p = fmaf(p, r, 1.f / 24.f);
  p = fmaf(p, r, 1.f / 6.f);
  p = fmaf(p, r, 0.5f);
  p = fmaf(p, r, 1.f);
  p = fmaf(p, r, 1.f);
  const float e = ldexpf(p, (int)k);
  return a > 103.f ? 0.f : e;
}
__device__ __forceinline__ float sqdist3(const float* a, const float* b) {
  float dx = a[0] - b[0], dy = a[1] - b[1], dz = a[2] - b[2];
  return (dx * dx + dy * dy) + dz * dz;
}
// |a - b|^2 of a filter range term: fma(dz, dz, fma(dy, dy, dx * dx)).
__device__ __forceinline__ float sqd_fma(const float* a, const float* b) {
  const float dx = a[0] - b[0], dy = a[1] - b[1], dz = a[2] - b[2];
  return __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
}
// Coordinate as the reference clamps it: (x + j) is unsigned, so a negative
// coordinate wraps and lands on the high edge (cudaBilateralFilter.cu:85).
__device__ __forceinline__ uint32_t ref_clamp_i(int v, uint32_t n) {
  return (v < 0 || (uint32_t)v >= n) ? n - 1 : (uint32_t)v;
}

constexpr int kTile = 16;
constexpr int kLdsRadius = 9;     // LDS tile path up to this radius, global reads beyond

// Cross-bilateral over colour/position/normal(/albedo) + the weighted squared
// residual of pt_calculateSquareError_kernel.  One exponential per tap: the
// range terms' exponents are summed, each scaled by its 1 / 2 sigma^2 (correctly rounded
// once per thread) and accumulated with fmas, so a tap takes no division.
// A pixel's guides, and for an image the pixel's own value and the sums so far,
// taps added in raster order.
struct FilterPixel {
  float p[3], n[3], d[3], z, iz;
};
struct FilterSums {
  float c[3], sum, t0, t1, t2;
};
struct FilterScale {
  float c, p, n, d, z;
};
struct FilterTap {
  float c[3], p[3], n[3], d[3], z, c2[3];
};
// The squared distances of a tap's guides.
struct FilterTerms {
  float p, n, d, z;
};
template <bool DIFF, bool DEPTH>
__device__ __forceinline__ FilterTerms filter_terms(const FilterPixel& P, const FilterTap& q) {
  FilterTerms t;
  t.p = sqd_fma(q.p, P.p);
  t.n = sqd_fma(q.n, P.n);
  t.d = DIFF ? sqd_fma(q.d, P.d) : 0.f;
  const float dz = DEPTH ? (q.z - P.z) * P.iz : 0.f;
  t.z = dz * dz;
  return t;
}
// The tap's negated exponent: 0 or more, or NaN (every scale is the reciprocal of a square).
template <bool DIFF, bool DEPTH>
__device__ __forceinline__ float filter_exponent(const float* c, const float* qc, const FilterTerms& t,
                                                 const FilterScale& k) {
  float a = sqd_fma(qc, c) * k.c;
  a = __builtin_fmaf(t.p, k.p, a);
  a = __builtin_fmaf(t.n, k.n, a);
  if (DIFF) a = __builtin_fmaf(t.d, k.d, a);
  if (DEPTH) a = __builtin_fmaf(t.z, k.z, a);
  return a;
}
__device__ __forceinline__ void filter_add(FilterSums& S, const float* qc, float a, float w) {
  const float f = w * cpt_exp_neg(a);
  S.t0 = __builtin_fmaf(f, qc[0], S.t0);
  S.t1 = __builtin_fmaf(f, qc[1], S.t1);
  S.t2 = __builtin_fmaf(f, qc[2], S.t2);
  S.sum = S.sum + f;
}
// A tap of exponent past 103 weighs exactly 0 and adds nothing to finite sums;
// infinite exponents (infinite guides) are left to the arithmetic.
__device__ __forceinline__ bool filter_zero(float a) { return a > 103.f && a < __builtin_huge_valf(); }
__device__ __forceinline__ void filter_store(const FilterArgs& fa, const FilterSums& S, uint32_t x, uint32_t y,
                                             const uint32_t* __restrict__ sample_n, float* __restrict__ filtered,
                                             float* __restrict__ err) {
  const size_t ind = (size_t)y * fa.width + x;
  const float o0 = S.t0 / S.sum, o1 = S.t1 / S.sum, o2 = S.t2 / S.sum;
  filtered[ind * 3] = o0;
  filtered[ind * 3 + 1] = o1;
  filtered[ind * 3 + 2] = o2;
  // pt_calculateSquareError_kernel (AdapBilatAtomic.cu:1143-1156)
  const uint32_t sn = sample_n[ind];
  float red = (float)fa.nd / (float)(fa.nd + sn);
  if (fa.nd + sn < sn) red = 0.f;
  const float d0 = o0 - S.c[0], d1 = o1 - S.c[1], d2 = o2 - S.c[2];
  err[ind] = red * ((d0 * d0 + d1 * d1) + d2 * d2) / 3.f;
}
template <bool DIFF, bool DEPTH>
__device__ __forceinline__ void filter_start(FilterPixel& P, const FilterTap& q) {
#pragma unroll
  for (int c = 0; c < 3; c++) {
    P.p[c] = q.p[c]; P.n[c] = q.n[c];
    P.d[c] = DIFF ? q.d[c] : 0.f;
  }
  P.z = DEPTH ? q.z : 0.f;
  P.iz = P.z > 0.f ? 1.f / P.z : 0.f;
}
__device__ __forceinline__ void filter_start(FilterSums& S, const float* qc) {
#pragma unroll
  for (int c = 0; c < 3; c++) S.c[c] = qc[c];
  S.sum = S.t0 = S.t1 = S.t2 = 0.f;
}
__device__ __forceinline__ FilterScale filter_scale(const FilterArgs& fa, bool depth) {
  return {1.f / fa.kc, 1.f / fa.kp, 1.f / fa.kn, 1.f / fa.kd, depth ? 1.f / fa.kz : 0.f};
}

// A 16 x 16 tile a workgroup.  Bound by the arithmetic of the taps (48 instructions each with
// the albedo guide; the SIMDs' every cycle is taken), so what is not arithmetic is
// kept small: the halo of (16 + 2R)^2 pixels lies in LDS as records
// of 12 words, read as 128-bit words that no two lanes of a 16-lane group
// share a bank for; the products of the spatial weights are tabled; the depth term is
// its own instance; a tap that weighs 0 in the whole wave ends early.  1920 x 1080,
// radius 5, with / without the albedo guide: 280 / 244 us; planes of single words,
// weights multiplied per tap and a depth branch took 381 / 305 (71 instructions a tap),
// at radius 7 735 / 558 against 524 / 467.  Two pixels of a column a thread, which share each
// record, 279 / 242 and 572 / 517: twice the LDS leaves half the waves.
// PAIR: a second image (color2) under the same guides in the same pass, whose taps share the
// records and the guides' distances; its pixels take the words of the record that are free.
// Image and second moment of the learned frames (1920 x 1080, radius 7, depth): 760 us,
// two passes 1044.
// REC: words a record.  At radius 9 records of 12 words leave two workgroups on a compute unit,
// of 10 three; without albedo and second image 10 hold a pixel (read as 64-bit words,
// again free of conflicts).  1000 x 700, radius 9: 399 us with 12, 290 with 10.
template <bool DIFF, bool DEPTH, bool PAIR, int REC>
__global__ __launch_bounds__(kTile * kTile) void k_filter_lds(FilterArgs fa, const float* __restrict__ color,
                                                              const float* __restrict__ gpos,
                                                              const float* __restrict__ gnrm,
                                                              const float* __restrict__ gdif,
                                                              const uint32_t* __restrict__ sample_n,
                                                              float* __restrict__ filtered, float* __restrict__ err,
                                                              const float* __restrict__ color2,
                                                              float* __restrict__ filtered2,
                                                              float* __restrict__ err2) {
  static_assert(!(DIFF && PAIR), "a pair's record has no room for the albedo");
  static_assert(REC == 12 || (REC == 10 && !DIFF && !PAIR), "words of a record");
  extern __shared__ float4 sm[];
  const int R = (int)fa.radius, D = 2 * R + 1, TW = kTile + 2 * R, TA = TW * TW;
  const uint32_t W = fa.width, H = fa.height;
  const int tx = threadIdx.x, ty = threadIdx.y, tid = ty * kTile + tx;
  const int bx = blockIdx.x * kTile, by = blockIdx.y * kTile;
  float* rec = (float*)sm;                         // c, p, n, then d, or z and two words of c2, or c2
  float* wt = rec + REC * (size_t)TA;              // spatial weight of tap (i, j)
  float* sz = wt + (size_t)D * D;                  // DEPTH: z (DIFF) or c2's last (PAIR) per halo pixel
  const float cam[3] = {fa.cam[0], fa.cam[1], fa.cam[2]};
  for (int k = tid; k < D * D; k += kTile * kTile) {
    const int i = k / D, j = k - i * D;
    wt[k] = fa.gauss[i] * fa.gauss[j];
  }
  for (int k = tid; k < TA; k += kTile * kTile) {
    const int hy = k / TW, hx = k - hy * TW;
    const size_t g = ((size_t)ref_clamp_i(by + hy - R, H) * W + ref_clamp_i(bx + hx - R, W)) * 3;
    float* r = rec + REC * k;
#pragma unroll
    for (int c = 0; c < 3; c++) {
      r[c] = color[g + c];
      r[3 + c] = gpos[g + c];
      r[6 + c] = gnrm[g + c];
      if (DIFF) r[9 + c] = gdif[g + c];
    }
    if (DEPTH) {
      const float z = sqrtf(sqdist3(gpos + g, cam));
      if (DIFF) sz[k] = z; else r[9] = z;
    }
    if (PAIR) {
      constexpr int at = DEPTH ? 10 : 9;
      r[at] = color2[g];
      r[at + 1] = color2[g + 1];
      if (DEPTH) sz[k] = color2[g + 2]; else r[11] = color2[g + 2];
    }
  }
  __syncthreads();
  const auto load = [&](int k) {
    FilterTap q;
    if constexpr (REC == 10) {
      const float2* r = (const float2*)(rec + 10 * k);
      const float2 a = r[0], b = r[1], c = r[2], d = r[3], e = r[4];
      q.c[0] = a.x; q.c[1] = a.y; q.c[2] = b.x;
      q.p[0] = b.y; q.p[1] = c.x; q.p[2] = c.y;
      q.n[0] = d.x; q.n[1] = d.y; q.n[2] = e.x;
      q.z = DEPTH ? e.y : 0.f;
      return q;
    }
    const float4* r = (const float4*)(rec + 12 * k);
    const float4 a = r[0], b = r[1], c = r[2];
    q.c[0] = a.x; q.c[1] = a.y; q.c[2] = a.z;
    q.p[0] = a.w; q.p[1] = b.x; q.p[2] = b.y;
    q.n[0] = b.z; q.n[1] = b.w; q.n[2] = c.x;
    q.d[0] = c.y; q.d[1] = c.z; q.d[2] = c.w;
    q.z = DEPTH ? (DIFF ? sz[k] : c.y) : 0.f;
    q.c2[0] = DEPTH ? c.z : c.y; q.c2[1] = DEPTH ? c.w : c.z; q.c2[2] = PAIR && DEPTH ? sz[k] : c.w;
    return q;
  };
  const FilterScale ks = filter_scale(fa, DEPTH);
  const uint32_t x = bx + tx, y = by + ty;
  FilterPixel P;
  FilterSums S, S2;
  {
    const FilterTap q = load((ty + R) * TW + tx + R);
    filter_start<DIFF, DEPTH>(P, q);
    filter_start(S, q.c);
    if (PAIR) filter_start(S2, q.c2);
  }
  for (int i = 0; i < D; i++) {
    const int row = (ty + i) * TW + tx;
    for (int j = 0; j < D; j++) {
      const FilterTap q = load(row + j);
      const FilterTerms t = filter_terms<DIFF, DEPTH>(P, q);
      const float a = filter_exponent<DIFF, DEPTH>(S.c, q.c, t, ks);
      const float a2 = PAIR ? filter_exponent<DIFF, DEPTH>(S2.c, q.c2, t, ks) : 0.f;
      if (__ballot(!(filter_zero(a) && (!PAIR || filter_zero(a2)))) == 0ull) continue;
      const float w = wt[i * D + j];
      filter_add(S, q.c, a, w);
      if (PAIR) filter_add(S2, q.c2, a2, w);
    }
  }
  if (x < W && y < H) {
    filter_store(fa, S, x, y, sample_n, filtered, err);
    if (PAIR) filter_store(fa, S2, x, y, sample_n, filtered2, err2);
  }
}

// Radii whose halo does not fit: every tap read from memory.
template <bool DIFF, bool DEPTH>
__global__ __launch_bounds__(kTile * kTile) void k_filter_mem(FilterArgs fa, const float* __restrict__ color,
                                                              const float* __restrict__ gpos,
                                                              const float* __restrict__ gnrm,
                                                              const float* __restrict__ gdif,
                                                              const uint32_t* __restrict__ sample_n,
                                                              float* __restrict__ filtered, float* __restrict__ err) {
  __shared__ float sg[2 * kMaxFilterRadius + 2];
  const int R = (int)fa.radius;
  const uint32_t W = fa.width, H = fa.height;
  const int tid = threadIdx.y * kTile + threadIdx.x;
  const uint32_t x = blockIdx.x * kTile + threadIdx.x, y = blockIdx.y * kTile + threadIdx.y;
  const float cam[3] = {fa.cam[0], fa.cam[1], fa.cam[2]};
  if (tid < 2 * R + 1) sg[tid] = fa.gauss[tid];
  __syncthreads();
  if (x >= W || y >= H) return;
  const auto load = [&](int yy, int xx) {
    const size_t g = ((size_t)ref_clamp_i(yy, H) * W + ref_clamp_i(xx, W)) * 3;
    FilterTap q;
#pragma unroll
    for (int c = 0; c < 3; c++) {
      q.c[c] = color[g + c]; q.p[c] = gpos[g + c]; q.n[c] = gnrm[g + c];
      q.d[c] = DIFF ? gdif[g + c] : 0.f;
    }
    q.z = DEPTH ? sqrtf(sqdist3(gpos + g, cam)) : 0.f;
    return q;
  };
  const FilterScale ks = filter_scale(fa, DEPTH);
  FilterPixel P;
  FilterSums S;
  {
    const FilterTap q = load((int)y, (int)x);
    filter_start<DIFF, DEPTH>(P, q);
    filter_start(S, q.c);
  }
  for (int i = -R; i <= R; i++)
    for (int j = -R; j <= R; j++) {
      const FilterTap q = load((int)y + i, (int)x + j);
      const float a = filter_exponent<DIFF, DEPTH>(S.c, q.c, filter_terms<DIFF, DEPTH>(P, q), ks);
      filter_add(S, q.c, a, sg[i + R] * sg[j + R]);
    }
  filter_store(fa, S, x, y, sample_n, filtered, err);
}

hipError_t launch_filter_error(const FilterArgs& fa, const float* color, const float* gpos, const float* gnrm,
                               const float* gdif, const uint32_t* sample_n, float* filtered, float* err,
                               hipStream_t st, const float* color2, float* filtered2, float* err2) {
  if (!color || !gpos || !gnrm || !sample_n || !filtered || !err || (fa.use_diff && !gdif) ||
      (color2 && (!filtered2 || !err2)) || (int)fa.radius > kMaxFilterRadius || fa.width == 0 || fa.height == 0)
    return hipErrorInvalidValue;
  const int R = (int)fa.radius, D = 2 * R + 1;
  const bool depth = fa.kz > 0.f, diff = fa.use_diff != 0, pair = color2 && !diff && R <= kLdsRadius;
  const dim3 block(kTile, kTile), grid((fa.width + kTile - 1) / kTile, (fa.height + kTile - 1) / kTile);
  const int TA = (kTile + 2 * R) * (kTile + 2 * R);
  const bool narrow = R == kLdsRadius && !diff && !pair;
  const size_t bytes =
      sizeof(float) * ((narrow ? 10 : 12) * (size_t)TA + (size_t)D * D + ((diff || pair) && depth ? TA : 0));
#define CPT_FILTER(DI, DE, PA, RE)                                                                                \
  {                                                                                                               \
    if (R > kLdsRadius)                                                                                           \
      k_filter_mem<DI, DE><<<grid, block, 0, st>>>(fa, color, gpos, gnrm, gdif, sample_n, filtered, err);         \
    else                                                                                                          \
      k_filter_lds<DI, DE, PA, RE><<<grid, block, bytes, st>>>(fa, color, gpos, gnrm, gdif, sample_n, filtered,   \
                                                               err, color2, filtered2, err2);                     \
  }
  if (diff) {
    if (depth) CPT_FILTER(true, true, false, 12) else CPT_FILTER(true, false, false, 12)
  } else if (pair) {
    if (depth) CPT_FILTER(false, true, true, 12) else CPT_FILTER(false, false, true, 12)
  } else if (narrow) {
    if (depth) CPT_FILTER(false, true, false, 10) else CPT_FILTER(false, false, false, 10)
  } else {
    if (depth) CPT_FILTER(false, true, false, 12) else CPT_FILTER(false, false, false, 12)
  }
#undef CPT_FILTER
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess || !color2 || pair) return e;
  return launch_filter_error(fa, color2, gpos, gnrm, gdif, sample_n, filtered2, err2, st, nullptr, nullptr, nullptr);
}

// Fixed-order double sum (stands in for thrust::reduce, AdapBilatAtomic.cu:1444):
// a pairwise tree inside each 256-element block; the same tree over each chunk
// of 256 block sums; the chunk sums in order.
__global__ __launch_bounds__(kBlock) void k_err_block_sums(const float* __restrict__ e, uint32_t n,
                                                           double* __restrict__ bs) {
  __shared__ double s[kBlock];
  uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  s[threadIdx.x] = i < n ? (double)e[i] : 0.0;
  __syncthreads();
  for (int stp = kBlock / 2; stp >= 1; stp >>= 1) {
    if ((int)threadIdx.x < stp) s[threadIdx.x] += s[threadIdx.x + stp];
    __syncthreads();
  }
  if (threadIdx.x == 0) bs[blockIdx.x] = s[0];
}
// One workgroup of four 256-thread groups, each reducing one chunk of block
// sums at a time (their loads in parallel, where one thread walking the block
// sums waits on every load in turn); the chunk sums wait in LDS for thread 0.
constexpr uint32_t kErrChunks = 1024;   // 2^26 pixels: 262,144 block sums
__global__ __launch_bounds__(1024) void k_err_final(const double* __restrict__ bs, uint32_t nb,
                                                    float* __restrict__ sum) {
  __shared__ double s[1024];
  __shared__ double cs[kErrChunks];
  const uint32_t g = threadIdx.x >> 8, t = threadIdx.x & 255u;
  const uint32_t nc = (nb + 255u) / 256u;
  for (uint32_t c0 = 0; c0 < nc; c0 += 4) {
    const uint32_t c = c0 + g, i = c * 256u + t;
    s[threadIdx.x] = (c < nc && i < nb) ? bs[i] : 0.0;
    __syncthreads();
    for (uint32_t stp = 128; stp >= 1; stp >>= 1) {
      if (t < stp) s[threadIdx.x] += s[threadIdx.x + stp];
      __syncthreads();
    }
    if (t == 0 && c < nc) cs[c] = s[threadIdx.x];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    double tot = 0.0;
    for (uint32_t c = 0; c < nc; c++) tot += cs[c];
    *sum = (float)tot;
  }
}
hipError_t launch_error_sum(const float* err, uint32_t n, double* block_sums, float* sum_out, hipStream_t st) {
  uint32_t nb = (n + kBlock - 1) / kBlock;
  if (n == 0 || (nb + 255u) / 256u > kErrChunks) return hipErrorInvalidValue;
  k_err_block_sums<<<nb, kBlock, 0, st>>>(err, n, block_sums);
  k_err_final<<<1, 1024, 0, st>>>(block_sums, nb, sum_out);
  return hipGetLastError();
}

// pt_genAdapPathQueue_kernel's per-pixel count (AdapBilatAtomic.cu:830-831).
__device__ __forceinline__ uint32_t prop_count(float e, float sum, uint32_t gen) {
  float r = (float)gen * (e / sum);
  if (!(r >= 0.f) || !(r < 4294967040.f)) return 0u;
  return (uint32_t)r;
}

constexpr int kScanPer = 4;                       // elements per thread in the scan
constexpr int kScanBlock = kBlock * kScanPer;     // 1024 elements per workgroup

// Counts and workgroup-local exclusive offsets.
// With a per-pixel cap (maxp > 0) a count stops at maxp - paths.
__device__ __forceinline__ uint32_t cap_count(uint32_t c, const uint32_t* __restrict__ paths, uint32_t maxp,
                                              uint32_t i) {
  if (maxp == 0u) return c;
  const uint32_t have = paths[i];
  const uint32_t room = have < maxp ? maxp - have : 0u;
  return c < room ? c : room;
}

__global__ __launch_bounds__(kBlock) void k_scan_local(const float* __restrict__ err, const float* __restrict__ sum,
                                                       uint32_t n, uint32_t gen, uint32_t* __restrict__ counts,
                                                       uint32_t* __restrict__ offsets, uint32_t* __restrict__ btot,
                                                       const uint32_t* __restrict__ paths, uint32_t maxp) {
  __shared__ uint32_t s[kBlock];
  const float sm = *sum;
  const uint32_t base = blockIdx.x * kScanBlock + threadIdx.x * kScanPer;
  uint32_t c[kScanPer], tsum = 0;
#pragma unroll
  for (int k = 0; k < kScanPer; k++) {
    uint32_t i = base + k;
    c[k] = i < n ? cap_count(prop_count(err[i], sm, gen), paths, maxp, i) : 0u;
    tsum += c[k];
  }
  s[threadIdx.x] = tsum;
  __syncthreads();
  for (int o = 1; o < kBlock; o <<= 1) {          // Hillis-Steele inclusive scan of thread sums
    uint32_t v = (int)threadIdx.x >= o ? s[threadIdx.x - o] : 0u;
    __syncthreads();
    s[threadIdx.x] += v;
    __syncthreads();
  }
  uint32_t run = s[threadIdx.x] - tsum;
#pragma unroll
  for (int k = 0; k < kScanPer; k++) {
    uint32_t i = base + k;
    if (i < n) { counts[i] = c[k]; offsets[i] = run; }
    run += c[k];
  }
  if (threadIdx.x == kBlock - 1) btot[blockIdx.x] = s[kBlock - 1];
}
// Exclusive scan of the workgroup totals (one workgroup, chunks of 256).
__global__ __launch_bounds__(kBlock) void k_scan_totals(uint32_t* __restrict__ btot, uint32_t nb,
                                                        uint32_t* __restrict__ total) {
  __shared__ uint32_t s[kBlock];
  __shared__ uint32_t carry;
  if (threadIdx.x == 0) carry = 0;
  __syncthreads();
  for (uint32_t c0 = 0; c0 < nb; c0 += kBlock) {
    uint32_t i = c0 + threadIdx.x;
    uint32_t v = i < nb ? btot[i] : 0u;
    s[threadIdx.x] = v;
    __syncthreads();
    for (int o = 1; o < kBlock; o <<= 1) {
      uint32_t w = (int)threadIdx.x >= o ? s[threadIdx.x - o] : 0u;
      __syncthreads();
      s[threadIdx.x] += w;
      __syncthreads();
    }
    if (i < nb) btot[i] = carry + s[threadIdx.x] - v;
    __syncthreads();
    if (threadIdx.x == 0) carry += s[kBlock - 1];
    __syncthreads();
  }
  if (threadIdx.x == 0) *total = carry;
}
__global__ __launch_bounds__(kBlock) void k_scan_add(uint32_t* __restrict__ offsets, const uint32_t* __restrict__ btot,
                                                     uint32_t n) {
  uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) offsets[i] += btot[i / kScanBlock];
}
hipError_t launch_alloc_scan(const float* err, const float* sum, uint32_t n, uint32_t gen, uint32_t* counts,
                             uint32_t* offsets, uint32_t* block_tot, uint32_t* total, uint32_t cap,
                             const uint32_t* paths, uint32_t maxp, hipStream_t st) {
  (void)cap;
  if (maxp && !paths) return hipErrorInvalidValue;
  uint32_t nb = (n + kScanBlock - 1) / kScanBlock;
  k_scan_local<<<nb, kBlock, 0, st>>>(err, sum, n, gen, counts, offsets, block_tot, paths, maxp);
  k_scan_totals<<<1, kBlock, 0, st>>>(block_tot, nb, total);
  k_scan_add<<<(n + kBlock - 1) / kBlock, kBlock, 0, st>>>(offsets, block_tot, n);
  return hipGetLastError();
}

// Multi-view adaptive batches scan each view's counts on their own: view v's
// offsets then move past the slots of views 0..v-1 (base: exclusive scan of
// the per-view totals, by k_scan_totals), so all views form one queue.
__global__ __launch_bounds__(kBlock) void k_offset_views(uint32_t* __restrict__ offsets, uint32_t n, FrameArgs fa,
                                                         const uint32_t* __restrict__ base) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) offsets[i] += base[view_of(fa, i)];
}
hipError_t launch_view_bases(uint32_t* view_totals, uint32_t n_views, uint32_t* total, hipStream_t st) {
  if (!view_totals || !total || n_views == 0) return hipErrorInvalidValue;
  k_scan_totals<<<1, kBlock, 0, st>>>(view_totals, n_views, total);
  return hipGetLastError();
}
hipError_t launch_offset_views(uint32_t* offsets, uint32_t n, const FrameArgs& fa, const uint32_t* base,
                               hipStream_t st) {
  if (!offsets || !base || !fa.views || fa.n_views == 0) return hipErrorInvalidValue;
  if (n == 0) return hipSuccess;
  k_offset_views<<<(n + kBlock - 1) / kBlock, kBlock, 0, st>>>(offsets, n, fa, base);
  return hipGetLastError();
}

// One eye path per queue slot: the pixel is the last one whose offset is
// <= slot (binary search), the sample index is slot - offset.
__global__ __launch_bounds__(kBlock) void k_gen_adaptive(FrameArgs fa, const uint32_t* __restrict__ offsets,
                                                         const uint32_t* __restrict__ counts,
                                                         const uint32_t* __restrict__ total, uint32_t cap,
                                                         PathBuf pb, SampleRec rec) {
  const uint32_t q = blockIdx.x * kBlock + threadIdx.x;
  uint32_t t = *total;
  if (t > cap) t = cap;
  if (q >= t) return;
  const uint32_t n = fa.width * fa.height;
  uint32_t lo = 0, hi = n;
  while (hi - lo > 1) {
    uint32_t mid = (lo + hi) >> 1;
    if (offsets[mid] <= q) lo = mid; else hi = mid;
  }
  const uint32_t k = q - offsets[lo];
  (void)counts;
  write_eye_path(fa, pb, q, lo, q, stream_key(fa.seed, fa.frame0, 1u, k));
  zero_rec(rec, q);
}
hipError_t launch_gen_adaptive(const FrameArgs& fa, const uint32_t* offsets, const uint32_t* counts,
                               const uint32_t* total, uint32_t cap, PathBuf pb, SampleRec rec, hipStream_t st) {
  if (!pathbuf_ok(pb) || !rec_ok(rec) || !offsets || !total) return hipErrorInvalidValue;
  k_gen_adaptive<<<(cap + kBlock - 1) / kBlock, kBlock, 0, st>>>(fa, offsets, counts, total, cap, pb, rec);
  return hipGetLastError();
}

// Running-mean update of one pixel from the sums of its new records.
__device__ __forceinline__ void accum_apply(uint32_t pix, uint32_t tN, f3 ts, f3 tp, f3 tn, f3 td, f3 tq,
                                            float* __restrict__ result, uint32_t* __restrict__ sample_n,
                                            float* __restrict__ gpos, float* __restrict__ gnrm,
                                            float* __restrict__ gdif, float* __restrict__ sq) {
  uint32_t nold = sample_n[pix], nn = tN + nold;
  if (nn > nold) {
    float ri = 1.f / (float)nn, oi = (float)nold * ri;
    float* r = result + (size_t)pix * 3;
    r[0] = fmaxf(ri * ts.x + oi * r[0], 0.f);
    r[1] = fmaxf(ri * ts.y + oi * r[1], 0.f);
    r[2] = fmaxf(ri * ts.z + oi * r[2], 0.f);
    sample_n[pix] = nold + tN;
    f3 vals[3] = {tp, tn, td};
    float* dst[3] = {gpos + (size_t)pix * 3, gnrm + (size_t)pix * 3, gdif + (size_t)pix * 3};
#pragma unroll
    for (int k = 0; k < 3; k++) {
      dst[k][0] = ri * vals[k].x + oi * dst[k][0];
      dst[k][1] = ri * vals[k].y + oi * dst[k][1];
      dst[k][2] = ri * vals[k].z + oi * dst[k][2];
    }
    float* q = sq + (size_t)pix * 3;                // squareResult (AdapEmp.cu:927-944)
    q[0] = fmaxf(ri * tq.x + oi * q[0], 0.f);
    q[1] = fmaxf(ri * tq.y + oi * q[1], 0.f);
    q[2] = fmaxf(ri * tq.z + oi * q[2], 0.f);
  }
}

// Adds record q to the running sums (records with N = 0 or an infinite
// component are skipped, AdapBilatAtomic.cu:1056-1060).
// One sample record: its four columns are loaded together (one round trip),
// then added in record order, so that loads of several records can be in
// flight while the sums keep their order.
struct RecVals {
  float4 a, p, n, d;
};
__device__ __forceinline__ RecVals load_record(const SampleRec& rec, uint32_t q) {
  RecVals r;
  r.a = rec.acc[q];
  r.p = rec.gpos[q];
  r.n = rec.gnrm[q];
  r.d = rec.gdif[q];
  return r;
}
__device__ __forceinline__ void add_record(const RecVals& r, f3& ts, f3& tp, f3& tn, f3& td, f3& tq, uint32_t& tN) {
  uint32_t N = __float_as_uint(r.a.w);
  f3 acc = ld3(r.a);
  if (N == 0 || isinf3(acc)) return;
  float nf = (float)N;
  ts = ts + acc;
  tq = tq + vmul(acc, acc);
  tN += N;
  tp = tp + ld3(r.p) * nf;
  tn = tn + ld3(r.n) * nf;
  td = td + ld3(r.d) * nf;
}
// Records q0, q0 + step, ... below q1 in order, four loads in flight.
__device__ __forceinline__ void accum_records(const SampleRec& rec, uint32_t q0, uint32_t q1, uint32_t step, f3& ts,
                                              f3& tp, f3& tn, f3& td, f3& tq, uint32_t& tN) {
  uint32_t q = q0;
  for (; q1 > 3 * step && q < q1 - 3 * step; q += 4 * step) {
    const RecVals r0 = load_record(rec, q), r1 = load_record(rec, q + step);
    const RecVals r2 = load_record(rec, q + 2 * step), r3 = load_record(rec, q + 3 * step);
    add_record(r0, ts, tp, tn, td, tq, tN);
    add_record(r1, ts, tp, tn, td, tq, tN);
    add_record(r2, ts, tp, tn, td, tq, tN);
    add_record(r3, ts, tp, tn, td, tq, tN);
  }
  for (; q < q1; q += step) add_record(load_record(rec, q), ts, tp, tn, td, tq, tN);
}

// Pixels with more records than this are summed by a whole workgroup.
constexpr uint32_t kAccumSerialMax = 32;


// pt_atomicApplyPathQueueResult_kernel + pt_accumTempResultToResult_kernel
// (AdapBilatAtomic.cu:1041-1141) with the per-pixel sums taken over the
// pixel's samples in queue order instead of float atomics.  Pixels holding
// more than kAccumSerialMax records are listed for k_accum_big.
__global__ __launch_bounds__(kBlock) void k_accum_adaptive(const uint32_t* __restrict__ offsets,
                                                           const uint32_t* __restrict__ counts, uint32_t n,
                                                           uint32_t cap, SampleRec rec, float* __restrict__ result,
                                                           uint32_t* __restrict__ sample_n, float* __restrict__ gpos,
                                                           float* __restrict__ gnrm, float* __restrict__ gdif,
                                                           float* __restrict__ sq, uint32_t* __restrict__ big_list,
                                                           uint32_t* __restrict__ big_n) {
  const uint32_t pix = blockIdx.x * kBlock + threadIdx.x;
  if (pix >= n) return;
  uint32_t q0 = offsets[pix], q1 = q0 + counts[pix];
  if (q1 > cap) q1 = cap;
  if (q0 > q1) q0 = q1;
  if (q1 > q0 + kAccumSerialMax) {
    big_list[atomicAdd(big_n, 1u)] = pix;
    return;
  }
  f3 ts = mk3(0.f, 0.f, 0.f), tp = ts, tn = ts, td = ts, tq = ts;
  uint32_t tN = 0;
  accum_records(rec, q0, q1, 1u, ts, tp, tn, td, tq, tN);
  accum_apply(pix, tN, ts, tp, tn, td, tq, result, sample_n, gpos, gnrm, gdif, sq);
}

// Heavily sampled pixels: one workgroup per pixel, thread t sums records
// q0 + t, q0 + t + 256, ..., then a fixed butterfly within each wave and the
// four wave sums in order (deterministic for a given record count).
__global__ __launch_bounds__(kBlock) void k_accum_big(const uint32_t* __restrict__ offsets,
                                                      const uint32_t* __restrict__ counts, uint32_t cap, SampleRec rec,
                                                      float* __restrict__ result, uint32_t* __restrict__ sample_n,
                                                      float* __restrict__ gpos, float* __restrict__ gnrm,
                                                      float* __restrict__ gdif, float* __restrict__ sq,
                                                      const uint32_t* __restrict__ big_list,
                                                      const uint32_t* __restrict__ big_n) {
  constexpr int kV = 15;
  __shared__ float red[kBlock / 64][kV];
  __shared__ uint32_t redn[kBlock / 64];
  const uint32_t nb = *big_n;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (uint32_t i = blockIdx.x; i < nb; i += gridDim.x) {
    const uint32_t pix = big_list[i];
    uint32_t q0 = offsets[pix], q1 = q0 + counts[pix];
    if (q1 > cap) q1 = cap;
    f3 ts = mk3(0.f, 0.f, 0.f), tp = ts, tn = ts, td = ts, tq = ts;
    uint32_t tN = 0;
    accum_records(rec, q0 + threadIdx.x, q1, kBlock, ts, tp, tn, td, tq, tN);
    float v[kV] = {ts.x, ts.y, ts.z, tp.x, tp.y, tp.z, tn.x, tn.y, tn.z, td.x, td.y, td.z, tq.x, tq.y, tq.z};
#pragma unroll
    for (int k = 0; k < kV; k++)
      for (int o = 32; o >= 1; o >>= 1) v[k] += __shfl_xor(v[k], o, 64);
    for (int o = 32; o >= 1; o >>= 1) tN += __shfl_xor(tN, o, 64);
    if (lane == 0) {
#pragma unroll
      for (int k = 0; k < kV; k++) red[wave][k] = v[k];
      redn[wave] = tN;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      float a[kV];
      uint32_t sN = 0;
#pragma unroll
      for (int k = 0; k < kV; k++) a[k] = 0.f;
      for (int w = 0; w < kBlock / 64; w++) {
#pragma unroll
        for (int k = 0; k < kV; k++) a[k] += red[w][k];
        sN += redn[w];
      }
      accum_apply(pix, sN, mk3(a[0], a[1], a[2]), mk3(a[3], a[4], a[5]), mk3(a[6], a[7], a[8]),
                  mk3(a[9], a[10], a[11]), mk3(a[12], a[13], a[14]), result, sample_n, gpos, gnrm, gdif, sq);
    }
    __syncthreads();
  }
}

hipError_t launch_accum_adaptive(const uint32_t* offsets, const uint32_t* counts, uint32_t n, uint32_t cap,
                                 SampleRec rec, float* result, uint32_t* sample_n, float* gpos, float* gnrm,
                                 float* gdif, float* sq, uint32_t* big_list, uint32_t* big_n, hipStream_t st) {
  if (!rec_ok(rec) || !offsets || !counts || !result || !sample_n || !gpos || !gnrm || !gdif || !sq || !big_list ||
      !big_n)
    return hipErrorInvalidValue;
  k_fill_u32<<<1, 1, 0, st>>>(big_n, 0u);
  k_accum_adaptive<<<(n + kBlock - 1) / kBlock, kBlock, 0, st>>>(offsets, counts, n, cap, rec, result, sample_n, gpos,
                                                                  gnrm, gdif, sq, big_list, big_n);
  k_accum_big<<<1024, kBlock, 0, st>>>(offsets, counts, cap, rec, result, sample_n, gpos, gnrm, gdif, sq, big_list,
                                       big_n);
  return hipGetLastError();
}

// ---- empirical error and round-based allocation -----------------------------

__global__ __launch_bounds__(kBlock) void k_emp_error(const float* __restrict__ r, const float* __restrict__ q,
                                                      const uint32_t* __restrict__ sample_n, uint32_t n,
                                                      float* __restrict__ err) {
  const uint32_t x = blockIdx.x * kBlock + threadIdx.x;
  if (x >= n) return;
  const uint32_t N = sample_n[x];
  const float* a = r + (size_t)x * 3;
  const float* b = q + (size_t)x * 3;
  float e = ((b[0] - a[0] * a[0]) + (b[1] - a[1] * a[1]) + (b[2] - a[2] * a[2])) * (float)N / ((float)(N - 1u) * 3.f);
  err[x] = fminf(e, 1.0f);
}
hipError_t launch_emp_error(const float* result, const float* sq, const uint32_t* sample_n, uint32_t n, float* err,
                            hipStream_t st) {
  if (!result || !sq || !sample_n || !err) return hipErrorInvalidValue;
  if (n == 0) return hipSuccess;
  k_emp_error<<<(n + kBlock - 1) / kBlock, kBlock, 0, st>>>(result, sq, sample_n, n, err);
  return hipGetLastError();
}

// Maximum with 0 as the initial value: non-negative floats order as their bits.
__global__ __launch_bounds__(kBlock) void k_error_max(const float* __restrict__ e, uint32_t n,
                                                      uint32_t* __restrict__ out) {
  uint32_t m = 0;
  for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock)
    m = max(m, __float_as_uint(fmaxf(e[i], 0.f)));
  for (int o = 32; o >= 1; o >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, o, 64));
  // one atomic a workgroup, of few: on one address they take about 12 ns each
  // (4,096 of them, one a wave of 1,024 workgroups, took 48 us)
  __shared__ uint32_t wm[kBlock / 64];
  if ((threadIdx.x & 63) == 0) wm[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kBlock / 64; w++) m = max(m, wm[w]);
    atomicMax(out, m);
  }
}
hipError_t launch_error_max(const float* err, uint32_t n, float* max_out, hipStream_t st) {
  if (!err || !max_out) return hipErrorInvalidValue;
  k_fill_u32<<<1, 1, 0, st>>>((uint32_t*)max_out, 0u);
  uint32_t nb = (n + kBlock - 1) / kBlock;
  if (nb > 256) nb = 256;
  if (nb) k_error_max<<<nb, kBlock, 0, st>>>(err, n, (uint32_t*)max_out);
  return hipGetLastError();
}

__global__ void k_round_init(RoundState* rs, uint32_t* kept, const float* maxe, uint32_t gen, uint32_t bisect,
                             float desired, float min_prob) {
  for (uint32_t i = threadIdx.x; i < 3 * kKeptSlots; i += blockDim.x) kept[i * kDealStride] = 0u;
  if (threadIdx.x != 0) return;
  RoundState s;
  s.maxe = *maxe;
  s.left = 0.f;
  s.right = s.maxe * 2.f;
  s.window = bisect ? (s.left + s.right) * 0.5f : s.maxe;
  s.accum = 0;
  s.gen = gen;
  s.done = gen == 0 ? 1u : 0u;
  s.rounds = 0;
  s.bisect = bisect;
  s.desired = desired;
  s.min_prob = min_prob;
  s.status = kRoundIdle;
  s.take = 0;
  *rs = s;
}
__global__ __launch_bounds__(kBlock) void k_zero_u32(uint32_t* __restrict__ p, uint32_t n) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) p[i] = 0u;
}
hipError_t launch_round_init(RoundState* rs, uint32_t* kept, const float* maxe, uint32_t gen, uint32_t bisect,
                             float desired, float min_prob, uint32_t* counts, uint32_t n, hipStream_t st) {
  if (!rs || !kept || !maxe || !counts) return hipErrorInvalidValue;
  k_round_init<<<1, 64, 0, st>>>(rs, kept, maxe, gen, bisect, desired, min_prob);
  if (n) k_zero_u32<<<(n + kBlock - 1) / kBlock, kBlock, 0, st>>>(counts, n);
  return hipGetLastError();
}

// remove_if + size bookkeeping + the bisection of AdapBilatBinary.cu:1363-1371,
// for the round that kept `kept` pixels.
__device__ __forceinline__ void round_update(RoundState& s, uint32_t kept) {
  const uint32_t take = min(kept, s.gen - s.accum);
  s.status = take < kept ? kRoundPartial : kRoundIdle;
  s.take = take;
  s.accum += take;
  s.rounds++;
  if (take == 0u) {
    s.done = 1u;
  } else if (s.bisect) {
    if ((float)take < s.desired) s.right = s.window;
    else if ((float)take > s.desired) s.left = s.window;
    s.window = (s.left + s.right) * 0.5f;
  }
  if (s.accum >= s.gen) s.done = 1u;
}
// One launch a round (keep = 0: only closes the last).  It closes the round
// before: every workgroup computes the state after it from the state it ran in and its
// kept pixels, one thread writes that for the next launch, and the kept
// pixels take one sample each, all of them unless more were kept than slots are
// left: that can only be the last round, whose ranks k_round_apply needs a scan for.
// Then pt_genTempAdapPathQueue_kernel: keep unless u * window > max(e, min_prob),
// u from the stream of (frame, slots filled so far) at the pixel; kept pixels are counted
// in kKeptSlots counters, of three sets in turn: read, added to, cleared.
// Six launches a round (keep, a scan of three, take, update) took 20 us, this 4.
__global__ __launch_bounds__(kBlock) void k_round(uint64_t seed, uint32_t frame, const float* __restrict__ err,
                                                  uint32_t n, const RoundState* __restrict__ from,
                                                  RoundState* __restrict__ to, const uint32_t* __restrict__ kept,
                                                  uint32_t* __restrict__ keeping, uint32_t* __restrict__ clear,
                                                  uint32_t* __restrict__ flags, uint32_t* __restrict__ counts,
                                                  int keep) {
  __shared__ uint32_t total, wc[kBlock / 64];
  RoundState s = *from;
  const bool pending = s.status == kRoundPending;
  if (threadIdx.x < 64) {
    const uint32_t t = wave_sum(pending ? kept[threadIdx.x * kDealStride] : 0u);
    if (threadIdx.x == 0) total = t;
    if (blockIdx.x == 0) clear[threadIdx.x * kDealStride] = 0u;
  }
  __syncthreads();
  if (pending) round_update(s, total);
  const bool all = pending && s.status == kRoundIdle;
  const bool next = keep && !s.done;
  const float window = s.window;
  if (next) s.status = kRoundPending;
  if (blockIdx.x == 0 && threadIdx.x == 0) *to = s;
  if (!all && !next) return;
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  bool k = false;
  if (i < n) {
    if (all && flags[i]) counts[i] += 1u;
    if (next) {
      uint64_t r = 0;
      const uint64_t inc = ((uint64_t)i << 1) | 1u;
      pcg32_seed(r, inc, stream_key(seed, frame, 3u, s.accum));
      const float u = uniform01(r, inc);
      k = !(u * window > fmaxf(err[i], s.min_prob));
      flags[i] = k ? 1u : 0u;
    }
  }
  if (!next) return;
  const uint64_t m = __ballot(k);
  if ((threadIdx.x & 63) == 0) wc[threadIdx.x >> 6] = (uint32_t)__popcll(m);
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t t = 0;
    for (int w = 0; w < kBlock / 64; w++) t += wc[w];
    if (t) atomicAdd(&keeping[(blockIdx.x % kKeptSlots) * kDealStride], t);
  }
}
// The last round's kept pixels of rank below its slots take one sample each.
__global__ __launch_bounds__(kBlock) void k_round_apply(const uint32_t* __restrict__ flags,
                                                        const uint32_t* __restrict__ rank, uint32_t n,
                                                        const RoundState* __restrict__ rs,
                                                        uint32_t* __restrict__ counts) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n && flags[i] && rank[i] < rs->take) counts[i] += 1u;
}
__global__ __launch_bounds__(kBlock) void k_round_fill(const RoundState* __restrict__ rs, uint32_t n,
                                                       uint32_t* __restrict__ counts) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const uint32_t unfilled = rs->gen > rs->accum ? rs->gen - rs->accum : 0u;
  counts[i] += unfilled / n + (i < unfilled % n ? 1u : 0u);
}

// Exclusive scan of given per-element values (SRC = 1) into offsets.
__global__ __launch_bounds__(kBlock) void k_scan_local_u32(const uint32_t* __restrict__ in, uint32_t n,
                                                           uint32_t* __restrict__ offsets,
                                                           uint32_t* __restrict__ btot) {
  __shared__ uint32_t s[kBlock];
  const uint32_t base = blockIdx.x * kScanBlock + threadIdx.x * kScanPer;
  uint32_t c[kScanPer], tsum = 0;
#pragma unroll
  for (int k = 0; k < kScanPer; k++) {
    uint32_t i = base + k;
    c[k] = i < n ? in[i] : 0u;
    tsum += c[k];
  }
  s[threadIdx.x] = tsum;
  __syncthreads();
  for (int o = 1; o < kBlock; o <<= 1) {
    uint32_t v = (int)threadIdx.x >= o ? s[threadIdx.x - o] : 0u;
    __syncthreads();
    s[threadIdx.x] += v;
    __syncthreads();
  }
  uint32_t run = s[threadIdx.x] - tsum;
#pragma unroll
  for (int k = 0; k < kScanPer; k++) {
    uint32_t i = base + k;
    if (i < n) offsets[i] = run;
    run += c[k];
  }
  if (threadIdx.x == kBlock - 1) btot[blockIdx.x] = s[kBlock - 1];
}
hipError_t launch_scan_counts(const uint32_t* counts, uint32_t n, uint32_t* offsets, uint32_t* block_tot,
                              uint32_t* total, hipStream_t st) {
  if (!counts || !offsets || !block_tot || !total) return hipErrorInvalidValue;
  uint32_t nb = (n + kScanBlock - 1) / kScanBlock;
  if (nb) k_scan_local_u32<<<nb, kBlock, 0, st>>>(counts, n, offsets, block_tot);
  k_scan_totals<<<1, kBlock, 0, st>>>(block_tot, nb, total);
  if (n) k_scan_add<<<(n + kBlock - 1) / kBlock, kBlock, 0, st>>>(offsets, block_tot, n);
  return hipGetLastError();
}
hipError_t launch_round(const FrameArgs& fa, const float* err, uint32_t n, RoundState* rs, uint32_t* kept, uint32_t j,
                        uint32_t* flags, uint32_t* counts, int keep, hipStream_t st) {
  if (!err || !rs || !flags || !kept || !counts || n == 0) return hipErrorInvalidValue;
  const auto set = [&](uint32_t k) { return kept + (size_t)(k % 3u) * kKeptSlots * kDealStride; };
  k_round<<<(n + kBlock - 1) / kBlock, kBlock, 0, st>>>(fa.seed, fa.frame0, err, n, rs + (j & 1u), rs + ((j + 1u) & 1u),
                                                        set(j), set(j + 1u), set(j + 2u), flags, counts, keep);
  return hipGetLastError();
}
hipError_t launch_round_rest(const RoundState* rs, const uint32_t* flags, uint32_t n, uint32_t* rank,
                             uint32_t* block_tot, uint32_t* total, uint32_t* counts, hipStream_t st) {
  if (!rs || !flags || !rank || !counts || n == 0) return hipErrorInvalidValue;
  const hipError_t e = launch_scan_counts(flags, n, rank, block_tot, total, st);
  if (e != hipSuccess) return e;
  k_round_apply<<<(n + kBlock - 1) / kBlock, kBlock, 0, st>>>(flags, rank, n, rs, counts);
  return hipGetLastError();
}
hipError_t launch_round_fill(const RoundState* rs, uint32_t n, uint32_t* counts, hipStream_t st) {
  if (!rs || !counts) return hipErrorInvalidValue;
  if (n) k_round_fill<<<(n + kBlock - 1) / kBlock, kBlock, 0, st>>>(rs, n, counts);
  return hipGetLastError();
}


// ---------------------------------------------------------------- per-pixel path caps
// A pixel that already has maxp paths gets no error weight (the allocation
// gives it nothing); counts of a round-based pass stop at maxp - paths.
__global__ __launch_bounds__(kBlock) void k_cap_error(float* __restrict__ err, const uint32_t* __restrict__ paths,
                                                      uint32_t maxp, uint32_t n) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n && paths[i] >= maxp) err[i] = 0.f;
}
__global__ __launch_bounds__(kBlock) void k_cap_counts(uint32_t* __restrict__ counts,
                                                       const uint32_t* __restrict__ paths, uint32_t maxp,
                                                       uint32_t n) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) counts[i] = cap_count(counts[i], paths, maxp, i);
}
// paths += counts (an adaptive pass), or += 1 (a warm-up frame); reset first
// when `reset`.
__global__ __launch_bounds__(kBlock) void k_add_paths(uint32_t* __restrict__ paths,
                                                      const uint32_t* __restrict__ counts, uint32_t n, int reset) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) paths[i] = (reset ? 0u : paths[i]) + (counts ? counts[i] : 1u);
}
hipError_t launch_cap_error(float* err, const uint32_t* paths, uint32_t maxp, uint32_t n, hipStream_t st) {
  if (!maxp || n == 0) return hipSuccess;
  k_cap_error<<<(n + kBlock - 1) / kBlock, kBlock, 0, st>>>(err, paths, maxp, n);
  return hipGetLastError();
}
hipError_t launch_cap_counts(uint32_t* counts, const uint32_t* paths, uint32_t maxp, uint32_t n, hipStream_t st) {
  if (!maxp || n == 0) return hipSuccess;
  k_cap_counts<<<(n + kBlock - 1) / kBlock, kBlock, 0, st>>>(counts, paths, maxp, n);
  return hipGetLastError();
}
hipError_t launch_add_paths(uint32_t* paths, const uint32_t* counts, uint32_t n, int reset, hipStream_t st) {
  if (n == 0) return hipSuccess;
  k_add_paths<<<(n + kBlock - 1) / kBlock, kBlock, 0, st>>>(paths, counts, n, reset);
  return hipGetLastError();
}
}  // namespace cpt
