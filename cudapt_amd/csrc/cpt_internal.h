// Internal layouts shared by the host library and the gfx950 kernels.
#pragma once
#include <cstdint>
#include <vector>

typedef uint32_t u32;
typedef uint64_t u64;
typedef int32_t i32;

namespace cpt {

// Reference constants (include/cudahelper.h:27-30).
constexpr float kInfF = 1e20f;                 // M_INF as float
constexpr double kBiasEps = 1e-4;              // M_FLT_BIAS_EPSILON
constexpr double kFltEps = 1e-5;               // M_FLT_EPSILON
constexpr double kEpsilon = 1e-9;              // M_EPSILON
constexpr u32 kInvalid = 0xFFFFFFFFu;

// Compact binary node of the reference layout (src/cudaRTCommon.cu:527-541):
// min/max bounds + (offset-or-triStart, triN).  triN == 0 marks an interior
// node; an empty leaf (a degenerate split) has inverted bounds.
struct BinNode {
  float mn[3], mx[3];
  u32 a, n;
};

// 4-wide node, 128 bytes = one 128-byte line: six 4-float slab planes, then
// per child either an interior node index (count == 0) or a leaf triangle
// range (child = first leaf-order triangle, count = #triangles).
// Unused slots have child = kInvalid and an empty box.
struct alignas(128) Node4 {
  float lox[4], hix[4], loy[4], hiy[4], loz[4], hiz[4];
  u32 child[4];
  u32 count[4];
};
static_assert(sizeof(Node4) == 128, "Node4 must be one 128-byte line");

// 8-wide node, 128 bytes = one line: child boxes as FP16 fractions h in [0, 1]
// of a power-of-two extent 2^(e-127) per axis from the origin o.  The host picks
// every h so that the box o + h * 2^(e-127) (in exact arithmetic) contains the
// child's FP32 box, so culling stays conservative and hits unchanged; a
// traversal multiplies them as they are (v_fma_mix_f32 takes FP16 operands).
// Children sit in eight slots; interior children (imask) are consecutive nodes
// from `child` on in slot order, and a leaf child's triangles (at most kLeaf8)
// are consecutive from `tri` on, slot by slot: bit 4 s + j of `valid` is set for
// triangle j of slot s.  Loaded as eight 16-byte vectors: {o, exponents +
// imask}, {child, tri, valid, -}, then lo and hi of each axis.
struct alignas(128) Node8 {
  float o[3];
  u32 exps;            // ex | ey << 8 | ez << 16 | imask << 24
  u32 child, tri, valid, pad;
  uint16_t h[3][2][8]; // [axis][lo, hi][slot]; an unused slot has no imask or valid bit
};
static_assert(sizeof(Node8) == 128, "Node8 must be one 128-byte line");
constexpr u32 kLeaf8 = 4;          // most triangles of an 8-wide leaf child
constexpr u32 kMaxNodes8 = 1u << 25;   // byte offsets of nodes fit 32 bits; a larger tree is not made
constexpr u32 kMaxDepth8 = 64;     // levels of the 8-wide tree (a traversal keeps at most one stack entry a level)

// Host result of the SAH build.
struct BvhHost {
  std::vector<BinNode> nodes;      // DFS preorder, reference CompactBVH order
  std::vector<u32> reorder;        // leaf order -> original triangle id
  std::vector<BinNode> dnodes;     // the device tree's binary SAH build, same format
  std::vector<u32> dreorder;       // device leaf order -> original triangle id
  std::vector<Node4> nodes4;       // 4-wide re-layout (BFS order, root 0)
  std::vector<Node8> nodes8;       // 8-wide quantized re-layout (BFS order, root 0)
  std::vector<u32> order8;         // its triangle order -> device leaf order
  float qmag = 1e-30f;             // max |o + q * step| over nodes8's planes, at least 1e-30
  u32 depth8 = 0;
  u32 depth4 = 0, leaves4 = 0;
};

// SAH build with NPBVHHelper semantics (src/bvhhelper.cpp:55-311).
bool build_bvh_sah(const float* pos3, const u32* idx3, u32 nt, u32 max_depth, BvhHost& out);
// The device tree: binned SAH over triangle bounds (dnodes / dreorder).
bool build_bvh_device(const float* pos3, const u32* idx3, u32 nt, BvhHost& out);
// Collapse the device binary tree into 4-wide nodes (SAH-optimal); a leaf
// range holds at most leaf_max triangles.
void collapse_bvh4(const float* pos3, const u32* idx3, BvhHost& b, u32 leaf_max);
// Collapse the device binary tree into 8-wide quantized nodes (SAH-optimal);
// a leaf child holds at most min(leaf_max, kLeaf8) triangles.  No nodes when
// they would exceed kMaxNodes8, an extent cannot be encoded or the tree is deeper than
// kMaxDepth8 (the FP32 layout serves such a scene); false when a vertex lies at
// minus infinity.
bool collapse_bvh8(BvhHost& b, u32 leaf_max);

}  // namespace cpt
