// bvh_build.h -- host SAH builder interface.
#pragma once
#include <stdint.h>

#include <vector>

namespace ne {

struct PrimInput {
  float bmin[3], bmax[3];
  uint32_t type;  // leaves never mix types
};

// 4-wide node, child boxes quantized to 8 bits per plane against the node's
// box, 16 floats:
//   (origin.xyz, exponents: byte a = e_a + 127)
//   (qlo.x, qlo.y, qlo.z, qhi.x) (qhi.y, qhi.z, meta, 0)
//   int child[4]
// Each q word holds one byte per child; child c's box on axis a is
// [origin_a + qlo_a[c] * 2^e_a, origin_a + qhi_a[c] * 2^e_a] in FP32 (the
// builder makes that decode contain the true box).  meta byte c is 0 for an
// inner child (child[c] = node index) or 0x80 | type << 4 | count for a leaf of
// count primitives of type (0 triangle, 1 sphere, 2 rectangle) at refs
// [child[c], child[c] + count).  child < 0: empty slot.
constexpr int kNodeFloats = 16;
constexpr uint32_t kMetaLeaf = 0x80;  // child meta byte: 0x80 | type << 4 | count for a leaf, 0 otherwise

struct BvhOutput {
  std::vector<float> nodes;     // kNodeFloats per node
  std::vector<uint32_t> refs;   // leaf slots -> input primitive index (leaves hold refs[first, first+count))
  std::vector<uint32_t> order;  // input primitive indices in leaf order
  uint32_t max_depth = 0;       // wide-node levels
  uint32_t max_stack = 0;       // deepest traversal stack (children pushed along any root path)
  uint32_t max_leaf = 0;
  bool quant_failed = false;    // some child box has no conservative 8-bit encoding (non-finite bounds)
};

void build_bvh(const std::vector<PrimInput>& prims, BvhOutput& out);

}  // namespace ne
