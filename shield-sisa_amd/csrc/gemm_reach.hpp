// Which elements of an operand row a GEMM lane reads, free of the HIP runtime.
#pragma once

namespace shv {

// gemm_wide_kernel with KS K steps: a lane of group g (0..3) reads 8 weights of a K-long row (K % 8 == 0) for step ks, this
// far from element 8 g: its chunk 32 ks + 8 g, or, where that lies past K (`in` false; the product's operand is zeroed), the
// row's chunk g.  A row of a single step may not have that one: there the row's first 8 (elsewhere the lane-dependent
// offset would cost registers that the kernel does not have: 183 -> 186 us at M 125,440, N 960, K 160 in fp16).
constexpr int wide_step(int KS, int ks, int g, bool in) { return in ? 32 * ks : KS == 1 ? -8 * g : 0; }

}  // namespace shv
