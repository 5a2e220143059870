// The 16-wide form of the hierarchy that tier 0 walks, one lane per child.
//
// A Karras subtree of s points has class 0 when s <= 32 (a leaf of the wide
// form) and class k when 32 * 8^(k-1) < s <= 32 * 8^k.  A wide node stands for
// a maximal subtree of its class (its parent has a higher class); its
// children are the maximal subtrees of lower classes below it, found by
// splitting those of a higher class until none is left or 16 are reached.  With a factor of 8 between classes a balanced subtree gives 8 to
// 15 children.  A subtree that would need more keeps its last oversize
// subtrees as references to binary nodes, which are walked as such.
//
// Wide nodes need no allocation: subtrees of one class are disjoint ranges of
// at least L = 32 * 8^(k-1) + 1 points, so first / L numbers them without
// collision.  The records of all classes (512 bytes each; for large n one per
// 28 points) fit into the 32 bytes per binary node of the refit's boxes at
// every n (wide_fits), and live there once the refit has read them.
#pragma once

#include "pg_common.hpp"

namespace pg {

constexpr int kWideLeaf = 32;
constexpr uint32_t kWideNone = 0xFFFFFFFFu;    // no child
constexpr uint32_t kWideBinary = 0x40000000u;  // reference to a binary node

struct alignas(16) WideChild {
    float4 lo;  // lo.xyz, max weight
    float4 hi;  // hi.xyz, reference (bits): leaf range, wide node or binary node
};

__host__ __device__ inline int wide_class(uint32_t s) {
    if (s <= (uint32_t)kWideLeaf) return 0;
    const int cl = 32 - __builtin_clz(s - 1u);  // ceil(log2 s) >= 6
    return (cl - 3) / 3;
}
// least size of class k >= 1
__host__ __device__ inline uint32_t wide_least(int k) { return ((uint32_t)kWideLeaf << (3 * (k - 1))) + 1u; }
// record of the class-k subtree that starts at sorted point `first`
__host__ __device__ inline uint32_t wide_slot(uint32_t n, int k, uint32_t first) {
    uint32_t at = first / wide_least(k);
    for (int j = 1; j < k; ++j) at += (n - 1u) / wide_least(j) + 1u;
    return at;
}
// reference to the subtree over points [first, first + s) (a maximal one of its class, or a cloud)
__host__ __device__ inline uint32_t wide_ref(uint32_t n, uint32_t first, uint32_t s) {
    const int k = wide_class(s);
    return k == 0 ? leaf_ref(first, s) : wide_slot(n, k, first);
}
// records that n points may use
__host__ __device__ inline uint64_t wide_records(uint32_t n) {
    uint64_t r = 0;
    for (int k = 1; k <= wide_class(n); ++k) r += (n - 1u) / wide_least(k) + 1u;
    return r;
}
// do they fit into the boxes of the n - 1 binary nodes?
__host__ __device__ inline bool wide_fits(uint32_t n) {
    return n <= (uint32_t)kWideLeaf || 16ull * sizeof(WideChild) * wide_records(n) <= 32ull * (n - 1u);
}

}  // namespace pg
