// The 16-wide form of the hierarchy that tier 0 walks, one lane per child.
//
// A Karras subtree of s points has class 0 when s <= 32 (a leaf of the wide
// form) and class k when 32 * 8^(k-1) < s <= 32 * 8^k.  A wide node stands for
// a maximal subtree of its class (its parent has a higher class); its
// children are the maximal subtrees of lower classes below it, found by
// splitting the largest one of a higher class until none is left or 16 are
// reached.  With a factor of 8 between classes a balanced subtree gives 8 to
// 15 children.  A subtree that would need more keeps its last oversize
// subtrees as references to binary nodes, which are walked as such.
//
// Wide nodes need no allocation: subtrees of one class are disjoint ranges of
// at least L = 32 * 8^(k-1) + 1 points, so first / L numbers them without
// collision.  All classes together take less than n / 28 records of 512
// bytes, less than the 32 bytes per point that the refit's boxes occupy, and
// live there once the refit has read them.
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

// Fills the wide node of binary node i (class k >= 1).
__host__ __device__ inline void wide_fill(uint32_t i, int k, uint32_t n, const Node *nodes, const uint2 *ranges,
                                          WideChild *out) {
    uint32_t at[16];             // child as parent << 1 | side
    uint32_t first[16], size[16];
    const uint32_t limit = wide_least(k) - 1u;  // children have at most this many points
    int m = 0;
    auto take = [&](int slot, uint32_t parent, uint32_t side) {
        const Node &nd = nodes[parent];
        uint32_t ref;
        memcpy(&ref, side ? &nd.hi1.w : &nd.hi0.w, 4);
        at[slot] = (parent << 1) | side;
        if (is_leaf(ref)) {
            first[slot] = leaf_first(ref);
            size[slot] = leaf_count(ref);
        } else {
            first[slot] = ranges[ref].x;
            size[slot] = ranges[ref].y - ranges[ref].x + 1u;
        }
    };
    take(m++, i, 0u);
    take(m++, i, 1u);
    while (m < 16) {
        int best = 0;
        for (int t = 1; t < m; ++t)
            if (size[t] > size[best]) best = t;
        if (size[best] <= limit) break;
        const Node &nd = nodes[at[best] >> 1];
        uint32_t ref;
        memcpy(&ref, (at[best] & 1u) ? &nd.hi1.w : &nd.hi0.w, 4);
        take(m++, ref, 1u);
        take(best, ref, 0u);
    }
    for (int t = 0; t < 16; ++t) {
        WideChild c;
        uint32_t ref = kWideNone;
        c.lo = make_float4(0.f, 0.f, 0.f, 0.f);
        c.hi = make_float4(0.f, 0.f, 0.f, 0.f);
        if (t < m) {
            const Node &nd = nodes[at[t] >> 1];
            c.lo = (at[t] & 1u) ? nd.lo1 : nd.lo0;
            c.hi = (at[t] & 1u) ? nd.hi1 : nd.hi0;
            if (size[t] <= limit) {
                ref = wide_ref(n, first[t], size[t]);
            } else {  // its own binary node
                memcpy(&ref, &c.hi.w, 4);
                ref |= kWideBinary;
            }
        }
        memcpy(&c.hi.w, &ref, 4);
        out[t] = c;
    }
}

}  // namespace pg
