// k nearest neighbours of every point over the LBVH (the reference's
// cuBQL_knn_kernel, pwr_bvh.cu:159-215: the K nearest by squared distance,
// the query's own id excluded, short lists padded with the last id found or
// 0).  Used for the learned radius features and as initial guesses.
//
// One lane per query in Morton order (neighbouring lanes walk neighbouring
// parts of the hierarchy).  Depth-first, nearer child first; the farther
// child waits on a per-lane stack in LDS as (parent << 1 | child) and is
// re-tested against the current K-th distance when it comes out.  A Karras
// hierarchy over 32-bit keys and < 2^26 points is less than 64 levels deep,
// and every level pushes at most one entry, so 64 entries never overflow.
// The first pass keeps 32 (half the LDS, so more waves per CU); the rare
// query that needs more is queued in the index workspace and redone by a
// second pass with 64.
#include "pg_common.hpp"
#include "pg_dpp.hpp"
#include "pg_kernels.hpp"
#include "pg_wide.hpp"

#include <float.h>

namespace pg {

constexpr int kKnnThreads = 128;
constexpr int kKnnStack = 64;      // deep pass: never overflows (see above)
constexpr int kKnnStackFast = 32;  // first pass: 16 KB of LDS per block instead of 32 KB
#ifndef PG_KNN_LOADS
#define PG_KNN_LOADS 2
#endif
constexpr int kLoads = PG_KNN_LOADS;  // leaf points loaded ahead

__device__ __forceinline__ float box_dist2(float4 lo, float4 hi, float qx, float qy, float qz) {
    const float dx = fmaxf(fmaxf(lo.x - qx, qx - hi.x), 0.0f);
    const float dy = fmaxf(fmaxf(lo.y - qy, qy - hi.y), 0.0f);
    const float dz = fmaxf(fmaxf(lo.z - qz, qz - hi.z), 0.0f);
    return dx * dx + dy * dy + dz * dz;
}

// S: stack entries.  The first pass (kDeep false) runs every query with a
// 32-entry stack; a query whose path needs more appends itself to `spill`
// and the deep pass (kDeep, 64 entries) redoes it, so no query's result
// depends on the stack size.
template <int K, int S, bool kDeep>
__device__ __forceinline__ void knn_body(int64_t n, IndexHeader *__restrict__ hdr, const float4 *__restrict__ pts,
                                         const uint32_t *__restrict__ perm, const Node *__restrict__ nodes, int k_out,
                                         int32_t *__restrict__ out_ids, float *__restrict__ out_d2,
                                         const IndexHeader *__restrict__ clouds, const int64_t *__restrict__ cloud_cells,
                                         int n_clouds, int sorted_rows, uint32_t *__restrict__ spill) {
    __shared__ uint32_t stack[S][kKnnThreads];
    int64_t i;
    if constexpr (kDeep) {
        const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
        if (t >= (int64_t)hdr->knn_spill) return;
        i = spill[t];
    } else {
        i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
        if (i >= n) return;
    }
    const float4 q = pts[i];
    float d[K];
    int32_t id[K];
#pragma unroll
    for (int t = 0; t < K; ++t) d[t] = FLT_MAX, id[t] = -1;
    // a node is pruned when its box is farther than the K-th distance (with
    // a relative margin for the rounding of the two squared distances)
    auto far = [&](float bd) { return bd * (1.0f - 1e-6f) > d[K - 1]; };
    auto offer = [&](const float4 &p, uint32_t j) {
        const float dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
        const float dd = dx * dx + dy * dy + dz * dz;
        if (dd < d[K - 1]) {  // sorted insertion, ties keep the earlier point
            d[K - 1] = dd;
            id[K - 1] = (int32_t)j;
#pragma unroll
            for (int u = K - 1; u > 0; --u) {
                if (d[u] < d[u - 1]) {
                    const float td = d[u];
                    d[u] = d[u - 1];
                    d[u - 1] = td;
                    const int32_t ti = id[u];
                    id[u] = id[u - 1];
                    id[u - 1] = ti;
                }
            }
        }
    };
    // a batch searches the query's own cloud (its subtree)
    uint32_t ref = hdr->root_ref;
    if (clouds != nullptr) {
        int lo = 0, hi = n_clouds - 1;  // largest c with cloud_cells[c] <= i
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (cloud_cells[mid] <= i) lo = mid;
            else hi = mid - 1;
        }
        ref = clouds[lo].root_ref;
    }
    int sp = 0;
    bool spilled = false;
    while (true) {
        if (is_leaf(ref)) {
            const uint32_t f = leaf_first(ref), c = leaf_count(ref);
            // kLoads loads in flight, then as many offers (leaf order kept)
            for (uint32_t t = 0; t < c; t += kLoads) {
                float4 p[kLoads];
#pragma unroll
                for (int u = 0; u < kLoads; ++u) p[u] = pts[f + min(t + (uint32_t)u, c - 1u)];
#pragma unroll
                for (int u = 0; u < kLoads; ++u) {
                    const uint32_t j = f + t + (uint32_t)u;
                    if (t + (uint32_t)u < c && (int64_t)j != i) offer(p[u], j);
                }
            }
        } else {
            const Node nd = nodes[ref];
            const float b0 = box_dist2(nd.lo0, nd.hi0, q.x, q.y, q.z);
            const float b1 = box_dist2(nd.lo1, nd.hi1, q.x, q.y, q.z);
            const bool near0 = b0 <= b1;
            const float bn = near0 ? b0 : b1, bf = near0 ? b1 : b0;
            if (!far(bf)) {
                if (sp == S) {
                    spilled = true;
                    break;
                }
                stack[sp++][threadIdx.x] = (ref << 1) | (near0 ? 1u : 0u);
            }
            if (!far(bn)) {
                ref = __float_as_uint(near0 ? nd.hi0.w : nd.hi1.w);
                continue;
            }
        }
        bool have = false;
        while (sp > 0 && !have) {
            const uint32_t e = stack[--sp][threadIdx.x];
            const Node nd = nodes[e >> 1];
            const float4 lo = (e & 1u) ? nd.lo1 : nd.lo0, hi = (e & 1u) ? nd.hi1 : nd.hi0;
            if (!far(box_dist2(lo, hi, q.x, q.y, q.z))) {
                ref = __float_as_uint(hi.w);
                have = true;
            }
        }
        if (!have) break;
    }
    if (!kDeep && spilled) {
        spill[atomicAdd(&hdr->knn_spill, 1u)] = (uint32_t)i;
        return;
    }
    // short lists repeat the last id found; with none found the reference
    // writes 0, a batch writes the point itself (0 may be another cloud's).
    // sorted_rows: row i (sorted order) of sorted ids, self as padding, and
    // (out_d2 non-null) out_d2[i] = the squared distance of the row's last
    // neighbour, FLT_MAX when the row is short (it then holds every other
    // point the search could reach).
    if (sorted_rows) {
        const int64_t o = i * k_out;
        int32_t last = (int32_t)i;
        float dk = FLT_MAX;
        for (int t = 0; t < k_out; ++t) {
            if (id[t] >= 0) last = id[t];
            out_ids[o + t] = last;
            dk = id[t] >= 0 ? d[t] : FLT_MAX;
        }
        if (out_d2) out_d2[i] = dk;
        return;
    }
    const int64_t o = (int64_t)perm[i] * k_out;
    int32_t last = clouds != nullptr ? (int32_t)perm[i] : 0;
    for (int t = 0; t < k_out; ++t) {
        if (id[t] >= 0) last = (int32_t)perm[id[t]];
        out_ids[o + t] = last;
        if (out_d2) out_d2[o + t] = id[t] >= 0 ? d[t] : FLT_MAX;
    }
}

// ------------------------------------------------------------------ guesses
constexpr int kDppXor3 = 0x1B;        // quad_perm [3, 2, 1, 0]
constexpr int kDppHalfMirror = 0x141;  // lane ^ 7
constexpr int kDppMirror = 0x140;      // lane ^ 15
constexpr int kGroupStack = 32;
// Up to this many queries a group of lanes each, above it a lane each.  One
// lane per query does less work in total but is a serial chain of some 300
// dependent loads, as long as the longest query of its wave, and few waves
// are in flight.  Whole calls with groups / with lanes: uniform points 1 k
// 0.55 / 0.74 ms, 16 k 0.93 / 1.10, 50 k 1.82 / 1.98, 100 k 2.65 / 2.73,
// 197 k 4.38 / 4.39, 350 k 7.18 / 7.14, 1.4 M 25.9 / 24.8; 90% in 64 clusters
// 50 k 2.06 / 2.39, 197 k 4.62 / 4.70, 350 k 7.60 / 7.53, 1.4 M 33.9 / 32.7; half
// in 256 clusters 197 k 4.58 / 4.68, 350 k 7.38 / 7.47, 700 k 13.4 / 13.2; LiDAR
// scans 50 k 7.26 / 7.48, 197 k 16.6 / 16.7, 350 k 20.9 / 20.8, 700 k 45.6 / 45.1.
// Only strongly graded points (x^4 of uniform ones) favour groups at every
// size: 197 k 5.2 / 6.5, 350 k 9.1 / 10.7, 1.4 M 38.4 / 40.9.
constexpr int64_t kGroupQueries = 3 << 16;

// One compare-exchange of a sorting network over a row: the lane and its
// partner (pd, pid) order their distances; `low`: the lane is the lower one.
__device__ __forceinline__ void exchange(uint32_t &d, int &id, uint32_t pd, int pid, bool low) {
    const uint32_t x = low ? min(d, pd) : max(d, pd);
    id = x == d ? id : pid;  // (equal distances stay where they are)
    d = x;
}
template <int C>
__device__ __forceinline__ void exchange(uint32_t &d, int &id, bool low) {
    exchange(d, id, (uint32_t)dpp<C>((int)d), dpp<C>(id), low);
}
__device__ __forceinline__ void exchange_xor4(uint32_t &d, int &id, bool low) {
    exchange(d, id, (uint32_t)dpp<kDppXor3>(dpp<kDppHalfMirror>((int)d)), dpp<kDppXor3>(dpp<kDppHalfMirror>(id)), low);
}

// The same neighbours as knn_kernel's, for rows of guesses: 16 lanes per
// query walk the 16-wide form of the hierarchy, a child per lane, and keep
// the 16 nearest sorted, one per lane.  A leaf's points come 16 at a time;
// if any is nearer than the K-th, the 16 are sorted and merged (a network of
// 15 exchanges).  The four queries of a wave step together.  Bound by VALU
// issue (about 110 instructions per step of the walk and 90 per merge).  It
// takes 32 us on 1 k points, 50 on 10 k and 106 on a 65 k LiDAR scan, where a
// lane per query takes 198, 240 and 273.  Of two points at the same distance
// either may take the last place.
__global__ void __launch_bounds__(256) knn_group_kernel(int64_t n, IndexHeader *__restrict__ hdr,
                                                        const float4 *__restrict__ pts,
                                                        const Node *__restrict__ nodes,
                                                        const WideChild *__restrict__ wide, int k,
                                                        int32_t *__restrict__ out_ids, float *__restrict__ out_d2,
                                                        const int64_t *__restrict__ cloud_cells, int n_clouds,
                                                        uint32_t *__restrict__ spill) {
    const int lane64 = threadIdx.x & 63, gl = threadIdx.x & 15;
    const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) >> 4;
    auto gballot = [&](bool p) {
        const uint64_t m = __ballot(p);
        return ((lane64 < 32 ? (uint32_t)m : (uint32_t)(m >> 32)) >> (lane64 & 16)) & 0xFFFFu;
    };
    bool go = i < n;
    const float4 q = pts[go ? i : 0];
    int64_t a = 0, z = n;
    if (cloud_cells != nullptr && go) {
        int lo = 0, hi = n_clouds - 1;  // largest c with cloud_cells[c] <= i
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (cloud_cells[mid] <= i) lo = mid;
            else hi = mid - 1;
        }
        a = cloud_cells[lo], z = cloud_cells[lo + 1];
    }
    const uint32_t root = wide_ref((uint32_t)n, (uint32_t)a, (uint32_t)(z - a));
    constexpr uint32_t kNone = 0x7F7FFFFFu;  // FLT_MAX
    uint32_t d = kNone;                      // (distances are >= 0: they order as their bits)
    int id = -1;
    float worst = FLT_MAX;
    // partly visited nodes: (reference, children left)
    __shared__ uint2 stack[kGroupStack][16];
    uint2 *const mine = &stack[0][threadIdx.x >> 4];
    int sz = 0;
    const bool root_leaf = is_leaf(root);
    uint32_t base = root_leaf ? leaf_first(root) : 0u;
    int o = 0, cnt = root_leaf ? (int)leaf_count(root) : 0;
    uint32_t node = root, left = root_leaf ? 0u : 0xFFFFu, ref = kWideNone;
    float key = FLT_MAX;
    bool fresh = root_leaf, spilled = false;
    const bool low1 = (gl & 1) == 0, low2 = (gl & 2) == 0, low4 = (gl & 4) == 0, low8 = (gl & 8) == 0;
    while (true) {
        bool walk = go && o >= cnt;
        while (__ballot(walk) != 0ull) {
            if (walk && !fresh) {
                const bool binary = (node & kWideBinary) != 0u;
                const float4 *box = binary ? (const float4 *)&nodes[node & ~kWideBinary] + 2 * (gl & 1)
                                           : (const float4 *)&wide[16u * node + (uint32_t)gl];
                const float4 lo = box[0], hi = box[1];
                ref = __float_as_uint(hi.w);
                if (binary) ref = gl < 2 ? (is_leaf(ref) ? ref : ref | kWideBinary) : kWideNone;
                const bool need = ((left >> gl) & 1u) != 0u && ref != kWideNone;
                left = gballot(need);
                key = need ? box_dist2(lo, hi, q.x, q.y, q.z) : FLT_MAX;
            }
            // the nearest child left that is not farther than the K-th (with
            // a relative margin for the rounding of the two distances)
            const uint32_t in = gballot(!(key * (1.0f - 1e-6f) > worst)) & left;
            uint32_t kmin = __float_as_uint(key);  // (keys are >= 0)
            kmin = min(kmin, (uint32_t)dpp<kDppXor1>((int)kmin));
            kmin = min(kmin, (uint32_t)dpp<kDppXor2>((int)kmin));
            kmin = min(kmin, (uint32_t)dpp<kDppRor4>((int)kmin));
            kmin = min(kmin, (uint32_t)dpp<kDppRor8>((int)kmin));
            const uint32_t at = gballot(__float_as_uint(key) == kmin) & in;
            const int c = (int)__builtin_ctz((at ? at : in) | 0x10000u) & 15;
            const uint32_t r = (uint32_t)__shfl((int)ref, c, 16);
            const bool has = walk & (in != 0u);
            left = walk ? in & ~(1u << c) : left;
            key = (has & (gl == c)) ? FLT_MAX : key;
            const bool leaf = has & is_leaf(r), down = has & !is_leaf(r), back = walk & !has;
            const bool end = back & (sz == 0), keep = down & (left != 0u), full = keep & (sz >= kGroupStack);
            if (keep & !full) mine[16 * sz] = make_uint2(node, left);
            const uint2 up = mine[16 * max(sz - 1, 0)];
            const bool pop = back & !end;
            sz += (keep & !full) ? 1 : (pop ? -1 : 0);
            node = down ? r : (pop ? up.x : node);
            left = down ? 0xFFFFu : (pop ? up.y : left);
            fresh = walk ? !(down | back) : fresh;
            base = leaf ? leaf_first(r) : base;
            cnt = leaf ? (int)leaf_count(r) : cnt;
            o = leaf ? 0 : o;
            spilled |= full;
            go &= !(end | full);
            walk &= !(leaf | end | full);
        }
        if (__ballot(go) == 0ull) break;
        const uint32_t j = base + (uint32_t)(o + gl);
        const bool has = go && o + gl < cnt && (int64_t)j != i;
        const float4 p = pts[has ? (int64_t)j : 0];
        const float dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
        const float dd = dx * dx + dy * dy + dz * dz;
        const bool nearer = has && dd < worst;
        o += go ? 16 : 0;
        if (__ballot(nearer) != 0ull) {
            uint32_t e = nearer ? __float_as_uint(dd) : kNone;
            int ie = nearer ? (int)j : -1;
            exchange<kDppXor1>(e, ie, low1);
            exchange<kDppXor3>(e, ie, low2);
            exchange<kDppXor1>(e, ie, low1);
            exchange<kDppHalfMirror>(e, ie, low4);
            exchange<kDppXor2>(e, ie, low2);
            exchange<kDppXor1>(e, ie, low1);
            exchange<kDppMirror>(e, ie, low8);
            exchange_xor4(e, ie, low4);
            exchange<kDppXor2>(e, ie, low2);
            exchange<kDppXor1>(e, ie, low1);
            // the 16 smaller ones of the two sorted rows, then their order
            exchange(d, id, (uint32_t)dpp<kDppMirror>((int)e), dpp<kDppMirror>(ie), true);
            exchange<kDppRor8>(d, id, low8);
            exchange_xor4(d, id, low4);
            exchange<kDppXor2>(d, id, low2);
            exchange<kDppXor1>(d, id, low1);
            worst = __uint_as_float((uint32_t)__shfl((int)d, k - 1, 16));
        }
        go &= o < cnt || left != 0u || sz > 0;
    }
    if (i >= n) return;
    if (spilled) {
        if (gl == 0) spill[atomicAdd(&hdr->knn_spill, 1u)] = (uint32_t)i;
        return;
    }
    // the row as knn_body writes it
    const int found = __popc(gballot(id >= 0));
    const int last = __shfl(id, found > 0 ? found - 1 : 0, 16);
    if (gl < k) out_ids[i * k + gl] = gl < found ? id : (found > 0 ? last : (int)i);
    if (out_d2 && gl == 0) out_d2[i] = found >= k ? worst : FLT_MAX;
}

#define PG_KNN_ARGS                                                                                                 \
    int64_t n, IndexHeader *__restrict__ hdr, const float4 *__restrict__ pts, const uint32_t *__restrict__ perm,    \
        const Node *__restrict__ nodes, int k_out, int32_t *__restrict__ out_ids, float *__restrict__ out_d2,       \
        const IndexHeader *__restrict__ clouds, const int64_t *__restrict__ cloud_cells, int n_clouds,               \
        int sorted_rows, uint32_t *__restrict__ spill
// first pass: 128 VGPRs and 16 KB of LDS per block, four waves per SIMD
template <int K>
__global__ void __launch_bounds__(kKnnThreads) __attribute__((amdgpu_waves_per_eu(4, 4)))
    knn_kernel(PG_KNN_ARGS) {
    knn_body<K, kKnnStackFast, false>(n, hdr, pts, perm, nodes, k_out, out_ids, out_d2, clouds, cloud_cells, n_clouds,
                                      sorted_rows, spill);
}
template <int K>
__global__ void __launch_bounds__(kKnnThreads) knn_deep_kernel(PG_KNN_ARGS) {
    knn_body<K, kKnnStack, true>(n, hdr, pts, perm, nodes, k_out, out_ids, out_d2, clouds, cloud_cells, n_clouds,
                                 sorted_rows, spill);
}
#undef PG_KNN_ARGS

__global__ void knn_reset_kernel(IndexHeader *hdr) { hdr->knn_spill = 0u; }

template <int K>
static void launch_knn(int64_t n, IndexHeader *hdr, const float4 *pts, const uint32_t *perm, const Node *nodes, int k,
                       int32_t *ids, float *d2, const IndexHeader *clouds, const int64_t *cloud_cells, int n_clouds,
                       int sorted, uint32_t *spill, hipStream_t stream) {
    const unsigned grid = (unsigned)((n + kKnnThreads - 1) / kKnnThreads);
    hipLaunchKernelGGL(knn_reset_kernel, dim3(1), dim3(1), 0, stream, hdr);
    hipLaunchKernelGGL(knn_kernel<K>, dim3(grid), dim3(kKnnThreads), 0, stream, n, hdr, pts, perm, nodes, k, ids, d2,
                       clouds, cloud_cells, n_clouds, sorted, spill);
    // the deep pass reads the spill count on the device; its grid covers
    // every query in case all of them spilled (blocks past the count exit)
    hipLaunchKernelGGL(knn_deep_kernel<K>, dim3(grid), dim3(kKnnThreads), 0, stream, n, hdr, pts, perm, nodes, k, ids,
                       d2, clouds, cloud_cells, n_clouds, sorted, spill);
}

hipError_t knn(int64_t n, void *index_ws, int k, int32_t *ids, float *d2, hipStream_t stream, int n_clouds,
               bool sorted_rows) {
    if (n <= 0) return hipSuccess;
    const IndexLayout L = make_index_layout(n);
    char *ws = (char *)index_ws;
    const IndexHeader *clouds = nullptr;
    const int64_t *cloud_cells = nullptr;
    if (n_clouds > 0) {
        const BatchLayout B = make_batch_layout(n, n_clouds);
        clouds = (const IndexHeader *)(ws + B.clouds);
        cloud_cells = (const int64_t *)(ws + B.offsets);
    }
    IndexHeader *hdr = (IndexHeader *)(ws + L.header);
    const float4 *pts = (const float4 *)(ws + L.points);
    const uint32_t *perm = (const uint32_t *)(ws + L.perm);
    const Node *nodes = (const Node *)(ws + L.nodes);
    uint32_t *spill = (uint32_t *)(ws + L.vals_alt);
    if (sorted_rows && k <= 16 && n <= kGroupQueries) {
        hipLaunchKernelGGL(knn_reset_kernel, dim3(1), dim3(1), 0, stream, hdr);
        hipLaunchKernelGGL(knn_group_kernel, dim3((unsigned)((n + 15) / 16)), dim3(256), 0, stream, n, hdr, pts, nodes,
                           (const WideChild *)(ws + L.boxes), k, ids, d2, cloud_cells, n_clouds, spill);
        hipLaunchKernelGGL(knn_deep_kernel<16>, dim3((unsigned)((n + kKnnThreads - 1) / kKnnThreads)),
                           dim3(kKnnThreads), 0, stream, n, hdr, pts, perm, nodes, k, ids, d2, clouds, cloud_cells,
                           n_clouds, 1, spill);
        return hipGetLastError();
    }
    if (k <= 8)
        launch_knn<8>(n, hdr, pts, perm, nodes, k, ids, d2, clouds, cloud_cells, n_clouds, sorted_rows ? 1 : 0, spill,
                      stream);
    else
        launch_knn<16>(n, hdr, pts, perm, nodes, k, ids, d2, clouds, cloud_cells, n_clouds, sorted_rows ? 1 : 0, spill,
                       stream);
    return hipGetLastError();
}

}  // namespace pg
