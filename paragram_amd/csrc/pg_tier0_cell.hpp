// Tier 0: every cell starts here.  16 lanes build one cell together in FP32,
// with the whole cell in LDS; a wave holds four cells.  Included by
// pg_cell.hip after pg_group_cell.hpp (the larger, FP64-capable tiers), whose
// reductions and row-pool helpers it shares.
//
// Per cell in LDS (about 3.2 KB):
//   vpos[64]  float4  vertex position y = N/D in seed-relative doubled
//                     coordinates, and a rigorous error radius (w)
//   vr2[64]   float   upper bound of |y|^2
//   vtri[64]  uint32  plane triple (i, j, k), ordered so that D > 0
//   pl[48]    float4  plane normal a and offset H (a . y <= H)
//   own[48]   int32   the plane's owner (sorted point id, or a negative
//                     box-plane code)
//   tmp[64]   uint32  clip and emission scratch
//   cand, cown [16]   planes and owners of the batch being offered
//   pm[24]    uint32  per plane, a 16-bit mask of the lanes whose removed
//                     triangle holds the plane; zero between clips
//   tent[8]   2 x u32 removal tests taken by their FP32 sign
// The nv vertices lie in slots 0 .. nv - 1 without gaps (slot v = lane + 16 k
// belongs to lane v mod 16): a clip puts its new vertices in the slots of the
// removed ones and, if there are fewer, moves the last vertices into the
// rest, so every sweep covers only the rows in use and needs no mask.
//
// Lane parallelism: vertex sweeps, the batch of up to 16 candidates (one per
// lane: tested against all vertices at once, then the few that may cut are
// offered in order), the 16 children of a node of the hierarchy's wide form, the
// boundary edges of a clip and the new vertices they make, bounds reductions
// and the row sort.  All control decisions are group-uniform.
//
// The kernel is bound by VALU issue (rocprofv3, 1 M uniform points: 7.89e9
// wave instructions fill 89% of the issue slots, with 38 of 64 lanes active), not
// by memory or latency, so a step is worth what it saves in instructions.
// Against four cells that share a binary walk (32 vertex slots with a valid
// mask, both children of a node tested by every lane), one group walking the
// 16-wide form for itself visits a tenth of the nodes, and its lanes test
// different boxes: 8.1e9 instructions in place of 10.2e9 on 1 M uniform
// points, and the tier took 15.7 ms in place of 20.2 (14.5 with the later
// steps).  The exact ball test of a child is put off until the walk comes to
// it, and is done by the whole group, a vertex per lane: testing it for each
// child by that child's lane took 23.7 ms.  The walk itself is written as
// selects in one loop that the wave steps through together (20.9 -> 20.0 ms):
// in divergent branches each join copies the walk's state.
//
// The lanes of a group exchange planes, vertices, lists and candidates through
// LDS; each exchange goes across lds_fence(), which costs nothing measurable
// (1 M uniform 17.28 -> 17.30 ms, 256 LiDAR clouds 572.8 -> 572.8).
#pragma once

namespace pg {

struct alignas(16) Tier0LDS {
    float4 vpos[64];  // y~ and w (see store_vertex)
    float4 pl[48];
    float4 cand[16];
    float vr2[64];
    int own[48];
    int cown[16];
    uint32_t vtri[64];
    uint32_t tmp[64];
    uint32_t pm[24];
    // removal tests taken by their FP32 sign: the vertex's plane triple
    // (slots, kept and renumbered by the plane collection), and the query
    // point with the sign taken in bit 31
    uint32_t tent[kTentMax][2];
    // their number (every lane of the group writes it, with the same value,
    // so each lane reads back its own store)
    uint32_t ntent;
};

struct Tier0 {
    static constexpr int G = 16, V = 64, P = 48;
    static constexpr int kRows = V / G;    // vertex slots per lane
    static constexpr int kPRows = P / G;   // plane slots per lane
    static constexpr int kB = 8;           // bits of a plane slot in a triple
    static constexpr uint32_t kBMask = (1u << kB) - 1u;
    static constexpr int kSlotShift = 24;  // a vertex slot above a triple in a word
    static constexpr int kStack = 32;      // partly visited nodes (at most one per level: 8 wide levels, and
                                           // binary ones below an oversize subtree; a cell
                                           // whose walk needs more goes to tier m)

    using LDS = Tier0LDS;
    LDS *S;
    uint32_t *ctr;  // the wave's diagnostics counters (LDS)
    uint32_t stk_node[kStack / G], stk_left[kStack / G];
    int gl;      // lane within the group
    int lane64;

    const float4 *pts;
    const Node *nodes;
    const WideChild *wide;
    const IndexHeader *hdr;
    uint32_t root;  // the cloud's wide form

    uint32_t seed;
    float sx, sy, sz, sw;
    int nv, np;  // vertices and planes held, in slots 0 .. nv - 1 and 0 .. np - 1
    float L_[3], U_[3];  // AABB of the cell
    float EM_;           // largest vertex error radius w of the cell
    float R2_;           // largest bound of |y|^2
    bool bounded;
    int status;
    bool overflow;  // the cell left this tier (capacity, or `bail`)
    // why the tier gave the cell up (0: it did not, or capacity): 1 more
    // undecided removal tests than the record holds, 2 an undecided vertex
    // orientation, 3 a predicted cube that cut the cell
    uint32_t bail;
    bool cube;      // the cell started inside a predicted cube (see init_box)
    bool active;  // the group holds a cell in this round
    bool dirty;   // the cell changed since the AABB was computed
    uint64_t bloom;
    bool in_guess;
    // After the pre-clip: every point nearer the seed than this (squared,
    // lowered by a margin) is one of the guesses already offered.
    float guess_r2;

    // diagnostics counters live in LDS (registers are the scarce resource)
    __device__ __forceinline__ void count(int slot, uint32_t v = 1u) const { atomicAdd(&ctr[slot], v); }

    // ---------------------------------------------------------- group ops
    // the group's bits of a wave mask, its lane 0 at bit 0
    __device__ __forceinline__ uint32_t gbits(uint64_t m) const {
        const uint32_t w = lane64 < 32 ? (uint32_t)m : (uint32_t)(m >> 32);
        return (w >> (lane64 & 16)) & 0xFFFFu;
    }
    __device__ __forceinline__ uint32_t gballot(bool p) const { return gbits(__ballot(p)); }
    __device__ __forceinline__ bool gany(bool p) const { return gballot(p) != 0u; }
    // set bits of a group mask below this lane
    __device__ __forceinline__ int grank(uint32_t bits) const { return __popc(bits & ((1u << gl) - 1u)); }
    __device__ __forceinline__ bool live() const { return active && status == kSuccess && !overflow; }
    __device__ __forceinline__ int gbi(int x, int k) const { return __shfl(x, k, G); }
    __device__ __forceinline__ float gbf(float x, int k) const { return __shfl(x, k, G); }
    __device__ __forceinline__ uint64_t gor64(uint64_t x) const {
        return ((uint64_t)row_or((uint32_t)(x >> 32)) << 32) | row_or((uint32_t)x);
    }
    // exclusive prefix sum over the group; total in `tot`
    __device__ __forceinline__ int gexcl(int x, int &tot) const {
        const int incl = row_scan(x);
        tot = dpp<kDppLast>(incl);
        return incl - x;
    }
    // ---------------------------------------------------------- vertices
    // Builds vertex (i, j, k) into `slot` (one lane).  With
    // |N - N~| <= g pN and |D - D~| <= g pD (g = 2e-6), the position error is
    // |y - N~/D~| <= (g pN + |y~| g pD) / (D~ - g pD), plus division rounding.
    // Returns false when the FP32 orientation is not safely positive (the cell
    // then goes to the FP64-capable tiers).  Ill-conditioned vertices (nearly
    // parallel or coaxial planes) are kept with their large radius: an FP64
    // call site here costs registers on every cell, and a test such a vertex
    // leaves open is recorded.
    __device__ __forceinline__ bool make_vertex(int slot, uint32_t i, uint32_t j, uint32_t k) {
        const float4 A = S->pl[i], B = S->pl[j], C = S->pl[k];
        const float pHA = plane_perm(A), pHB = plane_perm(B), pHC = plane_perm(C);
        const float c1x = B.y * C.z - B.z * C.y, c1y = B.z * C.x - B.x * C.z, c1z = B.x * C.y - B.y * C.x;
        const float c2x = C.y * A.z - C.z * A.y, c2y = C.z * A.x - C.x * A.z, c2z = C.x * A.y - C.y * A.x;
        const float c3x = A.y * B.z - A.z * B.y, c3y = A.z * B.x - A.x * B.z, c3z = A.x * B.y - A.y * B.x;
        const float D = A.x * c1x + A.y * c1y + A.z * c1z;
        const float Nx = A.w * c1x + B.w * c2x + C.w * c3x;
        const float Ny = A.w * c1y + B.w * c2y + C.w * c3y;
        const float Nz = A.w * c1z + B.w * c2z + C.w * c3z;
        const float ax = fabsf(A.x), ay = fabsf(A.y), az = fabsf(A.z);
        const float bx = fabsf(B.x), by = fabsf(B.y), bz = fabsf(B.z);
        const float cx = fabsf(C.x), cy = fabsf(C.y), cz = fabsf(C.z);
        const float q1x = by * cz + bz * cy, q1y = bz * cx + bx * cz, q1z = bx * cy + by * cx;
        const float q2x = cy * az + cz * ay, q2y = cz * ax + cx * az, q2z = cx * ay + cy * ax;
        const float q3x = ay * bz + az * by, q3y = az * bx + ax * bz, q3z = ax * by + ay * bx;
        const float pD = ax * q1x + ay * q1y + az * q1z;
        const float pNx = pHA * q1x + pHB * q2x + pHC * q3x;
        const float pNy = pHA * q1y + pHB * q2y + pHC * q3y;
        const float pNz = pHA * q1z + pHB * q2z + pHC * q3z;
        const uint32_t tri = tri_pack<kB>(i, j, k);
        const float eD = kG32 * pD;
        float4 pos = make_float4(0.f, 0.f, 0.f, -1.0f);
        bool ok = D > 2.0f * eD && pD > kTiny32;
        if (ok) {
            // hardware reciprocals (1 ulp): their error, and the products',
            // lie far inside the kSlack = 1e-6 relative terms of the bound
            const float inv = __builtin_amdgcn_rcpf(D);
            const float den = (1.0f + kSlack) * __builtin_amdgcn_rcpf(D - eD);
            const float x = Nx * inv, y = Ny * inv, z = Nz * inv;
            const float ex = (kG32 * pNx + fabsf(x) * eD) * den + fabsf(x) * kSlack;
            const float ey = (kG32 * pNy + fabsf(y) * eD) * den + fabsf(y) * kSlack;
            const float ez = (kG32 * pNz + fabsf(z) * eD) * den + fabsf(z) * kSlack;
            pos = make_float4(x, y, z, fmaxf(ex, fmaxf(ey, ez)) + kTiny32);
        } else if (D < -eD && pD > kTiny32 && S->ntent == 0u) {
            count(kStatInconsistent);
        }
        store_vertex(slot, pos);
        S->vtri[slot] = tri;
        return ok;
    }

    // The permanent of a plane's offset H = |a|^2 - dw, |a|^2 + |dw|, from
    // the plane (box planes have |a| = 1 and H >= 2, which gives H).
    __device__ __forceinline__ static float plane_perm(const float4 &A) {
        const float a2 = A.x * A.x + A.y * A.y + A.z * A.z;
        return a2 + fabsf(a2 - A.w);
    }

    // Vertex record: y~ and w = eps (1 + s) + 2e-6 max_k |y~_k|, which bounds
    // both the position error eps and the removal filter's rounding term
    // 2e-6 sum_k |a_k y~_k| <= 2e-6 |a|_1 max_k |y~_k|.  vr2 bounds |y|^2 (the ball
    // of balls_clear).
    __device__ __forceinline__ void store_vertex(int slot, float4 pos) {
        const float w = pos.w * (1.0f + kSlack) + kG32 * fmaxf(fabsf(pos.x), fmaxf(fabsf(pos.y), fabsf(pos.z)));
        S->vpos[slot] = make_float4(pos.x, pos.y, pos.z, w);
        const float rx = fabsf(pos.x) + w, ry = fabsf(pos.y) + w, rz = fabsf(pos.z) + w;
        S->vr2[slot] = fmaf(rx, rx, fmaf(ry, ry, rz * rz)) * (1.0f + 4.0f * kSlack);
    }

    // ---------------------------------------------------------- bounds
    __device__ __forceinline__ void update_bounds() {
        float lo0 = FLT_MAX, lo1 = FLT_MAX, lo2 = FLT_MAX, hi0 = -FLT_MAX, hi1 = -FLT_MAX, hi2 = -FLT_MAX, em = 0.0f;
        float r2 = 0.0f;
#pragma unroll
        for (int k = 0; k < kRows; ++k) {
            if (__ballot(nv > G * k) == 0ull) break;
            if (gl + G * k < nv) {
                const float4 p = S->vpos[gl + G * k];
                lo0 = fminf(lo0, p.x - p.w);
                hi0 = fmaxf(hi0, p.x + p.w);
                lo1 = fminf(lo1, p.y - p.w);
                hi1 = fmaxf(hi1, p.y + p.w);
                lo2 = fminf(lo2, p.z - p.w);
                hi2 = fmaxf(hi2, p.z + p.w);
                em = fmaxf(em, p.w);
                r2 = fmaxf(r2, S->vr2[gl + G * k]);
            }
        }
        L_[0] = row_min(lo0), L_[1] = row_min(lo1), L_[2] = row_min(lo2);
        U_[0] = row_max(hi0), U_[1] = row_max(hi1), U_[2] = row_max(hi2);
        EM_ = row_max(em);
        R2_ = row_max(r2);
        bounded = EM_ < FLT_MAX;
    }

    // Can the plane of candidate c not cut the cell?  max over the AABB of
    // a . y is sum_k max(a_k L_k, a_k U_k).
    __device__ __forceinline__ bool too_far(const float4 &c, float pH) const {
        if (!bounded) return false;
        const float S_ = fmaxf(c.x * L_[0], c.x * U_[0]) + fmaxf(c.y * L_[1], c.y * U_[1]) +
                         fmaxf(c.z * L_[2], c.z * U_[2]);
        const float M = fabsf(c.x) * fmaxf(fabsf(L_[0]), fabsf(U_[0])) +
                        fabsf(c.y) * fmaxf(fabsf(L_[1]), fabsf(U_[1])) +
                        fabsf(c.z) * fmaxf(fabsf(L_[2]), fabsf(U_[2]));
        return (c.w - S_) > kSlack * (pH + M) + kTiny32;
    }

    // Node prune.  Every point p of the box has a = p - s with |a| >= d and
    // H = |a|^2 - (w_p - w_s) >= |a|^2 - dw (dw = w_max - w_s).  Two tests,
    // either of which suffices:
    //  * octant radius (voronoi_bvh.cuh:71-107, pwr_bvh.cuh:150-185): a . y
    //    <= |a| rho with rho the largest AABB corner radius over the octants
    //    the box overlaps, so no cut when |a|^2 - rho |a| - dw >= 0 for all
    //    |a| >= d, i.e. 2d >= rho and (d^2 - dw)^2 >= rho^2 d^2, d^2 > dw;
    //  * the per-vertex balls (balls_clear), the exact form.
    // Each lane tests its own box.
    __device__ __forceinline__ bool octant_clear(const float4 &lo, const float4 &hi, float &key) const {
        const float alx = lo.x - sx, aly = lo.y - sy, alz = lo.z - sz;
        const float ahx = hi.x - sx, ahy = hi.y - sy, ahz = hi.z - sz;
        const float dx = fmaxf(fmaxf(alx, -ahx), 0.0f);
        const float dy = fmaxf(fmaxf(aly, -ahy), 0.0f);
        const float dz = fmaxf(fmaxf(alz, -ahz), 0.0f);
        const float d2 = dx * dx + dy * dy + dz * dz;
        const float dw = lo.w - sw;
        key = d2 - dw;
        // the octants a box overlaps form a product set, so the largest
        // corner radius over them is a sum of per-axis maxima
        const float rx = max0(alx <= 0.0f ? fabsf(L_[0]) : 0.0f, ahx >= 0.0f ? fabsf(U_[0]) : 0.0f);
        const float ry = max0(aly <= 0.0f ? fabsf(L_[1]) : 0.0f, ahy >= 0.0f ? fabsf(U_[1]) : 0.0f);
        const float rz = max0(alz <= 0.0f ? fabsf(L_[2]) : 0.0f, ahz >= 0.0f ? fabsf(U_[2]) : 0.0f);
        // (and no vertex is farther out than R2)
        const float rho2 = fminf(rx * rx + ry * ry + rz * rz, R2_) * (1.0f + kSlack);
        const float d2lo = d2 * (1.0f - kSlack);
        const float h = d2lo - dw - weight_slack(lo.w);
        return bounded & (4.0f * d2lo > rho2) & (h > 0.0f) & (h * h > rho2 * d2 * (1.0f + kSlack));
    }
    // the larger of two floats that are not negative, by their bits (fmaxf
    // would quiet a NaN of either first: two instructions more)
    __device__ __forceinline__ static float max0(float a, float b) {
        return __uint_as_float(max(__float_as_uint(a), __float_as_uint(b)));
    }
    __device__ __forceinline__ float weight_slack(float w) const { return kSlack * (fabsf(w) + fabsf(sw)) + kTiny32; }

    // Exact form of the prune, per vertex.  Vertex y is beyond the plane of
    // p iff a . y - |a|^2 + dw > 0, i.e. in doubled coordinates
    // |2a - y|^2 < |y|^2 + 4 dw: p lies in the ball about the vertex through
    // the seed (grown by the weight difference).  No point of the box cuts the
    // cell when the box misses every vertex's ball.  The box [2 al, 2 ah] is
    // widened by the cell's largest error radius (each coordinate of y lies
    // within w of y~), and vr2 = sum_k (|y~_k| + w)^2 bounds |y|^2.   Each lane
    // holds one box; the vertices are read in order, each by the whole group.
    __device__ __forceinline__ bool balls_clear(const float4 &lo, const float4 &hi) const {
        const float Ax = fmaf(2.0f, lo.x - sx, -EM_), Ay = fmaf(2.0f, lo.y - sy, -EM_), Az = fmaf(2.0f, lo.z - sz, -EM_);
        const float Bx = fmaf(2.0f, hi.x - sx, EM_), By = fmaf(2.0f, hi.y - sy, EM_), Bz = fmaf(2.0f, hi.z - sz, EM_);
        const float dw4 = 4.0f * (lo.w - sw + weight_slack(lo.w));
        bool cut = false;
#pragma unroll
        for (int k = 0; k < kRows; ++k) {
            if (__ballot(nv > G * k) == 0ull) break;
            const int v = gl + G * k;
            const float4 p = S->vpos[v];
            // distance to the box per axis: y minus y clamped to [A, B]
            // (A <= B; the same difference as A - y or y - B, so the same
            // rounding)
            const float tx = p.x - __builtin_amdgcn_fmed3f(p.x, Ax, Bx);
            const float ty = p.y - __builtin_amdgcn_fmed3f(p.y, Ay, By);
            const float tz = p.z - __builtin_amdgcn_fmed3f(p.z, Az, Bz);
            const float d2 = fmaf(tx, tx, fmaf(ty, ty, tz * tz));
            cut |= (v < nv) & !(d2 * (1.0f - kSlack) > S->vr2[v] + dw4);
        }
        return bounded & !gany(cut);
    }

    // ---------------------------------------------------------- planes
    // Planes referenced by some vertex (group-uniform mask of P bits).
    __device__ __forceinline__ uint64_t used_planes() const {
        uint64_t u = 0;
#pragma unroll
        for (int k = 0; k < kRows; ++k) {
            if (gl + G * k < nv) u |= planes_of(S->vtri[gl + G * k]);
        }
        return gor64(u);
    }
    __device__ __forceinline__ static uint64_t planes_of(uint32_t t) {
        return (1ull << tri_get<kB>(t, 0)) | (1ull << tri_get<kB>(t, 1)) | (1ull << tri_get<kB>(t, 2));
    }

    // a triple renumbered: each plane's new index is the count of used planes below it
    __device__ __forceinline__ static uint32_t renumber(uint64_t used, uint32_t t) {
        auto rank = [&](int e) { return (uint32_t)__popcll(used & ((1ull << tri_get<kB>(t, e)) - 1ull)); };
        return tri_pack<kB>(rank(0), rank(1), rank(2));
    }

    // Drops unreferenced planes and renumbers the vertex triples (the planes
    // of a recorded test's vertex stay, renumbered too, until the record is
    // written out with the cell).
    __device__ __forceinline__ void garbage_collect() {
        uint64_t used = used_planes();
        const uint32_t nt = S->ntent;
        for (uint32_t i = 0; i < nt; ++i) used |= planes_of(S->tent[i][0]);
#pragma unroll
        for (int k = 0; k < kPRows; ++k) {
            const int p = gl + G * k;
            const bool mv = p < np && ((used >> p) & 1ull);
            float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
            int o = 0;
            if (mv) {
                a = S->pl[p];
                o = S->own[p];
            }
            // every lane has read slot p before any lane writes a slot below
            // G (k + 1): all later reads are at or above that
            lds_fence();
            if (mv) {
                const int dst = __popcll(used & ((1ull << p) - 1ull));
                S->pl[dst] = a;
                S->own[dst] = o;
            }
        }
#pragma unroll
        for (int k = 0; k < kRows; ++k)
            if (gl + G * k < nv) S->vtri[gl + G * k] = renumber(used, S->vtri[gl + G * k]);
        if ((uint32_t)gl < nt) S->tent[gl][0] = renumber(used, S->tent[gl][0]);
        lds_fence();
        np = __popcll(used);
    }

    __device__ __forceinline__ bool has_plane(int owner) const {
        if (!(bloom & bloom_bit((uint32_t)owner))) return false;
        bool hit = false;
#pragma unroll
        for (int k = 0; k < kPRows; ++k) {
            const int p = gl + G * k;
            hit |= p < np && S->own[p] == owner;
        }
        return gany(hit);
    }

    __device__ __forceinline__ void empty_cell() {
        status = kEmptyCell;
        nv = 0;
    }

    // ---------------------------------------------------------- clipping
    // Offers the plane q (a, H) of point `owner` (group-uniform).  Returns
    // true when the cell changed.
    __device__ __forceinline__ bool clip(const float4 &q, int owner) {
        // Is vertex v strictly beyond the plane?  Filter: the error of
        // a~ . y~ - H~ against a . y - H is at most
        // |a|_1 eps + 2e-6 (sum |a_k y_k| + pH); with the stored w,
        // |a|_1 w + 2e-6 pH + tiny bounds the error of the FMA chain below.
        // A test inside that bound is undecided: it is taken by the sign of the
        // FP32 value and recorded; a pass after this tier decides it in FP64 and
        // sends the cell to the FP64-capable tiers if the sign was wrong.
        const float pa1 = fabsf(q.x) + fabsf(q.y) + fabsf(q.z);
        const float c2 = fmaf(kG32, plane_perm(q), kTiny32);
        // the removed vertices: bit v of the pair (the group's four rows; a
        // flag per row and lane instead is packed into bytes and unpacked:
        // 1.4% of the kernel, with the edges' places below from three ballots)
        uint32_t rem0 = 0u, rem1 = 0u;
        auto mine = [&](int k) { return (((k < 2 ? rem0 : rem1) >> (gl + 16 * (k & 1))) & 1u) != 0u; };
        bool open = false;
#pragma unroll
        for (int k = 0; k < kRows; ++k) {
            if (__ballot(nv > G * k) == 0ull) break;
            const float4 p = S->vpos[gl + G * k];
            const float Pv = fmaf(q.x, p.x, fmaf(q.y, p.y, fmaf(q.z, p.z, -q.w)));
            const float err = fmaf(pa1, p.w, c2);
            const bool in = gl + G * k < nv;
            const uint32_t bits = gballot(in & (Pv > 0.0f));  // (of a decided test; of an open one its FP32 sign)
            if (k < 2) rem0 |= bits << (16 * (k & 1));
            else rem1 |= bits << (16 * (k & 1));
            open |= in & !(fabsf(Pv) > err);
        }
        if (gany(open)) {  // (rare)
            uint32_t unsure = 0;
#pragma unroll
            for (int k = 0; k < kRows; ++k) {
                const float4 p = S->vpos[gl + G * k];
                const float Pv = fmaf(q.x, p.x, fmaf(q.y, p.y, fmaf(q.z, p.z, -q.w)));
                if (gl + G * k < nv && !(fabsf(Pv) > fmaf(pa1, p.w, c2))) unsure |= 1u << k;
            }
            const uint32_t n0 = S->ntent;
            int tot;
            uint32_t r = n0 + (uint32_t)gexcl(__popc(unsure), tot);
            if (n0 + (uint32_t)tot > (uint32_t)kTentMax) {
                overflow = true;
                bail = 1u;
                return false;
            }
#pragma unroll
            for (int k = 0; k < kRows; ++k) {
                if ((unsure >> k) & 1u) {
                    S->tent[r][0] = S->vtri[gl + G * k];
                    S->tent[r][1] = (uint32_t)owner | (mine(k) ? 0x80000000u : 0u);
                    ++r;
                }
            }
            S->ntent = n0 + (uint32_t)tot;
            lds_fence();
        }
        const int R = __popc(rem0) + __popc(rem1);
        if (R == 0) return false;  // the plane does not cut
        // listed in tmp[0, R) in slot order
#pragma unroll
        for (int k = 0; k < kRows; ++k) {
            if (__ballot(nv > G * k) == 0ull) break;
            if (mine(k)) {
                const int v = gl + G * k;
                const uint32_t lower = k & 1 ? ~(0xFFFF0000u << gl) : (1u << gl) - 1u;
                const int at = k < 2 ? __popc(rem0 & lower) : __popc(rem0) + __popc(rem1 & lower);
                S->tmp[at] = S->vtri[v] | ((uint32_t)v << kSlotShift);
            }
        }
        if (R == nv) {  // voronoi_convex_cell.cuh:430-435
            empty_cell();
            return true;
        }
        if (np >= P) {
            lds_fence();  // (the list; a lane stores to entries that others wrote)
            garbage_collect();
            if (np >= P) {
                overflow = true;
                return false;
            }
#pragma unroll
            for (int k = 0; k < kRows; ++k) {  // the listed triples were renumbered
                if (gl + G * k < R) {
                    const uint32_t v = S->tmp[gl + G * k] >> kSlotShift;
                    S->tmp[gl + G * k] = S->vtri[v] | (v << kSlotShift);
                }
            }
        }
        const int qs = np++;
        if (gl == 0) {
            S->pl[qs] = q;
            S->own[qs] = owner;
        }
        lds_fence();  // the list and the new plane
        if (in_guess) bloom |= bloom_bit((uint32_t)owner);
        // Boundary of the removed triangles: directed edges whose twin is not
        // removed.  Its nb edges are compacted into tmp[0, nb).
        int nb;
        int cycle = 0;  // every plane of the boundary cycle starts one edge and ends one
        uint32_t my_slot = 0u;  // (R <= G) slot of the gl-th removed vertex
        const bool spread = R <= G;
        if (spread) {
            // one removed triangle per lane, each lane checks its three edges
            // against all of them
            const bool has_tri = gl < R;
            uint32_t tr = 0u;
            if (has_tri) {
                const uint32_t w = S->tmp[gl];
                tr = w & 0xFFFFFFu;
                my_slot = w >> kSlotShift;
            }
            const uint32_t t0 = tri_get<kB>(tr, 0), t1 = tri_get<kB>(tr, 1), t2 = tri_get<kB>(tr, 2);
            bool tw0 = false, tw1 = false, tw2 = false;
            // The dual of a cell is a triangulated sphere: a pair of planes
            // lies in at most two triangles, which then share it as an edge.
            // So the twin of edge (x, y) is removed iff another removed
            // triangle holds both x and y: per plane, OR in the lanes whose
            // removed triangle holds it, intersect, and clear the words again.
            {
                const uint32_t bit = 1u << gl;
                const uint32_t s0 = (t0 & 1u) << 4, s1 = (t1 & 1u) << 4, s2 = (t2 & 1u) << 4;
                uint32_t *w0 = &S->pm[t0 >> 1], *w1 = &S->pm[t1 >> 1], *w2 = &S->pm[t2 >> 1];
                if (has_tri) {
                    atomicOr(w0, bit << s0);
                    atomicOr(w1, bit << s1);
                    atomicOr(w2, bit << s2);
                }
                lds_fence();
                if (has_tri) {
                    const uint32_t m0 = *w0 >> s0, m1 = *w1 >> s1, m2 = *w2 >> s2;
                    const uint32_t others = 0xFFFFu & ~bit;
                    tw0 = (m0 & m1 & others) != 0u;
                    tw1 = (m1 & m2 & others) != 0u;
                    tw2 = (m2 & m0 & others) != 0u;
                }
                lds_fence();
                if (has_tri) {
                    *w0 = 0u;
                    *w1 = 0u;
                    *w2 = 0u;
                }
            }
            const bool e0 = has_tri & !tw0, e1 = has_tri & !tw1, e2 = has_tri & !tw2;
            int j = gexcl((int)e0 + (int)e1 + (int)e2, nb);
            const int x0 = (int)(t0 * t0), x1 = (int)(t1 * t1), x2 = (int)(t2 * t2);
            cycle = (e0 ? x0 - x1 : 0) + (e1 ? x1 - x2 : 0) + (e2 ? x2 - x0 : 0);
            // (every lane has read its triangle above)
            if (e0) S->tmp[j] = t0 | (t1 << kB);
            j += (int)e0;
            if (e1) S->tmp[j] = t1 | (t2 << kB);
            j += (int)e1;
            if (e2) S->tmp[j] = t2 | (t0 << kB);
        } else {
            // clips that remove more triangles than the group has lanes: each
            // lane walks its own removed rows; an edge keeps the slot listed
            // in its word
            uint32_t emask = 0;
            boundary_rows(rem0, rem1, R, emask, cycle);
            lds_fence();  // (every lane has read the list)
            int j = gexcl(__popc(emask), nb);
            // (a removed set of R triangles without gaps has at most R + 2
            // boundary edges; more than tmp holds are never written)
            while (emask && j < V) {
                const int bit = (int)__builtin_ctz(emask);
                emask &= emask - 1u;
                const int k = bit / 3, e = bit - 3 * k;
                const uint32_t t = S->vtri[gl + G * k];
                const uint32_t slot = j < R ? S->tmp[j] >> kSlotShift : 0u;
                S->tmp[j++] = tri_get<kB>(t, e) | (tri_get<kB>(t, e == 2 ? 0 : e + 1) << kB) | (slot << kSlotShift);
            }
        }
        if (nb < 3 || row_sum(cycle) != 0) {
            status = kInconsistentBoundary;
            // (after a test taken by its FP32 sign the cell is rebuilt instead)
            if (gl == 0 && S->ntent == 0u) count(kStatInconsistent);
            return true;
        }
        const int kept = nv - R;
        if (kept + nb > V) {
            overflow = true;
            return false;
        }
        lds_fence();  // the edges
        // One new vertex (q, x, y) per boundary edge: the first R take the
        // removed ones' slots, the others follow the last vertex.
        bool bad = false;
        for (int e = gl; e < nb; e += G) {
            const uint32_t ed = S->tmp[e];
            const int slot = e >= R ? kept + e : (spread ? (int)my_slot : (int)(ed >> kSlotShift));
            bad |= !make_vertex(slot, (uint32_t)qs, ed & kBMask, (ed >> kB) & kBMask);
        }
        if (__ballot(nb < R) != 0ull) {
            // fewer new than removed: the last vertices move into the slots
            // left over (those of the removed list from nb on, in order)
            if (spread && gl >= nb && gl < R) S->tmp[gl] = my_slot;
            lds_fence();
            int m = nb;
#pragma unroll
            for (int k = 0; k < kRows; ++k) {
                const int v = gl + G * k;
                const bool mv = nb < R && v >= kept + nb && v < nv && !mine(k);
                const uint32_t bits = gballot(mv);
                if (mv) {
                    const uint32_t w = S->tmp[m + grank(bits)];
                    const int dst = (int)(spread ? w : w >> kSlotShift);
                    S->vpos[dst] = S->vpos[v];
                    S->vr2[dst] = S->vr2[v];
                    S->vtri[dst] = S->vtri[v];
                }
                m += __popc(bits);
            }
        }
        lds_fence();  // the vertices
        nv = kept + nb;
        if (gany(bad)) {
            overflow = true;
            bail = 2u;
            return false;
        }
        dirty = true;
        return true;
    }

    // Boundary edges of the lane's own removed rows: bit 3k + e of emask marks
    // edge e of row k.
    __device__ __forceinline__ void boundary_rows(uint32_t rem0, uint32_t rem1, int R, uint32_t &emask,
                                                  int &cycle) const {
#pragma unroll
        for (int k = 0; k < kRows; ++k) {
            if ((((k < 2 ? rem0 : rem1) >> (gl + 16 * (k & 1))) & 1u) == 0u) continue;
            const uint32_t t = S->vtri[gl + G * k];
            const uint32_t t0 = tri_get<kB>(t, 0), t1 = tri_get<kB>(t, 1), t2 = tri_get<kB>(t, 2);
            bool tw0 = false, tw1 = false, tw2 = false;
            for (int u = 0; u < R; ++u) {
                const uint32_t o = S->tmp[u];
                tw0 |= tri_has_edge<kB>(o, t1, t0);
                tw1 |= tri_has_edge<kB>(o, t2, t1);
                tw2 |= tri_has_edge<kB>(o, t0, t2);
            }
            const int x0 = (int)(t0 * t0), x1 = (int)(t1 * t1), x2 = (int)(t2 * t2);
            cycle += (tw0 ? 0 : x0 - x1) + (tw1 ? 0 : x1 - x2) + (tw2 ? 0 : x2 - x0);
            emask |= ((tw0 ? 0u : 1u) | (tw1 ? 0u : 2u) | (tw2 ? 0u : 4u)) << (3 * k);
        }
    }

    // ---------------------------------------------------------- candidates
    // Prepares the lane's candidate j (its plane); false when it cannot cut
    // the cell.  maybe_guess: j may be one of the guesses already offered
    // (only those can already own a plane of the cell): every guess lies
    // within the guess radius, up to the few ulps that its 3e-5 widening covers.
    __device__ __forceinline__ bool prepare(uint32_t j, float4 &c, bool &emptied, bool &maybe_guess) const {
        const float4 p = pts[j];
        c.x = p.x - sx;
        c.y = p.y - sy;
        c.z = p.z - sz;
        const float dw = p.w - sw;
        if (c.x == 0.0f && c.y == 0.0f && c.z == 0.0f) {
            emptied = dw > 0.0f;  // coincident point: half-space empty iff w_p > w_s
            return false;
        }
        const float a2 = c.x * c.x + c.y * c.y + c.z * c.z;
        if (a2 < guess_r2) return false;  // offered by the pre-clip; the cell has only shrunk since
        maybe_guess = guess_r2 == 0.0f || a2 < guess_r2 * 1.00003f;
        c.w = a2 - dw;
        return !too_far(c, a2 + fabsf(dw));
    }

    // May the plane of the lane's own candidate cut the cell: is some vertex
    // not certainly behind it (the test of clip(), so a candidate refused
    // here would be refused vertex by vertex there)?  The vertices are read
    // in order, each by the whole group at once.
    __device__ __forceinline__ bool may_cut(const float4 &c) const {
        const float pa1 = fabsf(c.x) + fabsf(c.y) + fabsf(c.z);
        const float c2 = fmaf(kG32, plane_perm(c), kTiny32);
        bool hit = false;
#pragma unroll 1
        for (int v = 0; v < V; v += 4) {
            if (__ballot(nv > v) == 0ull) break;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const float4 p = S->vpos[v + u];
                const float Pv = fmaf(c.x, p.x, fmaf(c.y, p.y, fmaf(c.z, p.z, -c.w)));
                hit |= (v + u < nv) & !(Pv < -fmaf(pa1, p.w, c2));
            }
        }
        return hit;
    }

    // Offers a batch of up to G candidates (lane-specific j when `has`).
    __device__ __forceinline__ void offer_batch(bool has, uint32_t j) {
        float4 c = make_float4(0.f, 0.f, 0.f, 0.f);
        bool emptied = false, maybe_guess = true;
        bool live_c = has && prepare(j, c, emptied, maybe_guess);
        if (gany(emptied)) {
            empty_cell();
            return;
        }
        uint32_t todo = gballot(live_c);
        const uint32_t skipped = gballot(has) & ~todo;
        if (gl == 0) {
            if (skipped) count(kStatSkipped, (uint32_t)__popc(skipped));
            if (todo) count(kStatCandidates, (uint32_t)__popc(todo));
        }
        if (!todo) return;
        // Every vertex against the lane's own candidate: one that lies
        // certainly behind all of them does not cut (the cell only shrinks
        // after this), so only the others are offered one at a time.
        // Nothing to gain on the initial box, which every guess cuts.
        if (np > 6) {
            const bool cuts = may_cut(c);  // (by all lanes of the group)
            live_c = live_c && cuts;
            todo = gballot(live_c);
            if (!todo) return;
        }
        // the owner's sign bit marks a candidate that may already own a plane
        if (live_c) {
            S->cand[gl] = c;
            S->cown[gl] = (int)(maybe_guess ? (j | 0x80000000u) : j);
        }
        lds_fence();
        float hkey = live_c ? c.w : FLT_MAX;
        while (todo) {
            // nearest plane first (smallest H = power distance of the point):
            // the cell shrinks fastest and fewer clips are undone later
            const float hmin = row_min(hkey);
            const uint32_t at = gballot(live_c && hkey == hmin) & todo;
            const int b = (int)__builtin_ctz(at ? at : todo);
            todo &= ~(1u << b);
            if (gl == b) hkey = FLT_MAX;
            const float4 q = S->cand[b];
            const int ow = S->cown[b];
            const int owner = ow & INT32_MAX;
            if (ow < 0 && bloom && has_plane(owner)) continue;
            if (clip(q, owner)) {
                if (gl == 0) count(kStatClips);
                if (status != kSuccess) return;
            } else if (overflow) {
                return;
            }
        }
        lds_fence();  // (the next batch is staged in the same place)
        if (dirty) {
            update_bounds();
            dirty = false;
        }
    }

    // Box plane `code` (2 axis + side) of the cell of seed point sp.  (A
    // lane-dependent choice among the members sx, sy, sz would be compiled
    // into a choice of addresses, moving them to scratch.)
    __device__ __forceinline__ float4 box_plane(int code, const float4 &sp) const {
        const int axis = code >> 1, side = code & 1;
        const float s = axis == 0 ? sp.x : (axis == 1 ? sp.y : sp.z);
        const float sg = side ? 1.0f : -1.0f;
        return make_float4(axis == 0 ? sg : 0.0f, axis == 1 ? sg : 0.0f, axis == 2 ? sg : 0.0f,
                           side ? 2.0f * (hdr->box_hi[axis] - s) : 2.0f * (s - hdr->box_lo[axis]));
    }

    // The initial cell: the box, or (cube_h > 0, a predicted half-width in
    // doubled coordinates) the box cut by the cube |y_k| <= cube_h, whose
    // planes carry owner codes -7..-12 and are written as bisectors of equal
    // weights (a = cube_h e_k, H = cube_h^2; see plane_perm).  A cell whose
    // final vertices touch a cube plane, or that empties, is rebuilt without
    // the cube.
    __device__ __forceinline__ void init_box(float cube_h = 0.0f) {
        bool from_cube = false;
        if (gl < 6) {
            float4 pl = box_plane(gl, pts[seed]);
            // (a cube so small that the products of three of its planes
            // leave the range of the filter is not used)
            from_cube = cube_h > 1e-8f && cube_h < pl.w;
            if (from_cube) pl = make_float4(pl.x * cube_h, pl.y * cube_h, pl.z * cube_h, cube_h * cube_h);
            S->pl[gl] = pl;
            S->own[gl] = (from_cube ? -7 : -1) - gl;
        }
        lds_fence();
        cube = gany(from_cube);
        np = 6;
        nv = 8;
        // the 8 corners go to slots 0..7 (lanes 0..7 of row 0)
        if (gl < 8) {
            const int cx = gl >> 2 & 1, cy = gl >> 1 & 1, cz = gl & 1;
            const uint32_t X = cx, Y = 2 + cy, Z = 4 + cz;
            const int sgn = (cx ? 1 : -1) * (cy ? 1 : -1) * (cz ? 1 : -1);
            // box corners: D = +- pD, always resolved in FP32
            if (sgn > 0) make_vertex(gl, X, Y, Z);
            else make_vertex(gl, X, Z, Y);
        }
        lds_fence();
        bloom = 0;
        update_bounds();
        dirty = false;
    }

    // ---------------------------------------------------------- traversal
    // Stack of partly visited nodes: entry t (node reference, mask of the
    // children left) sits in word t / 16 of lane t % 16.
    __device__ __forceinline__ void push(bool doit, int t, uint32_t node, uint32_t left) {
        const bool me = doit & (gl == (t & (G - 1)));
        const int sl = t / G;
#pragma unroll
        for (int j = 0; j < kStack / G; ++j) {
            stk_node[j] = (me & (j == sl)) ? node : stk_node[j];
            stk_left[j] = (me & (j == sl)) ? left : stk_left[j];
        }
    }
    __device__ __forceinline__ void pop(int t, uint32_t &node, uint32_t &left) const {
        const int sl = t / G;
        uint32_t a = stk_node[0], b = stk_left[0];
#pragma unroll
        for (int j = 1; j < kStack / G; ++j) {
            a = j == sl ? stk_node[j] : a;
            b = j == sl ? stk_left[j] : b;
        }
        node = (uint32_t)gbi((int)a, t & (G - 1));
        left = (uint32_t)gbi((int)b, t & (G - 1));
    }

    // Builds cell `cell`: the initial polytope, clipped by its guesses and by
    // the points of the hierarchy that may cut it.
    //
    // Each cell walks the 16-wide hierarchy on its own, depth first, one lane
    // per child: a node's children are tested against the cell's box on arrival
    // (and again, those left, when the walk comes back from below), then taken
    // by the smallest lower bound of H, each after a test against the vertices
    // that the cell has by then.  The groups of a wave step
    // until each has a leaf to offer or has ended, and offer their batches
    // together, so the candidates and clips of the four cells share their
    // instructions.  The reference pops the smallest key from a list instead
    // (voronoi_bvh.cuh:246-283); after the pre-clip the order changes little
    // of the work, and the diagram does not depend on it.  There is one call
    // of offer_batch() for guesses and leaves: a copy of the clip for each
    // would not fit the instruction cache.
    __device__ __forceinline__ void build(uint32_t cell, const CellParams *sprm) {
        bool guesses = false;       // the current source: the guesses, then the hierarchy
        int o = 0, n = 0;           // batch position and size of the current source or leaf
        uint32_t base = 0u;         // first point of the leaf
        uint32_t node = 0u;         // current node and its children left
        uint32_t left = 0u;
        bool fresh = true;          // key, ref and box are those of the node's children
        float key = FLT_MAX;        // the lane's child: bound, reference and box
        uint32_t ref = kWideNone;
        float4 lo = make_float4(0.f, 0.f, 0.f, 0.f), hi = lo;
        int sz = 0;
        uint32_t n_nodes = 0u, n_leaves = 0u;
        if (active) {
            const CellParams &prm = *reread(sprm);
            begin(cell, prm);
            guesses = true;
            n = first_count(prm);
        }
        bool go = active;
        while (true) {
            if (go && guesses && o >= n) {  // all offered: the hierarchy next
                guesses = false;
                in_guess = false;
                guess_r2 = first_radius2(*reread(sprm));
                o = 0;
                n = 0;
                node = root;
                left = 0xFFFFu;
                fresh = false;
                if (is_leaf(root)) {
                    n_leaves = 1u;
                    base = leaf_first(root);
                    n = (int)leaf_count(root);
                    left = 0u;
                }
            }
            // The wave steps as one, without branches but for the loads: the
            // many values that a step may change would be copied at each
            // join of divergent paths.
            bool walk = go && o >= n;
            while (__ballot(walk) != 0ull) {
                const bool arrive = walk && !fresh;
                if (arrive) {
                    // the children left against the cell's AABB
                    const bool binary = (node & kWideBinary) != 0u;
                    const float4 *box = binary ? (const float4 *)&nodes[node & ~kWideBinary] + 2 * (gl & 1)
                                               : (const float4 *)&wide[16u * node + (uint32_t)gl];
                    lo = box[0], hi = box[1];
                    ref = __float_as_uint(hi.w);
                    if (binary) ref = gl < 2 ? (is_leaf(ref) ? ref : ref | kWideBinary) : kWideNone;
                    const bool clear = octant_clear(lo, hi, key);
                    const bool need = ((left >> gl) & 1u) & (ref != kWideNone) & !clear;
                    left = gballot(need);
                    key = need ? key : FLT_MAX;
                    n_nodes++;
                }
                fresh = true;
                // the nearest child left that every vertex of the cell, as it
                // is now, does not rule out
                bool look = walk & (left != 0u), visit = false;
                uint32_t r = 0u;
                while (__ballot(look) != 0ull) {
                    const float kmin = row_min(key);
                    const uint32_t at = gballot(key == kmin) & left;
                    const int c = (int)__builtin_ctz((at ? at : left) | 0x10000u) & (G - 1);
                    const uint32_t rc = (uint32_t)gbi((int)ref, c);
                    const float4 clo = make_float4(gbf(lo.x, c), gbf(lo.y, c), gbf(lo.z, c), gbf(lo.w, c));
                    const float4 chi = make_float4(gbf(hi.x, c), gbf(hi.y, c), gbf(hi.z, c), 0.0f);
                    const bool pass = !balls_clear(clo, chi);
                    left = look ? left & ~(1u << c) : left;
                    key = (look & (gl == c)) ? FLT_MAX : key;
                    r = (look & pass) ? rc : r;
                    visit |= look & pass;
                    look &= !pass & (left != 0u);
                }
                const bool leaf = visit & is_leaf(r), down = visit & !is_leaf(r);
                const bool back = walk & !visit;  // nothing left here: the last node with children left
                const bool keep = down & (left != 0u);
                const bool full = keep & (sz >= kStack);
                const bool end = back & (sz == 0);
                uint32_t up_node, up_left;
                pop(sz > 0 ? sz - 1 : 0, up_node, up_left);
                push(keep, sz, node, left);
                sz += keep ? 1 : ((back & !end) ? -1 : 0);
                node = down ? r : ((back & !end) ? up_node : node);
                left = down ? 0xFFFFu : ((back & !end) ? up_left : left);
                fresh = !(down | back);
                base = leaf ? leaf_first(r) : base;
                n = leaf ? (int)leaf_count(r) : n;
                o = leaf ? 0 : o;
                n_leaves += leaf ? 1u : 0u;
                overflow |= full;
                go &= !(end | full);
                walk &= !(leaf | end | full);
            }
            if (__ballot(go) == 0ull) break;
            if (go) {
                uint32_t j = 0;
                bool has = false;
                if (guesses) {
                    has = first_point(*reread(sprm), o + gl, n, j);
                } else {
                    j = base + (uint32_t)(o + gl);
                    has = o + gl < n && j != seed;
                }
                o += G;
                offer_batch(has, j);
                go = live() && (guesses || o < n || left != 0u || sz > 0);
            }
        }
        if (active && gl == 0) {
            count(kStatNodes, n_nodes);
            count(kStatLeaves, n_leaves);
        }
    }

    // The cell's seed and its initial polytope (the box, or the predicted cube).
    __device__ __forceinline__ void begin(uint32_t cell, const CellParams &prm) {
        seed = cell;
        S->ntent = 0u;
        const float4 s = pts[cell];
        sx = s.x, sy = s.y, sz = s.z, sw = s.w;
        status = kSuccess;
        overflow = false;
        bail = 0u;
        init_box(prm.init_h ? 2.0f * prm.init_h[prm.perm[cell]] : 0.0f);
        in_guess = true;
        guess_r2 = 0.0f;
    }

    // The points the cell is clipped by first: its guesses (rows by original
    // id, or Morton-ordered rows of sorted ids, the library's own kNN
    // pre-clip), or its Morton neighbours (the cheap analogue of clipping by
    // the k nearest neighbours, voronoi_ultra.cu:70-85; the order does not
    // change the result, only how fast the cell shrinks).
    __device__ __forceinline__ int first_count(const CellParams &prm) const {
        if (!prm.guesses) return prm.seed_window;
        if (prm.guess_stride > 0) return prm.guess_stride;
        const uint32_t orig = prm.perm[seed];
        return prm.guess_offsets[orig + 1] - prm.guess_offsets[orig];
    }
    // The i-th of them (of n); false when there is none.
    __device__ __forceinline__ bool first_point(const CellParams &prm, int i, int n, uint32_t &j) const {
        j = 0;
        if (i >= n) return false;
        if (!prm.guesses) {
            const int64_t t = (int64_t)seed - n / 2 + i + (i >= n / 2 ? 1 : 0);
            j = (uint32_t)(t < 0 ? 0 : t);
            return t >= 0 && t < prm.n;
        }
        const int64_t at = prm.guess_stride > 0 ? (int64_t)seed * prm.guess_stride
                                                : (int64_t)prm.guess_offsets[prm.perm[seed]];
        const int32_t gid = prm.guesses[at + i];
        if (gid < 0 || (int64_t)gid >= prm.n) return false;  // voronoi_ultra.cu:76-78 skips negative ids
        j = (prm.guess_stride > 0 || prm.guesses_sorted) ? (uint32_t)gid : prm.inv[gid];
        return j != seed;
    }
    // The row holds the guess_stride nearest points (kNN order, ties and
    // all); a point off the row has squared distance >= the row's last, up to
    // the few ulps of the two FP32 evaluations of |p - s|^2, which the 1e-5
    // relative margin covers.
    __device__ __forceinline__ float first_radius2(const CellParams &prm) const {
        return prm.guesses && prm.guess_stride > 0 && prm.guess_d2 ? prm.guess_d2[seed] * (1.0f - 1e-5f) : 0.0f;
    }

    // ---------------------------------------------------------- output
    // Row = sorted original ids of the owners of referenced planes
    // (voronoi_ultra.cu:125-138).  stage_row() returns the row length F
    // (group-uniform; the ids are staged unsorted in tmp[0, F)), the caller
    // takes F entries of the row pool, and write_row() writes the sorted row
    // there.  With duplicate points a row also holds every exact duplicate of
    // an owner (a second copy of a plane removes no vertex, so at most one
    // plane per group of duplicates is referenced); lane 0 builds such rows.
    __device__ __forceinline__ int stage_row(const CellParams &prm) const {
        if (status == kEmptyCell) return 0;
        const uint64_t used = used_planes();
        if (hdr->has_duplicates != 0u) {
            int F = 0;
            if (gl == 0) {
                for (int p = 0; p < np; ++p) {
                    if (!((used >> p) & 1ull)) continue;
                    const int owner = S->own[p];
                    if (owner < 0) continue;
                    for (uint32_t m = prm.dup_head[owner]; m != 0xFFFFFFFFu; m = prm.dup_next[m]) F++;
                }
            }
            return gbi(F, 0);
        }
        int32_t ids[kPRows];
        int mine = 0;
#pragma unroll
        for (int k = 0; k < kPRows; ++k) {
            const int p = gl + G * k;
            ids[k] = -1;
            if (p < np && ((used >> p) & 1ull)) {
                const int owner = S->own[p];
                if (owner >= 0) {
                    ids[k] = (int32_t)prm.perm[owner];
                    mine++;
                }
            }
        }
        int F;
        int at = gexcl(mine, F);
#pragma unroll
        for (int k = 0; k < kPRows; ++k)
            if (ids[k] >= 0) S->tmp[at++] = (uint32_t)ids[k];
        lds_fence();
        return F;
    }

    // Writes the staged row (sorted) to row_out and the cell's count, status
    // and extent.
    __device__ __forceinline__ void write_row(const CellParams &prm, uint32_t orig, int32_t *row_out, int F) const {
        if (F > 0) {
            if (hdr->has_duplicates != 0u) {
                // insertion into the sorted row, dropping repeats
                int len = 0;
                const uint64_t used = used_planes();
                if (gl == 0) {
                    for (int p = 0; p < np; ++p) {
                        if (!((used >> p) & 1ull)) continue;
                        const int owner = S->own[p];
                        if (owner < 0) continue;
                        for (uint32_t m = prm.dup_head[owner]; m != 0xFFFFFFFFu; m = prm.dup_next[m]) {
                            const int32_t id = (int32_t)prm.perm[m];
                            int k = len;
                            while (k > 0 && row_out[k - 1] > id) k--;
                            if (k > 0 && row_out[k - 1] == id) continue;
                            if (len >= F) break;  // (F bounds the distinct ids)
                            for (int t = len; t > k; --t) row_out[t] = row_out[t - 1];
                            row_out[k] = id;
                            len++;
                        }
                    }
                }
                F = gbi(len, 0);
            } else {
                // rank of each id among the row (ids are distinct)
                for (int t = gl; t < F; t += G) {
                    const int32_t x = (int32_t)S->tmp[t];
                    int rank = 0;
                    for (int u = 0; u < F; ++u) rank += (int32_t)S->tmp[u] < x;
                    row_out[rank] = x;
                }
            }
        }
        if (gl == 0) {
            prm.counts[orig] = F;
            prm.status[orig] = status;
            if (prm.extent)
                prm.extent[orig] = status == kEmptyCell ? 0.0f
                                                       : 0.5f * fmaxf(fmaxf(fmaxf(-L_[0], U_[0]), fmaxf(-L_[1], U_[1])),
                                                                      fmaxf(-L_[2], U_[2]));
        }
    }

    // Does a final vertex lie on a plane of the predicted cube (group op)?
    __device__ __forceinline__ bool cube_touched() const {
        const uint64_t used = used_planes();
        bool hit = false;
#pragma unroll
        for (int k = 0; k < kPRows; ++k) {
            const int p = gl + G * k;
            if (p < np && ((used >> p) & 1ull)) hit |= S->own[p] <= -7;
        }
        return gany(hit);
    }

    // The owners of the planes held, in plane order (point ids in the index's
    // order, negative for the box planes, -1 past them), for the large tier
    // (group op).
    __device__ __forceinline__ void store_owners(int32_t *out) const {
#pragma unroll
        for (int k = 0; k < kPRows; ++k) {
            const int p = gl + G * k;
            if (p < kPromoPlanes) out[p] = p < np ? S->own[p] : -1;
        }
    }

    __device__ __forceinline__ void setup(const CellParams &prm, LDS *s, uint32_t *counters) {
        const int lane = threadIdx.x & (kWave - 1);
        S = s;
        ctr = counters;
#pragma unroll
        for (int j = 0; j < kStack / G; ++j) stk_node[j] = stk_left[j] = 0u;
        gl = lane & (G - 1);
        lane64 = lane;
        pts = prm.pts;
        nodes = prm.nodes;
        wide = prm.wide;
        if (prm.clouds == nullptr) set_cloud(prm.hdr, wide_ref((uint32_t)prm.n, 0u, (uint32_t)prm.n));
        if (lane < kNumCtr) ctr[lane] = 0u;
        for (int w = gl; w < (int)(sizeof(S->pm) / 4); w += G) S->pm[w] = 0u;
    }

    // The cloud the next cells belong to: its clipping box and wide form.
    __device__ __forceinline__ void set_cloud(const IndexHeader *h, uint32_t r) {
        hdr = h;
        root = r;
    }

    // Adds the wave's counters to the launch's (cells: every lane's count).
    __device__ __forceinline__ void flush(const CellParams &prm, uint32_t cells) const {
        lds_fence();
        const uint32_t total = wave_sum(cells);
        if (lane64 < kNumCtr) {
            const uint32_t s = lane64 == kStatCells ? total : ctr[lane64];
            if (s) atomicAdd(&prm.stats[ctr_stat_slot(lane64)], (unsigned long long)s);
        }
    }
};

// Tier 0's waves take Morton-consecutive quads of cells from a global
// counter (a batch's quads each lie in one cloud; kSmall: cells_per_wave cells
// of one cloud, see launch_cells).  A cell the tier gives up
// on (`bail`) is flagged, one that outgrows it queued, for tier m.
template <bool kSmall>
__device__ __forceinline__ void tier0_body(const CellParams &prm) {
    constexpr int kCellsPerWave = kWave / kT0Lanes;
    __shared__ Tier0::LDS lds[kT0Threads / kT0Lanes];
    __shared__ uint32_t ctrs[kT0Threads / kWave][kNumCtr];
    __shared__ CellParams sprm;
    // each wave's unused part of the row pool: next entry and entries left
    __shared__ unsigned long long chunk_at[kT0Threads / kWave];
    __shared__ uint32_t chunk_left[kT0Threads / kWave];
    if (threadIdx.x == 0) sprm = prm;
    if (threadIdx.x < kT0Threads / kWave) {
        chunk_at[threadIdx.x] = 0ull;
        chunk_left[threadIdx.x] = 0u;
    }
    __syncthreads();
    const int lane = threadIdx.x & (kWave - 1);
    const int grp = lane / kT0Lanes;
    Tier0 g;
    g.setup(prm, &lds[(threadIdx.x / kWave) * kCellsPerWave + grp], ctrs[threadIdx.x / kWave]);
    uint32_t cells = 0;
    const int64_t count = prm.end - prm.begin;
    while (true) {
        uint32_t k = 0;
        if (lane == 0) k = atomicAdd(&prm.counters[0], 1u);
        const int64_t quad = (int64_t)uniform(k);
        int64_t c = kCellsPerWave * quad + grp, last = count;  // the group's cell, from prm.begin
        if (kSmall) {
            c = grp < prm.cells_per_wave ? prm.cells_per_wave * quad + grp : count;
            if (prm.cells_per_wave * quad >= count) break;
        } else if (prm.clouds == nullptr) {
            if (kCellsPerWave * quad >= count) break;
        } else {
            // a batch: the quad's cells share their cloud's subtree
            if (quad >= prm.quads[prm.n_clouds]) break;
            const int cl = uniform(batch_find(prm.quads, prm.n_clouds, quad));
            const int64_t a = prm.cloud_cells[cl], z = prm.cloud_cells[cl + 1];
            g.set_cloud(&prm.clouds[cl], wide_ref((uint32_t)prm.n, (uint32_t)a, (uint32_t)(z - a)));
            c = max(a, prm.begin) + kCellsPerWave * (quad - prm.quads[cl]) - prm.begin + grp;
            last = min(z, prm.end) - prm.begin;
        }
        const uint64_t t0 = clock64();
        const bool active = c < last;
        g.active = active;
        const uint32_t cell = (uint32_t)(prm.begin + (active ? c : 0));
        g.build(cell, &sprm);
        // the launch's fields read again rather than kept in registers across
        // the traversal
        const CellParams &P = *reread(&sprm);
        const uint32_t orig = P.perm[cell];
        // a cell built inside a predicted cube stands only if the cube cut nothing
        if (active && !g.overflow && g.cube && (g.status != kSuccess || g.cube_touched())) g.overflow = true, g.bail = 3u;
        // the removal tests taken by their FP32 sign go to the record for the
        // FP64 check after this tier, with the cell; a cell that ended
        // inconsistent after such a test, or that the record cannot hold, goes
        // to tier m instead
        const uint32_t nt = active && !g.overflow ? g.S->ntent : 0u;
        if (nt > 0u && g.status == kInconsistentBoundary) {
            g.overflow = true, g.bail = 1u;
        } else if (nt > 0u) {
            // (the base comes from the group's lane 0 through a shuffle: a
            // store and load of one LDS word by different lanes are not
            // ordered for the compiler)
            uint32_t base = 0u;
            if (g.gl == 0) base = atomicAdd(&P.counters[7], nt);
            base = (uint32_t)g.gbi((int)base, 0);
            const bool fits = (uint64_t)base + nt <= (uint64_t)P.tent_cap;
            if ((uint32_t)g.gl < nt && (uint64_t)base + g.gl < (uint64_t)P.tent_cap) {
                uint32_t *rec = P.tent + 5 * ((uint64_t)base + g.gl);
                const uint32_t t = g.S->tent[g.gl][0];
                rec[0] = fits ? cell : kNoCell;
                rec[1] = (uint32_t)g.S->own[tri_get<Tier0::kB>(t, 0)];
                rec[2] = (uint32_t)g.S->own[tri_get<Tier0::kB>(t, 1)];
                rec[3] = (uint32_t)g.S->own[tri_get<Tier0::kB>(t, 2)];
                rec[4] = g.S->tent[g.gl][1];
            }
            if (!fits) g.overflow = true, g.bail = 1u;
        }
        const bool emit = active && !g.overflow;
        const int F = emit ? g.stage_row(P) : 0;
        // the wave's four rows, back to back in the wave's current pool chunk
        // (whose position lives in LDS, not in registers across the traversal)
        const int f0 = rl(F, 0), f1 = rl(F, 16), f2 = rl(F, 32), f3 = rl(F, 48);
        const uint32_t need = (uint32_t)(f0 + f1 + f2 + f3);
        const int wv = threadIdx.x / kWave;
        uint32_t left = uniform(chunk_left[wv]);
        uint64_t at;
        if (need > left) {
            left = need > P.pool_chunk ? need : P.pool_chunk;
            at = pool_take(P, left);
        } else {
            const unsigned long long a = chunk_at[wv];
            at = ((uint64_t)uniform((uint32_t)(a >> 32)) << 32) | (uint64_t)uniform((uint32_t)a);
        }
        const uint64_t base = at + (uint64_t)(grp > 0 ? f0 : 0) + (uint64_t)(grp > 1 ? f1 : 0) +
                              (uint64_t)(grp > 2 ? f2 : 0);
        if (lane == 0) {
            chunk_at[wv] = at + need;
            chunk_left[wv] = left - need;
        }
        uint32_t slot = 0u;
        if (emit) {
            if (base + (uint64_t)F <= P.rows_elems) {
                if (g.gl == 0) P.row_offsets[cell] = (int64_t)base;
                g.write_row(P, orig, P.rows + base, F);
            } else if (g.gl == 0) {
                pool_short(P, cell, orig, base + (uint64_t)F);
            }
        } else if (active && g.gl == 0) {
            if (g.bail) {  // flag for tier m
                if (g.bail < 3u) g.count(g.bail == 1u ? kCtrBailTest : kCtrBailVertex);
                P.exact_list[c] = 1u;
                atomicAdd(&P.counters[5], 1u);
            } else {  // queue for tier m
                g.count(kStatPromoted);
                slot = atomicAdd(&P.counters[1], 1u);
                if (slot < P.queue_cap) P.mid_list[slot] = cell;
                else truncate_cell(P, orig);
            }
        }
        // with the promotion, the owners of the planes held (tier m starts
        // from them); the slot comes from the group's lane 0
        if (active && !emit && !g.bail) {
            slot = (uint32_t)g.gbi((int)slot, 0);
            if (slot < P.promo_cap) g.store_owners(P.promo + (size_t)slot * kPromoPlanes);
        }
        if (active && P.cycles && g.gl == 0) P.cycles[orig] = (uint32_t)min(clock64() - t0, (uint64_t)0x7fffffff);
        if (active && g.gl == 0) cells++;
    }
    g.flush(prm, cells);
}

__global__ void __launch_bounds__(kT0Threads) __attribute__((amdgpu_waves_per_eu(3, 3))) cell_group_kernel(const CellParams prm) {
    tier0_body<false>(prm);
}
// An instance of its own: the choice made in the kernel above costs it 0.7%.
__global__ void __launch_bounds__(kT0Threads) __attribute__((amdgpu_waves_per_eu(3, 3)))
cell_group_small_kernel(const CellParams prm) {
    tier0_body<true>(prm);
}

}  // namespace pg
