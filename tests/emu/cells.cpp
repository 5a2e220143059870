// The cell tiers of csrc/pg_cell.hip on the CPU: one group of lanes builds cell
// after cell, over a hierarchy of wide records made here.  Reads a request from
// stdin, writes rows and what else is asked for to stdout.
#include <float.h>
#include <math.h>
#include <stdio.h>
#include <stdlib.h>

#include <algorithm>
#include <vector>

#include "../../paragram_amd/csrc/pg_cell.hip"

namespace pg {
// (elsewhere in the library)
hipError_t fill_u32(uint32_t *, int64_t, uint32_t, hipStream_t) { return hipSuccess; }
}  // namespace pg

#include "rt.hpp"

using namespace pg;

namespace {

struct Request {
    int32_t n, tier, cells, stride, fanout, binary_below, seed, has_d2;
    int64_t limit;
};

void get(void *p, size_t bytes) {
    if (bytes && fread(p, 1, bytes, stdin) != bytes) {
        fprintf(stderr, "emulator: short request\n");
        exit(4);
    }
}
template <class T>
std::vector<T> get(size_t m) {
    std::vector<T> v(m);
    get(v.data(), m * sizeof(T));
    return v;
}

std::vector<float4> pts;
std::vector<Node> nodes;
std::vector<WideChild> wide;

void box_of(uint32_t a, uint32_t z, float4 &lo, float4 &hi) {
    lo = make_float4(FLT_MAX, FLT_MAX, FLT_MAX, -FLT_MAX);
    hi = make_float4(-FLT_MAX, -FLT_MAX, -FLT_MAX, 0.0f);
    for (uint32_t i = a; i < z; ++i) {
        const float4 p = pts[i];
        lo.x = fminf(lo.x, p.x), lo.y = fminf(lo.y, p.y), lo.z = fminf(lo.z, p.z), lo.w = fmaxf(lo.w, p.w);
        hi.x = fmaxf(hi.x, p.x), hi.y = fmaxf(hi.y, p.y), hi.z = fmaxf(hi.z, p.z);
    }
}
uint32_t binary_over(uint32_t a, uint32_t z) {
    if (z - a <= (uint32_t)kWideLeaf) return leaf_ref(a, z - a);
    const uint32_t at = (uint32_t)nodes.size(), m = (a + z) / 2;
    nodes.emplace_back();
    Node nd;
    box_of(a, m, nd.lo0, nd.hi0);
    box_of(m, z, nd.lo1, nd.hi1);
    const uint32_t r0 = binary_over(a, m), r1 = binary_over(m, z);
    nd.hi0.w = __uint_as_float(r0);
    nd.hi1.w = __uint_as_float(r1);
    nodes[at] = nd;
    return at;
}
// a wide record of up to `fanout` children; subtrees of fewer than `below` points are binary ones
uint32_t wide_over(uint32_t a, uint32_t z, uint32_t fanout, uint32_t below) {
    if (z - a <= (uint32_t)kWideLeaf) return leaf_ref(a, z - a);
    const uint32_t at = (uint32_t)(wide.size() / 16);
    wide.resize(wide.size() + 16);
    for (uint32_t c = 0; c < 16; ++c) {
        WideChild ch{};
        ch.hi.w = __uint_as_float(kWideNone);
        const uint32_t u = a + (uint32_t)((uint64_t)(z - a) * c / fanout), v = a + (uint32_t)((uint64_t)(z - a) * (c + 1) / fanout);
        if (c < fanout && v > u) {
            box_of(u, v, ch.lo, ch.hi);
            uint32_t r;
            if (v - u > (uint32_t)kWideLeaf && v - u < below) r = binary_over(u, v) | kWideBinary;
            else r = wide_over(u, v, fanout, below);
            ch.hi.w = __uint_as_float(r);
        }
        wide[16ull * at + c] = ch;
    }
    return at;
}

CellParams prm{};
std::vector<int32_t> cells;
std::vector<std::vector<int32_t>> rows, planes;
std::vector<int32_t> info;  // per cell: 1 kept, vertices, planes, status, open tests, clips
uint32_t root;
IndexHeader hdr{};

void fail(const char *what, int cell) {
    fprintf(stderr, "emulator: %s (cell %d)\n", what, cell);
    exit(5);
}

void put(bool kept, int nv, int np, int status, int open, int clips, int F, const int32_t *row, std::vector<int32_t> held) {
    for (int v : {kept ? 1 : 0, nv, np, status, open, clips}) info.push_back(v);
    rows.emplace_back(row, row + F);
    planes.push_back(std::move(held));
}

int32_t row_out[1 << 16];

Tier0::LDS lds0;
uint32_t ctr0[kNumCtr];
void body0(void *) {
    Tier0 g;
    g.setup(prm, &lds0, ctr0);
    g.set_cloud(&hdr, root);
    for (int32_t cell : cells) {
        g.active = true;
        const uint32_t before = ctr0[kStatClips];
        g.build((uint32_t)cell, &prm);
        if (g.nv < 0 || g.nv > Tier0::V || g.np < 0 || g.np > Tier0::P) fail("vertices or planes out of range", cell);
        const bool kept = !g.overflow;
        const int F = kept ? g.stage_row(prm) : 0;
        if (kept) g.write_row(prm, (uint32_t)cell, row_out, F);
        emu::fence();
        if (g.gl == 0) {
            for (uint32_t w : lds0.pm)
                if (w) fail("plane masks not cleared", cell);
            std::vector<int32_t> held;
            for (int p = 0; p < g.np; ++p) held.push_back(lds0.own[p]);
            put(kept, g.nv, g.np, g.status, (int)lds0.ntent, (int)(ctr0[kStatClips] - before), prm.counts[cell] * kept,
                row_out, held);
        }
        emu::fence();
    }
}

template <class T, int V, int P>
struct Larger {
    static struct Both {
        GroupLDS<V, P> lds;
        CandLDS<64> cand;
    } both;
    static void body(void *) {
        T g;
        g.setup(prm, &both.lds, &both.cand);
        g.set_cloud(&hdr, root);
        emu::fence();
        for (int32_t cell : cells) {
            g.active = true;
            const uint32_t before = g.gl == 0 ? both.lds.ctr[kStatClips] : 0u;
            g.start((uint32_t)cell, prm);
            if (prm.promo) g.offer_owners(prm.promo, kPromoPlanes);
            if (g.live()) g.traverse();
            if (g.np < 0 || g.np > P) fail("planes out of range", cell);
            const bool kept = !g.overflow;
            const int F = kept ? g.stage_row(prm) : 0;
            if (kept) g.write_row(prm, (uint32_t)cell, row_out, F);
            emu::fence();
            if (g.gl == 0) {
                std::vector<int32_t> held;
                for (int p = 0; p < g.np; ++p) held.push_back(__float_as_int(both.lds.plx[p].y));
                put(kept, mask_popc(g.valid), g.np, g.status, 0, (int)(both.lds.ctr[kStatClips] - before),
                    prm.counts[cell] * kept, row_out, held);
            }
            emu::fence();
        }
    }
    static void go(const Request &q) {
        emu::watch(&both, sizeof both);
        emu::run(64, (unsigned)q.seed, q.limit, body, nullptr);
    }
};
template <class T, int V, int P>
typename Larger<T, V, P>::Both Larger<T, V, P>::both;

void write(const std::vector<std::vector<int32_t>> &v) {
    for (const auto &r : v) {
        const int32_t m = (int32_t)r.size();
        fwrite(&m, 4, 1, stdout);
        fwrite(r.data(), 4, r.size(), stdout);
    }
}

}  // namespace

int main() {
    Request q;
    get(&q, sizeof q);
    pts = get<float4>(q.n);
    cells = get<int32_t>(q.cells);
    std::vector<int32_t> guesses = get<int32_t>((size_t)q.n * q.stride);
    std::vector<float> d2 = get<float>(q.has_d2 ? q.n : 0);
    float box[6];
    get(box, sizeof box);
    for (int k = 0; k < 3; ++k) hdr.box_lo[k] = box[k], hdr.box_hi[k] = box[3 + k];
    hdr.n = (uint32_t)q.n;
    std::vector<uint32_t> ids(q.n), one(q.n), none(q.n, 0xFFFFFFFFu);
    for (int i = 0; i < q.n; ++i) ids[i] = one[i] = (uint32_t)i;
    std::vector<int32_t> counts(q.n), status(q.n);
    nodes.reserve(q.n + 1);
    root = wide_over(0, (uint32_t)q.n, (uint32_t)q.fanout, (uint32_t)q.binary_below);
    nodes.emplace_back();
    wide.resize(wide.size() + 16);
    prm.n = q.n;
    prm.hdr = &hdr;
    prm.pts = pts.data();
    prm.perm = prm.inv = ids.data();
    prm.nodes = nodes.data();
    prm.wide = wide.data();
    prm.dup_head = one.data();
    prm.dup_next = none.data();
    prm.end = q.n;
    if (q.stride > 0) {
        prm.guesses = guesses.data();
        prm.guess_stride = q.stride;
        if (q.has_d2) prm.guess_d2 = d2.data();
    }
    prm.counts = counts.data();
    prm.status = status.data();
    if (q.tier == 0) {
        emu::watch(&lds0, sizeof lds0);
        // (every lane stores the number of recorded tests, and reads its own store back)
        emu::leave_out(&lds0.ntent, sizeof lds0.ntent);
        emu::run(16, (unsigned)q.seed, q.limit, body0, nullptr);
    } else if (q.tier == 1) {
        Larger<TierM, kTmVerts, kTmPlanes>::go(q);
    } else if (q.tier == 2) {
        Larger<Tier1, kT1Verts, kT1Planes>::go(q);
    } else {
        Larger<Tier2, kT2Verts, kT2Planes>::go(q);
    }
    fwrite(info.data(), 4, info.size(), stdout);
    write(rows);
    write(planes);
    emu::report(stderr);
    return 0;
}
