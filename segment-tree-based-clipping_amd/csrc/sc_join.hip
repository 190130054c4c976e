// sc_join.hip -- candidate pairs of a clip by a join of bounding boxes.
//
// The pairs that the stab finds (sc_stab.hip) are those whose boxes overlap
// (LSMF) and whose lineSegmentIntersection2 type is not 0; the tree only
// narrows down which pairs are tested.  A clip needs the pairs and not the
// tree, and a ring's own order narrows them down without any sort: 64
// consecutive edges are connected, so their box is small.  The join keeps
// one box per leaf (64 consecutive edges of a ring) and one per group (64
// consecutive leaves of a base ring):
//   k_join_leaves  box and place of every leaf, in single precision rounded
//                  outward; notes inputs that the join must not take
//   k_join_groups  box of every group of base leaves
//   k_join_tiles   one wave per overlay leaf: the base groups, then the base
//                  leaves, whose boxes meet it; each is a tile of at most
//                  64 x 64 edge pairs
//   k_join_pairs   one wave per tile: rows and columns that miss the other
//                  leaf's box drop out, the boxes of the rest are compared in
//                  single precision, the pairs that pass ("near") are queued
//                  in LDS and go through LSMF and the classification on the
//                  doubles with all lanes busy
//
// When the pair set equals the tree's.  Take a pair that LSMF keeps, with key
// intervals [s1,t1] and [s2,t2], s1 <= s2.  If no edge is vertical in the
// keys, every distinct endpoint value but the largest is one elementary point
// (k_unique_flags), so: for s1 < s2 the second edge's "before" leaf ends at s2
// and lies in the first edge's leaf range, which covers one of its ancestors;
// for s1 == s2 both ranges start at the same leaf, and either both edges cover
// the same node or the shorter range's "after" leaf lies under the longer
// one's first covered node.  The tree tests the pair either way.  Vertical
// edges bring repeated and missing points by the reference's rules, and the
// tree then misses pairs that touch there; NaN and infinities have no order.
// Rings with any of these go to the tree (join_candidates returns false).
//
// Measured (tree stages + stab + sort of the duplicates -> join + sort of the
// pairs): 200,000 x 1,000,000 harmonic rings 2.02 -> 0.32 ms (the join's
// kernels 0.15 ms), 100,000 x 4,096 star overlays 19.2 -> 1.94 ms, 1,000 x
// 1,000 stars 0.51 -> 0.08 ms, 256 pairs of 10,000 to 200,000 vertices 40 -> 1.25 ms.
#include "sc_ctx.hpp"
#include "sc_fp64.hpp"
#include "sc_wave.hpp"

#include <algorithm>

namespace sc {

namespace {

constexpr int BLK = 256;
constexpr int WPB = BLK / WAVE;

inline unsigned grid_for(int64_t n, int per = BLK) {
    int64_t g = ceil_div(n, per);
    if (g < 1) g = 1;
    return unsigned(g);
}

int bits_for(int64_t n) { // bits to hold values in [0, n)
    int b = 0;
    while ((int64_t(1) << b) < n) b++;
    return b < 1 ? 1 : b;
}

// The rings of the context: base rings 0..nbr-1, then overlays; loff holds
// their first leaves (nbr + K + 1 entries).
struct RingTab {
    const double2 *bpoly, *cpoly;
    const int *loff, *bvoff, *beoff, *coff, *eoff;
    const double *shift; // per ring of a pair, or null
    int nbr, K;
    uint32_t lb, nleaf; // base leaves, all leaves
    uint32_t call;      // this join's number: what "bad" holds where its rings are not for the join
};
// first vertex, edges, first edge (base: global, overlay: 0) and ring (overlay: 1-based) of a leaf
struct __align__(16) Leaf {
    uint32_t vert, n, edge, ring;
};

__device__ inline BoxF boxf_readlane(const BoxF &b, int l) {
    BoxF r;
    r.minx = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(b.minx), l));
    r.maxx = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(b.maxx), l));
    r.miny = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(b.miny), l));
    r.maxy = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(b.maxy), l));
    return r;
}
__device__ inline BoxF boxf_wave(const BoxF &b) { // no NaN: finite boxes and the empty box
    BoxF r;
    r.minx = wave_min(b.minx);
    r.maxx = wave_max(b.maxx);
    r.miny = wave_min(b.miny);
    r.maxy = wave_max(b.maxy);
    return r;
}
// ballot of the lanes whose box overlaps q (finite boxes; the empty box overlaps none)
__device__ inline uint64_t meets(const BoxF &b, const BoxF &q) {
    return __builtin_amdgcn_ballot_w64(b.minx <= q.maxx) & __builtin_amdgcn_ballot_w64(b.maxx >= q.minx) &
           __builtin_amdgcn_ballot_w64(b.miny <= q.maxy) & __builtin_amdgcn_ballot_w64(b.maxy >= q.miny);
}
__device__ inline BoxF edge_boxf(const double2 &a, const double2 &b) {
    return boxf_of(box_of(a.x, a.y, b.x, b.y));
}

// Tiles (base leaf, overlay leaf) go to TILE_SEGS segments, each with its own
// counter on its own 128-byte line, staged per wave (one same-address counter
// costs about 5 ns an atomic).
constexpr int TILE_SEGS = 512;
constexpr int TILE_PAD = 32; // u32 per counter line
constexpr int TSTG = 256;

// One wave per leaf.  Bound by the read of the vertices (16 bytes each).
// Clears the words that the tiles and pairs are counted in as well.
__global__ __launch_bounds__(BLK) void k_join_leaves(RingTab t, BoxF *__restrict__ box, Leaf *__restrict__ desc,
                                                     uint32_t *__restrict__ bad,
                                                     unsigned long long *__restrict__ sum,
                                                     uint32_t *__restrict__ counter) {
    const int lane = threadIdx.x & (WAVE - 1);
    const uint32_t w = uni(blockIdx.x * WPB + threadIdx.x / WAVE);
    for (uint32_t i = blockIdx.x * BLK + threadIdx.x; i < TILE_SEGS; i += gridDim.x * BLK) {
        counter[size_t(i) * TILE_PAD] = 0u;
        if (i < 3) sum[i] = 0ull;
    }
    if (w >= t.nleaf) return;
    const int r = seg_of(t.loff, t.nbr + t.K, w);
    const bool base = r < t.nbr;
    const int k = r - t.nbr;
    const double2 *P = base ? t.bpoly : t.cpoly;
    const uint32_t v0 = uint32_t(base ? t.bvoff[r] : t.coff[k]);
    const uint32_t e0 = uint32_t(base ? t.beoff[r] : t.eoff[k]);
    const uint32_t n = uint32_t(base ? t.beoff[r + 1] : t.eoff[k + 1]) - e0;
    const uint32_t first = (w - uint32_t(t.loff[r])) * uint32_t(WAVE);
    const uint32_t cnt = min(uint32_t(WAVE), n - first);
    BoxF b = boxf_empty();
    bool no = false;
    if (uint32_t(lane) < cnt) {
        const double2 p = P[v0 + first + lane], q = P[v0 + first + lane + 1];
        b = edge_boxf(p, q);
        const double sh = t.shift ? t.shift[base ? r : k] : 0.0;
        const double kp = p.x + sh, kq = q.x + sh; // the tree's keys (k_edges)
        no = kp == kq || !(fabs(kp) < INFINITY) || !(fabs(p.y) < INFINITY) || !(fabs(kq) < INFINITY) ||
             !(fabs(q.y) < INFINITY);
    }
    if (__ballot(no)) {
        if (lane == 0) *bad = t.call;
        return; // the join's results are not used
    }
    b = boxf_wave(b);
    if (lane == 0) {
        box[w] = b;
        Leaf d;
        d.vert = v0 + first;
        d.n = cnt;
        d.edge = base ? e0 + first : first;
        d.ring = uint32_t(base ? r : k + 1);
        desc[w] = d;
    }
}

// Group slots: the groups of base ring r start at loff[r] / 64 + r (a ring of
// n leaves has at most n / 64 + 1 groups, so the slots of two rings never meet).
__device__ inline uint32_t group_slot(const int *loff, int r) { return uint32_t(loff[r]) / uint32_t(WAVE) + uint32_t(r); }

// One wave per group slot of the base rings.
__global__ __launch_bounds__(BLK) void k_join_groups(RingTab t, const BoxF *__restrict__ box, uint32_t nslot,
                                                     BoxF *__restrict__ gbox, const uint32_t *__restrict__ bad) {
    const int lane = threadIdx.x & (WAVE - 1);
    const uint32_t w = uni(blockIdx.x * WPB + threadIdx.x / WAVE);
    if (w >= nslot || *bad == t.call) return;
    int lo = 0, hi = t.nbr - 1; // last ring whose first slot is <= w
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (group_slot(t.loff, mid) <= w) lo = mid;
        else hi = mid - 1;
    }
    const uint32_t l = uint32_t(t.loff[lo]) + (w - group_slot(t.loff, lo)) * uint32_t(WAVE) + uint32_t(lane);
    BoxF b = boxf_empty();
    if (l < uint32_t(t.loff[lo + 1])) b = box[l];
    b = boxf_wave(b);
    if (lane == 0) gbox[w] = b;
}

struct TileArgs {
    RingTab t;
    const BoxF *box, *gbox;
    const Leaf *desc;
    bool paired;
    uint32_t chunk;      // base groups per wave
    const uint32_t *bad;
    uint2 *out;
    uint32_t cap;        // per segment
    uint32_t *counter;
};

// One wave per overlay leaf and chunk of base groups: 64 boxes a step.
__global__ __launch_bounds__(BLK) void k_join_tiles(TileArgs a) {
    __shared__ uint2 stage_all[WPB][TSTG];
    const int lane = threadIdx.x & (WAVE - 1);
    const uint32_t wv = uni(threadIdx.x / WAVE);
    const uint32_t w = blockIdx.x * WPB + wv;
    const uint32_t L = a.t.lb + w;
    if (L >= a.t.nleaf || *a.bad == a.t.call) return;
    const BoxF cb = a.box[L];
    const int r = a.paired ? int(a.desc[L].ring) - 1 : 0;
    const uint32_t l0 = uint32_t(a.t.loff[r]), nl = uint32_t(a.t.loff[r + 1]) - l0;
    uint2 *stage = stage_all[wv];
    const uint32_t seg = (w + blockIdx.y * 61u) % uint32_t(TILE_SEGS);
    const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (WAVE - lane));
    uint32_t cnt = 0;
    auto flush = [&]() {
        uint32_t base = 0;
        if (lane == 0) base = atomicAdd(a.counter + size_t(seg) * TILE_PAD, cnt);
        base = uni(base);
        uint2 *out = a.out + size_t(seg) * a.cap;
        for (uint32_t i = lane; i < cnt; i += WAVE)
            if (base + i < a.cap) out[base + i] = stage[i];
        cnt = 0;
    };
    // the 64 leaves from 'f' (ring-local) against this overlay leaf
    auto leaves = [&](uint32_t f) {
        const uint32_t l = f + uint32_t(lane);
        const BoxF b = l < nl ? a.box[l0 + l] : boxf_empty();
        const uint64_t m = meets(b, cb);
        if (!m) return;
        const uint32_t nh = uint32_t(__popcll(m));
        if (cnt + nh > uint32_t(TSTG)) flush();
        if ((m >> lane) & 1ull) stage[cnt + uint32_t(__popcll(m & lt))] = make_uint2(l0 + l, L);
        cnt += nh;
    };
    const uint32_t ng = (nl + WAVE - 1) / WAVE;
    const uint32_t g0 = blockIdx.y * a.chunk, g1 = min(ng, g0 + a.chunk);
    if (ng == 1) {
        if (g0 == 0) leaves(0);
    } else {
        const uint32_t gs = group_slot(a.t.loff, r);
        for (uint32_t g = g0; g < g1; g += WAVE) {
            const uint32_t gi = g + uint32_t(lane);
            const BoxF b = gi < g1 ? a.gbox[gs + gi] : boxf_empty();
            uint64_t m = meets(b, cb);
            while (m) {
                const int i = __builtin_ctzll(m);
                m &= m - 1ull;
                leaves((g + uint32_t(i)) * uint32_t(WAVE));
            }
        }
    }
    if (cnt) flush();
}

struct PairArgs {
    const double2 *bpoly, *cpoly;
    const BoxF *box;
    const Leaf *desc;
    const int *coff;
    bool paired;
    const uint32_t *bad;
    uint32_t call;
    const uint2 *tiles;
    uint32_t cap;
    const uint32_t *counter;
    int bits_b, bits_c;
    uint64_t *out;
    uint64_t out_cap;
    unsigned long long *sum; // [0] pairs, [1] tiles, [2] largest segment
};

constexpr int QNEAR = 2 * WAVE;      // near pairs classified per step, two per lane
constexpr int QCAP = QNEAR + WAVE;   // queue: a row adds at most 64
// Found pairs staged per wave.  A flush takes its place in the output with an
// atomic on one word, and those queue up: 20 million pairs with 256 staged took
// 1.35 ms, with 640 (five blocks of LDS still fit a CU) 0.87; eight counters
// with parts of the output to pack afterwards gain nothing more.
constexpr int HSTG = 10 * WAVE;

// One wave per run of tiles; the grid covers the chip and strides over the
// tiles.  A block's waves take its turns from a counter in LDS: tiles differ a
// lot in the rows that survive, and with a fixed share per wave a third of the
// launched waves were in flight on average (the join's kernels at 200,000 x
// 1,000,000 vertices: 192 -> 161 us, at 100,000 x 4,096 overlays: 1.00 -> 0.94
// ms).  Blocks of five or ten waves share better and run slower (181, 190).
// Bound by VALU issue: about 14 instructions per surviving row and 64 columns,
// and the classification's FP64 work per near pair.
__global__ __launch_bounds__(BLK) void k_join_pairs(PairArgs a) {
    __shared__ uint32_t toff[TILE_SEGS + 1]; // first tile of each segment
    __shared__ uint32_t next;                // the block's turns taken so far
    __shared__ uint32_t qb[WPB][QCAP], qc[WPB][QCAP], qk[WPB][QCAP];
    __shared__ uint64_t hits_all[WPB][HSTG];
    if (*a.bad == a.call) return; // every block reads the same word
    const int lane = threadIdx.x & (WAVE - 1);
    const uint32_t wv = uni(threadIdx.x / WAVE);
    if (wv == 0) { // segment counts to offsets, eight segments per lane
        constexpr int PER = TILE_SEGS / WAVE;
        uint32_t c[PER], s = 0, mx = 0;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const uint32_t raw = a.counter[size_t(lane * PER + i) * TILE_PAD];
            mx = max(mx, raw);
            c[i] = min(raw, a.cap);
            s += c[i];
        }
        uint32_t incl = s;
        for (int d = 1; d < WAVE; d <<= 1) {
            const uint32_t o = __shfl_up(incl, d, WAVE);
            if (lane >= d) incl += o;
        }
        uint32_t at = incl - s;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            toff[lane * PER + i] = at;
            at += c[i];
        }
        if (lane == WAVE - 1) toff[TILE_SEGS] = at;
        mx = wave_reduce(mx, [](uint32_t x, uint32_t y) { return max(x, y); });
        if (lane == 0) next = 0u;
        if (blockIdx.x == 0 && lane == WAVE - 1) {
            a.sum[1] = at;
            a.sum[2] = mx;
        }
    }
    __syncthreads();
    // Fewer than eight turns per wave: 2 to 16 waves share a tile, each walking
    // every 2nd to 16th of its rows or columns (two stars of 1,000 and 1,100
    // vertices have 272 tiles, which took 36 us a wave each, 13 shared).  At
    // 200,000 x 1,000,000 vertices, 3 tiles a wave, halves of tiles take the
    // join from 161 to 153 us; quarters repeat the tiles' set-up too often (with
    // fixed shares: whole tiles 192 us, halves 176, quarters 205).
    const uint32_t nw = gridDim.x * WPB;
    uint32_t parts = 1;
    while (parts < 16u && uint64_t(toff[TILE_SEGS]) * parts * 2u <= 8u * uint64_t(nw)) parts *= 2u;
    const uint32_t ntile = toff[TILE_SEGS] * parts; // shares of tiles
    const uint64_t share = ~0ull / ((1ull << parts) - 1ull); // every parts-th row
    uint32_t *vb = qb[wv], *vc = qc[wv], *vk = qk[wv];
    uint64_t *hits = hits_all[wv];
    const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (WAVE - lane));
    const int sb = a.bits_b + a.bits_c;
    uint32_t nq = 0, nh = 0;
    auto flush = [&]() {
        unsigned long long base = 0;
        if (lane == 0) base = atomicAdd(a.sum, (unsigned long long)nh);
        base = (uint64_t(uni(uint32_t(base >> 32))) << 32) | uni(uint32_t(base));
        for (uint32_t i = lane; i < nh; i += WAVE)
            if (base + i < a.out_cap) a.out[base + i] = hits[i];
        nh = 0;
    };
    // the first n queued near pairs (n <= QNEAR), two per lane
    auto classify_queue = [&](uint32_t n) {
        double2 B0[2], B1[2], C0[2], C1[2];
        uint32_t b[2], c[2], k[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const uint32_t i = uint32_t(u * WAVE + lane);
            if (i >= n) continue;
            b[u] = vb[i];
            c[u] = vc[i];
            k[u] = vk[i];
            B0[u] = a.bpoly[b[u]];
            B1[u] = a.bpoly[b[u] + 1];
            C0[u] = a.cpoly[c[u]];
            C1[u] = a.cpoly[c[u] + 1];
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            bool hit = false;
            if (uint32_t(u * WAVE + lane) < n)
                hit = box_overlap(box_of(B0[u].x, B0[u].y, B1[u].x, B1[u].y),
                                  box_of(C0[u].x, C0[u].y, C1[u].x, C1[u].y)) &&
                      classify_pre(B0[u].x, B0[u].y, B1[u].x, B1[u].y, C0[u].x, C0[u].y, C1[u].x, C1[u].y) != 0;
            const uint64_t m = __ballot(hit);
            if (!m) continue;
            const uint32_t add = uint32_t(__popcll(m));
            if (nh + add > uint32_t(HSTG)) flush();
            if (hit) {
                // a base vertex is its edge plus one per ring before (closing vertices)
                const uint32_t be = b[u] - (a.paired ? k[u] - 1u : 0u);
                const uint32_t local = c[u] - uint32_t(a.coff[k[u] - 1u]);
                hits[nh + uint32_t(__popcll(m & lt))] =
                    (uint64_t(k[u]) << sb) | (uint64_t(be) << a.bits_c) | uint64_t(local);
            }
            nh += add;
        }
    };
    const uint32_t per = min(8u, max(1u, ntile / (4u * nw))); // tiles per turn
    int sg = 0;
    for (;;) {
        uint32_t turn = 0;
        if (lane == 0) turn = atomicAdd(&next, 1u);
        const uint64_t at0 = (uint64_t(uni(turn)) * gridDim.x + blockIdx.x) * per;
        if (at0 >= ntile) break;
        const uint32_t t0 = uint32_t(at0), t1 = min(ntile, t0 + per);
        int hi = TILE_SEGS; // toff[sg] <= t0 < toff[hi]: later turns search on from the last segment
        while (hi - sg > 1) {
            const int mid = (sg + hi) >> 1;
            if (toff[mid] * parts <= t0) sg = mid;
            else hi = mid;
        }
        for (uint32_t t = t0; t < t1; ++t) {
            const uint32_t tile = t / parts;
            while (toff[sg + 1] <= tile) ++sg; // tile < toff[TILE_SEGS]: ends at the last non-empty segment
            const uint2 tl = a.tiles[size_t(sg) * a.cap + (tile - toff[sg])];
            const uint32_t lb = uni(tl.x), lc = uni(tl.y);
            const Leaf db = a.desc[lb], dc = a.desc[lc];
            const BoxF bb = a.box[lb], cb = a.box[lc];
            BoxF rb = boxf_empty(), cl = boxf_empty();
            if (uint32_t(lane) < db.n) rb = edge_boxf(a.bpoly[db.vert + lane], a.bpoly[db.vert + lane + 1]);
            if (uint32_t(lane) < dc.n) cl = edge_boxf(a.cpoly[dc.vert + lane], a.cpoly[dc.vert + lane + 1]);
            const uint64_t R = meets(rb, cb), C = meets(cl, bb);
            // walk the side with fewer survivors, the other side in lanes
            const bool rows = __popcll(R) <= __popcll(C);
            uint64_t set = (rows ? R : C) & (share << (t % parts));
            const uint64_t other = rows ? C : R;
            const BoxF mine = rows ? cl : rb, walk = rows ? rb : cl;
            while (set) {
                const int i = __builtin_ctzll(set);
                set &= set - 1ull;
                const uint64_t m = meets(mine, boxf_readlane(walk, i)) & other;
                if (!m) continue;
                if ((m >> lane) & 1ull) {
                    const uint32_t at = nq + uint32_t(__popcll(m & lt));
                    vb[at] = db.vert + uint32_t(rows ? i : lane);
                    vc[at] = dc.vert + uint32_t(rows ? lane : i);
                    vk[at] = dc.ring;
                }
                nq += uint32_t(__popcll(m));
                if (nq >= uint32_t(QNEAR)) {
                    classify_queue(QNEAR);
                    nq -= uint32_t(QNEAR); // fewer than 64 are left: move them to the front
                    if (uint32_t(lane) < nq) {
                        vb[lane] = vb[QNEAR + lane];
                        vc[lane] = vc[QNEAR + lane];
                        vk[lane] = vk[QNEAR + lane];
                    }
                }
            }
        }
    }
    if (nq) classify_queue(nq);
    if (nh) flush();
}

} // namespace

bool join_candidates(Ctx &c) {
    SC_REQUIRE(c.ne > 0, SC_ESTATE, "polygons not set");
    hipStream_t s = c.stream;
    c.bits_b = bits_for(c.nb);
    c.bits_c = bits_for(c.maxcsz);
    c.bits_k = bits_for(int64_t(c.K) + 1);
    SC_REQUIRE(c.bits_b + c.bits_c + c.bits_k <= 64, SC_ERANGE, "pair key does not fit in 64 bits");
    key_shifts(c);
    const int R = c.nbr + c.K;
    const uint32_t nleaf = uint32_t(c.loff[R]), lb = uint32_t(c.loff[c.nbr]), lc = nleaf - lb;
    RingTab t;
    t.bpoly = reinterpret_cast<const double2 *>(c.bpoly.p);
    t.cpoly = reinterpret_cast<const double2 *>(c.cpoly.p);
    t.loff = c.d_loff;
    t.bvoff = c.d_bvoff;
    t.beoff = c.d_beoff;
    t.coff = c.d_coff;
    t.eoff = c.d_eoff;
    t.shift = c.paired ? c.d_shift.p : nullptr;
    t.nbr = c.nbr;
    t.K = c.K;
    t.lb = lb;
    t.nleaf = nleaf;
    // boxes and places: leaves, then the base rings' groups (their slots end below lb / 64 + nbr + 1)
    const uint32_t nslot = lb / uint32_t(WAVE) + uint32_t(c.nbr);
    BoxF *box = reinterpret_cast<BoxF *>(c.join_box.ensure(2 * (size_t(nleaf) + nslot)));
    BoxF *gbox = box + nleaf;
    Leaf *desc = reinterpret_cast<Leaf *>(c.join_leaf.ensure(2 * size_t(nleaf)));
    // control words: pairs, tiles, largest segment (64 bits each), the "bad" flag, then the segment counters
    const bool fresh = c.join_ctl.cap == 0; // holds nothing yet
    if (++c.join_call == 0) c.join_call = 1;
    t.call = c.join_call;
    uint32_t *ctl = c.join_ctl.ensure(size_t(TILE_PAD) * (TILE_SEGS + 1));
    unsigned long long *sum = reinterpret_cast<unsigned long long *>(ctl);
    uint32_t *bad = ctl + 6, *counter = ctl + TILE_PAD;
    if (c.join_seg_cap == 0) c.join_seg_cap = std::max<int64_t>(64, ceil_div(16 * int64_t(nleaf), TILE_SEGS));
    if (c.cand_cap == 0) c.cand_cap = std::max<int64_t>(1 << 16, 2 * int64_t(c.ne));
    uint32_t maxng = 1;
    for (int r = 0; r < c.nbr; ++r)
        maxng = std::max(maxng, uint32_t(ceil_div(c.loff[r + 1] - c.loff[r], WAVE)));
    // few overlay leaves: a leaf's base groups are split over more waves
    const uint32_t chunk = lc >= 16384u ? uint32_t(WAVE) : lc >= 2048u ? 16u : 4u;
    uint64_t h[4] = {0, 0, 0, 0};
    for (int attempt = 0; attempt < 3; ++attempt) {
        c.join_tile.ensure(size_t(c.join_seg_cap) * TILE_SEGS);
        c.pairs.ensure(size_t(c.cand_cap));
        if (attempt > 0 || fresh) {
            FillBatch fb(s);
            fb.add(ctl, int64_t(TILE_PAD) * (TILE_SEGS + 1), 0u);
            fb.flush();
        }
        c.mark(8);
        if (attempt == 0) {
            k_join_leaves<<<grid_for(nleaf, WPB), BLK, 0, s>>>(t, box, desc, bad, sum, counter);
            SC_HIP(hipGetLastError());
            if (maxng > 1) {
                k_join_groups<<<grid_for(nslot, WPB), BLK, 0, s>>>(t, box, nslot, gbox, bad);
                SC_HIP(hipGetLastError());
            }
        }
        TileArgs a;
        a.t = t;
        a.box = box;
        a.gbox = gbox;
        a.desc = desc;
        a.paired = c.paired;
        a.chunk = chunk;
        a.bad = bad;
        a.out = reinterpret_cast<uint2 *>(c.join_tile.p);
        a.cap = uint32_t(c.join_seg_cap);
        a.counter = counter;
        k_join_tiles<<<dim3(grid_for(lc, WPB), unsigned(ceil_div(maxng, chunk))), BLK, 0, s>>>(a);
        SC_HIP(hipGetLastError());
        PairArgs p;
        p.bpoly = t.bpoly;
        p.cpoly = t.cpoly;
        p.box = box;
        p.desc = desc;
        p.coff = t.coff;
        p.paired = c.paired;
        p.bad = bad;
        p.call = t.call;
        p.tiles = a.out;
        p.cap = a.cap;
        p.counter = counter;
        p.bits_b = c.bits_b;
        p.bits_c = c.bits_c;
        p.out = c.pairs;
        p.out_cap = uint64_t(c.cand_cap);
        p.sum = sum;
        int cus = 256, v = 0;
        if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, c.device) == hipSuccess && v > 0) cus = v;
        k_join_pairs<<<unsigned(cus) * 5u, BLK, 0, s>>>(p);
        SC_HIP(hipGetLastError());
        c.mark(9);
        ReadBack rb(c);
        rb.add(h, reinterpret_cast<const uint64_t *>(ctl), 4);
        rb.run();
        if (uint32_t(h[3]) == t.call) return false;
        const int64_t seg_max = int64_t(h[2]), np = int64_t(h[0]);
        if (seg_max > int64_t(UINT32_MAX / TILE_SEGS)) return false; // tiles are counted in 32 bits
        if (seg_max > c.join_seg_cap) {
            c.join_seg_cap = seg_max + seg_max / 4 + 64;
            continue;
        }
        if (np <= c.cand_cap) break;
        c.cand_cap = np + np / 4 + 1024;
    }
    SC_REQUIRE(int64_t(h[2]) <= c.join_seg_cap && int64_t(h[0]) <= c.cand_cap, SC_EHIP,
               "join buffer overflow after resize");
    // every pair was found once; sorted by (overlay, base edge, overlay-local edge).
    // One overlay has one overlay field, and a pair's base edges already follow
    // the pair order, so both leave that field out of the sort.
    const int64_t n = int64_t(h[0]);
    const int kb = c.bits_b + c.bits_c + (c.paired || c.K == 1 ? 0 : c.bits_k);
    if (n <= SMALL_SORT_MAX) sort_small_u64(c.pairs, c.cand.ensure(size_t(n) + 1), int(n), s); // whole keys: the same order
    else radix_sort_u64_buf(c.pairs, c.cand, nullptr, nullptr, n, 0, kb, c.rs, s);
    c.n_pairs = n;
    pair_offsets(c);
    c.n_cand = c.n_near = c.n_tests = c.n_units = 0;
    c.joined = true;
    return true;
}

} // namespace sc
