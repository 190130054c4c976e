// sc_small.hip -- a batch of small independent pairs clipped by one kernel: one
// wave per pair, the whole clip of a pair in LDS (rows A8-A17 for rings of up to 64 vertices).
//
// A pair's candidate set is the brute-force set {(b, c): LSMF and a non-zero
// lineSegmentIntersection2 type}, which equals the set the reference's tree
// emits for rings without vertical edges (saveIntersectionsIdsMulticore,
// oacc:6010-6244; a vertical edge's one-point range can miss its partners in
// the tree, never here), in (base edge, overlay edge) order.  Then,
// as the staged path and the oracle do (clip:522-601, oacc:7257-7988):
// per-edge counts, intersection points and quantised alpha / beta, every
// edge's intersections ordered by (alpha modulo 1e9, pair), augmented rings
// with neighbour links, initial labels.  Labelling, traversal and clean-up
// follow labelIntersections2 / createResult2 / cleanUpResult2
// (foster/polyclip.h:337-787), on slot numbers and bit sets instead of linked
// vertices.
//
// A wave never waits on one lane: pair tests spread over (base edge, overlay
// edge) and again over the boxes that overlap, both edge orders by counting
// the smaller keys, a lane per pair for slots and labels, the entry/exit
// status from the number of crossings before a slot.  The traversal steps from
// crossing to crossing on 192-bit sets held in scalar registers and the wave
// copies each piece's slots; clean-up checks every vertex at once against its
// neighbours and runs in order, on one lane, only for a ring that loses one.
//
// Bound by VALU issue (FP64 predicates): 2,170 vector instructions per wave
// for rings of 4 to 64 vertices keep the units about half busy.  16,384 such
// pairs take 112 us where sizes are log-uniform, 160 where they are uniform; the
// version that linked vertices in LDS (28 KB a pair, five pairs a CU) and walked
// them on one lane took 700 on the former.
//
// Covered here: pairs whose intersection vertices are all labelled CROSSING
// or BOUNCING, whose rings keep a plain vertex, with no bouncing pair to
// split, every intersection given a slot, quantised alphas in range, and
// sizes within the LDS capacities below.  Any other pair sets its fallback
// word and the host reruns the whole batch on the staged path.
#include "sc_ctx.hpp"
#include "sc_fp64.hpp"

namespace sc {

namespace {

constexpr int SP_NV = 64;                    // ring vertices per side
constexpr int SP_I = 128;                    // intersections per pair
constexpr int SP_AUG = SP_NV + SP_I;         // augmented ring slots per side
constexpr int SP_OUTR = 64;                  // output rings per pair
constexpr int SP_OUTV = 2 * SP_AUG;          // output vertices per pair
constexpr int SP_C0 = SP_NV + 1;             // point codes: base vertices, overlay vertices (each ring
constexpr int SP_P0 = 2 * (SP_NV + 1);       // with its closing vertex), intersections
constexpr int SP_NONE = 255;                 // no slot
constexpr int SP_NOV = -100;
constexpr int SP_WORDS = SP_AUG / 64;        // a bit per slot of one side

enum : int { L_NONE = 0, L_CROSSING = 1, L_BOUNCING = 2 };
// fallback reasons, per pair
enum : int {
    F_SIZE = 1, F_PAIRS = 2, F_SLOT = 4, F_ALPHA = 8, F_WALK = 16, F_LABEL = 32, F_PLAIN = 64, F_SPLIT = 128,
    F_TRAV = 256, F_OUT = 512
};

// 7.9 KB, so that 20 pairs are in flight on a CU: a slot or an output vertex
// is a code into the one array of points, never a copy of it.
struct SmallLDS {
    double X[SP_P0 + SP_I], Y[SP_P0 + SP_I];
    union {
        struct {
            int qa[SP_I], qb[SP_I]; // quantised alpha / beta, until the pairs are ordered
        };
        uint16_t ord[SP_OUTV];      // output vertices, ring after ring
    };
    uint16_t code[2][SP_AUG];       // per side and slot: its point
    uint8_t nb[2][SP_AUG];          // the partner slot (SP_NONE: a plain vertex)
    uint8_t lab[SP_AUG];            // label of a base slot (of its partner too)
    uint8_t pe[2][SP_I], pt[SP_I];  // per pair: its edges and type
    uint8_t srt[2][SP_I];           // per side: position in the order by (edge, parameter modulo 1e9, pair) -> pair
    uint8_t ps[2][SP_I];            // per side and pair: its slot
    uint8_t cnt[2][SP_NV + 1], nd[2][SP_NV + 1]; // per edge: pairs / inserted ones on earlier edges
    uint16_t cand[WAVE];
    uint16_t rbeg[SP_OUTR], rlen[SP_OUTR];
};

struct SmallArgs {
    int J;
    const int *bvoff, *nb, *cvoff, *nc; // per job: ring offsets (vertices, closing vertices included) and sizes
    const double *bpoly, *cpoly;
    int *fail;                          // per job: fallback reasons (0: clipped here)
    int *route;                         // per job: 0 crossing traversal, 1 no crossing vertex
    int *job_nv, *job_nr;               // per job: output vertices and rings
    double *out_x, *out_y;              // per job slot of SP_OUTV vertices
    int *out_len;                       // per job slot of SP_OUTR ring lengths
    double *out4;                       // areas and IoU instead of the rings, 4 x J (the batch-area layout)
    uint32_t *anyfail;                  // optional: set when some job falls back
};

// LDS of one wave: its accesses stay in order, so the compiler's order is all
// that a step needs from the one before
__device__ inline void step() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

__device__ inline int wave_sum(int v) {
    for (int d = WAVE / 2; d > 0; d >>= 1) v += __shfl_xor(v, d, WAVE);
    return v;
}
__device__ inline int wave_excl(int v, int lane, int &total) {
    int inc = v;
    for (int d = 1; d < WAVE; d <<= 1) {
        const int y = __shfl_up(inc, d, WAVE);
        if (lane >= d) inc += y;
    }
    total = __builtin_amdgcn_readlane(inc, WAVE - 1);
    return inc - v;
}
__device__ inline uint64_t lane64(uint64_t v, int l) { // lane l's value (l the same on every lane)
    const uint32_t lo = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(v)), l));
    const uint32_t hi = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(v >> 32)), l));
    return (uint64_t(hi) << 32) | lo;
}

// a bit per slot of one side's augmented ring, in scalar registers
struct Slots {
    uint64_t w[SP_WORDS];
};
__device__ inline bool has(const Slots &m, int s) {
    const uint64_t v = s < 64 ? m.w[0] : (s < 128 ? m.w[1] : m.w[2]);
    return (v >> (s & 63)) & 1u;
}
__device__ inline Slots pick(bool second, const Slots &a, const Slots &b) {
    Slots r;
#pragma unroll
    for (int k = 0; k < SP_WORDS; ++k) r.w[k] = second ? b.w[k] : a.w[k];
    return r;
}
__device__ inline Slots only(int s) {
    Slots r;
#pragma unroll
    for (int k = 0; k < SP_WORDS; ++k) r.w[k] = (s >> 6) == k ? 1ull << (s & 63) : 0ull;
    return r;
}
__device__ inline void drop(Slots &m, int s) {
    const Slots b = only(s);
#pragma unroll
    for (int k = 0; k < SP_WORDS; ++k) m.w[k] &= ~b.w[k];
}
__device__ inline bool any(const Slots &m) { return (m.w[0] | m.w[1] | m.w[2]) != 0; }
__device__ inline int lowest(const Slots &m) { // of a set that is not empty
    if (m.w[0]) return __ffsll((unsigned long long)m.w[0]) - 1;
    if (m.w[1]) return 63 + __ffsll((unsigned long long)m.w[1]);
    return 127 + __ffsll((unsigned long long)m.w[2]);
}
__device__ inline int highest(const Slots &m) {
    if (m.w[2]) return 191 - __clzll((long long)m.w[2]);
    if (m.w[1]) return 127 - __clzll((long long)m.w[1]);
    return 63 - __clzll((long long)m.w[0]);
}
__device__ inline Slots above(int s) { // the slots after s
    Slots r;
#pragma unroll
    for (int k = 0; k < SP_WORDS; ++k) {
        const int b = s - 64 * k;
        r.w[k] = b < 0 ? ~0ull : (b >= 63 ? 0ull : ~0ull << (b + 1));
    }
    return r;
}
// the next slot of a non-empty set from s on, forwards or backwards round the ring (s itself last)
__device__ inline int next_slot(const Slots &m, int s, bool fwd) {
    const Slots a = above(s);
    Slots x;
#pragma unroll
    for (int k = 0; k < SP_WORDS; ++k) x.w[k] = m.w[k] & (fwd ? a.w[k] : ~a.w[k]);
    if (fwd) return any(x) ? lowest(x) : lowest(m);
    drop(x, s);
    return any(x) ? highest(x) : highest(m);
}
__device__ inline int below(uint64_t m) { // bits of m below this lane
    return int(__builtin_amdgcn_mbcnt_hi(uint32_t(m >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(m), 0)));
}

// winding test of (rx, ry) against an augmented ring of n slots
// (polygon::pointInPoly, polygon.h:435-457): an integer sum of per-edge terms,
// so the lanes may add them in any order
__device__ bool point_in_ring(const SmallLDS &L, const uint16_t *code, int n, double rx, double ry, int lane) {
    int w = 0;
    for (int k = lane; k < n; k += WAVE) {
        const int one = code[k], two = code[k + 1 == n ? 0 : k + 1];
        const double p0x = L.X[one], p0y = L.Y[one], p1x = L.X[two], p1y = L.Y[two];
        if ((p0y < ry) != (p1y < ry)) {
            const int dir = 2 * (p1y > p0y) - 1;
            if (p0x >= rx) {
                if (p1x > rx) w += dir;
                else if ((areaA(p0x, p0y, p1x, p1y, rx, ry) > 0) == (p1y > p0y)) w += dir;
            } else if (p1x > rx) {
                if ((areaA(p0x, p0y, p1x, p1y, rx, ry) > 0) == (p1y > p0y)) w += dir;
            }
        }
    }
    return (wave_sum(w) % 2) != 0;
}

// the first slot without an intersection, -1 if there is none
__device__ inline int first_plain(const Slots &inter, int n) {
    Slots p;
#pragma unroll
    for (int k = 0; k < SP_WORDS; ++k) p.w[k] = ~inter.w[k];
    const int v = any(p) ? lowest(p) : SP_AUG; // slots past the ring have no intersection either
    return v < n ? v : -1;
}

// From the first plain vertex v on, the k-th crossing after it gets ENTRY/EXIT
// alternately starting from ENTRY (EXIT when v lies inside the other ring); a
// bouncing vertex met in the EXIT state is a split candidate.
__device__ inline void states(const Slots &cross, const Slots &inter, int v, bool inside, int lane, Slots &exits,
                              Slots &split) {
    const Slots after = above(v);
    int upto = 0, m = 0; // crossings before v (v is none), crossings
#pragma unroll
    for (int k = 0; k < SP_WORDS; ++k) {
        upto += __popcll(cross.w[k] & ~after.w[k]);
        m += __popcll(cross.w[k]);
    }
    int at = 0;
#pragma unroll
    for (int k = 0; k < SP_WORDS; ++k) {
        const int c = at + below(cross.w[k]) - upto + (64 * k + lane < v ? m : 0);
        const uint64_t ex = __ballot(((c & 1) != 0) != inside);
        exits.w[k] = ex & cross.w[k];
        split.w[k] = ex & inter.w[k] & ~cross.w[k];
        at += __popcll(cross.w[k]);
    }
}

__device__ inline bool flat(const SmallLDS &L, int a, int b, int c) { // codes of three points
    return fabs(areaA(L.X[a], L.Y[a], L.X[b], L.Y[b], L.X[c], L.Y[c])) < EPS;
}

// Shoelace sums in the order of the batch-area kernels, so both give the same
// bits: a ring's terms x_i y_(i+1) - x_(i+1) y_i added per lane over
// i = lane, lane + 64, ... and then by a shuffle tree (32, 16, ..., 1); an input
// ring (at most 64 vertices) and the sum of a job's |S| over its rings (at most
// 64) as those kernels' 256-thread block sums, whose two upper tree steps add
// zeros.
__device__ inline double wave_tree(double s) {
    for (int d = WAVE / 2; d > 0; d >>= 1) s += __shfl_down(s, d, WAVE);
    return __shfl(s, 0, WAVE);
}
__device__ double input_ring_sum2(const double *x, const double *y, int n, int lane) {
    double s = 0.0;
    if (lane < n) s += x[lane] * y[lane + 1] - x[lane + 1] * y[lane];
    s = (s + 0.0) + 0.0;
    return wave_tree(s);
}
__device__ void pair_areas(const SmallArgs &a, const SmallLDS &L, int j, int nb, int nc, int nr, int lane) {
    double mine = 0.0; // lane r: |S| of output ring r
    for (int r = 0; r < nr; ++r) {
        const int at = L.rbeg[r], len = L.rlen[r];
        double s = 0.0;
        for (int i = lane; i < len; i += WAVE) {
            const int v = L.ord[at + i], w = L.ord[at + (i + 1 == len ? 0 : i + 1)];
            s += L.X[v] * L.Y[w] - L.X[w] * L.Y[v];
        }
        const double rs = wave_tree(s);
        if (lane == r) mine += fabs(rs);
    }
    const double out2 = wave_tree((mine + 0.0) + 0.0);
    const double P2 = input_ring_sum2(L.X, L.Y, nb, lane), Q2 = input_ring_sum2(L.X + SP_C0, L.Y + SP_C0, nc, lane);
    if (lane == 0) {
        const int J = a.J;
        const double I = 0.5 * out2, P = 0.5 * fabs(P2), Q = 0.5 * fabs(Q2);
        const double U = P + Q - I;
        a.out4[j] = I;
        a.out4[J + j] = P;
        a.out4[2 * J + j] = Q;
        a.out4[3 * J + j] = U != 0.0 ? I / U : 0.0;
    }
}

// one pair, the whole wave; returns the fallback reasons (0: clipped)
__device__ int clip_pair(const SmallArgs &a, SmallLDS &L, int j, int lane, int &route, int &nv_out, int &nr_out) {
    const int nb = a.nb[j], nc = a.nc[j];
    nv_out = nr_out = 0;
    route = 0;
    if (nb > SP_NV || nc > SP_NV || nb < 3 || nc < 3) return F_SIZE;
    {
        const double *B = a.bpoly + 2 * int64_t(a.bvoff[j]);
        const double *C = a.cpoly + 2 * int64_t(a.cvoff[j]);
        for (int i = lane; i <= nb; i += WAVE) {
            L.X[i] = B[2 * i];
            L.Y[i] = B[2 * i + 1];
        }
        for (int i = lane; i <= nc; i += WAVE) {
            L.X[SP_C0 + i] = C[2 * i];
            L.Y[SP_C0 + i] = C[2 * i + 1];
        }
    }
    step();

    // ---- pairs with overlapping boxes: as many lanes per base edge as fit, the overlay edges between them ----
    uint64_t boxes = 0; // lane = base edge: its overlay edges
    {
        const int G = WAVE / nb, g = lane / nb, e = lane - g * nb;
        uint64_t m = 0;
        if (g < G) {
            const double b1x = L.X[e], b1y = L.Y[e], b2x = L.X[e + 1], b2y = L.Y[e + 1];
            for (int c = g; c < nc; c += G)
                if (lsmf(b1x, b1y, b2x, b2y, L.X[SP_C0 + c], L.Y[SP_C0 + c], L.X[SP_C0 + c + 1], L.Y[SP_C0 + c + 1]))
                    m |= 1ull << c;
        }
        boxes = m;
        for (int k = 1; k < G; ++k) boxes |= __shfl((unsigned long long)m, (lane + k * nb) & (WAVE - 1), WAVE);
        if (lane >= nb) boxes = 0;
    }
    // ---- the pairs that intersect, 64 tests at a time, in (base edge, overlay edge) order ----
    int I = 0;
    bool alpha_bad = false;
    {
        int tests, f = wave_excl(__popcll(boxes), lane, tests);
        for (int t0 = 0; t0 < tests; t0 += WAVE) {
            for (; boxes && f < t0 + WAVE; boxes &= boxes - 1, ++f)
                L.cand[f - t0] = uint16_t((lane << 6) | (__ffsll((unsigned long long)boxes) - 1));
            step();
            int t = 0, e = 0, c = 0;
            double al = 0.0, be = 0.0, x = 0.0, y = 0.0;
            if (t0 + lane < tests) {
                e = L.cand[lane] >> 6;
                c = L.cand[lane] & 63;
                const double b1x = L.X[e], b1y = L.Y[e], b2x = L.X[e + 1], b2y = L.Y[e + 1];
                const double c1x = L.X[SP_C0 + c], c1y = L.Y[SP_C0 + c];
                t = classify(b1x, b1y, b2x, b2y, c1x, c1y, L.X[SP_C0 + c + 1], L.Y[SP_C0 + c + 1], al, be);
                intersection_point(t, al, b1x, b1y, b2x, b2y, c1x, c1y, x, y);
            }
            const uint64_t hit = __ballot(t != 0);
            const int p = I + below(hit);
            if (t != 0) {
                alpha_bad |= !alpha_in_range(al) || !alpha_in_range(be);
                if (p < SP_I) {
                    L.pe[0][p] = uint8_t(e);
                    L.pe[1][p] = uint8_t(c);
                    L.pt[p] = uint8_t(t);
                    L.X[SP_P0 + p] = x;
                    L.Y[SP_P0 + p] = y;
                    L.qa[p] = alpha_to_int(al);
                    L.qb[p] = alpha_to_int(be);
                }
            }
            I += __popcll(hit);
            step();
        }
    }
    if (I > SP_I) return F_PAIRS;
    if (__ballot(alpha_bad)) return F_ALPHA;

    // ---- both sides' orders by (edge, parameter modulo 1e9, pair) and the counts per edge
    // (countEdgeIntersections, clip:522-601): a lane per pair and per edge, the other pairs read lane by lane ----
    int ndt0 = 0, ndt1 = 0; // inserted intersections of either side
    {
        int cB = 0, cC = 0, nB = 0, nC = 0;
        for (int p0 = 0; p0 < I || p0 == 0; p0 += WAVE) {
            const int p = p0 + lane;
            uint64_t kB = 0, kC = 0;
            if (p < I) {
                kB = (uint64_t(L.pe[0][p]) << 32) | uint32_t(L.qa[p] % 1000000000);
                kC = (uint64_t(L.pe[1][p]) << 32) | uint32_t(L.qb[p] % 1000000000);
            }
            int rB = 0, rC = 0;
            for (int q0 = 0; q0 < I; q0 += WAVE) {
                const int q = q0 + lane;
                uint64_t oB = kB, oC = kC;
                int fl = 0;
                if (q < I) {
                    if (q0 != p0) {
                        oB = (uint64_t(L.pe[0][q]) << 32) | uint32_t(L.qa[q] % 1000000000);
                        oC = (uint64_t(L.pe[1][q]) << 32) | uint32_t(L.qb[q] % 1000000000);
                    }
                    fl = (nondeg_b(L.pt[q]) ? 1 : 0) | (nondeg_c(L.pt[q]) ? 2 : 0);
                }
                const uint64_t insB = __ballot(fl & 1), insC = __ballot(fl & 2);
                const int nq = min(WAVE, I - q0);
                for (int i = 0; i < nq; ++i) {
                    const uint64_t vB = lane64(oB, i), vC = lane64(oC, i);
                    const bool before = q0 + i < p;
                    rB += (vB < kB || (vB == kB && before)) ? 1 : 0;
                    rC += (vC < kC || (vC == kC && before)) ? 1 : 0;
                    if (p0 == 0) {
                        const bool eB = int(vB >> 32) < lane, eC = int(vC >> 32) < lane;
                        cB += eB ? 1 : 0;
                        cC += eC ? 1 : 0;
                        nB += eB ? int((insB >> i) & 1u) : 0;
                        nC += eC ? int((insC >> i) & 1u) : 0;
                    }
                }
                if (p0 == 0) {
                    ndt0 += __popcll(insB);
                    ndt1 += __popcll(insC);
                }
            }
            if (p < I) {
                L.srt[0][rB] = uint8_t(p);
                L.srt[1][rC] = uint8_t(p);
            }
        }
        if (lane < nb) {
            L.cnt[0][lane] = uint8_t(cB);
            L.nd[0][lane] = uint8_t(nB);
        }
        if (lane < nc) {
            L.cnt[1][lane] = uint8_t(cC);
            L.nd[1][lane] = uint8_t(nC);
        }
        if (lane < 2) {
            L.cnt[lane][lane ? nc : nb] = uint8_t(I);
            L.nd[lane][lane ? nc : nb] = uint8_t(lane ? ndt1 : ndt0);
        }
    }
    const int n0 = nb + ndt0, n1 = nc + ndt1; // augmented ring sizes
    for (int s = lane; s < n0; s += WAVE) L.nb[0][s] = SP_NONE;
    for (int s = lane; s < n1; s += WAVE) L.nb[1][s] = SP_NONE;
    step();

    // ---- augmented rings (copyIntersectionsParallel, oacc:7508-7664): every ring vertex has a slot, a
    // degenerate first intersection of an edge takes its first vertex's, the others follow in order while
    // the edge has slots for them ----
    bool walk = false;
#pragma unroll
    for (int side = 0; side < 2; ++side) {
        const int ne = side ? nc : nb, v0 = side ? SP_C0 : 0;
        if (lane < ne) L.code[side][lane + L.nd[side][lane]] = uint16_t(v0 + lane);
        for (int t = lane; t < I; t += WAVE) {
            const int p = L.srt[side][t], e = L.pe[side][p];
            const int g0 = L.cnt[side][e], s0 = e + L.nd[side][e], room = L.nd[side][e + 1] - L.nd[side][e];
            const int t0 = L.pt[L.srt[side][g0]];
            const int k = (side ? degen_c_first(t0) : degen_b_first(t0)) ? 1 : 0;
            const int i = t - g0;
            int s = SP_NONE;
            if (i < k) {
                s = s0;
            } else if (i - k < room) {
                s = s0 + 1 + i - k;
                L.code[side][s] = uint16_t(SP_P0 + p);
                // The reference matches the augmented arrays to the rings by coordinates (copyToLinkedList,
                // clip:606-695); that walk keeps slot order unless an inserted intersection equals the next
                // ring vertex, which falls back.
                const int nx = v0 + (e + 1 == ne ? 0 : e + 1);
                if (L.X[SP_P0 + p] == L.X[nx] && L.Y[SP_P0 + p] == L.Y[nx]) walk = true;
            }
            L.ps[side][p] = uint8_t(s);
        }
    }
    step();
    // every pair holds a slot on both rings, else the reference leaves it out (undefined)
    bool bad = false;
    for (int p = lane; p < I; p += WAVE) {
        const int s = L.ps[0][p], q = L.ps[1][p];
        if (s == SP_NONE || q == SP_NONE) {
            bad = true;
        } else {
            L.nb[0][s] = uint8_t(q);
            L.nb[1][q] = uint8_t(s);
        }
    }
    if (__ballot(bad)) return F_SLOT;
    step();

    // ---- initial labels (calculateInitLabelParallel, oacc:7925-7988), a lane per pair ----
    bool odd_label = false;
    for (int p = lane; p < I; p += WAVE) {
        const int i = L.ps[0][p], q = L.ps[1][p];
        const int tm = i == 0 ? n0 - 1 : i - 1, tp = i + 1 == n0 ? 0 : i + 1;
        const int qm = q == 0 ? n1 - 1 : q - 1, qp = q + 1 == n1 ? 0 : q + 1;
        const int pMN = L.nb[0][tm] != SP_NONE ? L.nb[0][tm] : SP_NOV;
        const int pPN = L.nb[0][tp] != SP_NONE ? L.nb[0][tp] : SP_NOV;
        const int cm = L.code[0][tm], ci = L.code[0][i], cp = L.code[0][tp], dm = L.code[1][qm], dp = L.code[1][qp];
        const int lab = label_of(pMN, pPN, qm, qp, L.X[dm], L.Y[dm], L.X[dp], L.Y[dp], L.X[cm], L.Y[cm], L.X[ci],
                                 L.Y[ci], L.X[cp], L.Y[cp]);
        L.lab[i] = uint8_t(lab);
        if (lab != L_CROSSING && lab != L_BOUNCING) odd_label = true;
    }
    if (__ballot(walk)) return F_WALK;
    // labels other than CROSSING / BOUNCING (chains, ON labels, no rule) take the staged path
    if (__ballot(odd_label)) return F_LABEL;
    step();

    // ---- labelIntersections2: crossings, special cases, entry/exit ----
    Slots inter[2], cross[2];
#pragma unroll
    for (int side = 0; side < 2; ++side)
#pragma unroll
        for (int k = 0; k < SP_WORDS; ++k) {
            const int s = 64 * k + lane;
            bool in = false, cr = false;
            if (s < (side ? n1 : n0)) {
                const int q = L.nb[side][s];
                in = q != SP_NONE;
                cr = in && L.lab[side ? q : s] == L_CROSSING;
            }
            inter[side].w[k] = __ballot(in);
            cross[side].w[k] = __ballot(cr);
        }
    const bool crossing = any(cross[0]); // a crossing has its partner on the other ring
    route = crossing ? 0 : 1;
    int top = 0, nr = 0; // output vertices and rings
    Slots exits0, exits1;   // crossings met in the EXIT state
    Slots split0, split1;   // bouncing vertices met in it
    const int v0 = first_plain(inter[0], n0), v1 = first_plain(inter[1], n1);
    if (v0 < 0 || v1 < 0) return F_PLAIN;
    const int c0 = L.code[0][v0], c1 = L.code[1][v1];
    const bool in0 = point_in_ring(L, L.code[1], n1, L.X[c0], L.Y[c0], lane);
    const bool in1 = point_in_ring(L, L.code[0], n0, L.X[c1], L.Y[c1], lane);
    if (crossing) {
        // 4) entry/exit
        states(cross[0], inter[0], v0, in0, lane, exits0, split0);
        states(cross[1], inter[1], v1, in1, lane, exits1, split1);
    } else {
        // 3.5) a ring without crossing vertices is an output ring when inside the other
        for (int side = 0; side < 2; ++side) {
            const int n = side ? n1 : n0;
            if (!(side ? in1 : in0)) continue;
            for (int s = lane; s < n; s += WAVE) L.ord[top + s] = L.code[side][s];
            if (lane == 0) {
                L.rbeg[nr] = uint16_t(top);
                L.rlen[nr] = uint16_t(n);
            }
            top += n;
            ++nr;
        }
    }

    int fail = 0;
    if (crossing) {
        // 5) a P candidate whose partner is a Q candidate is split: staged path
        bool sp = false;
        for (int p = lane; p < I; p += WAVE) sp |= has(split0, L.ps[0][p]) && has(split1, L.ps[1][p]);
        if (__ballot(sp)) return F_SPLIT;
        // ---- createResult2, a piece between two crossings at a time: the whole wave walks the crossings'
        // bits and copies the piece's slots ----
        Slots left = cross[0]; // crossings of P that start a ring unless a walk passes them
        const int bound = 4 * (n0 + n1) + 16;
        while (any(left) && !fail) {
            const int I0 = lowest(left), beg = top;
            if (nr >= SP_OUTR) {
                fail = F_OUT;
                break;
            }
            int V = I0, side = 0;
            drop(left, V);
            const Slots start = only(I0);
            for (;;) {
                const int n = side ? n1 : n0;
                const Slots cs = pick(side, cross[0], cross[1]), xs = pick(side, exits0, exits1);
                const bool fwd = !has(xs, V); // on from an entry, back from an exit, to the next of the other kind
                Slots stop;
#pragma unroll
                for (int k = 0; k < SP_WORDS; ++k) // the start ends the walk in either state
                    stop.w[k] = (fwd ? xs.w[k] : cs.w[k] & ~xs.w[k]) | (side == 0 ? start.w[k] : 0ull);
                if (!any(stop)) {
                    fail = F_TRAV;
                    break;
                }
                const int W = next_slot(stop, V, fwd);
                int len = fwd ? W - V : V - W;
                if (len <= 0) len += n;
                if (top + len > SP_OUTV) {
                    fail = F_OUT;
                    break;
                }
                if (top + len - beg > bound) {
                    fail = F_TRAV;
                    break;
                }
                for (int i = lane; i < len; i += WAVE) {
                    int s = fwd ? V + 1 + i : V - 1 - i;
                    if (s >= n) s -= n;
                    if (s < 0) s += n;
                    L.ord[top + i] = L.code[side][s];
                }
                if (side == 0) { // the slots passed start no ring any more
#pragma unroll
                    for (int k = 0; k < SP_WORDS; ++k) {
                        const int s = 64 * k + lane;
                        int d = fwd ? s - V : V - s;
                        if (d <= 0) d += n;
                        left.w[k] &= ~__ballot(d <= len);
                    }
                }
                top += len;
                if (side == 0 && W == I0) break;
                V = __builtin_amdgcn_readfirstlane(int(L.nb[side][W]));
                side ^= 1;
                if (side == 0) {
                    drop(left, V);
                    if (V == I0) break;
                }
            }
            if (lane == 0) {
                L.rbeg[nr] = uint16_t(beg);
                L.rlen[nr] = uint16_t(top - beg);
            }
            ++nr;
        }
    }
    if (fail) return fail;
    step();

    // ---- cleanUpResult2: vertices with |A(last kept, v, next)| < eps go, the first ones of a ring while
    // A(its last vertex, v, next) is that small; decided at once where no vertex goes, by one lane otherwise ----
    int rings = 0, verts = 0;
    for (int r = 0; r < nr; ++r) {
        const int beg = __builtin_amdgcn_readfirstlane(int(L.rbeg[r]));
        const int n = __builtin_amdgcn_readfirstlane(int(L.rlen[r])), last = n - 1;
        int root = -1;
        for (int s0 = 0; s0 < n && root < 0; s0 += WAVE) {
            const int s = s0 + lane;
            const bool ok = s < n && !flat(L, L.ord[beg + last], L.ord[beg + s], L.ord[beg + min(s + 1, last)]);
            const uint64_t m = __ballot(ok);
            if (m) root = s0 + __ffsll((unsigned long long)m) - 1;
        }
        if (root < 0) continue;
        bool gone = false;
        for (int s = root + 1 + lane; s < n; s += WAVE)
            gone |= flat(L, L.ord[beg + s - 1], L.ord[beg + s], L.ord[beg + (s == last ? root : s + 1)]);
        int len = n - root, at = beg + root;
        if (__ballot(gone)) {
            if (lane == 0) {
                int k = root, prev = L.ord[beg + root];
                const int first = prev;
                for (int s = root + 1; s < n; ++s) {
                    const int v = L.ord[beg + s];
                    if (flat(L, prev, v, s == last ? first : int(L.ord[beg + s + 1]))) continue;
                    L.ord[beg + ++k] = uint16_t(v);
                    prev = v;
                }
                len = k + 1 - root;
            }
            len = __builtin_amdgcn_readfirstlane(len);
            step();
        }
        if (lane == 0) { // r >= rings: this ring's own entry has been read
            L.rbeg[rings] = uint16_t(at);
            L.rlen[rings] = uint16_t(len);
        }
        step();
        if (!a.out4) {
            const int64_t o = int64_t(j) * SP_OUTV + verts;
            for (int i = lane; i < len; i += WAVE) {
                const int v = L.ord[at + i];
                a.out_x[o + i] = L.X[v];
                a.out_y[o + i] = L.Y[v];
            }
            if (lane == 0) a.out_len[int64_t(j) * SP_OUTR + rings] = len;
        }
        verts += len;
        ++rings;
    }
    nv_out = verts;
    nr_out = rings;
    if (a.out4) pair_areas(a, L, j, nb, nc, rings, lane);
    return 0;
}

// One wave per pair and a block per wave, handed out by the hardware as LDS
// comes free (a queue of pairs costs an atomic on one address per pair).
__global__ __launch_bounds__(WAVE, 5) void k_small_pairs(SmallArgs a) {
    __shared__ SmallLDS L;
    const int lane = threadIdx.x, j = blockIdx.x;
    int route = 0, nv = 0, nr = 0;
    const int f = clip_pair(a, L, j, lane, route, nv, nr);
    if (lane == 0) {
        a.fail[j] = f;
        a.route[j] = route;
        a.job_nv[j] = f ? 0 : nv;
        a.job_nr[j] = f ? 0 : nr;
        if (f && a.anyfail) atomicOr(a.anyfail, 1u);
    }
}

// output rings of every job at their final offsets: one block per job
__global__ void k_small_emit(int J, const int *__restrict__ voff, const int *__restrict__ roff,
                             const int *__restrict__ job_nr, const double *__restrict__ ox,
                             const double *__restrict__ oy, const int *__restrict__ olen, double *rx, double *ry,
                             int *ring_off) {
    const int j = blockIdx.x;
    const int v0 = voff[j], nv = voff[j + 1] - v0, r0 = roff[j], nr = job_nr[j];
    for (int i = threadIdx.x; i < nv; i += blockDim.x) {
        rx[v0 + i] = ox[int64_t(j) * SP_OUTV + i];
        ry[v0 + i] = oy[int64_t(j) * SP_OUTV + i];
    }
    if (threadIdx.x == 0) {
        int at = v0;
        for (int r = 0; r < nr; ++r) {
            ring_off[r0 + r] = at;
            at += olen[int64_t(j) * SP_OUTR + r];
        }
        if (j == J - 1) ring_off[roff[J]] = voff[J]; // the closing entry
    }
}

// rings given back to back without closing vertices (the set_pairs layout)
// into the resident layout with the closing vertex; one thread per vertex
__global__ void k_pairs_layout(const double *__restrict__ xy, int64_t n, const int *__restrict__ in_off,
                               const int *__restrict__ out_off, int R, double *out) {
    const int64_t g = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (g >= n) return;
    const int r = seg_of_wave(in_off, R, g);
    const int local = int(g - in_off[r]);
    const double x = xy[2 * g], y = xy[2 * g + 1];
    const int64_t d = int64_t(out_off[r]) + local;
    out[2 * d] = x;
    out[2 * d + 1] = y;
    if (local == 0) {
        const int64_t cl = int64_t(out_off[r]) + (in_off[r + 1] - in_off[r]);
        out[2 * cl] = x;
        out[2 * cl + 1] = y;
    }
}

struct SmallScratch {
    DBuf<int> jobs, fail, route, nv, nr, voff, olen;
    DBuf<double> ox, oy;
};

SmallScratch &sscratch() {
    thread_local SmallScratch *p = new SmallScratch();
    return *p;
}

} // namespace

bool small_batch_eligible(const Ctx &c, int k0, int k1) {
    if (!c.paired || c.prov || !c.small_fused || c.uni) return false;
    for (int k = k0; k <= k1; ++k)
        if (c.bsz[k - 1] > SP_NV || c.csz[k - 1] > SP_NV) return false;
    return true;
}

bool clip_small_batch(Ctx &c, int k0, int k1) {
    hipStream_t s = c.stream;
    const int J = k1 - k0 + 1;
    SmallScratch &S = sscratch();
    c.hold_scratch(); // another context's batch may still be read out of it
    std::vector<int> h(4 * size_t(J));
    for (int j = 0; j < J; ++j) {
        const int k = k0 + j, br = job_base(c, k);
        h[j] = c.bvoff[br];
        h[J + j] = c.bsz[br];
        h[2 * J + j] = c.coff[k - 1];
        h[3 * J + j] = c.csz[k - 1];
    }
    int *dj = S.jobs.ensure(4 * size_t(J));
    c.upload(dj, h.data(), sizeof(int) * h.size());
    SmallArgs a;
    a.J = J;
    a.bvoff = dj;
    a.nb = dj + J;
    a.cvoff = dj + 2 * J;
    a.nc = dj + 3 * J;
    a.bpoly = c.bpoly;
    a.cpoly = c.cpoly;
    a.fail = S.fail.ensure(J);
    a.route = S.route.ensure(J);
    a.job_nv = S.nv.ensure(size_t(J) + 1);
    a.job_nr = S.nr.ensure(size_t(J) + 1);
    a.out_x = S.ox.ensure(size_t(J) * SP_OUTV);
    a.out_y = S.oy.ensure(size_t(J) * SP_OUTV);
    a.out_len = S.olen.ensure(size_t(J) * SP_OUTR);
    {
        FillBatch fb(s);
        fb.add(a.job_nv + J, 1, 0u);
        fb.add(a.job_nr + J, 1, 0u);
        fb.flush();
    }
    a.out4 = nullptr;
    a.anyfail = nullptr;
    k_small_pairs<<<J, WAVE, 0, s>>>(a);
    SC_HIP(hipGetLastError());
    int *voff = S.voff.ensure(size_t(J) + 1), *roff = c.jobs.d_ring.ensure(size_t(J) + 1); // rings: for the areas too
    scan_exclusive_u32_2(reinterpret_cast<const uint32_t *>(a.job_nv), reinterpret_cast<uint32_t *>(voff), J + 1,
                         nullptr, reinterpret_cast<const uint32_t *>(a.job_nr), reinterpret_cast<uint32_t *>(roff),
                         J + 1, nullptr, s);
    // one read-back: ring offsets per job, vertex total, fallback reasons, routes
    JobSet &js = c.jobs;
    js.ring_off.assign(size_t(J) + 1, 0);
    std::vector<int> fails(static_cast<size_t>(J)), routes(static_cast<size_t>(J));
    int NV = 0;
    {
        ReadBack rb(c);
        rb.add(js.ring_off.data(), static_cast<const int *>(roff), size_t(J) + 1);
        rb.add(&NV, static_cast<const int *>(voff + J), 1);
        rb.add(fails.data(), static_cast<const int *>(a.fail), size_t(J));
        rb.add(routes.data(), static_cast<const int *>(a.route), size_t(J));
        rb.run();
    }
    int any = 0;
    for (int f : fails) any |= f;
    c.small_fail = any;
    if (any) return false; // the staged path reruns the batch
    const int NR = js.ring_off[J];
    c.d_ring_off.ensure(size_t(NR) + 1);
    c.d_ring_x.ensure(size_t(NV > 0 ? NV : 1));
    c.d_ring_y.ensure(size_t(NV > 0 ? NV : 1));
    c.hold_scratch(); // read after the return: a wait here costs 16,384 pairs 27 us of 315
    k_small_emit<<<J, 256, 0, s>>>(J, voff, roff, a.job_nr, a.out_x, a.out_y, a.out_len, c.d_ring_x, c.d_ring_y,
                                   c.d_ring_off);
    SC_HIP(hipGetLastError());
    c.nrings = NR;
    c.n_out = NV;
    c.long_rings = false;
    c.undefined = 0;
    c.cur_k = J == 1 ? k0 : 0;
    c.flags_pending = false;
    js.k0 = k0;
    js.J = J;
    js.resident = true;
    js.prov = false;
    js.flags.assign(size_t(J), 0);
    js.route = routes;
    js.reason.assign(size_t(J), 0);
    return true;
}

void pairs_graph_reset(Ctx &c) {
    Ctx::PairsGraph &g = c.pg;
    if (g.exec) (void)hipGraphExecDestroy(g.exec);
    if (g.graph) (void)hipGraphDestroy(g.graph);
    g.exec = nullptr;
    g.graph = nullptr;
    g.bxy = g.cxy = nullptr;
    g.out4 = nullptr;
}

void pairs_area_graph(Ctx &c, const double *bxy, const double *cxy, double *out4) {
    SC_REQUIRE(c.paired && c.K >= 1, SC_ESTATE, "pairs not set (segclip_set_pairs)");
    SC_REQUIRE(!c.uni, SC_ESTATE, "the area / IoU graph is defined for the intersection");
    SC_REQUIRE(bxy && cxy && out4, SC_EINVAL, "null pointer");
    for (int k = 0; k < c.K; ++k)
        SC_REQUIRE(c.bsz[k] <= SP_NV && c.csz[k] <= SP_NV, SC_EINVAL,
                   "the graph forward takes rings of at most 64 vertices");
    hipStream_t s = c.stream;
    const int J = c.K;
    Ctx::PairsGraph &g = c.pg;
    if (!g.exec || g.bxy != bxy || g.cxy != cxy || g.out4 != out4) {
        pairs_graph_reset(c);
        // tables: job (bvoff, nb, cvoff, nc), base input / output offsets (J+1, J), overlay ones (J+1, J)
        std::vector<int> h(4 * size_t(J) + 2 * (2 * size_t(J) + 1));
        int *t = h.data();
        for (int j = 0; j < J; ++j) {
            t[j] = c.bvoff[j];
            t[J + j] = c.bsz[j];
            t[2 * J + j] = c.coff[j];
            t[3 * J + j] = c.csz[j];
        }
        int *bin = t + 4 * J, *bout = bin + J + 1, *cin = bout + J, *cout = cin + J + 1;
        for (int j = 0; j <= J; ++j) {
            bin[j] = c.beoff[j];
            cin[j] = c.eoff[j] - c.nb;
            if (j < J) {
                bout[j] = c.bvoff[j];
                cout[j] = c.coff[j];
            }
        }
        int *dt = g.tables.ensure(h.size());
        SC_HIP(hipMemcpyAsync(dt, h.data(), sizeof(int) * h.size(), hipMemcpyHostToDevice, s));
        uint32_t *words = g.words.ensure(1);
        SmallArgs a;
        a.J = J;
        a.bvoff = dt;
        a.nb = dt + J;
        a.cvoff = dt + 2 * J;
        a.nc = dt + 3 * J;
        a.bpoly = c.bpoly;
        a.cpoly = c.cpoly;
        a.anyfail = words;
        a.fail = g.fail.ensure(J);
        a.route = g.route.ensure(J);
        a.job_nv = g.nv.ensure(size_t(J) + 1);
        a.job_nr = g.nr.ensure(size_t(J) + 1);
        a.out_x = a.out_y = nullptr; // areas only
        a.out_len = nullptr;
        a.out4 = out4;
        SC_HIP(hipStreamSynchronize(s)); // the tables are on the device before the capture
        const int64_t nbt = c.nb, nct = c.nct;
        const int dbin = int(bin - t), dbout = int(bout - t), dcin = int(cin - t), dcout = int(cout - t);
        SC_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeRelaxed));
        hipGraph_t graph = nullptr;
        try {
            // fill kernels, no memset nodes, inside the graph
            FillBatch fb(s);
            fb.add(words, 1, 0u);
            fb.flush();
            k_pairs_layout<<<unsigned(ceil_div(nbt, 256)), 256, 0, s>>>(bxy, nbt, dt + dbin, dt + dbout, J,
                                                                        c.bpoly);
            k_pairs_layout<<<unsigned(ceil_div(nct, 256)), 256, 0, s>>>(cxy, nct, dt + dcin, dt + dcout, J,
                                                                        c.cpoly);
            k_small_pairs<<<J, WAVE, 0, s>>>(a);
            SC_HIP(hipGetLastError());
        } catch (...) {
            (void)hipStreamEndCapture(s, &graph); // the stream leaves capture mode either way
            if (graph) (void)hipGraphDestroy(graph);
            throw;
        }
        SC_HIP(hipStreamEndCapture(s, &graph));
        g.graph = graph;
        SC_HIP(hipGraphInstantiateWithFlags(&g.exec, g.graph, 0));
        g.bxy = bxy;
        g.cxy = cxy;
        g.out4 = out4;
    }
    SC_HIP(hipGraphLaunch(g.exec, s));
    rings_moved(c);
    uint32_t anyfail = 0;
    {
        ReadBack rb(c);
        rb.add(&anyfail, static_cast<const uint32_t *>(g.words.p), 1);
        rb.run();
    }
    if (!anyfail) return;
    // some pair is not covered: the staged path on the same rings (the
    // context's rings now hold the caller's coordinates; the set-up is redone
    // for them, which drops the graph)
    std::vector<int> bsz = c.bsz, csz = c.csz;
    ctx_set_pairs(c, bxy, bsz.data(), cxy, csz.data(), J, true);
    const int keep = c.small_fused;
    c.small_fused = 0;
    try {
        clip_jobs(c, 1, J);
    } catch (...) {
        c.small_fused = keep;
        throw;
    }
    c.small_fused = keep;
    batch_area(c, out4);
    c.wait(); // out4 is written on return, and the thread's scratch is free
    c.small_fail = 1;
}

} // namespace sc
