// sc_foster.hip -- Foster/Greiner-Hormann labelling, traversal and clean-up
// (rows A16-A17) on the GPU, for a batch of jobs in the same launches.
//
// Reference: copyToLinkedList (src/clip.cpp:606-695), labelIntersections2,
// createResult2, cleanUpResult2 (foster/polyclip.h:337-787), for the
// intersection (UNION = false) and, on the sequential route, the union.  The
// augmented rings built by post_jobs are the linked lists of copyToLinkedList laid out in ring order: slot i of a job's base
// ring P is followed by slot i+1 (mod its length), likewise for the overlay
// ring Q; a slot is an intersection vertex when its alpha (P) or neighbour
// (Q) is set.  Job j owns P slots [AB[j], AB[j+1]) and Q slots
// [AC[j], AC[j+1]); neighbour links are 1-based within the job.
//
// Every job takes one of three routes:
//  - crossing (every label CROSSING or BOUNCING, a plain vertex on both
//    rings, crossings alternate, no interior bouncing pair): the entry/exit
//    status of a crossing vertex is the parity of the crossings met since the
//    first plain vertex (one prefix count); a traversal piece runs from a
//    crossing vertex to the next crossing vertex in the walking direction,
//    then jumps to the neighbour of that vertex on the other ring.  Pieces
//    form cycles; a cycle's output component is started at its base-ring
//    vertex that comes first in base-ring order, and the pieces of a
//    component are laid out by their distance from that start (both found by
//    walks between every eighth crossing and doubling over those; by
//    doubling alone for few crossings);
//  - no crossing (same conditions, no crossing vertex): each ring is output
//    when its first plain vertex lies inside the other ring;
//  - sequential: everything else -- intersection chains (LEFT_ON ...
//    ON_RIGHT), split bouncing pairs, rings made only of intersections,
//    inconsistent labels, the union -- runs the reference's sequential
//    algorithm: large jobs over the whole device (sc_walk.hip), small ones
//    and what that leaves in one block each.
// The outputs of all jobs are laid out job after job, then cleaned up.
//
// Clean-up: the reference removes, in one pass from the root, every vertex
// nearly collinear (|A| < 1e-9) with the last kept vertex and its successor,
// after first dropping collinear roots.  The decisions are computed as the
// unique fixed point of keep[i] = |A(last kept before i, i, i+1)| >= eps,
// iterated in parallel from the guess "predecessor kept"; the fixed point
// equals the sequential result because it is determined left to right.  A wave
// decides a tile in order from a guess of the last vertex kept before it (one
// window of vertices further back decides the guess), skipping runs of kept
// vertices by ballots; a tile whose guess was wrong is decided again.
//
// Provenance: every output vertex carries the slot it came from (a P slot g
// as g, a Q slot g as ~g, none as SRC_NONE) for the area gradient.
#include "sc_ctx.hpp"
#include "sc_fp64.hpp"
#include "sc_seg.hpp"
#include "sc_seqroute.hpp"

#include <algorithm>
#include <climits>

namespace sc {

namespace {

constexpr int BLK = 256;
inline unsigned grid_for(int64_t n, int per = BLK) {
    int64_t g = ceil_div(n, per);
    if (g < 1) g = 1;
    return unsigned(g);
}

// reasons for taking the sequential route
enum : int { SLOW_LABEL = 1, SLOW_NOPLAIN = 2, SLOW_ODD = 4, SLOW_SPLIT = 8, SLOW_LINK = 16, SLOW_UNION = 32 };
// routes
enum : int { K_CROSS = 0, K_NOCROSS = 1, K_SEQ = 2 };

// one side (all P rings or all Q rings) of a batch
struct Side {
    const int *off;  // J+1 slot offsets of this side's rings
    const int *ooff; // J+1 slot offsets of the other side's rings
    const double *x, *y;
    const int *lab, *nbr, *av; // av null: intersection iff nbr set
};

__device__ inline bool inter_at(const Side &s, int64_t i) { return s.av ? s.av[i] != -100 : s.nbr[i] != -100; }

// Crossing flags with their closing entry, label and link checks of both sides
// (blockIdx.y 0: P, 1: Q), and the first plain vertex of each job's rings
// (blockIdx.y 2: P, skipped for the sparse base; 3: Q).  At ordinary sizes the
// stage is bound by its launches, not by their work, so steps of both sides share
// one: two stars of 1,000 and 1,100 vertices are labelled in 0.24 ms instead of
// 0.39, 20,000 against 51,000 in 0.30 instead of 0.39.
struct ClassifyArgs {
    Side s[2];
    int J, per;
    int64_t n[2];  // flags of the sides: their slots or more
    const int *pj; // jobs of a sparse base side's slots (its pairs' jobs), else null
    uint32_t *cross[2];
    int *slow, *first[2];
    int *bounce; // per job: its base side has a bouncing vertex
};
__global__ __launch_bounds__(BLK) void k_jclassify(ClassifyArgs a) {
    const int y = blockIdx.y & 1;
    const Side &s = a.s[y];
    const int lane = threadIdx.x & (WAVE - 1);
    if (blockIdx.y < 2) {
        const int *pj = y ? nullptr : a.pj;
        const int64_t n = s.off[a.J];
        WaveSpan w(s.off, a.J, pj ? 0 : n, a.per);
        for (int q = 0; q < a.per && w.at <= a.n[y]; ++q, w.at += WAVE) {
            const int64_t i = w.at + lane;
            const int js = pj ? 0 : w.of(s.off, a.J, lane);
            if (i > a.n[y]) continue;
            uint32_t c = 0;
            if (i < n && inter_at(s, i)) {
                const int j = pj ? pj[i] : js;
                const int lab = s.lab[i];
                if (lab != L_CROSSING && lab != L_BOUNCING) atomicOr(&a.slow[j], SLOW_LABEL);
                const int nb = s.nbr[i];
                if (nb < 1 || nb > s.ooff[j + 1] - s.ooff[j]) atomicOr(&a.slow[j], SLOW_LINK);
                c = lab == L_CROSSING ? 1u : 0u;
                if (y == 0 && lab == L_BOUNCING) a.bounce[j] = 1;
            }
            a.cross[y][i] = c;
        }
        return;
    }
    // first plain vertex (local index, -1 if none): one wave per job
    const int j = int((int64_t(blockIdx.x) * blockDim.x + threadIdx.x) / WAVE);
    if (!a.first[y] || j >= a.J) return; // whole wave
    const int64_t b = s.off[j], e = s.off[j + 1];
    int res = -1;
    for (int64_t base = b; base < e; base += WAVE) {
        const int64_t v = base + lane;
        const uint64_t m = __ballot(v < e && !inter_at(s, v));
        if (m) {
            res = int(base - b) + __ffsll((unsigned long long)m) - 1;
            break;
        }
    }
    if (lane == 0) a.first[y][j] = res;
}

// winding test of polygon::pointInPoly (polygon.h:435-457) of each job's
// query point (the other ring's first plain vertex) against this side's
// rings, summed per job; blockIdx.y picks the side (a null wind: not this way)
struct WindSide {
    Side r;
    Side from;        // the other side, whose first plain vertices are the query points
    const int *first;
    const double *q;  // or the points, x,y per job (sparse base side)
    int *wind;
};
struct JobState {
    int J;
    int uni; // the union: every job takes the sequential route
    const int *AB, *AC;
    int *slow, *firstP, *firstQ, *windP, *windQ, *kind, *mP, *mQ, *cP0, *cQ0;
    int *vP, *vQ; // crossings of the batch before each ring's first plain vertex
};
struct WindSides {
    WindSide s[2];
    int J, per;
    JobState st;
    const uint32_t *ccP, *ccQ;
    int sparse;
    SparseP sp;
    const int *flags;
};
// route of each job; first crossing index of each job on both sides (J+1 threads)
__device__ inline void decide(const WindSides &a, int j) {
    const JobState &s = a.st;
    const uint32_t *ccP = a.ccP, *ccQ = a.ccQ;
    if (j > s.J) return;
    s.cP0[j] = int(ccP[s.AB[j]]);
    s.cQ0[j] = int(ccQ[s.AC[j]]);
    if (j == s.J) return;
    int mp = int(ccP[s.AB[j + 1]] - ccP[s.AB[j]]), mq = int(ccQ[s.AC[j + 1]] - ccQ[s.AC[j]]);
    s.mP[j] = mp;
    s.mQ[j] = mq;
    int sl = s.slow[j];
    const int fp = s.firstP[j], fq = s.firstQ[j];
    if (fp < 0 || fq < 0) {
        sl |= SLOW_NOPLAIN;
    } else {
        // sparse: the slots before the first plain one are the job's first positions
        // (a flagged job's slots may not ascend: as the searches find it)
        s.vP[j] = int(ccP[!a.sparse ? s.AB[j] + fp : (a.flags[j] ? sp_lower(a.sp, j, fp) : a.sp.P0[j] + fp)]);
        s.vQ[j] = int(ccQ[s.AC[j] + fq]);
    }
    if (mp != mq || (mp & 1)) sl |= SLOW_ODD;
    if (s.uni) sl |= SLOW_UNION;
    s.slow[j] = sl;
    s.kind[j] = sl ? K_SEQ : (mp == 0 ? K_NOCROSS : K_CROSS);
}
__global__ __launch_bounds__(BLK) void k_jwinding(WindSides a) {
    if (blockIdx.y == 2) { // the routes need no winding and share the launch
        decide(a, blockIdx.x * blockDim.x + threadIdx.x);
        return;
    }
    const WindSide &z = a.s[blockIdx.y];
    if (!z.wind) return;
    const Side &r = z.r;
    const int64_t n = r.off[a.J];
    const int lane = threadIdx.x & (WAVE - 1);
    WaveSpan s(r.off, a.J, n, a.per);
    int sum = 0, of = s.seg; // terms of job 'of', not added yet
    auto add = [&]() {
        for (int d = WAVE / 2; d > 0; d >>= 1) sum += __shfl_down(sum, d, WAVE);
        if (lane == 0 && sum) atomicAdd(&z.wind[of], sum);
        sum = 0;
    };
    for (int q = 0; q < a.per && s.at < n; ++q, s.at += WAVE) {
        const int64_t i = s.at + lane;
        const int j = s.of(r.off, a.J, lane);
        int w = 0;
        const int fp = i < n ? z.first[j] : -1;
        if (fp >= 0) {
            const int64_t nx = i + 1 == r.off[j + 1] ? r.off[j] : i + 1;
            const int64_t v = z.q ? 0 : int64_t(z.from.off[j]) + fp;
            const double qx = z.q ? z.q[2 * j] : z.from.x[v], qy = z.q ? z.q[2 * j + 1] : z.from.y[v];
            w = wind_edge(r.x[i], r.y[i], r.x[nx], r.y[nx], qx, qy);
        }
        const int j0 = __builtin_amdgcn_readfirstlane(j);
        if (j0 != of) {
            add();
            of = j0;
        }
        if (j0 == s.seg) { // the whole wave inside one job
            sum += w;
        } else {
            if (j == j0) sum += w;
            else if (w) atomicAdd(&z.wind[j], w);
        }
    }
    add();
}

// query points of a batch with a sparse base ring: each ring's first plain vertex
__global__ void k_query_pts(int J, Side Q, SparseP sp, const int *firstP, const int *firstQ, double *pq, double *qq,
                            int *qok) {
    int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= J) return;
    const int fp = firstP[j], fq = firstQ[j];
    qok[j] = fq >= 0;
    double x = 0, y = 0;
    if (fp >= 0) {
        const SlotInfo si = sp_slot(sp, j, fp);
        x = si.x;
        y = si.y;
    }
    pq[2 * j] = x;
    pq[2 * j + 1] = y;
    x = y = 0;
    if (fq >= 0) {
        x = Q.x[Q.off[j] + fq];
        y = Q.y[Q.off[j] + fq];
    }
    qq[2 * j] = x;
    qq[2 * j + 1] = y;
}

// ---- sparse base ring (one-to-many batches) ----

// first plain slot of each job's virtual base ring: the first slot not held by
// an intersection; one wave per job over its ascending slot list
__global__ __launch_bounds__(BLK) void k_sp_first_plain(SparseP sp, int J, int *first) {
    const int j = int((int64_t(blockIdx.x) * blockDim.x + threadIdx.x) / WAVE);
    const int lane = threadIdx.x & (WAVE - 1);
    if (j >= J) return; // whole wave
    const int a = sp.P0[j], b = sp.P0[j + 1];
    const int nslots = sp.AB[j + 1] - sp.AB[j];
    int res = b - a < nslots ? b - a : -1;
    for (int base = a; base < b; base += WAVE) {
        const int i = base + lane;
        const bool gap = i < b && sp.slot[i] != i - a;
        const uint64_t m = __ballot(gap);
        if (m) {
            res = base - a + __ffsll((unsigned long long)m) - 1;
            break;
        }
    }
    if (lane == 0) first[j] = res < nslots ? res : -1;
}

// winding of each job's query point against every base edge (all jobs share
// the base ring); corrected below on the edges that hold intersections
constexpr int WCH = 4096; // base edges per block
__global__ __launch_bounds__(BLK) void k_sp_wind_base(int J, int nb, const double *__restrict__ bpoly,
                                                      const double *__restrict__ qq, const int *__restrict__ qok,
                                                      int *wind) {
    __shared__ int sh[BLK / WAVE];
    const int chunks = (nb + WCH - 1) / WCH;
    const int j = blockIdx.x / chunks, ch = blockIdx.x % chunks;
    if (j >= J || !qok[j]) return; // whole block
    const double rx = qq[2 * j], ry = qq[2 * j + 1];
    const int e1 = min(nb, (ch + 1) * WCH);
    int w = 0;
    for (int e = ch * WCH + threadIdx.x; e < e1; e += BLK) {
        const double *P = bpoly + 2 * int64_t(e);
        w += wind_edge(P[0], P[1], P[2], P[3], rx, ry);
    }
    for (int d = WAVE / 2; d > 0; d >>= 1) w += __shfl_down(w, d, WAVE);
    if ((threadIdx.x & (WAVE - 1)) == 0) sh[threadIdx.x / WAVE] = w;
    __syncthreads();
    if (threadIdx.x == 0) {
        int t = 0;
        for (int k = 0; k < BLK / WAVE; ++k) t += sh[k];
        if (t) atomicAdd(&wind[j], t);
    }
}

// an edge split by non-degenerate intersections: replace its full-edge term
// by the terms of its pieces (source vertex -> X1 -> ... -> next vertex)
__global__ void k_sp_wind_fix(int I, const int *__restrict__ pj, SparseP sp, const double *__restrict__ qq,
                              const int *__restrict__ qok, int *wind) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= I) return;
    const int j = pj[i];
    if (!qok[j]) return;
    const int e = sp.edge[i];
    auto is_nd = [&](int k) { return sp.slot[k] >= 0 && sp.slot[k] == sp.edge[k] + 1 + sp.ndx[k]; };
    if (!is_nd(i)) return;
    // Base edge e = (a, b) with the run of points p1..pm inserted on it counts
    // -w(a, b) + w(a, p1) + w(p1, p2) + ... + w(pm, b) instead of w(a, b):
    // each point adds the term of the piece that ends at it, the last point
    // also the closing piece, the first the removal of the whole edge.
    const double rx = qq[2 * j], ry = qq[2 * j + 1];
    const double *V = sp.bpoly + 2 * int64_t(sp.bvoff[j]);
    const double ax = V[2 * e], ay = V[2 * e + 1], bx = V[2 * e + 2], by = V[2 * e + 3]; // closing vertex repeated
    const bool first = !(i > sp.P0[j] && sp.edge[i - 1] == e && is_nd(i - 1));
    const bool last = !(i + 1 < sp.P0[j + 1] && sp.edge[i + 1] == e && is_nd(i + 1));
    const double px = first ? ax : sp.x[i - 1], py = first ? ay : sp.y[i - 1];
    const double x = sp.x[i], y = sp.y[i];
    int w = wind_edge(px, py, x, y, rx, ry);
    if (first) w -= wind_edge(ax, ay, bx, by, rx, ry);
    if (last) w += wind_edge(x, y, bx, by, rx, ry);
    if (w) atomicAdd(&wind[j], w);
}

// Entry/exit status of every crossing vertex from the parity of crossings
// since the first plain vertex V; bouncing vertices met with status EXIT are
// split candidates (labelIntersections2 step 4, polyclip.h:551-635), and a job
// with a P candidate linked to a Q candidate takes the sequential route
// (blockIdx.y 2).  A crossing is a step of the crossing counts, so a plain slot
// is one word read and nothing written; statuses are kept per crossing, the
// bouncing ones computed where a job has any (the status and split arrays over
// all slots took 0.81 ms for 35 million slots and 24 million positions, now
// 0.65; for 40 million dense slots 0.47, now 0.21).
struct EnexSide {
    Side r;
    int64_t n;
    const int *pj;   // jobs of a sparse base side's positions, else null
    const int *slot; // their slots
    const uint32_t *cc; // crossings before each slot (closing entry included)
    const int *first, *wind, *m, *v; // per job: first plain slot, winding, crossings, those before it
    int *enex, *cpos; // per crossing: status, slot
};
struct EnexSides {
    EnexSide s[2]; // P, Q
    int J, per;
    const int *kind, *bounce;
    uint32_t *linkP, *linkQ; // crossing -> the crossing it is linked to on the other side (linkQ: as P's links have it)
    int *slow;
};
// status on meeting slot i (local slot sl) of job j's ring
__device__ inline int status_at(const EnexSide &z, int j, int sl, uint32_t before) {
    const uint32_t c = before - uint32_t(z.v[j]) + (sl < z.first[j] ? uint32_t(z.m[j]) : 0u);
    return ((z.wind[j] % 2) != 0 ? EXIT : ENTRY) ^ int(c & 1u);
}
__global__ __launch_bounds__(BLK) void k_jenex(EnexSides a) {
    const bool splits = blockIdx.y == 2;
    const EnexSide &z = a.s[blockIdx.y & 1];
    const int lane = threadIdx.x & (WAVE - 1);
    WaveSpan w(z.r.off, a.J, z.pj ? 0 : z.n, a.per);
    for (int q = 0; q < a.per && w.at < z.n; ++q, w.at += WAVE) {
        const int64_t i = w.at + lane;
        const int js = z.pj ? 0 : w.of(z.r.off, a.J, lane);
        if (i >= z.n) continue;
        if (splits) {
            const int j = z.pj ? z.pj[i] : js;
            if (!a.bounce[j] || a.kind[j] != K_CROSS || z.r.lab[i] != L_BOUNCING || !inter_at(z.r, i)) continue;
            if (status_at(z, j, z.slot ? z.slot[i] : int(i) - z.r.off[j], z.cc[i]) != EXIT) continue;
            const EnexSide &o = a.s[1];
            const int sl = z.r.nbr[i] - 1;
            const int64_t g = int64_t(o.r.off[j]) + sl;
            if (o.r.lab[g] == L_BOUNCING && inter_at(o.r, g) && status_at(o, j, sl, o.cc[g]) == EXIT)
                atomicOr(&a.slow[j], SLOW_SPLIT);
            continue;
        }
        const uint32_t ci = z.cc[i];
        if (z.cc[i + 1] == ci) continue; // no crossing
        z.cpos[ci] = int(i);
        const int j = z.pj ? z.pj[i] : js;
        if (a.kind[j] != K_CROSS) {
            z.enex[ci] = NEITHER;
            continue;
        }
        if (blockIdx.y == 0) {
            const int64_t o = int64_t(z.r.ooff[j]) + (z.r.nbr[i] - 1);
            const uint32_t l = a.s[1].cc[o];
            const bool ok = a.s[1].cc[o + 1] != l;
            a.linkP[ci] = ok ? l : NIL;
            if (ok) a.linkQ[l] = ci;
        }
        z.enex[ci] = status_at(z, j, z.slot ? z.slot[i] : int(i) - z.r.off[j], ci);
    }
}

struct PieceArgs {
    int J;
    Side P, Q;
    const int *PAB;  // J+1 slot offsets of the base rings (virtual in the sparse layout)
    int sparse;      // base side given as positions of a sparse ring
    SparseP sp;
    const int *cposP, *cposQ;
    const uint32_t *crossP, *ccountP;
    const uint32_t *linkP, *linkQ;
    const int *enexP, *enexQ; // per crossing
    const int *cP0, *cQ0, *kind;
    int mP, mQ; // crossing totals of the batch
    int *ppos, *plen, *pdir, *pj;
    uint32_t *succ, *val;
    int *slow;
    const int *flags; // a flagged job's sparse slots may not ascend: as the searches find them
};

// Pieces: crossing x (P crossings first, then Q crossings; blockIdx.y picks the
// side) to the next crossing in its walking direction; ppos is local to the
// job's ring.  A P crossing's value orders the starts: even for its own index
// (crossings ascend with their slots), odd for the far one's.
// Bound by gathers: crossings find one another by the indices that the kernel
// before left (linkP, linkQ), so a Q crossing on a shared base ring needs no
// search among the job's slots (18 million crossings: 1.32 -> 0.67 ms; the
// starts by index instead of slot, below: 1.09 -> 0.39).
__global__ __launch_bounds__(BLK) void k_jpieces(PieceArgs a) {
    const bool onP = blockIdx.y == 0;
    const int xl = blockIdx.x * blockDim.x + threadIdx.x;
    if (xl >= (onP ? a.mP : a.mQ)) return;
    const int x = onP ? xl : a.mP + xl;
    const Side &R = onP ? a.P : a.Q;
    const int *cpos = onP ? a.cposP : a.cposQ;
    const int *c0 = onP ? a.cP0 : a.cQ0;
    const int *enex = onP ? a.enexP : a.enexQ;
    const int j = seg_of_wave(c0, a.J, xl);
    a.pj[x] = j;
    if (a.kind[j] != K_CROSS) {
        a.ppos[x] = 0;
        a.plen[x] = 0;
        a.pdir[x] = 1;
        a.succ[x] = uint32_t(x);
        a.val[x] = NIL;
        return;
    }
    const int m = c0[j + 1] - c0[j];
    const int jl = xl - c0[j];
    const int pos = cpos[xl];
    const int e = enex[xl];
    const int d = e == ENTRY ? 1 : -1;
    int jw = jl + d;
    if (jw < 0) jw += m;
    if (jw >= m) jw -= m;
    const int xw = c0[j] + jw; // the far crossing
    const int posW = cpos[xw];
    if (enex[xw] != (e ^ 1)) atomicOr(&a.slow[j], SLOW_ODD);
    // local slots of the two crossings and the ring length
    int sl, slW, n;
    if (onP) {
        n = a.PAB[j + 1] - a.PAB[j];
        sl = a.sparse ? a.sp.slot[pos] : pos - R.off[j];
        slW = a.sparse ? a.sp.slot[posW] : posW - R.off[j];
    } else {
        n = R.off[j + 1] - R.off[j];
        sl = pos - R.off[j];
        slW = posW - R.off[j];
    }
    int len = d > 0 ? slW - sl : sl - slW;
    if (len <= 0) len += n;
    // the neighbour of the far crossing on the other ring, as a crossing index
    uint32_t s = uint32_t(x);
    bool ok;
    uint32_t occw = 0;
    if (onP) {
        occw = a.linkP[xw];
        ok = occw != NIL;
    } else {
        const int wl = R.nbr[posW] - 1; // local slot on the other ring
        // the P crossing that is linked here, where that is the one this side is linked to
        const uint32_t l = a.linkQ[xw];
        ok = false;
        if (l >= uint32_t(a.cP0[j]) && l < uint32_t(a.cP0[j + 1]) && !(a.sparse && a.flags[j])) {
            const int g = a.cposP[l];
            ok = (a.sparse ? a.sp.slot[g] : g - a.PAB[j]) == wl;
            occw = l;
        }
        if (!ok && a.sparse) {
            const int k = sp_find(a.sp, j, wl);
            ok = k >= 0 && a.crossP[k] != 0;
            occw = k >= 0 ? a.ccountP[k] : 0u;
        } else if (!ok) {
            const int64_t w = int64_t(R.ooff[j]) + wl;
            ok = a.crossP[w] != 0;
            occw = a.ccountP[w];
        }
    }
    if (!ok) atomicOr(&a.slow[j], SLOW_LINK);
    else s = (onP ? uint32_t(a.mP) : 0u) + occw;
    a.ppos[x] = sl;
    a.plen[x] = len;
    a.pdir[x] = d;
    a.succ[x] = s;
    a.val[x] = onP ? min(2u * uint32_t(x), 2u * uint32_t(xw) + 1u) : NIL;
}

// Cycles of the crossing graph by doubling.  On a crossing job successors
// alternate between P and Q crossings and only P crossings carry values, so
// the doubling runs over the P crossings alone, stepping two pieces at a time
// (a P piece and the Q piece after it).  After r rounds the record of P
// crossing x describes the window of 2^r such steps from x (wrapping around
// x's cycle): the window's minimum value, the summed piece lengths before
// that minimum's first occurrence, the summed lengths of the whole window and
// the P crossing after the window.  A window sum is read only when the window
// holds no occurrence of the cycle's minimum, so does not wrap and stays below
// the cycle's total; the 32-bit wrap-around of longer windows is never read.
struct JumpArgs {
    int mP, M;
    const uint32_t *val, *succ;
    const int *plen, *pj, *kind, *slow;
};
// A job found inconsistent while its pieces were built takes the sequential
// route: its crossings stand alone.
__device__ inline uint4 jump_first(const JumpArgs &a, int x) {
    const int j = a.pj[x];
    if (a.kind[j] != K_CROSS || a.slow[j]) return make_uint4(NIL, 0u, 0u, uint32_t(x));
    const uint32_t q = a.succ[x];
    uint32_t n2 = q < uint32_t(a.M) ? a.succ[q] : uint32_t(x);
    if (n2 >= uint32_t(a.mP)) n2 = uint32_t(x); // not a P-Q-P step: a crossing outside the traversed jobs
    const uint32_t w = uint32_t(a.plen[x]) + (q < uint32_t(a.M) && q != uint32_t(x) ? uint32_t(a.plen[q]) : 0u);
    return make_uint4(a.val[x], 0u, w, n2);
}
__device__ inline uint4 jump_join(const uint4 &a, const uint4 &b) { // the window of a, then that of b
    uint4 o;
    o.x = a.x <= b.x ? a.x : b.x;
    o.y = a.x <= b.x ? a.y : a.z + b.y;
    o.z = a.z + b.z;
    o.w = b.w;
    return o;
}
__global__ void k_jump_init(JumpArgs a, uint4 *rec, uint2 *cov) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    if (x >= a.mP) return;
    rec[x] = jump_first(a, x);
    cov[x] = make_uint2(NIL, 0u);
}

// More crossings than one block holds: one of every RULE crossings, at a place
// that a hash picks, is a ruler.  A ruler walks to the next one and leaves every
// crossing it passes its name and the distance; only the rulers' windows are
// doubled; and a cycle without a ruler, short as it then is, is walked from each
// of its crossings.  9 million crossings: 0.84 ms, doubling all of them 1.70
// (19 rounds of three 16-byte accesses each).
// The links are a permutation; a walk of more than RULE_CAP steps says that
// they are not, and the caller then doubles every crossing's window.
constexpr int RULE = 8, RULE_CAP = 4096;
__device__ inline uint32_t ruler_of(uint32_t g) { // group g's ruler
    uint32_t h = g * 0x9E3779B1u;
    h ^= h >> 15;
    h *= 0x85EBCA77u;
    return g * RULE + (h >> 29);
}
__device__ inline bool is_ruler(uint32_t x) { return ruler_of(x / RULE) == x; }

__global__ void k_ruler_walk(int mP, int G, const uint4 *__restrict__ rec, uint2 *cov, uint4 *rule, uint32_t *over) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= G) return;
    uint32_t x = ruler_of(uint32_t(g));
    if (x >= uint32_t(mP)) { // the last group may end before its ruler
        rule[g] = rule[G + g] = make_uint4(NIL, 0u, 0u, uint32_t(g));
        return;
    }
    uint4 a = rec[x]; // minimum, its distance, length, next
    cov[x] = make_uint2(uint32_t(g), 0u);
    a.y = 0u;
    int steps = 0;
    while (!is_ruler(a.w)) {
        if (++steps > RULE_CAP) {
            *over = 1u;
            break;
        }
        const uint4 b = rec[a.w];
        cov[a.w] = make_uint2(uint32_t(g), a.z);
        a = jump_join(a, make_uint4(b.x, 0u, b.z, b.w));
    }
    a.w = is_ruler(a.w) ? a.w / RULE : uint32_t(g);
    rule[g] = rule[G + g] = a; // the stretch, and the window that is doubled
}

// every crossing's cycle minimum and the distance to it: from its ruler's
// window (rule1: whole cycles), or, where the minimum lies behind it on its
// ruler's stretch (rule0), from the next ruler's
__global__ void k_ruler_final(int mP, const uint4 *__restrict__ rec, const uint2 *__restrict__ cov,
                              const uint4 *__restrict__ rule0, const uint4 *__restrict__ rule1, uint2 *out,
                              uint32_t *over) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    if (x >= mP) return;
    const uint2 c = cov[x];
    if (c.x != NIL) {
        const uint4 r = rule1[c.x];
        uint32_t d = r.y - c.y;
        if (r.y < c.y) {
            const uint4 r0 = rule0[c.x];
            d = rule1[r0.w].y + (r0.z - c.y);
        }
        out[x] = make_uint2(r.x, d);
        return;
    }
    uint4 a = rec[x];
    for (int steps = 0; a.w != uint32_t(x); ) {
        if (++steps > RULE_CAP) {
            *over = 1u;
            break;
        }
        const uint4 b = rec[a.w];
        a = jump_join(a, make_uint4(b.x, 0u, b.z, b.w));
    }
    out[x] = make_uint2(a.x, a.y);
}
__global__ void k_jump_out(int mP, const uint4 *__restrict__ rec, uint2 *out) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    if (x < mP) out[x] = make_uint2(rec[x].x, rec[x].y);
}

// Round r makes every window four times as long (4^r records to 4^(r+1)) and
// sets moved[r] when some window's minimum changed.  Values on a cycle are
// distinct, so a round that moves no minimum finds every cycle no longer than
// the windows it read: minima and distances are final in both buffers (the
// round copied them unchanged), and every later round returns at once.
// Doubling takes twice the launches (2.6 us each also where they return) and a
// read and a write more of every record for one gather less: labelling of
// 200,000 x 1,000,000 vertices 0.488 -> 0.470 ms, of 100,000 x 4,096 overlays
// 7.10 -> 7.04 ms.
__global__ void k_jump_rank(int mP, const uint4 *__restrict__ rec, uint4 *__restrict__ rec2, uint32_t *moved,
                            int r) {
    if (r > 0 && moved[r - 1] == 0u) return;
    int x = blockIdx.x * blockDim.x + threadIdx.x;
    if (x >= mP) return;
    const uint4 a = rec[x];
    uint4 o = jump_join(a, rec[a.w]);
    o = jump_join(o, rec[o.w]);
    o = jump_join(o, rec[o.w]);
    rec2[x] = o;
    if (o.x != a.x) moved[r] = 1u;
}

// The rounds, doubling, for at most JUMP_SMALL records, by one block with
// the records in LDS (64 KB): a round is a barrier instead of a launch (12
// launches of 2.5 us and their gaps at 1,400 crossings).
constexpr int JUMP_SMALL = 4096, JUMP_BLK = 1024, JUMP_PER = JUMP_SMALL / JUMP_BLK;
__device__ inline void jump_all(uint4 (&a)[JUMP_PER], int n, int rounds) { // thread t: records t, t + JUMP_BLK, ...
    __shared__ uint4 r[JUMP_SMALL];
    for (int q = 0; q < JUMP_PER; ++q) {
        const int x = q * JUMP_BLK + int(threadIdx.x);
        if (x < n) r[x] = a[q];
    }
    __syncthreads();
    for (int k = 0; k < rounds; ++k) {
        int moved = 0;
        for (int q = 0; q < JUMP_PER; ++q) {
            const int x = q * JUMP_BLK + int(threadIdx.x);
            if (x >= n) continue;
            const uint4 o = jump_join(a[q], r[a[q].w]);
            moved |= o.x != a[q].x ? 1 : 0;
            a[q] = o;
        }
        moved = __syncthreads_or(moved); // every record is read before the next round's are written
        if (!moved) break;
        for (int q = 0; q < JUMP_PER; ++q) {
            const int x = q * JUMP_BLK + int(threadIdx.x);
            if (x < n) r[x] = a[q];
        }
        __syncthreads();
    }
}
// the crossings' own records
__global__ __launch_bounds__(JUMP_BLK) void k_jump_small(JumpArgs ja, int rounds, uint2 *out) {
    uint4 a[JUMP_PER];
    for (int q = 0; q < JUMP_PER; ++q) {
        const int x = q * JUMP_BLK + int(threadIdx.x);
        if (x < ja.mP) a[q] = jump_first(ja, x);
    }
    jump_all(a, ja.mP, rounds);
    for (int q = 0; q < JUMP_PER; ++q) {
        const int x = q * JUMP_BLK + int(threadIdx.x);
        if (x < ja.mP) out[x] = make_uint2(a[q].x, a[q].y);
    }
}
// the rulers'
__global__ __launch_bounds__(JUMP_BLK) void k_rule_small(uint4 *rec, int n, int rounds) {
    uint4 a[JUMP_PER];
    for (int q = 0; q < JUMP_PER; ++q) {
        const int x = q * JUMP_BLK + int(threadIdx.x);
        if (x < n) a[q] = rec[x];
    }
    jump_all(a, n, rounds);
    for (int q = 0; q < JUMP_PER; ++q) {
        const int x = q * JUMP_BLK + int(threadIdx.x);
        if (x < n) rec[x] = a[q];
    }
}

// Per crossing (P and Q): the list start of a traversed cycle (the P crossing
// whose even value, twice its index, is the cycle's minimum; every other value
// on the cycle is larger) and the summed piece lengths from the crossing up to
// that start, the whole cycle's total at the start itself.
// Equivalent to the list ranking of the cycle broken before its start.
// For the P crossings also the ring starts and their totals in base-ring
// order, each with a closing entry.
__global__ void k_rank_final(int M, int mP, const uint2 *__restrict__ rec, const uint32_t *succ, const int *plen,
                             uint32_t *inode, uint32_t *dist, uint32_t *tot, uint32_t *isstart) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    if (x == 0) tot[mP] = isstart[mP] = 0u;
    if (x >= M) return;
    // the P crossing whose record describes x's cycle: x itself, or a Q crossing's successor
    const uint32_t p = x < mP ? uint32_t(x) : succ[x];
    uint32_t m = NIL, dp = 0u;
    if (p < uint32_t(mP)) {
        const uint2 r = rec[p];
        m = r.x;
        dp = r.y;
    }
    const bool trav = m != NIL && (m & 1u) == 0u;
    const uint32_t I = trav ? m >> 1 : NIL;
    inode[x] = I;
    uint32_t d = 0u;
    if (trav) {
        if (x >= mP) {
            d = uint32_t(plen[x]) + (p == I ? 0u : dp);
        } else if (uint32_t(x) != I) {
            d = dp;
        } else { // the start: the whole cycle, its own piece then the Q piece after it and on
            const uint32_t q = succ[x], n2 = succ[q];
            d = uint32_t(plen[x]) + uint32_t(plen[q]) + (n2 == I || n2 >= uint32_t(mP) ? 0u : rec[n2].y);
        }
    }
    dist[x] = d;
    if (x < mP) {
        const bool st = I == uint32_t(x);
        tot[x] = st ? d : 0u;
        isstart[x] = st ? 1u : 0u;
    }
}

struct CountArgs {
    int J;
    const int *AB, *AC, *kind, *slow, *windP, *windQ, *cP0, *sidx, *seq_res; // seq_res null: not run (yet)
    const uint32_t *base, *ridx;
    uint32_t *jv, *jr;
};

// output vertices and rings of every job before clean-up
__global__ void k_jcounts(CountArgs a) {
    int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j > a.J) return;
    if (j == a.J) { // closing entries of their scans
        a.jv[j] = a.jr[j] = 0u;
        return;
    }
    uint32_t v = 0, r = 0;
    const int k = a.kind[j];
    if (k == K_CROSS && !a.slow[j]) {
        v = a.base[a.cP0[j + 1]] - a.base[a.cP0[j]];
        r = a.ridx[a.cP0[j + 1]] - a.ridx[a.cP0[j]];
    } else if (k == K_NOCROSS) {
        bool ip = (a.windP[j] % 2) != 0, iq = (a.windQ[j] % 2) != 0;
        v = (ip ? uint32_t(a.AB[j + 1] - a.AB[j]) : 0u) + (iq ? uint32_t(a.AC[j + 1] - a.AC[j]) : 0u);
        r = uint32_t(ip) + uint32_t(iq);
    } else if (a.seq_res) {
        int s = a.sidx[j];
        r = uint32_t(a.seq_res[3 * s]);
        v = uint32_t(a.seq_res[3 * s + 1]);
    }
    a.jv[j] = v;
    a.jr[j] = r;
}

// every piece's first output vertex carries the piece (its index + 1); what the
// output needs of a piece in one record; ring offsets at the starts
struct HeadArgs {
    int M, mP;
    const uint32_t *inode, *dist, *base, *ridx;
    const int *pj, *cP0, *ppos, *plen, *pdir;
    const uint32_t *JV, *JR;
    uint32_t *head;
    int4 *piece; // first output vertex, length, slot (walked on) or ~slot (walked back), job
    int *off;
};
__global__ void k_jheads(HeadArgs a) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    if (x >= a.M) return;
    const int j = a.pj[x];
    const int c0 = a.cP0[j];
    if (x < a.mP && a.ridx[x + 1] != a.ridx[x])
        a.off[a.JR[j] + a.ridx[x] - a.ridx[c0]] = int(a.JV[j] + a.base[x] - a.base[c0]);
    const uint32_t I = a.inode[x];
    if (I == NIL) return;
    const uint32_t o = a.JV[j] + (a.base[I] - a.base[c0]) + (a.dist[I] - a.dist[x]);
    a.head[o] = uint32_t(x) + 1u;
    const int sl = a.ppos[x];
    a.piece[x] = make_int4(int(o), a.plen[x], a.pdir[x] > 0 ? sl : ~sl, j);
}

struct EmitArgs {
    int J, mP;
    const int *PAB; // base ring slot offsets (virtual in the sparse layout)
    int sparse;
    SparseP sp;
    const int *cP0, *cposP, *flags;
    const uint32_t *head;
    const int4 *piece;
    Side P, Q;
    double *ox, *oy;
    int *osrc;
};

// Output vertex i from the piece it lies on: the last head up to i names one
// (of an earlier job where i is not on a piece: then it ends before i).  The
// piece's record replaces a search for the job, its crossings' positions the
// search among the job's slots (24 million vertices: 0.85 -> 0.63 ms, bound by
// gathers of points).
__global__ __launch_bounds__(BLK) void k_jemit(EmitArgs a, int64_t n_out) {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n_out) return;
    const uint32_t h = a.head[i];
    if (h == 0u) return;
    const int x = int(h - 1u);
    const int4 pc = a.piece[x];
    const int k = int(i - int64_t(uint32_t(pc.x))) + 1;
    if (k > pc.y) return;
    const int j = pc.w;
    const bool on = pc.z >= 0; // walked on
    const int sl = on ? pc.z : ~pc.z;
    const bool onP = x < a.mP;
    const int *off = onP ? a.PAB : a.Q.off;
    const int n = off[j + 1] - off[j];
    int pos = (sl + (on ? k : -k)) % n;
    if (pos < 0) pos += n;
    if (onP && a.sparse) {
        // its place among the job's positions, between the piece's two crossings (or, past the ring's
        // end, its first or last one): most pieces leave nothing to search
        int lo = a.sp.P0[j], hi = a.sp.P0[j + 1];
        const int c0 = a.cP0[j], c1 = a.cP0[j + 1];
        if (a.flags[j]) { // slots that may not ascend: the whole job, as elsewhere
        } else if (on) {
            if (pos > sl) {
                lo = a.cposP[x] + 1;
                if (x + 1 < c1) hi = a.cposP[x + 1];
            } else {
                hi = a.cposP[c0];
            }
        } else {
            if (pos < sl) {
                hi = a.cposP[x];
                if (x > c0) lo = a.cposP[x - 1];
            } else {
                lo = a.cposP[c1 - 1];
            }
        }
        const SlotInfo si = sp_slot_in(a.sp, j, pos, lo, hi);
        a.ox[i] = si.x;
        a.oy[i] = si.y;
        a.osrc[i] = SRC_NONE;
    } else {
        const Side &R = onP ? a.P : a.Q;
        const int g = off[j] + pos;
        a.ox[i] = R.x[g];
        a.oy[i] = R.y[g];
        a.osrc[i] = onP ? g : ~g;
    }
}

// the base rings of no-crossing jobs in the sparse layout, by output position
__global__ void k_sp_nocross_p(int64_t n_out, int J, const uint32_t *JV, const int *kind, const int *windP,
                               SparseP sp, double *ox, double *oy, int *osrc) {
    int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n_out) return;
    const int j = seg_of(reinterpret_cast<const int *>(JV), J, i);
    if (kind[j] != K_NOCROSS || (windP[j] % 2) == 0) return;
    const int q = int(i - JV[j]);
    if (q >= sp.AB[j + 1] - sp.AB[j]) return; // the overlay part
    const SlotInfo si = sp_slot(sp, j, q);
    ox[i] = si.x;
    oy[i] = si.y;
    osrc[i] = SRC_NONE;
}

// dense copies of the sparse base rings of the sequential jobs
__global__ void k_sp_materialize(int q0, int nseq, const int *jobs_of, const int64_t *moff, SparseP sp,
                                 const int *av, const int *nbr, const int *lab, double *mx, double *my, int *mav,
                                 int *mnbr, int *mlab) {
    const int q = q0 + int(blockIdx.y);
    if (q >= nseq) return;
    const int j = jobs_of[q];
    const int n = sp.AB[j + 1] - sp.AB[j];
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) {
        const SlotInfo si = sp_slot(sp, j, t);
        const int64_t o = moff[q] + t;
        mx[o] = si.x;
        my[o] = si.y;
        mav[o] = si.pos >= 0 ? av[si.pos] : -100;
        mnbr[o] = si.pos >= 0 ? nbr[si.pos] : -100;
        mlab[o] = si.pos >= 0 ? lab[si.pos] : 0;
    }
}

// rings of no-crossing jobs: P's ring when its plain vertex lies inside Q, then Q's
__global__ void k_jcopy_nocross(Side s, bool sideP, int J, int64_t n, const int *kind, const int *windP,
                                const int *windQ, const int *AB, const uint32_t *JV, double *ox, double *oy,
                                int *osrc) {
    int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int j = seg_of(s.off, J, i);
    if (kind[j] != K_NOCROSS) return;
    bool ip = (windP[j] % 2) != 0, iq = (windQ[j] % 2) != 0;
    if (sideP ? !ip : !iq) return;
    int64_t dst = JV[j] + (sideP || !ip ? 0 : (AB[j + 1] - AB[j])) + (i - s.off[j]);
    ox[dst] = s.x[i];
    oy[dst] = s.y[i];
    osrc[dst] = sideP ? int(i) : ~int(i);
}

__global__ void k_jnocross_off(int J, const int *kind, const int *windP, const int *windQ, const int *AB,
                               const uint32_t *JV, const uint32_t *JR, int *off) {
    int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= J || kind[j] != K_NOCROSS) return;
    bool ip = (windP[j] % 2) != 0, iq = (windQ[j] % 2) != 0;
    uint32_t r = JR[j];
    if (ip) off[r++] = int(JV[j]);
    if (iq) off[r] = int(JV[j] + (ip ? uint32_t(AB[j + 1] - AB[j]) : 0u));
}

// ---------------------------------------------------------------------------
// ---------------------------------------------------------------------------
// clean-up (cleanUpResult2)
// ---------------------------------------------------------------------------
__device__ inline bool collinear(const double *x, const double *y, int a, int b, int c) {
    return fabs(areaA(x[a], y[a], x[b], y[b], x[c], y[c])) < EPS;
}

// drop collinear roots: the root's predecessor stays the ring's last vertex
__global__ void k_root_loop(int nr, const int *off, const double *x, const double *y, int *rstart) {
    int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= nr) return;
    int s = off[r], last = off[r + 1] - 1;
    int root = s;
    while (root <= last) {
        int nx = root == last ? root : root + 1;
        int pv = root == last ? root : last;
        if (collinear(x, y, pv, root, nx)) ++root;
        else break;
    }
    rstart[r] = root;
}

// Which vertices stay.  In a ring, the vertices before its root go, the root
// stays, and a later vertex stays unless it is collinear with the last vertex
// kept before it and its successor (the root, for the ring's last vertex).
// One wave decides a span from left to right, 64 vertices a window: while the
// vertex before is kept a vertex's decision needs only its two neighbours (k0,
// all lanes at once), so a step goes to the next vertex dropped that way;
// after a drop the last kept vertex L is fixed until the next kept one, so one
// step tests all later lanes against L.  A step is one test per lane and a
// ballot, however long the run of dropped vertices is.  Rounds that each let
// one more vertex of every run see its last kept vertex took 6 launches of 15
// us on 1.4 M vertices, and 48 of 54 us and then 6.4 ms of one lane per ring on
// 27 M (short edges drop in long runs); now 39 us and 0.26 ms.
constexpr int KEEP_WIN = 4;                  // windows per tile, their loads issued together
constexpr int KEEP_TILE = KEEP_WIN * WAVE;
constexpr int64_t KEEP_FIRST_TWO = 1 << 18; // vertices beyond which two rounds are run before the first check
constexpr int KEEP_ROUNDS = 50;              // rounds before one wave per ring
constexpr uint32_t KEEP_ANY = 0xffffffffu;   // the tile's first vertex needs no vertex before it

struct KeepArgs {
    int64_t n;
    const int *ringid, *off, *rstart;
    const double *x, *y;
    uint32_t *keep;
    uint32_t *used;      // per tile: the mark (last kept index + 1) before it that it was decided with
    const uint32_t *last; // per tile, previous round: its last kept index + 1, 0 for none
    uint32_t *last_out;
    uint32_t *changed;   // per round: some tile's last kept vertex moved
    int64_t ntiles;
};

__device__ inline double lane_value(double v, int l) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane(int(b), l), hi = __builtin_amdgcn_readlane(int(b >> 32), l);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

// vertices [base, min(base + NW * 64, end)), flags written from 'out' (a window's
// start) on; mark: last kept index + 1 before base.  Returns the span's last
// kept index + 1, or mark; used: the mark before 'out', KEEP_ANY when the vertex
// there needs none.  Run by a whole wave, uniform arguments.
template <int NW>
__device__ inline uint32_t keep_span(const KeepArgs &a, int64_t base, int64_t out, int64_t end, uint32_t mark,
                                     uint32_t &used) {
    const int lane = threadIdx.x & (WAVE - 1);
    int rs[NW], rl[NW];
    double X[NW], Y[NW], XN[NW], YN[NW];
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        const int64_t i = base + w * WAVE + lane;
        rs[w] = rl[w] = -1;
        X[w] = Y[w] = XN[w] = YN[w] = 0.0;
        if (i < end) {
            rl[w] = a.ringid[i];
            X[w] = a.x[i];
            Y[w] = a.y[i];
        }
    }
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        const int64_t i = base + w * WAVE + lane;
        if (i < end) {
            rs[w] = a.rstart[rl[w]];
            rl[w] = a.off[rl[w] + 1] - 1; // the ring's last vertex
        }
    }
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        const int64_t i = base + w * WAVE + lane;
        if (i < end) {
            const int64_t nx = i == rl[w] ? rs[w] : i + 1;
            if (rs[w] <= rl[w]) { // else no vertex of the ring stays and none is tested
                XN[w] = a.x[nx];
                YN[w] = a.y[nx];
            }
        }
    }
    double px = 0.0, py = 0.0; // the vertex before the window
    if (base > 0) {
        px = a.x[base - 1];
        py = a.y[base - 1];
    }
    used = KEEP_ANY;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        const int64_t b = base + w * WAVE, i = b + lane;
        if (b >= end) break; // uniform
        const bool valid = i < end, fixed = valid && i <= rs[w];
        double XP = __shfl_up(X[w], 1, WAVE), YP = __shfl_up(Y[w], 1, WAVE); // every lane active
        if (lane == 0) {
            XP = px;
            YP = py;
        }
        const bool k0 = fixed ? i == rs[w] : valid && !(fabs(areaA(XP, YP, X[w], Y[w], XN[w], YN[w])) < EPS);
        const uint64_t K0 = __ballot(k0), FIX = __ballot(fixed);
        const int nv = int(end - b < WAVE ? end - b : WAVE);
        const uint64_t V = nv == WAVE ? ~0ull : ((1ull << nv) - 1ull);
        uint64_t K = 0;
        int p = 0;
        double Lx = 0.0, Ly = 0.0;
        bool yes = (FIX & 1ull) || mark == uint32_t(b); // the vertex before lane p is kept, or lane p needs none
        if (b == out) used = (FIX & 1ull) ? KEEP_ANY : mark;
        if (!yes) {
            Lx = a.x[mark - 1u];
            Ly = a.y[mark - 1u];
        }
        while (p < nv) {
            const uint64_t from = ~0ull << p;
            if (yes) {
                const uint64_t D = V & ~K0 & ~FIX & from;
                const int z = D ? int(__builtin_ctzll(D)) : nv;
                K |= K0 & from & (z == WAVE ? ~0ull : ((1ull << z) - 1ull));
                if (z < nv) {
                    Lx = z ? lane_value(X[w], z - 1) : px;
                    Ly = z ? lane_value(Y[w], z - 1) : py;
                    yes = false;
                }
                p = z + 1;
            } else {
                const bool stop = valid && lane >= p &&
                                  (fixed || !(fabs(areaA(Lx, Ly, X[w], Y[w], XN[w], YN[w])) < EPS));
                const uint64_t F = __ballot(stop);
                if (!F) break;
                const int f = int(__builtin_ctzll(F));
                yes = true;
                if ((FIX >> f) & 1ull) {
                    p = f;
                } else {
                    K |= 1ull << f;
                    p = f + 1;
                }
            }
        }
        if (valid && i >= out) a.keep[i] = uint32_t((K >> lane) & 1ull);
        if (K) mark = uint32_t(b) + uint32_t(WAVE - __builtin_clzll(K));
        px = lane_value(X[w], WAVE - 1);
        py = lane_value(Y[w], WAVE - 1);
    }
    return mark;
}

// Round 0: every tile, one wave each, from one window before it, as if the
// vertex before that window were kept: only a run of dropped vertices as long
// as the window leaves the tile with another start than its true one.
__global__ __launch_bounds__(BLK) void k_keep_first(KeepArgs a) {
    const int64_t t = int64_t(__builtin_amdgcn_readfirstlane(int(blockIdx.x * (BLK / WAVE) + threadIdx.x / WAVE)));
    if (t >= a.ntiles) return;
    const int64_t out = t * KEEP_TILE, end = min(out + KEEP_TILE, a.n);
    uint32_t used, m;
    if (t == 0) m = keep_span<KEEP_WIN>(a, 0, 0, end, 0u, used);
    else m = keep_span<KEEP_WIN + 1>(a, out - WAVE, out, end, uint32_t(out - WAVE), used);
    if ((threadIdx.x & (WAVE - 1)) == 0) {
        a.used[t] = used;
        a.last_out[t] = m > uint32_t(out) ? m : 0u;
    }
}

// Later rounds: a tile whose last kept vertex before it is another one than it
// was decided with is decided again.  A round that moves no tile's last kept
// vertex leaves every tile right, and later rounds return at once.  One wave
// looks at 64 tiles; hardly any is decided again (a run of dropped vertices has
// to cross a tile's edge).
__global__ __launch_bounds__(BLK) void k_keep_fix(KeepArgs a, int round) {
    if (round > 1 && a.changed[round - 1] == 0u) return;
    const int lane = threadIdx.x & (WAVE - 1);
    const int64_t t0 = int64_t(__builtin_amdgcn_readfirstlane(int(blockIdx.x * (BLK / WAVE) + threadIdx.x / WAVE))) * WAVE;
    if (t0 >= a.ntiles) return;
    const int64_t t = t0 + lane;
    uint32_t in = 0u;
    bool again = false;
    if (t < a.ntiles) {
        const uint32_t u = a.used[t];
        if (u != KEEP_ANY) { // its ring's root, which is kept, lies before the tile
            int64_t q = t - 1;
            while (q > 0 && a.last[q] == 0u) --q;
            in = a.last[q];
            again = in != u;
        }
        if (!again) a.last_out[t] = a.last[t];
    }
    uint64_t m = __ballot(again);
    while (m) {
        const int l = int(__builtin_ctzll(m));
        m &= m - 1ull;
        const int64_t tt = t0 + l, base = tt * KEEP_TILE;
        const uint32_t mk = uint32_t(__builtin_amdgcn_readlane(int(in), l));
        uint32_t used;
        const uint32_t r = keep_span<KEEP_WIN>(a, base, base, min(base + KEEP_TILE, a.n), mk, used);
        if (lane == 0) {
            const uint32_t lk = r > uint32_t(base) ? r : 0u;
            a.used[tt] = mk;
            a.last_out[tt] = lk;
            if (lk != a.last[tt]) a.changed[round] = 1u;
        }
    }
}

// one wave per ring from its first vertex to its last (runs that need too many rounds)
__global__ __launch_bounds__(BLK) void k_keep_rings(KeepArgs a, int nr) {
    const int r = __builtin_amdgcn_readfirstlane(int(blockIdx.x * (BLK / WAVE) + threadIdx.x / WAVE));
    if (r >= nr) return;
    const int64_t end = a.off[r + 1];
    uint32_t mark = 0u;
    uint32_t used;
    for (int64_t b = a.off[r]; b < end; b += KEEP_TILE)
        mark = keep_span<KEEP_WIN>(a, b, b, min(b + KEEP_TILE, end), mark, used);
}

// ring heads carry their ring index; an inclusive max-scan spreads it
__global__ void k_ring_heads(int nr, const int *off, uint32_t *head) {
    int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= nr) return;
    if (off[r + 1] > off[r]) head[off[r]] = uint32_t(r);
}

// vertices left of every ring, and whether there are any (nr + 1 threads: the closing entry)
__global__ void k_ring_counts(int nr, const int *off, const uint32_t *kscan, uint32_t *cnt, uint32_t *nonempty,
                              uint32_t *longest) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r > nr) return;
    const uint32_t c = r < nr ? kscan[off[r + 1]] - kscan[off[r]] : 0u;
    if (c > uint32_t(LONG_RING)) *longest = 1u;
    if (r < nr) cnt[r] = c;
    nonempty[r] = c > 0u ? 1u : 0u;
}

// the vertices kept, and the offsets of the rings that have any (with the closing one)
__global__ void k_compact_out(int64_t n, const uint32_t *keep, const uint32_t *kscan, const double *x,
                              const double *y, const int *src, double *x2, double *y2, int *src2, int nr,
                              const uint32_t *cnt, const uint32_t *nonempty, const int *off, int *off2) {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i <= nr && (i == nr || cnt[i])) off2[nonempty[i]] = int(kscan[off[i]]);
    if (i >= n || !keep[i]) return;
    const uint32_t o = kscan[i];
    x2[o] = x[i];
    y2[o] = y[i];
    src2[o] = src[i];
}

__global__ void k_job_rings(int J, const uint32_t *jr, const uint32_t *nonempty, uint32_t *out, int *ring) {
    int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j > J) return;
    const uint32_t r = nonempty[jr[j]];
    out[j] = r;
    ring[j] = int(r);
}

// ---------------------------------------------------------------------------
// sequential path: the reference's algorithm on index-linked vertices, one thread
// ---------------------------------------------------------------------------
struct SeqArgs {
    int nP, nQ, cap; // ring nodes of P and Q (an intersection vertex or a run of plain vertices)
    // node records: P nodes [0,nP), Q nodes [nP,nP+nQ)
    const double *nx0, *ny0, *nx1, *ny1; // first / last vertex of the node
    const int *nlen, *nslot, *ninter, *nlab, *nnb;
    const double *px, *py, *qx, *qy; // ring vertices by slot (run expansion)
    int windP, windQ;                // winding of each ring's first plain vertex w.r.t. the other ring
    double *vx, *vy, *vx1, *vy1;
    int *vlen, *vslot, *nx, *pv, *nb, *lab, *enex;
    uint8_t *inter;
    int *cand; // scratch list, cap entries
    int *seen; // 2 per vertex: the traversal component that last walked it in each direction
    int4 *rec; // per node for createResult2's walks: nx, pv, nb, enex | vlen << 2
    int *pstep; // per walk candidate: its walk's node count, then its first step record
    int2 *emit; // 2 * cap step records (node << 1 | forward, output place) of one round of walks
    double *ox, *oy;
    int *vsrc, *osrc; // provenance of inserted vertices / output vertices (slot reference)
    int P0, Q0;       // first slot of the job's rings in the batch arrays
    int uni;          // 1: the union (UNION of foster/polyclip.h:39 and its XORs)
    int par;          // 1: createResult2's rings walked one per lane first
    int out_cap;
    int *ring_off;
    int ring_cap;
    int *result; // [0] rings, [1] vertices, [2] status bits
};

// vertex t of node V in ring order
__device__ inline void seq_vertex(const SeqArgs &a, int V, int t, double &x, double &y) {
    if (a.vslot[V] >= 0 && a.vlen[V] > 1) {
        const bool onP = V < a.nP;
        const int sl = a.vslot[V] + t;
        x = onP ? a.px[sl] : a.qx[sl];
        y = onP ? a.py[sl] : a.qy[sl];
    } else {
        x = a.vx[V];
        y = a.vy[V];
    }
}

// point-in-polygon over the ring from root, every vertex of every node
__device__ __attribute__((always_inline)) bool seq_point_in(SeqArgs &a, int root, double rx, double ry) {
    int w = 0, one = root;
    bool have = false;
    double fx = 0, fy = 0, px = 0, py = 0;
    do {
        for (int t = 0; t < a.vlen[one]; ++t) {
            double cx, cy;
            seq_vertex(a, one, t, cx, cy);
            if (!have) {
                fx = cx;
                fy = cy;
                have = true;
            } else {
                w += wind_edge(px, py, cx, cy, rx, ry);
            }
            px = cx;
            py = cy;
        }
        one = a.nx[one];
    } while (one != root);
    w += wind_edge(px, py, fx, fy, rx, ry);
    return (w % 2) != 0;
}

// provenance of a single-vertex node
__device__ inline int seq_src(const SeqArgs &a, int V) {
    if (a.vslot[V] < 0) return a.vsrc[V];
    return V < a.nP ? a.P0 + a.vslot[V] : ~(a.Q0 + a.vslot[V]);
}

// node records -> the job's linked rings (all threads of the block)
// createResult2's walks, one per lane (see seq_run).  Returns PT_DONE with
// rings/outn advanced and the rings written, PT_FAIL when the single walk
// would fail (a ring that revisits a (node, direction) state, a jump to no
// neighbour, or the output capacities), or PT_FALLBACK after clearing what it
// wrote.  Candidate ranks live in seen[2v] (rank + 1) and the first ring that
// visits a candidate in seen[2v + 1] (as SEEN_FIRST - ring, kept by atomicMax),
// both zero before and after.
enum : int { PT_DONE = 0, PT_FAIL = 1, PT_FALLBACK = 2 };
constexpr int PT_MAX_STEPS = 1 << 15; // a longer ring walks in the single walk
constexpr int SEEN_FIRST = 1 << 30;
constexpr int PT_CHUNK = 2048; // candidates per round of walks

// one ring's walk from node I by one lane, as createResult2 walks it
// (foster/polyclip.h:717-759): returns 0 when it closes, 1 when it fails, 2
// when it is longer than PT_MAX_STEPS, 3 when 'visit' asks it to stop.
// 'visit' sees every node the walk marks (the start, every node stepped to,
// every jump target); 'step' sees every node stepped to with its direction
// and vertex count (the emitted ones).  A node's links, label and length come
// in one 16-byte record, so a step waits for one load.
template <class Visit, class Step>
__device__ __attribute__((always_inline)) int pt_walk(const SeqArgs &a, int I, Visit visit, Step step) {
    const bool uni = a.uni != 0;
    int V = I;
    if (visit(V)) return 3;
    int4 r = a.rec[V];
    int steps = 0, lam = 0, power = 1, sv = -1, sd = -1; // Brent's cycle test on (node, direction)
    do {
        const int e = r.w & 3;
        const int st = e == ENTRY ? EXIT : (e == EXIT ? ENTRY : e);
        do {
            const bool fwd = (st == EXIT) != uni;
            V = fwd ? r.x : r.y;
            const int dir = fwd ? 1 : 0;
            if (V == sv && dir == sd) return 1; // a state seen again: the walk never closes
            if (++lam == power) {
                sv = V;
                sd = dir;
                power <<= 1;
                lam = 0;
            }
            if (++steps > PT_MAX_STEPS) return 2;
            r = a.rec[V];
            if (visit(V)) return 3;
            step(V, fwd, r.w >> 2);
        } while (!((r.w & 3) == st) && V != I);
        if (V != I) {
            V = r.z;
            if (V < 0) return 1;
            if (visit(V)) return 3;
            r = a.rec[V];
        }
    } while (V != I);
    return 0;
}

// what the walks need from the wave that ran the steps before them, and
// what they give back (in LDS, one per block)
struct SeqShared {
    int go;                // 2: the entry/exit walks run, 1: createResult2's walks run, 0: result written
    int n, status;         // nodes (inserted ones included), status bits so far
    int rings, outn;       // rings and output vertices written so far
    int ptr;               // the walks' outcome (PT_*)
    int scan[2], sV[2];    // ring s: its entry/exit walk runs on every wave, from node sV[s]
    int sst[2];            //   with this status at sV[s]
    int nsplit[2], ncross[2]; // the split / crossing candidate lists' lengths
};

constexpr int SEQ_BLK = 1024; // threads of a sequential job's block

// exclusive scan of one value per thread over the block, in thread order;
// tot = the block's sum.  Every thread of the block calls it.
template <class T> __device__ inline T seq_block_scan(T c, T &tot, T *s_w) {
    const int lane = threadIdx.x & (WAVE - 1), wid = threadIdx.x / WAVE, nw = blockDim.x / WAVE;
    T incl = c;
    for (int d = 1; d < WAVE; d <<= 1) {
        const T o = __shfl_up(incl, d, WAVE);
        if (lane >= d) incl += o;
    }
    if (lane == WAVE - 1) s_w[wid] = incl;
    __syncthreads();
    T before = 0, t = 0;
    for (int w = 0; w < nw; ++w) {
        const T v = s_w[w];
        if (w < wid) before += v;
        t += v;
    }
    __syncthreads(); // s_w is free for the next call
    tot = t;
    return before + incl - c;
}

// minimum of one value per thread over the block.  Every thread calls it.
__device__ inline int seq_block_min(int x, int *s_w) {
    const int lane = threadIdx.x & (WAVE - 1), wid = threadIdx.x / WAVE, nw = blockDim.x / WAVE;
    for (int d = 1; d < WAVE; d <<= 1) x = min(x, __shfl_xor(x, d, WAVE));
    if (lane == 0) s_w[wid] = x;
    __syncthreads();
    int m = INT_MAX;
    for (int w = 0; w < nw; ++w) m = min(m, s_w[w]);
    __syncthreads();
    return m;
}

// Run by every thread of the block, with the same control flow in every
// wave (all loop bounds and branches that reach a barrier come from LDS or
// from values every thread computes alike).
__device__ __attribute__((always_inline)) int seq_par_traverse(SeqArgs &a, SeqShared &sh) {
    const int tid = threadIdx.x, nthr = blockDim.x;
    const int n = sh.n, rings = sh.rings, outn = sh.outn;
    const int n0 = a.nP + a.nQ; // nodes before any insertion; inserted nodes follow
    if (n - n0 > 4096) return PT_FALLBACK;
    __shared__ int s_w[SEQ_BLK / WAVE];
    __shared__ int64_t s_w64[SEQ_BLK / WAVE];
    __shared__ int s_next, s_qend, s_long, s_res;
    const int half = a.cap / 2;
    int *cand = a.cand, *info = a.cand + half;
    // the walks' node records (the walks change none of these fields)
    for (int v = tid; v < n; v += nthr) a.rec[v] = make_int4(a.nx[v], a.pv[v], a.nb[v], a.enex[v] | (a.vlen[v] << 2));
    // 1) the candidates in ring order from the root: original P nodes in index
    //    order, each followed by the nodes inserted after it
    auto is_cand = [&](int v) { return a.inter[v] != 0 && a.lab[v] == L_CROSSING; };
    int ncand = 0;
    // back to all-zero state words (listed candidates only carry marks)
    auto clear = [&]() {
        __syncthreads();
        for (int q = tid; q < ncand; q += nthr) {
            const int v = cand[q];
            a.seen[2 * v] = 0;
            a.seen[2 * v + 1] = 0;
        }
        __syncthreads();
    };
    for (int w = 0; w < a.nP; w += nthr) {
        const int v = w + tid;
        int c = 0;
        if (v < a.nP) {
            c = is_cand(v) ? 1 : 0;
            for (int x = a.nx[v], g = 0; x >= n0 && g <= n - n0; x = a.nx[x], ++g) c += is_cand(x) ? 1 : 0;
        }
        int tot;
        const int ex = seq_block_scan(c, tot, s_w);
        if (ncand + tot > half) {
            clear();
            return PT_FALLBACK;
        }
        int q = ncand + ex;
        if (v < a.nP) {
            if (is_cand(v)) {
                cand[q] = v;
                a.seen[2 * v] = ++q;
            }
            for (int x = a.nx[v], g = 0; x >= n0 && g <= n - n0; x = a.nx[x], ++g)
                if (is_cand(x)) {
                    cand[q] = x;
                    a.seen[2 * x] = ++q;
                }
        }
        ncand += tot;
    }
    __syncthreads();
    // 2)-4) in chunks of PT_CHUNK candidates in rank order, so that the
    // single walk's first failing ring is found without walking every
    // candidate after it.
    int nring = 0;    // rings of the chunks before
    int64_t nout = 0; // their vertices
    for (int c0 = 0; c0 < ncand; c0 += PT_CHUNK) {
        const int c1 = min(ncand, c0 + PT_CHUNK);
        // 2) every candidate walks without writing until it marks a candidate
        //    of smaller rank (then it does not own its ring); an owner's walk
        //    gives its ring's vertex count or its failure.  The single walk
        //    ends at the first failing ring: nothing after that owner's rank
        //    matters.  Threads take candidates from a counter in LDS as their
        //    walks end, so a long walk holds one lane, not the others.
        if (tid == 0) {
            s_next = c0 + nthr;
            s_qend = c1;
            s_long = 0;
        }
        __syncthreads();
        for (int q = c0 + tid; q < c1;) {
            if (q >= __hip_atomic_load(&s_qend, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) break;
            int cnt = 0, nst = 0;
            const int res = pt_walk(
                a, cand[q],
                [&](int v) {
                    const int r = a.seen[2 * v];
                    return r > 0 && r < q + 1;
                },
                [&](int, bool, int len) {
                    cnt += len;
                    ++nst;
                });
            if (res == 2) atomicOr(&s_long, 1);
            if (res == 1) atomicMin(&s_qend, q + 1);
            info[q] = res == 3 ? -1 : (res == 1 ? -2 : cnt);
            a.pstep[q] = nst;
            q = atomicAdd(&s_next, 1);
        }
        __syncthreads();
        const int qend = s_qend;
        const bool lng = s_long != 0;
        if (lng) {
            clear();
            return PT_FALLBACK;
        }
        const bool fail = qend < c1 || info[c1 - 1] == -2;
        // 3) ring order: owner r (in the order of the starts) gets ring index
        //    r (kept in its seen[2v], still positive) and its output place
        //    from a running sum (kept in info); then the owners walk again in
        //    any order, and every candidate a walk marks keeps the first ring
        //    that marked it
        const int nring0 = nring;
        const int64_t out0 = int64_t(outn) + nout; // the chunk's first output vertex
        int nrec = 0;                              // the chunk's step records
        bool allw = !fail;                         // every owner of the chunk writes
        for (int q0 = c0; q0 < qend; q0 += nthr) {
            const int q = q0 + tid;
            const int inf = q < qend ? info[q] : -1;
            const bool owner = inf != -1;
            int otot;
            const int oex = seq_block_scan(owner ? 1 : 0, otot, s_w);
            const int64_t c = owner && inf > 0 ? inf : 0;
            int64_t ctot;
            const int64_t cex = seq_block_scan(c, ctot, s_w64);
            int stot;
            const int sex = seq_block_scan(owner ? a.pstep[q] : 0, stot, s_w);
            const int r = nring + oex;
            const int64_t at = int64_t(outn) + nout + cex;
            bool write = true;
            if (owner) {
                write = !fail && rings + r < a.ring_cap && at + c <= a.out_cap;
                if (write) a.ring_off[rings + r] = int(at);
                a.seen[2 * cand[q]] = r + 1;
                info[q] = write ? int(at) : -3; // -3: an owner that writes nothing
                a.pstep[q] = nrec + sex;
            }
            int wtot;
            (void)seq_block_scan(write ? 0 : 1, wtot, s_w);
            if (wtot) allw = false;
            nring += otot;
            nout += ctot;
            nrec += stot;
        }
        // rings that share (node, direction) states can exceed the records'
        // room (2 per node); the single walk then decides
        if (allw && nrec > 2 * a.cap) {
            clear();
            return PT_FALLBACK;
        }
        if (tid == 0) s_next = c0 + nthr;
        __syncthreads();
        for (int q = c0 + tid; q < qend; q = atomicAdd(&s_next, 1)) {
            const int inf = info[q];
            if (inf == -1) continue;
            const int X = cand[q];
            const int tag = SEEN_FIRST - (a.seen[2 * X] - 1);
            const bool write = inf >= 0 && allw;
            int at = inf, k = a.pstep[q];
            (void)pt_walk(
                a, X,
                [&](int v) {
                    if (a.seen[2 * v] > 0) atomicMax(&a.seen[2 * v + 1], tag);
                    return false;
                },
                [&](int v, bool fwd, int len) {
                    if (write) a.emit[k++] = make_int2(v << 1 | (fwd ? 1 : 0), at);
                    at += len;
                });
        }
        __syncthreads();
        // the rings' vertices, one thread per output vertex: the step record
        // of vertex o is the last one placed at or before it (records follow
        // the output order)
        if (allw && nrec > 0) {
            const int O = int(int64_t(outn) + nout - out0);
            for (int o = tid; o < O; o += nthr) {
                const int oo = int(out0) + o;
                int lo = 0, hi = nrec - 1;
                while (lo < hi) {
                    const int mid = (lo + hi + 1) >> 1;
                    if (a.emit[mid].y <= oo) lo = mid;
                    else hi = mid - 1;
                }
                const int2 e = a.emit[lo];
                const int v = e.x >> 1, t = oo - e.y, len = a.rec[v].w >> 2;
                const int u = (e.x & 1) ? t : len - 1 - t;
                const int vs = a.vslot[v];
                const bool onP = v < a.nP;
                double x, y;
                if (vs >= 0 && len > 1) {
                    x = onP ? a.px[vs + u] : a.qx[vs + u];
                    y = onP ? a.py[vs + u] : a.qy[vs + u];
                } else {
                    x = a.vx[v];
                    y = a.vy[v];
                }
                a.ox[oo] = x;
                a.oy[oo] = y;
                a.osrc[oo] = vs >= 0 ? (onP ? a.P0 + vs + u : ~(a.Q0 + vs + u)) : a.vsrc[v];
            }
        }
        __syncthreads();
        // 4) the check: an owner is first marked by its own ring, any other
        //    candidate by a ring whose start comes before it.  At the first
        //    candidate where that does not hold, a candidate no earlier ring
        //    marked is where the single walk starts its next ring: if a full
        //    walk from it fails, the single walk fails there too.
        int before = nring0;
        for (int q0 = c0; q0 < qend; q0 += nthr) {
            const int q = q0 + tid;
            const int inf = q < qend ? info[q] : -1;
            const bool owner = inf != -1;
            int otot;
            const int r = before + seq_block_scan(owner ? 1 : 0, otot, s_w);
            bool bad = false, unmarked = false;
            if (q < qend) {
                const int fv = a.seen[2 * cand[q] + 1];
                const int first = fv > 0 ? SEEN_FIRST - fv : INT_MAX;
                bad = owner ? first != r : first >= r;
                unmarked = !owner && first >= r;
            }
            const int fb = seq_block_min(bad ? tid : INT_MAX, s_w);
            if (fb != INT_MAX) {
                if (tid == fb) {
                    int res = 0;
                    if (unmarked)
                        res = pt_walk(
                            a, cand[q], [&](int) { return false; }, [&](int, bool, int) {});
                    s_res = unmarked && res == 1 ? PT_FAIL : PT_FALLBACK;
                }
                __syncthreads();
                const int out = s_res;
                clear();
                return out;
            }
            before += otot;
        }
        if (fail) {
            clear();
            return PT_FAIL;
        }
    }
    clear();
    if (rings + nring > a.ring_cap || int64_t(outn) + nout > a.out_cap) return PT_FAIL;
    if (tid == 0) {
        sh.rings = rings + nring;
        sh.outn = outn + int(nout);
    }
    return PT_DONE;
}

// The entry/exit walks of the rings marked in sh.scan, on every thread of the
// block: ring s from the node after sh.sV[s] around to sh.sV[s], WAVE x
// waves nodes per round.  Each wave scans its nodes' tables, the waves'
// composed tables give every wave the state the walk enters its nodes in
// (LDS), and each lane applies its node's effect; list appends keep ring
// order (ballot ranks within a wave, counts across waves) and the lists'
// bounds.  Every branch that reaches a barrier depends on LDS values only.
__device__ __attribute__((always_inline)) void seq_enex_block(SeqArgs &a, SeqShared &sh) {
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), wid = tid / WAVE, nw = blockDim.x / WAVE;
    const int nthr = blockDim.x;
    const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (WAVE - lane));
    __shared__ uint32_t s_tab[SEQ_BLK / WAVE];
    __shared__ int s_cs[SEQ_BLK / WAVE], s_cc[SEQ_BLK / WAVE];
    const int half = a.cap / 2, lim = half / 2;
    const bool uni = a.uni != 0;
    for (int s = 0; s < 2; ++s) {
        if (!sh.scan[s]) continue;
        int *splitL = s ? a.cand + half / 2 : a.cand;
        int *crossL = s ? a.cand + half + half / 2 : a.cand + half;
        const int r0 = s ? a.nP : 0, m = s ? a.nQ : a.nP, v0 = sh.sV[s] - r0;
        int state = sh.sst[s] | 2; // first = true
        int nsplit = sh.nsplit[s], ncross = sh.ncross[s];
        for (int pb = 1; pb < m; pb += nthr) {
            const int p = pb + wid * WAVE + lane;
            const bool on = p < m;
            int I = -1, lab = L_NONE;
            bool it = false;
            if (on) {
                I = r0 + (v0 + p >= m ? v0 + p - m : v0 + p);
                lab = a.lab[I];
                it = a.inter[I] != 0;
            }
            uint32_t P = it ? seq_table(lab) : SEQ_TAB_ID;
            for (int d = 1; d < WAVE; d <<= 1) {
                const uint32_t o = uint32_t(__shfl_up(int(P), d, WAVE));
                if (lane >= d) P = seq_tcompose(o, P);
            }
            // lanes past the ring's end hold the identity: lane 63 has the wave's table
            if (lane == WAVE - 1) s_tab[wid] = P;
            __syncthreads();
            int sw = state, send = state;
            for (int w = 0; w < nw; ++w) {
                const uint32_t t = s_tab[w];
                if (w < wid) sw = seq_tapply(t, sw);
                send = seq_tapply(t, send);
            }
            const uint32_t Pex = uint32_t(__shfl_up(int(P), 1, WAVE));
            const int sin = lane == 0 ? sw : seq_tapply(Pex, sw);
            const int sst = sin & 1;
            const bool sfirst = (sin >> 1) != 0;
            bool addS = false, addC = false;
            if (it) {
                if (lab == L_CROSSING) {
                    a.enex[I] = sst;
                } else if (lab == L_BOUNCING) {
                    addS = (sst == EXIT) != uni;
                } else if (lab == L_DCROSS) {
                    a.enex[I] = sst;
                    if (sfirst ? ((sst == EXIT) != uni) : ((sst == ENTRY) != uni)) a.lab[I] = L_CROSSING;
                } else if (lab == L_DBOUNCE) {
                    a.enex[I] = sst;
                    addC = sfirst ? ((sst == EXIT) != uni) : ((sst == ENTRY) != uni);
                }
            }
            const uint64_t ms = __ballot(addS), mc = __ballot(addC);
            if (lane == 0) {
                s_cs[wid] = int(__popcll(ms));
                s_cc[wid] = int(__popcll(mc));
            }
            __syncthreads();
            int bs = 0, bc = 0, ts = 0, tc = 0;
            for (int w = 0; w < nw; ++w) {
                const int cs = s_cs[w], cc = s_cc[w];
                if (w < wid) {
                    bs += cs;
                    bc += cc;
                }
                ts += cs;
                tc += cc;
            }
            if (addS) {
                const int q = nsplit + bs + int(__popcll(ms & lt));
                if (q < lim) splitL[q] = I;
            }
            if (addC) {
                const int q = ncross + bc + int(__popcll(mc & lt));
                if (q < lim) crossL[q] = I;
            }
            nsplit = min(nsplit + ts, lim);
            ncross = min(ncross + tc, lim);
            state = send;
            __syncthreads(); // s_tab, s_cs and s_cc are rewritten next round
        }
        if (tid == 0) {
            sh.nsplit[s] = nsplit;
            sh.ncross[s] = ncross;
        }
    }
}

// The reference's sequential algorithm on the job's rings, run by one wave
// with uniform control flow: every lane holds the same walk state.  Part 0
// runs the steps before the entry/exit walks and leaves its state in sh
// (sh.go = 2), part 2 the steps after them up to createResult2's walks
// (sh.go = 1); either writes the job's result instead when it fails (sh.go =
// 0).  Part 1 takes the walks' outcome (sh.ptr), runs the single walk when
// they fell back, and writes the result.  Lane i
// caches the hot fields of node w0 + i (a window of 64 consecutive nodes,
// w0 a multiple of 64), so a walk in ring order reads registers and reloads
// one coalesced window every 64 nodes.  Every write goes to memory (from all
// lanes, the same value) and to the window.  Output runs are written one
// vertex per lane.
__device__ __attribute__((always_inline)) void seq_run(SeqArgs &a, SeqShared &sh, int part) {
    const int lane = threadIdx.x & (WAVE - 1);
    int status = 0;
    // ring nodes already laid out by seq_init: P = [0,nP), Q = [nP,nP+nQ)
    int n = a.nP + a.nQ;
    int w0 = -(1 << 30);
    int c_nx = 0, c_pv = 0, c_nb = 0, c_lab = 0, c_enex = 0, c_inter = 0;
    int c_seen0 = 0, c_seen1 = 0, c_vlen = 0, c_vslot = 0;
    auto fill = [&](int I) {
        w0 = I & ~(WAVE - 1);
        const int j = w0 + lane;
        if (j < n) {
            c_nx = a.nx[j];
            c_pv = a.pv[j];
            c_nb = a.nb[j];
            c_lab = a.lab[j];
            c_enex = a.enex[j];
            c_inter = a.inter[j];
            const int2 sn = reinterpret_cast<const int2 *>(a.seen)[j];
            c_seen0 = sn.x;
            c_seen1 = sn.y;
            c_vlen = a.vlen[j];
            c_vslot = a.vslot[j];
        }
        // wait for the window here, so that its later reads wait for nothing
        // (the walk's own stores share the same counter)
        __builtin_amdgcn_s_waitcnt(0x0f70); // vmcnt(0), other counters free
    };
    auto slot = [&](int I) {
        if (unsigned(I - w0) >= unsigned(WAVE)) fill(I);
        return I - w0;
    };
    auto NX_ = [&](int I) { const int k = slot(I); return __builtin_amdgcn_readlane(c_nx, k); };
    auto PV_ = [&](int I) { const int k = slot(I); return __builtin_amdgcn_readlane(c_pv, k); };
    auto NB_ = [&](int I) { const int k = slot(I); return __builtin_amdgcn_readlane(c_nb, k); };
    auto LAB_ = [&](int I) { const int k = slot(I); return __builtin_amdgcn_readlane(c_lab, k); };
    auto ENEX_ = [&](int I) { const int k = slot(I); return __builtin_amdgcn_readlane(c_enex, k); };
    auto INTER_ = [&](int I) { const int k = slot(I); return __builtin_amdgcn_readlane(c_inter, k); };
    auto VLEN_ = [&](int I) { const int k = slot(I); return __builtin_amdgcn_readlane(c_vlen, k); };
    auto VSLOT_ = [&](int I) { const int k = slot(I); return __builtin_amdgcn_readlane(c_vslot, k); };
    // the traversal's state words, 2 per node (direction d)
    auto SEEN_ = [&](int I, int d) {
        const int k = slot(I);
        return d ? __builtin_amdgcn_readlane(c_seen1, k) : __builtin_amdgcn_readlane(c_seen0, k);
    };
    auto set_seen = [&](int I, int d, int v) {
        a.seen[2 * I + d] = v;
        if (I - w0 == lane) {
            if (d) c_seen1 = v;
            else c_seen0 = v;
        }
    };
    auto set_nx = [&](int I, int v) { a.nx[I] = v; if (I - w0 == lane) c_nx = v; };
    auto set_pv = [&](int I, int v) { a.pv[I] = v; if (I - w0 == lane) c_pv = v; };
    auto set_nb = [&](int I, int v) { a.nb[I] = v; if (I - w0 == lane) c_nb = v; };
    auto set_lab = [&](int I, int v) { a.lab[I] = v; if (I - w0 == lane) c_lab = v; };
    auto set_enex = [&](int I, int v) { a.enex[I] = v; if (I - w0 == lane) c_enex = v; };
    auto set_inter = [&](int I, int v) { a.inter[I] = uint8_t(v); if (I - w0 == lane) c_inter = v; };
    // a new single-vertex node (its own ring until inserted), -1 when full
    auto snew = [&](double x, double y, int src) -> int {
        if (n >= a.cap) return -1;
        const int v = n++;
        a.vx[v] = x;
        a.vy[v] = y;
        a.vx1[v] = x;
        a.vy1[v] = y;
        a.vlen[v] = 1;
        a.vslot[v] = -1;
        a.vsrc[v] = src;
        if (v - w0 == lane) {
            c_vlen = 1;
            c_vslot = -1;
            c_seen0 = c_seen1 = 0; // zeroed with the rest at set-up
        }
        set_nx(v, v);
        set_pv(v, v);
        set_nb(v, -1);
        set_lab(v, L_NONE);
        set_enex(v, NEITHER);
        set_inter(v, 0);
        return v;
    };
    auto sinsert = [&](int V, int curr) {
        const int c = NX_(curr);
        set_nx(PV_(c), V);
        set_pv(V, PV_(c));
        set_nx(V, c);
        set_pv(c, V);
    };
    // the vertices of node V, walking forward or backward, one per lane
    auto semit = [&](int &outn, int V, bool forward) -> bool {
        const int len = VLEN_(V);
        if (outn + len > a.out_cap) return false;
        const int vs = VSLOT_(V);
        const bool onP = V < a.nP;
        for (int t0 = 0; t0 < len; t0 += WAVE) {
            const int t = t0 + lane;
            if (t < len) {
                const int u = forward ? t : len - 1 - t;
                double x, y;
                seq_vertex(a, V, u, x, y);
                a.ox[outn + t] = x;
                a.oy[outn + t] = y;
                a.osrc[outn + t] = vs >= 0 ? (onP ? a.P0 + vs + u : ~(a.Q0 + vs + u)) : a.vsrc[V];
            }
        }
        outn += len;
        return true;
    };
    const int rootP = 0, rootQ = a.nP;
    const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (WAVE - lane));
    if (part == 1) {
        n = sh.n;
        status = sh.status;
        int rings = sh.rings, outn = sh.outn;
        if (sh.ptr == PT_FAIL) goto done;
        if (sh.ptr == PT_FALLBACK) {
            int root = rootP, I = root;
            bool have = INTER_(I) && LAB_(I) == L_CROSSING;
            if (!have) {
                do { I = NX_(I); } while (!(INTER_(I) && LAB_(I) == L_CROSSING) && I != root);
                have = I != root;
            }
            long bound = 4L * n + 16;
            int comp = 0;
            while (have) {
                if (rings >= a.ring_cap) goto done;
                a.ring_off[rings++] = outn;
                int V = I;
                set_inter(V, 0);
                long steps = 0;
                ++comp;
                do {
                    int st = seq_toggle(ENEX_(V));
                    do {
                        const bool fwd = (st == EXIT) != (a.uni != 0); // (status == EXIT) ^ UNION, polyclip.h:740
                        V = fwd ? NX_(V) : PV_(V);
                        set_inter(V, 0);
                        // within one component the walk is determined by (vertex, direction):
                        // a repeated state can never reach I again (the reference loops forever)
                        const int dir = fwd ? 1 : 0;
                        if (SEEN_(V, dir) == comp) goto done;
                        set_seen(V, dir, comp);
                        if (++steps > bound || !semit(outn, V, fwd)) goto done;
                    } while (!(ENEX_(V) == st) && V != I);
                    if (V != I) {
                        V = NB_(V);
                        if (V < 0) goto done;
                        set_inter(V, 0);
                    }
                } while (V != I);
                do { I = NX_(I); } while (!(INTER_(I) && LAB_(I) == L_CROSSING) && I != root);
                have = I != root;
            }
        }
        a.ring_off[rings] = outn;
        a.result[0] = rings;
        a.result[1] = outn;
        a.result[2] = status;
        return;
    }
    if (part == 2) {
        n = sh.n;
        status = sh.status;
        const int rings = sh.rings, outn = sh.outn;
        const int half = a.cap / 2;
        const int nsplit[2] = {sh.nsplit[0], sh.nsplit[1]}, ncross[2] = {sh.ncross[0], sh.ncross[1]};
        int *splitL[2] = {a.cand, a.cand + half / 2};
        int *crossL[2] = {a.cand + half, a.cand + half + half / 2};
        // membership of the Q lists, marked in the traversal's (still zero)
        // state words: -1 in slot 2V for the split list, in 2V+1 for the crossing list
        const int nmark = n;
        for (int j = 0; j < nsplit[1]; ++j) set_seen(splitL[1][j], 0, -1);
        for (int j = 0; j < ncross[1]; ++j) set_seen(crossL[1][j], 1, -1);
        // 5) split interior bouncing pairs
        for (int i = 0; i < nsplit[0]; ++i) {
            int IP = splitL[0][i], IQ = NB_(IP);
            if (!(IQ >= 0 && IQ < nmark && SEEN_(IQ, 0) == -1)) continue;
            int VP = snew(a.vx[IP], a.vy[IP], seq_src(a, IP));
            int VQ = snew(a.vx[IQ], a.vy[IQ], seq_src(a, IQ));
            if (VP < 0 || VQ < 0) { status |= UB_TRAVERSAL; goto done; }
            // the vertex before IP is the last vertex of its previous node, the one after the first of the next
            double sP = areaA(a.vx1[PV_(IP)], a.vy1[PV_(IP)], a.vx[IP], a.vy[IP], a.vx[NX_(IP)], a.vy[NX_(IP)]);
            double sQ = areaA(a.vx1[PV_(IQ)], a.vy1[PV_(IQ)], a.vx[IQ], a.vy[IQ], a.vx[NX_(IQ)], a.vy[NX_(IQ)]);
            if (sP * sQ > 0) {
                set_nb(IP, VQ); set_nb(VQ, IP); set_inter(IP, 1); set_inter(VQ, 1);
                set_nb(IQ, VP); set_nb(VP, IQ); set_inter(IQ, 1); set_inter(VP, 1);
            } else {
                set_nb(VP, VQ); set_nb(VQ, VP); set_inter(VP, 1); set_inter(VQ, 1);
            }
            sinsert(VP, IP);
            sinsert(VQ, IQ);
            if (!a.uni) {
                set_enex(IP, EXIT); set_enex(VP, ENTRY); set_enex(IQ, EXIT); set_enex(VQ, ENTRY);
            } else {
                set_enex(IP, ENTRY); set_enex(VP, EXIT); set_enex(IQ, ENTRY); set_enex(VQ, EXIT);
            }
            set_lab(IP, L_CROSSING); set_lab(VP, L_CROSSING); set_lab(IQ, L_CROSSING); set_lab(VQ, L_CROSSING);
        }
        // 6) crossing candidates
        for (int i = 0; i < ncross[0]; ++i) {
            int IP = crossL[0][i], IQ = NB_(IP);
            if (IQ >= 0 && IQ < nmark && SEEN_(IQ, 1) == -1) {
                set_lab(IP, L_CROSSING);
                set_lab(IQ, L_CROSSING);
            }
        }
        for (int j = 0; j < nsplit[1]; ++j) set_seen(splitL[1][j], 0, 0);
        for (int j = 0; j < ncross[1]; ++j) set_seen(crossL[1][j], 1, 0);
        // createResult2.  First the walks run one per lane (seq_par_traverse,
        // every wave of the block): every candidate start (a P crossing, in
        // ring order from the root) walks its ring without writing; the
        // candidate with the smallest rank on a ring owns it; the owners walk
        // again and write the rings.  The reference's single walk starts a
        // ring at the first candidate that no earlier ring visited, so the
        // result is the same when every owner is first visited by its own
        // ring and every other candidate by a ring that starts before it;
        // that is checked, and otherwise (or when a walk is too long or too
        // many nodes were inserted) the single walk of part 1 runs.
        __threadfence_block(); // this wave's stores, before the other waves read them
        if (lane == 0) {
            sh.n = n;
            sh.status = status;
            sh.rings = rings;
            sh.outn = outn;
            sh.go = 1;
        }
        return;
    }
    // 2) intersection chains.  Before any insertion ring P is nodes [0, nP) in
    // ring order from its root, so the chain starts (intersections labelled
    // LEFT_ON or RIGHT_ON) are found 64 nodes per ballot, in that order, and
    // walked one after another.  A start that an earlier chain relabelled is
    // checked again and skipped, and a later block reads the labels the chains
    // before it wrote: the reference's single walk, step for step.
    for (int w = 0; w < a.nP; w += WAVE) {
        const int v = w + lane;
        bool start = false;
        if (v < a.nP) {
            const int lb = a.lab[v];
            start = a.inter[v] != 0 && (lb == L_LEFT_ON || lb == L_RIGHT_ON);
        }
        uint64_t starts = __ballot(start);
        while (starts) {
            const int I = w + __builtin_ctzll(starts);
            starts &= starts - 1ull;
            if (INTER_(I) && (LAB_(I) == L_LEFT_ON || LAB_(I) == L_RIGHT_ON)) {
                int x = LAB_(I) == L_LEFT_ON ? 0 : 1;
                int X = I, J = I, guard = 0;
                do {
                    set_lab(J, L_NONE);
                    if (NB_(J) >= 0) set_lab(NB_(J), L_NONE);
                    J = NX_(J);
                    if (++guard > n) { status |= UB_TRAVERSAL; goto done; }
                } while (LAB_(J) == L_ON_ON);
                int y = LAB_(J) == L_ON_LEFT ? 0 : 1;
                int ct = x != y ? L_DCROSS : L_DBOUNCE;
                set_lab(X, ct);
                set_lab(J, ct);
                if (NB_(X) >= 0) set_lab(NB_(X), ct);
                if (NB_(J) >= 0) set_lab(NB_(J), ct);
            }
        }
    }
    {
        int rings = 0, outn = 0;
        int roots[2] = {rootP, rootQ};
        bool noInter[2] = {false, false}, ident[2] = {false, false};
        // rings in index order (no insertion yet): ring s is nodes [ring0[s], ring0[s] + ringn[s])
        const int ring0[2] = {rootP, rootQ}, ringn[2] = {a.nP, a.nQ};
        // the ring's first node in ring order that is not an intersection, or -1
        auto first_plain = [&](int s) {
            for (int w = 0; w < ringn[s]; w += WAVE) {
                const int v = ring0[s] + w + lane;
                const uint64_t m = __ballot(w + lane < ringn[s] && a.inter[v] == 0);
                if (m) return ring0[s] + w + int(__builtin_ctzll(m));
            }
            return -1;
        };
        // 3.5) rings without crossing vertices (64 nodes per ballot)
        for (int s = 0; s < 2; ++s) {
            int A = roots[s], B = roots[1 - s];
            bool nocross = true, allon = true;
            int V = A;
            for (int w = 0; w < ringn[s] && nocross; w += WAVE) {
                const int v = ring0[s] + w + lane;
                bool cr = false, notOn = false;
                if (w + lane < ringn[s]) {
                    const int lb = a.lab[v];
                    const bool it = a.inter[v] != 0;
                    cr = it && (lb == L_CROSSING || lb == L_DCROSS);
                    // polygon::noCrossingVertex(union_case), polygon.h:465-475
                    if (a.uni && it && (lb == L_BOUNCING || lb == L_DBOUNCE)) cr = true;
                    notOn = lb != L_ON_ON;
                }
                if (__ballot(cr)) nocross = false;
                if (__ballot(notOn)) allon = false;
            }
            if (!nocross) continue;
            noInter[s] = true;
            if (allon) {
                ident[s] = true;
                continue;
            }
            double qx = 0, qy = 0;
            bool found = false, plain = false;
            V = first_plain(s);
            if (V >= 0) {
                qx = a.vx[V];
                qy = a.vy[V];
                found = plain = true;
            }
            if (!found) {
                V = A;
                do {
                    int nxv = NX_(V), nbv = NB_(V);
                    if (nbv >= 0 && NB_(nxv) != PV_(nbv) && NB_(nxv) != NX_(nbv)) {
                        qx = 0.5 * (a.vx[V] + a.vx[nxv]);
                        qy = 0.5 * (a.vy[V] + a.vy[nxv]);
                        found = true;
                        break;
                    }
                    V = NX_(V);
                } while (V != A);
            }
            if (!found) { status |= UB_TRAVERSAL; goto done; }
            // the ring's first plain vertex: its winding against the other ring is known
            const bool in = plain ? ((s == 0 ? a.windP : a.windQ) % 2) != 0 : seq_point_in(a, B, qx, qy);
            if (in != (a.uni != 0)) { // isInside ^ UNION, polyclip.h:470
                if (rings >= a.ring_cap) { status |= UB_TRAVERSAL; goto done; }
                a.ring_off[rings++] = outn;
                int W = A;
                do {
                    if (!semit(outn, W, true)) { status |= UB_TRAVERSAL; goto done; }
                    W = NX_(W);
                } while (W != A);
            }
        }
        if (ident[0] && ident[1]) {
            int target = NB_(rootP), V = rootQ;
            bool found = false;
            do {
                if (V == target) found = true;
                V = NX_(V);
            } while (V != rootQ);
            if (found) {
                if (rings >= a.ring_cap) { status |= UB_TRAVERSAL; goto done; }
                a.ring_off[rings++] = outn;
                int W = rootP;
                do {
                    if (!semit(outn, W, true)) { status |= UB_TRAVERSAL; goto done; }
                    W = NX_(W);
                } while (W != rootP);
            }
        }
        // 4) entry/exit flags; split and crossing candidates in scratch
        int nsplit[2] = {0, 0}, ncross[2] = {0, 0};
        bool inserted[2] = {false, false};
        int half = a.cap / 2; // cand[0..half) split lists, [half..cap) crossing lists
        int *splitL[2] = {a.cand, a.cand + half / 2};
        int *crossL[2] = {a.cand + half, a.cand + half + half / 2};
        // the entry/exit walk's state (status, first of a delayed pair) as 2 bits
        // x = st | first << 1 (EXIT = 0, ENTRY = 1); a node's effect on it is a
        // 4-entry table of 2-bit states, and tables compose along the ring
        if (lane == 0) sh.scan[0] = sh.scan[1] = 0;
        for (int s = 0; s < 2; ++s) {
            if (noInter[s]) continue;
            int A = roots[s], B = roots[1 - s];
            int V = first_plain(s), W = A; // ring s has no inserted node yet
            if (V < 0) {
                W = A;
                do {
                    int nxv = NX_(W), nbv = NB_(W);
                    if (nbv >= 0 && NB_(nxv) != PV_(nbv) && NB_(nxv) != NX_(nbv)) {
                        int T = snew(0.5 * (a.vx[W] + a.vx[nxv]), 0.5 * (a.vy[W] + a.vy[nxv]), SRC_NONE);
                        if (T < 0) { status |= UB_TRAVERSAL; goto done; }
                        sinsert(T, W);
                        inserted[s] = true;
                        V = T;
                        break;
                    }
                    W = NX_(W);
                } while (W != A);
            }
            if (V < 0) { status |= UB_TRAVERSAL; goto done; }
            int st = ENTRY;
            // V is the ring's first plain vertex unless a midpoint had to be inserted;
            // its winding against ring B is known while B has no inserted vertex
            const bool known = a.vslot[V] >= 0 && !inserted[1 - s];
            const bool in = known ? ((s == 0 ? a.windP : a.windQ) % 2) != 0 : seq_point_in(a, B, a.vx[V], a.vy[V]);
            if (in) st = seq_toggle(st);
            bool first = true;
            if (!inserted[s]) {
                // the walk from the node after V around to V runs on every wave
                // (seq_enex_block); no other step before it reads this ring's
                // labels or lists
                if (lane == 0) {
                    sh.scan[s] = 1;
                    sh.sV[s] = V;
                    sh.sst[s] = st;
                }
                continue;
            }
            int I = NX_(V);
            while (I != V) {
                if (INTER_(I)) {
                    int lab = LAB_(I);
                    if (lab == L_CROSSING) {
                        set_enex(I, st);
                        st = seq_toggle(st);
                    }
                    if (lab == L_BOUNCING && ((st == EXIT) != (a.uni != 0)) && nsplit[s] < half / 2)
                        splitL[s][nsplit[s]++] = I;
                    if (lab == L_DCROSS) {
                        set_enex(I, st);
                        if (first) {
                            if ((st == EXIT) != (a.uni != 0)) set_lab(I, L_CROSSING);
                            first = false;
                        } else {
                            if ((st == ENTRY) != (a.uni != 0)) set_lab(I, L_CROSSING);
                            first = true;
                            st = seq_toggle(st);
                        }
                    }
                    if (lab == L_DBOUNCE) {
                        set_enex(I, st);
                        if (first) {
                            if (((st == EXIT) != (a.uni != 0)) && ncross[s] < half / 2) crossL[s][ncross[s]++] = I;
                            first = false;
                        } else {
                            if (((st == ENTRY) != (a.uni != 0)) && ncross[s] < half / 2) crossL[s][ncross[s]++] = I;
                            first = true;
                        }
                        st = seq_toggle(st);
                    }
                }
                I = NX_(I);
            }
        }
        __threadfence_block(); // this wave's stores, before the other waves read them
        if (lane == 0) {
            sh.n = n;
            sh.status = status;
            sh.rings = rings;
            sh.outn = outn;
            sh.nsplit[0] = nsplit[0];
            sh.nsplit[1] = nsplit[1];
            sh.ncross[0] = ncross[0];
            sh.ncross[1] = ncross[1];
            sh.go = 2;
        }
        return;
    }
done:
    if (lane == 0) sh.go = 0;
    a.result[0] = 0;
    a.result[1] = 0;
    a.result[2] = status | UB_TRAVERSAL;
    a.ring_off[0] = 0;
}


// one block per sequential job: its threads lay out the rings, its first wave
// runs the algorithm (no barrier after that point)
__global__ __launch_bounds__(SEQ_BLK) void k_sequential(SeqBatch b) {
    if (b.done && b.done[blockIdx.x]) return;
    const SeqJob jb = b.jobs[blockIdx.x];
    SeqArgs a;
    a.nP = jb.nPn;
    a.nQ = jb.nQn;
    a.cap = jb.cap;
    a.P0 = jb.P0;
    a.Q0 = jb.Q0;
    a.uni = b.uni;
    a.par = b.par;
    a.nx0 = b.nx0 + jb.node0; a.ny0 = b.ny0 + jb.node0; a.nx1 = b.nx1 + jb.node0; a.ny1 = b.ny1 + jb.node0;
    a.nlen = b.nlen + jb.node0; a.nslot = b.nslot + jb.node0; a.ninter = b.ninter + jb.node0;
    a.nlab = b.nlab + jb.node0; a.nnb = b.nnb + jb.node0;
    a.px = b.px + jb.P0; a.py = b.py + jb.P0; a.qx = b.qx + jb.Q0; a.qy = b.qy + jb.Q0;
    a.windP = b.windP[jb.j];
    a.windQ = b.windQ[jb.j];
    a.vx = b.vx + jb.vbase; a.vy = b.vy + jb.vbase; a.vx1 = b.vx1 + jb.vbase; a.vy1 = b.vy1 + jb.vbase;
    a.vlen = b.vlen + jb.vbase; a.vslot = b.vslot + jb.vbase;
    a.nx = b.nx + jb.vbase; a.pv = b.pv + jb.vbase; a.nb = b.nb + jb.vbase; a.lab = b.lab + jb.vbase;
    a.enex = b.enex + jb.vbase; a.vsrc = b.vsrc + jb.vbase; a.cand = b.cand + jb.vbase;
    a.seen = b.seen + 2 * jb.vbase;
    a.rec = b.rec + jb.vbase;
    a.pstep = b.pstep + jb.vbase;
    a.emit = b.emit + 2 * jb.vbase;
    a.inter = b.inter + jb.vbase;
    a.ox = b.ox + jb.obase; a.oy = b.oy + jb.obase; a.osrc = b.osrc + jb.obase; a.out_cap = jb.out_cap;
    a.ring_off = b.ring_off + jb.rbase; a.ring_cap = jb.ring_cap;
    a.result = b.result + 3 * int64_t(blockIdx.x);
    if (jb.nPn + jb.nQn > jb.cap) { // cannot happen: cap is sized from the node counts
        if (threadIdx.x == 0) {
            a.result[0] = 0;
            a.result[1] = 0;
            a.result[2] = UB_TRAVERSAL;
            a.ring_off[0] = 0;
        }
        return;
    }
    __shared__ SeqShared sh;
    if (threadIdx.x == 0) sh.go = 0;
    __syncthreads();
    if (threadIdx.x < WAVE) seq_run(a, sh, 0); // wave 0: the steps before the entry/exit walks
    __syncthreads();
    if (!sh.go) return; // the job's result is written
    seq_enex_block(a, sh); // every wave
    __syncthreads();
    if (threadIdx.x < WAVE) seq_run(a, sh, 2); // wave 0: split and crossing candidates
    __syncthreads();
    if (!sh.go) return;
    const int ptr = a.par ? seq_par_traverse(a, sh) : PT_FALLBACK; // every wave
    __syncthreads();
    if (threadIdx.x == 0) sh.ptr = ptr;
    __syncthreads();
    if (threadIdx.x < WAVE) seq_run(a, sh, 1); // wave 0: the single walk if needed, the result
}

// Every sequential job's working rings before any insertion: its P and Q
// rings in node order (node v of the job at slot vbase + v), nothing
// inserted, no walk state.  Job q owns nodes [nodeoff[2q], nodeoff[2q+2]).
// Again before k_sequential for the jobs that the device-wide steps left.
__global__ void k_seq_init(SeqBatch b, const int64_t *__restrict__ nodeoff, int nseq, int64_t N) {
    const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= N) return;
    int lo = 0, hi = nseq - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (nodeoff[2 * mid] <= t) lo = mid;
        else hi = mid - 1;
    }
    if (b.done && b.done[lo]) return;
    const SeqJob &jb = b.jobs[lo];
    const int v = int(t - jb.node0);
    const int64_t w = jb.vbase + v;
    b.seen[2 * w] = 0;
    b.seen[2 * w + 1] = 0;
    b.vx[w] = b.nx0[t];
    b.vy[w] = b.ny0[t];
    b.vx1[w] = b.nx1[t];
    b.vy1[w] = b.ny1[t];
    b.vlen[w] = b.nlen[t];
    b.vslot[w] = b.nslot[t];
    b.vsrc[w] = SRC_NONE;
    b.lab[w] = b.nlab[t];
    const bool it = b.ninter[t] != 0;
    b.inter[w] = it ? 1 : 0;
    b.enex[w] = NEITHER;
    b.nb[w] = it ? b.nnb[t] : -1;
    const bool onP = v < jb.nPn;
    const int r0 = onP ? 0 : jb.nPn, m = onP ? jb.nPn : jb.nQn, i = v - r0;
    b.nx[w] = r0 + (i + 1 == m ? 0 : i + 1);
    b.pv[w] = r0 + (i == 0 ? m - 1 : i - 1);
}

// Ring nodes of the sequential jobs: every intersection slot is a node, every
// maximal run of plain slots is one node.  Segment g = 2q (ring P of sequential
// job q) or 2q+1 (its ring Q) covers flat slots [segoff[g], segoff[g+1]).
struct NodeArgs {
    int nseg;
    const int64_t *segoff;
    const SeqJob *jobs;
    const double *px, *py, *qx, *qy;
    const int *avP, *labP, *nbrP, *labQ, *nbrQ;
};

__device__ inline bool node_inter(const NodeArgs &a, int g, int s) {
    const SeqJob &jb = a.jobs[g >> 1];
    return (g & 1) ? a.nbrQ[jb.Q0 + s] != -100 : a.avP[jb.P0 + s] != -100;
}

// node offset of every segment: the node-start scan at the segment's first slot
__global__ void k_seg_node_offsets(int nseg, const int64_t *segoff, const uint32_t *nidx, int64_t *nodeoff) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g <= nseg) nodeoff[g] = int64_t(nidx[segoff[g]]);
}

__global__ void k_node_flags(NodeArgs a, int64_t S, uint32_t *flag) {
    const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= S) return;
    int lo = 0, hi = a.nseg - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (a.segoff[mid] <= t) lo = mid;
        else hi = mid - 1;
    }
    const int g = lo, s = int(t - a.segoff[g]);
    flag[t] = (s == 0 || node_inter(a, g, s) || node_inter(a, g, s - 1)) ? 1u : 0u;
}

// node records (start slot, interior flag, first vertex, label, neighbour slot)
__global__ void k_node_fill(NodeArgs a, int64_t S, const uint32_t *flag, const uint32_t *nidx, int *nslot,
                            int *ninter, double *nx0, double *ny0, int *nlab, int *nnb) {
    const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= S || !flag[t]) return;
    int lo = 0, hi = a.nseg - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (a.segoff[mid] <= t) lo = mid;
        else hi = mid - 1;
    }
    const int g = lo, s = int(t - a.segoff[g]);
    const SeqJob &jb = a.jobs[g >> 1];
    const uint32_t k = nidx[t];
    const bool onQ = g & 1;
    const bool in = node_inter(a, g, s);
    nslot[k] = s;
    ninter[k] = in ? 1 : 0;
    nx0[k] = onQ ? a.qx[jb.Q0 + s] : a.px[jb.P0 + s];
    ny0[k] = onQ ? a.qy[jb.Q0 + s] : a.py[jb.P0 + s];
    nlab[k] = onQ ? a.labQ[jb.Q0 + s] : a.labP[jb.P0 + s];
    nnb[k] = in ? (onQ ? a.nbrQ[jb.Q0 + s] : a.nbrP[jb.P0 + s]) - 1 : -1;
}

// run lengths, last vertices and neighbour nodes (node indices local to the job)
__global__ void k_node_finish(NodeArgs a, int64_t N, const int64_t *nodeoff, const uint32_t *flag,
                              const uint32_t *nidx, const int *nslot, const int *ninter, int *nlen, double *nx1,
                              double *ny1, int *nnb) {
    const int64_t k = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (k >= N) return;
    int lo = 0, hi = a.nseg - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (nodeoff[mid] <= k) lo = mid;
        else hi = mid - 1;
    }
    const int g = lo;
    const SeqJob &jb = a.jobs[g >> 1];
    const bool onQ = g & 1;
    const int nsl = int(a.segoff[g + 1] - a.segoff[g]);
    const int end = k + 1 < nodeoff[g + 1] ? nslot[k + 1] : nsl;
    const int len = end - nslot[k];
    nlen[k] = len;
    const int sl = nslot[k] + len - 1;
    nx1[k] = onQ ? a.qx[jb.Q0 + sl] : a.px[jb.P0 + sl];
    ny1[k] = onQ ? a.qy[jb.Q0 + sl] : a.py[jb.P0 + sl];
    if (ninter[k]) {
        const int og = g ^ 1; // the other ring of the same job
        const int w = nnb[k];
        const int on = int(a.segoff[og + 1] - a.segoff[og]);
        if (w < 0 || w >= on) {
            nnb[k] = -1;
        } else {
            const int64_t t = a.segoff[og] + w;
            const int64_t node = int64_t(nidx[t]) + int64_t(flag[t]) - 1; // node holding that slot
            nnb[k] = int(node - nodeoff[g & ~1]);
        }
    }
}

// rings of the sequential jobs into the batch output (one block per job)
__global__ void k_jseq_copy(const SeqJob *jobs, const int *done, const int *result, const uint32_t *JV, const uint32_t *JR,
                            const double *sx, const double *sy, const int *ssrc, const int *sroff, double *ox,
                            double *oy, int *osrc, int *off) {
    if (done && done[blockIdx.x]) return; // written by walk_emit
    const SeqJob jb = jobs[blockIdx.x];
    const int rings = result[3 * blockIdx.x], verts = result[3 * blockIdx.x + 1];
    const int64_t o = JV[jb.j];
    for (int i = threadIdx.x; i < verts; i += blockDim.x) {
        ox[o + i] = sx[jb.obase + i];
        oy[o + i] = sy[jb.obase + i];
        osrc[o + i] = ssrc[jb.obase + i];
    }
    for (int r = threadIdx.x; r < rings; r += blockDim.x) off[JR[jb.j] + r] = int(o + sroff[jb.rbase + r]);
}

// scratch owned by this stage
struct FosterScratch {
    DBuf<uint32_t> crossP, crossQ, ccP, ccQ;
    DBuf<uint32_t> jring; // per job first ring after clean-up, then the output totals
    DBuf<int> enexP, enexQ, cposP, cposQ;
    DBuf<int> ppos, plen, pdir, pj;
    DBuf<int4> piece;        // per crossing what the output needs of its piece
    DBuf<uint4> jrec, jrec2, jrule; // records of the crossing cycles, of their rulers
    DBuf<uint2> jcov, jend;         // per crossing: its ruler; its cycle's minimum and the distance to it
    DBuf<uint32_t> succ, val, ringid, inode, dist, tot, isstart, ringidx, head, linkP, linkQ;
    DBuf<int> jst;
    DBuf<uint32_t> jv, jr;
    DBuf<double> ox, oy, qpts, mx, my, nx0, ny0, nx1, ny1, vx1, vy1;
    DBuf<int> osrc, qoks, mav, mnbr, mlab, mjob, nslot, ninter, nlab, nnb, nlen, vlen, vslot, seen;
    DBuf<int64_t> moff, segoff, nodeoff;
    DBuf<uint32_t> nflag, nidx;
    DBuf<int> off, rstart;
    DBuf<uint32_t> keep, kscan, rcnt, nonempty, kctl, ktstate;
    // sequential route
    DBuf<SeqJob> sjobs;
    DBuf<int> sres, sroff, sosrc;
    DBuf<double> vx, vy, sox, soy;
    DBuf<int> nx, pv, nb, lab, enex, vsrc, cand;
    DBuf<uint8_t> inter;
    DBuf<int4> srec;
    DBuf<uint32_t> jmoved; // per doubling round: some cycle minimum moved
    DBuf<int> spstep;
    DBuf<int2> semit;
    DBuf<int> sdone;
};

FosterScratch &fscratch() {
    thread_local FosterScratch *p = new FosterScratch();
    return *p;
}

template <class T> void d2h_sync(Ctx &c, T *h, const T *d, int64_t n) {
    ReadBack rb(c);
    rb.add(h, d, size_t(n));
    rb.run();
}

// clean-up of nr rings laid out at off[0..nr] in (ox, oy, osrc), the vertices'
// rings in ringid and keep's closing entry and the round flags cleared by the
// caller; result into Ctx.  job_ring gets, per job, its first ring after it (J+1
// entries, from the jobs' first rings before it, jr on the device)
void cleanup_rings(Ctx &c, FosterScratch &f, int nr, int64_t n, int J, const uint32_t *jr,
                   std::vector<uint32_t> &job_ring) {
    hipStream_t s = c.stream;
    int *dring = c.jobs.d_ring.ensure(size_t(J) + 1); // job_ring on the device, for the areas
    if (nr == 0 || n == 0) {
        job_ring.assign(size_t(J) + 1, 0u);
        c.nrings = 0;
        c.n_out = 0;
        FillBatch fb(s);
        fb.add(c.d_ring_off.ensure(1), 1, 0u);
        fb.add(dring, int64_t(J) + 1, 0u);
        fb.flush();
        c.wait(); // the labelling's scratch is the host thread's, for any context and stream
        return;
    }
    int *rstart = f.rstart.ensure(nr);
    k_root_loop<<<grid_for(nr), BLK, 0, s>>>(nr, f.off, f.ox, f.oy, rstart);
    uint32_t *keep = f.keep;
    const int64_t ntiles = (n + KEEP_TILE - 1) / KEEP_TILE;
    uint32_t *changed = f.kctl;
    uint32_t *state = f.ktstate.ensure(3 * size_t(ntiles));
    uint32_t *nonempty = f.nonempty.ensure(size_t(nr) + 1);
    KeepArgs ka;
    ka.n = n;
    ka.ringid = reinterpret_cast<const int *>(f.ringid.p);
    ka.off = f.off;
    ka.rstart = rstart;
    ka.x = f.ox;
    ka.y = f.oy;
    ka.keep = keep;
    ka.used = state;
    ka.last = nullptr;
    ka.last_out = state + ntiles;
    ka.changed = changed;
    ka.ntiles = ntiles;
    k_keep_first<<<grid_for(ntiles, BLK / WAVE), BLK, 0, s>>>(ka);
    SC_HIP(hipGetLastError());
    ka.last = state + 2 * ntiles;
    uint32_t *kscan = f.kscan.ensure(size_t(n) + 1);
    uint32_t *rcnt = f.rcnt.ensure(size_t(nr) + 1);
    uint32_t *jring = f.jring.ensure(size_t(J) + 3);
    job_ring.resize(size_t(J) + 3);
    // rounds until one moves nothing (of many vertices some tile nearly always
    // moves in the first); the counts that follow are taken before
    // that is known (one wait instead of two), and again if it was not the last
    for (int it = 1;;) {
        const int end = std::min(it + (it > 1 ? 8 : (n > KEEP_FIRST_TWO ? 2 : 1)), KEEP_ROUNDS);
        const bool rings = it >= end;
        if (rings) {
            k_keep_rings<<<grid_for(nr, BLK / WAVE), BLK, 0, s>>>(ka, nr);
        } else {
            for (; it < end; ++it) {
                const uint32_t *prev = ka.last_out;
                ka.last_out = const_cast<uint32_t *>(ka.last);
                ka.last = prev;
                k_keep_fix<<<grid_for(ntiles, BLK), BLK, 0, s>>>(ka, it);
            }
        }
        SC_HIP(hipGetLastError());
        // compaction counts: vertices, surviving rings, the jobs' first rings
        scan_exclusive_u32(keep, kscan, n + 1, jring + J + 1, s);
        k_ring_counts<<<grid_for(int64_t(nr) + 1), BLK, 0, s>>>(nr, f.off, kscan, rcnt, nonempty, changed + KEEP_ROUNDS);
        SC_HIP(hipGetLastError());
        scan_exclusive_u32(nonempty, nonempty, int64_t(nr) + 1, jring + J + 2, s);
        k_job_rings<<<grid_for(int64_t(J) + 1), BLK, 0, s>>>(J, jr, nonempty, jring, dring);
        SC_HIP(hipGetLastError());
        uint32_t moved = 0, longest = 0;
        ReadBack rb(c);
        rb.add(job_ring.data(), static_cast<const uint32_t *>(jring), size_t(J) + 3);
        if (!rings) rb.add(&moved, static_cast<const uint32_t *>(changed + it - 1), 1);
        rb.add(&longest, static_cast<const uint32_t *>(changed + KEEP_ROUNDS), 1);
        rb.run();
        c.long_rings = longest != 0u; // set by a round that was not the last, it costs launches and no more
        if (!moved) break;
    }
    const uint32_t nout = job_ring[size_t(J) + 1];
    c.nrings = int(job_ring[size_t(J) + 2]);
    job_ring.resize(size_t(J) + 1);
    c.n_out = nout;
    c.d_ring_x.ensure(nout);
    c.d_ring_y.ensure(nout);
    c.d_ring_src.ensure(nout);
    int *off2 = c.d_ring_off.ensure(size_t(c.nrings) + 1);
    k_compact_out<<<grid_for(std::max(n, int64_t(nr) + 1)), BLK, 0, s>>>(n, keep, kscan, f.ox, f.oy, f.osrc,
                                                                        c.d_ring_x, c.d_ring_y, c.d_ring_src, nr,
                                                                        rcnt, nonempty, f.off, off2);
    SC_HIP(hipGetLastError());
    c.wait();
}

} // namespace

void release_foster_scratch() {
    FosterScratch &f = fscratch();
    for (DBuf<uint32_t> *b : {&f.jring, &f.crossP, &f.crossQ, &f.ccP, &f.ccQ, &f.succ, &f.val, &f.ringid,
                              &f.inode, &f.dist, &f.tot, &f.isstart, &f.ringidx, &f.head, &f.linkP, &f.linkQ,
                              &f.jv, &f.jr, &f.keep, &f.kscan, &f.rcnt, &f.nonempty, &f.kctl, &f.ktstate,
                              &f.jmoved})
        b->release();
    f.srec.release();
    f.spstep.release();
    f.semit.release();
    f.sdone.release();
    release_walk_scratch();
    f.jrec.release();
    f.jrec2.release();
    f.jrule.release();
    f.jcov.release();
    f.jend.release();
    f.piece.release();
    for (DBuf<int> *b : {&f.enexP, &f.enexQ, &f.cposP, &f.cposQ, &f.ppos, &f.plen, &f.pdir, &f.pj, &f.jst,
                         &f.osrc, &f.off, &f.rstart, &f.sres, &f.sroff, &f.sosrc, &f.nx, &f.pv, &f.nb,
                         &f.lab, &f.enex, &f.vsrc, &f.cand})
        b->release();
    for (DBuf<double> *b : {&f.ox, &f.oy, &f.vx, &f.vy, &f.sox, &f.soy, &f.qpts, &f.mx, &f.my, &f.nx0, &f.ny0,
                             &f.nx1, &f.ny1, &f.vx1, &f.vy1})
        b->release();
    for (DBuf<int> *b : {&f.qoks, &f.mav, &f.mnbr, &f.mlab, &f.mjob, &f.nslot, &f.ninter, &f.nlab, &f.nnb, &f.nlen,
                         &f.vlen, &f.vslot, &f.seen})
        b->release();
    f.moff.release();
    f.segoff.release();
    f.nodeoff.release();
    f.nflag.release();
    f.nidx.release();
    f.inter.release();
    f.sjobs.release();
}

void label_and_traverse(Ctx &c) {
    JobSet &js = c.jobs;
    SC_REQUIRE(js.J >= 1 && (js.late || int(js.AB.size()) == js.J + 1), SC_ESTATE,
               "segclip_intersections must run first");
    hipStream_t s = c.stream;
    FosterScratch &f = fscratch();
    const int J = js.J;
    const bool sparse = c.sparseP;
    const int *AB = js.d_AB.p, *AC = js.d_AC.p;
    // the base side is either its dense rings (slots) or, in the sparse layout,
    // its intersections (positions); the overlay side is always dense
    const SparseP sp = sparse ? sparse_view(c) : SparseP{};
    const int *PO = sparse ? js.d_p0 : AB; // offsets of the base-side arrays
    // slots of either side, or the most they can be until the offsets are read back
    const bool late = js.late;
    int64_t nP = sparse ? js.p0[J] : (late ? js.cap_b : js.AB[J]), nQ = late ? js.cap_c : js.AC[J];
    const Side P = sparse ? Side{PO, AC, c.sp_x, c.sp_y, c.sp_lab, c.sp_nbr, c.sp_av}
                          : Side{AB, AC, c.aug_bx, c.aug_by, c.lab_b, c.nbr_b, c.av_b};
    const Side Q{AC, AB, c.aug_cx, c.aug_cy, c.lab_c, c.nbr_c, nullptr};
    // per-job words
    int *jw = f.jst.ensure(14 * int64_t(J) + 4);
    {
        FillBatch fb(s);
        fb.add(jw, 14 * int64_t(J) + 4, 0u);
        fb.flush();
    }
    JobState st;
    st.J = J;
    st.uni = c.uni;
    st.AB = PO;
    st.AC = AC;
    st.slow = jw;
    st.firstP = jw + J;
    st.firstQ = jw + 2 * J;
    st.windP = jw + 3 * J;
    st.windQ = jw + 4 * J;
    st.kind = jw + 5 * J;
    st.mP = jw + 6 * J;
    st.mQ = jw + 7 * J;
    st.cP0 = jw + 8 * J;          // J+1
    st.cQ0 = jw + 9 * J + 1;      // J+1
    int *sidx = jw + 10 * J + 2;  // J
    st.vP = jw + 11 * J + 2;
    st.vQ = jw + 12 * J + 2;
    int *bounce = jw + 13 * J + 2;
    uint32_t *crossP = f.crossP.ensure(nP + 1), *crossQ = f.crossQ.ensure(nQ + 1);
    ClassifyArgs cl;
    cl.s[0] = P;
    cl.s[1] = Q;
    cl.J = J;
    cl.pj = sparse ? c.p_j.p : nullptr;
    cl.n[0] = nP;
    cl.n[1] = nQ;
    cl.cross[0] = crossP;
    cl.cross[1] = crossQ;
    cl.slow = st.slow;
    cl.bounce = bounce;
    cl.first[0] = sparse ? nullptr : st.firstP;
    cl.first[1] = st.firstQ;
    int64_t most = std::max(nP, nQ); // slots of the larger side
    int per = cl.per = span_per(most);
    k_jclassify<<<dim3(std::max(grid_for(most + 1, BLK * per), grid_for(int64_t(J) * WAVE)), 4), BLK, 0, s>>>(cl);
    if (sparse) k_sp_first_plain<<<grid_for(int64_t(J) * WAVE), BLK, 0, s>>>(sp, J, st.firstP);
    SC_HIP(hipGetLastError());
    uint32_t *ccP = f.ccP.ensure(nP + 1), *ccQ = f.ccQ.ensure(nQ + 1);
    uint32_t *tot = c.d_u32_total.ensure(2);
    scan_exclusive_u32_2(crossP, ccP, nP + 1, tot, crossQ, ccQ, nQ + 1, tot + 1, s);
    // point-in-polygon of each ring's first plain vertex w.r.t. the other ring
    double *pq = nullptr, *qq = nullptr;
    int *qok = nullptr;
    if (sparse) {
        pq = f.qpts.ensure(4 * size_t(J));
        qq = pq + 2 * size_t(J);
        qok = f.qoks.ensure(size_t(J));
        k_query_pts<<<grid_for(J), BLK, 0, s>>>(J, Q, sp, st.firstP, st.firstQ, pq, qq, qok);
        SC_HIP(hipGetLastError());
    }
    WindSides wd;
    wd.s[0] = WindSide{Q, P, st.firstP, pq, st.windP};
    wd.s[1] = WindSide{P, Q, st.firstQ, nullptr, sparse ? nullptr : st.windQ};
    wd.J = J;
    wd.per = per;
    wd.st = st;
    wd.ccP = ccP;
    wd.ccQ = ccQ;
    wd.sparse = sparse ? 1 : 0;
    wd.sp = sp;
    wd.flags = c.flags;
    k_jwinding<<<dim3(std::max(grid_for(sparse ? nQ : most, BLK * per), grid_for(int64_t(J) + 1)), 3), BLK, 0, s>>>(wd);
    if (sparse) {
        const int chunks = (c.nb + WCH - 1) / WCH;
        k_sp_wind_base<<<unsigned(int64_t(J) * chunks), BLK, 0, s>>>(J, c.nb, c.bpoly, qq, qok, st.windQ);
        if (nP > 0) k_sp_wind_fix<<<grid_for(nP), BLK, 0, s>>>(int(nP), c.p_j, sp, qq, qok, st.windQ);
    }
    SC_HIP(hipGetLastError());
    uint32_t htot[2], hseg[2 * SEG_CTL] = {};
    {
        ReadBack rb(c); // with the post stage's job flags and offsets, when still on the device
        rb.add(htot, static_cast<const uint32_t *>(tot), 2);
        const bool fl = c.flags_pending;
        if (fl) rb.add(js.flags.data(), static_cast<const int *>(c.flags.p), size_t(J));
        if (late) {
            js.AB.resize(size_t(J) + 1);
            js.AC.resize(size_t(J) + 1);
            rb.add(js.AB.data(), AB, size_t(J) + 1);
            rb.add(js.AC.data(), AC, size_t(J) + 1);
            if (c.I > 0) rb.add(hseg, static_cast<const uint32_t *>(c.seg_ctl.p), 2 * SEG_CTL);
        }
        rb.run();
        if (fl) {
            c.flags_pending = false;
            int any = 0;
            for (int v : js.flags) any |= v;
            c.undefined = any;
        }
    }
    if (late) {
        js.late = false;
        if (hseg[2] | hseg[SEG_CTL + 2]) { // a group too large for the ordering: again, with the radix sort
            post_jobs(c, js.k0, js.k0 + J - 1);
            label_and_traverse(c);
            return;
        }
        c.nbaug = js.AB[J];
        c.ncaug = js.AC[J];
        if (!sparse) nP = js.AB[J];
        nQ = js.AC[J];
        most = std::max(nP, nQ);
        per = span_per(most);
    }
    const int mP = int(htot[0]), mQ = int(htot[1]);
    const int M = mP + mQ;
    // entry/exit status, split pairs and pieces of the crossing jobs
    PieceArgs pa;
    if (M > 0) {
        int *cposP = f.cposP.ensure(mP + 1), *cposQ = f.cposQ.ensure(mQ + 1);
        EnexSides en;
        en.s[0] = EnexSide{P, nP, cl.pj, sparse ? sp.slot : nullptr, ccP, st.firstP, st.windP, st.mP, st.vP,
                           f.enexP.ensure(mP + 1), cposP};
        en.s[1] = EnexSide{Q, nQ, nullptr, nullptr, ccQ, st.firstQ, st.windQ, st.mQ, st.vQ, f.enexQ.ensure(mQ + 1),
                           cposQ};
        en.J = J;
        en.per = per;
        en.kind = st.kind;
        en.bounce = bounce;
        en.linkP = f.linkP.ensure(mP + 1);
        en.linkQ = f.linkQ.ensure(mQ + 1);
        en.slow = st.slow;
        k_jenex<<<dim3(grid_for(most, BLK * per), 3), BLK, 0, s>>>(en);
        pa.J = J;
        pa.P = P;
        pa.Q = Q;
        pa.PAB = AB;
        pa.sparse = sparse ? 1 : 0;
        pa.sp = sp;
        pa.cposP = cposP;
        pa.cposQ = cposQ;
        pa.crossP = crossP;
        pa.ccountP = ccP;
        pa.linkP = en.linkP;
        pa.linkQ = en.linkQ;
        pa.enexP = f.enexP;
        pa.enexQ = f.enexQ;
        pa.cP0 = st.cP0;
        pa.cQ0 = st.cQ0;
        pa.kind = st.kind;
        pa.mP = mP;
        pa.mQ = mQ;
        pa.ppos = f.ppos.ensure(M);
        pa.plen = f.plen.ensure(M);
        pa.pdir = f.pdir.ensure(M);
        pa.pj = f.pj.ensure(M);
        pa.succ = f.succ.ensure(M);
        pa.val = f.val.ensure(M);
        pa.slow = st.slow;
        pa.flags = c.flags;
        k_jpieces<<<dim3(grid_for(std::max(mP, mQ)), 2), BLK, 0, s>>>(pa);
        SC_HIP(hipGetLastError());
    }
    // routes and crossing counts on the host
    std::vector<int> hk(3 * size_t(J));
    const int *hkind = hk.data(), *hmP = hk.data() + J, *hmQ = hk.data() + 2 * J;
    js.reason.resize(size_t(J));
    int maxm = 0, maxmP = 0; // crossings of the largest traversed job, and its P crossings
    std::vector<int> seq_jobs;
    bool any_nocross = false;
    auto add_routes = [&](ReadBack &rb) {
        rb.add(hk.data(), static_cast<const int *>(st.kind), 3 * size_t(J));
        rb.add(js.reason.data(), static_cast<const int *>(st.slow), size_t(J));
    };
    auto take_routes = [&] {
        js.route.assign(hkind, hkind + J);
        for (int j = 0; j < J; ++j) {
            if (hkind[j] == K_CROSS && js.reason[j]) js.route[j] = K_SEQ; // found inconsistent later
            if (js.route[j] == K_CROSS) {
                maxm = std::max(maxm, hmP[j] + hmQ[j]);
                maxmP = std::max(maxmP, hmP[j]);
            }
            else if (js.route[j] == K_SEQ) seq_jobs.push_back(j);
            else any_nocross = true;
        }
    };
    // cycles of the crossing jobs: minimum and distance to it by doubling
    uint32_t *dist = nullptr, *inode = nullptr;
    uint32_t *base = f.tot.ensure(int64_t(mP) + 1), *ridx = f.ringidx.ensure(int64_t(mP) + 1);
    const uint32_t *gave_up = nullptr; // set where the crossings' links are no permutation
    // longest: as many P crossings as a cycle may hold
    auto rank_cycles = [&](int longest, bool every) {
        const int rounds = ilog2_exact(longest);
        const JumpArgs ja{mP, M, pa.val, pa.succ, pa.plen, pa.pj, st.kind, st.slow};
        uint2 *ends = f.jend.ensure(mP > 0 ? mP : 1);
        uint32_t *moved = f.jmoved.ensure(size_t(rounds) + 1); // per round, and whether a walk gave up
        // the windows of the n records a, lengthened until they hold whole cycles
        auto doubled = [&](int n, uint4 *a, uint4 *b) {
            for (int r = 0; r < (rounds + 1) / 2; ++r) {
                k_jump_rank<<<grid_for(n), BLK, 0, s>>>(n, a, b, moved, r);
                std::swap(a, b);
            }
            return a;
        };
        if (mP > 0 && mP <= JUMP_SMALL) {
            k_jump_small<<<1, JUMP_BLK, 0, s>>>(ja, rounds, ends);
        } else if (mP > 0) {
            const int G = int(ceil_div(int64_t(mP), int64_t(RULE)));
            uint4 *rec = f.jrec.ensure(mP), *rule = f.jrule.ensure(3 * size_t(G));
            uint2 *cov = f.jcov.ensure(mP);
            {
                FillBatch fb(s);
                fb.add(moved, rounds + 1, 0u);
                fb.flush();
            }
            k_jump_init<<<grid_for(mP), BLK, 0, s>>>(ja, rec, cov);
            if (every) {
                const uint4 *whole = doubled(mP, rec, f.jrec2.ensure(mP));
                k_jump_out<<<grid_for(mP), BLK, 0, s>>>(mP, whole, ends);
            } else {
                k_ruler_walk<<<grid_for(G), BLK, 0, s>>>(mP, G, rec, cov, rule, moved + rounds);
                const uint4 *whole = rule + G;
                if (G <= JUMP_SMALL) k_rule_small<<<1, JUMP_BLK, 0, s>>>(rule + G, G, rounds);
                else whole = doubled(G, rule + G, rule + 2 * size_t(G));
                k_ruler_final<<<grid_for(mP), BLK, 0, s>>>(mP, rec, cov, rule, whole, ends, moved + rounds);
                gave_up = moved + rounds;
            }
        }
        inode = f.inode.ensure(M);
        dist = f.dist.ensure(M);
        uint32_t *isstart = f.isstart.ensure(int64_t(mP) + 1);
        k_rank_final<<<grid_for(M), BLK, 0, s>>>(M, mP, ends, pa.succ, pa.plen, inode, dist, base, isstart);
        SC_HIP(hipGetLastError());
        scan_exclusive_u32_2(base, base, int64_t(mP) + 1, nullptr, isstart, ridx, int64_t(mP) + 1, nullptr, s);
    };
    // per-job output sizes before clean-up, and their offsets
    uint32_t *jv = f.jv.ensure(J + 1), *jr = f.jr.ensure(J + 1);
    CountArgs ca;
    ca.J = J;
    ca.AB = AB;
    ca.AC = AC;
    ca.kind = st.kind;
    ca.slow = st.slow;
    ca.windP = st.windP;
    ca.windQ = st.windQ;
    ca.cP0 = st.cP0;
    ca.sidx = sidx;
    ca.seq_res = nullptr;
    ca.base = base;
    ca.ridx = ridx;
    ca.jv = jv;
    ca.jr = jr;
    auto totals = [&](bool routes) {
        k_jcounts<<<grid_for(int64_t(J) + 1), BLK, 0, s>>>(ca);
        SC_HIP(hipGetLastError());
        scan_exclusive_u32_2(jv, jv, int64_t(J) + 1, tot, jr, jr, int64_t(J) + 1, tot + 1, s);
        uint32_t over = 0;
        ReadBack rb(c);
        rb.add(htot, static_cast<const uint32_t *>(tot), 2);
        if (gave_up) rb.add(&over, gave_up, 1);
        if (routes) add_routes(rb);
        rb.run();
        return over == 0u;
    };
    // Few crossings: their cycles are ranked before the routes are known, and
    // one read-back brings the routes and the totals (which stand where no job
    // is sequential).  Many: the routes come first, so that the sequential jobs
    // run beside the ranking.
    const bool few = mP <= RULE * JUMP_SMALL; // no launch per round
    bool counted = false;
    if (few) {
        if (mP > 0) rank_cycles(mP, false);
        if (!totals(true)) {
            gave_up = nullptr;
            rank_cycles(mP, true);
            totals(true);
        }
        take_routes();
        counted = seq_jobs.empty();
    } else {
        ReadBack rb(c);
        add_routes(rb);
        rb.run();
        take_routes();
    }
    // sequential route
    const int nseq = int(seq_jobs.size());
    std::vector<SeqJob> sj(static_cast<size_t>(nseq));
    WalkIn wi;
    int *done = nullptr; // per sequential job: run by walk_jobs
    bool walked = false;
    if (nseq > 0) {
        std::vector<int> hsidx(static_cast<size_t>(J), -1);
        int64_t mb = 0;
        std::vector<int64_t> moff(static_cast<size_t>(nseq)), segoff(2 * size_t(nseq) + 1, 0);
        for (int q = 0; q < nseq; ++q) {
            const int j = seq_jobs[q];
            SeqJob &b = sj[q];
            b.j = j;
            b.nP = js.AB[j + 1] - js.AB[j];
            b.nQ = js.AC[j + 1] - js.AC[j];
            // sparse layout: the base ring is materialised densely for this job
            moff[q] = mb;
            b.P0 = sparse ? int(mb) : js.AB[j];
            mb += b.nP;
            b.Q0 = js.AC[j];
            segoff[2 * q + 1] = segoff[2 * q] + b.nP;
            segoff[2 * q + 2] = segoff[2 * q + 1] + b.nQ;
            hsidx[j] = q;
        }
        SeqJob *djobs = f.sjobs.ensure(nseq);
        c.upload(djobs, sj.data(), sizeof(SeqJob) * nseq);
        c.upload(sidx, hsidx.data(), sizeof(int) * J);
        SeqBatch b;
        b.jobs = djobs;
        b.done = nullptr;
        b.uni = c.uni;
        b.par = c.seq_par;
        b.px = c.aug_bx; b.py = c.aug_by; b.qx = c.aug_cx; b.qy = c.aug_cy;
        const int *avP = c.av_b, *labP = c.lab_b, *nbrP = c.nbr_b;
        if (sparse) {
            double *mx = f.mx.ensure(mb), *my = f.my.ensure(mb);
            int *mav = f.mav.ensure(mb), *mnbr = f.mnbr.ensure(mb), *mlab = f.mlab.ensure(mb);
            int *djob = f.mjob.ensure(nseq);
            int64_t *dmoff = f.moff.ensure(nseq);
            c.upload(djob, seq_jobs.data(), sizeof(int) * nseq);
            c.upload(dmoff, moff.data(), sizeof(int64_t) * nseq);
            for (int q0 = 0; q0 < nseq; q0 += 65535) {
                dim3 g(64, unsigned(std::min(65535, nseq - q0)));
                k_sp_materialize<<<g, BLK, 0, s>>>(q0, nseq, djob, dmoff, sp, c.sp_av, c.sp_nbr, c.sp_lab, mx, my,
                                                   mav, mnbr, mlab);
                SC_HIP(hipGetLastError());
            }
            b.px = mx; b.py = my;
            avP = mav; labP = mlab; nbrP = mnbr;
        }
        // ring nodes
        const int nseg = 2 * nseq;
        const int64_t S = segoff[nseg];
        int64_t *dseg = f.segoff.ensure(nseg + 1);
        c.upload(dseg, segoff.data(), sizeof(int64_t) * (nseg + 1));
        NodeArgs na;
        na.nseg = nseg;
        na.segoff = dseg;
        na.jobs = djobs;
        na.px = b.px; na.py = b.py; na.qx = b.qx; na.qy = b.qy;
        na.avP = avP; na.labP = labP; na.nbrP = nbrP; na.labQ = c.lab_c; na.nbrQ = c.nbr_c;
        uint32_t *flag = f.nflag.ensure(S + 1), *nidx = f.nidx.ensure(S + 1);
        k_node_flags<<<grid_for(S), BLK, 0, s>>>(na, S, flag);
        SC_HIP(hipGetLastError());
        SC_HIP(hipMemsetAsync(flag + S, 0, sizeof(uint32_t), s));
        scan_exclusive_u32(flag, nidx, S + 1, nullptr, s);
        // node offsets of the segments, gathered on the device and read back at once
        std::vector<int64_t> nodeoff(size_t(nseg) + 1);
        int64_t *dnodeoff = f.nodeoff.ensure(nseg + 1);
        k_seg_node_offsets<<<grid_for(int64_t(nseg) + 1), BLK, 0, s>>>(nseg, dseg, nidx, dnodeoff);
        SC_HIP(hipGetLastError());
        {
            ReadBack rb(c);
            rb.add(nodeoff.data(), static_cast<const int64_t *>(dnodeoff), size_t(nseg) + 1);
            rb.run();
        }
        const int64_t N = nodeoff[nseg];
        int *nslot = f.nslot.ensure(N), *ninter = f.ninter.ensure(N), *nlab = f.nlab.ensure(N);
        int *nnb = f.nnb.ensure(N), *nlen = f.nlen.ensure(N);
        double *nx0 = f.nx0.ensure(N), *ny0 = f.ny0.ensure(N), *nx1 = f.nx1.ensure(N), *ny1 = f.ny1.ensure(N);
        k_node_fill<<<grid_for(S), BLK, 0, s>>>(na, S, flag, nidx, nslot, ninter, nx0, ny0, nlab, nnb);
        k_node_finish<<<grid_for(N), BLK, 0, s>>>(na, N, dnodeoff, flag, nidx, nslot, ninter, nlen, nx1, ny1, nnb);
        SC_HIP(hipGetLastError());
        // scratch per job, sized by its nodes
        int64_t vb = 0, ob = 0, rb = 0;
        wi.nwalk = 0;
        for (int q = 0; q < nseq; ++q) {
            SeqJob &j = sj[q];
            j.node0 = int(nodeoff[2 * q]);
            j.nPn = int(nodeoff[2 * q + 1] - nodeoff[2 * q]);
            j.nQn = int(nodeoff[2 * q + 2] - nodeoff[2 * q + 1]);
            j.cap = 2 * (j.nPn + j.nQn) + 64;
            j.out_cap = 2 * (j.nP + j.nQ) + 64;
            j.ring_cap = j.nP + j.nQ + 8;
            j.walk = j.nPn + j.nQn >= WALK_MIN_NODES ? wi.nwalk++ : -1;
            j.vbase = vb;
            j.obase = ob;
            j.rbase = rb;
            vb += j.cap;
            ob += j.out_cap;
            rb += j.ring_cap + 1;
        }
        c.upload(djobs, sj.data(), sizeof(SeqJob) * nseq);
        b.nx0 = nx0; b.ny0 = ny0; b.nx1 = nx1; b.ny1 = ny1;
        b.nlen = nlen; b.nslot = nslot; b.ninter = ninter; b.nlab = nlab; b.nnb = nnb;
        b.windP = st.windP;
        b.windQ = st.windQ;
        b.vx = f.vx.ensure(vb); b.vy = f.vy.ensure(vb); b.vx1 = f.vx1.ensure(vb); b.vy1 = f.vy1.ensure(vb);
        b.vlen = f.vlen.ensure(vb); b.vslot = f.vslot.ensure(vb);
        b.nx = f.nx.ensure(vb); b.pv = f.pv.ensure(vb); b.nb = f.nb.ensure(vb); b.lab = f.lab.ensure(vb);
        b.enex = f.enex.ensure(vb); b.vsrc = f.vsrc.ensure(vb); b.cand = f.cand.ensure(vb);
        b.seen = f.seen.ensure(2 * vb);
        b.inter = f.inter.ensure(vb);
        b.rec = f.srec.ensure(vb);
        b.pstep = f.spstep.ensure(vb);
        b.emit = f.semit.ensure(2 * vb);
        b.ox = f.sox.ensure(ob); b.oy = f.soy.ensure(ob); b.osrc = f.sosrc.ensure(ob);
        b.ring_off = f.sroff.ensure(rb);
        b.result = f.sres.ensure(3 * int64_t(nseq));
        // the jobs' working rings and zeroed walk state, spread over the device
        {
            FillBatch fb(s);
            fb.add(b.seen, 2 * vb, 0u);
            fb.flush();
        }
        k_seq_init<<<grid_for(N), BLK, 0, s>>>(b, dnodeoff, nseq, N);
        SC_HIP(hipGetLastError());
        // the sequential jobs run beside the crossing jobs' labelling
        c.ensure_side_stream();
        SC_HIP(hipEventRecord(c.ev_fork, s));
        SC_HIP(hipStreamWaitEvent(c.stream2, c.ev_fork, 0));
        if (c.seq_par) {
            wi.b = b;
            wi.jobs = &sj;
            wi.nodeoff = dnodeoff;
            wi.segoff = dseg;
            wi.nidx = nidx;
            wi.N = N;
            wi.firstP = st.firstP;
            wi.firstQ = st.firstQ;
            done = f.sdone.ensure(nseq);
            {
                FillBatch fb(c.stream2);
                fb.add(done, nseq, 0u);
                fb.flush();
            }
            walked = walk_jobs(wi, done, c.stream2);
            if (walked) { // the others from their initial state
                b.done = done;
                k_seq_init<<<grid_for(N), BLK, 0, c.stream2>>>(b, dnodeoff, nseq, N);
                SC_HIP(hipGetLastError());
            }
        }
        k_sequential<<<nseq, SEQ_BLK, 0, c.stream2>>>(b);
        SC_HIP(hipGetLastError());
        SC_HIP(hipEventRecord(c.ev_join, c.stream2));
    }
    if (!few && maxm > 0) rank_cycles(maxmP, false);
    if (!counted) {
        if (nseq > 0) {
            ca.seq_res = f.sres;
            SC_HIP(hipStreamWaitEvent(s, c.ev_join, 0));
        }
        if (!totals(false)) {
            gave_up = nullptr;
            rank_cycles(maxmP, true);
            totals(false);
        }
    }
    const int64_t NV = htot[0];
    const int NR = int(htot[1]);
    f.ox.ensure(NV + 1);
    f.oy.ensure(NV + 1);
    f.osrc.ensure(NV + 1);
    int *off = f.off.ensure(int64_t(NR) + 1);
    // the rings' first vertices and the pieces' by position, each the maximum up
    // to it after one scan of both; ring offsets come from every route first
    uint32_t *head = f.head.ensure(NV + 1);
    uint32_t *ringid = f.ringid.ensure(size_t(NV) + 1);
    const bool cross = maxm > 0 && NV > 0;
    {
        FillBatch fb(s);
        fb.add(off + NR, 1, uint32_t(int(NV)));
        fb.add(head, cross ? NV : 0, 0u);
        fb.add(ringid, NV, 0u);
        fb.add(f.keep.ensure(size_t(NV) + 1) + NV, 1, 0u); // closing entry of the clean-up's scan
        fb.add(f.kctl.ensure(KEEP_ROUNDS + 1), KEEP_ROUNDS + 1, 0u); // and the long-ring word
        fb.flush();
    }
    int4 *piece = f.piece.ensure(M > 0 ? M : 1);
    if (cross) {
        HeadArgs ha;
        ha.M = M;
        ha.mP = mP;
        ha.inode = inode;
        ha.dist = dist;
        ha.base = base;
        ha.ridx = ridx;
        ha.pj = pa.pj;
        ha.cP0 = st.cP0;
        ha.ppos = pa.ppos;
        ha.plen = pa.plen;
        ha.pdir = pa.pdir;
        ha.JV = jv;
        ha.JR = jr;
        ha.head = head;
        ha.piece = piece;
        ha.off = off;
        k_jheads<<<grid_for(M), BLK, 0, s>>>(ha);
    }
    SC_HIP(hipGetLastError());
    if (any_nocross) {
        if (sparse)
            k_sp_nocross_p<<<grid_for(NV), BLK, 0, s>>>(NV, J, jv, st.kind, st.windP, sp, f.ox, f.oy, f.osrc);
        else
            k_jcopy_nocross<<<grid_for(nP), BLK, 0, s>>>(P, true, J, nP, st.kind, st.windP, st.windQ, AB, jv, f.ox,
                                                         f.oy, f.osrc);
        k_jcopy_nocross<<<grid_for(nQ), BLK, 0, s>>>(Q, false, J, nQ, st.kind, st.windP, st.windQ, AB, jv, f.ox,
                                                     f.oy, f.osrc);
        k_jnocross_off<<<grid_for(J), BLK, 0, s>>>(J, st.kind, st.windP, st.windQ, AB, jv, jr, off);
        SC_HIP(hipGetLastError());
    }
    std::vector<int> hres(3 * size_t(nseq));
    if (nseq > 0) {
        if (walked) walk_emit(wi, done, jv, jr, f.ox, f.oy, f.osrc, off, s);
        k_jseq_copy<<<nseq, BLK, 0, s>>>(f.sjobs, walked ? done : nullptr, f.sres, jv, jr, f.sox, f.soy, f.sosrc, f.sroff, f.ox, f.oy,
                                          f.osrc, off);
        SC_HIP(hipGetLastError());
    }
    if (NR > 0 && NV > 0) {
        k_ring_heads<<<grid_for(NR), BLK, 0, s>>>(NR, off, ringid);
        SC_HIP(hipGetLastError());
        scan_inclusive_last_u32_2(ringid, ringid, NV, head, head, cross ? NV : 0, s);
    }
    if (cross) {
        EmitArgs ea;
        ea.J = J;
        ea.mP = mP;
        ea.PAB = AB;
        ea.sparse = sparse ? 1 : 0;
        ea.sp = sp;
        ea.cP0 = st.cP0;
        ea.cposP = pa.cposP;
        ea.flags = c.flags;
        ea.head = head;
        ea.piece = piece;
        ea.P = P;
        ea.Q = Q;
        ea.ox = f.ox;
        ea.oy = f.oy;
        ea.osrc = f.osrc;
        k_jemit<<<grid_for(NV), BLK, 0, s>>>(ea, NV);
        SC_HIP(hipGetLastError());
    }
    if (nseq > 0) {
        ReadBack rb(c);
        rb.add(hres.data(), static_cast<const int *>(f.sres.p), 3 * size_t(nseq));
        rb.run();
    }
    for (int q = 0; q < nseq; ++q) {
        js.flags[sj[q].j] |= hres[3 * q + 2];
        c.undefined |= hres[3 * q + 2];
    }
    std::vector<uint32_t> job_ring;
    cleanup_rings(c, f, NR, NV, J, jr, job_ring);
    js.ring_off.resize(size_t(J) + 1);
    for (int j = 0; j <= J; ++j) js.ring_off[j] = int(job_ring[j]);
}

void clip_jobs(Ctx &c, int k0, int k1) {
    SC_REQUIRE(k0 >= 1 && k1 <= c.K && k0 <= k1, SC_EINVAL, "overlay index out of range");
    StageTimes t;
    // independent small pairs: one launch (sc_small.hip); a batch
    // it does not cover runs on the staged path below
    if (small_batch_eligible(c, k0, k1)) {
        for (int i = 0; i <= 6; ++i) c.mark(i);
        if (clip_small_batch(c, k0, k1)) {
            c.mark(7);
            if (c.timing) {
                SC_HIP(hipEventSynchronize(c.ev[7]));
                t.label = c.elapsed(6, 7);
                c.times = t;
            }
            return;
        }
    }
    // candidate pairs, where no call has found them yet: from the box join, or,
    // where it refuses the rings, from the tree (built here unless all of it is there)
    const bool cand = int(c.pair_off.size()) != c.K + 1;
    c.mark(10);
    const bool joined = cand && join_candidates(c);
    const bool tree = cand && !joined && c.built != TREE_ALL;
    c.mark(0);
    if (tree) {
        build_edges(c);
        build_elementary(c);
    }
    c.mark(1);
    if (tree) build_node_intervals(c);
    c.mark(2);
    if (tree) build_leaf_end_entries(c);
    c.mark(3);
    if (tree) build_cover_lists(c);
    c.mark(4);
    if (cand && !joined) find_candidates(c);
    c.moved = false;
    c.mark(5);
    post_jobs(c, k0, k1, true);
    c.mark(6);
    label_and_traverse(c);
    c.mark(7);
    if (c.timing) {
        SC_HIP(hipEventSynchronize(c.ev[7]));
        t.elementary = c.elapsed(0, 1);
        t.tree = c.elapsed(1, 2);
        t.endlist = c.elapsed(2, 3);
        t.cover = c.elapsed(3, 4);
        t.candidates = c.elapsed(joined ? 10 : 4, 5);
        t.stab_kernel = cand ? c.elapsed(8, 9) : 0.0f;
        t.post = c.elapsed(5, 6);
        t.label = c.elapsed(6, 7);
        c.times = t;
    }
}

void clip_all(Ctx &c, int k) { clip_jobs(c, k, k); }

} // namespace sc
