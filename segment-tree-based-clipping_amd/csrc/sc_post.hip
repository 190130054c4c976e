// sc_post.hip -- intersection bookkeeping (rows A11-A15) for a batch of jobs.
//
// A job clips one base ring against one overlay ring (overlay k, base
// job_base(k)); all jobs of a batch run in the same launches, their arrays
// laid out job after job.
//
// Reference (src/clip.cpp / oacc_segment_tree.cpp):
//  - countEdgeIntersections + isNonDegenerateCase + exclusive scans
//    (clip:508-601, 1858-1861): per edge all / non-degenerate counts; a pair
//    is non-degenerate for the base edge if type in {1,3,5,7}, for the
//    overlay edge if type in {1,2,6}
//  - saveIntersectionsParallel (oacc:7257-7341): intersection point by type,
//    alpha/beta quantised with alphaToInt
//  - sortIntersectionsAtEdgesParallel (oacc:7436-7473): per edge, stable sort
//    by the quantised alpha (nine decimal digits, i.e. modulo 1e9)
//  - copyIntersectionsParallel (oacc:7508-7664): augmented rings, source
//    vertex i at i + (non-degenerate intersections before it); a leading
//    degenerate intersection marks the source vertex, the non-degenerate ones
//    follow it in alpha order; neighbour links are 1-based cross indices
//  - calculateInitLabelParallel (oacc:7925-7988): initial Foster labels
// Order: pairs come in (base edge, overlay edge) order and every edge's
// intersections are sorted by quantised alpha (ties keep that order).  On
// inputs where the reference is well defined this gives its result; the
// cases where it is not (an intersection never given a slot) are reported
// through the undefined-behaviour flags instead of being guessed.
#include "sc_ctx.hpp"
#include "sc_seg.hpp"
#include "sc_fp64.hpp"

namespace sc {

namespace {

constexpr int BLK = 256;
inline unsigned grid_for(int64_t n, int per = BLK) {
    int64_t g = ceil_div(n, per);
    if (g < 1) g = 1;
    return unsigned(g);
}

enum : int { UB_UNASSIGNED = 1, UB_ALPHA_RANGE = 16 };

struct JobArgs {
    int J;
    const int *p0;     // J+1 pair offsets (relative to the batch's first pair)
    const int *bvoff;  // base ring vertex offset in bpoly
    const int *beoff;  // base ring first global edge
    const int *nb, *nc;
    const int *cvoff;  // overlay vertex offset in cpoly
    const int *JB, *JC; // J+1 offsets of the per-edge count arrays (n+1 per job)
};

__global__ void k_pair_decode(JobArgs ja, const uint64_t *__restrict__ pairs, int I, int bits_b, int bits_c,
                              const double *__restrict__ bpoly, const double *__restrict__ cpoly, int *pj, int *pb,
                              int *pc, int *pt, double *px, double *py, int *qa, int *qb, int *all_b, int *dg_b,
                              int *all_c, int *dg_c, int *flags, int *arr_b, int *arr_c, uint32_t *starts,
                              uint64_t *KB) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    const int lane = threadIdx.x & (WAVE - 1);
    bool counted = false; // a pair inside its job's rings
    int gb = -1, t = 0;
    if (p < I) {
        const int j = seg_of_wave(ja.p0, ja.J, p);
        const uint64_t key = pairs[p];
        const int b = int((key >> bits_c) & ((1ull << bits_b) - 1ull)) - ja.beoff[j];
        const int cl = int(key & ((1ull << bits_c) - 1ull));
        pj[p] = j;
        // sparse base side: pairs of one base edge are one run, which starts here or not
        if (starts)
            starts[p] = (p == ja.p0[j] || (((pairs[p - 1] ^ key) >> bits_c) & ((1ull << bits_b) - 1ull)) != 0) ? 1u : 0u;
        if (b < 0 || b >= ja.nb[j] || cl >= ja.nc[j]) { // a pair outside the job's rings
            atomicOr(&flags[j], UB_UNASSIGNED);
            arr_c[p] = -1;
            if (arr_b) arr_b[p] = -1;
            pb[p] = 0;
            pc[p] = 0;
            pt[p] = 0;
            px[p] = 0.0;
            py[p] = 0.0;
            qa[p] = 0;
            qb[p] = 0;
            if (KB) KB[p] = uint32_t(p);
        } else {
            const int64_t bId = 2 * int64_t(ja.bvoff[j] + b), cId = 2 * int64_t(ja.cvoff[j] + cl);
            const double b1x = bpoly[bId], b1y = bpoly[bId + 1], b2x = bpoly[bId + 2], b2y = bpoly[bId + 3];
            const double c1x = cpoly[cId], c1y = cpoly[cId + 1], c2x = cpoly[cId + 2], c2y = cpoly[cId + 3];
            double al, be;
            t = classify(b1x, b1y, b2x, b2y, c1x, c1y, c2x, c2y, al, be);
            double x, y;
            intersection_point(t, al, b1x, b1y, b2x, b2y, c1x, c1y, x, y);
            pb[p] = b;
            pc[p] = cl;
            pt[p] = t;
            px[p] = x;
            py[p] = y;
            const int ia = alpha_to_int(al);
            qa[p] = ia;
            qb[p] = alpha_to_int(be);
            if (KB) KB[p] = (uint64_t(uint32_t(ia % 1000000000)) << 32) | uint32_t(p);
            if (!alpha_in_range(al) || !alpha_in_range(be)) atomicOr(&flags[j], UB_ALPHA_RANGE);
            arr_c[p] = atomicAdd(&all_c[ja.JC[j] + cl], 1); // arrival inside the overlay edge's group
            if (!nondeg_c(t)) atomicAdd(&dg_c[ja.JC[j] + cl], 1);
            gb = ja.JB[j] + b;
            counted = true;
        }
    }
    if (!all_b) return; // uniform
    // pairs are sorted by (job, base edge): each run of one base edge inside
    // the wave adds its counts with one atomic per counter
    const int prev = __shfl_up(gb, 1, WAVE);
    const bool head = counted && (lane == 0 || prev != gb);
    const uint64_t hm = __ballot(head), cm = __ballot(counted), dgm = __ballot(counted && !nondeg_b(t));
    int base = 0;
    if (head) {
        const uint64_t above = lane == WAVE - 1 ? 0ull : hm & (~0ull << (lane + 1));
        const int nxt = above ? __ffsll((unsigned long long)above) - 1 : WAVE;
        const uint64_t run = (nxt == WAVE ? ~0ull : ((1ull << nxt) - 1ull)) & (~0ull << lane) & cm;
        base = atomicAdd(&all_b[gb], __popcll(run));
        const int n_dg = __popcll(run & dgm);
        if (n_dg) atomicAdd(&dg_b[gb], n_dg);
    }
    // arrival inside the base edge's group: the run's base plus the counted lanes before this one
    const uint64_t upto = lane == WAVE - 1 ? ~0ull : ((2ull << lane) - 1ull);
    const int h = (hm & upto) ? 63 - __clzll(hm & upto) : 0; // this lane's run head
    const int hb = __shfl(base, h, WAVE);
    if (counted) arr_b[p] = hb + __popcll(cm & ((1ull << lane) - 1ull) & ~((1ull << h) - 1ull));
}

// Per-edge alpha order without a global sort.  Every counted pair has an
// arrival index inside its edge's group (taken from the counting atomics), so
// the groups are filled at their exclusive count offsets; inside a group the
// pairs are then ranked by (quantised alpha, pair index), keys that are all
// distinct.  The result equals a stable sort of the pairs (in pair order) by
// (edge slot, quantised alpha): ties keep pair order.
struct ScatterSide {
    const int *edge_of, *JX, *scan, *arr, *q;
    uint64_t *K;
};
struct ScatterSides {
    ScatterSide s[2];
};
__global__ void k_seg_scatter(int I, const int *__restrict__ pj, ScatterSides sides) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= I) return;
    const ScatterSide &z = sides.s[blockIdx.y];
    const int a = z.arr[p];
    if (a < 0) return; // not counted (flagged job)
    const int pos = z.scan[z.JX[pj[p]] + z.edge_of[p]] + a;
    z.K[pos] = (uint64_t(uint32_t(z.q[p] % 1000000000)) << 32) | uint32_t(p);
}

// The sparse base side has far more edges than pairs (one ring per job), but
// its pairs are already in (job, base edge) order: the runs of one edge are
// its groups.  start[r] of run r; start was filled with I, so runs past the
// last one are empty.
__global__ void k_run_starts(int I, const uint32_t *__restrict__ head, const uint32_t *__restrict__ run, int *start) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < I && head[p]) start[run[p]] = p;
}

// keys for the per-edge alpha order: the edge's slot over the batch above
// the quantised alpha modulo 1e9 (the nine decimal digits the reference's
// LSD sort looks at, sortIntersectionsAtEdgesParallel oacc:7436-7473) in the
// low 30 bits; values are pair indices
__global__ void k_edge_alpha_keys(const int *__restrict__ edge_of, const int *__restrict__ pj,
                                  const int *__restrict__ off, const int *__restrict__ q, int I, uint64_t *keys,
                                  uint32_t *vals) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= I) return;
    keys[i] = (uint64_t(uint32_t(off[pj[i]] + edge_of[i])) << 30) | uint64_t(uint32_t(q[i] % 1000000000));
    vals[i] = uint32_t(i);
}

__global__ void k_copy_order(const uint32_t *__restrict__ vals, int I, int *ord) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < I) ord[i] = int(vals[i]);
}

// Augmented ring offsets per job: sizes nb + (non-degenerate intersections on
// the base; ndg: their counts by pair position in the sparse layout), likewise
// overlay, scanned by one block (J + 1 entries each), JOB_PER jobs per thread:
// one launch where sizes, closing entries and their scans took five.  More jobs
// than one chunk are gathered by as many blocks and scanned in two launches
// (16,384 jobs: 81 us in four chunks of one block, 14 so).
// Pairs up to which launches and read-backs are saved at the price of more loads:
// a clip with 22,000 pairs takes 368 us instead of 406, with 56,000 448 instead of
// 496.  Beyond the line it would gain less and less (106,000: 478 for 523, 473,000:
// 609 for 630), for buffers with a spare slot per pair; with tens of millions of
// slots the links by slot are the faster ones.
constexpr int LATE_MAX = 1 << 16;
constexpr int JOB_BLK = 1024, JOB_PER = 4;
// Scanned counts of the edges' non-degenerate pairs: of all pairs less the
// degenerate ones.  Those are few as a rule, so that a pair takes one counting
// atomic for its overlay edge and not two: the stage of 4,096 overlays with 20
// million pairs 5.08 -> 4.93 ms, of 200,000 x 1,000,000 vertices 0.306 -> 0.298.
struct NdScan {
    const int *all, *dg;
    __device__ int operator[](int64_t i) const { return all[i] - dg[i]; }
};
__global__ void k_job_sizes(JobArgs ja, NdScan nd_b, const uint32_t *__restrict__ ndg, NdScan nd_c, int *nba,
                            int *nca) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j > ja.J) return;
    int b = 0, c = 0;
    if (j < ja.J) {
        b = ja.nb[j] + (nd_b.all ? nd_b[ja.JB[j + 1]] - nd_b[ja.JB[j]] : int(ndg[ja.p0[j + 1]] - ndg[ja.p0[j]]));
        c = ja.nc[j] + (nd_c[ja.JC[j + 1]] - nd_c[ja.JC[j]]);
    }
    nba[j] = b;
    nca[j] = c;
}
__global__ __launch_bounds__(JOB_BLK) void k_job_offsets(JobArgs ja, NdScan nd_b, const uint32_t *__restrict__ ndg,
                                                       NdScan nd_c, int *nba, int *nca) {
    __shared__ int sb[JOB_BLK / WAVE], sc[JOB_BLK / WAVE];
    const int lane = threadIdx.x & (WAVE - 1), wid = threadIdx.x / WAVE;
    const int j0 = int(threadIdx.x) * JOB_PER;
    int vb[JOB_PER], vc[JOB_PER], tb = 0, tc = 0;
#pragma unroll
    for (int q = 0; q < JOB_PER; ++q) {
        const int j = j0 + q;
        vb[q] = vc[q] = 0;
        if (j < ja.J) {
            vb[q] = ja.nb[j] + (nd_b.all ? nd_b[ja.JB[j + 1]] - nd_b[ja.JB[j]] : int(ndg[ja.p0[j + 1]] - ndg[ja.p0[j]]));
            vc[q] = ja.nc[j] + (nd_c[ja.JC[j + 1]] - nd_c[ja.JC[j]]);
        }
        tb += vb[q];
        tc += vc[q];
    }
    int ib = tb, ic = tc;
    for (int d = 1; d < WAVE; d <<= 1) {
        const int ob = __shfl_up(ib, d, WAVE), oc = __shfl_up(ic, d, WAVE);
        if (lane >= d) {
            ib += ob;
            ic += oc;
        }
    }
    if (lane == WAVE - 1) {
        sb[wid] = ib;
        sc[wid] = ic;
    }
    __syncthreads();
    int bb = ib - tb, bc = ic - tc; // before this thread's jobs
    for (int w = 0; w < wid; ++w) {
        bb += sb[w];
        bc += sc[w];
    }
#pragma unroll
    for (int q = 0; q < JOB_PER; ++q) {
        if (j0 + q <= ja.J) {
            nba[j0 + q] = bb;
            nca[j0 + q] = bc;
        }
        bb += vb[q];
        bc += vc[q];
    }
}

// the two sides of the augmented rings, one per blockIdx.y (a null ax: not in this batch)
struct AugSide {
    const int *JX, *nverts, *voff, *AX;
    const double *poly;
    const int *all_scan;
    NdScan nd_scan;
    const int *edge_of, *ord, *q;
    double *ax, *ay;
    int *av, *nbr, *lab, *from, *slot;
};
struct AugSides {
    AugSide s[2];
};

// Source vertices: count slot i of job j is vertex i - JX[j] (the last slot of
// a job is padding).  Every slot of the augmented rings is written once, in
// full: a source's here, an inserted intersection's by aug_segment (an edge
// has a slot per non-degenerate intersection, and no fewer positions to fill
// them from), so nothing is cleared first.  Bound by the stores, 32 bytes a slot.
template <bool ONE>
__device__ inline void aug_source(int J, const AugSide &z, bool side_b, const int *__restrict__ pt, int64_t i) {
    if (!z.ax || i >= z.JX[J]) return;
    const int j = seg_of_wave(z.JX, J, i);
    const int j0 = z.JX[j], v = int(i - j0);
    if (v >= z.nverts[j]) return;
    const int64_t pos = z.AX[j] + v + (z.nd_scan[i] - z.nd_scan[j0]);
    const double2 V = reinterpret_cast<const double2 *>(z.poly)[int64_t(z.voff[j]) + v];
    z.ax[pos] = V.x;
    z.ay[pos] = V.y;
    int av = -100; // or the parameter of the degenerate intersection that leads its edge's order
    if (ONE) {
        const int s = z.all_scan[i];
        if (z.all_scan[i + 1] > s) {
            const int p = z.ord[s];
            if (side_b ? degen_b_first(pt[p]) : degen_c_first(pt[p])) av = z.q[p];
        }
    }
    z.av[pos] = av;
    z.nbr[pos] = -100;
    z.lab[pos] = 0;
    if (z.from) z.from[pos] = v;
}

// one thread per position of the per-edge alpha order: a leading degenerate
// intersection takes its edge's source slot, the non-degenerate ones fill
// the slots after it in order
template <bool ONE>
__device__ inline void aug_segment(const int *__restrict__ pj, int I, const int *__restrict__ pt,
                                   const double *__restrict__ px, const double *__restrict__ py, int *flags,
                                   const AugSide &z, bool side_b, int i) {
    if (!z.ax || i >= I) return;
    const int p = z.ord[i];
    const int j = pj[p];
    const int e = z.edge_of[p];
    const int gi = z.JX[j] + e;
    const int s = z.all_scan[gi], t = z.all_scan[gi + 1];
    const int nd = z.nd_scan[gi + 1] - z.nd_scan[gi];
    const int src = z.AX[j] + e + (z.nd_scan[gi] - z.nd_scan[z.JX[j]]);
    const int first = i == s ? p : z.ord[s];
    const int k0 = (side_b ? degen_b_first(pt[first]) : degen_c_first(pt[first])) ? 1 : 0;
    if (i == s && k0 + nd != t - s) atomicOr(&flags[j], UB_UNASSIGNED);
    if (i == s && k0) {
        if (!ONE) z.av[src] = z.q[p];
        z.slot[p] = src;
        return;
    }
    const int k = i - s - k0;
    if (k >= nd) return; // more positions than non-degenerate slots: flagged above
    if (!(side_b ? nondeg_b(pt[p]) : nondeg_c(pt[p]))) atomicOr(&flags[j], UB_UNASSIGNED);
    const int sl = src + 1 + k;
    z.ax[sl] = px[p];
    z.ay[sl] = py[p];
    z.av[sl] = z.q[p];
    z.nbr[sl] = -100;
    z.lab[sl] = 0;
    z.slot[p] = sl;
    if (z.from) z.from[sl] = ~p;
}
// words of the ordering that say that a group was too large for it
__device__ inline bool unordered_words(const uint32_t *over) { return over && (over[2] | over[SEG_CTL + 2]) != 0u; }
// blockIdx.y: the sources of either side, then the intersections, in one
// launch: a source looks up whether an intersection leads its edge's order
__global__ __launch_bounds__(BLK) void k_augment(int J, const int *__restrict__ pj, int I, const int *__restrict__ pt,
                                               const double *__restrict__ px, const double *__restrict__ py,
                                               int *flags, AugSides sides, const uint32_t *over) {
    if (unordered_words(over)) return;
    const AugSide &z = sides.s[blockIdx.y & 1];
    const bool side_b = (blockIdx.y & 1) == 0;
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (blockIdx.y < 2) aug_source<true>(J, z, side_b, pt, i);
    else if (i < I) aug_segment<true>(pj, I, pt, px, py, flags, z, side_b, int(i));
}
// Many slots take two launches, and the intersection tells its source slot (256
// pairs with 32 million sources: 0.7 ms, with the look-ups 0.8; one kernel with
// both parts takes 0.15 longer than two).
__global__ void k_aug_sources(int J, AugSides sides) {
    aug_source<false>(J, sides.s[blockIdx.y], blockIdx.y == 0, nullptr,
                      int64_t(blockIdx.x) * blockDim.x + threadIdx.x);
}
__global__ void k_aug_segments(const int *__restrict__ pj, int I, const int *__restrict__ pt,
                               const double *__restrict__ px, const double *__restrict__ py, int *flags,
                               AugSides sides) {
    aug_segment<false>(pj, I, pt, px, py, flags, sides.s[blockIdx.y], blockIdx.y == 0,
                       int(blockIdx.x * blockDim.x + threadIdx.x));
}

// Neighbour links, 1-based and local to the job's rings (as the reference's
// arrays), and initial labels, by position on the base rings: the slots beside
// an intersection's are those of the positions beside it, or plain (a position
// without a slot, in a flagged job, is passed over).  over: words that say that
// an order is still to come.
struct LabelArgs {
    int J, I;
    const int *pj, *ord, *JB, *scan, *slot_b, *slot_c, *AB, *AC;
    const double *bx, *by, *cx, *cy;
    int *nbr_b, *nbr_c, *lab_b, *lab_c, *flags;
    const uint32_t *over;
};
__global__ __launch_bounds__(BLK) void k_link_labels(LabelArgs a) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (unordered_words(a.over) || i >= a.scan[a.JB[a.J]]) return;
    const int p = a.ord[i], j = a.pj[p];
    const int g = a.slot_b[p], h = a.slot_c[p];
    if (g < 0 || h < 0) {
        atomicOr(&a.flags[j], UB_UNASSIGNED);
        return;
    }
    const int B0 = a.AB[j], C0 = a.AC[j], nbaug = a.AB[j + 1] - B0, ncaug = a.AC[j + 1] - C0;
    a.nbr_b[g] = h - C0 + 1;
    a.nbr_c[h] = g - B0 + 1;
    const int first = a.scan[a.JB[j]], end = a.scan[a.JB[j + 1]]; // the job's positions
    // the partner of slot s (-100: a plain vertex, -101: an intersection without one), from position k on in steps d
    auto partner = [&](int s, int k, int d) {
        while (k >= first && k < end && a.slot_b[a.ord[k]] < 0) k += d;
        if (k < first || k >= end) return -100;
        const int q = a.ord[k];
        if (a.slot_b[q] != s) return -100;
        return a.slot_c[q] < 0 ? -101 : a.slot_c[q] - C0;
    };
    const int t = g - B0, tm = t == 0 ? nbaug - 1 : t - 1, tp = t + 1 == nbaug ? 0 : t + 1;
    const int pMN = partner(B0 + tm, t == 0 ? end - 1 : i - 1, -1);
    const int pPN = partner(B0 + tp, t + 1 == nbaug ? first : i + 1, 1);
    const int n = h - C0, qm = n == 0 ? ncaug - 1 : n - 1, qp = n + 1 == ncaug ? 0 : n + 1;
    const int lab = label_of(pMN, pPN, qm, qp, a.cx[C0 + qm], a.cy[C0 + qm], a.cx[C0 + qp], a.cy[C0 + qp],
                             a.bx[B0 + tm], a.by[B0 + tm], a.bx[g], a.by[g], a.bx[B0 + tp], a.by[B0 + tp]);
    a.lab_b[g] = lab;
    a.lab_c[h] = lab;
}

// The same in two launches, by pair and by slot: for many pairs, whose
// neighbours' pairs are worth more loads than a look at every slot (256 pairs
// with 40 million slots: 0.15 ms less).  The labels also of rings whose links
// are given.
__global__ void k_link(const int *__restrict__ sb, const int *__restrict__ scn, const int *__restrict__ pj, int I,
                       const int *__restrict__ AB, const int *__restrict__ AC, int *nbr_b, int *nbr_c, int *flags) {
    int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= I) return;
    int a = sb[p], b = scn[p], j = pj[p];
    if (a < 0 || b < 0) {
        atomicOr(&flags[j], UB_UNASSIGNED);
        return;
    }
    nbr_b[a] = b - AC[j] + 1;
    nbr_c[b] = a - AB[j] + 1;
}
__global__ void k_init_labels(int J, const int *__restrict__ AB, const int *__restrict__ AC,
                              const double *__restrict__ bx, const double *__restrict__ by,
                              const int *__restrict__ avb, const int *__restrict__ nbrb,
                              const double *__restrict__ cx, const double *__restrict__ cy, int *labb, int *labc,
                              int *flags) {
    int64_t g = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (g >= AB[J]) return;
    if (avb[g] == -100) return;
    int j = seg_of(AB, J, g);
    const int B0 = AB[j], nbaug = AB[j + 1] - B0, C0 = AC[j], ncaug = AC[j + 1] - C0;
    const int i = int(g - B0);
    int tm = i - 1 < 0 ? nbaug - 1 : i - 1;
    int tp = i + 1 == nbaug ? 0 : i + 1;
    int pMN = avb[B0 + tm] != -100 ? nbrb[B0 + tm] - 1 : -100;
    int pPN = avb[B0 + tp] != -100 ? nbrb[B0 + tp] - 1 : -100;
    int nId = nbrb[g] - 1;
    if (nId < 0 || nId >= ncaug) {
        atomicOr(&flags[j], UB_UNASSIGNED);
        return;
    }
    int qm = nId - 1 < 0 ? ncaug - 1 : nId - 1;
    int qp = nId + 1 == ncaug ? 0 : nId + 1;
    int lab = label_of(pMN, pPN, qm, qp, cx[C0 + qm], cy[C0 + qm], cx[C0 + qp], cy[C0 + qp], bx[B0 + tm],
                       by[B0 + tm], bx[g], by[g], bx[B0 + tp], by[B0 + tp]);
    labb[g] = lab;
    labc[C0 + nId] = lab;
}

// ---- sparse base ring ----

// per position: leading-degenerate / non-degenerate class (B side)
__global__ void k_sp_mark(int I, const int *__restrict__ ord, const int *__restrict__ pj, const int *__restrict__ pb,
                          const int *__restrict__ pt, const int *__restrict__ p0, int *kind, uint32_t *ndf,
                          int *flags, const uint32_t *__restrict__ unordered) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= I) return;
    if (unordered && *unordered) { // ord is not there yet: only the jobs' totals, which need no order
        ndf[i] = nondeg_b(pt[i]) ? 1u : 0u;
        return;
    }
    int p = ord[i], j = pj[p], e = pb[p], t = pt[p];
    bool start = i == p0[j] || pb[ord[i - 1]] != e;
    bool nd = nondeg_b(t), lead = start && degen_b_first(t);
    if (!nd && !lead) atomicOr(&flags[j], UB_UNASSIGNED);
    kind[i] = lead ? 1 : (nd ? 2 : 0);
    ndf[i] = nd ? 1u : 0u;
}

__global__ void k_sp_fill(int I, const int *__restrict__ ord, const int *__restrict__ pj, const int *__restrict__ pb,
                          const int *__restrict__ p0, const uint32_t *__restrict__ ndg, const int *__restrict__ bvoff,
                          const double *__restrict__ bpoly, const double *__restrict__ px,
                          const double *__restrict__ py, const int *__restrict__ qa, int *slot, int *ndx, int *edge,
                          int *av, int *nbr, int *lab, double *x, double *y, const int *kind,
                          const uint32_t *__restrict__ unordered) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= I) return;
    if (unordered && *unordered) {
        // No slot anywhere until the order is there: the labelling's first kernels
        // run before the host learns of it, and take an edge from a position that
        // holds a slot.
        slot[i] = -1;
        ndx[i] = 0;
        edge[i] = 0;
        av[i] = -100;
        nbr[i] = -100;
        lab[i] = 0;
        x[i] = 0.0;
        y[i] = 0.0;
        return;
    }
    int p = ord[i], j = pj[p], e = pb[p];
    int rel = int(ndg[i] - ndg[p0[j]]);
    int k = kind[i];
    slot[i] = k == 1 ? e + rel : (k == 2 ? e + 1 + rel : -1);
    ndx[i] = rel;
    edge[i] = e;
    av[i] = qa[p];
    nbr[i] = -100;
    lab[i] = 0;
    if (k == 2) {
        x[i] = px[p];
        y[i] = py[p];
    } else {
        const double *V = bpoly + 2 * (int64_t(bvoff[j]) + e);
        x[i] = V[0];
        y[i] = V[1];
    }
}

// links and labels on the sparse base ring
struct SpLabelArgs {
    int I, J;
    const int *pj, *ord, *slot_c, *AC;
    SparseP sp;
    const double *cx, *cy;
    int *nbr_p, *nbr_c, *lab_p, *lab_c, *flags;
    const uint32_t *over;
};
__global__ __launch_bounds__(BLK) void k_sp_link_labels(SpLabelArgs a) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.I || unordered_words(a.over)) return;
    const SparseP &sp = a.sp;
    const int j = a.pj[i], q = sp.slot[i], h = a.slot_c[a.ord[i]];
    if (q < 0 || h < 0 || h >= a.AC[a.J]) {
        atomicOr(&a.flags[j], UB_UNASSIGNED);
        return;
    }
    const int C0 = a.AC[j], ncaug = a.AC[j + 1] - C0, nbaug = sp.AB[j + 1] - sp.AB[j];
    a.nbr_p[i] = h - C0 + 1;
    a.nbr_c[h] = q + 1;
    const int tm = q == 0 ? nbaug - 1 : q - 1, tp = q + 1 == nbaug ? 0 : q + 1;
    // The slots beside q are held by the positions beside i or plain (slots ascend
    // with the positions unless the job was flagged); at the ring's ends by the
    // last position, or one past it, and by the first.
    SlotInfo pm, pp;
    if (a.flags[j] & UB_UNASSIGNED) {
        pm = sp_slot(sp, j, tm);
        pp = sp_slot(sp, j, tp);
    } else {
        const int first = sp.P0[j], end = sp.P0[j + 1];
        const int last = sp.slot[end - 1] == nbaug - 1 ? end - 1 : end;
        pm = sp_slot_at(sp, j, tm, q == 0 ? last : (i > first && sp.slot[i - 1] == tm ? i - 1 : i));
        pp = sp_slot_at(sp, j, tp, q + 1 == nbaug ? first : i + 1);
    }
    auto partner = [&](const SlotInfo &s) {
        if (s.pos < 0) return -100;
        const int o = a.slot_c[a.ord[s.pos]];
        return o < 0 || o >= a.AC[a.J] ? -101 : o - C0;
    };
    const int n = h - C0;
    if (n < 0 || n >= ncaug) {
        atomicOr(&a.flags[j], UB_UNASSIGNED);
        return;
    }
    const int qm = n == 0 ? ncaug - 1 : n - 1, qp = n + 1 == ncaug ? 0 : n + 1;
    const int lab = label_of(partner(pm), partner(pp), qm, qp, a.cx[C0 + qm], a.cy[C0 + qm], a.cx[C0 + qp],
                             a.cy[C0 + qp], pm.x, pm.y, sp.x[i], sp.y[i], pp.x, pp.y);
    a.lab_p[i] = lab;
    a.lab_c[h] = lab;
}

int bits_for(int64_t n) {
    int b = 0;
    while ((int64_t(1) << b) < n) b++;
    return b < 1 ? 1 : b;
}

} // namespace

// late: the augmented rings' offsets may stay on the device (js.late), where
// label_and_traverse reads them back with its own first values; a group too
// large for the ordering is then found there, and nothing after the ordering has
// run.  A read-back costs a small clip 20 us of 400.
void post_jobs(Ctx &c, int k0, int k1, bool late) {
    SC_REQUIRE(k0 >= 1 && k1 <= c.K && k0 <= k1, SC_EINVAL, "overlay index out of range");
    SC_REQUIRE(int(c.pair_off.size()) == c.K + 1, SC_ESTATE, "candidates not computed");
    hipStream_t s = c.stream;
    const int J = k1 - k0 + 1;
    JobSet &js = c.jobs;
    js.k0 = k0;
    js.J = J;
    js.resident = true;
    js.prov = c.prov;
    js.p0.assign(J + 1, 0);
    js.bvoff.resize(J);
    js.beoff.resize(J);
    js.nb.resize(J);
    js.nc.resize(J);
    js.cvoff.resize(J);
    js.JB.assign(J + 1, 0);
    js.JC.assign(J + 1, 0);
    js.cin.resize(J + 1);
    const int64_t P0 = c.pair_off[k0 - 1];
    for (int j = 0; j < J; ++j) {
        int k = k0 + j, br = job_base(c, k);
        js.p0[j + 1] = int(c.pair_off[k] - P0);
        js.bvoff[j] = c.bvoff[br];
        js.beoff[j] = c.beoff[br];
        js.nb[j] = c.bsz[br];
        js.nc[j] = c.csz[k - 1];
        js.cvoff[j] = c.coff[k - 1];
        js.cin[j] = c.eoff[k - 1] - c.nb;
        js.JB[j + 1] = js.JB[j] + js.nb[j] + 1;
        js.JC[j + 1] = js.JC[j] + js.nc[j] + 1;
    }
    const int I = js.p0[J];
    c.cur_k = J == 1 ? k0 : 0;
    c.I = I;
    js.cin[J] = c.eoff[k1] - c.nb;
    {
        // the job arrays back to back, one copy to the device
        const std::vector<int> *parts[] = {&js.p0, &js.bvoff, &js.beoff, &js.nb, &js.nc,
                                           &js.cvoff, &js.JB, &js.JC, &js.cin};
        int **views[] = {&js.d_p0, &js.d_bvoff, &js.d_beoff, &js.d_nb, &js.d_nc,
                         &js.d_cvoff, &js.d_JB, &js.d_JC, &js.d_cin};
        size_t tot = 0;
        for (const std::vector<int> *v : parts) tot += v->size();
        js.h_pack.resize(tot);
        int *dp = js.d_pack.ensure(tot);
        size_t at = 0;
        for (int q = 0; q < 9; ++q) {
            std::copy(parts[q]->begin(), parts[q]->end(), js.h_pack.begin() + at);
            *views[q] = dp + at;
            at += parts[q]->size();
        }
        c.upload(dp, js.h_pack.data(), sizeof(int) * tot);
    }
    JobArgs ja;
    ja.J = J;
    ja.p0 = js.d_p0;
    ja.bvoff = js.d_bvoff;
    ja.beoff = js.d_beoff;
    ja.nb = js.d_nb;
    ja.nc = js.d_nc;
    ja.cvoff = js.d_cvoff;
    ja.JB = js.d_JB;
    ja.JC = js.d_JC;
    const int nJB = js.JB[J], nJC = js.JC[J];
    const int Ia = I > 0 ? I : 1;
    // one-to-many batches keep the shared base ring sparse (no dense copy per job)
    const bool sparse = !c.paired && !c.prov && J >= 2;
    c.sparseP = sparse;
    c.p_j.ensure(Ia); c.p_b.ensure(Ia); c.p_c.ensure(Ia); c.p_type.ensure(Ia); c.p_x.ensure(Ia); c.p_y.ensure(Ia);
    c.p_qa.ensure(Ia); c.p_qb.ensure(Ia); c.ordB.ensure(Ia); c.ordC.ensure(Ia);
    c.slot_b.ensure(Ia); c.slot_c.ensure(Ia);
    FillBatch fb(s);
    int *all_b = nullptr, *dg_b = nullptr;
    if (!sparse) {
        all_b = c.all_b.ensure(nJB + 1);
        dg_b = c.dg_b.ensure(nJB + 1);
        fb.add(all_b, nJB + 1, 0u);
        fb.add(dg_b, nJB + 1, 0u);
    }
    int *all_c = c.all_c.ensure(nJC + 1), *dg_c = c.dg_c.ensure(nJC + 1);
    int *flags = c.flags.ensure(J);
    fb.add(flags, J, 0u);
    fb.add(all_c, nJC + 1, 0u);
    fb.add(dg_c, nJC + 1, 0u);
    fb.add(c.slot_b.p, Ia, ~0u);
    fb.add(c.slot_c.p, Ia, ~0u);
    uint32_t *segctl = c.seg_ctl.ensure(2 * SEG_CTL); // per side: list counts, too-large flag
    fb.add(segctl, 2 * SEG_CTL, 0u);
    if (sparse) {
        fb.add(c.sp_ndf.ensure(size_t(I) + 1) + I, 1, 0u); // closing entry of its scan
        fb.add(c.run_start.ensure(size_t(I) + 1), int64_t(I) + 1, uint32_t(I));
    }
    fb.flush();
    if (I > 0) {
        k_pair_decode<<<grid_for(I), BLK, 0, s>>>(ja, c.pairs.p + P0, I, c.bits_b, c.bits_c, c.bpoly, c.cpoly, c.p_j,
                                                  c.p_b, c.p_c, c.p_type, c.p_x, c.p_y, c.p_qa, c.p_qb, all_b, dg_b,
                                                  all_c, dg_c, flags, sparse ? nullptr : c.arr_b.ensure(Ia),
                                                  c.arr_c.ensure(Ia),
                                                  sparse ? c.run_head.ensure(Ia) : nullptr,
                                                  sparse ? c.seg_kb.ensure(Ia) : nullptr);
        SC_HIP(hipGetLastError());
    }
    {
        uint32_t *arr[4] = {reinterpret_cast<uint32_t *>(all_c), reinterpret_cast<uint32_t *>(dg_c),
                            reinterpret_cast<uint32_t *>(all_b), reinterpret_cast<uint32_t *>(dg_b)};
        const int64_t n[4] = {int64_t(nJC) + 1, int64_t(nJC) + 1, int64_t(nJB) + 1, int64_t(nJB) + 1};
        scan_exclusive_u32_4(sparse ? 2 : 4, arr, n, s);
    }

    // Per edge alpha order on each side (positions = the edge groups' count
    // offsets, on a sparse base side the runs of pairs of one edge): by ranking
    // inside the groups, or (a group beyond SEG_LDS_MAX) by one stable radix
    // sort of the pairs (in pair order) by (edge slot, quantised alpha).  The base
    // side of 4,096 jobs with 24 million pairs, most of them on edges with 64 to
    // 512, is ordered in 0.55 ms, by the sort's eight passes in 1.85.  Pairs are in (job, base edge,
    // overlay edge) order, so ties keep the base side's pair order and, on the
    // overlay side, base-edge order.
    const int bits_eb = bits_for(int64_t(nJB) + 1), bits_ec = bits_for(int64_t(nJC) + 1);
    SC_REQUIRE(bits_eb + 30 <= 64 && bits_ec + 30 <= 64, SC_ERANGE, "edge order key too wide");
    auto radix_order = [&](bool side_b) {
        const int *edge_of = side_b ? c.p_b.p : c.p_c.p;
        const int *JX = side_b ? ja.JB : ja.JC;
        k_edge_alpha_keys<<<grid_for(I), BLK, 0, s>>>(edge_of, c.p_j, JX, side_b ? c.p_qa : c.p_qb, I,
                                                      c.ord_key.ensure(Ia), c.ord_val.ensure(Ia));
        SC_HIP(hipGetLastError());
        radix_sort_u64_buf(c.ord_key, c.ord_key_alt, &c.ord_val, &c.ord_val_alt, I, 0,
                           (side_b ? bits_eb : bits_ec) + 30, c.rs, s);
        k_copy_order<<<grid_for(I), BLK, 0, s>>>(c.ord_val, I, side_b ? c.ordB : c.ordC);
        SC_HIP(hipGetLastError());
    };
    if (I > 0) {
        // the sides sorted inside their groups: the overlays, then the base rings (not sparse)
        ScatterSides sc{};
        SegSets ss{};
        auto groups = [&](const int *scan, int nseg, const uint64_t *K, DBuf<uint32_t> &wl, DBuf<uint32_t> &bl,
                          uint32_t *ctl, int *ord) {
            // listed groups hold more than SEG_THREAD (wave list) or SEG_WAVE_MAX (block list) pairs each
            const int64_t nw = std::min<int64_t>(nseg, int64_t(I) / (SEG_THREAD + 1)) + 1;
            const int64_t nb = std::min<int64_t>(nseg, int64_t(I) / (SEG_WAVE_MAX + 1)) + 1;
            ss.s[ss.count++] = SegSet{nseg, scan, K, ord, wl.ensure(size_t(nw)), bl.ensure(size_t(nb)), ctl};
        };
        sc.s[0] = ScatterSide{c.p_c, ja.JC, all_c, c.arr_c, c.p_qb, c.seg_kc.ensure(Ia)};
        groups(all_c, nJC, c.seg_kc, c.seg_wc, c.seg_bc, segctl + SEG_CTL, c.ordC);
        if (sparse) {
            uint32_t *run = c.u32c.ensure(Ia);
            scan_exclusive_u32(c.run_head, run, I, nullptr, s);
            k_run_starts<<<grid_for(I), BLK, 0, s>>>(I, c.run_head, run, c.run_start);
            groups(c.run_start, I, c.seg_kb, c.seg_wb, c.seg_bb, segctl, c.ordB);
        } else {
            sc.s[1] = ScatterSide{c.p_b, ja.JB, all_b, c.arr_b, c.p_qa, c.seg_kb.ensure(Ia)};
            groups(all_b, nJB, c.seg_kb, c.seg_wb, c.seg_bb, segctl, c.ordB);
        }
        k_seg_scatter<<<dim3(grid_for(I), sparse ? 1 : 2), BLK, 0, s>>>(I, c.p_j, sc);
        SC_HIP(hipGetLastError());
        seg_sort<false>(ss, I, s);
    }
    // augmented ring sizes and offsets per job
    int *nba = js.d_AB.ensure(J + 1), *nca = js.d_AC.ensure(J + 1);
    // sparse: the virtual slot of every base-side intersection (unordered: a
    // word that says that the base side's order is still to come)
    auto sparse_slots = [&](const uint32_t *unordered) {
        int *kind = reinterpret_cast<int *>(c.u32c.ensure(Ia));
        uint32_t *ndf = reinterpret_cast<uint32_t *>(c.sp_ndf.p);
        if (I > 0) {
            k_sp_mark<<<grid_for(I), BLK, 0, s>>>(I, c.ordB, c.p_j, c.p_b, c.p_type, ja.p0, kind, ndf, flags,
                                                  unordered);
            SC_HIP(hipGetLastError());
        }
        scan_exclusive_u32(ndf, ndf, int64_t(I) + 1, nullptr, s);
        int *slot = c.sp_slot.ensure(Ia), *ndx = c.sp_ndx.ensure(Ia), *edge = c.sp_edge.ensure(Ia);
        int *sav = c.sp_av.ensure(Ia), *snbr = c.sp_nbr.ensure(Ia);
        double *sx = c.sp_x.ensure(Ia), *sy = c.sp_y.ensure(Ia);
        c.sp_lab.ensure(Ia);
        if (I > 0) {
            k_sp_fill<<<grid_for(I), BLK, 0, s>>>(I, c.ordB, c.p_j, c.p_b, ja.p0, ndf, ja.bvoff, c.bpoly, c.p_x,
                                                  c.p_y, c.p_qa, slot, ndx, edge, sav, snbr, c.sp_lab, sx, sy,
                                                  kind, unordered);
            SC_HIP(hipGetLastError());
        }
    };
    if (sparse) sparse_slots(segctl + 2);
    const uint32_t *ndg = sparse ? reinterpret_cast<const uint32_t *>(c.sp_ndf.p) : nullptr;
    if (J < JOB_BLK * JOB_PER) {
        k_job_offsets<<<1, JOB_BLK, 0, s>>>(ja, NdScan{all_b, dg_b}, ndg, NdScan{all_c, dg_c}, nba, nca);
    } else {
        k_job_sizes<<<grid_for(int64_t(J) + 1), BLK, 0, s>>>(ja, NdScan{all_b, dg_b}, ndg, NdScan{all_c, dg_c}, nba, nca);
        uint32_t *ub = reinterpret_cast<uint32_t *>(nba), *uc = reinterpret_cast<uint32_t *>(nca);
        scan_exclusive_u32_2(ub, ub, int64_t(J) + 1, nullptr, uc, uc, int64_t(J) + 1, nullptr, s);
    }
    SC_HIP(hipGetLastError());
    js.late = late && I <= LATE_MAX;
    js.AB.clear();
    js.AC.clear();
    js.cap_b = int64_t(nJB) - J + I;
    js.cap_c = int64_t(nJC) - J + I;
    if (!js.late) {
        js.AB.resize(J + 1);
        js.AC.resize(J + 1);
    }
    uint32_t hseg[2 * SEG_CTL] = {};
    if (!js.late) {
        ReadBack rb(c);
        rb.add(js.AB.data(), static_cast<const int *>(nba), size_t(J) + 1);
        rb.add(js.AC.data(), static_cast<const int *>(nca), size_t(J) + 1);
        if (I > 0) rb.add(hseg, static_cast<const uint32_t *>(segctl), size_t(2 * SEG_CTL));
        rb.run();
    }
    // a group too large for LDS: that side's order by the radix sort instead
    if (hseg[2]) {
        radix_order(true);
        if (sparse) sparse_slots(nullptr);
    }
    if (hseg[SEG_CTL + 2]) radix_order(false);
    const int64_t nba_tot = js.late ? js.cap_b : js.AB[J], nca_tot = js.late ? js.cap_c : js.AC[J];
    c.nbaug = js.late ? 0 : int(nba_tot);
    c.ncaug = js.late ? 0 : int(nca_tot);
    const uint32_t *over = js.late && I > 0 ? segctl : nullptr;

    const int64_t nbaA = nba_tot > 0 ? nba_tot : 1, ncaA = nca_tot > 0 ? nca_tot : 1;
    c.aug_cx.ensure(ncaA); c.aug_cy.ensure(ncaA); c.av_c.ensure(ncaA); c.nbr_c.ensure(ncaA); c.lab_c.ensure(ncaA);
    int *from_b = c.prov ? c.from_b.ensure(nbaA) : nullptr, *from_c = c.prov ? c.from_c.ensure(ncaA) : nullptr;
    AugSides as{};
    if (!sparse) {
        c.aug_bx.ensure(nbaA); c.aug_by.ensure(nbaA); c.av_b.ensure(nbaA); c.nbr_b.ensure(nbaA); c.lab_b.ensure(nbaA);
        as.s[0] = AugSide{ja.JB, ja.nb, ja.bvoff, nba, c.bpoly, all_b, NdScan{all_b, dg_b}, c.p_b, c.ordB, c.p_qa, c.aug_bx,
                          c.aug_by, c.av_b, c.nbr_b, c.lab_b, from_b, c.slot_b};
    }
    as.s[1] = AugSide{ja.JC, ja.nc, ja.cvoff, nca, c.cpoly, all_c, NdScan{all_c, dg_c}, c.p_c, c.ordC, c.p_qb, c.aug_cx,
                      c.aug_cy, c.av_c, c.nbr_c, c.lab_c, from_c, c.slot_c};
    // (the sparse base side has slots by the hundred million and none of these arrays)
    const int64_t nsrc = sparse ? nJC : std::max(nJB, nJC);
    if (over || std::max<int64_t>(I, nsrc) < SPAN_MIN) {
        k_augment<<<dim3(grid_for(std::max<int64_t>(I, nsrc)), I > 0 ? 4 : 2), BLK, 0, s>>>(
            J, c.p_j, I, c.p_type, c.p_x, c.p_y, flags, as, over);
    } else {
        k_aug_sources<<<dim3(grid_for(nsrc), 2), BLK, 0, s>>>(J, as);
        if (I > 0) k_aug_segments<<<dim3(grid_for(I), 2), BLK, 0, s>>>(c.p_j, I, c.p_type, c.p_x, c.p_y, flags, as);
    }
    SC_HIP(hipGetLastError());
    if (I > 0) {
        if (sparse) {
            SpLabelArgs la{I, J, c.p_j, c.ordB, c.slot_c, nca, sparse_view(c), c.aug_cx, c.aug_cy, c.sp_nbr, c.nbr_c,
                           c.sp_lab, c.lab_c, flags, over};
            k_sp_link_labels<<<grid_for(I), BLK, 0, s>>>(la);
        } else if (I > LATE_MAX) {
            k_link<<<grid_for(I), BLK, 0, s>>>(c.slot_b, c.slot_c, c.p_j, I, nba, nca, c.nbr_b, c.nbr_c, flags);
            k_init_labels<<<grid_for(nba_tot), BLK, 0, s>>>(J, nba, nca, c.aug_bx, c.aug_by, c.av_b, c.nbr_b,
                                                            c.aug_cx, c.aug_cy, c.lab_b, c.lab_c, flags);
        } else {
            LabelArgs la{J, I, c.p_j, c.ordB, ja.JB, all_b, c.slot_b, c.slot_c, nba, nca, c.aug_bx, c.aug_by, c.aug_cx,
                         c.aug_cy, c.nbr_b, c.nbr_c, c.lab_b, c.lab_c, flags, over};
            k_link_labels<<<grid_for(I), BLK, 0, s>>>(la);
        }
        SC_HIP(hipGetLastError());
    }
    js.flags.assign(size_t(J), 0);
    c.flags_pending = true; // read back later, with the next read-back that needs a wait anyway
}

void fetch_flags(Ctx &c) {
    if (!c.flags_pending) return;
    JobSet &js = c.jobs;
    ReadBack rb(c);
    rb.add(js.flags.data(), static_cast<const int *>(c.flags.p), size_t(js.J));
    rb.run();
    c.flags_pending = false;
    int any = 0;
    for (int f : js.flags) any |= f;
    c.undefined = any;
}

void post_overlay(Ctx &c, int k) {
    pairs_after_move(c);
    post_jobs(c, k, k);
}

SparseP sparse_view(Ctx &c) {
    SparseP v;
    v.P0 = c.jobs.d_p0;
    v.AB = c.jobs.d_AB;
    v.nbv = c.jobs.d_nb;
    v.bvoff = c.jobs.d_bvoff;
    v.slot = c.sp_slot;
    v.ndx = c.sp_ndx;
    v.edge = c.sp_edge;
    v.x = c.sp_x;
    v.y = c.sp_y;
    v.bpoly = c.bpoly;
    return v;
}

void init_labels_one(Ctx &c, int nba, int nca, const double *bx, const double *by, const int *avb, const int *nbrb,
                     const double *cx, const double *cy, int *labb, int *labc, int *flags) {
    hipStream_t s = c.stream;
    std::vector<int> off = {0, nba, 0, nca};
    thread_local DBuf<int> *dd = new DBuf<int>(); // scratch, kept for the thread's lifetime
    int *d = dd->ensure(4);
    SC_HIP(hipMemcpyAsync(d, off.data(), sizeof(int) * 4, hipMemcpyHostToDevice, s));
    {
        FillBatch fb(s);
        fb.add(labb, nba, 0u);
        fb.add(labc, nca, 0u);
        fb.flush();
    }
    k_init_labels<<<grid_for(nba), BLK, 0, s>>>(1, d, d + 2, bx, by, avb, nbrb, cx, cy, labb, labc, flags);
    SC_HIP(hipGetLastError());
    SC_HIP(hipStreamSynchronize(s)); // off is a stack vector
}

} // namespace sc
