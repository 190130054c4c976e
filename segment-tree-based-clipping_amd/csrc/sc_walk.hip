// sc_walk.hip -- the sequential labelling route run over the whole device.
//
// The route takes the jobs whose crossings are not plainly alternating: rings
// with intersection chains, split bouncing pairs, an odd number of crossings,
// a link that was never made, and every union.  On large rings these are
// accidents: a few of a million crossings fall within the reference's 1e-9.
// One block per job (k_sequential) spends 1 to 4 seconds on such a pair of
// 200,000 x 1,000,000 vertices, most of it in one lane walking one long
// ring a node at a time.  Here the same steps run on every CU and the single
// walk is left only around the accidents:
//   - chains (labelIntersections2 step 2), split pairs and crossing
//     candidates (steps 5, 6) one after another by one thread, from short
//     lists that the whole device gathers;
//   - entry/exit flags (step 4) by a scan of state tables;
//   - createResult2's walks on "specials": the nodes with an entry/exit flag
//     and the crossing candidates.  From special i the walk goes to the next
//     special a in its direction; if a carries the opposite flag the piece
//     ends there and the walk goes on from a's neighbour s.  A step is plain
//     when that holds, s carries a flag and its neighbour is a.  Steps that
//     are not plain mark every special that they visit as touched.  Plain
//     steps none of whose specials (i, a, s) is touched are linked: each
//     special has at most one linked step in and one out, so the links form
//     cycles and paths, found by doubling with the distance in vertices to
//     the cycle's smallest candidate or to the path's end.
//     A cycle is a ring of its own: no other step visits its specials, the
//     reversed cycle visits the same ones, and the reference starts it at
//     their smallest base-ring candidate.  Everything else is walked in
//     the reference's order by one thread per job that crosses a path in one
//     step, and stops where its start is visited again.
//   - the check of the walked rings: every start is first visited by its own
//     ring and every other candidate by a ring that starts before it.  Then
//     the single walk would give the same rings (by induction over the
//     starts).
// A job that exceeds a list, has a ring without plain or crossing vertices, or
// fails the check is left to k_sequential (its 'old' word is set).
//
// Measured (MI355X, 200,000 x 1,000,000 harmonic rings with 1 to 15 such
// accidents): the whole clip 970 to 4,100 ms -> 1.3 to 3.6; 13 to 16 such
// overlays among 100,000 x 4,096: their labelling 52 -> 12.9 ms.
#include "sc_fp64.hpp"
#include "sc_seqroute.hpp"

#include <algorithm>

namespace sc {

namespace {

constexpr int BLK = 256;
constexpr int LIST = 256;         // chain starts, split pairs, crossing candidates per job
constexpr int TERMS = 2048;       // specials per job whose step is not linked
constexpr int SINGLES = 4096;     // their walked steps per job
constexpr int WALK_ROUNDS = 4;    // walks and their check
constexpr int MAX_MICRO = 1 << 15; // specials stepped over singly by one job's walks
constexpr uint32_t DEAD = 0xfffffffeu; // no neighbour node
constexpr uint32_t ONCYCLE = 0x80000000u;

inline unsigned grid_for(int64_t n, int per = BLK) {
    int64_t g = ceil_div(n, per);
    if (g < 1) g = 1;
    return unsigned(g);
}

struct WalkJob {
    int old;                 // left to k_sequential
    int V[2];                // first plain node of each ring
    int cross[2];            // ring has a crossing vertex
    int nchain, nsplit[2], ncross[2];
    int n;                   // nodes, inserted ones included
    uint32_t nterm, fail;    // specials without a linked step; the start whose walk never closes
    uint32_t nsingle;
    uint32_t wrong;          // the smallest candidate that the last check did not accept
    uint32_t extra[WALK_ROUNDS]; // candidates that earlier checks found unvisited
    int nextra;
};
// a walked stretch of a path: its specials with distance in (lo, hi] to the
// path's end, 'off' vertices after the start of the ring that begins at 'ring';
// at 'last' the ring closes before the jump
struct Stretch {
    uint32_t lo, hi, off, ring, last;
};
// per special without a linked step; rings that run into one another walk a
// path more than once, each output keeps its own copy
constexpr int STRETCHES = 4;
struct Term {
    uint32_t i;        // the special
    uint32_t cand;     // smallest candidate whose own step lies on the path that ends here
    uint32_t nst, pad; // stretches used
    Stretch st[STRETCHES];
};
// a walked step that is not linked: from special i, 'off' vertices after ring 'ring's start
struct Single {
    uint32_t i, off, ring, pad;
};

struct WalkArgs {
    SeqBatch b;
    const int64_t *nodeoff, *segoff;
    const uint32_t *nidx;
    const int *firstP, *firstQ;
    int nseq;
    int64_t N;
    uint32_t cap;            // specials
    WalkJob *gj;
    uint64_t *lists;         // per walking job (SeqJob::walk): chain starts, P split list, P crossing list, of LIST entries
    uint32_t *tab, *tsum;    // state tables by node, per block
    uint32_t *cnt, *ins;     // per node: specials / inserted nodes there, then before it (N + 1)
    // per special
    uint32_t *spn;           // node -> special (NIL: none), in k_sequential's node numbering
    uint32_t *sw, *su, *sinfo, *snb, *slen, *succ, *tpos, *mark;
    uint8_t *touched, *linked;
    uint4 *rec, *rec2;
    Term *terms;
    Single *singles;
    uint32_t *isstart, *tot; // then their scans
    uint32_t *head, *piece;  // by output vertex, job after job at obase
    int *done;
};

__device__ inline int seg_find(const int64_t *off, int n, int64_t t) { // last g with off[g] <= t
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (off[mid] <= t) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}
__device__ inline uint32_t specials(const WalkArgs &a) { return a.cnt[a.N]; }
// ring g = 2q + (0: P, 1: Q) of the jobs: its specials are [ring_first, ring_first of g + 1)
__device__ inline uint32_t ring_first(const WalkArgs &a, int g) { return a.cnt[a.nodeoff[g]]; }
// sinfo: enex | candidate << 2 | ring g << 3
__device__ inline int info_enex(uint32_t f) { return int(f & 3u); }
__device__ inline bool info_cand(uint32_t f) { return (f & 4u) != 0u; }
__device__ inline int info_ring(uint32_t f) { return int(f >> 3); }

// ---- chains ----

__global__ void k_walk_init(WalkArgs a) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= a.nseq) return;
    const SeqJob &jb = a.b.jobs[q];
    WalkJob g;
    const int fp = a.firstP[jb.j], fq = a.firstQ[jb.j];
    g.old = jb.walk < 0 || jb.nPn + jb.nQn > jb.cap || fp < 0 || fq < 0 ? 1 : 0;
    g.V[0] = g.V[1] = 0;
    if (!g.old) { // a first plain slot starts a node
        g.V[0] = int(int64_t(a.nidx[a.segoff[2 * q] + fp]) - a.nodeoff[2 * q]);
        g.V[1] = int(int64_t(a.nidx[a.segoff[2 * q + 1] + fq]) - a.nodeoff[2 * q]);
    }
    g.cross[0] = g.cross[1] = 0;
    g.nchain = g.nsplit[0] = g.nsplit[1] = g.ncross[0] = g.ncross[1] = 0;
    g.n = jb.nPn + jb.nQn;
    g.nterm = g.nsingle = 0;
    g.fail = g.wrong = NIL;
    g.nextra = 0;
    a.gj[q] = g;
}

// chain starts: P intersections labelled LEFT_ON or RIGHT_ON
__global__ void k_walk_chain_starts(WalkArgs a) {
    const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= a.N) return;
    const int g = seg_find(a.nodeoff, 2 * a.nseq, t), q = g >> 1;
    if ((g & 1) || a.gj[q].old) return;
    const int v = int(t - a.nodeoff[2 * q]);
    const int64_t w = a.b.jobs[q].vbase + v;
    const int lb = a.b.lab[w];
    if (!a.b.inter[w] || (lb != L_LEFT_ON && lb != L_RIGHT_ON)) return;
    const int k = atomicAdd(&a.gj[q].nchain, 1);
    if (k < LIST) a.lists[int64_t(a.b.jobs[q].walk) * 3 * LIST + k] = uint64_t(v);
}

// ascending order of a short list, by one block (every thread calls it)
__device__ inline void sort_list(uint64_t *l, int n, uint64_t *s) {
    for (int i = threadIdx.x; i < n; i += blockDim.x) s[i] = l[i];
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        int r = 0;
        for (int j = 0; j < n; ++j) r += s[j] < s[i] ? 1 : 0; // keys are distinct
        l[r] = s[i];
    }
    __syncthreads();
}

// the chains in ring order, one block per job, walked by one thread: the
// reference's loop over the starts, a start relabelled by an earlier chain skipped
__global__ __launch_bounds__(BLK) void k_walk_chains(WalkArgs a) {
    __shared__ uint64_t s[LIST];
    const int q = blockIdx.x;
    WalkJob &g = a.gj[q];
    const int n = g.nchain;
    if (g.old || n == 0) return;
    if (n > LIST) {
        __syncthreads();
        if (threadIdx.x == 0) g.old = 1;
        return;
    }
    uint64_t *l = a.lists + int64_t(a.b.jobs[q].walk) * 3 * LIST;
    sort_list(l, n, s);
    if (threadIdx.x != 0) return;
    const int64_t vb = a.b.jobs[q].vbase;
    int *lab = a.b.lab + vb;
    const int *nb = a.b.nb + vb, *nx = a.b.nx + vb;
    for (int k = 0; k < n; ++k) {
        const int X = int(l[k]);
        if (lab[X] != L_LEFT_ON && lab[X] != L_RIGHT_ON) continue;
        const int x = lab[X] == L_LEFT_ON ? 0 : 1;
        int J = X, guard = 0;
        do {
            lab[J] = L_NONE;
            if (nb[J] >= 0) lab[nb[J]] = L_NONE;
            J = nx[J];
            if (++guard > g.n) {
                g.old = 1;
                return;
            }
        } while (lab[J] == L_ON_ON);
        const int y = lab[J] == L_ON_LEFT ? 0 : 1;
        const int ct = x != y ? L_DCROSS : L_DBOUNCE;
        lab[X] = ct;
        lab[J] = ct;
        if (nb[X] >= 0) lab[nb[X]] = ct;
        if (nb[J] >= 0) lab[nb[J]] = ct;
    }
}

// ---- entry/exit flags ----

// Node tables scanned in node order.  Bit 8 marks a table that starts anew: a
// ring's first node, and its first plain node, whose table is constant (the
// status there is known).  op(x, y): x first.
constexpr uint32_t TAB_HEAD = 0x100u;
__device__ inline uint32_t tab_op(uint32_t x, uint32_t y) {
    return (y & TAB_HEAD) ? y : ((x & TAB_HEAD) | seq_tcompose(x & 0xffu, y & 0xffu));
}
constexpr int TAB_ITEMS = 8;
constexpr int TAB_TILE = BLK * TAB_ITEMS;

// exclusive composition over the block's threads; tot: the block's
__device__ inline uint32_t tab_block(uint32_t x, uint32_t *s_w, uint32_t &tot) {
    const int lane = threadIdx.x & (WAVE - 1), wid = threadIdx.x / WAVE;
    uint32_t inc = x;
    for (int d = 1; d < WAVE; d <<= 1) {
        const uint32_t o = __shfl_up(inc, d, WAVE);
        if (lane >= d) inc = tab_op(o, inc);
    }
    if (lane == WAVE - 1) s_w[wid] = inc;
    __syncthreads();
    uint32_t ex = __shfl_up(inc, 1, WAVE);
    if (lane == 0) ex = SEQ_TAB_ID;
    uint32_t before = SEQ_TAB_ID, t = SEQ_TAB_ID;
    for (int w = 0; w < BLK / WAVE; ++w) {
        if (w < wid) before = tab_op(before, s_w[w]);
        t = tab_op(t, s_w[w]);
    }
    __syncthreads();
    tot = t;
    return tab_op(before, ex);
}

__global__ __launch_bounds__(BLK) void k_walk_tables(WalkArgs a) {
    __shared__ uint32_t s_w[BLK / WAVE];
    const int64_t t0 = int64_t(blockIdx.x) * TAB_TILE + int64_t(threadIdx.x) * TAB_ITEMS;
    uint32_t acc = SEQ_TAB_ID;
    int g = -1;
    int64_t gend = 0;
    for (int it = 0; it < TAB_ITEMS; ++it) {
        const int64_t t = t0 + it;
        if (t >= a.N) break;
        if (g < 0 || t >= gend) {
            g = seg_find(a.nodeoff, 2 * a.nseq, t);
            gend = a.nodeoff[g + 1];
        }
        const int q = g >> 1, sd = g & 1;
        uint32_t tab = SEQ_TAB_ID;
        if (!a.gj[q].old) {
            const SeqJob &jb = a.b.jobs[q];
            const int v = int(t - a.nodeoff[2 * q]);
            const int64_t w = jb.vbase + v;
            const int lb = a.b.lab[w];
            if (a.b.inter[w]) {
                tab = seq_table(lb);
                bool cr = lb == L_CROSSING || lb == L_DCROSS;
                if (a.b.uni && (lb == L_BOUNCING || lb == L_DBOUNCE)) cr = true;
                if (cr && !a.gj[q].cross[sd]) a.gj[q].cross[sd] = 1; // noCrossingVertex
            }
            if (v == a.gj[q].V[sd]) {
                const bool in = ((sd ? a.b.windQ : a.b.windP)[jb.j] % 2) != 0;
                const uint32_t x = uint32_t(in ? EXIT : ENTRY) | 2u; // first = true
                tab = TAB_HEAD | (x * 0x55u);
            } else if (t == a.nodeoff[g]) {
                tab |= TAB_HEAD;
            }
        }
        a.tab[t] = tab;
        acc = tab_op(acc, tab);
    }
    uint32_t tot;
    (void)tab_block(acc, s_w, tot);
    if (threadIdx.x == 0) a.tsum[blockIdx.x] = tot;
}

// the tiles' tables to the composition before each tile (one block)
__global__ __launch_bounds__(BLK) void k_walk_tab_sums(uint32_t *sum, int n) {
    __shared__ uint32_t s_w[BLK / WAVE];
    uint32_t carry = SEQ_TAB_ID;
    for (int b = 0; b < n; b += BLK * TAB_ITEMS) {
        const int i0 = b + int(threadIdx.x) * TAB_ITEMS;
        uint32_t v[TAB_ITEMS], acc = SEQ_TAB_ID;
#pragma unroll
        for (int it = 0; it < TAB_ITEMS; ++it) {
            v[it] = i0 + it < n ? sum[i0 + it] : SEQ_TAB_ID;
            acc = tab_op(acc, v[it]);
        }
        uint32_t tot;
        uint32_t run = tab_op(carry, tab_block(acc, s_w, tot));
#pragma unroll
        for (int it = 0; it < TAB_ITEMS; ++it) {
            if (i0 + it < n) sum[i0 + it] = run;
            run = tab_op(run, v[it]);
        }
        carry = tab_op(carry, tot);
    }
}

// inclusive composition at every node, in place
__global__ __launch_bounds__(BLK) void k_walk_tab_scan(WalkArgs a) {
    __shared__ uint32_t s_w[BLK / WAVE];
    const int64_t t0 = int64_t(blockIdx.x) * TAB_TILE + int64_t(threadIdx.x) * TAB_ITEMS;
    uint32_t v[TAB_ITEMS], acc = SEQ_TAB_ID;
#pragma unroll
    for (int it = 0; it < TAB_ITEMS; ++it) {
        v[it] = t0 + it < a.N ? a.tab[t0 + it] : SEQ_TAB_ID;
        acc = tab_op(acc, v[it]);
    }
    uint32_t tot;
    uint32_t run = tab_op(a.tsum[blockIdx.x], tab_block(acc, s_w, tot));
#pragma unroll
    for (int it = 0; it < TAB_ITEMS; ++it) {
        run = tab_op(run, v[it]);
        if (t0 + it < a.N) a.tab[t0 + it] = run;
    }
}

// flags, relabelled delayed crossings, split and crossing lists (labelIntersections2 step 4)
__global__ void k_walk_enex(WalkArgs a) {
    const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= a.N) return;
    const int g = seg_find(a.nodeoff, 2 * a.nseq, t), q = g >> 1, sd = g & 1;
    WalkJob &wj = a.gj[q];
    if (wj.old) return;
    const int64_t r0 = a.nodeoff[g], r1 = a.nodeoff[g + 1];
    const int v = int(t - a.nodeoff[2 * q]), V = wj.V[sd];
    if (t == r0 && !wj.cross[sd]) wj.old = 1; // a ring without crossings is output whole: k_sequential
    const SeqJob &jb = a.b.jobs[q];
    const int64_t w = jb.vbase + v;
    if (!a.b.inter[w]) return;
    const int lab = a.b.lab[w];
    const uint32_t E = t == r0 ? SEQ_TAB_ID : (a.tab[t - 1] & 0xffu);
    // before the first plain node: the state carried around the ring's end
    const int x = v > V ? seq_tapply(E, 0) : seq_tapply(E, seq_tapply(a.tab[r1 - 1] & 0xffu, 0));
    const int st = x & 1;
    const bool first = (x >> 1) != 0, uni = a.b.uni != 0;
    bool addS = false, addC = false;
    if (lab == L_CROSSING) {
        a.b.enex[w] = st;
    } else if (lab == L_BOUNCING) {
        addS = (st == EXIT) != uni;
    } else if (lab == L_DCROSS) {
        a.b.enex[w] = st;
        if (first ? ((st == EXIT) != uni) : ((st == ENTRY) != uni)) a.b.lab[w] = L_CROSSING;
    } else if (lab == L_DBOUNCE) {
        a.b.enex[w] = st;
        addC = first ? ((st == EXIT) != uni) : ((st == ENTRY) != uni);
    }
    if (!addS && !addC) return;
    const int k = atomicAdd(addS ? &wj.nsplit[sd] : &wj.ncross[sd], 1);
    if (sd) { // membership marks
        a.b.seen[2 * w + (addS ? 0 : 1)] = -1;
    } else if (k < LIST) {
        const int m = int(r1 - r0), p = v > V ? v - V : v - V + m; // place on the walk
        a.lists[int64_t(jb.walk) * 3 * LIST + (addS ? LIST : 2 * LIST) + k] = (uint64_t(uint32_t(p)) << 32) | uint32_t(v);
    }
}

// split bouncing pairs and crossing candidates in walk order (steps 5, 6), one thread per job
__global__ __launch_bounds__(BLK) void k_walk_split(WalkArgs a) {
    __shared__ uint64_t s[LIST];
    const int q = blockIdx.x;
    WalkJob &wj = a.gj[q];
    const int old = wj.old, nS = wj.nsplit[0], nC = wj.ncross[0];
    const SeqJob &jb = a.b.jobs[q];
    // beyond the lists here or k_sequential's (cap / 4 entries): left to it
    const int lim = jb.cap / 4;
    const bool over = nS > LIST || nC > LIST || nS > lim || nC > lim || wj.nsplit[1] > lim || wj.ncross[1] > lim;
    __syncthreads();
    if (old) return;
    if (over) {
        if (threadIdx.x == 0) wj.old = 1;
        return;
    }
    uint64_t *lS = a.lists + int64_t(jb.walk) * 3 * LIST + LIST, *lC = lS + LIST;
    sort_list(lS, nS, s);
    sort_list(lC, nC, s);
    if (threadIdx.x != 0) return;
    const int64_t vb = jb.vbase;
    double *vx = a.b.vx + vb, *vy = a.b.vy + vb, *vx1 = a.b.vx1 + vb, *vy1 = a.b.vy1 + vb;
    int *nx = a.b.nx + vb, *pv = a.b.pv + vb, *nb = a.b.nb + vb, *lab = a.b.lab + vb, *enex = a.b.enex + vb;
    int *vlen = a.b.vlen + vb, *vslot = a.b.vslot + vb, *vsrc = a.b.vsrc + vb;
    const int *seen = a.b.seen + 2 * vb;
    uint8_t *inter = a.b.inter + vb;
    const int n0 = jb.nPn + jb.nQn;
    int n = n0;
    auto snew = [&](int I) { // a copy of node I's vertex, its own ring until inserted
        const int v = n++;
        vx[v] = vx1[v] = vx[I];
        vy[v] = vy1[v] = vy[I];
        vlen[v] = 1;
        vslot[v] = -1;
        vsrc[v] = vslot[I] < 0 ? vsrc[I] : (I < jb.nPn ? jb.P0 + vslot[I] : ~(jb.Q0 + vslot[I]));
        nx[v] = pv[v] = v;
        return v;
    };
    auto insert = [&](int V, int curr) {
        const int c = nx[curr];
        nx[pv[c]] = V;
        pv[V] = pv[c];
        nx[V] = c;
        pv[c] = V;
    };
    for (int i = 0; i < nS; ++i) {
        const int IP = int(uint32_t(lS[i])), IQ = nb[IP];
        if (!(IQ >= 0 && IQ < n0 && seen[2 * IQ] == -1)) continue;
        if (n + 2 > jb.cap) { // cannot happen: cap is over twice the nodes
            wj.old = 1;
            return;
        }
        const int VP = snew(IP), VQ = snew(IQ);
        const double sP = areaA(vx1[pv[IP]], vy1[pv[IP]], vx[IP], vy[IP], vx[nx[IP]], vy[nx[IP]]);
        const double sQ = areaA(vx1[pv[IQ]], vy1[pv[IQ]], vx[IQ], vy[IQ], vx[nx[IQ]], vy[nx[IQ]]);
        inter[VP] = inter[VQ] = 1;
        if (sP * sQ > 0) {
            nb[IP] = VQ;
            nb[VQ] = IP;
            nb[IQ] = VP;
            nb[VP] = IQ;
            inter[IP] = inter[IQ] = 1;
        } else {
            nb[VP] = VQ;
            nb[VQ] = VP;
        }
        insert(VP, IP);
        insert(VQ, IQ);
        enex[IP] = enex[IQ] = a.b.uni ? ENTRY : EXIT;
        enex[VP] = enex[VQ] = a.b.uni ? EXIT : ENTRY;
        lab[IP] = lab[VP] = lab[IQ] = lab[VQ] = L_CROSSING;
    }
    for (int i = 0; i < nC; ++i) {
        const int IP = int(uint32_t(lC[i])), IQ = nb[IP];
        if (IQ >= 0 && IQ < n0 && seen[2 * IQ + 1] == -1) {
            lab[IP] = L_CROSSING;
            lab[IQ] = L_CROSSING;
        }
    }
    wj.n = n;
}

// ---- specials ----

__device__ inline bool is_special(const SeqBatch &b, int64_t w) {
    return (b.inter[w] != 0 && b.lab[w] == L_CROSSING) || b.enex[w] != NEITHER;
}

// specials and inserted nodes at every node (an inserted node counts with the node before it)
__global__ void k_walk_count(WalkArgs a) {
    const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t > a.N) return;
    uint32_t c = 0, ni = 0;
    if (t < a.N) {
        const int q = seg_find(a.nodeoff, 2 * a.nseq, t) >> 1;
        const WalkJob &wj = a.gj[q];
        if (!wj.old) {
            const SeqJob &jb = a.b.jobs[q];
            const int n0 = jb.nPn + jb.nQn;
            const int64_t w = jb.vbase + (t - a.nodeoff[2 * q]);
            c = is_special(a.b, w) ? 1u : 0u;
            if (wj.n > n0)
                for (int x = a.b.nx[w], k = n0; x >= n0 && k < wj.n; x = a.b.nx[jb.vbase + x], ++k) {
                    c += is_special(a.b, jb.vbase + x) ? 1u : 0u;
                    ++ni;
                }
        }
    }
    a.cnt[t] = c;
    a.ins[t] = ni;
}

__global__ void k_walk_specials(WalkArgs a) {
    const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= a.N) return;
    const int g = seg_find(a.nodeoff, 2 * a.nseq, t), q = g >> 1;
    const WalkJob &wj = a.gj[q];
    if (wj.old) return;
    const SeqJob &jb = a.b.jobs[q];
    const int n0 = jb.nPn + jb.nQn;
    const int64_t w0 = jb.vbase + (t - a.nodeoff[2 * q]);
    uint32_t i = a.cnt[t];
    // first vertex of the node in its ring: its slot and one per node inserted before it
    uint32_t u = uint32_t(a.b.vslot[w0]) + (a.ins[t] - a.ins[a.nodeoff[g]]);
    int64_t w = w0;
    for (int k = n0;; ++k) {
        const bool cand = a.b.inter[w] != 0 && a.b.lab[w] == L_CROSSING;
        const int e = a.b.enex[w];
        a.spn[w] = cand || e != NEITHER ? i : NIL;
        if (cand || e != NEITHER) {
            a.sw[i] = uint32_t(w - jb.vbase);
            a.su[i] = u;
            a.sinfo[i] = uint32_t(e) | (cand ? 4u : 0u) | (uint32_t(g) << 3);
            a.touched[i] = 0;
            a.mark[i] = NIL;
            ++i;
        }
        if (wj.n <= n0 || k > wj.n) break;
        u += uint32_t(a.b.vlen[w]);
        const int x = a.b.nx[w];
        if (x < n0) break;
        w = jb.vbase + x;
    }
}

__global__ void k_walk_links(WalkArgs a) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= specials(a)) return;
    const int64_t vb = a.b.jobs[info_ring(a.sinfo[i]) >> 1].vbase;
    const int nb = a.b.nb[vb + a.sw[i]];
    a.snb[i] = nb < 0 ? DEAD : a.spn[vb + nb];
}

// the direction of the walk from a special with flag e
__device__ inline bool walks_fwd(int e, int uni) { return (seq_toggle(e) == EXIT) != (uni != 0); }
// the special after c in that direction on its ring [r0, r1)
__device__ inline uint32_t next_special(uint32_t c, bool fwd, uint32_t r0, uint32_t r1) {
    return fwd ? (c + 1 == r1 ? r0 : c + 1) : (c == r0 ? r1 - 1 : c - 1);
}
// vertices of ring g, inserted ones included
__device__ inline uint32_t ring_vertices(const WalkArgs &a, int g) {
    const SeqJob &jb = a.b.jobs[g >> 1];
    return uint32_t((g & 1) ? jb.nQ : jb.nP) + (a.ins[a.nodeoff[g + 1]] - a.ins[a.nodeoff[g]]);
}
// vertices stepped over from special c to special d
__device__ inline uint32_t step_len(const WalkArgs &a, uint32_t c, uint32_t d, bool fwd, uint32_t total) {
    const int l = fwd ? int(a.su[d]) - int(a.su[c]) : int(a.su[c]) - int(a.su[d]);
    return uint32_t(l <= 0 ? l + int(total) : l);
}

// plain steps; the others mark what they visit
__global__ void k_walk_steps(WalkArgs a) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= specials(a)) return;
    const uint32_t f = a.sinfo[i];
    const int g = info_ring(f), e = info_enex(f);
    const uint32_t r0 = ring_first(a, g), r1 = ring_first(a, g + 1);
    const bool fwd = walks_fwd(e, a.b.uni);
    const int st = seq_toggle(e);
    uint32_t c = next_special(i, fwd, r0, r1);
    uint32_t s = NIL;
    bool plain = false;
    if (e != NEITHER && info_enex(a.sinfo[c]) == st) {
        s = a.snb[c];
        plain = s < DEAD && info_enex(a.sinfo[s]) != NEITHER && a.snb[s] == c;
    }
    a.linked[i] = plain ? 1 : 0;
    a.succ[i] = plain ? s : i;
    a.slen[i] = plain ? step_len(a, i, c, fwd, ring_vertices(a, g)) : 0u;
    if (plain) return;
    a.touched[i] = 1;
    if (e == NEITHER) return;
    for (int k = 0; k < MAX_MICRO; ++k) {
        a.touched[c] = 1;
        if (info_enex(a.sinfo[c]) == st) {
            const uint32_t n = a.snb[c];
            if (n < DEAD) a.touched[n] = 1;
            return;
        }
        if (c == i) return; // around the ring: no special ends the step
        c = next_special(c, fwd, r0, r1);
    }
    a.gj[g >> 1].old = 1;
}

// links between untouched specials; doubling records (see k_walk_jump)
__global__ void k_walk_cut(WalkArgs a) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= specials(a)) return;
    const uint32_t f = a.sinfo[i];
    const int g = info_ring(f), q = g >> 1;
    bool link = a.linked[i] != 0;
    uint32_t c = 0;
    if (link) {
        c = next_special(i, walks_fwd(info_enex(f), a.b.uni), ring_first(a, g), ring_first(a, g + 1));
        link = !a.touched[i] && !a.touched[c] && !a.touched[a.succ[i]];
    }
    a.tpos[i] = NIL;
    if (link) {
        // candidates of this step on the base ring: i by its own step, c reached by it
        uint32_t v = 0x7fffffffu;
        if (!(g & 1)) {
            if (info_cand(f)) v = 2u * i;
            if (info_cand(a.sinfo[c])) v = min(v, 2u * c + 1u);
        }
        a.linked[i] = 2;
        a.rec[i] = make_uint4(ONCYCLE | v, 0u, a.slen[i], a.succ[i]);
        return;
    }
    a.rec[i] = make_uint4(i, 0u, 0u, i);
    const uint32_t k = atomicAdd(&a.gj[q].nterm, 1u);
    if (k >= uint32_t(TERMS)) {
        a.gj[q].old = 1;
        return;
    }
    Term t;
    t.i = i;
    t.cand = NIL;
    t.nst = t.pad = 0;
    const int64_t at = int64_t(a.b.jobs[q].walk) * TERMS + k;
    a.terms[at] = t;
    a.tpos[i] = uint32_t(at);
}

// Doubling over the links.  A record: (smallest value of the window, vertices
// from the special to where that value is, vertices of the window, the special
// after it).  A path's last special has its own index as value, below every
// candidate's (ONCYCLE | 2 * special + (0: by its own step, 1: reached)), and
// links to itself with no vertices.  A round that moves no smallest value has
// windows as long as every cycle and path, and later rounds return at once;
// a window sum is read only when its window holds no occurrence of the final
// value, so it does not wrap.
__global__ void k_walk_jump(WalkArgs a, const uint4 *__restrict__ rec, uint4 *__restrict__ rec2, uint32_t *moved,
                            int r) {
    if (r > 0 && moved[r - 1] == 0u) return;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= specials(a)) return;
    const uint4 x = rec[i];
    const uint4 y = rec[x.w];
    uint4 o;
    o.x = x.x <= y.x ? x.x : y.x;
    o.y = x.x <= y.x ? x.y : x.z + y.y;
    o.z = x.z + y.z;
    o.w = y.w;
    rec2[i] = o;
    if (o.x != x.x) moved[r] = 1u;
}

// per path: the smallest base candidate whose own step lies on it
__global__ void k_walk_paths(WalkArgs a) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= specials(a) || a.linked[i] != 2) return;
    const uint32_t f = a.sinfo[i], m = a.rec[i].x;
    if ((m & ONCYCLE) || (info_ring(f) & 1) || !info_cand(f)) return;
    const uint32_t k = a.tpos[m];
    if (k == NIL) return; // over the list: the job is old
    if (i < __hip_atomic_load(&a.terms[k].cand, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        atomicMin(&a.terms[k].cand, i);
}

// ---- the walks off the cycles: one block per job, walked by thread 0 ----
// Starts are taken in order from the candidates that look unvisited: ends of
// paths by their marks, paths as a whole.  A path that was walked in part can
// hold more: the check then names the first, and the next round walks again
// with it among the candidates.
__global__ __launch_bounds__(BLK) void k_walk_walks(WalkArgs a, int again) {
    __shared__ uint32_t s_min[BLK / WAVE];
    __shared__ int s_end;
    const int q = blockIdx.x;
    WalkJob &wj = a.gj[q];
    if (wj.old) return; // uniform: written by earlier launches only
    if (again && wj.wrong == NIL) return;
    const int nt = int(wj.nterm);
    const int walk = a.b.jobs[q].walk;
    Term *T = a.terms + int64_t(walk) * TERMS;
    const int uni = a.b.uni;
    const int lane = threadIdx.x & (WAVE - 1), wid = threadIdx.x / WAVE;
    int micro = 0; // thread 0: specials stepped over singly so far
    if (again) { // marks and starts are cleared (k_walk_reset)
        __syncthreads();
        if (threadIdx.x == 0) {
            wj.extra[wj.nextra++] = wj.wrong; // one per round
            wj.wrong = wj.fail = NIL;
            wj.nsingle = 0;
        }
        for (int k = threadIdx.x; k < nt; k += BLK) T[k].nst = 0;
        __syncthreads();
    }
    // the special reached by the linked step from i
    auto reached = [&](uint32_t i) {
        const uint32_t f = a.sinfo[i];
        const int g = info_ring(f);
        return next_special(i, walks_fwd(info_enex(f), uni), ring_first(a, g), ring_first(a, g + 1));
    };
    for (;;) {
        // the smallest candidate not visited yet: an end of a path (visited: marked, or reached by
        // a walked path's link), or a path no ring has walked in either direction
        uint32_t m = NIL;
        for (int k = threadIdx.x; k < nt; k += BLK) {
            const Term &t = T[k];
            const uint32_t f = a.sinfo[t.i];
            if (!(info_ring(f) & 1) && info_cand(f) && a.mark[t.i] == NIL) {
                bool seen = false;
                if (a.linked[t.i] == 1) { // a plain step: its far special may link back to t.i
                    const uint32_t w = reached(t.i);
                    if (a.linked[w] == 2 && reached(w) == t.i) {
                        const uint32_t x = a.rec[w].x;
                        seen = (x & ONCYCLE) || a.terms[a.tpos[x]].nst > 0;
                    }
                }
                if (!seen) m = min(m, t.i);
            }
            if (t.cand != NIL && t.nst == 0 && a.mark[t.cand] == NIL) {
                const uint32_t w = reached(t.cand); // the reversed path visits the same specials
                bool seen = false;
                if (a.linked[w] == 2) {
                    const uint32_t x = a.rec[w].x;
                    seen = (x & ONCYCLE) || a.terms[a.tpos[x]].nst > 0;
                }
                if (!seen) m = min(m, t.cand);
            }
        }
        // linked candidates named by the checks: visited by a stretch over their own step
        // or over the one that reaches them
        if (int(threadIdx.x) < wj.nextra) {
            const uint32_t x = wj.extra[threadIdx.x];
            if (a.linked[x] == 2 && a.mark[x] == NIL) {
                auto walked = [&](uint32_t i) {
                    const uint4 r = a.rec[i];
                    if (r.x & ONCYCLE) return true;
                    const Term &t = a.terms[a.tpos[r.x]];
                    for (uint32_t k = 0; k < t.nst; ++k)
                        if (r.y > t.st[k].lo && r.y <= t.st[k].hi) return true;
                    return false;
                };
                const uint32_t w = reached(x);
                if (!walked(x) && !(a.linked[w] == 2 && reached(w) == x && walked(w))) m = min(m, x);
            }
        }
        for (int d = 1; d < WAVE; d <<= 1) m = min(m, uint32_t(__shfl_xor(int(m), d, WAVE)));
        if (lane == 0) s_min[wid] = m;
        __syncthreads();
        if (threadIdx.x == 0) {
            uint32_t x = NIL;
            for (int w = 0; w < BLK / WAVE; ++w) x = min(x, s_min[w]);
            s_end = x == NIL ? 1 : 0;
            if (x != NIL) {
                const uint32_t I = x;
                uint32_t cur = I, off = 0;
                int ends = 0;
                bool closed = false;
                a.mark[I] = min(a.mark[I], I);
                while (!closed) {
                    const uint4 r = a.rec[cur];
                    if (a.linked[cur] == 2) {
                        // along a path: to its end, or to the start where that lies on the way
                        if (r.x & ONCYCLE) { // off the cycles no walk enters one
                            wj.old = 1;
                            break;
                        }
                        Term &t = a.terms[a.tpos[r.x]];
                        uint32_t lo = 0, last = NIL;
                        const uint4 ri = a.rec[I];
                        if (ri.x == r.x && ri.y < r.y) { // jumped to
                            lo = ri.y;
                            closed = true;
                        }
                        const uint32_t fI = a.sinfo[I];
                        // the special whose linked step reaches I: the one I's own flag points to
                        if (info_enex(fI) != NEITHER) {
                            const uint32_t w = reached(I);
                            if (a.linked[w] == 2 && reached(w) == I) {
                                const uint4 rw = a.rec[w];
                                if (rw.x == r.x && rw.y <= r.y && rw.y > lo) {
                                    lo = rw.y - 1u; // w's own step is walked
                                    last = w;
                                    closed = true;
                                }
                            }
                        }
                        bool twice = false; // entered there before: the walk never closes
                        for (uint32_t k = 0; k < t.nst; ++k)
                            if (t.st[k].ring == I && t.st[k].hi == r.y) twice = true;
                        if (twice) {
                            closed = false;
                            wj.fail = I;
                            break;
                        }
                        if (t.nst >= uint32_t(STRETCHES)) {
                            closed = false;
                            wj.old = 1;
                            break;
                        }
                        Stretch sg;
                        sg.lo = lo;
                        sg.hi = r.y;
                        sg.off = off;
                        sg.ring = I;
                        sg.last = last;
                        t.st[t.nst++] = sg;
                        if (last != NIL) off += r.y - a.rec[last].y + a.slen[last];
                        else off += r.y - lo;
                        if (!closed) {
                            cur = r.x;
                            a.mark[cur] = min(a.mark[cur], I);
                            if (cur == I) closed = true;
                        }
                        continue;
                    }
                    // a step that is not linked, special by special
                    if (++ends > nt) { // some end twice: the walk never closes
                        wj.fail = I;
                        break;
                    }
                    const uint32_t f = a.sinfo[cur];
                    const int g = info_ring(f), e = info_enex(f), st = seq_toggle(e);
                    if (e == NEITHER || wj.nsingle >= uint32_t(SINGLES)) {
                        wj.old = 1;
                        break;
                    }
                    const uint32_t r0 = ring_first(a, g), r1 = ring_first(a, g + 1), total = ring_vertices(a, g);
                    const bool fwd = walks_fwd(e, uni);
                    uint32_t c = cur, len = 0;
                    bool stop = false;
                    for (;;) {
                        const uint32_t d = next_special(c, fwd, r0, r1);
                        len += step_len(a, c, d, fwd, total);
                        c = d;
                        a.mark[c] = min(a.mark[c], I);
                        if (c == I) {
                            closed = true;
                            break;
                        }
                        if (info_enex(a.sinfo[c]) == st) break;
                        if (c == cur) { // around the ring: the walk never closes
                            wj.fail = I;
                            stop = true;
                            break;
                        }
                        if (++micro > MAX_MICRO) {
                            wj.old = 1;
                            stop = true;
                            break;
                        }
                    }
                    if (stop) break;
                    Single sg;
                    sg.i = cur;
                    sg.off = off;
                    sg.ring = I;
                    sg.pad = 0;
                    a.singles[int64_t(walk) * SINGLES + wj.nsingle++] = sg;
                    off += len;
                    if (closed) break;
                    const uint32_t n = a.snb[c];
                    if (n == DEAD) { // createResult2 jumps to no neighbour
                        wj.fail = I;
                        break;
                    }
                    if (n == NIL) {
                        wj.old = 1;
                        break;
                    }
                    a.mark[n] = min(a.mark[n], I);
                    if (n == I) closed = true;
                    cur = n;
                }
                if (closed) {
                    a.isstart[I] = 1u;
                    a.tot[I] = off;
                } else {
                    s_end = 1;
                }
            }
            __threadfence_block();
        }
        __syncthreads();
        if (s_end) return;
    }
}

// before another round: jobs whose check named a candidate start over
__global__ void k_walk_reset(WalkArgs a) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= specials(a)) return;
    const WalkJob &wj = a.gj[info_ring(a.sinfo[i]) >> 1];
    if (wj.wrong == NIL || (a.rec[i].x & ONCYCLE)) return;
    a.mark[i] = NIL;
    a.isstart[i] = a.tot[i] = 0u;
}

// what the walked stretches of linked steps visit
__global__ void k_walk_marks(WalkArgs a) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= specials(a) || a.linked[i] != 2) return;
    const uint4 r = a.rec[i];
    if (r.x & ONCYCLE) return;
    const uint32_t f = a.sinfo[i];
    const int g = info_ring(f);
    if (a.gj[g >> 1].old) return;
    const Term &t = a.terms[a.tpos[r.x]];
    for (uint32_t k = 0; k < t.nst; ++k) {
        const Stretch s = t.st[k];
        if (!(r.y > s.lo && r.y <= s.hi)) continue;
        const uint32_t c = next_special(i, walks_fwd(info_enex(f), a.b.uni), ring_first(a, g), ring_first(a, g + 1));
        atomicMin(&a.mark[c], s.ring);
        if (i != s.last) atomicMin(&a.mark[a.succ[i]], s.ring);
    }
}

// The check, and the cycles' starts.  Off the cycles every start is first
// visited by its own ring, every other candidate by a ring that starts before
// it; where a walk never closes, the same for the candidates before that
// start, and no earlier ring visits it.
__global__ void k_walk_check(WalkArgs a) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= specials(a)) return;
    const uint32_t f = a.sinfo[i];
    const int g = info_ring(f);
    WalkJob &wj = a.gj[g >> 1];
    if ((g & 1) || !info_cand(f)) return;
    const uint4 r = a.rec[i];
    if (r.x & ONCYCLE) {
        const uint32_t v = r.x & 0x7fffffffu;
        if (v == 2u * i) { // the cycle's smallest candidate, by its own step
            const uint32_t s = a.succ[i];
            a.isstart[i] = 1u;
            a.tot[i] = a.slen[i] + (s == i ? 0u : a.rec[s].y);
        }
        return;
    }
    if (i > wj.fail) return;
    const uint32_t m = a.mark[i];
    const bool ok = i == wj.fail ? m >= i : (a.isstart[i] ? m == i : m < i);
    if (!ok) atomicMin(&wj.wrong, i);
}

// starts of jobs that failed or are left to k_sequential do not count
__global__ void k_walk_drop(WalkArgs a) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= specials(a) || !a.isstart[i]) return;
    const WalkJob &wj = a.gj[info_ring(a.sinfo[i]) >> 1];
    if (wj.old || wj.wrong != NIL || wj.fail != NIL) a.isstart[i] = a.tot[i] = 0u;
}

// rings and vertices of every job (isstart and tot hold their scans now)
__global__ void k_walk_result(WalkArgs a) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= a.nseq) return;
    const WalkJob &wj = a.gj[q];
    const SeqJob &jb = a.b.jobs[q];
    const uint32_t i0 = ring_first(a, 2 * q), i1 = ring_first(a, 2 * q + 1);
    const uint32_t rings = a.isstart[i1] - a.isstart[i0], verts = a.tot[i1] - a.tot[i0];
    const bool fail = wj.fail != NIL;
    if (wj.old || wj.wrong != NIL || (!fail && (rings > uint32_t(jb.ring_cap) || verts > uint32_t(jb.out_cap)))) {
        a.done[q] = 0;
        return;
    }
    a.done[q] = 1;
    int *res = a.b.result + 3 * q;
    res[0] = int(rings);
    res[1] = int(verts);
    res[2] = fail ? int(UB_TRAVERSAL) : 0;
    a.b.ring_off[jb.rbase] = 0;
}

// every step's first output vertex carries the step's special; ring offsets
__device__ inline void place(const WalkArgs &a, int q, uint32_t I, uint32_t off, uint32_t i) {
    const int64_t o = a.b.jobs[q].obase + (a.tot[I] - a.tot[ring_first(a, 2 * q)]) + off;
    a.head[o] = uint32_t(o);
    a.piece[o] = i;
}
__global__ void k_walk_heads(WalkArgs a) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= specials(a)) return;
    const int q = info_ring(a.sinfo[i]) >> 1;
    if (!a.done[q] || a.gj[q].fail != NIL) return;
    if (a.isstart[i + 1] != a.isstart[i]) {
        const uint32_t i0 = ring_first(a, 2 * q);
        a.b.ring_off[a.b.jobs[q].rbase + (a.isstart[i] - a.isstart[i0])] = int(a.tot[i] - a.tot[i0]);
    }
    if (a.linked[i] != 2) return;
    const uint4 r = a.rec[i];
    if (r.x & ONCYCLE) {
        const uint32_t v = r.x & 0x7fffffffu;
        if (v == 0x7fffffffu || (v & 1u)) return; // no candidate, or the reversed cycle
        const uint32_t I = v >> 1, L = a.tot[I + 1] - a.tot[I];
        place(a, q, I, i == I ? 0u : L - r.y, i);
    } else {
        const Term &t = a.terms[a.tpos[r.x]];
        for (uint32_t k = 0; k < t.nst; ++k)
            if (r.y > t.st[k].lo && r.y <= t.st[k].hi) place(a, q, t.st[k].ring, t.st[k].off + (t.st[k].hi - r.y), i);
    }
}
__global__ void k_walk_single_heads(WalkArgs a) { // one block per job
    const int q = blockIdx.x;
    if (!a.done[q] || a.gj[q].fail != NIL) return;
    for (uint32_t k = threadIdx.x; k < a.gj[q].nsingle; k += blockDim.x) {
        const Single t = a.singles[int64_t(a.b.jobs[q].walk) * SINGLES + k];
        place(a, q, t.ring, t.off, t.i);
    }
}

// the rings' vertices into the batch's output, grid-stride over each job
__global__ void k_walk_emit(WalkArgs a, const uint32_t *JV, const uint32_t *JR, double *ox, double *oy, int *osrc,
                            int *off, int q0) {
    const int q = q0 + int(blockIdx.y);
    if (!a.done[q]) return;
    const SeqJob &jb = a.b.jobs[q];
    const int rings = a.b.result[3 * q], verts = a.b.result[3 * q + 1];
    const uint32_t V0 = JV[jb.j], R0 = JR[jb.j];
    const int n0 = jb.nPn + jb.nQn, ni = a.gj[q].n - n0;
    for (int r = blockIdx.x * blockDim.x + threadIdx.x; r < rings; r += gridDim.x * blockDim.x)
        off[R0 + r] = int(V0) + a.b.ring_off[jb.rbase + r];
    for (int o = blockIdx.x * blockDim.x + threadIdx.x; o < verts; o += gridDim.x * blockDim.x) {
        const uint32_t h = a.head[jb.obase + o];
        const uint32_t i = a.piece[h];
        const uint32_t f = a.sinfo[i];
        const int g = info_ring(f);
        const int total = int(ring_vertices(a, g));
        const int k = int(uint32_t(jb.obase + o) - h) + 1;
        int u = (int(a.su[i]) + (walks_fwd(info_enex(f), a.b.uni) ? k : -k)) % total;
        if (u < 0) u += total;
        int slot = u;
        int64_t node = -1; // an inserted node's vertex
        if (ni > 0) {
            // the node of vertex u: last t of the ring whose first vertex is at or before u
            int64_t lo = a.nodeoff[g], hi = a.nodeoff[g + 1] - 1;
            const uint32_t b0 = a.ins[lo];
            const int64_t t0 = a.nodeoff[2 * q];
            while (lo < hi) {
                const int64_t mid = (lo + hi + 1) >> 1;
                if (a.b.vslot[jb.vbase + (mid - t0)] + int(a.ins[mid] - b0) <= u) lo = mid;
                else hi = mid - 1;
            }
            const int64_t w = jb.vbase + (lo - t0);
            int d = u - (a.b.vslot[w] + int(a.ins[lo] - b0)) - a.b.vlen[w];
            slot = u - int(a.ins[lo] - b0);
            if (d >= 0) { // the d-th node inserted after it
                node = jb.vbase + a.b.nx[w];
                for (; d > 0; --d) node = jb.vbase + a.b.nx[node];
            }
        }
        const bool onP = !(g & 1);
        double x, y;
        int src;
        if (node >= 0) {
            x = a.b.vx[node];
            y = a.b.vy[node];
            src = a.b.vsrc[node];
        } else {
            x = (onP ? a.b.px + jb.P0 : a.b.qx + jb.Q0)[slot];
            y = (onP ? a.b.py + jb.P0 : a.b.qy + jb.Q0)[slot];
            src = onP ? jb.P0 + slot : ~(jb.Q0 + slot);
        }
        ox[V0 + o] = x;
        oy[V0 + o] = y;
        osrc[V0 + o] = src;
    }
}

struct WalkScratch {
    DBuf<uint64_t> gj, lists, terms, singles, rec, rec2;
    DBuf<uint32_t> tab, tsum, cnt, ins, spn, special, moved, head, piece, starts;
    DBuf<uint8_t> bytes;
};
WalkScratch &scratch() {
    thread_local WalkScratch *p = new WalkScratch();
    return *p;
}

WalkArgs walk_args(const WalkIn &in, int *done) {
    WalkScratch &f = scratch();
    WalkArgs a;
    a.b = in.b;
    a.nodeoff = in.nodeoff;
    a.segoff = in.segoff;
    a.nidx = in.nidx;
    a.firstP = in.firstP;
    a.firstQ = in.firstQ;
    a.nseq = int(in.jobs->size());
    a.N = in.N;
    a.cap = uint32_t(in.N) + 2u * uint32_t(LIST) * uint32_t(in.nwalk);
    a.done = done;
    const SeqJob &lastj = in.jobs->back();
    const int64_t nv = lastj.vbase + lastj.cap, no = lastj.obase + lastj.out_cap;
    a.gj = reinterpret_cast<WalkJob *>(f.gj.ensure(size_t(a.nseq) * ((sizeof(WalkJob) + 7) / 8)));
    a.lists = f.lists.ensure(size_t(in.nwalk) * 3 * LIST);
    a.terms = reinterpret_cast<Term *>(f.terms.ensure(size_t(in.nwalk) * TERMS * sizeof(Term) / 8));
    a.singles = reinterpret_cast<Single *>(f.singles.ensure(size_t(in.nwalk) * SINGLES * sizeof(Single) / 8));
    a.rec = reinterpret_cast<uint4 *>(f.rec.ensure(2 * size_t(a.cap)));
    a.rec2 = reinterpret_cast<uint4 *>(f.rec2.ensure(2 * size_t(a.cap)));
    a.tab = f.tab.ensure(size_t(a.N));
    a.tsum = f.tsum.ensure(size_t(ceil_div(a.N, TAB_TILE)));
    a.cnt = f.cnt.ensure(size_t(a.N) + 1);
    a.ins = f.ins.ensure(size_t(a.N) + 1);
    a.spn = f.spn.ensure(size_t(nv));
    uint32_t *sp = f.special.ensure(8 * size_t(a.cap));
    a.sw = sp;
    a.su = sp + size_t(a.cap);
    a.sinfo = sp + 2 * size_t(a.cap);
    a.snb = sp + 3 * size_t(a.cap);
    a.slen = sp + 4 * size_t(a.cap);
    a.succ = sp + 5 * size_t(a.cap);
    a.tpos = sp + 6 * size_t(a.cap);
    a.mark = sp + 7 * size_t(a.cap);
    a.touched = f.bytes.ensure(2 * size_t(a.cap));
    a.linked = a.touched + a.cap;
    uint32_t *st = f.starts.ensure(2 * (size_t(a.cap) + 1));
    a.isstart = st;
    a.tot = st + size_t(a.cap) + 1;
    a.head = f.head.ensure(size_t(no));
    a.piece = f.piece.ensure(size_t(no));
    return a;
}

static_assert(sizeof(Term) % 8 == 0 && sizeof(Single) % 8 == 0, "allocated in 8-byte words");

} // namespace

bool walk_jobs(const WalkIn &in, int *done, hipStream_t s) {
    uint32_t most = 1;
    for (const SeqJob &j : *in.jobs)
        if (j.walk >= 0) most = std::max(most, uint32_t(j.nPn + j.nQn) + 2u * uint32_t(LIST));
    const int nseq = int(in.jobs->size());
    // specials are counted in 30 bits, output places in 32
    const SeqJob &lastj = in.jobs->back();
    if (in.nwalk == 0 || in.N + 2 * int64_t(LIST) * in.nwalk >= (int64_t(1) << 29) ||
        lastj.obase + lastj.out_cap >= (int64_t(1) << 32) - 1)
        return false;
    WalkArgs a;
    try {
        a = walk_args(in, done);
    } catch (const Error &e) { // 300 KB a job: k_sequential needs none of it
        if (e.code != SC_ENOMEM) throw;
        release_walk_scratch();
        return false;
    }
    const int64_t no = lastj.obase + lastj.out_cap;
    const unsigned gn = grid_for(a.N), gs = grid_for(a.cap), gq = grid_for(nseq);
    const unsigned nt = unsigned(ceil_div(a.N, TAB_TILE));
    const int rounds = ilog2_exact(most);
    uint32_t *moved = scratch().moved.ensure(size_t(rounds) + 1);
    {
        FillBatch fb(s);
        fb.add(moved, rounds + 1, 0u);
        fb.add(a.isstart, 2 * (int64_t(a.cap) + 1), 0u); // and tot
        fb.add(a.head, no, 0u);
        fb.flush();
    }
    k_walk_init<<<gq, BLK, 0, s>>>(a);
    k_walk_chain_starts<<<gn, BLK, 0, s>>>(a);
    k_walk_chains<<<unsigned(nseq), BLK, 0, s>>>(a);
    k_walk_tables<<<nt, BLK, 0, s>>>(a);
    k_walk_tab_sums<<<1, BLK, 0, s>>>(a.tsum, int(nt));
    k_walk_tab_scan<<<nt, BLK, 0, s>>>(a);
    k_walk_enex<<<gn, BLK, 0, s>>>(a);
    k_walk_split<<<unsigned(nseq), BLK, 0, s>>>(a);
    k_walk_count<<<grid_for(a.N + 1), BLK, 0, s>>>(a);
    SC_HIP(hipGetLastError());
    scan_exclusive_u32_2(a.cnt, a.cnt, a.N + 1, nullptr, a.ins, a.ins, a.N + 1, nullptr, s);
    k_walk_specials<<<gn, BLK, 0, s>>>(a);
    k_walk_links<<<gs, BLK, 0, s>>>(a);
    k_walk_steps<<<gs, BLK, 0, s>>>(a);
    k_walk_cut<<<gs, BLK, 0, s>>>(a);
    for (int r = 0; r < rounds; ++r) {
        k_walk_jump<<<gs, BLK, 0, s>>>(a, a.rec, a.rec2, moved, r);
        std::swap(a.rec, a.rec2);
    }
    k_walk_paths<<<gs, BLK, 0, s>>>(a);
    for (int r = 0; r < WALK_ROUNDS; ++r) {
        if (r > 0) k_walk_reset<<<gs, BLK, 0, s>>>(a);
        k_walk_walks<<<unsigned(nseq), BLK, 0, s>>>(a, r);
        k_walk_marks<<<gs, BLK, 0, s>>>(a);
        k_walk_check<<<gs, BLK, 0, s>>>(a);
    }
    k_walk_drop<<<gs, BLK, 0, s>>>(a);
    SC_HIP(hipGetLastError());
    scan_exclusive_u32_2(a.isstart, a.isstart, int64_t(a.cap) + 1, nullptr, a.tot, a.tot, int64_t(a.cap) + 1, nullptr,
                         s);
    k_walk_result<<<gq, BLK, 0, s>>>(a);
    k_walk_heads<<<gs, BLK, 0, s>>>(a);
    k_walk_single_heads<<<unsigned(nseq), BLK, 0, s>>>(a);
    SC_HIP(hipGetLastError());
    scan_inclusive_max_u32(a.head, a.head, no, s);
    return true;
}

void walk_emit(const WalkIn &in, const int *done, const uint32_t *JV, const uint32_t *JR, double *ox, double *oy,
               int *osrc, int *off, hipStream_t s) {
    WalkArgs a = walk_args(in, const_cast<int *>(done));
    int64_t big = 1;
    for (const SeqJob &j : *in.jobs) big = std::max<int64_t>(big, int64_t(j.nP) + j.nQ);
    const unsigned bx = unsigned(std::min<int64_t>(ceil_div(big, BLK), 8192));
    for (int q0 = 0; q0 < a.nseq; q0 += 65535) {
        k_walk_emit<<<dim3(bx, unsigned(std::min(65535, a.nseq - q0))), BLK, 0, s>>>(a, JV, JR, ox, oy, osrc, off, q0);
        SC_HIP(hipGetLastError());
    }
}

void release_walk_scratch() {
    WalkScratch &f = scratch();
    for (DBuf<uint64_t> *b : {&f.gj, &f.lists, &f.terms, &f.singles, &f.rec, &f.rec2}) b->release();
    for (DBuf<uint32_t> *b : {&f.tab, &f.tsum, &f.cnt, &f.ins, &f.spn, &f.special, &f.moved, &f.head, &f.piece,
                              &f.starts})
        b->release();
    f.bytes.release();
}

} // namespace sc
