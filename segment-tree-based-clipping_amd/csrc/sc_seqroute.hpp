// sc_seqroute.hpp -- jobs of the sequential labelling route, shared by the
// kernels that run the reference's steps one after another (sc_foster.hip)
// and those that run them over the whole device (sc_walk.hip).
#pragma once
#include "sc_ctx.hpp"

#include <climits>

namespace sc {

enum : int {
    L_NONE = 0, L_CROSSING = 1, L_BOUNCING = 2, L_LEFT_ON = 3, L_RIGHT_ON = 4, L_ON_ON = 5,
    L_ON_LEFT = 6, L_ON_RIGHT = 7, L_DCROSS = 8, L_DBOUNCE = 9
};
enum : int { EXIT = 0, ENTRY = 1, NEITHER = 2 };
enum : int { UB_TRAVERSAL = 4 };
constexpr int SRC_NONE = INT_MIN;
constexpr uint32_t NIL = 0xffffffffu;

__device__ inline int seq_toggle(int s) { return s == ENTRY ? EXIT : (s == EXIT ? ENTRY : s); }

// the entry/exit walk's state (status, first of a delayed pair) as 2 bits
// x = st | first << 1 (EXIT = 0, ENTRY = 1); a node's effect on it is a
// 4-entry table of 2-bit states, and tables compose along the ring
constexpr uint32_t SEQ_TAB_ID = 0xE4u;
__device__ inline int seq_tapply(uint32_t t, int x) { return int((t >> (2 * x)) & 3u); }
__device__ inline uint32_t seq_tcompose(uint32_t f, uint32_t g) { // f first, then g
    uint32_t h = 0;
#pragma unroll
    for (int x = 0; x < 4; ++x) h |= ((g >> (2 * ((f >> (2 * x)) & 3u))) & 3u) << (2 * x);
    return h;
}
__device__ inline uint32_t seq_table(int lab) { // of an intersection with this label
    if (lab == L_CROSSING) return 0xB1u; // status toggles
    if (lab == L_DCROSS) return 0x4Bu;   // first: clear it; else set it, toggle
    if (lab == L_DBOUNCE) return 0x1Bu;  // first flips, status toggles
    return SEQ_TAB_ID;
}

// sequential route for several jobs: one block per job, its first wave runs seq_run
struct SeqJob {
    int j;                     // job
    int nP, nQ, P0, Q0;        // ring sizes (slots) and first slots in the dense ring arrays
    int node0, nPn, nQn;       // first node, node counts of P and Q
    int cap, out_cap, ring_cap;
    int walk;                  // its place among the jobs that sc_walk.hip takes, -1: none of them
    int64_t vbase, obase, rbase; // scratch bases: vertices, output vertices, ring offsets
};

struct SeqBatch {
    const SeqJob *jobs;
    const double *px, *py, *qx, *qy;
    const double *nx0, *ny0, *nx1, *ny1;
    const int *nlen, *nslot, *ninter, *nlab, *nnb;
    const int *windP, *windQ;
    double *vx, *vy, *vx1, *vy1;
    int *vlen, *vslot, *nx, *pv, *nb, *lab, *enex, *vsrc, *cand, *seen;
    uint8_t *inter;
    int4 *rec;
    int *pstep;
    int2 *emit;
    double *ox, *oy;
    int *osrc, *ring_off, *result;
    const int *done; // per job: its result is there already (sc_walk.hip), or null
    int uni;
    int par;
};

// sc_walk.hip: the route's steps over the whole device.  walk_jobs runs them
// on 'stream' for the jobs of at least WALK_MIN_NODES nodes and fills their
// result words and done flags (a job it leaves keeps done = 0 and is not
// written); walk_emit writes their rings to the batch's output.
struct WalkIn {
    SeqBatch b;
    const std::vector<SeqJob> *jobs; // host copy
    int nwalk;                       // jobs with a place among them
    const int64_t *nodeoff, *segoff; // 2 * nseq + 1 node / slot offsets (device)
    const uint32_t *nidx;            // node index by slot (exclusive scan of node starts)
    int64_t N;                       // nodes of all jobs
    const int *firstP, *firstQ;      // per batch job: first plain slot of each ring
};
// below, one block per job is as fast: on unions of 300 nodes 0.99 ms a clip against
// 0.98 device-wide, of 1,000 nodes 1.22 against 0.98 (the launches cost 0.15 ms)
constexpr int WALK_MIN_NODES = 512;
bool walk_jobs(const WalkIn &in, int *done, hipStream_t s); // false: no job is large enough, or no memory for them
void walk_emit(const WalkIn &in, const int *done, const uint32_t *JV, const uint32_t *JR, double *ox, double *oy,
               int *osrc, int *off, hipStream_t s);
void release_walk_scratch();

} // namespace sc
