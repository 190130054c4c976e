// sc_area.hip -- differentiable intersection area and IoU of a batch of jobs
// (row A19; the reference has no counterpart: it only writes the rings).
//
// Forward, per job: A_I = sum of the unsigned shoelace areas of the job's
// cleaned output rings, A_P / A_Q = unsigned shoelace areas of its base /
// overlay ring, IoU = A_I / (A_P + A_Q - A_I).  Twice the signed area of a
// ring is S = sum_i (x_i y_{i+1} - x_{i+1} y_i) and its area is |S| / 2: the
// input rings may run either way round, and with a clockwise input one job's
// output can hold rings of both orientations.  An intersection of two simple
// rings has no holes, so every output ring counts positively.  Each sum is
// reduced in a fixed order, so repeated runs give the same bits.
//
// Backward, with the combinatorics of the forward held fixed: an output
// vertex gets d|S|/dx_i = sgn(S) (y_{i+1} - y_{i-1}), d|S|/dy_i =
// sgn(S) (x_{i-1} - x_{i+1}) with S its ring's signed sum, routed by its
// provenance (the augmented slot it was emitted from):
//  - a source vertex of either ring, or an intersection located at an input
//    vertex (types 2-8: at b1 or c1 as the intersection stage places them),
//    passes the gradient to that input vertex;
//  - a proper crossing (type 1) X = (1-alpha) b1 + alpha b2 with
//    alpha = AP1 / (AP1 - AP2), AP1 = A(b1,c1,c2), AP2 = A(b2,c1,c2)
//    (lineSegmentIntersection2, oacc_segment_tree.cpp:5520-5611) passes it to
//    b1, b2 directly and through alpha to b1, b2, c1, c2.
// Contributions meet at input vertices: gathered there, or, where jobs share a
// base ring, through FP64 atomic adds.
#include "sc_ctx.hpp"
#include "sc_fp64.hpp"

#include <climits>

namespace sc {

namespace {

constexpr int BLK = 256;
constexpr int SRC_NONE = INT_MIN;

inline unsigned grid_for(int64_t n, int per = BLK) {
    int64_t g = ceil_div(n, per);
    if (g < 1) g = 1;
    return unsigned(g);
}

__device__ inline double block_sum(double v, double *sh) {
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int d = BLK / 2; d > 0; d >>= 1) {
        if (int(threadIdx.x) < d) sh[threadIdx.x] += sh[threadIdx.x + d];
        __syncthreads();
    }
    return sh[0];
}

// Twice the signed area of the input rings of both sides (blockIdx.z; vertices
// voff[r] .. voff[r+1]-1, the last one the repeated closing vertex), a block per
// RING_CHUNK vertices: one block per ring left 256 rings of 10,000 to 200,000
// vertices to as many blocks (0.25 ms for 32 million vertices, now 0.09).
// Chunk q of ring r is part[voff[r] / RING_CHUNK + r + q]: no two rings meet.
constexpr int64_t RING_CHUNK = 4096;
struct RingSide {
    int rings, r0;
    const double *poly;
    const int *voff;
    double *part, *out;
};
struct RingSides {
    RingSide s[2];
};
__global__ __launch_bounds__(BLK) void k_ring_area2(RingSides sides) {
    __shared__ double sh[BLK];
    const RingSide &z = sides.s[blockIdx.z];
    if (int(blockIdx.y) >= z.rings) return;
    const int r = z.r0 + blockIdx.y;
    const int64_t a = z.voff[r], n = z.voff[r + 1] - a - 1;
    for (int64_t q = blockIdx.x; q == 0 || q * RING_CHUNK < n; q += gridDim.x) {
        const int64_t end = n < (q + 1) * RING_CHUNK ? n : (q + 1) * RING_CHUNK;
        // thread t adds the terms of vertices t, t + BLK, ... in that order; four
        // terms are loaded before they are added (the same order and bits)
        double s = 0.0;
        int64_t i = q * RING_CHUNK + threadIdx.x;
        for (; i + 3 * BLK < end; i += 4 * BLK) {
            const double *p0 = z.poly + 2 * (a + i), *p1 = p0 + 2 * BLK, *p2 = p1 + 2 * BLK, *p3 = p2 + 2 * BLK;
            const double t0 = p0[0] * p0[3] - p0[2] * p0[1], t1 = p1[0] * p1[3] - p1[2] * p1[1];
            const double t2 = p2[0] * p2[3] - p2[2] * p2[1], t3 = p3[0] * p3[3] - p3[2] * p3[1];
            s += t0;
            s += t1;
            s += t2;
            s += t3;
        }
        for (; i < end; i += BLK) {
            const double *p = z.poly + 2 * (a + i);
            s += p[0] * p[3] - p[2] * p[1];
        }
        const double t = block_sum(s, sh);
        if (threadIdx.x == 0) (n <= RING_CHUNK ? z.out[blockIdx.y] : z.part[a / RING_CHUNK + r + q]) = t;
        __syncthreads(); // sh is written again
    }
}
// The same for rings of at most RING_WAVE vertices, a wave each: lane l holds the
// sums of the block's threads l, l + 64, l + 128 and l + 192 and adds them in the
// block's order (16,384 pairs of 4 to 64 vertices: 28 us with a block per ring,
// 10 so).
constexpr int RING_WAVE = BLK;
__device__ inline double wave_block_sum(double (&s)[BLK / WAVE]) {
    static_assert(BLK == 4 * WAVE, "the block sum's tree: 128, 64, then 32 to 1");
    s[0] += s[2];
    s[1] += s[3];
    s[0] += s[1];
    for (int d = WAVE / 2; d > 0; d >>= 1) s[0] += __shfl_down(s[0], d, WAVE);
    return s[0]; // lane 0
}
__global__ __launch_bounds__(BLK) void k_ring_area2_few(RingSides sides) {
    const RingSide &z = sides.s[blockIdx.y];
    const int k = int(blockIdx.x) * (BLK / WAVE) + int(threadIdx.x) / WAVE, lane = threadIdx.x & (WAVE - 1);
    if (k >= z.rings) return;
    const int r = z.r0 + k;
    const int64_t a = z.voff[r], n = z.voff[r + 1] - a - 1;
    double s[BLK / WAVE];
    for (int q = 0; q < BLK / WAVE; ++q) {
        const int64_t i = q * WAVE + lane;
        s[q] = 0.0;
        if (i < n) {
            const double *p = z.poly + 2 * (a + i);
            s[q] += p[0] * p[3] - p[2] * p[1];
        }
    }
    const double t = wave_block_sum(s);
    if (lane == 0) z.out[k] = t;
}
// rings of more than one chunk: its chunks in order
__global__ void k_ring_parts(RingSides sides) {
    const RingSide &z = sides.s[blockIdx.y];
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= z.rings) return;
    const int r = z.r0 + k;
    const int64_t a = z.voff[r], n = z.voff[r + 1] - a - 1;
    if (n <= RING_CHUNK) return;
    const double *p = z.part + (a / RING_CHUNK + r);
    double s = p[0];
    for (int64_t q = 1; q * RING_CHUNK < n; ++q) s += p[q];
    z.out[k] = s;
}

// Twice the signed area of every output ring.  A ring of at most AREA_CHUNK
// vertices is summed by one wave: lanes stride the ring and a fixed shuffle
// tree adds their sums (the order of the small-pair kernel).  Four rings of at
// most 16 vertices share the wave: the tree's steps over 32 and 16 lanes would
// add zeros to such a ring, and most are this short (the output rings of 256
// large pairs: 0.19 -> 0.06 ms).
// A longer ring is summed in chunks of AREA_CHUNK vertices, one wave per
// chunk, and its chunk sums are added in chunk order.
constexpr int AREA_CHUNK = LONG_RING;
constexpr int AREA_WAVES = 8192; // waves of the short-ring grid (32 per CU)
constexpr int RING_LANES = 16, RING_SET = WAVE / RING_LANES; // lanes of a short ring, rings a wave takes at once

__device__ inline double wave_ring_sum(const double *__restrict__ x, const double *__restrict__ y, int64_t a,
                                       int64_t b, int64_t c0, int64_t c1, int lane) {
    // eight terms are loaded before they are added (the same order and bits): a
    // wave alone on a long ring does little but wait for its loads
    constexpr int AHEAD = 8;
    double s = 0.0;
    int64_t i = c0 + lane;
    for (; i + (AHEAD - 1) * WAVE < c1 && i + (AHEAD - 1) * WAVE + 1 < b; i += AHEAD * WAVE) {
        double t[AHEAD];
#pragma unroll
        for (int q = 0; q < AHEAD; ++q) {
            const int64_t k = i + q * WAVE;
            t[q] = x[k] * y[k + 1] - x[k + 1] * y[k];
        }
#pragma unroll
        for (int q = 0; q < AHEAD; ++q) s += t[q];
    }
    for (; i < c1; i += WAVE) {
        const int64_t nx = i + 1 == b ? a : i + 1;
        s += x[i] * y[nx] - x[nx] * y[i];
    }
    for (int d = WAVE / 2; d > 0; d >>= 1) s += __shfl_down(s, d, WAVE);
    return s;
}

// set: the rings that a wave takes at once, RING_SET or, where there are waves
// for all, one: a set's longer rings are summed one after the other (300 pairs
// of 50 to 3,000 vertices: 31 -> 15 us with eight loads ahead instead of four,
// 31 pairs of 1,000 to 20,000: 39 -> 21).
__global__ __launch_bounds__(BLK) void k_out_ring_area2(int nrings, int set, const int *__restrict__ roff,
                                                        const double *__restrict__ x, const double *__restrict__ y,
                                                        double *out) {
    const int lane = int(threadIdx.x) & (WAVE - 1), l = lane & (RING_LANES - 1), q = lane / RING_LANES;
    const int stride = int(gridDim.x) * (BLK / WAVE) * set;
    for (int r0 = (int(blockIdx.x) * (BLK / WAVE) + int(threadIdx.x) / WAVE) * set; r0 < nrings; r0 += stride) {
        const int r = q < set ? r0 + q : nrings;
        const int64_t a = r < nrings ? roff[r] : 0, b = r < nrings ? roff[r + 1] : 0;
        double s = 0.0;
        if (b - a <= RING_LANES && a + l < b) {
            const int64_t i = a + l, nx = i + 1 == b ? a : i + 1;
            s += x[i] * y[nx] - x[nx] * y[i];
        }
        for (int d = RING_LANES / 2; d > 0; d >>= 1) s += __shfl_down(s, d, RING_LANES);
        if (l == 0 && r < nrings && b - a <= RING_LANES) out[r] = s;
        for (uint64_t m = __ballot(l == 0 && b - a > RING_LANES && b - a <= AREA_CHUNK); m; m &= m - 1) {
            const int from = __ffsll((unsigned long long)m) - 1;
            const int64_t ra = __shfl(int(a), from, WAVE), rb = __shfl(int(b), from, WAVE);
            const double t = wave_ring_sum(x, y, ra, rb, ra, rb, lane);
            if (lane == 0) out[r0 + from / RING_LANES] = t;
        }
    }
}

// chunks of each long ring (0 for a ring of at most AREA_CHUNK vertices;
// cnt[nrings] = 0 closes the scan)
__global__ void k_ring_chunks(int nrings, const int *__restrict__ roff, uint32_t *cnt) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r > nrings) return;
    if (r == nrings) {
        cnt[r] = 0u;
        return;
    }
    const int64_t len = roff[r + 1] - roff[r];
    cnt[r] = len <= AREA_CHUNK ? 0u : uint32_t((len + AREA_CHUNK - 1) / AREA_CHUNK);
}

// chunk q of the *total (choff: exclusive scan of the chunk counts)
__global__ __launch_bounds__(BLK) void k_out_chunk_area2(int nrings, const int *__restrict__ roff,
                                                         const uint32_t *__restrict__ choff,
                                                         const uint32_t *__restrict__ total, int64_t cap,
                                                         const double *__restrict__ x, const double *__restrict__ y,
                                                         double *part) {
    const int64_t q = int64_t(blockIdx.x) * (BLK / WAVE) + int64_t(threadIdx.x) / WAVE;
    const int lane = int(threadIdx.x) & (WAVE - 1);
    if (q >= int64_t(*total) || q >= cap) return; // whole wave
    int lo = 0, hi = nrings - 1; // the ring: the first r with choff[r + 1] > q
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (int64_t(choff[mid + 1]) > q) hi = mid;
        else lo = mid + 1;
    }
    const int64_t a = roff[lo], b = roff[lo + 1];
    const int64_t c0 = a + (q - int64_t(choff[lo])) * AREA_CHUNK;
    const int64_t c1 = c0 + AREA_CHUNK < b ? c0 + AREA_CHUNK : b;
    const double s = wave_ring_sum(x, y, a, b, c0, c1, lane);
    if (lane == 0) part[q] = s;
}

__global__ void k_ring_chunk_sum(int nrings, const uint32_t *__restrict__ choff, int64_t cap,
                                 const double *__restrict__ part, double *out) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= nrings) return;
    const int64_t k0 = choff[r], k1 = int64_t(choff[r + 1]) < cap ? int64_t(choff[r + 1]) : cap;
    if (k0 >= k1) return; // a short ring
    double s = part[k0];
    for (int64_t k = k0 + 1; k < k1; ++k) s += part[k];
    out[r] = s;
}

// The areas and IoU of each job, a block per job: thread t adds |S| of rings t,
// t + 256, ... (four loaded ahead), then a fixed tree.  Where jobs are many they
// have a ring or two each and a wave per job adds in the same order (EACH;
// 16,384 jobs: 14 us with a block per job, 6 so).
constexpr int JOBS_EACH = 2048;
template <bool EACH>
__global__ __launch_bounds__(BLK) void k_job_areas(int J, int paired, const int *__restrict__ jring,
                                                   const double *__restrict__ ring2,
                                                   const double *__restrict__ barea2,
                                                   const double *__restrict__ carea2, double *out4) {
    __shared__ double sh[EACH ? 1 : BLK];
    const int lane = threadIdx.x & (WAVE - 1);
    const int j = EACH ? int(blockIdx.x) * (BLK / WAVE) + int(threadIdx.x) / WAVE : int(blockIdx.x);
    if (EACH && j >= J) return; // whole wave
    const int r0 = jring[j], r1 = jring[j + 1];
    double t;
    if (EACH) {
        double s[BLK / WAVE] = {};
        for (int r = r0; r < r1; r += BLK)
            for (int q = 0; q < BLK / WAVE; ++q) {
                const int k = r + q * WAVE + lane;
                if (k < r1) s[q] += fabs(ring2[k]);
            }
        t = wave_block_sum(s);
        if (lane != 0) return;
    } else {
        double s = 0.0;
        int r = r0 + int(threadIdx.x);
        for (; r + 3 * BLK < r1; r += 4 * BLK) {
            const double v0 = ring2[r], v1 = ring2[r + BLK], v2 = ring2[r + 2 * BLK], v3 = ring2[r + 3 * BLK];
            s += fabs(v0);
            s += fabs(v1);
            s += fabs(v2);
            s += fabs(v3);
        }
        for (; r < r1; r += BLK) s += fabs(ring2[r]);
        t = block_sum(s, sh);
        if (threadIdx.x != 0) return;
    }
    const double I = 0.5 * t, P = 0.5 * fabs(barea2[paired ? j : 0]), Q = 0.5 * fabs(carea2[j]);
    const double U = P + Q - I;
    out4[j] = I;
    out4[J + j] = P;
    out4[2 * J + j] = Q;
    out4[3 * J + j] = U != 0.0 ? I / U : 0.0;
}

__device__ inline double sgn1(double v) { return v < 0.0 ? -1.0 : 1.0; }

// per job: coefficients of d(2A_I) (per output ring, times its orientation
// sign in k_output_grad), d(S_P) and d(S_Q) in the loss, S the signed sums
__global__ void k_coef(int J, int paired, const double *out4, const double *barea2, const double *carea2,
                       const double *g_area, const double *g_iou, double *cI, double *cQ, double *cPr) {
    int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= J) return;
    double I = out4[j], P = out4[J + j], Q = out4[2 * J + j];
    double U = P + Q - I;
    double ga = g_area ? g_area[j] : 0.0, gi = g_iou ? g_iou[j] : 0.0;
    double dI = ga, dP = 0.0;
    if (U != 0.0) {
        dI += gi * (U + I) / (U * U);
        dP = -gi * I / (U * U);
    }
    cI[j] = 0.5 * dI;
    cQ[j] = 0.5 * dP * sgn1(carea2[j]);
    // the base ring may be shared by every job (one-to-many)
    unsafeAtomicAdd(&cPr[paired ? j : 0], 0.5 * dP * sgn1(barea2[paired ? j : 0]));
}

// d(2A)/d(vertex) of the input rings: base rings (all of them, coefficient per
// ring) or overlays (coefficient per overlay, zero outside the batch); input
// vertex i of ring r sits at i + r in the layout with closing vertices.
// Plain stores: this is the first writer of the gradient arrays.
__global__ void k_input_ring_grad(int64_t n, const int *__restrict__ off, int R, const double *__restrict__ poly,
                                  const double *__restrict__ coef, double *grad) {
    int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int r = seg_of(off, R, i);
    const int64_t v = i - off[r], m = off[r + 1] - off[r];
    const double *P = poly + 2 * (int64_t(off[r]) + r);
    const int64_t nx = v + 1 == m ? 0 : v + 1, pv = v == 0 ? m - 1 : v - 1;
    const double c = coef[r];
    grad[2 * i] = c * (P[2 * nx + 1] - P[2 * pv + 1]);
    grad[2 * i + 1] = c * (P[2 * pv] - P[2 * nx]);
}

struct ProvArgs {
    int J, nrings;
    const int *jring, *roff, *src;
    const uint32_t *rid; // output ring of every output vertex
    const double *ox, *oy;
    const double *cI;
    const double *ring2; // signed 2A of every output ring
    const int *from_b, *from_c;
    const int *p_b, *p_c, *p_type;
    const int *bvoff, *beoff, *nb, *cvoff, *cin, *nc; // per job
    const double *bpoly, *cpoly;
    double *grad_b, *grad_c;
    int *bad;
};

__device__ inline void add_b(const ProvArgs &a, int j, int v, double gx, double gy) {
    int64_t i = int64_t(a.beoff[j]) + v;
    unsafeAtomicAdd(&a.grad_b[2 * i], gx);
    unsafeAtomicAdd(&a.grad_b[2 * i + 1], gy);
}
__device__ inline void add_c(const ProvArgs &a, int j, int v, double gx, double gy) {
    int64_t i = int64_t(a.cin[j]) + v;
    unsafeAtomicAdd(&a.grad_c[2 * i], gx);
    unsafeAtomicAdd(&a.grad_c[2 * i + 1], gy);
}

// gradient (gx, gy) on the crossing X of the edges B = b1 b2 and C = c1 c2:
// what b1, b2 (gb) and c1, c2 (gc) get of it
__device__ inline void crossing_grad(const double *__restrict__ B, const double *__restrict__ C, double gx, double gy,
                                     double *gb, double *gc) {
    const double b1x = B[0], b1y = B[1], b2x = B[2], b2y = B[3];
    const double c1x = C[0], c1y = C[1], c2x = C[2], c2y = C[3];
    const double AP1 = areaA(b1x, b1y, c1x, c1y, c2x, c2y);
    const double AP2 = areaA(b2x, b2y, c1x, c1y, c2x, c2y);
    const double D = AP1 - AP2;
    const double al = AP1 / D;
    // X = (1-al) b1 + al b2
    const double gal = gx * (b2x - b1x) + gy * (b2y - b1y);
    double gb1x = (1.0 - al) * gx, gb1y = (1.0 - al) * gy, gb2x = al * gx, gb2y = al * gy;
    // al = AP1 / (AP1 - AP2)
    const double g1 = -gal * AP2 / (D * D), g2 = gal * AP1 / (D * D);
    // A(p,q,r): d/dp = (qy-ry, rx-qx), d/dq = (ry-py, px-rx), d/dr = (py-qy, qx-px)
    gb1x += g1 * (c1y - c2y);
    gb1y += g1 * (c2x - c1x);
    gb2x += g2 * (c1y - c2y);
    gb2y += g2 * (c2x - c1x);
    gc[0] = g1 * (c2y - b1y) + g2 * (c2y - b2y);
    gc[1] = g1 * (b1x - c2x) + g2 * (b2x - c2x);
    gc[2] = g1 * (b1y - c1y) + g2 * (b2y - c1y);
    gc[3] = g1 * (c1x - b1x) + g2 * (c1x - b2x);
    gb[0] = gb1x;
    gb[1] = gb1y;
    gb[2] = gb2x;
    gb[3] = gb2y;
}

// gradient (gx, gy) on the point of pair p, seen from side P (onP) or Q
__device__ void pair_grad(const ProvArgs &a, int j, int p, bool onP, double gx, double gy) {
    const int t = a.p_type[p], b = a.p_b[p], c = a.p_c[p];
    if (t != 1) {
        // types 3,5,7 sit at c1 (base side), 2,6 at b1 (overlay side)
        if (onP) add_c(a, j, c, gx, gy);
        else add_b(a, j, b, gx, gy);
        return;
    }
    const int nb = a.nb[j], nc = a.nc[j];
    double gb[4], gc[4];
    crossing_grad(a.bpoly + 2 * (int64_t(a.bvoff[j]) + b), a.cpoly + 2 * (int64_t(a.cvoff[j]) + c), gx, gy, gb, gc);
    add_b(a, j, b, gb[0], gb[1]);
    add_b(a, j, b + 1 == nb ? 0 : b + 1, gb[2], gb[3]);
    add_c(a, j, c, gc[0], gc[1]);
    add_c(a, j, c + 1 == nc ? 0 : c + 1, gc[2], gc[3]);
}

// ring heads for the output ring index (rid zero-filled, then max-scanned)
__global__ void k_out_ring_heads(int nrings, const int *__restrict__ roff, uint32_t *rid) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= nrings) return;
    if (roff[r + 1] > roff[r]) rid[roff[r]] = uint32_t(r);
}

__global__ void k_output_grad(ProvArgs a, int64_t v0, int64_t v1) {
    int64_t i = v0 + int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= v1) return;
    const int r = int(a.rid[i]);
    const int j = seg_of(a.jring, a.J, r);
    const int64_t rb = a.roff[r], re = a.roff[r + 1];
    const int64_t nx = i + 1 == re ? rb : i + 1, pv = i == rb ? re - 1 : i - 1;
    const double c = a.cI[j] * sgn1(a.ring2[r]);
    const double gx = c * (a.oy[nx] - a.oy[pv]), gy = c * (a.ox[pv] - a.ox[nx]);
    const int s = a.src[i];
    if (s == SRC_NONE) {
        atomicOr(a.bad, 1);
        return;
    }
    if (s >= 0) {
        const int v = a.from_b[s];
        if (v >= 0) add_b(a, j, v, gx, gy);
        else pair_grad(a, j, ~v, true, gx, gy);
    } else {
        const int v = a.from_c[~s];
        if (v >= 0) add_c(a, j, v, gx, gy);
        else pair_grad(a, j, ~v, false, gx, gy);
    }
}

// ---- gradients without an atomic per contribution ----
// Where every input ring belongs to one job, an output vertex leaves its
// gradient and, at the input vertex or the pair it came from, its index.  An
// input vertex stores its ring's term and its output vertex's; a pair turns
// what its two visits left into shares of its edges' ends, which a wave sums
// over the pairs of one edge before it adds them.  FP64 atomics pass the caches
// of the eight dies: 256 pairs with 32 million input vertices spent 1.86 ms in
// them and 0.39 in the rings' terms; these kernels take 0.88.  Jobs that
// share a base ring keep an atomic per contribution (k_output_grad).
struct GatherGrad {
    ProvArgs a;
    int I;
    int64_t n_out;
    const int *jv0;      // J + 1: first output vertex of each job
    double2 *og;         // per output vertex
    int *inv_b, *inv_c;  // per input vertex: its output vertex, -1 for none
    int *inv_p, *inv_q;  // per pair: the output vertex of its base / overlay visit
    double4 *rec;        // per pair: shares of c1 and c2
    const int *ord_c, *pj;
    uint32_t *found;     // output vertices found from the other side, per block of the kernels that look
    int nfound;
};

// first output vertex of each job (J + 1 threads)
__global__ void k_job_first_out(int J, const int *__restrict__ jring, const int *__restrict__ roff, int *jv0) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j <= J) jv0[j] = roff[jring[j]];
}

__global__ __launch_bounds__(BLK) void k_output_terms(GatherGrad g, int per) {
    const ProvArgs &a = g.a;
    const int lane = threadIdx.x & (WAVE - 1);
    WaveSpan w(g.jv0, a.J, g.n_out, per);
    for (int q = 0; q < per && w.at < g.n_out; ++q, w.at += WAVE) {
        const int64_t i = w.at + lane;
        const int j = w.of(g.jv0, a.J, lane);
        if (i >= g.n_out) continue;
        const int r = int(a.rid[i]);
        const int64_t rb = a.roff[r], re = a.roff[r + 1];
        const int64_t nx = i + 1 == re ? rb : i + 1, pv = i == rb ? re - 1 : i - 1;
        const double c = a.cI[j] * sgn1(a.ring2[r]);
        g.og[i] = make_double2(c * (a.oy[nx] - a.oy[pv]), c * (a.ox[pv] - a.ox[nx]));
        const int s = a.src[i];
        if (s == SRC_NONE) {
            atomicOr(a.bad, 1);
            continue;
        }
        const int v = s >= 0 ? a.from_b[s] : a.from_c[~s];
        if (v >= 0) (s >= 0 ? g.inv_b + a.beoff[j] : g.inv_c + a.cin[j])[v] = int(i);
        else (s >= 0 ? g.inv_p : g.inv_q)[~v] = int(i);
    }
}

// a block's count at its place in the list (an atomic per wave on one word took
// longer than the kernels' own work)
__device__ inline void put_count(uint32_t *at, uint32_t n) { // all threads
    __shared__ uint32_t part[BLK / WAVE];
    for (int d = WAVE / 2; d > 0; d >>= 1) n += uint32_t(__shfl_xor(int(n), d, WAVE));
    if ((threadIdx.x & (WAVE - 1)) == 0) part[threadIdx.x / WAVE] = n;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t t = 0;
        for (int q = 0; q < BLK / WAVE; ++q) t += part[q];
        *at = t;
    }
}

// Sums g over each run of lanes with the same key (n lanes hold one) and gives
// the run's last lane the sum; whether this lane is one.
__device__ inline bool run_sums(int64_t key, bool have, double (&g)[4]) {
    const int lane = threadIdx.x & (WAVE - 1);
    const int64_t k = have ? key : -1 - lane;
    const int lo = int(uint32_t(uint64_t(k))), hi = int(uint32_t(uint64_t(k) >> 32));
    const bool head = lane == 0 || __shfl_up(lo, 1, WAVE) != lo || __shfl_up(hi, 1, WAVE) != hi;
    const uint64_t heads = __ballot(head);
    const uint64_t upto = ~0ull >> (WAVE - 1 - lane);
    const int first = 63 - __clzll((long long)(heads & upto)); // this lane's run
    for (int d = 1; d < WAVE && __ballot(lane - first >= d); d <<= 1)
        for (int q = 0; q < 4; ++q) {
            const double y = __shfl_up(g[q], d, WAVE);
            if (lane - first >= d) g[q] += y;
        }
    return have && (lane == WAVE - 1 || ((heads >> (lane + 1)) & 1u));
}

// pairs in (job, base edge) order: the base side's shares
__global__ __launch_bounds__(BLK) void k_pair_terms(GatherGrad g) {
    const ProvArgs &a = g.a;
    uint32_t found = 0;
    const int64_t step = int64_t(gridDim.x) * blockDim.x;
    for (int64_t p0 = int64_t(blockIdx.x) * blockDim.x; p0 < g.I; p0 += step) {
        const int64_t p = p0 + threadIdx.x;
        double gb[4] = {}, gc[4] = {};
        int j = 0, b = 0;
        if (p < g.I) {
            const int ip = g.inv_p[p], iq = g.inv_q[p], c = a.p_c[p];
            j = g.pj[p];
            b = a.p_b[p];
            if (ip >= 0 || iq >= 0) {
                const double2 gp = ip >= 0 ? g.og[ip] : make_double2(0.0, 0.0);
                const double2 gq = iq >= 0 ? g.og[iq] : make_double2(0.0, 0.0);
                found += (ip >= 0 ? 1u : 0u) + (iq >= 0 ? 1u : 0u);
                if (a.p_type[p] == 1) {
                    crossing_grad(a.bpoly + 2 * (int64_t(a.bvoff[j]) + b), a.cpoly + 2 * (int64_t(a.cvoff[j]) + c),
                                  gp.x + gq.x, gp.y + gq.y, gb, gc);
                } else { // types 3,5,7 sit at c1 (base side), 2,6 at b1 (overlay side)
                    gb[0] = gq.x;
                    gb[1] = gq.y;
                    gc[0] = gp.x;
                    gc[1] = gp.y;
                }
            }
            g.rec[p] = make_double4(gc[0], gc[1], gc[2], gc[3]);
        }
        if (run_sums(int64_t(a.beoff[j]) + b, p < g.I, gb)) {
            if (gb[0] != 0.0 || gb[1] != 0.0) add_b(a, j, b, gb[0], gb[1]);
            if (gb[2] != 0.0 || gb[3] != 0.0) add_b(a, j, b + 1 == a.nb[j] ? 0 : b + 1, gb[2], gb[3]);
        }
    }
    put_count(g.found + blockIdx.x, found);
}

// pairs in (job, overlay edge) order: the overlay side's
__global__ __launch_bounds__(BLK) void k_pair_terms_c(GatherGrad g) {
    const ProvArgs &a = g.a;
    const int64_t k = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    double gc[4] = {};
    int j = 0, c = 0;
    if (k < g.I) {
        const int p = g.ord_c[k];
        j = g.pj[p];
        c = a.p_c[p];
        const double4 t = g.rec[p];
        gc[0] = t.x;
        gc[1] = t.y;
        gc[2] = t.z;
        gc[3] = t.w;
    }
    if (run_sums(int64_t(a.cin[j]) + c, k < g.I, gc)) {
        if (gc[0] != 0.0 || gc[1] != 0.0) add_c(a, j, c, gc[0], gc[1]);
        if (gc[2] != 0.0 || gc[3] != 0.0) add_c(a, j, c + 1 == a.nc[j] ? 0 : c + 1, gc[2], gc[3]);
    }
}

struct VertexSide {
    int64_t n;
    const int *off; // input vertex offsets of the rings
    int R;
    const double *poly, *coef;
    const int *inv;
    double *grad;
};
struct VertexSides {
    VertexSide s[2];
    const double2 *og;
    int per;
    uint32_t *found;
};
// input vertex i of ring r sits at i + r in the layout with closing vertices
__global__ __launch_bounds__(BLK) void k_vertex_grad(VertexSides a) {
    const VertexSide &z = a.s[blockIdx.y];
    const int lane = threadIdx.x & (WAVE - 1);
    uint32_t found = 0;
    WaveSpan w(z.off, z.R, z.n, a.per);
    for (int q = 0; q < a.per && w.at < z.n; ++q, w.at += WAVE) {
        const int64_t i = w.at + lane;
        const int r = w.of(z.off, z.R, lane);
        if (i >= z.n) continue;
        const int64_t v = i - z.off[r], m = z.off[r + 1] - z.off[r];
        const double *P = z.poly + 2 * (int64_t(z.off[r]) + r);
        const int64_t nx = v + 1 == m ? 0 : v + 1, pv = v == 0 ? m - 1 : v - 1;
        const double c = z.coef[r];
        double gx = c * (P[2 * nx + 1] - P[2 * pv + 1]), gy = c * (P[2 * pv] - P[2 * nx]);
        const int o = z.inv[i];
        if (o >= 0) {
            const double2 t = a.og[o];
            gx += t.x;
            gy += t.y;
            ++found;
        }
        z.grad[2 * i] = gx;
        z.grad[2 * i + 1] = gy;
    }
    put_count(a.found + blockIdx.y * gridDim.x + blockIdx.x, found);
}

// Output vertices that share their input vertex or visit with another one, of
// which only the last was found; returns at once where there is none.
__global__ __launch_bounds__(BLK) void k_grad_rest(GatherGrad g) {
    const ProvArgs &a = g.a;
    __shared__ uint32_t total;
    if (threadIdx.x == 0) total = 0;
    __syncthreads();
    uint32_t n = 0;
    for (int k = threadIdx.x; k < g.nfound; k += BLK) n += g.found[k];
    for (int d = WAVE / 2; d > 0; d >>= 1) n += uint32_t(__shfl_xor(int(n), d, WAVE));
    if ((threadIdx.x & (WAVE - 1)) == 0) atomicAdd(&total, n);
    __syncthreads();
    if (int64_t(total) == g.n_out) return;
    const int64_t step = int64_t(gridDim.x) * blockDim.x;
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < g.n_out; i += step) {
        const int s = a.src[i];
        if (s == SRC_NONE) continue;
        const int j = seg_of(g.jv0, a.J, i);
        const int v = s >= 0 ? a.from_b[s] : a.from_c[~s];
        const double2 t = g.og[i];
        if (v >= 0) {
            if ((s >= 0 ? g.inv_b + a.beoff[j] : g.inv_c + a.cin[j])[v] == int(i)) continue;
            if (s >= 0) add_b(a, j, v, t.x, t.y);
            else add_c(a, j, v, t.x, t.y);
        } else if ((s >= 0 ? g.inv_p : g.inv_q)[~v] != int(i)) {
            pair_grad(a, j, ~v, s >= 0, t.x, t.y);
        }
    }
}

struct AreaScratch {
    DBuf<double> ring2, barea2, carea2, out4, cI, cQ, cPr, part, rpart;
    DBuf<int> bad, bin_off;
    DBuf<uint32_t> chunks, choff, tot, rid, gfound;
    // gathered gradients
    DBuf<int> jv0, inv;
    DBuf<double2> og;
    DBuf<double4> rec;
};

AreaScratch &ascratch(Ctx &) {
    thread_local AreaScratch *p = new AreaScratch();
    return *p;
}

} // namespace

void batch_area(Ctx &c, double *out4) {
    SC_REQUIRE(!c.uni, SC_ESTATE, "area / IoU are defined for the intersection (a union output may hold holes)");
    JobSet &js = c.jobs;
    SC_REQUIRE(js.J >= 1 && int(js.ring_off.size()) == js.J + 1, SC_ESTATE, "no clipped batch");
    SC_REQUIRE(js.resident, SC_ESTATE, "the batch was clipped from other rings");
    hipStream_t s = c.stream;
    AreaScratch &a = ascratch(c);
    const int J = js.J;
    double *barea2 = a.barea2.ensure(c.nbr), *carea2 = a.carea2.ensure(J);
    double *ring2 = a.ring2.ensure(size_t(c.nrings > 0 ? c.nrings : 1));
    if (c.nrings > 0) {
        const int nr = c.nrings;
        const int set = nr <= AREA_WAVES ? 1 : RING_SET;
        const int64_t wgrid = std::min<int64_t>(ceil_div(int64_t(nr), set * (BLK / WAVE)), AREA_WAVES / (BLK / WAVE));
        k_out_ring_area2<<<unsigned(wgrid), BLK, 0, s>>>(nr, set, c.d_ring_off, c.d_ring_x, c.d_ring_y, ring2);
        if (c.long_rings) {
            uint32_t *cnt = a.chunks.ensure(size_t(nr) + 1), *choff = a.choff.ensure(size_t(nr) + 1);
            uint32_t *tot = a.tot.ensure(1);
            // a long ring has at most one chunk more than its AREA_CHUNK-vertex
            // multiples, and there are at most n_out / AREA_CHUNK long rings
            const int64_t cap = 2 * (c.n_out / AREA_CHUNK) + 1;
            double *part = a.part.ensure(size_t(cap));
            k_ring_chunks<<<grid_for(int64_t(nr) + 1), BLK, 0, s>>>(nr, c.d_ring_off, cnt);
            scan_exclusive_u32(cnt, choff, int64_t(nr) + 1, tot, s);
            k_out_chunk_area2<<<grid_for(cap, BLK / WAVE), BLK, 0, s>>>(nr, c.d_ring_off, choff, tot, cap,
                                                                        c.d_ring_x, c.d_ring_y, part);
            k_ring_chunk_sum<<<grid_for(nr), BLK, 0, s>>>(nr, choff, cap, part, ring2);
        }
    }
    RingSides rs;
    const int64_t pb = (c.nb + c.nbr) / RING_CHUNK + c.nbr + 1, pc = (c.nct + c.K) / RING_CHUNK + c.K + 1;
    double *part = a.rpart.ensure(size_t(pb + pc));
    rs.s[0] = RingSide{c.paired ? J : 1, c.paired ? js.k0 - 1 : 0, c.bpoly, c.d_bvoff, part, barea2};
    rs.s[1] = RingSide{J, js.k0 - 1, c.cpoly, c.d_coff, part + pb, carea2};
    // blocks for a ring's chunks, where there are not many rings anyway
    const int64_t longest = ceil_div(int64_t(std::max(c.maxbsz, c.maxcsz)), RING_CHUNK);
    const int64_t bx = std::max<int64_t>(1, std::min<int64_t>(longest, 32768 / J));
    const bool few = std::max(c.maxbsz, c.maxcsz) <= RING_WAVE; // a wave's worth of vertices per ring
    if (few) k_ring_area2_few<<<dim3(grid_for(J, BLK / WAVE), 2), BLK, 0, s>>>(rs);
    for (int r = 0; r < J && !few; r += 65535) { // grid dimension limit
        RingSides part_of = rs;
        for (RingSide &z : part_of.s) {
            z.rings = std::max(0, std::min(65535, z.rings - r));
            z.r0 += r;
            z.out += r;
        }
        k_ring_area2<<<dim3(unsigned(bx), unsigned(std::min(65535, J - r)), 2), BLK, 0, s>>>(part_of);
    }
    if (longest > 1) k_ring_parts<<<dim3(grid_for(J), 2), BLK, 0, s>>>(rs);
    const int paired = c.paired ? 1 : 0;
    if (J >= JOBS_EACH)
        k_job_areas<true><<<grid_for(J, BLK / WAVE), BLK, 0, s>>>(J, paired, js.d_ring, ring2, barea2, carea2, out4);
    else k_job_areas<false><<<J, BLK, 0, s>>>(J, paired, js.d_ring, ring2, barea2, carea2, out4);
    SC_HIP(hipGetLastError());
}

void batch_area_backward(Ctx &c, const double *g_area, const double *g_iou, double *grad_b, double *grad_c) {
    JobSet &js = c.jobs;
    SC_REQUIRE(c.prov && js.prov, SC_ESTATE, "the batch was clipped without provenance (segclip_set_provenance)");
    hipStream_t s = c.stream;
    AreaScratch &a = ascratch(c);
    const int J = js.J;
    double *out4 = a.out4.ensure(4 * size_t(J));
    batch_area(c, out4);
    double *cI = a.cI.ensure(J), *cQ = a.cQ.ensure(c.K), *cPr = a.cPr.ensure(c.nbr);
    SC_HIP(hipMemsetAsync(cPr, 0, sizeof(double) * c.nbr, s));
    SC_HIP(hipMemsetAsync(cQ, 0, sizeof(double) * c.K, s));
    // k_coef writes cQ for the batch's jobs at their overlay index
    k_coef<<<grid_for(J), BLK, 0, s>>>(J, c.paired ? 1 : 0, out4, a.barea2, a.carea2, g_area, g_iou, cI,
                                       cQ + (js.k0 - 1), c.paired ? cPr + (js.k0 - 1) : cPr);
    SC_HIP(hipGetLastError());
    // input ring terms: base rings (input offsets beoff), all overlays (input offsets eoff - nb)
    int *boff = c.d_beoff;
    const bool gather = c.paired || (J == 1 && c.K == 1); // every input ring in one job at most
    if (!gather) k_input_ring_grad<<<grid_for(c.nb), BLK, 0, s>>>(c.nb, boff, c.nbr, c.bpoly, cPr, grad_b);
    std::vector<int> cinall(size_t(c.K) + 1);
    for (int k = 0; k <= c.K; ++k) cinall[k] = c.eoff[k] - c.nb;
    int *dci = a.bin_off.ensure(c.K + 1);
    c.upload(dci, cinall.data(), sizeof(int) * (c.K + 1));
    if (!gather) k_input_ring_grad<<<grid_for(c.nct), BLK, 0, s>>>(c.nct, dci, c.K, c.cpoly, cQ, grad_c);
    SC_HIP(hipGetLastError());
    // output vertices of the batch
    ProvArgs p;
    p.J = J;
    p.nrings = c.nrings;
    p.jring = js.d_ring;
    p.roff = c.d_ring_off;
    p.src = c.d_ring_src;
    p.ox = c.d_ring_x;
    p.oy = c.d_ring_y;
    p.cI = cI;
    p.ring2 = a.ring2;
    p.from_b = c.from_b;
    p.from_c = c.from_c;
    p.p_b = c.p_b;
    p.p_c = c.p_c;
    p.p_type = c.p_type;
    p.bvoff = js.d_bvoff;
    p.beoff = js.d_beoff;
    p.nb = js.d_nb;
    p.cvoff = js.d_cvoff;
    p.cin = js.d_cin;
    p.nc = js.d_nc;
    p.bpoly = c.bpoly;
    p.cpoly = c.cpoly;
    p.grad_b = grad_b;
    p.grad_c = grad_c;
    p.bad = a.bad.ensure(1);
    SC_HIP(hipMemsetAsync(p.bad, 0, sizeof(int), s));
    const int I = gather ? js.p0[J] : 0;
    const bool outs = c.n_out > 0 && c.nrings > 0;
    GatherGrad g{};
    {
        FillBatch fb(s);
        if (outs) fb.add(a.rid.ensure(size_t(c.n_out)), c.n_out, 0u);
        if (gather) {
            const int64_t nv = int64_t(c.nb) + c.nct;
            int *inv = a.inv.ensure(size_t(nv + 2 * int64_t(I)));
            g.inv_b = inv;
            g.inv_c = inv + c.nb;
            g.inv_p = inv + nv;
            g.inv_q = inv + nv + I;
            fb.add(inv, nv + 2 * int64_t(I), ~0u);
        }
        fb.flush();
    }
    if (outs) {
        // the ring of every output vertex: ring heads, then a max-scan
        uint32_t *rid = a.rid;
        k_out_ring_heads<<<grid_for(c.nrings), BLK, 0, s>>>(c.nrings, c.d_ring_off, rid);
        scan_inclusive_max_u32(rid, rid, c.n_out, s);
        p.rid = rid;
        if (!gather) k_output_grad<<<grid_for(c.n_out), BLK, 0, s>>>(p, 0, c.n_out);
    }
    if (gather) {
        g.a = p;
        g.I = I;
        g.n_out = outs ? c.n_out : 0;
        g.jv0 = a.jv0.ensure(size_t(J) + 1);
        g.og = a.og.ensure(size_t(g.n_out > 0 ? g.n_out : 1));
        g.rec = a.rec.ensure(size_t(I) + 1);
        g.ord_c = c.ordC;
        g.pj = c.p_j;
        if (g.n_out > 0) {
            k_job_first_out<<<grid_for(int64_t(J) + 1), BLK, 0, s>>>(J, js.d_ring, c.d_ring_off, a.jv0);
            const int per = span_per(g.n_out);
            k_output_terms<<<grid_for(g.n_out, BLK * per), BLK, 0, s>>>(g, per);
        }
        const int blocks = 2048; // eight waves per SIMD
        VertexSides vs{};
        vs.s[0] = VertexSide{c.nb, boff, c.nbr, c.bpoly, cPr, g.inv_b, grad_b};
        vs.s[1] = VertexSide{c.nct, dci, c.K, c.cpoly, cQ, g.inv_c, grad_c};
        vs.og = g.og;
        const int64_t most = std::max<int64_t>(c.nb, c.nct);
        vs.per = int(std::max<int64_t>(1, ceil_div(most, int64_t(blocks) * BLK)));
        const int vblocks = int(grid_for(most, BLK * vs.per)), pblocks = I > 0 ? std::min(blocks, int(grid_for(I))) : 0;
        g.nfound = 2 * vblocks + pblocks;
        vs.found = a.gfound.ensure(size_t(g.nfound));
        k_vertex_grad<<<dim3(unsigned(vblocks), 2), BLK, 0, s>>>(vs);
        g.found = vs.found + 2 * vblocks;
        if (I > 0) {
            k_pair_terms<<<pblocks, BLK, 0, s>>>(g);
            k_pair_terms_c<<<grid_for(I), BLK, 0, s>>>(g);
        }
        g.found = vs.found;
        if (g.n_out > 0) k_grad_rest<<<std::min(blocks, int(grid_for(g.n_out))), BLK, 0, s>>>(g);
    }
    SC_HIP(hipGetLastError());
    int bad = 0;
    {
        ReadBack rb(c);
        rb.add(&bad, static_cast<const int *>(p.bad), 1);
        rb.run();
    }
    SC_REQUIRE(!bad, SC_EUNDEF, "an output vertex has no provenance (sequential route midpoint vertex)");
}

} // namespace sc
