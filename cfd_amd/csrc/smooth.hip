// Start-up mesh smoothing: smoothing_mod::smoothing (smoothing.f90:21-75),
// the quality-driven node relocation the main program runs once before the
// time loop (ns2DComp.ALE.f90:76).
//
// The reference:
//   checkMesh: nodes of elements with quality mu < 0.85 become smoothable;
//     H_MIN_GLOBAL = min(1, min over elements of h);
//   two Laplacian passes: each smoothable free node moves to the mean of its
//     neighbours (or a tol_move-sized step towards it), restored when its
//     worst element gets worse;
//   up to 100 sweeps: each smoothable free node clears its flag and, when its
//     worst element is below 0.85, climbs the worst element's quality along a
//     one-sided-difference gradient (2 steps of up to 8 halving tries, the
//     tries accumulating), re-marking its neighbours when it moved; the
//     sweeps stop when the largest squared move is below 0.01 H_MIN_GLOBAL.
// Every pass updates the nodes in place, in index order, so each node reads
// the new positions of the lower-numbered neighbours moved before it.  On an
// O-grid numbered ring by ring that order is a chain through every node of
// the mesh (node (r, 0) follows node (r-1, last) through the seam), so the
// reference's result is inherently sequential.
//
// Two schedules of the same per-node arithmetic (same operations, same order,
// contraction off):
//   order 0 - the reference's node order, bit for bit its result, for small
//             meshes: one wave per pass walks the nodes, its lanes forming a
//             node's elements (and its tries) side by side, while the waves of
//             the next passes, on other CUs, follow behind (k_sm_passes);
//   order 1 - colour by colour: a greedy colouring of the node graph (no two
//             nodes of one colour share an element, so nodes of a colour read
//             and write disjoint data), side by side, colours in
//             sequence.  The same per-node updates in another order: a
//             different, equally admissible smoothing (every accepted move
//             still raises the node's worst element).
#include <algorithm>

#include "cfd_internal.hpp"
#include "crmath.hpp"
#include "reduce.hpp"

namespace cfd {

namespace {

constexpr int kSmSweeps = 100;       // NITER
constexpr int kSmSteps = 2;          // MITER
constexpr int kSmTries = 8;          // NTRY
constexpr double kSmTolMetric = .85; // TOL_METRIC
constexpr double kSmTolDist = 1e-2;  // FACTOR_TOL_DIST
constexpr double kSmDelta = 1e-2;    // FACTOR_DELTA
constexpr double kSmPlus = 1.0;      // FACTOR_PLUS
constexpr double kSmStep = 3.0;      // FACTOR_STEP
constexpr double kTwoSqrt3 = 3.46410161513775;

struct SmDev {
    const int *inpoel, *esup1, *esup2, *psup1, *psup2, *fixed;
    double *X, *Y;
    int* smoothable;
    const double* tol_move;  // null: setTol_move not called
    const double* hmin;      // H_MIN_GLOBAL, device scalar
};

// smoothing.f90:344-355 mu and :357-365 h of the element's three nodes
__device__ inline double sm_mu(const SmDev& d, int e) {
    const int* n = d.inpoel + 3 * e;
    const double X1 = d.X[n[0] - 1], X2 = d.X[n[1] - 1], X3 = d.X[n[2] - 1];
    const double Y1 = d.Y[n[0] - 1], Y2 = d.Y[n[1] - 1], Y3 = d.Y[n[2] - 1];
    const double area = X2 * Y3 + X3 * Y1 + X1 * Y2 - (X2 * Y1 + X3 * Y2 + X1 * Y3);
    const double l1 = (X3 - X2) * (X3 - X2) + (Y3 - Y2) * (Y3 - Y2);
    const double l2 = (X1 - X3) * (X1 - X3) + (Y1 - Y3) * (Y1 - Y3);
    const double l3 = (X2 - X1) * (X2 - X1) + (Y2 - Y1) * (Y2 - Y1);
    const double l = l1 + l2 + l3;
    return kTwoSqrt3 * area / l;
}

__device__ inline double sm_h(const SmDev& d, int e) {
    const int* n = d.inpoel + 3 * e;
    const double X1 = d.X[n[0] - 1], X2 = d.X[n[1] - 1], X3 = d.X[n[2] - 1];
    const double Y1 = d.Y[n[0] - 1], Y2 = d.Y[n[1] - 1], Y3 = d.Y[n[2] - 1];
    const double area = X2 * Y3 + X3 * Y1 + X1 * Y2 - (X2 * Y1 + X3 * Y2 + X1 * Y3);
    const double d1 = fabs(X3 - X2) + fabs(Y3 - Y2);
    const double d2 = fabs(X1 - X3) + fabs(Y1 - Y3);
    const double d3 = fabs(X2 - X1) + fabs(Y2 - Y1);
    const double dd = d1 + d2 + d3;
    return fabs(area) / dd;
}

// getMu_min (:199-215)
__device__ inline double sm_mu_min(const SmDev& d, int ip) {
    double m = 1;
    for (int s = d.esup2[ip - 1]; s < d.esup2[ip]; ++s) {
        const double mu1 = sm_mu(d, d.esup1[s] - 1);
        if (mu1 <= m) m = mu1;
    }
    return m;
}

// laplacianSmoothing (:77-111), node ip
__device__ void sm_laplacian_node(const SmDev& d, int ip) {
    if (!(d.smoothable[ip - 1] && !d.fixed[ip - 1])) return;
    double xn = 0, yn = 0;
    const double mu_old = sm_mu_min(d, ip);
    const double xo = d.X[ip - 1], yo = d.Y[ip - 1];
    const int n = d.psup2[ip] - d.psup2[ip - 1];
    for (int s = d.psup2[ip - 1]; s < d.psup2[ip]; ++s) {
        xn = xn + d.X[d.psup1[s] - 1];
        yn = yn + d.Y[d.psup1[s] - 1];
    }
    xn = xn / n;
    yn = yn / n;
    if (d.tol_move) {
        const double dX = xn - d.X[ip - 1], dY = yn - d.Y[ip - 1];
        const double tm = d.tol_move[ip - 1];
        d.X[ip - 1] = d.X[ip - 1] + dX / (fabs(dX) + fabs(dY)) * tm / 2 * kSmStep;
        d.Y[ip - 1] = d.Y[ip - 1] + dY / (fabs(dX) + fabs(dY)) * tm / 2 * kSmStep;
    } else {
        d.X[ip - 1] = xn;
        d.Y[ip - 1] = yn;
    }
    if (sm_mu_min(d, ip) < mu_old) {  // if worse, restore
        d.X[ip - 1] = xo;
        d.Y[ip - 1] = yo;
    }
}

// checkMesh (:367-385): smoothable marks and per-block partials of min h
// and of "some element below 0.85"
__global__ void __launch_bounds__(kBlock)
k_sm_check(int nelem, SmDev d, double* __restrict__ hpart, double* __restrict__ anypart) {
    double hm = 1.0, any = 0.0;
    for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < nelem; e += gridDim.x * blockDim.x) {
        if (sm_mu(d, e) < kSmTolMetric) {
            const int* n = d.inpoel + 3 * e;
            for (int k = 0; k < 3; ++k) d.smoothable[n[k] - 1] = 1;
            any = 1.0;
        }
        const double h1 = sm_h(d, e);
        if (h1 < hm) hm = h1;
    }
    block_partial(hm, OpMin(), hpart);
    block_partial(any, OpMax(), anypart);
}

// H_MIN_GLOBAL = min(1, partials) and the "any" flag
__global__ void __launch_bounds__(256)
k_sm_check_fin(const double* __restrict__ hpart, const double* __restrict__ anypart, int nb,
               double* __restrict__ out) {
    const double h = combine_partials(hpart, nb, 1.0, OpMin());
    const double a = combine_partials(anypart, nb, 0.0, OpMax());
    if (threadIdx.x == 0) {
        out[0] = h;
        out[1] = a;
    }
}

// v of a lane that every lane names alike
__device__ __forceinline__ double lane_of(double v, int lane) {
    const int l = __builtin_amdgcn_readfirstlane(lane);
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                            __builtin_amdgcn_readlane(__double2loint(v), l));
}
// v of another lane of the row of 16 by the DPP control kCtrl (no LDS round trip)
template <int kCtrl>
__device__ __forceinline__ double dpp_of(double v) {
    const int hi = __double2hiint(v), lo = __double2loint(v);
    return __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, kCtrl, 0xf, 0xf, false),
                            __builtin_amdgcn_update_dpp(lo, lo, kCtrl, 0xf, 0xf, false));
}
constexpr int kDppXor1 = 0xB1, kDppXor2 = 0x4E, kDppHalfMirror = 0x141, kDppMirror = 0x140;

// One node's update by a wave: lane k of each group of G lanes forms the node's
// k-th element (esup order), the groups the tries and the three points of a
// gradient.  pos(i) is node i's position (0-based).
template <class Pos>
struct SmNode {
    const SmDev& d;
    Pos pos;
    int ip, id[3], G, k, g;  // the node; the lane's element; lanes a group, lane, group
    bool act;                // the lane has an element
    double2 own;
    double cx[3], cy[3], X[3], Y[3], area;  // the element's corners; those of the last evaluation

    static __device__ __forceinline__ int lanes(int cnt) { return cnt <= 8 ? 8 : cnt <= 16 ? 16 : 32; }
    // ids: the nodes of the lane's element (0-based; read where it has one)
    __device__ __forceinline__ SmNode(const SmDev& d, Pos pos, int ip, int cnt, const int (&ids)[3])
        : d(d), pos(pos), ip(ip), G(lanes(cnt)) {
        const int lane = threadIdx.x & 63;
        k = lane & (G - 1);
        g = lane / G;
        act = k < cnt;
#pragma unroll
        for (int v = 0; v < 3; ++v) {
            id[v] = act ? ids[v] : ip;
            const double2 c = pos(id[v]);
            cx[v] = c.x;
            cy[v] = c.y;
        }
        own = pos(ip);
    }
    // quality (sm_mu) of the lane's element with the node at x, y
    __device__ __forceinline__ double mu(double x, double y) {
#pragma unroll
        for (int v = 0; v < 3; ++v) {
            X[v] = id[v] == ip ? x : cx[v];
            Y[v] = id[v] == ip ? y : cy[v];
        }
        area = X[1] * Y[2] + X[2] * Y[0] + X[0] * Y[1] -
               (X[1] * Y[0] + X[2] * Y[1] + X[0] * Y[2]);
        const double l1 = (X[2] - X[1]) * (X[2] - X[1]) + (Y[2] - Y[1]) * (Y[2] - Y[1]);
        const double l2 = (X[0] - X[2]) * (X[0] - X[2]) + (Y[0] - Y[2]) * (Y[0] - Y[2]);
        const double l3 = (X[1] - X[0]) * (X[1] - X[0]) + (Y[1] - Y[0]) * (Y[1] - Y[0]);
        const double l = l1 + l2 + l3;
        return quot(kTwoSqrt3 * area, l);
    }
    // h (sm_h) at the corners of the last evaluation
    __device__ __forceinline__ double h_at() const {
        const double d1 = fabs(X[2] - X[1]) + fabs(Y[2] - Y[1]);
        const double d2 = fabs(X[0] - X[2]) + fabs(Y[0] - Y[2]);
        const double d3 = fabs(X[1] - X[0]) + fabs(Y[1] - Y[0]);
        return quot(fabs(area), d1 + d2 + d3);
    }
    // smallest of the group's v where ok (init where none is smaller; NaN never
    // is), known to the whole group
    __device__ __forceinline__ double group_min(double v, bool ok, double init) const {
        double m1 = ok && v < init ? v : init;
        auto take = [&](double o) {
            if (o < m1) m1 = o;
        };
        take(dpp_of<kDppXor1>(m1));
        take(dpp_of<kDppXor2>(m1));
        take(dpp_of<kDppHalfMirror>(m1));  // quads hold one value each
        if (G > 8) take(dpp_of<kDppMirror>(m1));
        if (G > 16) take(__shfl_xor(m1, 16, 64));
        return m1;
    }
    // getMu_vec's min_idx (smoothing.f90:174-197): the first element with the
    // smallest quality below 1 (element 0 when none is), and its quality
    __device__ __forceinline__ int worst(double v, double& vm) const {
        vm = group_min(v, act, 1.0);
        const unsigned long long hit = __ballot(act && v < 1.0 && v == vm);
        const unsigned long long mine = (hit >> (g * G)) & ((1ull << G) - 1ull);
        if (__any(!mine)) {
            const double v0 = __shfl(v, g * G, 64);
            if (!mine) vm = v0;
        }
        return mine ? (int)__builtin_ctzll(mine) : 0;
    }
    // laplacianSmoothing (:77-111): the node's new position
    __device__ __forceinline__ double2 laplacian() {
        const double x = own.x, y = own.y;
        const int lane = threadIdx.x & 63;
        const double mu_old = group_min(mu(x, y), act, 1.0);
        const int s0 = d.psup2[ip], np = d.psup2[ip + 1] - s0;
        const double2 nb = pos(lane < np ? d.psup1[s0 + lane] - 1 : ip);
        double xn = 0, yn = 0;
        for (int v = 0; v < np; ++v) {
            xn = xn + lane_of(nb.x, v);
            yn = yn + lane_of(nb.y, v);
        }
        xn = xn / np;
        yn = yn / np;
        if (d.tol_move) {
            const double dX = xn - x, dY = yn - y, tm = d.tol_move[ip];
            xn = x + dX / (fabs(dX) + fabs(dY)) * tm / 2 * kSmStep;
            yn = y + dY / (fabs(dX) + fabs(dY)) * tm / 2 * kSmStep;
        }
        if (group_min(mu(xn, yn), act, 1.0) < mu_old) return own;  // if worse, restored
        return make_double2(xn, yn);
    }
    // One node of an optimisation sweep: moveIpoin (:113-171) with getG
    // (:217-236) and getStep (:238-270).  False when its worst element is good
    // enough (:54-63); else *to is where it goes.  The tries accumulate: a failed
    // try is not undone before the next, half as long, is added.
    __device__ __forceinline__ bool sweep(double delta, const Recip& by_delta, double2& to) {
        double x = own.x, y = own.y;
        // The qualities v at x, y and those at x + delta and y + delta (getG) in
        // one evaluation: a group each
        const auto three = [&](double xo, double yo) {
            return mu(g == 1 ? xo + delta : xo, g == 2 ? yo + delta : yo);
        };
        double m = G < 32 ? three(x, y) : mu(x, y), mu_min;
        int mi = worst(m, mu_min);  // group 0's: its result counts
        mi = __builtin_amdgcn_readfirstlane(mi);
        mu_min = lane_of(mu_min, 0);
        if (!(mu_min < kSmTolMetric)) return false;
        for (int it = 0; it < kSmSteps; ++it) {
            const double xo = x, yo = y;
            double v, vx, vy, h;
            if (G < 32) {
                if (it > 0) m = three(xo, yo);
                h = h_at();
                v = __shfl(m, k, 64);
                vx = __shfl(m, G + k, 64);
                vy = __shfl(m, 2 * G + k, 64);
            } else {
                v = it > 0 ? mu(xo, yo) : m;
                h = h_at();
                vx = mu(xo + delta, yo);
                vy = mu(xo, yo + delta);
            }
            const double gx = quot(vx - v, by_delta), gy = quot(vy - v, by_delta);
            // getStep: the largest step along the worst element's gradient before
            // another element's linearised quality falls to the worst one's
            const double gxm = lane_of(gx, mi), gym = lane_of(gy, mi);
            const double g2 = gxm * gxm + gym * gym;
            double step;
            if (d.tol_move) {
                step = d.tol_move[ip] / ((fabs(gxm) + fabs(gym)) * (double)kSmSweeps);
            } else {  // group 0's h
                h = lane_of(group_min(h, act, 1.0), 0);
                step = quot(h * kSmStep, fabs(gxm) + fabs(gym));
            }
            const double gg = gxm * gx + gym * gy;
            step = group_min(quot(v - mu_min, g2 - gg), act && gg < 0, step);
            // the tries, a group each, in batches of 64 / G
            bool accepted = false;
            for (int t0 = 0; t0 < kSmTries && !accepted; t0 += 64 / G) {
                double xs = x, ys = y;
                for (int u = 0; u < 64 / G; ++u) {
                    const double dx = step * gxm, dy = step * gym;
                    if (u <= g) {
                        xs = xs + dx;
                        ys = ys + dy;
                    }
                    step = .5 * step;
                }
                const double nv = mu(xs, ys);
                double best;
                const int nmi = worst(nv, best);
                const unsigned long long ok = __ballot(best > mu_min * kSmPlus);
                // the first group that raised the worst element, else the last
                // try's position
                const int sel = ok ? (int)__builtin_ctzll(ok) / G : 64 / G - 1;
                x = lane_of(xs, sel * G);
                y = lane_of(ys, sel * G);
                if (ok) {
                    mi = __builtin_amdgcn_readlane(nmi, __builtin_amdgcn_readfirstlane(sel * G));
                    mu_min = lane_of(best, sel * G);
                    accepted = true;
                }
            }
            if (!accepted) {  // restore and stop
                x = xo;
                y = yo;
                break;
            }
        }
        to = make_double2(x, y);
        return true;
    }
};

// ---------------------------------------------------------------------------
// order 0: up to kSmPasses consecutive passes in one launch, a block of one wave
// per pass, each on a CU of its own.
//
// A node's update reads its ring (the nodes that share an element with it) and
// marks it, and changes nothing else but the node itself.  So pass w + 1 may
// update node i as soon as pass w is past i and past every node of i's ring:
// each block publishes how far it is (prog, after every 64 nodes) and the next
// one follows that far behind, taking the positions and marks that it left.
// Every update then reads exactly the values and marks that it would read with
// the passes one after the other.  Block 0 waits for nothing and block w only
// for block w - 1, and the twelve blocks of every launch in flight (one a stream,
// a few streams on the hardware's queues) are far fewer than the CUs: each has a
// CU as soon as other kernels' blocks leave one, so each wait ends.  Should one not
// (its predecessor has no CU for so long, or is lost), the block gives up when it has
// seen no progress for `limit`, says so behind prog, and the call fails; those behind
// it see no progress either.  On a ring by ring numbering the passes run one ring and
// a chunk apart; on one where every node has a far neighbour they run one after the
// other.
//
// Marks: a sweep that moves node i marks its ring.  Nodes after i take their
// turn in the same sweep (the block's own marks), those before i in the next
// one (a row of bits in memory, read once that sweep may pass them).
//
// Inside a wave the lanes form the qualities of the node's elements, 8, 16 or
// 32 lanes a group, and the groups the tries (their positions are the running
// sums that the sequential loop forms) and the three points of a gradient.
//
// Whether a sweep is the last is known when it ends, while the next ones are
// on their way: each block leaves its pass's positions in hist, and the result
// is taken from the last sweep that counts.
//
// Bound by the chain of one node's update (3 us: about 700 instructions with
// the lanes' exchanges and eight divisions in sequence), node after node, on
// one wave; the positions stay in LDS while they fit.  64 x 128 cylinder (8,192
// nodes, 2 + 8 passes): 28.7 ms; 42.7 with the passes as twelve waves of one
// block (three to a SIMD share its instructions), 1,524 with one lane per pass
// and the passes one by one.
// ---------------------------------------------------------------------------
constexpr int kSmPasses = 12;
struct SmSeq {
    SmDev d;               // topology, tol_move, hmin
    const int *ring, *need;  // per esup entry its element's nodes (0-based); per node
                             // how far the pass before has to be
    const double2* xy;     // positions before the launch's first pass
    double2* hist;         // positions after each pass of the launch
    // rows of a bit per node: row 0 the marks before the first sweep, row w + 1
    // those that pass w leaves to the next; then the free nodes
    unsigned* rows;
    int* prog;             // per pass: nodes done; then 1 when a pass gave up
    double* dmax;          // per pass: the largest squared move
    int n, nlap;           // nodes; Laplacian passes of the launch, the first ones
    long long limit;       // of a wait without progress, ticks of wall_clock64()
};
__host__ __device__ constexpr int sm_words(int n) { return (n + 63) / 64 * 2; }

template <bool kLds>
__global__ void __launch_bounds__(64)
k_sm_passes(SmSeq q) {
    extern __shared__ double2 smem_sm[];
    const int n = q.n, nw = sm_words(n), lane = threadIdx.x, w = blockIdx.x;
    double2* own_hist = q.hist + (size_t)w * n;
    double2* xy = kLds ? smem_sm : own_hist;
    unsigned* marks = reinterpret_cast<unsigned*>(smem_sm + (kLds ? n : 0));
    const unsigned* free_ = q.rows + (size_t)(kSmPasses + 1) * nw;
    const double2* src = w > 0 ? own_hist - n : q.xy;
    const unsigned* in_row = q.rows + (size_t)w * nw;
    unsigned* out_row = q.rows + (size_t)(w + 1) * nw;
    const bool lap = w < q.nlap;
    for (int i = lane; i < nw; i += 64) marks[i] = w <= q.nlap ? q.rows[i] : 0u;
    __syncthreads();
    {
        const double delta = *q.d.hmin * kSmDelta;
        const Recip by_delta = recip(delta);
        double d_max = 0.0;
        int taken = 0;  // positions of the pass before that are here
        for (int c0 = 0; c0 < n; c0 += 64) {
            const int node = c0 + lane;
            const bool in = node < n;
            const int b_l = in ? q.d.esup2[node] : 0, e_l = in ? q.d.esup2[node + 1] : 0;
            int need = in ? q.need[node] : 0;
            for (int off = 32; off > 0; off >>= 1) need = max(need, __shfl_xor(need, off, 64));
            if (w > 0) {
                long long since = wall_clock64();
                for (int at, seen = -1;;) {
                    at = __builtin_amdgcn_readfirstlane(__hip_atomic_load(
                        &q.prog[w - 1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
                    if (at >= need) break;
                    const long long now = wall_clock64();
                    if (at != seen) {
                        seen = at;
                        since = now;
                    } else if (now - since > q.limit) {
                        if (lane == 0)
                            __hip_atomic_store(&q.prog[kSmPasses], 1, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT);
                        return;
                    }
                    __builtin_amdgcn_s_sleep(16);
                }
                __threadfence();
            }
            for (int i = taken + lane; i < need; i += 64) xy[i] = src[i];
            taken = max(taken, need);
            if (w > q.nlap && lane < 2) marks[c0 / 32 + lane] |= in_row[c0 / 32 + lane];
            __syncthreads();
            unsigned long long passed = 0;
            int next = -1, nid[3];  // the entries of the node expected next
            const unsigned long long fr =
                (unsigned long long)free_[c0 / 32] | ((unsigned long long)free_[c0 / 32 + 1] << 32);
            for (;;) {
                const volatile unsigned* mv = marks + c0 / 32;
                const unsigned long long m =
                    ((unsigned long long)mv[0] | ((unsigned long long)mv[1] << 32)) & fr & ~passed;
                if (!m) break;
                const int j = __builtin_ctzll(m);
                passed |= (2ull << j) - 1ull;
                const int ip = c0 + j;
                const int b = __builtin_amdgcn_readlane(b_l, j);
                const int cnt = __builtin_amdgcn_readlane(e_l, j) - b;
                const auto at = [xy](int i) { return xy[i]; };
                const int G = SmNode<decltype(at)>::lanes(cnt), k = lane & (G - 1);
                int id[3] = {ip, ip, ip};
                if (k < cnt)
#pragma unroll
                    for (int v = 0; v < 3; ++v)
                        id[v] = next == j ? nid[v] : q.ring[3 * (b + k) + v];
                SmNode<decltype(at)> node_(q.d, at, ip, cnt, id);
                if (j < 63) {  // most nodes marked: the next one's entries, in flight meanwhile
                    next = j + 1;
                    const int b1 = __builtin_amdgcn_readlane(b_l, next);
                    const int e1 = __builtin_amdgcn_readlane(e_l, next);
                    const int k1 = lane & (SmNode<decltype(at)>::lanes(e1 - b1) - 1);
                    if (b1 + k1 < e1)
                        for (int v = 0; v < 3; ++v) nid[v] = q.ring[3 * (b1 + k1) + v];
                }
                double2 to;
                if (lap) {
                    to = node_.laplacian();
                } else {
                    if (lane == 0) atomicAnd(&marks[ip >> 5], ~(1u << (ip & 31)));
                    if (!node_.sweep(delta, by_delta, to)) continue;
                    const double ex = to.x - node_.own.x, ey = to.y - node_.own.y;
                    const double d_move = ex * ex + ey * ey;
                    if (d_move > d_max) d_max = d_move;
                    if (d_move > __DBL_MIN__ && node_.act && node_.g == 0)  // update_list (:289-298)
#pragma unroll
                        for (int u = 0; u < 3; ++u) {
                            const int m = node_.id[u];
                            if (m != ip)
                                atomicOr(&(m > ip ? marks : out_row)[m >> 5], 1u << (m & 31));
                        }
                }
                if (lane == 0) xy[ip] = to;
                // the wave's other lanes read it: LDS takes a wave's accesses in order
                if (kLds) asm volatile("" ::: "memory");
                else __threadfence_block();
            }
            if (kLds && in) own_hist[node] = xy[node];
            __threadfence();
            if (lane == 0)
                __hip_atomic_store(&q.prog[w], min(c0 + 64, n), __ATOMIC_RELEASE,
                                   __HIP_MEMORY_SCOPE_AGENT);
        }
        if (lane == 0) q.dmax[w] = d_max;
    }
}

// Before a launch: the first sweep's marks (of the check, or what row `last`
// was left), empty rows behind them, the free nodes, no pass begun.  A thread
// per word.
__global__ void k_sm_rows(const int* __restrict__ smoothable, const int* __restrict__ fixed,
                          unsigned* __restrict__ rows, int* __restrict__ prog, int n, int last) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, nw = sm_words(n);
    if (i <= kSmPasses) prog[i] = 0;
    if (i >= nw) return;
    unsigned m = 0, f = 0;
    for (int b = 0; b < 32 && 32 * i + b < n; ++b) {
        if (smoothable[32 * i + b]) m |= 1u << b;
        if (!fixed[32 * i + b]) f |= 1u << b;
    }
    rows[i] = last > 0 ? rows[(size_t)last * nw + i] : m;
    for (int r = 1; r <= kSmPasses; ++r) rows[(size_t)r * nw + i] = 0;
    rows[(size_t)(kSmPasses + 1) * nw + i] = f;
}

// per node: its ring (the nodes of its elements, in esup order) and how far the
// pass before has to be for it
__global__ void k_sm_ring(const int* __restrict__ inpoel, const int* __restrict__ esup1,
                          const int* __restrict__ esup2, int* __restrict__ ring,
                          int* __restrict__ need, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int far = i;
    for (int s = esup2[i]; s < esup2[i + 1]; ++s)
        for (int k = 0; k < 3; ++k) {
            const int m = inpoel[3 * (esup1[s] - 1) + k] - 1;
            ring[3 * s + k] = m;
            far = max(far, m);
        }
    need[i] = far + 1;
}

__global__ void k_sm_pack(const double* __restrict__ X, const double* __restrict__ Y,
                          double2* __restrict__ xy, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) xy[i] = make_double2(X[i], Y[i]);
}

__global__ void k_sm_unpack(const double2* __restrict__ xy, double* __restrict__ X,
                            double* __restrict__ Y, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    X[i] = xy[i].x;
    Y[i] = xy[i].y;
}

// order 1, the Laplacian passes: one lane per node of a colour (12 us a colour of
// 13,000 nodes; a wave per node takes 22: most of it loads of one position a
// lane)
__global__ void __launch_bounds__(kBlock)
k_sm_laplacian_colour(SmDev d, const int* __restrict__ nodes, int count) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q < count) sm_laplacian_node(d, nodes[q]);
}

// order 1, a sweep: one wave per node of a colour, four a block.  A colour of
// 13,000 nodes takes 19 us; with one lane per node, which keeps its elements'
// qualities and gradients in scratch memory and tries one position after the
// other, 52.
constexpr int kColourWaves = 4;
__global__ void __launch_bounds__(64 * kColourWaves)
k_sm_sweep_colour(SmDev d, const int* __restrict__ nodes, int count, double* __restrict__ dmove) {
    const int q = __builtin_amdgcn_readfirstlane(blockIdx.x * kColourWaves + (threadIdx.x >> 6));
    if (q >= count) return;
    const int lane = threadIdx.x & 63, ip = nodes[q] - 1;
    if (!(d.smoothable[ip] && !d.fixed[ip])) return;
    const int b = d.esup2[ip];
    const auto at = [&d](int i) { return make_double2(d.X[i], d.Y[i]); };
    const int cnt = d.esup2[ip + 1] - b, k = lane & (SmNode<decltype(at)>::lanes(cnt) - 1);
    int id[3] = {ip, ip, ip};
    if (k < cnt) {
        const int* n = d.inpoel + 3 * (d.esup1[b + k] - 1);
#pragma unroll
        for (int v = 0; v < 3; ++v) id[v] = n[v] - 1;
    }
    SmNode<decltype(at)> node(d, at, ip, cnt, id);
    if (lane == 0) d.smoothable[ip] = 0;
    const double delta = *d.hmin * kSmDelta;
    double2 to;
    if (!node.sweep(delta, recip(delta), to)) return;
    const double ex = to.x - node.own.x, ey = to.y - node.own.y;
    const double d_move = ex * ex + ey * ey;
    if (d_move > __DBL_MIN__ && node.act && node.g == 0)  // update_list (:289-298)
#pragma unroll
        for (int u = 0; u < 3; ++u)
            if (node.id[u] != ip) d.smoothable[node.id[u]] = 1;
    if (lane == 0) {
        dmove[ip] = d_move;
        d.X[ip] = to.x;
        d.Y[ip] = to.y;
    }
}

// largest squared move of a colour sweep (moves are >= 0 or NaN; NaN is
// skipped as the reference's "d_move > d_max" skips it)
__global__ void __launch_bounds__(kBlock)
k_sm_max(const double* __restrict__ v, int n, double* __restrict__ partials) {
    double m = 0.0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        if (v[i] > m) m = v[i];
    block_partial(m, OpMax(), partials);
}

__global__ void __launch_bounds__(256)
k_sm_max_fin(const double* __restrict__ partials, int nb, double* __restrict__ out) {
    const double m = combine_partials(partials, nb, 0.0, OpMax());
    if (threadIdx.x == 0) *out = m;
}

}  // namespace

void SmoothPlan::build(const Tables& t, const int* fixed_host, hipStream_t s) {
    const int n = t.npoin;
    std::vector<int> e2(n + 1), p2(n + 1), p1(t.npsup);
    t.esup2.download(e2.data(), n + 1, s);
    t.psup2.download(p2.data(), n + 1, s);
    t.psup1.download(p1.data(), t.npsup, s);
    CFD_HIP(hipStreamSynchronize(s));
    max_elems = 0;
    for (int i = 0; i < n; ++i) max_elems = std::max(max_elems, e2[i + 1] - e2[i]);
    // greedy colouring in node order: the smallest colour no lower-numbered
    // neighbour holds
    std::vector<int> colour(n, -1), seen;
    int ncol = 0;
    for (int i = 0; i < n; ++i) {
        seen.assign(ncol + 1, 0);
        for (int q = p2[i]; q < p2[i + 1]; ++q) {
            const int c = colour[p1[q] - 1];
            if (c >= 0) seen[c] = 1;
        }
        int c = 0;
        while (seen[c]) ++c;
        colour[i] = c;
        ncol = std::max(ncol, c + 1);
    }
    // free nodes by colour, ascending within a colour
    colour_ptr.assign(ncol + 1, 0);
    for (int i = 0; i < n; ++i)
        if (!fixed_host[i]) ++colour_ptr[colour[i] + 1];
    for (int c = 0; c < ncol; ++c) colour_ptr[c + 1] += colour_ptr[c];
    std::vector<int> nodes(std::max(1, colour_ptr[ncol])), fill(colour_ptr.begin(), colour_ptr.end() - 1);
    for (int i = 0; i < n; ++i)
        if (!fixed_host[i]) nodes[fill[colour[i]]++] = i + 1;
    colour_nodes.alloc(nodes.size());
    colour_nodes.upload(nodes.data(), nodes.size(), s);
    fixed.alloc(std::max(1, n));
    fixed.upload(fixed_host, n, s);
    smoothable.alloc(std::max(1, n));
    dmove.alloc(std::max(1, n));
    partials.alloc(2 * (size_t)kRedBlocks);
    scal.alloc(4);
}

bool smooth_check(const Tables& t, SmoothPlan& plan, double* X, double* Y, double* hmin_host,
                  hipStream_t s) {
    SmDev d{t.inpoel.p, t.esup1.p, t.esup2.p, t.psup1.p, t.psup2.p, plan.fixed.p,
            X, Y, plan.smoothable.p, nullptr, plan.scal.p};
    plan.smoothable.zero(s);
    const int nb = std::min<int>(grid_for(t.nelem), kRedBlocks);
    k_sm_check<<<nb, kBlock, 0, s>>>(t.nelem, d, plan.partials.p, plan.partials.p + kRedBlocks);
    k_sm_check_fin<<<1, 256, 0, s>>>(plan.partials.p, plan.partials.p + kRedBlocks, nb, plan.scal.p);
    CFD_HIP(hipGetLastError());
    double hs[2];
    CFD_HIP(hipMemcpyAsync(hs, plan.scal.p, sizeof(hs), hipMemcpyDeviceToHost, s));
    CFD_HIP(hipStreamSynchronize(s));
    plan.hmin = hs[0];
    if (hmin_host) *hmin_host = hs[0];
    return hs[1] != 0.0;
}

// order 0 (see k_sm_passes)
static int smooth_run_seq(const Tables& t, SmoothPlan& plan, const SmDev& d, hipStream_t s) {
    const int n = t.npoin, nw = sm_words(n);
    if (plan.ring.n != 9 * (size_t)t.nelem) {  // kept with the mesh's plan (ring, the last: all of it)
        plan.need.alloc(n);
        plan.xy.alloc(n);
        plan.hist.alloc((size_t)kSmPasses * n);
        plan.dmax_pass.alloc(kSmPasses);
        plan.rows.alloc((size_t)(kSmPasses + 2) * nw);
        plan.prog.alloc(kSmPasses + 1);
        plan.ring.alloc(9 * (size_t)t.nelem);
    }
    k_sm_ring<<<grid_for(n), kBlock, 0, s>>>(t.inpoel.p, t.esup1.p, t.esup2.p, plan.ring.p,
                                             plan.need.p, n);
    k_sm_pack<<<grid_for(n), kBlock, 0, s>>>(d.X, d.Y, plan.xy.p, n);
    // the positions in LDS while they fit (9,600 nodes in 160 KB)
    const size_t base = (size_t)nw * sizeof(unsigned), full = base + (size_t)n * sizeof(double2);
    int dev = 0, most = 0;
    CFD_HIP(hipGetDevice(&dev));
    CFD_HIP(hipDeviceGetAttribute(&most, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
    const bool lds = full <= (size_t)most;
    if (lds)  // the limit holds for the process: the same for every mesh
        CFD_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k_sm_passes<true>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, most));
    int khz = 0;
    CFD_HIP(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev));
    const long long limit = (long long)(1.0e3 * khz * plan.wait_s);
    const double tol_dist = kSmTolDist * plan.hmin;
    const double2* result = plan.xy.p;
    int sweep = 0, nlap = 2, last = 0;
    for (bool end = false; !end && sweep < kSmSweeps; nlap = 0) {
        const int nsw = std::min(kSmPasses - nlap, kSmSweeps - sweep), np = nlap + nsw;
        if (last > 0)  // the next passes start from the last one's positions
            CFD_HIP(hipMemcpyAsync(plan.xy.p, result, sizeof(double2) * n, hipMemcpyDeviceToDevice, s));
        k_sm_rows<<<grid_for(std::max(nw, kSmPasses + 1)), kBlock, 0, s>>>(
            plan.smoothable.p, plan.fixed.p, plan.rows.p, plan.prog.p, n, last);
        const SmSeq q{d, plan.ring.p, plan.need.p, plan.xy.p, plan.hist.p, plan.rows.p,
                      plan.prog.p, plan.dmax_pass.p, n, nlap, limit};
        if (lds) k_sm_passes<true><<<np, 64, full, s>>>(q);
        else k_sm_passes<false><<<np, 64, base, s>>>(q);
        CFD_HIP(hipGetLastError());
        last = np;
        double dmax[kSmPasses];
        int lost = 0;
        CFD_HIP(hipMemcpyAsync(dmax, plan.dmax_pass.p, sizeof(dmax), hipMemcpyDeviceToHost, s));
        CFD_HIP(hipMemcpyAsync(&lost, plan.prog.p + kSmPasses, sizeof(lost), hipMemcpyDeviceToHost, s));
        CFD_HIP(hipStreamSynchronize(s));
        CFD_CHECK(!lost, "smoothing: a pass saw no progress of the one before for " +
                             std::to_string(plan.wait_s) + " s");
        for (int k = nlap; k < np && !end; ++k) {
            ++sweep;
            end = dmax[k] < tol_dist;
            result = plan.hist.p + (size_t)k * n;
        }
    }
    k_sm_unpack<<<grid_for(n), kBlock, 0, s>>>(result, d.X, d.Y, n);
    CFD_HIP(hipGetLastError());
    return sweep;
}

int smooth_run(const Tables& t, SmoothPlan& plan, double* X, double* Y, const double* tol_move,
               int order, hipStream_t s) {
    const int n = t.npoin;
    SmDev d{t.inpoel.p, t.esup1.p, t.esup2.p, t.psup1.p, t.psup2.p, plan.fixed.p,
            X, Y, plan.smoothable.p, tol_move, plan.scal.p};
    if (order == 0) return smooth_run_seq(t, plan, d, s);
    const int ncol = (int)plan.colour_ptr.size() - 1;
    auto colour_pass = [&](auto launch) {
        for (int c = 0; c < ncol; ++c) {
            const int b = plan.colour_ptr[c], cnt = plan.colour_ptr[c + 1] - b;
            if (cnt > 0) launch(plan.colour_nodes.p + b, cnt);
        }
    };
    for (int it = 0; it < 2; ++it) {
        colour_pass([&](const int* nodes, int cnt) {
            k_sm_laplacian_colour<<<grid_for(cnt), kBlock, 0, s>>>(d, nodes, cnt);
        });
    }
    CFD_HIP(hipGetLastError());
    const double tol_dist = kSmTolDist * plan.hmin;
    const int nbm = std::min<int>(grid_for(n), kRedBlocks);
    int sweep = 1;
    for (; sweep <= kSmSweeps; ++sweep) {
        plan.dmove.zero(s);
        colour_pass([&](const int* nodes, int cnt) {
            k_sm_sweep_colour<<<(cnt + kColourWaves - 1) / kColourWaves, 64 * kColourWaves, 0, s>>>(
                d, nodes, cnt, plan.dmove.p);
        });
        k_sm_max<<<nbm, kBlock, 0, s>>>(plan.dmove.p, n, plan.partials.p);
        k_sm_max_fin<<<1, 256, 0, s>>>(plan.partials.p, nbm, plan.scal.p + 2);
        CFD_HIP(hipGetLastError());
        double dmax;
        CFD_HIP(hipMemcpyAsync(&dmax, plan.scal.p + 2, sizeof(double), hipMemcpyDeviceToHost, s));
        CFD_HIP(hipStreamSynchronize(s));
        if (dmax < tol_dist) break;
    }
    return std::min(sweep, kSmSweeps);
}

}  // namespace cfd
