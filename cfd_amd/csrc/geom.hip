// Geometry kernels of the path: P1 gradients and areas (deriv), lumped mass
// (MASAS), mesh-Laplace values (mLaplace), the GCL mass update (gcl.f90),
// wall normals (NORMALES), and the small per-set loops of fluidStructure
// (FORCES, TRANSF).
//
// Node-owned results are gathers over each node's esup segment in ascending
// element order: that is the order in which the reference's sequential
// element-order scatter adds into the node, so sums are bitwise identical and
// no atomics are needed.  All of these are HBM-bound integer/gather work.
#include <type_traits>

#include "cfd_internal.hpp"
#include "forces.hpp"
#include "reduce.hpp"
#include "crmath.hpp"

namespace cfd {
namespace {

// mLaplace.f90:188-200
__device__ inline double quality_mu(double X1, double X2, double X3, double Y1, double Y2, double Y3) {
    const double TWOSQRT3 = 3.46410161513775;
    double ar = X2 * Y3 + X3 * Y1 + X1 * Y2 - (X2 * Y1 + X3 * Y2 + X1 * Y3);
    double l1 = (X3 - X2) * (X3 - X2) + (Y3 - Y2) * (Y3 - Y2);
    double l2 = (X1 - X3) * (X1 - X3) + (Y1 - Y3) * (Y1 - Y3);
    double l3 = (X2 - X1) * (X2 - X1) + (Y2 - Y1) * (Y2 - Y1);
    double l = l1 + l2 + l3;
    return TWOSQRT3 * ar / l;
}

// an element's weight in laplace, 1/mu^2 (mLaplace.f90:120-148)
__device__ inline double lap_weight(double X1, double X2, double X3, double Y1, double Y2, double Y3) {
    const double mu = quality_mu(X1, X2, X3, Y1, Y2, Y3);
    return 1.0 / (mu * mu);
}
// an element's two terms of gcl.f90:218-236: its W's divergence by area/3 now,
// and the old W's by the old area's
__device__ inline double2 gcl_terms(const double* nx, const double* ny, int n0, int n1, int n2,
                                    const double* Wx, const double* wy, const double* Wxo,
                                    const double* wyo, double area, double area_old) {
    const double divW = nx[0] * Wx[n0] + nx[1] * Wx[n1] + nx[2] * Wx[n2] + ny[0] * wy[n0] +
                        ny[1] * wy[n1] + ny[2] * wy[n2];
    const double divWo = nx[0] * Wxo[n0] + nx[1] * Wxo[n1] + nx[2] * Wxo[n2] + ny[0] * wyo[n0] +
                         ny[1] * wyo[n1] + ny[2] * wyo[n2];
    return make_double2(divW * area / 3.0, divWo * area_old / 3.0);
}

// subrutinas.f90:99-125, and what else the nodes' kernel needs of an element:
// its weight in laplace and (kGcl) its terms of the GCL, formed once here
// instead of by each of its nodes
template <bool kGcl>
__global__ void __launch_bounds__(kBlock)
k_deriv(const int* __restrict__ inpoel, const double* __restrict__ X, const double* __restrict__ Y,
        double* __restrict__ area, double* __restrict__ dNx, double* __restrict__ dNy,
        double* __restrict__ HH, double* __restrict__ HHX, double* __restrict__ HHY, int nelem,
        double* __restrict__ partials, ElemTerms x) {
    double hm = __builtin_huge_val();
    for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < nelem; e += gridDim.x * blockDim.x) {
        int n1 = inpoel[3 * e] - 1, n2 = inpoel[3 * e + 1] - 1, n3 = inpoel[3 * e + 2] - 1;
        double X1 = X[n1], X2 = X[n2], X3 = X[n3];
        double Y1 = Y[n1], Y2 = Y[n2], Y3 = Y[n3];
        double a = (X2 * Y3 + X3 * Y1 + X1 * Y2 - (X2 * Y1 + X3 * Y2 + X1 * Y3)) / 2.0;
        const double old = kGcl ? area[e] : 0.0;
        area[e] = a;
        double a2 = 2.0 * a;
        const double nx[3] = {(Y2 - Y3) / a2, (Y3 - Y1) / a2, (Y1 - Y2) / a2};
        const double ny[3] = {(X3 - X2) / a2, (X1 - X3) / a2, (X2 - X1) / a2};
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            dNx[3 * e + j] = nx[j];
            dNy[3 * e + j] = ny[j];
        }
        if (x.lapw) x.lapw[e] = lap_weight(X1, X2, X3, Y1, Y2, Y3);
        if (kGcl) {
            x.area_old[e] = old;
            x.gcl[e] = gcl_terms(nx, ny, n1, n2, n3, x.Wx, x.mode ? x.Wy : x.Wx, x.Wxo,
                                 x.mode ? x.Wyo : x.Wxo, a, old);
        }
        double h = sqrt(a);
        HH[e] = h;
        if (h < hm) hm = h;
        double mx = X3 - X2, my = Y3 - Y2;
        if (X1 - X3 < mx) mx = X1 - X3;
        if (X2 - X1 < mx) mx = X2 - X1;
        if (Y1 - Y3 < my) my = Y1 - Y3;
        if (Y2 - Y1 < my) my = Y2 - Y1;
        HHX[e] = fabs(mx);
        HHY[e] = fabs(my);
    }
    block_partial(hm, OpMin(), partials);
}

// subrutinas.f90:137-152: M(i) = sum of area/3 over i's elements, ascending
__global__ void __launch_bounds__(kBlock)
k_masas(const int* __restrict__ esup1, const int* __restrict__ esup2, const double* __restrict__ area,
        double* __restrict__ M, int npoin) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= npoin) return;
    double m = 0.0;
    for (int s = esup2[i]; s < esup2[i + 1]; ++s) m = m + area[esup1[s] - 1] / 3.0;
    M[i] = m;
}

// mLaplace.f90:120-148, one row per thread; column positions from the slot
// map.  A row of up to kLapRow entries accumulates in LDS (the same sequence
// of additions per entry as in memory), column-major over the block's
// threads so lanes hit distinct banks; longer rows accumulate in memory.  The
// solves' ELL copy is written from the same row (width > 0): a pass over the
// matrix and a launch of 4.8 us less per step.
constexpr int kLapRow = 16;

// row i's contributions in esup order; acc(k) is the accumulator of CSR
// entry r0 + k, the first one the diagonal's; weight(e): the element's weight;
// each(e): the node's other sums
template <class Weight, class Acc, class Each>
__device__ inline void laplace_row(int r0, int s0, int s1, const int* __restrict__ esup1,
                                   const int* __restrict__ lslot, Weight weight,
                                   const double* __restrict__ dNx, const double* __restrict__ dNy,
                                   Acc acc, Each each) {
    for (int s = s0; s < s1; ++s) {
        const int e = esup1[s] - 1;
        int slot[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) slot[j] = lslot[3 * s + j] - r0;
        const int li = slot[0] == 0 ? 0 : slot[1] == 0 ? 1 : 2;  // the row's own node
        const double q = weight(e);
        double nx[3], ny[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            nx[j] = dNx[3 * e + j];
            ny[j] = dNy[3 * e + j];
        }
        const double ax = li == 0 ? nx[0] : li == 1 ? nx[1] : nx[2];
        const double ay = li == 0 ? ny[0] : li == 1 ? ny[1] : ny[2];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            double& a = acc(slot[j]);
            a = a + (ax * nx[j] + ay * ny[j]) * q;
        }
        each(e);
    }
}

// laplace's rows, and the nodes' masses in the same pass over their elements:
// MASAS, or the GCL's update from the terms that k_deriv left; one more block
// folds k_deriv's minima of HH (a launch of 4.7 us less).  Blocks of one wave in XCD
// order (a node's elements are its ring neighbours' too).
//
// Formed from the coordinates, gradients and W per node and element, in launches
// of their own (laplace + GCL / laplace + MASAS), and so, k_deriv's 15 us more for
// the GCL's terms not counted: 4,608 nodes 8.6 + 7.4 / 8.6 + 4.2 us, now 5.7 / 5.6;
// 524,288 nodes 100 + 91 / 100 + 10 us, now 95 / 85 (blocks of 256 in natural order
// 102 / 92, 7.4 us on the small mesh).  Bound by the lines that a node's scattered
// elements share with others: 520 MB are fetched past the L2s for 150 MB of
// tables.  Fewer loads (a packed slot record, the products instead of the
// gradients) and rows staged for coalesced CSR stores left it at 88-92.
constexpr int kLapThreads = 64;
// kMassNone: the host entry, without masses and with the weights formed here from the
// coordinates (one matrix: a pass over the elements before it costs it more)
enum { kMassNone, kMassMasas, kMassGcl };
struct LapWeights {
    const double* w;  // from k_deriv, or (kMassNone) null:
    const int* inpoel;
    const double *X, *Y;
};
template <int kMass>
__global__ void __launch_bounds__(kLapThreads)
k_laplace(const int* __restrict__ esup1, const int* __restrict__ esup2,
          const int* __restrict__ rowptr, const int* __restrict__ lslot,
          LapWeights lw, const double* __restrict__ dNx,
          const double* __restrict__ dNy, double* __restrict__ lap, double* __restrict__ diag,
          int npoin, int width, double* __restrict__ ell, NodeMass m, HminFold h) {
    __shared__ double srow[kLapRow * kLapThreads];
    // the fold is the first block's: on a large mesh it takes longer than a row block
    // and ends beside them instead of behind (33.5M triangles: 2,011 us, as the last
    // block's 2,077, in a launch of its own 2,018 + 29)
    const int nblk = (npoin + kLapThreads - 1) / kLapThreads, fold = h.out ? 1 : 0;
    if ((int)blockIdx.x < fold) {  // subrutinas.f90:124-125: hmin = min(minval(HH), 1e10)
        const double v = combine_partials(h.partials, h.nb, __builtin_huge_val(), OpMin());
        if (threadIdx.x == 0) *h.out = v > 1.0e10 ? 1.0e10 : v;
        return;
    }
    const int i = xcd_block((int)blockIdx.x - fold, nblk) * kLapThreads + threadIdx.x;
    if (i >= npoin) return;
    const int r0 = rowptr[i], len = rowptr[i + 1] - r0, s0 = esup2[i], s1 = esup2[i + 1];
    const auto weight = [&lw](int e) {
        if (kMass != kMassNone) return lw.w[e];
        const int n1 = lw.inpoel[3 * e] - 1, n2 = lw.inpoel[3 * e + 1] - 1, n3 = lw.inpoel[3 * e + 2] - 1;
        return lap_weight(lw.X[n1], lw.X[n2], lw.X[n3], lw.Y[n1], lw.Y[n2], lw.Y[n3]);
    };
    double tot1 = 0.0, tot2 = 0.0;
    auto each = [&](int e) {
        if (kMass == kMassMasas) tot1 = tot1 + m.area[e] / 3.0;  // subrutinas.f90:137-152
        if (kMass == kMassGcl) {  // gcl.f90:218-236
            const double2 g = m.gcl[e];
            tot1 = tot1 + g.x;
            tot2 = tot2 + g.y;
        }
    };
    if (len <= kLapRow) {
        double* sr = srow + threadIdx.x;
        for (int j = 0; j < len; ++j) sr[j * kLapThreads] = 0.0;
        laplace_row(r0, s0, s1, esup1, lslot, weight, dNx, dNy,
                    [sr](int k) -> double& { return sr[k * kLapThreads]; }, each);
        for (int j = 0; j < len; ++j) lap[r0 + j] = sr[j * kLapThreads];
        for (int j = 0; j < width; ++j)
            ell[(size_t)j * npoin + i] = j < len ? sr[j * kLapThreads] : 0.0;
        diag[i] = sr[0];
    } else {
        double* row = lap + r0;
        for (int j = 0; j < len; ++j) row[j] = 0.0;
        laplace_row(r0, s0, s1, esup1, lslot, weight, dNx, dNy,
                    [row](int k) -> double& { return row[k]; }, each);
        for (int j = 0; j < width; ++j) ell[(size_t)j * npoin + i] = j < len ? row[j] : 0.0;
        diag[i] = row[0];
    }
    if (kMass == kMassMasas) m.M[i] = tot1;
    if (kMass == kMassGcl) m.M[i] = m.M[i] + *m.dt * (tot1 + tot2) / 2.0;
}

// gcl.f90:218-236 per node: both divergence sums in ascending element order (the
// host entry, whose gradients come from the caller)
__global__ void __launch_bounds__(kBlock)
k_gcl(const int* __restrict__ inpoel, const int* __restrict__ esup1, const int* __restrict__ esup2,
      double* __restrict__ M, const double* __restrict__ Wx, const double* __restrict__ Wy,
      const double* __restrict__ Wxo, const double* __restrict__ Wyo, const double* __restrict__ dNx,
      const double* __restrict__ dNy, const double* __restrict__ area,
      const double* __restrict__ area_old, const double* __restrict__ dtp, int mode, int npoin) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= npoin) return;
    const double dt = *dtp;
    const double* wy = mode ? Wy : Wx;     // as written, the y-part reads W_x
    const double* wyo = mode ? Wyo : Wxo;
    double tot1 = 0.0, tot2 = 0.0;
    for (int s = esup2[i]; s < esup2[i + 1]; ++s) {
        int e = esup1[s] - 1;
        const int n0 = inpoel[3 * e] - 1, n1 = inpoel[3 * e + 1] - 1, n2 = inpoel[3 * e + 2] - 1;
        const double2 g = gcl_terms(dNx + 3 * e, dNy + 3 * e, n0, n1, n2, Wx, wy, Wxo, wyo, area[e],
                                    area_old[e]);
        tot1 = tot1 + g.x;
        tot2 = tot2 + g.y;
    }
    M[i] = M[i] + dt * (tot1 + tot2) / 2.0;
}

// subrutinas.f90:26-63 per wall node; incident wall edges in ascending order
__global__ void k_normales(int nw, const int* __restrict__ wnode_bc, const int* __restrict__ wnode_ptr,
                           const int* __restrict__ wnode_edges, const int* __restrict__ wall,
                           const double* __restrict__ X, const double* __restrict__ Y,
                           int* __restrict__ flags, double* __restrict__ vals) {
    int w = blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= nw) return;
    double nlx = 0.0, nly = 0.0, den = 0.0;
    for (int q = wnode_ptr[w]; q < wnode_ptr[w + 1]; ++q) {
        int ed = wnode_edges[q];
        int a = wall[2 * ed] - 1, b = wall[2 * ed + 1] - 1;
        double lx = Y[b] - Y[a];
        double ly = -(X[b] - X[a]);
        double l = sqrt(lx * lx + ly * ly);
        nlx = nlx + lx;
        nly = nly + ly;
        den = den + l;
    }
    int bi = wnode_bc[w];
    int f = flags[bi] & ~2;
    if (den > 1.0e-6) {
        double lx = nlx / den, ly = nly / den;
        double ln = sqrt(lx * lx + ly * ly);
        if (ln > 0.2) {
            f |= 2;
            vals[8 * bi + 2] = lx / ln;
            vals[8 * bi + 3] = ly / ln;
        }
    }
    flags[bi] = f;
}

// subrutinas.f90:75-84 on the nodes NORMALES marked (flag bit 1): the
// velocity relative to the mesh keeps its tangential part, then W is added
__global__ void k_normalvel(const int* __restrict__ bcidx, const int* __restrict__ flags,
                            const double* __restrict__ vals, double* __restrict__ VX,
                            double* __restrict__ VY, const double* __restrict__ WX,
                            const double* __restrict__ WY, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int bi = bcidx[i];
    if (bi < 0 || !(flags[bi] & 2)) return;
    const double nx = vals[8 * bi + 2], ny = vals[8 * bi + 3];
    const double vx = VX[i], vy = VY[i], wx = WX[i], wy = WY[i];
    const double p = -ny * (vx - wx) + nx * (vy - wy);
    VX[i] = -ny * p + wx;
    VY[i] = nx * p + wy;
}

// One wave per 64 edges: lane l forms edge 64 b + l, the wave sums the terms
// by a fixed shuffle tree and lane 0 stores the block's five partials at
// part[q * nb + b].
template <bool kPress, bool kVisc>
__global__ void __launch_bounds__(64)
k_forces_part(int nedge, const int* __restrict__ iset, const double* __restrict__ X,
              const double* __restrict__ Y, const double* __restrict__ P, double xref,
              double yref, ViscIn v, double* __restrict__ part) {
    const int nb = gridDim.x, b = blockIdx.x;
    const int i = b * 64 + threadIdx.x;
    double r[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    if (i < nedge) force_terms<kPress, kVisc>(i, iset, X, Y, P, xref, yref, v, r);
#pragma unroll
    for (int q = 0; q < 5; ++q) {
        if (q < 3 && !kPress) continue;
        if (q >= 3 && !kVisc) continue;
        const double t = wave_reduce(r[q], OpSum());
        if (threadIdx.x == 0) part[q * nb + b] = t;
    }
}

// One wave folds the nb block partials: lane l sums partials l, l + 64, ...
// in that order, then the shuffle tree.  zero4 (when given) receives four zeros
// in the same launch (the iteration counts and residuals of mesh solves that
// stop at once on a mesh that does not move).
template <bool kPress, bool kVisc>
__global__ void __launch_bounds__(64)
k_forces_fin(int nb, const double* __restrict__ part, double* __restrict__ out,
             double* __restrict__ outv, double* __restrict__ zero4) {
    const int l = threadIdx.x;
#pragma unroll
    for (int q = 0; q < 5; ++q) {
        if (q < 3 && !kPress) continue;
        if (q >= 3 && !kVisc) continue;
        double a = 0.0;
        for (int k = l; k < nb; k += 64) a = a + part[q * nb + k];
        a = wave_reduce(a, OpSum());
        if (l == 0) {
            if (q < 3)
                out[q] = a;
            else
                outv[q - 3] = a;
        }
    }
    if (zero4 && l < 4) zero4[l] = 0.0;
}

// Both in one block, a wave per 64-edge piece and the pieces' sums in LDS: the
// same trees in the same order, one launch instead of two.  Up to kForcesOne
// pieces (us a step with / without: 128 edges 49.5 / 52.0, 512 edges 93.8 /
// 94.1); above, one CU's gathers take longer than a launch (1,024 edges 232 /
// 226, 2,048 866 / 852).
template <bool kPress, bool kVisc>
__global__ void __launch_bounds__(64 * kForcesOne)
k_forces_one(ForceIn f) {
    forces_block<kPress, kVisc>(f);
}

// meshMove.f90:378-389, one set; kForces: the last block forms FORCES instead (two
// chains of loads side by side: a step of a small moving mesh 4.4 us less)
template <bool kForces>
__global__ void __launch_bounds__(kBlock)
k_transf(int nedge, const int* __restrict__ iset, const double* __restrict__ X,
         const double* __restrict__ Y, const double* __restrict__ cs, double yposr, double xref,
         double yref, double* __restrict__ DXPOS, double* __restrict__ DYPOS, ForceIn forces) {
    if (kForces && blockIdx.x == gridDim.x - 1) {
        forces_block<true, false>(forces);
        return;
    }
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nedge) return;
    const double ca = cs[0], sa = cs[1];
    for (int jj = 0; jj < 2; ++jj) {
        int n = iset[3 * i + jj] - 1;
        double distx = X[n] - xref;
        double disty = Y[n] - yref + yposr;
        DXPOS[n] = ca * distx + sa * disty - distx;
        DYPOS[n] = -(sa * distx) + ca * disty - disty + yposr;
    }
}

}  // namespace

void launch_deriv(const Tables& t, const double* X, const double* Y, double* area, double* dNx,
                  double* dNy, double* HH, double* HHX, double* HHY, double* hmin_out,
                  double* partials, hipStream_t s, const ElemTerms& x) {
    const unsigned g = grid_for(t.nelem);
    const auto kernel = x.gcl ? k_deriv<true> : k_deriv<false>;
    kernel<<<g, kBlock, 0, s>>>(t.inpoel.p, X, Y, area, dNx, dNy, HH, HHX, HHY, t.nelem, partials, x);
    // hmin = minval(HH), capped at 1e10 (subrutinas.f90:124-125)
    if (hmin_out)
        k_min_finalize<<<1, 256, 0, s>>>(partials, (int)g, __builtin_huge_val(), 1.0e10, hmin_out);
    CFD_HIP(hipGetLastError());
}

void launch_masas(const Tables& t, const double* area, double* M, hipStream_t s) {
    k_masas<<<grid_for(t.npoin), kBlock, 0, s>>>(t.esup1.p, t.esup2.p, area, M, t.npoin);
    CFD_HIP(hipGetLastError());
}

static void laplace(const Tables& t, const LapWeights& w, const double* dNx, const double* dNy,
                    double* lap, double* diag, hipStream_t s, EllLap* ell, const NodeMass& m, HminFold h) {
    const auto kernel = m.gcl ? k_laplace<kMassGcl> : m.area ? k_laplace<kMassMasas> : k_laplace<kMassNone>;
    const int nblk = (t.npoin + kLapThreads - 1) / kLapThreads + (h.out ? 1 : 0);
    kernel<<<nblk, kLapThreads, 0, s>>>(t.esup1.p, t.esup2.p, t.rowptr.p, t.lslot.p, w, dNx, dNy, lap,
                                        diag, t.npoin, ell ? ell->width : 0,
                                        ell ? ell->val.p : nullptr, m, h);
    CFD_HIP(hipGetLastError());
}

void launch_laplace(const Tables& t, const double* lapw, const double* dNx, const double* dNy,
                    double* lap, double* diag, hipStream_t s, EllLap* ell, const NodeMass& m, HminFold h) {
    CFD_CHECK(m.area || m.gcl, "internal: laplace with the masses");
    laplace(t, {lapw, nullptr, nullptr, nullptr}, dNx, dNy, lap, diag, s, ell, m, h);
}

void launch_laplace(const Tables& t, const double* X, const double* Y, const double* dNx,
                    const double* dNy, double* lap, double* diag, hipStream_t s) {
    laplace(t, {nullptr, t.inpoel.p, X, Y}, dNx, dNy, lap, diag, s, nullptr, NodeMass{}, HminFold{});
}

void launch_gcl(const Tables& t, double* M, const double* Wx, const double* Wy, const double* Wxo,
                const double* Wyo, const double* dNx, const double* dNy, const double* area,
                const double* area_old, const double* dt, int mode, hipStream_t s) {
    k_gcl<<<grid_for(t.npoin), kBlock, 0, s>>>(t.inpoel.p, t.esup1.p, t.esup2.p, M, Wx, Wy, Wxo, Wyo,
                                               dNx, dNy, area, area_old, dt, mode, t.npoin);
    CFD_HIP(hipGetLastError());
}

void launch_normales(const BcTable& bc, int nw, const int* wnode_bc, const int* wnode_ptr,
                     const int* wnode_edges, const int* wall, const double* X, const double* Y,
                     hipStream_t s) {
    if (nw == 0) return;
    k_normales<<<grid_for(nw), kBlock, 0, s>>>(nw, wnode_bc, wnode_ptr, wnode_edges, wall, X, Y,
                                               bc.flags.p, bc.vals.p);
    CFD_HIP(hipGetLastError());
}

void launch_normalvel(const BcTable& bc, double* VX, double* VY, const double* WX,
                      const double* WY, hipStream_t s) {
    const int n = (int)bc.bcidx.n;
    if (bc.nb == 0 || n == 0) return;
    k_normalvel<<<grid_for(n), kBlock, 0, s>>>(bc.bcidx.p, bc.flags.p, bc.vals.p, VX, VY, WX, WY,
                                               n);
    CFD_HIP(hipGetLastError());
}

size_t forces_part_size(int nedge) { return 5 * (size_t)std::max(1, (nedge + 63) / 64); }

void launch_forces(int nedge, const int* iset, const double* X, const double* Y, const double* P,
                   double xref, double yref, double* out3, const ViscIn* visc, double* out2,
                   double* part, double* zero4, hipStream_t s) {
    if (nedge == 0 || (!out3 && !visc)) {
        if (zero4) {
            k_forces_fin<false, false><<<1, 64, 0, s>>>(0, part, out3, out2, zero4);
            CFD_HIP(hipGetLastError());
        }
        return;
    }
    const ViscIn v = visc ? *visc : ViscIn{};
    const int nb = (nedge + 63) / 64;
    auto go = [&](auto press, auto vis) {
        constexpr bool kP = decltype(press)::value, kV = decltype(vis)::value;
        if (nb <= kForcesOne) {
            k_forces_one<kP, kV><<<1, 64 * std::max(5, nb), 0, s>>>(
                ForceIn{nedge, iset, X, Y, P, xref, yref, v, out3, out2, zero4});
            return;
        }
        k_forces_part<kP, kV><<<nb, 64, 0, s>>>(nedge, iset, X, Y, P, xref, yref, v, part);
        k_forces_fin<kP, kV><<<1, 64, 0, s>>>(nb, part, out3, out2, zero4);
    };
    if (out3 && visc) go(std::true_type{}, std::true_type{});
    else if (out3) go(std::true_type{}, std::false_type{});
    else go(std::false_type{}, std::true_type{});
    CFD_HIP(hipGetLastError());
}

void launch_transf(int nedge, const int* iset, const double* X, const double* Y, const double* cs,
                   double yposr, double xref, double yref, double* DXPOS, double* DYPOS,
                   hipStream_t s, const ForceIn* forces) {
    if (nedge == 0) return;
    const auto kernel = forces ? k_transf<true> : k_transf<false>;
    kernel<<<grid_for(nedge) + (forces ? 1 : 0), kBlock, 0, s>>>(
        nedge, iset, X, Y, cs, yposr, xref, yref, DXPOS, DYPOS, forces ? *forces : ForceIn{});
    CFD_HIP(hipGetLastError());
}

}  // namespace cfd
