// Forces on one edge set: the terms of an edge, and the whole sum by one block.
#pragma once

#include "cfd_internal.hpp"
#include "crmath.hpp"
#include "reduce.hpp"

namespace cfd {
namespace {

// meshMove.f90:167-192 FORCES and ns2DComp.ALE.f90:839-887 FORCE_VISC, one
// set.  FORCE_VISC's traction is that of the full stress tensor (-p I +
// viscous, with the element-average pressure), Sutherland mu at the
// edge-average temperature, on the edge normal (Y2-Y1, -(X2-X1)) / |edge|.
// r = FX, FY, RM, F_VX, F_VY terms of edge i.
template <bool kPress, bool kVisc>
__device__ __forceinline__ void force_terms(int i, const int* __restrict__ iset,
                                            const double* __restrict__ X,
                                            const double* __restrict__ Y,
                                            const double* __restrict__ P, double xref,
                                            double yref, const ViscIn& v, double r[5]) {
    const int n1 = iset[3 * i] - 1, n2 = iset[3 * i + 1] - 1;
    if (kPress) {
        const double d_press = (P[n1] + P[n2]) / 2.0;
        const double rlx = X[n1] - X[n2];
        const double rly = Y[n2] - Y[n1];
        const double dfx = d_press * rly, dfy = d_press * rlx;
        const double xc = (X[n1] + X[n2]) / 2.0;
        const double yc = (Y[n2] + Y[n1]) / 2.0;
        r[0] = dfx;
        r[1] = dfy;
        r[2] = dfy * (xc - xref) - dfx * (yc - yref);
    }
    if (kVisc) {
        const int ie = iset[3 * i + 2] - 1;
        const double temp = (v.T[n1] + v.T[n2]) / 2.0;
        const double smu = 110.0;
        const double fmu = 0.017 * pow_3_2(temp / v.t_inf) * (v.t_inf + smu) / (temp + smu);
        double rly = -(X[n2] - X[n1]);
        double rlx = Y[n2] - Y[n1];
        const double rmod = sqrt(rlx * rlx + rly * rly);
        rlx = rlx / rmod;
        rly = rly / rmod;
        double dux = 0.0, duy = 0.0, dvx = 0.0, dvy = 0.0, press = 0.0;
#pragma unroll
        for (int jj = 0; jj < 3; ++jj) {
            const int nn = v.inpoel[3 * ie + jj] - 1;
            const double nx = v.dNx[3 * ie + jj], ny = v.dNy[3 * ie + jj];
            const double vx = v.VX[nn], vy = v.VY[nn];
            dux = dux + nx * vx;
            duy = duy + ny * vx;
            dvx = dvx + nx * vy;
            dvy = dvy + ny * vy;
            press = press + P[nn];
        }
        press = press / 3.0;
        const double txx = -press - fmu * (2.0 / 3.0 * (dux + dvy) - 2.0 * dux);
        const double txy = fmu * (duy + dvx);
        const double tyy = -press - fmu * (2.0 / 3.0 * (dux + dvy) - 2.0 * dvy);
        r[3] = (txx * rlx + txy * rly) * rmod;
        r[4] = (txy * rlx + tyy * rly) * rmod;
    }
}

// The sums of up to kForcesOne pieces of 64 edges by one block (a multiple of 64
// threads): a wave per piece, then a wave per sum, the trees and the order of
// k_forces_part and k_forces_fin.  Every thread of the block calls it.
template <bool kPress, bool kVisc>
__device__ __forceinline__ void forces_block(const ForceIn& f) {
    __shared__ double part[5][kForcesOne];
    const int nb = (f.nedge + 63) / 64, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int nw = blockDim.x >> 6;
    for (int b = w; b < nb; b += nw) {
        const int i = b * 64 + lane;
        double r[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
        if (i < f.nedge)
            force_terms<kPress, kVisc>(i, f.iset, f.X, f.Y, f.P, f.xref, f.yref, f.v, r);
#pragma unroll
        for (int q = 0; q < 5; ++q) {
            if (q < 3 && !kPress) continue;
            if (q >= 3 && !kVisc) continue;
            const double t = wave_reduce(r[q], OpSum());
            if (lane == 0) part[q][b] = t;
        }
    }
    __syncthreads();
    for (int q = w; q < 5; q += nw) {
        if (!(q < 3 ? kPress : kVisc)) continue;
        double a = 0.0;
        for (int k = lane; k < nb; k += 64) a = a + part[q][k];
        a = wave_reduce(a, OpSum());
        if (lane == 0) {
            if (q < 3) f.out[q] = a;
            else f.outv[q - 3] = a;
        }
    }
    if (f.zero4 && threadIdx.x < 4) f.zero4[threadIdx.x] = 0.0;
}

}  // namespace
}  // namespace cfd
