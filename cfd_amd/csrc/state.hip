// Session state helpers shared by the single-case session and the batch:
// the boundary-condition table, the free-stream start, step control.
#include <map>

#include "cfd_internal.hpp"
#include "reduce.hpp"
#include "stepctl.hpp"

namespace cfd {

namespace {
// free stream (ns2DComp.ALE.f90:409-420) plus the start values of the work arrays
__global__ void k_freestream(double* __restrict__ U, double* __restrict__ U1, double* __restrict__ VX,
                             double* __restrict__ VY, double* __restrict__ T, double* __restrict__ GAMM,
                             double* __restrict__ RHO, double* __restrict__ E, double* __restrict__ WX,
                             double* __restrict__ WY, double rho, double u, double v, double t,
                             double gama, double pamb, int n) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    GAMM[i] = gama;
    double energia = pamb / ((gama - 1.0) * rho) + 0.5 * (u * u + v * v);
    double u4 = energia * rho;
    double4 q = make_double4(rho, rho * u, rho * v, u4);
    reinterpret_cast<double4*>(U)[i] = q;
    reinterpret_cast<double4*>(U1)[i] = q;
    VX[i] = u;
    VY[i] = v;
    T[i] = t;
    RHO[i] = rho;
    E[i] = u4 / rho;
    WX[i] = -0.0;
    WY[i] = 0.0;
}
// Step control (stepctl.hpp).  Block c serves case c: its partials are [pb[c],
// pb[c+1]) (all nb when pb is null), its scalars the X_NCTL slots from ctl_all
// + c * X_NCTL.
__global__ void __launch_bounds__(256)
k_step_ctl(const double* __restrict__ partials, const int* __restrict__ pb, int nb,
           double* __restrict__ ctl_all, StepLaw law) {
    const int cs = blockIdx.x;
    const int b0 = pb ? pb[cs] : 0, b1 = pb ? pb[cs + 1] : nb;
    const double m = combine_partials(partials + b0, b1 - b0, 1.0e20, OpMin());
    if (threadIdx.x != 0) return;
    double* ctl = ctl_all + (size_t)cs * X_NCTL;
    step_control(ctl, m, ctl[CFD_S_DTMIN1], ctl[CFD_S_BANDERA], law);
}

// DT clipped at 10*min(DT) (subrutinas.f90:210-216), then DTL = DTMIN, or
// DTMIN*f + DT*(1-f) with local time stepping (ns2DComp.ALE.f90:158-164);
// element e reads the scalars of case ecase[e] (case 0 when ecase is null)
__global__ void k_dt_finish(double* __restrict__ DT, double* __restrict__ DTL,
                            const double* __restrict__ ctl_all, const int* __restrict__ ecase,
                            int blend, int n) {
    int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n) return;
    const double* ctl = ctl_all + (ecase ? (size_t)ecase[e] * X_NCTL : 0);
    const double cota = 10.0 * ctl[X_RAW], dtmin = ctl[CFD_S_DTMIN];
    double d = DT[e];
    if (d > cota) {
        d = cota;
        DT[e] = d;
    }
    if (blend) {
        const double f = ctl[X_FDTL];
        DTL[e] = dtmin * f + d * (1.0 - f);
    } else {
        DTL[e] = dtmin;
    }
}

// One thread per entity.  Bound by the scattered side (32-byte records of U
// fill a memory sector each): U of 2,097,152 nodes 64 MB in, 64 MB out.  In
// place of a loop on the host, which took 20 of the 24 ms of reading U; up to
// kRenumberHost doubles the loop takes less than the launch (us a read of U by the
// loop / so: 1,152 nodes 26 / 39, 8,192 27 / 34, 16,000 48 / 44, 32,768 111 / 79).
constexpr size_t kRenumberHost = 40000;
template <int W, bool kScatter>
void renumber_host_w(const double* in, double* out, const int* map, int n) {
    for (int i = 0; i < n; ++i) {
        const size_t a = W * (size_t)(kScatter ? i : map[i]), b = W * (size_t)(kScatter ? map[i] : i);
        for (int c = 0; c < W; ++c) out[b + c] = in[a + c];
    }
}
template <bool kScatter>
void renumber_host(const double* in, double* out, const FieldMap& m) {
    if (m.w == 4) renumber_host_w<4, kScatter>(in, out, m.host, m.n);
    else if (m.w == 3) renumber_host_w<3, kScatter>(in, out, m.host, m.n);
    else renumber_host_w<1, kScatter>(in, out, m.host, m.n);
}
template <int W, bool kScatter>
__global__ void k_renumber(const double* __restrict__ in, double* __restrict__ out,
                           const int* __restrict__ map, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const size_t a = kScatter ? i : map[i], b = kScatter ? map[i] : i;
    if constexpr (W == 4) {
        reinterpret_cast<double4*>(out)[b] = reinterpret_cast<const double4*>(in)[a];
    } else {
#pragma unroll
        for (int c = 0; c < W; ++c) out[W * b + c] = in[W * a + c];
    }
}

template <bool kScatter>
void renumber(const double* in, double* out, const int* map, int n, int w, hipStream_t s) {
    if (n <= 0) return;
    const unsigned g = grid_for(n);
    if (w == 4) k_renumber<4, kScatter><<<g, kBlock, 0, s>>>(in, out, map, n);
    else if (w == 3) k_renumber<3, kScatter><<<g, kBlock, 0, s>>>(in, out, map, n);
    else k_renumber<1, kScatter><<<g, kBlock, 0, s>>>(in, out, map, n);
    CFD_HIP(hipGetLastError());
}

}  // namespace

void read_field(const double* state, double* host, const FieldMap& m, FieldStage& st, hipStream_t s) {
    const size_t n = (size_t)m.n * m.w;
    if (n <= kRenumberHost) {
        std::vector<double> tmp(n);
        CFD_HIP(hipMemcpyAsync(tmp.data(), state, sizeof(double) * n, hipMemcpyDeviceToHost, s));
        CFD_HIP(hipStreamSynchronize(s));
        renumber_host<true>(tmp.data(), host, m);
        return;
    }
    std::lock_guard<std::mutex> hold(st.mu);
    double* out = st.room(n);
    renumber<true>(state, out, m.dev, m.n, m.w, s);
    CFD_HIP(hipMemcpyAsync(host, out, sizeof(double) * n, hipMemcpyDeviceToHost, s));
    CFD_HIP(hipStreamSynchronize(s));
}

void write_field(const double* host, double* state, const FieldMap& m, FieldStage& st, hipStream_t s) {
    const size_t n = (size_t)m.n * m.w;
    if (n <= kRenumberHost) {
        std::vector<double> tmp(n);
        renumber_host<false>(host, tmp.data(), m);
        CFD_HIP(hipMemcpyAsync(state, tmp.data(), sizeof(double) * n, hipMemcpyHostToDevice, s));
        CFD_HIP(hipStreamSynchronize(s));
        return;
    }
    std::lock_guard<std::mutex> hold(st.mu);
    double* in = st.room(n);
    CFD_HIP(hipMemcpyAsync(in, host, sizeof(double) * n, hipMemcpyHostToDevice, s));
    renumber<false>(in, state, m.dev, m.n, m.w, s);
    CFD_HIP(hipStreamSynchronize(s));
}

// ---------------------------------------------------------------------------
// Boundary-condition table (host construction, reference list semantics)
// ---------------------------------------------------------------------------


BcHost build_bc_host(int npoin, const cfd_bc_lists* bc) {
    BcHost h;
    h.bcidx.assign(npoin, -1);
    auto entry = [&](int node) -> int {
        CFD_CHECK(node >= 1 && node <= npoin, "boundary list node id out of range");
        int& b = h.bcidx[node - 1];
        if (b < 0) {
            b = (int)h.nodes.size();
            h.nodes.push_back(node);
            h.flags.push_back(0);
            h.vals.insert(h.vals.end(), 8, 0.0);
        }
        return b;
    };
    if (!bc) return h;
    for (int i = 0; i < bc->nfixv; ++i) {           // FIXVEL: last occurrence wins
        int b = entry(bc->ifixv_node[i]);
        h.flags[b] |= 1;
        h.vals[8 * b + 0] = bc->rfixv_valuex[i];
        h.vals[8 * b + 1] = bc->rfixv_valuey[i];
    }
    for (int i = 0; i < bc->nfixrho; ++i) {
        int b = entry(bc->ifixrho_node[i]);
        h.flags[b] |= 4;
        h.vals[8 * b + 4] = bc->rfixrho_value[i];
    }
    for (int i = 0; i < bc->nfixt; ++i) {
        int b = entry(bc->ifixt_node[i]);
        h.flags[b] |= 8;
        h.vals[8 * b + 5] = bc->rfixt_value[i];
    }
    // wall nodes: incident edges in ascending edge order (NORMALES sums)
    std::map<int, std::vector<int>> inc;
    for (int e = 0; e < bc->nwall; ++e)
        for (int j = 0; j < 2; ++j) inc[bc->wall[2 * e + j]].push_back(e);
    h.wnode_ptr.push_back(0);
    for (auto& kv : inc) {
        int b = entry(kv.first);
        h.wnode_bc.push_back(b);
        for (int e : kv.second) h.wnode_edges.push_back(e);
        h.wnode_ptr.push_back((int)h.wnode_edges.size());
    }
    return h;
}

Consts consts_of(const cfd_consts* c) {
    Consts k;
    k.gama = c->gama; k.fr = c->fr; k.fmu = c->fmu; k.fk = c->fk; k.fcv = c->fcv;
    k.t_inf = c->t_inf; k.rho_inf = c->rho_inf; k.u_inf = c->u_inf; k.v_inf = c->v_inf;
    k.cte = c->cte; k.fsafe = c->fsafe;
    return k;
}

void launch_freestream(const NodeState& ns, const Consts& c, int n, hipStream_t s) {
    if (n <= 0) return;
    const double pamb = c.rho_inf * c.fr * c.t_inf;
    k_freestream<<<grid_for(n), kBlock, 0, s>>>(ns.U, ns.U1, ns.VX, ns.VY, ns.T, ns.GAMM, ns.RHO, ns.E,
                                               ns.WX, ns.WY, c.rho_inf, c.u_inf, c.v_inf, c.t_inf,
                                               c.gama, pamb, n);
    CFD_HIP(hipGetLastError());
}

void launch_step_ctl(const double* partials, const int* pb, int nb, double* ctl, int ncases,
                     int itlocal, int motion, double amp, double omega, hipStream_t s) {
    k_step_ctl<<<ncases, 256, 0, s>>>(partials, pb, nb, ctl, StepLaw{itlocal, motion, amp, omega});
    CFD_HIP(hipGetLastError());
}

void launch_dt_finish(double* DT, double* DTL, const double* ctl, const int* ecase, bool blend,
                      int nelem, hipStream_t s) {
    k_dt_finish<<<grid_for(nelem), kBlock, 0, s>>>(DT, DTL, ctl, ecase, blend ? 1 : 0, nelem);
    CFD_HIP(hipGetLastError());
}

}  // namespace cfd
