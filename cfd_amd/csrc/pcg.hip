// Jacobi-preconditioned CG of biconjGrad.f90:8-62 (named biCG there).
//
// Reference sequence (one solve):
//   x(fix) = x_fix; y = A x; y(fix) = 1e30 x(fix); r = b - y; r(fix) = 0
//   if r.r < tol: return
//   p = r/diag; e = r.p; y = A p (fix rows 1e30 p); alfa = e/p.y; x += alfa p
//   while |e_old| > tol and k < 1000:
//     k++; r -= alfa y; z = r/diag; e = r.z; beta = e/e_old; p = beta p + z
//     y = A p (fix rows 1e30 p); alfa = e/p.y; x += alfa p; e_old = e
//
// On the device one iteration is two full-grid kernels:
//   A (k_cg_a): alfa and the loop test; x += alfa p, r -= alfa y, z = r/diag,
//      block partials of r.z;
//   B (k_cg_b): beta; each row forms p_new = beta p_old + z for its columns on
//      the fly, y = A p_new, stores its own p_new (double-buffered p), block
//      partials of p.y.
// Every block of A (of B) first combines the p.y (the r.z) partials that the
// kernel before left, all in the same fixed order, so each has the scalars it
// needs without a launch of its own for them; the first block stores them for
// the kernels after (no kernel reads a scalar that it writes).  Above
// kFoldMax partials a one-block kernel per scalar combines them instead.
//
// x is read and written in every second iteration only: p is double-buffered,
// so A still has the previous iteration's p and adds both updates, in order,
// at once (the same operations on every x; half of x's traffic).
//
// The scalars live in device memory.  Kernels queued after a loop has ended
// return at once (done flag), so the host queues batches of iterations
// between polls.  Several independent systems on one matrix (the x and y mesh
// solves) run interleaved and share the polls.  Dot products combine block
// partials in a fixed tree, so the iteration sequence is deterministic (not
// the serial summation order of the reference).
//
// Two systems on one matrix (the x and y mesh solves) iterate in lockstep:
// one launch per kernel for both, each matrix entry read once for both
// products, and row blocks in XCD order (xcd_block: a row's neighbours' blocks
// mostly on the same XCD).  Partials belong to logical blocks of 256 rows
// whatever the launch shape, so a system's iterates do not depend on whether
// it runs alone or in a pair, nor on its blocks' size; a system that has
// finished is skipped inside the paired kernels.
//
// Small systems run a whole solve in one launch instead (k_cg_whole).
//
// Relative mode (rel = 1): the two tests use tol^2 times the r.r and r.z of
// the residual of the guess that is zero off the fixed nodes, so the stopping
// point does not depend on the initial guess (warm starts compare at equal
// tolerance).
#include <mutex>
#include <type_traits>

#include "cfd_internal.hpp"
#include "reduce.hpp"

namespace cfd {
namespace {

// scal[] slots
enum {
    S_ALFA = 0, S_BETA, S_EOLD, S_ENEW, S_PY, S_RR, S_K, S_DONE, S_STOP, S_CONV, S_TOL, S_MAXIT,
    S_TOLR, S_TOLZ, S_ALFA0, S_NSCAL = 16
};

// The CSR entries of a block's rows [i0, i1) are one contiguous range
// [rowptr[i0], rowptr[i1]).  They are staged through LDS in chunks with
// coalesced loads; each row then visits its own entries in order,
// f(a_ij, column j (0-based)).  Every thread of the block must call this
// (rows without work pass an empty range b == e).
constexpr int kSpChunk = 2048;

template <class F>
__device__ inline void staged_rows(const double* __restrict__ A, const int* __restrict__ idx,
                                   int s0, int s1, int b, int e, double* sA, int* sI, F f) {
    for (int c0 = s0; c0 < s1; c0 += kSpChunk) {
        const int c1 = min(c0 + kSpChunk, s1);
        __syncthreads();
        for (int q = c0 + (int)threadIdx.x; q < c1; q += (int)blockDim.x) {
            sA[q - c0] = A[q];
            sI[q - c0] = idx[q] - 1;
        }
        __syncthreads();
        const int lo = max(b, c0), hi = min(e, c1);
        for (int j = lo; j < hi; ++j) f(sA[j - c0], sI[j - c0]);
    }
}

// One system of a launch (the kernels take one or two)
struct CgSys {
    double *x, *r, *z, *y, *scal;
    double *prr, *prz, *ppy;  // block partials: residual (3 nb), r.z, p.y
    const double* p;  // the current p
    double* pother;   // the other buffer: the p before in A, the next p in B
    unsigned char* fixflag;
    const double *b, *x_fix;
    const int* fix_idx;
    int nfix;
};
// NS systems of a block: both of a pair (NS = 2), or the one of the block's
// grid row (NS = 1, blockIdx.y)
struct CgBoth {
    CgSys s[2];
};
template <int NS>
struct CgArgs {
    CgSys s[NS];
    __device__ __forceinline__ explicit CgArgs(const CgBoth& b) {
        if (NS == 1) {
            s[0] = b.s[blockIdx.y];
        } else {
            s[0] = b.s[0];
            s[NS - 1] = b.s[1];
        }
    }
};

// The sums of NS arrays of nb block partials, in the order of
// combine_partials on one block of 256 threads (thread t adds partials t, t +
// 256, ... to 0, then the waves' trees, then the waves in order), known to
// every thread.  Blocks of 512 threads or more give each array its own 256
// threads; smaller ones (256) add the arrays side by side.  nb <= kFoldMax.
constexpr int kFoldSmall = 1024, kFoldMid = 2048, kFoldMax = 3072;
// Loads of the partials, issued before the caller's own loads so that the sum
// waits for nothing else.  Blocks of 256 threads: every thread its own
// partials of every array; blocks of 1024: every thread a quarter of them,
// handed over through LDS (12 loads in 24 registers a thread would cost the
// kernels a wave per SIMD).
template <int kG, int NS>
struct Fold {
    static constexpr int kMax = kG == 1 ? kFoldSmall : kG == 2 ? kFoldMid : kFoldMax;
    static constexpr int kL = kMax / (kG * kBlock);
    double v[NS][kL];
    __device__ __forceinline__ void load(const double* part0, const double* part1, int nb) {
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            const double* p = k == 0 ? part0 : part1;
#pragma unroll
            for (int q = 0; q < kL; ++q) {
                const int j = threadIdx.x + q * kG * kBlock;
                v[k][q] = j < nb ? p[j] : 0.0;
            }
        }
    }
    // out[k]: the sum of array k
    __device__ __forceinline__ void sum(int nb, double (&out)[NS]) {
        __shared__ double sh[NS][kBlock / 64];
        const int t = threadIdx.x & (kBlock - 1), g = threadIdx.x / kBlock;
        if constexpr (kG == 1) {
#pragma unroll
            for (int k = 0; k < NS; ++k) {
                double acc = 0.0;
#pragma unroll
                for (int q = 0; q < kL; ++q)
                    if (t + q * kBlock < nb) acc = acc + v[k][q];
                acc = wave_reduce(acc, OpSum());
                if ((t & 63) == 0) sh[k][t >> 6] = acc;
            }
        } else {
            __shared__ double sp[NS][kMax];
#pragma unroll
            for (int k = 0; k < NS; ++k)
#pragma unroll
                for (int q = 0; q < kL; ++q) sp[k][threadIdx.x + q * kG * kBlock] = v[k][q];
            __syncthreads();
            if (g < NS) {  // 256 threads per array
                double acc = 0.0;
#pragma unroll
                for (int q = 0; q < kMax / kBlock; ++q)
                    if (t + q * kBlock < nb) acc = acc + sp[g][t + q * kBlock];
                acc = wave_reduce(acc, OpSum());
                if ((t & 63) == 0) sh[g][t >> 6] = acc;
            }
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            double s = sh[k][0];
#pragma unroll
            for (int w = 1; w < kBlock / 64; ++w) s = s + sh[k][w];
            out[k] = s;
        }
    }
};

// Partials of NS values per row (block_partial's tree per 256 rows): one per
// logical block lb0 .. lb0 + kG - 1.  Every thread of the block calls this.
template <int kG, int NS>
__device__ __forceinline__ void cg_partials(const double (&v)[NS], double* const (&part)[NS],
                                            int lb0, int nb) {
    __shared__ double sh[NS][kG * (kBlock / 64)];
    const int t = threadIdx.x;
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        const double w = wave_reduce(v[k], OpSum());
        if ((t & 63) == 0) sh[k][t >> 6] = w;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        const int g = t - 64 * k;  // wave k stores system k's
        if (g < 0 || g >= kG || !part[k] || lb0 + g >= nb) continue;
        double s = sh[k][g * (kBlock / 64)];
#pragma unroll
        for (int w = 1; w < kBlock / 64; ++w) s = s + sh[k][g * (kBlock / 64) + w];
        part[k][lb0 + g] = s;
    }
}

// fixflag = 0; scalars reset (block 0)
template <int NS>
__global__ void k_cg_init(int n, CgBoth sys, double tol, int maxit) {
    const CgArgs<NS> a(sys);
    int i = blockIdx.x * blockDim.x + threadIdx.x;
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        if (i < n) a.s[k].fixflag[i] = 0;
        if (i < S_NSCAL)
            a.s[k].scal[i] = i == S_TOL ? tol : i == S_MAXIT ? (double)maxit : 0.0;
    }
}

template <int NS>
__global__ void k_cg_fix(CgBoth sys) {
    const CgArgs<NS> a(sys);
    int q = blockIdx.x * blockDim.x + threadIdx.x;
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        if (q >= a.s[k].nfix) continue;
        int i = a.s[k].fix_idx[q] - 1;
        a.s[k].fixflag[i] = 1;
        a.s[k].x[i] = 1.0 * a.s[k].x_fix[q];
    }
}

// The matrix rows of a kernel: f(a_ij, column j (0-based)) over row i's
// entries in CSR order, from the CSR arrays (staged; every thread of the
// block calls it, rows without work with on = false) or the ELL copy.
struct CsrRows {
    static constexpr bool kFew = false, kMany = false, kAlone = false;
    const double* A;
    const int *idx, *rowptr;
    template <class F>
    __device__ __forceinline__ void visit(int n, int i0, int i, bool on, F f) const {
        __shared__ double sA[kSpChunk];
        __shared__ int sI[kSpChunk];
        staged_rows(A, idx, rowptr[i0], rowptr[min(i0 + (int)blockDim.x, n)], on ? rowptr[i] : 0,
                    on ? rowptr[i + 1] : 0, sA, sI, f);
    }
    template <int NS>
    struct Ahead {  // nothing is loaded ahead
        __device__ __forceinline__ void load(const CsrRows&, int, int, const CgArgs<NS>&, int) {}
        __device__ __forceinline__ void dots(const CsrRows& m, int n, int i0, int i, bool work,
                                             const bool (&row)[NS], const CgArgs<NS>& a, int first,
                                             const double (&beta)[NS], double (&dot)[NS]) const {
            m.visit(n, i0, i, work, [&](double aij, int c) {
#pragma unroll
                for (int k = 0; k < NS; ++k) {
                    if (!row[k]) continue;
                    const double pc = first ? a.s[k].z[c] : beta[k] * a.s[k].p[c] + a.s[k].z[c];
                    dot[k] = dot[k] + aij * pc;
                }
            });
        }
    };
};
// kW: most entries of a row; kShort: columns as 16-bit distances from the
// row; kAhead: k_cg_b loads the entries (1), and gathers their p and z too
// (2), ahead of the scalars.  The rows that with_rows takes each form for leave some
// kernels without use: kFew: up to kFoldSmall partials, kMany: above, kAlone: a pair
// of systems never shares a thread
template <int kW, bool kShort, int kAhead>
struct EllRows {
    EllMat m;
    static constexpr bool kDeep = kAhead == 2, kFew = kAhead > 0, kAlone = kDeep;
    static constexpr bool kMany = kW == 8 && kShort && kAhead == 0;
    template <class F>
    __device__ __forceinline__ void visit(int n, int, int i, bool on, F f) const {
        if (!on) return;
        const int l = m.len[i];
#pragma unroll
        for (int k = 0; k < kW; ++k) {
            if (k < l) {
                const size_t q = (size_t)k * n + i;
                f(m.val[q], kShort ? i + (int)m.dcol[q] : m.col[q]);
            }
        }
    }
    // k_cg_b's entries of row i, loaded ahead of the scalars (slots beyond a
    // row's length hold 0 and the row's own column, and are not added)
    template <int NS>
    struct Ahead {
        int len, col[kW];
        double val[kW];
        double p[kDeep ? NS : 1][kDeep ? kW : 1], z[kDeep ? NS : 1][kDeep ? kW : 1];
        __device__ __forceinline__ void load(const EllRows& r, int n, int i, const CgArgs<NS>& a,
                                             int first) {
            if constexpr (kAhead == 0) return;
            len = r.m.len[i];
#pragma unroll
            for (int j = 0; j < kW; ++j) {
                if (j >= r.m.width) continue;
                const size_t q = (size_t)j * n + i;
                val[j] = r.m.val[q];
                col[j] = kShort ? i + (int)r.m.dcol[q] : r.m.col[q];
            }
            if constexpr (kDeep) {
#pragma unroll
                for (int j = 0; j < kW; ++j) {
                    if (j >= r.m.width) continue;
#pragma unroll
                    for (int k = 0; k < NS; ++k) {
                        z[k][j] = a.s[k].z[col[j]];
                        if (!first) p[k][j] = a.s[k].p[col[j]];
                    }
                }
            }
        }
        __device__ __forceinline__ void dots(const EllRows& r, int n, int, int i, bool work,
                                             const bool (&row)[NS], const CgArgs<NS>& a, int first,
                                             const double (&beta)[NS], double (&dot)[NS]) const {
            if (!work) return;
            const int len = kAhead ? this->len : (int)r.m.len[i];
#pragma unroll
            for (int j = 0; j < kW; ++j) {
                if (j >= len) continue;
                const size_t q = (size_t)j * n + i;
                const double aij = kAhead ? val[j] : r.m.val[q];
                const int c = kAhead ? col[j] : kShort ? i + (int)r.m.dcol[q] : r.m.col[q];
#pragma unroll
                for (int k = 0; k < NS; ++k) {
                    if (!row[k]) continue;
                    double zc, pc = 0.0;
                    if constexpr (kDeep) {
                        zc = z[k][j];
                        pc = first ? zc : beta[k] * p[k][j] + zc;
                    } else {
                        zc = a.s[k].z[c];
                        pc = first ? zc : beta[k] * a.s[k].p[c] + zc;
                    }
                    dot[k] = dot[k] + aij * pc;
                }
            }
        }
    };
};

// r = -1*(A x) + b with fixed rows y = 1e30 x and r(fix) = 0; partials of r.r
// and, in relative mode, of rd.rd and rd.(rd/diag) for the residual rd of the
// guess that is zero off the fixed nodes.  kFirst: the first preconditioned
// residual too, z = r/diag with the partials of r.z (used only when the first
// test does not end the solve; a launch of its own for it costs 4.5 us)
template <class Rows, int NS, bool kFirst>
__global__ void __launch_bounds__(kBlock)
k_cg_residual(int n, Rows rows, const double* __restrict__ diag, CgBoth sys, int rel, int nb) {
    const CgArgs<NS> a(sys);
    const int lb = xcd_block(blockIdx.x, gridDim.x);
    const int i0 = lb * kBlock, i = i0 + threadIdx.x;
    const bool act = i < n;
    bool row[NS], any = false;
    double dot[NS], dotd[NS];
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        row[k] = act && !a.s[k].fixflag[i];
        any = any || row[k];
        dot[k] = dotd[k] = 0.0;
    }
    rows.visit(n, i0, i, any, [&](double aij, int c) {
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            if (!row[k]) continue;
            const double xc = a.s[k].x[c];
            dot[k] = dot[k] + aij * xc;
            if (rel && a.s[k].fixflag[c]) dotd[k] = dotd[k] + aij * xc;
        }
    });
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        const CgSys& q = a.s[k];
        double v = 0.0, vdr = 0.0, vdz = 0.0, vz = 0.0;
        if (act) {
            double ri = 0.0;
            if (row[k]) {
                ri = -1.0 * dot[k] + q.b[i];
                if (rel) {
                    const double rd = -1.0 * dotd[k] + q.b[i];
                    vdr = rd * rd;
                    vdz = rd * (rd / diag[i]);
                }
            }
            q.r[i] = ri;
            v = ri * ri;
            if (kFirst) {
                const double zi = ri / diag[i];
                q.z[i] = zi;
                vz = ri * zi;
            }
        }
        block_partial(v, OpSum(), q.prr, lb);
        if (kFirst) block_partial(vz, OpSum(), q.prz, lb);
        if (rel) {
            block_partial(vdr, OpSum(), q.prr + nb, lb);
            block_partial(vdz, OpSum(), q.prr + 2 * nb, lb);
        }
    }
}

// The first residual test.  A residual that is exactly zero ends the solve too: in
// relative mode the threshold is zero where the residual that it refers to is (no
// fixed node displaced and b = 0, or every row fixed).
__device__ __forceinline__ bool cg_solved(double rr, double tolr) { return rr < tolr || rr == 0.0; }
// The step length e / p.y; none where a residual that has become exactly zero has
// left no direction (p and p.y are zero then, or underflowed to it).
__device__ __forceinline__ double cg_step(double e, double py) { return py == 0.0 ? 0.0 : e / py; }

// the first residual test (block k: system k)
__global__ void __launch_bounds__(256)
k_cg_test(CgBoth a, int nb, int rel) {
    const CgSys& q = a.s[blockIdx.x];
    const double rr = combine_partials(q.prr, nb, 0.0, OpSum());
    double dr = 0.0, dz = 0.0;
    if (rel) {
        dr = combine_partials(q.prr + nb, nb, 0.0, OpSum());
        dz = combine_partials(q.prr + 2 * nb, nb, 0.0, OpSum());
    }
    if (threadIdx.x == 0) {
        double* scal = q.scal;
        const double tol = scal[S_TOL];
        const double tolr = rel ? tol * tol * dr : tol;
        const double tolz = rel ? tol * tol * dz : tol;
        scal[S_TOLR] = tolr;
        scal[S_TOLZ] = tolz;
        scal[S_RR] = rr;
        if (cg_solved(rr, tolr)) {
            scal[S_DONE] = 1.0;
            scal[S_CONV] = 1.0;
            scal[S_EOLD] = rr;
        }
    }
}

// The scalars a kernel starts from
struct CgScalars {
    double alfa, alfa0, beta, eold, enew, k, done, stop, maxit, tolz;
    __device__ __forceinline__ void load(const double* scal) {
        alfa = scal[S_ALFA];
        alfa0 = scal[S_ALFA0];
        beta = scal[S_BETA];
        eold = scal[S_EOLD];
        enew = scal[S_ENEW];
        k = scal[S_K];
        done = scal[S_DONE];
        stop = scal[S_STOP];
        maxit = scal[S_MAXIT];
        tolz = scal[S_TOLZ];
    }
};

// A's step length, and whether the loop goes on
__device__ __forceinline__ double cg_alfa(const CgScalars& c, double py, bool& more) {
    more = fabs(c.enew) > c.tolz && c.k < c.maxit;
    return cg_step(c.enew, py);
}

// Kernel A of an iteration (see the file header).  both: x takes the previous
// iteration's update and this one's; else x is left for the next iteration,
// unless this is the last.  kFold: the p.y partials are combined here, else
// k_cg_fin_b has left alfa and the loop test.
//
// An iteration of one system / two in A and B, with the one-block kernels and x
// in every iteration before and now (us): 32,768 rows 15.2 / 17 -> 9.4 / 10.5;
// 131,072 rows 17.5 / 20.7 -> 11.0 / 12.9; 524,288 rows 27 / 38 -> 19.9 / 31.
// What bounds it: below 131,072 rows the launches and one chain of dependent
// loads in each kernel; above, the bytes (A 56 a row and system on average, B
// 103 with the matrix, from the Infinity Cache at 524,288 rows: A 7.8 us, B 12.2).
template <int kG, int NS, bool kFold>
__global__ void __launch_bounds__(kG * kBlock)
k_cg_a(int n, const double* __restrict__ diag, CgBoth sys, int nb, int both) {
    const CgArgs<NS> a(sys);
    const int pb = xcd_block(blockIdx.x, gridDim.x);
    const int i = pb * (kG * kBlock) + threadIdx.x;
    // every load of the kernel is issued before the first wait: the partials,
    // the rows' own values, the scalars
    Fold<kG, NS> fold;
    if (kFold) fold.load(a.s[0].ppy, a.s[NS - 1].ppy, nb);
    double p[NS], y[NS], r[NS], x[NS], p0[NS], d = 1.0;
    if (i < n) {
        d = diag[i];
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            const CgSys& q = a.s[k];
            y[k] = q.y[i];
            r[k] = q.r[i];
            if (both) {
                p[k] = q.p[i];
                p0[k] = q.pother[i];
                x[k] = q.x[i];
            }
        }
    }
    CgScalars sc[NS];
    bool on[NS], any = false;
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        sc[k].load(a.s[k].scal);
        on[k] = sc[k].done == 0.0;
        any = any || on[k];
    }
    if (!any) return;  // uniform over the grid
    double alfa[NS], py[NS];
    bool stop[NS];
    if (kFold) fold.sum(nb, py);
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        if (kFold) {
            bool more;
            alfa[k] = cg_alfa(sc[k], py[k], more);
            stop[k] = !more;
        } else {
            alfa[k] = sc[k].alfa;
            stop[k] = sc[k].stop != 0.0;
        }
    }
    double v[NS];
    double* part[NS];
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        const CgSys& q = a.s[k];
        v[k] = 0.0;
        part[k] = on[k] && !stop[k] ? q.prz : nullptr;
        if (!on[k]) continue;
        if (kFold && pb == 0 && threadIdx.x == 0) {
            q.scal[S_PY] = py[k];
            q.scal[S_EOLD] = sc[k].enew;
            if (!both) q.scal[S_ALFA0] = alfa[k];
            if (stop[k]) q.scal[S_STOP] = 1.0;
        }
        if (i >= n) continue;
        if (both) q.x[i] = alfa[k] * p[k] + (sc[k].alfa0 * p0[k] + x[k]);
        else if (stop[k]) q.x[i] = alfa[k] * q.p[i] + q.x[i];
        if (stop[k]) continue;  // the loop test failed: only the last x update remained
        const double ri = -alfa[k] * y[k] + r[k];
        q.r[i] = ri;
        const double zi = ri / d;
        q.z[i] = zi;
        v[k] = ri * zi;
    }
    cg_partials<kG, NS>(v, part, pb * kG, nb);
}

// Kernel B: p_new = beta p_old + z on the fly (first: p_new = z), y = A p_new.
// kFold: the r.z partials are combined here, else k_cg_fin_a has left beta.
// As in A every load that depends on no other kernel's scalar is issued
// before the first wait; with kDeep the gathered p and z of all entries too
// (blocks of one per CU: nothing else hides their latency).
template <int kG, class Rows, int NS, bool kFold>
__global__ void __launch_bounds__(kG * kBlock) __attribute__((amdgpu_waves_per_eu(kG > 1 ? 8 : 1)))
k_cg_b(int n, Rows rows, CgBoth sys, int nb, int first) {
    const CgArgs<NS> a(sys);
    const int pb = xcd_block(blockIdx.x, gridDim.x);
    const bool lead = pb == 0 && threadIdx.x == 0;
    const int i0 = pb * (kG * kBlock), i = i0 + threadIdx.x;
    const bool act = i < n;
    Fold<kG, NS> fold;
    if (kFold) fold.load(a.s[0].prz, a.s[NS - 1].prz, nb);
    typename Rows::template Ahead<NS> ahead;
    ahead.load(rows, n, act ? i : n - 1, a, first);
    bool fixed[NS];
    double zi[NS], pi[NS];
    if (act) {
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            fixed[k] = a.s[k].fixflag[i];
            zi[k] = a.s[k].z[i];
            if (!first) pi[k] = a.s[k].p[i];
        }
    }
    CgScalars sc[NS];
    bool on[NS], any = false;
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        sc[k].load(a.s[k].scal);
        on[k] = sc[k].done == 0.0 && sc[k].stop == 0.0;
        any = any || on[k];
        if (kFold && lead && sc[k].stop != 0.0 && sc[k].done == 0.0) {
            a.s[k].scal[S_CONV] = fabs(sc[k].eold) > sc[k].tolz ? 0.0 : 1.0;
            a.s[k].scal[S_DONE] = 1.0;  // read by the other blocks only beside STOP
        }
    }
    if (!any) return;  // uniform over the grid
    bool row[NS], work = false;
    double beta[NS], e[NS], dot[NS];
    if (kFold) fold.sum(nb, e);
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        row[k] = on[k] && act && !fixed[k];
        work = work || row[k];
        dot[k] = 0.0;
        beta[k] = kFold ? (first ? 0.0 : e[k] / sc[k].eold) : sc[k].beta;
        if (kFold && lead && on[k]) {
            double* scal = a.s[k].scal;
            scal[S_ENEW] = e[k];
            if (!first) {
                scal[S_BETA] = beta[k];
                scal[S_K] = sc[k].k + 1.0;
            }
        }
    }
    ahead.dots(rows, n, i0, i, work, row, a, first, beta, dot);
    double v[NS];
    double* part[NS];
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        const CgSys& q = a.s[k];
        v[k] = 0.0;
        part[k] = on[k] ? q.ppy : nullptr;
        if (!on[k] || !act) continue;
        const double pn = first ? zi[k] : beta[k] * pi[k] + zi[k];
        const double yi = row[k] ? dot[k] : 1.0e30 * pn;
        q.pother[i] = pn;
        q.y[i] = yi;
        v[k] = pn * yi;
    }
    cg_partials<kG, NS>(v, part, pb * kG, nb);
}

// The scalars between A and B, and between B and A, of systems with more than
// kFoldMax partials: block k combines system k's
__global__ void __launch_bounds__(256)
k_cg_fin_a(CgBoth a, int nb, int first) {
    const CgSys& q = a.s[blockIdx.x];
    double* scal = q.scal;
    if (scal[S_DONE] != 0.0) return;
    if (scal[S_STOP] != 0.0) {
        if (threadIdx.x == 0) {
            scal[S_DONE] = 1.0;
            scal[S_CONV] = fabs(scal[S_EOLD]) > scal[S_TOLZ] ? 0.0 : 1.0;
        }
        return;
    }
    const double e = combine_partials(q.prz, nb, 0.0, OpSum());
    if (threadIdx.x == 0) {
        scal[S_ENEW] = e;
        if (first) return;
        scal[S_K] = scal[S_K] + 1.0;
        scal[S_BETA] = e / scal[S_EOLD];
    }
}

__global__ void __launch_bounds__(256)
k_cg_fin_b(CgBoth a, int nb) {
    const CgSys& q = a.s[blockIdx.x];
    double* scal = q.scal;
    if (scal[S_DONE] != 0.0 || scal[S_STOP] != 0.0) return;
    const double py = combine_partials(q.ppy, nb, 0.0, OpSum());
    if (threadIdx.x == 0) {
        bool more;
        CgScalars c;
        c.load(scal);
        const double alfa = cg_alfa(c, py, more);
        scal[S_PY] = py;
        scal[S_ALFA0] = scal[S_ALFA];
        scal[S_ALFA] = alfa;
        scal[S_EOLD] = scal[S_ENEW];
        if (!more) scal[S_STOP] = 1.0;
    }
}

// ELL row lengths and columns (EllLap::build): distances from the row (kShort,
// *far = 1 when one has more than 16 bits) or column numbers
template <bool kShort, class C>
__global__ void k_ell_col(int n, int width, const int* __restrict__ rowptr,
                          const int* __restrict__ idx, C* __restrict__ col,
                          unsigned char* __restrict__ len, int* __restrict__ far) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int b = rowptr[i], cnt = rowptr[i + 1] - b;
    len[i] = (unsigned char)cnt;
    bool out = false;
    for (int k = 0; k < width; ++k) {
        const int c = k < cnt ? idx[b + k] - 1 : i;
        const int d = kShort ? c - i : c;
        out = out || d < -32768 || d > 32767;
        col[(size_t)k * n + i] = (C)d;
    }
    if (kShort && out) *far = 1;
}

__global__ void k_ell_val(int n, int width, const int* __restrict__ rowptr,
                          const double* __restrict__ A, double* __restrict__ val) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int b = rowptr[i], len = rowptr[i + 1] - b;
    for (int k = 0; k < width; ++k) val[(size_t)k * n + i] = k < len ? A[b + k] : 0.0;
}

// meshMove.f90:99-104 for both axes in one launch, with the outcomes of their
// solves (a launch of its own costs the step more than what it does)
struct MoveAxis {
    const double *scal, *pos;
    double *X, *X1, *W, *Wold, *iters, *rz;
};
__global__ void k_mesh_move(MoveAxis ax, MoveAxis ay, double* __restrict__ itsum,
                            double* __restrict__ unconv, const double* __restrict__ dtminp, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const double dtmin = *dtminp;
    if (i < n) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const MoveAxis& a = k ? ay : ax;
            const double d = a.pos[i];
            if (a.Wold) a.Wold[i] = a.W[i];
            a.X[i] = a.X[i] + d;
            a.X1[i] = a.X1[i] + d;
            a.W[i] = d / dtmin;
        }
    }
    if (i != 0) return;
    *ax.iters = ax.scal[S_K];
    *ax.rz = ax.scal[S_EOLD];
    *ay.iters = ay.scal[S_K];
    *ay.rz = ay.scal[S_EOLD];
    *itsum = *itsum + ax.scal[S_K] + ay.scal[S_K];
    *unconv = *unconv + (ax.scal[S_CONV] == 0.0 ? 1.0 : 0.0) + (ay.scal[S_CONV] == 0.0 ? 1.0 : 0.0);
}

// z = x (the guess), no row fixed yet; system blockIdx.y
__global__ void k_cg_guess(int n, CgBoth a) {
    const CgSys& q = a.s[blockIdx.y];
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    q.z[i] = q.x[i];
    q.fixflag[i] = 0;
}

// out[k] = the sum of system k's residual partials (block k)
__global__ void __launch_bounds__(256)
k_cg_rr(CgBoth a, int nb, double* __restrict__ out) {
    const double s = combine_partials(a.s[blockIdx.x].prr, nb, 0.0, OpSum());
    if (threadIdx.x == 0) out[blockIdx.x] = s;
}

CgSys cg_sys(const PcgSystem& q, int cur) {
    PcgWork& w = *q.w;
    double* pbuf[2] = {w.pa.p, w.pb.p};
    const size_t nb = w.nblocks;
    return CgSys{q.x, w.r.p, w.z.p, w.y.p, w.scal.p, w.partial.p, w.partial.p + 3 * nb,
                 w.partial.p + 4 * nb, pbuf[cur], pbuf[cur ^ 1], w.fixflag.p, q.b,
                 q.x_fix, q.x_fix_idx, q.nfix};
}

// Rows up to which k_cg_b loads a row's entries (kAheadRows), and gathers
// their p and z too (kDeepRows), before it has beta.  Measured per iteration,
// one system / two: 32,768 rows 9.6 / 13.4 us with no loads ahead, 9.5 / 13.1
// with the entries, 9.2 / 12.5 with the gathers; 131,072 rows 10.9 / 18.7,
// 10.8 / 16.6, 10.9 / 16.4; 245,760 rows 13.8 / 23.3, 12.7 / 21.0, 13.6 / 21.6;
// 524,288 rows (bound by bandwidth: the registers cost waves) 21.2 / 31.9,
// 24.7 / 38.6, 24.5 / 39.3.
constexpr int kDeepRows = 160 * 1024, kAheadRows = 256 * 1024;
// Two systems up to kRowsApart rows: a grid row of blocks each, since latency and
// not the matrix's bytes is what an iteration costs (4,608 rows 12.6 us with both in
// each thread); above, both in each thread, which reads the matrix once.
constexpr int kRowsApart = 160 * 1024;
static_assert(kAheadRows == kFoldSmall * kBlock && kDeepRows <= kRowsApart,
              "the row readers' kFew, kMany and kAlone");
// calls f with the row reader of the matrix: the ELL copy when there is one
template <class F>
void with_rows(int n, const double* A, const int* idx, const int* rowptr, const EllMat* ell, F f) {
    if (!ell) f(CsrRows{A, idx, rowptr});
    else if (ell->width <= 8 && ell->dcol && n <= kDeepRows) f(EllRows<8, true, 2>{*ell});
    else if (ell->width <= 8 && ell->dcol && n <= kAheadRows) f(EllRows<8, true, 1>{*ell});
    else if (ell->width <= 8 && ell->dcol) f(EllRows<8, true, 0>{*ell});
    else if (ell->width <= 8) f(EllRows<8, false, 0>{*ell});
    else if (ell->dcol) f(EllRows<kEllMaxWidth, true, 0>{*ell});
    else f(EllRows<kEllMaxWidth, false, 0>{*ell});
}

}  // namespace

// Four launches for both systems; one system at a time from the CSR rows, with
// a copy and a set-up launch of its own, took ten (5-8 us each on 131,584
// rows, the residual 6.7).
void pcg_initial_rr(const PcgSystem (&sys)[2], int npoin, const double* A, const int* idx,
                    const int* rowptr, const double* diag, const EllMat* ell, double* rr_out,
                    hipStream_t s) {
    CgBoth a{};
    for (int k = 0; k < 2; ++k) {
        sys[k].w->ensure(npoin);
        a.s[k] = cg_sys(sys[k], 0);
    }
    const int nb = (int)grid_for(npoin), nfix = std::max(sys[0].nfix, sys[1].nfix);
    k_cg_guess<<<dim3(nb, 2), kBlock, 0, s>>>(npoin, a);
    for (auto& q : a.s) q.x = q.z;
    if (nfix > 0) k_cg_fix<1><<<dim3(grid_for(nfix), 2), kBlock, 0, s>>>(a);
    with_rows(npoin, A, idx, rowptr, ell, [&](auto rows) {
        k_cg_residual<decltype(rows), 1, false><<<dim3(nb, 2), kBlock, 0, s>>>(npoin, rows, diag, a, 0, nb);
    });
    k_cg_rr<<<2, 256, 0, s>>>(a, nb, rr_out);
    CFD_HIP(hipGetLastError());
}

void launch_mesh_move(const MeshAxis& x, const MeshAxis& y, double* itsum, double* unconv,
                      const double* dtmin, int n, hipStream_t s) {
    auto axis = [](const MeshAxis& a) {
        return MoveAxis{a.w->scal.p, a.pos, a.X, a.X1, a.W, a.Wold, a.iters, a.rz};
    };
    k_mesh_move<<<grid_for(n), kBlock, 0, s>>>(axis(x), axis(y), itsum, unconv, dtmin, n);
    CFD_HIP(hipGetLastError());
}

bool EllLap::build(int npoin, long long nnz, const int* rowptr, const int* idx, const int* rowptr_host,
                   hipStream_t s) {
    n = npoin;
    width = 0;
    if (n <= 0 || nnz <= 0) return false;
    int w = 0, least = 0;
    for (int i = 0; i < n; ++i) {
        const int l = rowptr_host[i + 1] - rowptr_host[i];
        w = std::max(w, l);
        least = std::min(least, l);
    }
    if (least < 0 || w <= 0 || w > kEllMaxWidth || (double)w * n > 1.5 * (double)nnz) return false;
    dcol.alloc((size_t)w * n);
    len.alloc(n);
    val.alloc((size_t)w * n);
    DBuf<int> far(1);
    far.zero(s);
    k_ell_col<true><<<grid_for(n), kBlock, 0, s>>>(n, w, rowptr, idx, dcol.p, len.p, far.p);
    CFD_HIP(hipGetLastError());
    int out = 0;
    CFD_HIP(hipMemcpyAsync(&out, far.p, sizeof(int), hipMemcpyDeviceToHost, s));
    CFD_HIP(hipStreamSynchronize(s));
    if (out) {
        dcol.release();
        col.alloc((size_t)w * n);
        k_ell_col<false><<<grid_for(n), kBlock, 0, s>>>(n, w, rowptr, idx, col.p, len.p, far.p);
        CFD_HIP(hipGetLastError());
        CFD_HIP(hipStreamSynchronize(s));  // far goes out of scope
    }
    width = w;
    return true;
}

bool EllLap::build(const Tables& t, hipStream_t s) {
    std::vector<int> rp(t.npoin + 1);  // the row lengths, on the host (once per session)
    t.rowptr.download(rp.data(), t.npoin + 1, s);
    CFD_HIP(hipStreamSynchronize(s));
    return build(t.npoin, t.nnz, t.rowptr.p, t.idx.p, rp.data(), s);
}

void EllLap::refresh(const int* rowptr, const double* A, hipStream_t s) {
    if (!width) return;
    k_ell_val<<<grid_for(n), kBlock, 0, s>>>(n, width, rowptr, A, val.p);
    CFD_HIP(hipGetLastError());
}

void PcgWork::ensure(int npoin) {
    if (npoin == n) return;
    n = 0;  // until every part is there
    nblocks = (int)grid_for(npoin);
    r.alloc(npoin);
    z.alloc(npoin);
    y.alloc(npoin);
    pa.alloc(npoin);
    pb.alloc(npoin);
    fixflag.alloc(npoin);
    partial.alloc(kPcgPartials * (size_t)nblocks);
    scal.alloc(S_NSCAL);
    hpin.alloc(2 * S_NSCAL);
    for (auto& e : ev)
        if (!e) CFD_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    n = npoin;
}

PcgWork::~PcgWork() {
    for (auto e : ev)
        if (e) (void)hipEventDestroy(e);
}

namespace {

// the scalars of the systems to the host's pinned copies
__global__ void k_cg_poll(CgBoth a, double* h0, double* h1) {
    const double* scal = a.s[blockIdx.x].scal;
    (blockIdx.x ? h1 : h0)[threadIdx.x] = scal[threadIdx.x];
}

// Launches of one solve on rows of type Rows: the start, and single
// iterations, of one system (q.s[0]) or two.
template <class Rows>
struct CgLaunch {
    int n, nb;
    Rows rows;
    const double* diag;
    hipStream_t s;
    static constexpr bool kEll = !std::is_same<Rows, CsrRows>::value;
    // Up to kFoldSmall partials blocks of 256 threads that each combine them
    // all (4 loads a thread); up to kFoldMid blocks of 512 and up to kFoldMax
    // of 1024, so that fewer blocks read them (an iteration of one system /
    // two at 320,000 rows: 16.2 / 25.3 us with 512 threads, 17.8 / 27.9 with
    // 1024); above, the one-block kernels (524,288 rows: 23.0 / 34.7 us with
    // them, 19.8 / 31.2 without; 980,000 rows 38.8 / 57.5 either way).  CSR
    // rows are staged by 256 threads.
    // f(systems in a thread, grid rows of systems)
    template <class F>
    void shaped(int nsys, F f) const {
        if constexpr (!Rows::kAlone) {
            if (nsys == 2 && n > kRowsApart) {
                f(std::integral_constant<int, 2>{}, 1);
                return;
            }
        }
        f(std::integral_constant<int, 1>{}, nsys);
    }

    template <int NS>
    void start_ns(const CgBoth& q, int rows_y, double tol, int maxit, int rel) const {
        const dim3 g(nb, rows_y), blk(kBlock);
        k_cg_init<NS><<<g, blk, 0, s>>>(n, q, tol, maxit);
        const int nfix = std::max(q.s[0].nfix, q.s[1].nfix);
        if (nfix > 0) k_cg_fix<NS><<<dim3(grid_for(nfix), rows_y), blk, 0, s>>>(q);
        k_cg_residual<Rows, NS, true><<<g, blk, 0, s>>>(n, rows, diag, q, rel, nb);
        k_cg_test<<<NS * rows_y, 256, 0, s>>>(q, nb, rel);
    }
    void start(const CgBoth& q, int nsys, double tol, int maxit, int rel) const {
        shaped(nsys, [&](auto ns, int y) { start_ns<decltype(ns)::value>(q, y, tol, maxit, rel); });
    }
    template <int NS>
    void a_ns(const CgBoth& q, int rows_y, int both) const {
        if (nb <= kFoldSmall) {
            k_cg_a<1, NS, true><<<dim3(nb, rows_y), kBlock, 0, s>>>(n, diag, q, nb, both);
        } else if (kEll && nb <= kFoldMid) {
            k_cg_a<2, NS, true><<<dim3((nb + 1) / 2, rows_y), 2 * kBlock, 0, s>>>(n, diag, q, nb, both);
        } else if (kEll && nb <= kFoldMax) {
            k_cg_a<4, NS, true><<<dim3((nb + 3) / 4, rows_y), 4 * kBlock, 0, s>>>(n, diag, q, nb, both);
        } else {
            k_cg_a<1, NS, false><<<dim3(nb, rows_y), kBlock, 0, s>>>(n, diag, q, nb, both);
            k_cg_fin_a<<<NS * rows_y, 256, 0, s>>>(q, nb, 0);
        }
    }
    void a(const CgBoth& q, int nsys, int both) const {
        shaped(nsys, [&](auto ns, int y) { a_ns<decltype(ns)::value>(q, y, both); });
    }
    template <int NS>
    void b_ns(const CgBoth& q, int rows_y, int first) const {
        CFD_CHECK(nb <= kFoldSmall ? !Rows::kMany : !Rows::kFew, "internal: PCG row reader");
        if constexpr (!Rows::kMany) {
            if (nb <= kFoldSmall) {
                k_cg_b<1, Rows, NS, true><<<dim3(nb, rows_y), kBlock, 0, s>>>(n, rows, q, nb, first);
                return;
            }
        }
        if constexpr (!Rows::kFew) {
            if constexpr (kEll) {
                if (nb <= kFoldMid) {
                    k_cg_b<2, Rows, NS, true>
                        <<<dim3((nb + 1) / 2, rows_y), 2 * kBlock, 0, s>>>(n, rows, q, nb, first);
                    return;
                }
                if (nb <= kFoldMax) {
                    k_cg_b<4, Rows, NS, true>
                        <<<dim3((nb + 3) / 4, rows_y), 4 * kBlock, 0, s>>>(n, rows, q, nb, first);
                    return;
                }
            }
            if (first) k_cg_fin_a<<<NS * rows_y, 256, 0, s>>>(q, nb, 1);
            k_cg_b<1, Rows, NS, false><<<dim3(nb, rows_y), kBlock, 0, s>>>(n, rows, q, nb, first);
            k_cg_fin_b<<<NS * rows_y, 256, 0, s>>>(q, nb);
        }
    }
    void b(const CgBoth& q, int nsys, int first) const {
        shaped(nsys, [&](auto ns, int y) { b_ns<decltype(ns)::value>(q, y, first); });
    }
};


// ---------------------------------------------------------------------------
// Small systems: a whole solve in one launch, one block per system.  Thread t
// of kT holds rows t, t + kT, ..., kR of them; a wave's rows s kT + 64 w ..
// belong to logical block (s kT + 64 w) / 256, so every sum has the pieces and
// the order of the kernels above (the same bits).  r, diag and z or y (never
// both alive) stay in registers, p is in LDS for the gathers, the matrix in
// registers and LDS as far as it fits.  The scalars never leave the block: no
// launch, no round trip through memory and no poll between the iterations, and a
// mesh that moves in steps does not wait for the host (under the absolute rule with
// a learned start the host waits, at the next step's solves, for these to have ended:
// pcg_ask_iterations).
//
// An iteration of one system / two against the two launches above (us): 768
// rows 1.6 / 1.65 against 7.9 / 8.3, 2,048 rows 2.3 / 2.45, 3,072 rows 3.1 /
// 3.3, 3,840 rows 3.8 / 4.0, 4,608 rows 5.3 / 5.7 against 7.9 / 8.35.  Bound by
// the one CU: FP64 instructions (about 0.35 us per 512 rows), three barriers and
// two trees (1 us).  The forms of 512 threads (up to 3,072 rows) spill nothing; those
// of 1,024 are at their 128 VGPRs and keep 23 (up to 4,096 rows) to 35 registers a
// thread in scratch, which the 4,608 rows' time includes.  Above kWholeRows the matrix no longer fits beside p (6,144
// rows 8.9 / 8.9, 8,192 rows 13 / 13 against 7.8 / 8.0).
// ---------------------------------------------------------------------------

__device__ __forceinline__ double first_lane(double v) {
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)),
                            __builtin_amdgcn_readfirstlane(__double2loint(v)));
}

// a becomes {a's lower half, b's lower half}, b {a's upper, b's upper}; kRows:
// the same of neighbouring rows of 16 lanes
template <bool kRows>
__device__ __forceinline__ void swap_parts(double& a, double& b) {
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    auto half = [](int u, int v) {
        return kRows ? (u32x2)__builtin_amdgcn_permlane16_swap((unsigned)u, (unsigned)v, false, false)
                     : (u32x2)__builtin_amdgcn_permlane32_swap((unsigned)u, (unsigned)v, false, false);
    };
    const u32x2 hi = half(__double2hiint(a), __double2hiint(b));
    const u32x2 lo = half(__double2loint(a), __double2loint(b));
    a = __hiloint2double((int)hi.x, (int)lo.x);
    b = __hiloint2double((int)hi.y, (int)lo.y);
}
// wave_reduce's sums of kR values a lane, out[s * stride] for value s: after the
// step of half waves two values share a register, after the next four
template <int kR>
__device__ __forceinline__ void wave_sums(double (&v)[kR], double* out, int stride) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int g = 0; g < kR; g += 4) {
        double a[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) a[j] = g + j < kR ? v[g + j] : 0.0;
        swap_parts<false>(a[0], a[1]);
        a[0] = a[0] + a[1];
        if (g + 2 < kR) {
            swap_parts<false>(a[2], a[3]);
            a[2] = a[2] + a[3];
        }
        swap_parts<true>(a[0], a[2]);
        double t = a[0] + a[2];
        t = t + lane_above<8>(t);
        t = t + lane_above<4>(t);
        t = t + lane_above<2>(t);
        t = t + lane_above<1>(t);
        // rows of 16 lanes: values g, g + 2, g + 1, g + 3
        const int s = g + (lane >> 5) + 2 * (lane >> 4 & 1);
        if ((lane & 15) == 0 && s < kR) out[s * stride] = t;
    }
}

template <int kT, int kW, int kR, int kKeep, int kLds, bool kX>
__global__ void __launch_bounds__(kT)
k_cg_whole(int n, EllMat m, const double* __restrict__ diag, CgBoth sys, double tol, int maxit,
           int rel) {
    extern __shared__ double sp[];  // p (first: x), kLds values per row, a byte per row: fixed
    __shared__ double sums[3][kR * (kT / 64)];
    unsigned char* fixed = reinterpret_cast<unsigned char*>(sp + (kX ? 1 + kLds : 2 + kLds) * n);
    const CgSys& q = sys.s[blockIdx.x];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, nb = (n + kBlock - 1) / kBlock;
    // the waves' sums into sums[k], and all of sums[k]
    auto put = [&](int k, double (&v)[kR]) { wave_sums(v, &sums[k][w], (kT / 64)); };
    auto total = [&](int k) {
        double acc = 0.0;
        if (lane < nb) {
            const double* p = &sums[k][4 * lane];
            double b = p[0];
            b = b + p[1];
            b = b + p[2];
            b = b + p[3];
            acc = acc + b;
        }
        return first_lane(wave_reduce(acc, OpSum())) + 0.0;
    };
    // x in registers (kX) or in LDS
    double x[kX ? kR : 1], d[kR], r[kR], yz[kR], v[kR];
    double *sx = sp + n, *sv = sx + (kX ? 0 : n);
    int fix = 0;  // bit s: row 1024 s + t is fixed
    for (int i = t; i < n; i += kT) {
        sp[i] = q.x[i];
        fixed[i] = 0;
    }
    __syncthreads();
    for (int f = t; f < q.nfix; f += kT) {
        const int i = q.fix_idx[f] - 1;
        sp[i] = 1.0 * q.x_fix[f];
        fixed[i] = 1;
    }
    __syncthreads();
    // the rows' entries: their columns as packed offsets into p, the lengths,
    // the first kKeep values, and the next kLds in LDS; the others are read in
    // each use, at an offset of a zero that the compiler can't see through (it
    // would keep them all, in scratch).  Slots beyond the matrix's width repeat
    // its last.
    constexpr int kPairs = (kW + 1) / 2;
    unsigned at[kR][kPairs], full = 0;  // full: rows s of the wave all of kW entries
    unsigned long long lens = 0;
    double kept[kR][kKeep > 0 ? kKeep : 1];
    const int last = m.width - 1;
#pragma unroll
    for (int s = 0; s < kR; ++s) {
        const int i = min(s * kT + t, n - 1);
        lens |= (unsigned long long)m.len[i] << (4 * s);
        if (__all(m.len[i] == kW)) full |= 1u << s;
#pragma unroll
        for (int j = 0; j < kW; ++j) {
            const unsigned c = 8u * (unsigned)(i + m.dcol[min(j, last) * n + i]);
            at[s][j / 2] = j & 1 ? at[s][j / 2] | c << 16 : c;
            if (j < kKeep) kept[s][j] = m.val[min(j, last) * n + i];
            else if (j < kKeep + kLds) sv[(j - kKeep) * n + i] = m.val[min(j, last) * n + i];
        }
    }
    // f(in the row, a_ij, byte offset of column j's p) over the slots of the
    // thread's row s, in order
    auto row = [&](int s, int zero, auto all, auto f) {
        const int i = min(s * kT + t, n - 1);
        unsigned len = (unsigned)(lens >> (4 * s)) & 15u, o[kPairs];
        double a[kW];
#pragma unroll
        for (int j = kKeep; j < kW; ++j)
            a[j] = j < kKeep + kLds ? sv[(j - kKeep) * n + i] : m.val[min(j, last) * n + i + zero];
#pragma unroll
        for (int j = 0; j < kPairs; ++j) {
            o[j] = at[s][j];
            asm volatile("" : "+v"(o[j]));
        }
        asm volatile("" : "+v"(len));
#pragma unroll
        for (int j = 0; j < kW; ++j)
            f(all.value || (unsigned)j < len, j < kKeep ? kept[s][j] : a[j],
              j & 1 ? o[j / 2] >> 16 : o[j / 2] & 0xffffu);
    };
    auto p_at = [&](unsigned o) {
        return *reinterpret_cast<const double*>(reinterpret_cast<const char*>(sp) + o);
    };
    double vr[kR], vz[kR];
#pragma unroll
    for (int s = 0; s < kR; ++s) {
        const int i = s * kT + t;
        r[s] = yz[s] = vr[s] = vz[s] = 0.0;
        d[s] = 1.0;
        if (i < n) {
            if (kX) x[s] = sp[i];
            else sx[i] = sp[i];
            d[s] = diag[i];
            double dot = 0.0, dotd = 0.0;
            row(s, 0, std::false_type{}, [&](bool in, double aij, unsigned o) {
                const double xc = p_at(o);
                dot = in ? dot + aij * xc : dot;
                dotd = in && fixed[o / 8] ? dotd + aij * xc : dotd;
            });
            if (fixed[i]) {
                fix |= 1 << s;
            } else {
                const double bi = q.b[i];
                r[s] = -1.0 * dot + bi;
                const double rd = -1.0 * dotd + bi;
                vr[s] = rd * rd;
                vz[s] = rd * (rd / d[s]);
            }
        }
        v[s] = r[s] * r[s];
    }
    put(0, v);
    if (rel) {
        put(1, vr);
        put(2, vz);
    }
    __syncthreads();
    const double rr = total(0);
    const double tolr = rel ? tol * tol * total(1) : tol, tolz = rel ? tol * tol * total(2) : tol;
    double e = rr, k = 0.0, conv = 1.0;
    if (!cg_solved(rr, tolr)) {
        __syncthreads();  // sums are read
#pragma unroll
        for (int s = 0; s < kR; ++s) {
            yz[s] = r[s] / d[s];
            v[s] = r[s] * yz[s];
        }
        put(0, v);
        __syncthreads();
        e = total(0);
        double beta = 0.0;
        for (bool first = true;; first = false) {
            // B: p = beta p + z, y = A p
#pragma unroll
            for (int s = 0; s < kR; ++s) {
                const int i = s * kT + t;
                if (i < n) sp[i] = first ? yz[s] : beta * sp[i] + yz[s];
            }
            __syncthreads();
            int zero = 0;
            asm volatile("" : "+s"(zero));
#pragma unroll
            for (int s = 0; s < kR; ++s) {
                const int i = s * kT + t;
                const double pn = sp[min(i, n - 1)];
                double dot = 0.0;
                const auto add = [&](bool in, double aij, unsigned o) {
                    const double c = dot + aij * p_at(o);
                    dot = in ? c : dot;
                };
                if (full >> s & 1) row(s, zero, std::true_type{}, add);
                else row(s, zero, std::false_type{}, add);
                yz[s] = fix >> s & 1 ? 1.0e30 * pn : dot;
                v[s] = i < n ? pn * yz[s] : 0.0;
            }
            put(1, v);
            __syncthreads();
            // A: x += alfa p, r -= alfa y, z = r / diag
            const double alfa = cg_step(e, total(1)), eold = e;
            const bool more = fabs(e) > tolz && k < (double)maxit;
#pragma unroll
            for (int s = 0; s < kR; ++s) {
                const int i = s * kT + t;
                if (i >= n) continue;
                double& xi = kX ? x[s] : sx[i];
                xi = alfa * sp[i] + xi;
            }
            if (!more) break;
#pragma unroll
            for (int s = 0; s < kR; ++s) {
                if (s * kT + t < n) r[s] = -alfa * yz[s] + r[s];
                double ds = d[s];
                asm volatile("" : "+v"(ds));  // else the divisor's reciprocals are kept, in scratch
                yz[s] = r[s] / ds;
                v[s] = r[s] * yz[s];
            }
            put(0, v);
            __syncthreads();
            e = total(0);
            beta = e / eold;
            k = k + 1.0;
        }
        conv = fabs(e) > tolz ? 0.0 : 1.0;
    }
#pragma unroll
    for (int s = 0; s < kR; ++s) {
        const int i = s * kT + t;
        if (i < n) q.x[i] = kX ? x[s] : sx[i];
    }
    if (t < S_NSCAL)
        q.scal[t] = t == S_K ? k : t == S_EOLD ? e : t == S_CONV ? conv : t == S_DONE ? 1.0
                  : t == S_TOL ? tol : t == S_MAXIT ? (double)maxit : t == S_TOLR ? tolr
                  : t == S_TOLZ ? tolz : t == S_RR ? rr : 0.0;
}

// The rows up to which a solve runs in k_cg_whole (33 bytes of LDS a row in
// its largest form), and the iteration cap (one launch of at most 0.15 s)
constexpr int kWholeRows = 4864, kWholeIters = 20000;
// A caller's matrix gets its ELL copy (EllMaker) when the first test has not ended the
// solve of a small system, and from so many iterations on that of a larger one, about
// where the copy has cost what it gains (us: the copy, an iteration from CSR rows and
// from it: 8,192 rows 65, 9.2, 7.7; 32,768 rows 60, 9.1, 7.6; 180,000 130, 12.5, 11.0;
// 524,288 1,400, 30, 19; 2.1M 2,700, 88, 66).
inline long ell_from(int n) { return n <= 128 * 1024 ? 28 : 96; }

template <int kT, int kW, int kR, int kKeep, int kLds, bool kX>
void launch_whole(int n, const EllMat& m, const double* diag, const CgBoth& q, int nsys, double tol,
                  int maxit, int rel, hipStream_t s) {
    const auto kernel = k_cg_whole<kT, kW, kR, kKeep, kLds, kX>;
    const size_t lds = (size_t)n * ((kX ? 1 + kLds : 2 + kLds) * sizeof(double) + 1);
    // the kernel's limit holds for the process: always that of its largest n, so
    // that threads with systems of different sizes set the same
    constexpr int kMost = std::min(kT * kR, kWholeRows) * ((kX ? 1 + kLds : 2 + kLds) * 8 + 1);
    if (kMost > 48 * 1024)
        CFD_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, kMost));
    kernel<<<nsys, kT, lds, s>>>(n, m, diag, q, tol, maxit, rel);
    CFD_HIP(hipGetLastError());
}

}  // namespace

void pcg_launch_multi(const PcgSystem* sys, int nsys, int npoin, const double* A, const int* idx,
                      const int* rowptr, const double* diag, double tol, int maxit, int rel,
                      hipStream_t s, const EllMat* ell, const EllMaker& late) {
    CFD_CHECK(npoin > 0, "arg: PCG needs npoin > 0");
    constexpr int kMaxSys = 2;
    CFD_CHECK(nsys >= 1 && nsys <= kMaxSys, "internal: PCG systems per launch");
    const int nb = (int)grid_for(npoin);
    for (int k = 0; k < nsys; ++k) sys[k].w->ensure(npoin);
    const bool small = npoin <= kWholeRows && maxit <= kWholeIters;
    // small systems: the whole solve in one launch; false where its rule does not hold
    auto whole = [&]() {
        if (!small || !ell || ell->width > 8 || !ell->dcol) return false;
        CgBoth q{};
        for (int k = 0; k < nsys; ++k) {
            q.s[k] = cg_sys(sys[k], 0);
            sys[k].w->polled_iters = -1.0;
        }
        // Threads, rows a thread and where the matrix is kept, by what fits: up
        // to 3,072 rows all of it in registers; above, values beside p in LDS,
        // and above 4,096 rows x there too and two or three values a row read
        // from L2 (5.3 us an iteration at 4,608 rows; 6.1 with three in LDS and
        // x in registers, which spills more; 6.8 with x in place; 8.0 in 512 threads
        // of ten rows).
        const int half = (npoin + 511) / 512;
        const auto pick = [&](auto width) {
            constexpr int kW = decltype(width)::value;
            return half <= 2   ? launch_whole<512, kW, 2, kW, 0, true>
                   : half <= 4 ? launch_whole<512, kW, 4, kW, 0, true>
                   : half <= 6 ? launch_whole<512, kW, 6, kW, 0, true>
                   : half <= 8 ? launch_whole<1024, kW, 4, 4, 3, true>
                               : launch_whole<1024, kW, 5, 2, 2, false>;
        };
        const auto go = ell->width <= 7 ? pick(std::integral_constant<int, 7>{})
                                        : pick(std::integral_constant<int, 8>{});
        go(npoin, *ell, diag, q, nsys, tol, maxit, rel, s);
        return true;
    };
    if (whole()) return;
    // pbuf[cur] holds the current p; both systems' buffers flip together
    int cur = 1;
    bool done[kMaxSys] = {false, nsys == 1};
    // the systems of a launch: both, or the one that is not done
    auto args = [&]() {
        CgBoth q{};
        int m = 0;
        for (int k = 0; k < nsys; ++k)
            if (!done[k]) q.s[m++] = cg_sys(sys[k], cur);
        return q;
    };
    auto count = [&]() { return (int)!done[0] + (int)!done[1]; };
    // Polls: a kernel writes the scalars to the host's pinned copies (two of
    // them, so that a poll may be waited for while the next iterations are
    // queued); without pinned memory a copy to the stack.
    double local[kMaxSys][S_NSCAL];
    const bool pinned = sys[0].w->hpin.p && sys[nsys - 1].w->hpin.p;
    auto host = [&](int k, int slot) {
        return pinned ? sys[k].w->hpin.p + slot * S_NSCAL : local[k];
    };
    auto ask = [&](int slot) {
        if (pinned) {
            CgBoth q{};
            for (int k = 0; k < nsys; ++k) q.s[k] = cg_sys(sys[k], cur);
            k_cg_poll<<<nsys, S_NSCAL, 0, s>>>(q, host(0, slot), host(nsys - 1, slot));
            CFD_HIP(hipEventRecord(sys[0].w->ev[slot], s));
            return;
        }
        for (int k = 0; k < nsys; ++k)
            CFD_HIP(hipMemcpyAsync(local[k], sys[k].w->scal.p, sizeof(local[k]),
                                   hipMemcpyDeviceToHost, s));
    };
    auto told = [&](int slot) {
        if (pinned) CFD_HIP(hipEventSynchronize(sys[0].w->ev[slot]));
        else CFD_HIP(hipStreamSynchronize(s));
        for (int k = 0; k < nsys; ++k) {
            done[k] = done[k] || host(k, slot)[S_DONE] != 0.0;
            sys[k].w->polled_iters = host(k, slot)[S_K];
        }
        return count() == 0;
    };
    int chunk = 4, slot = 0, both = 0;
    long launched = 0;
    enum { kStart, kProduct, kLoop } at = kStart;
    bool waits = (bool)late;
    // from where the solve stands; false: not done, and now is the time for the late copy
    auto solve = [&](auto rows) {
        const CgLaunch<decltype(rows)> go{npoin, nb, rows, diag, s};
        if (at == kStart) {
            // the first poll before the first product, which only solves that go on
            // need: a solve that the first test ends is known 5 us earlier
            go.start(args(), nsys, tol, maxit, rel);
            ask(slot);
            at = kProduct;
            if (waits && told(slot)) return true;
            if (waits && small) return false;
        }
        if (at == kProduct) {
            go.b(args(), nsys, 1);  // p0 = z0 into pbuf[0]
            cur = 0;
            at = kLoop;
            CFD_HIP(hipGetLastError());
        }
        auto iterate = [&](int m) {
            for (int q = 0; q < m; ++q) {
                go.a(args(), count(), both);
                go.b(args(), count(), 0);
                cur ^= 1;
                both ^= 1;
            }
            CFD_HIP(hipGetLastError());
        };
        // Most warm-started mesh solves stop at the first residual test;
        // batches grow while a solve runs on (few polls, few launches after
        // its end).  From kAsyncFrom iterations on the next batch is queued
        // before a poll is waited for: a poll's round trip costs an idle GPU
        // about 15 us, the batch queued in vain at the end about 50.
        constexpr long kAsyncFrom = 128;
        constexpr int kAsyncBatch = 8;
        while (!told(slot)) {
            CFD_CHECK(launched <= 4L * maxit + 64, "PCG did not terminate");
            if (waits && launched >= ell_from(npoin)) return false;
            if (pinned && launched >= kAsyncFrom) break;
            iterate(chunk);
            launched += chunk;
            chunk = std::min(chunk * 2, 16);
            ask(slot);
        }
        if (count() == 0) return true;
        iterate(kAsyncBatch);
        ask(slot);
        for (bool end = false; !end; slot ^= 1) {
            launched += kAsyncBatch;
            CFD_CHECK(launched <= 4L * maxit + 64, "PCG did not terminate");
            iterate(kAsyncBatch);
            ask(slot ^ 1);
            end = told(slot);
        }
        return true;
    };
    bool end = false;
    with_rows(npoin, A, idx, rowptr, ell, [&](auto rows) { end = solve(rows); });
    if (end) return;
    // it goes on with the late copy: small systems in one launch, from the start (the
    // one above has set the fixed values only), others where they stand
    waits = false;
    ell = late();
    if (!whole()) with_rows(npoin, A, idx, rowptr, ell, [&](auto rows) { solve(rows); });
}

bool pcg_ask_iterations(PcgWork& x, PcgWork& y, hipStream_t s) {
    if (x.polled_iters >= 0.0 && y.polled_iters >= 0.0) return false;
    CgBoth q{};
    q.s[0].scal = x.scal.p;
    q.s[1].scal = y.scal.p;
    k_cg_poll<<<2, S_NSCAL, 0, s>>>(q, x.hpin.p, y.hpin.p);
    CFD_HIP(hipEventRecord(x.ev[0], s));
    return true;
}

double pcg_told_iterations(PcgWork& x, PcgWork& y) {
    if (x.polled_iters < 0.0 || y.polled_iters < 0.0) {
        CFD_HIP(hipEventSynchronize(x.ev[0]));
        x.polled_iters = x.hpin.p[S_K];
        y.polled_iters = y.hpin.p[S_K];
    }
    return x.polled_iters + y.polled_iters;
}

void pcg_launch(PcgWork& w, int npoin, const double* A, const int* idx, const int* rowptr,
                const double* diag, double* x, const double* b, const double* x_fix,
                const int* x_fix_idx, int nfix, double tol, int maxit, int rel, hipStream_t s,
                const EllMaker& late) {
    PcgSystem sys{&w, x, b, x_fix, x_fix_idx, nfix};
    pcg_launch_multi(&sys, 1, npoin, A, idx, rowptr, diag, tol, maxit, rel, s, nullptr, late);
}

PcgResult pcg_result(const PcgWork& w, hipStream_t s) {
    double h[S_NSCAL];
    CFD_HIP(hipMemcpyAsync(h, w.scal.p, sizeof(h), hipMemcpyDeviceToHost, s));
    CFD_HIP(hipStreamSynchronize(s));
    PcgResult res;
    res.iters = (int)h[S_K];
    res.rz = h[S_EOLD];
    res.converged = h[S_CONV] != 0.0;
    return res;
}

}  // namespace cfd

// ---------------------------------------------------------------------------
// The same solve with no allocation (cfd_bicg_ex_noalloc): every work vector
// lives in one file-scope device array, `scratch`, sized for kNoAllocRows
// rows; its address on each device comes from hipGetSymbolAddress once, with
// that device current, and only that address is handed to kernels and copies.
// Calls on one device share the array: overlapping calls there race.
// ---------------------------------------------------------------------------
namespace cfd {
namespace {

constexpr int kNoAllocRows = 1 << 19;  // 524,288 rows
constexpr int kNoAllocBlocks = (kNoAllocRows + kBlock - 1) / kBlock;
constexpr size_t kAlign = 32;  // doubles: 256-byte sub-array alignment
constexpr size_t align_up(size_t v) { return (v + kAlign - 1) / kAlign * kAlign; }
// layout (in doubles): r, z, y, pa, pb (kNoAllocRows each), partial
// (kPcgPartials kNoAllocBlocks), scal (S_NSCAL), fixflag (kNoAllocRows bytes),
// the CSR check flag (one int32, in its own slot)
constexpr size_t kOffVec = 0;
constexpr size_t kOffPartial = align_up(kOffVec + 5 * (size_t)kNoAllocRows);
constexpr size_t kOffScal = align_up(kOffPartial + kPcgPartials * (size_t)kNoAllocBlocks);
constexpr size_t kOffFix = align_up(kOffScal + S_NSCAL);
constexpr size_t kOffFlag = align_up(kOffFix + kNoAllocRows / 8);
constexpr size_t kScratchDoubles = align_up(kOffFlag + 1);

}  // namespace

// about 22 MB per device, held until the process ends
static __device__ __align__(256) double scratch[kScratchDoubles];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double* g_scratch_ptr[kMaxDevices] = {};

double* scratch_on_current_device() {
    int dev = 0;
    CFD_HIP(hipGetDevice(&dev));
    CFD_CHECK(dev >= 0 && dev < kMaxDevices, "device id beyond the scratch table");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* ptr = nullptr;
        CFD_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
        CFD_CHECK(ptr != nullptr, "hipGetSymbolAddress(scratch) returned null");
        g_scratch_ptr[dev] = static_cast<double*>(ptr);
    }
    return g_scratch_ptr[dev];
}

// The row pointer starts at 0 and never decreases, every column index and
// fixed-node index lies in 1..n: else *flag = 1 (flag cleared by the caller's
// first launch, block 0 thread 0 of k_csr_flag_clear).
__global__ void k_csr_flag_clear(int* __restrict__ flag) { *flag = 0; }

__global__ void k_csr_check(int n, const int* __restrict__ rowptr, const int* __restrict__ idx,
                            const int* __restrict__ fix_idx, int nfix, int* __restrict__ flag) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x, nt = gridDim.x * blockDim.x;
    if (t == 0 && rowptr[0] != 0) *flag = 1;
    for (int i = t; i < n; i += nt)
        if (rowptr[i + 1] < rowptr[i]) *flag = 1;
    const int nnz = rowptr[n];
    for (int q = t; q < nnz; q += nt) {
        const int c = idx[q];
        if (c < 1 || c > n) *flag = 1;
    }
    for (int q = t; q < nfix; q += nt) {
        const int c = fix_idx[q];
        if (c < 1 || c > n) *flag = 1;
    }
}

}  // namespace
}  // namespace cfd

extern "C" int cfd_bicg_ex_noalloc(int npoin, const double* spMtx, const int* spIdx,
                                   const int* spRowptr, const double* diagMtx, double* x,
                                   const double* b, const double* x_fix, const int* x_fixIdx,
                                   int nfix, double tol, int maxit, int rel, void* stream,
                                   int* iters, double* rz, int* converged) {
    using namespace cfd;
    CFD_TRY({
        CFD_ARG(npoin > 0 && spMtx && spIdx && spRowptr && diagMtx && x && b, "null argument");
        CFD_ARG(npoin <= kNoAllocRows, "npoin " + std::to_string(npoin) + " exceeds the " +
                                           std::to_string(kNoAllocRows) +
                                           " rows of the allocation-free scratch");
        CFD_ARG(tol > 0.0 && maxit >= 0 && (rel == 0 || rel == 1), "tol > 0, maxit >= 0, rel 0/1");
        CFD_ARG(nfix >= 0 && (nfix == 0 || (x_fix && x_fixIdx)), "fixed-node lists");
        hipStream_t s = static_cast<hipStream_t>(stream);
        double* base = scratch_on_current_device();
        // the CSR and fixed-node indices are checked on the device first
        int* flag = reinterpret_cast<int*>(base + kOffFlag);
        k_csr_flag_clear<<<1, 1, 0, s>>>(flag);
        k_csr_check<<<1024, kBlock, 0, s>>>(npoin, spRowptr, spIdx, x_fixIdx, nfix, flag);
        CFD_HIP(hipGetLastError());
        int bad = 0;
        CFD_HIP(hipMemcpyAsync(&bad, flag, sizeof(int), hipMemcpyDeviceToHost, s));
        CFD_HIP(hipStreamSynchronize(s));
        CFD_ARG(bad == 0, "row pointer, column index or fixed-node index out of range");
        PcgWork w;  // views of the scratch array; nothing is allocated
        const int nb = (int)grid_for(npoin);
        w.n = npoin;
        w.nblocks = nb;
        w.r.borrow(base + kOffVec, npoin);
        w.z.borrow(base + kOffVec + (size_t)kNoAllocRows, npoin);
        w.y.borrow(base + kOffVec + 2 * (size_t)kNoAllocRows, npoin);
        w.pa.borrow(base + kOffVec + 3 * (size_t)kNoAllocRows, npoin);
        w.pb.borrow(base + kOffVec + 4 * (size_t)kNoAllocRows, npoin);
        w.partial.borrow(base + kOffPartial, kPcgPartials * (size_t)nb);
        w.scal.borrow(base + kOffScal, S_NSCAL);
        w.fixflag.borrow(reinterpret_cast<unsigned char*>(base + kOffFix), npoin);
        pcg_launch(w, npoin, spMtx, spIdx, spRowptr, diagMtx, x, b, x_fix, x_fixIdx, nfix, tol,
                   maxit, rel, s);
        PcgResult res = pcg_result(w, s);
        if (iters) *iters = res.iters;
        if (rz) *rz = res.rz;
        if (converged) *converged = res.converged;
    })
}
