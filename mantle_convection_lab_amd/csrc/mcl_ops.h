// Device operators shared by the FP64 and mixed-precision kernels: ELL row
// products, the gradient G and divergence G^T applied from element tables, the
// hanging-node constraints.  Sums run in the reference's order (sorted ELL
// columns; a row's elements ascending; an element's rows ascending).
#pragma once
#include "mcl_kernels.h"

// Agent-scope accesses of vectors that other workgroups write or read between
// two grid waits (GridSync).
__device__ __forceinline__ double ald(const double *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void ast(double *p, double v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ------------------------------------------------------------- sparse products

// (the vector's values read through load(j))
template <typename LD>
__device__ __forceinline__ double ell_row_ld(const int *__restrict__ col, const double *__restrict__ val, int ncol,
                                             int n, int row, LD load)
{
    // loads issued nine entries at a time (one memory round trip per chunk
    // instead of per entry); the sum keeps the ascending-column order
    double s = 0.0;
    int j = 0;
    for (; j + 9 <= ncol; j += 9) {
        int c[9];
        double v[9], x[9];
#pragma unroll
        for (int u = 0; u < 9; u++) {
            c[u] = col[(j + u) * n + row];
            v[u] = val[(j + u) * n + row];
        }
#pragma unroll
        for (int u = 0; u < 9; u++) x[u] = load(c[u]);
#pragma unroll
        for (int u = 0; u < 9; u++) s += v[u] * x[u];
    }
    if (j < ncol) {
        // the rest (a boundary row's, or of a longer row) in one round trip too
        int c[8];
        double v[8], x[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const bool in = j + u < ncol;
            c[u] = in ? col[(j + u) * n + row] : -1;
            v[u] = in ? val[(j + u) * n + row] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < 8; u++) x[u] = c[u] >= 0 ? load(c[u]) : 0.0;
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (c[u] >= 0) s += v[u] * x[u];
    }
    return s;
}

__device__ __forceinline__ double ell_row(const int *__restrict__ col, const double *__restrict__ val, int ncol,
                                          int n, int row, const double *__restrict__ x)
{
    return ell_row_ld(col, val, ncol, n, row, [&](int j) { return x[j]; });
}

// Products of a persistent solve whose threads own at most one row each (row
// = global thread number): the workgroup's rows are consecutive, so the vector
// entries they read lie in a window of the vector (the rows of a few mesh
// lines), which is read once, in order, into LDS; the row itself -- offsets
// into the window and values -- stays in registers over the whole solve.
// Gathering through agent-scope loads instead moves every entry up to 18 times
// past the L2.  Both forms of a solve pass different waits, so all workgroups
// take the same one: the host decides (fits) from the widest window of the mesh.
struct Window {
    double *buf;    // LDS
    int w0, n;      // vector entries [w0, w0 + n)
    bool fits;
    // the entries value(j) of the window into LDS, four loads in flight
    template <typename F>
    __device__ __forceinline__ void fill(F value) const
    {
        for (int j = threadIdx.x; j < n; j += 4 * MCL_BLOCK) {
            double v[4];
#pragma unroll
            for (int k = 0; k < 4; k++) v[k] = j + k * MCL_BLOCK < n ? value(w0 + j + k * MCL_BLOCK) : 0.0;
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (j + k * MCL_BLOCK < n) buf[j + k * MCL_BLOCK] = v[k];
        }
        __syncthreads();
    }
};

template <int W>
struct RowReg {
    int n;             // entries
    unsigned off[W];   // byte offsets in the window
    double v[W];
    // the row times the window's vector, in ell_row's order; skip: a slot
    // left out (-1: none)
    __device__ __forceinline__ double dot(const double *buf, int skip = -1) const
    {
        double x[W], s = 0.0;
#pragma unroll
        for (int u = 0; u < W; u++) x[u] = *(const double *)((const char *)buf + off[u]);
        // opaque to the compiler, which would otherwise keep the comparisons
        // of every slot with them in scalar registers over the whole solve
        int m = n, k = skip;
        asm volatile("" : "+v"(m), "+v"(k));
#pragma unroll
        for (int u = 0; u < W; u++)
            if (u < m && u != k) s += v[u] * x[u];
        return s;
    }
};

// This thread's row of a matrix (row < rows: col, val slot-major) and the
// workgroup's window.  fits = false (more slots than W, more rows than threads,
// or a window of some workgroup wider than the LDS buffer): neither is used.
template <int W>
__device__ __forceinline__ Window row_window(RowReg<W> &r, const int *__restrict__ col, const int *__restrict__ ncol,
                                             const double *__restrict__ val, int rows, double *buf, bool fits)
{
    __shared__ int lo, hi;
    const int row = blockIdx.x * blockDim.x + threadIdx.x;
    Window w{buf, 0, 0, fits};
    if (!fits) return w;
    if (threadIdx.x == 0) {
        lo = 0x7fffffff;
        hi = -1;
    }
    __syncthreads();
    r.n = row < rows ? ncol[row] : 0;
    int c[W], l = 0x7fffffff, h = -1;
#pragma unroll
    for (int u = 0; u < W; u++) {
        c[u] = u < r.n ? col[u * rows + row] : row;
        r.v[u] = u < r.n ? val[u * rows + row] : 0.0;
        if (u < r.n) {
            l = min(l, c[u]);
            h = max(h, c[u]);
        }
    }
    if (row < rows) {
        atomicMin(&lo, min(l, row));
        atomicMax(&hi, max(h, row));
    }
    __syncthreads();
    w.w0 = hi < 0 ? 0 : lo;
    w.n = hi < 0 ? 0 : hi - lo + 1;
#pragma unroll
    for (int u = 0; u < W; u++) r.off[u] = 8u * (unsigned)(u < r.n ? c[u] - w.w0 : 0);
    return w;
}

// G and G^T are applied from tables of a row's elements (an element's rows) and
// the entries: the index and the entry come in one round trip, the vector in a
// second.  (Through node, adjacency, element level and gradient table it took
// five: an Uzawa iteration's own phases at 32x32 17 us, 14 so; 27 and 22 at
// 256x256.)

// (G p)[P], G_prod_p (Solver.c:569-591): the row's elements ascending, their
// values read through load(e)
template <typename LD>
__device__ __forceinline__ double g_row_ld(const LevelDev &L, int P, LD load)
{
    int e[4];
    double v[4], x[4], s = 0.0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        e[k] = L.g_el[k * L.neq + P];
        v[k] = L.g_val[k * L.neq + P];
    }
#pragma unroll
    for (int k = 0; k < 4; k++) x[k] = e[k] >= 0 ? load(e[k]) : 0.0;
#pragma unroll
    for (int k = 0; k < 4; k++)
        if (e[k] >= 0) s += v[k] * x[k];
    return s;
}

__device__ __forceinline__ double g_row(const LevelDev &L, int P, const double *__restrict__ p)
{
    return g_row_ld(L, P, [&](int e) { return p[e]; });
}

// (G^T x)[e], GT_prod_d (Solver.c:645-666): rows of the element ascending,
// with the velocity values read through load(r).
template <typename LD>
__device__ __forceinline__ double gt_elem_ld(const LevelDev &L, int e, LD load)
{
    int r[8];
    double v[8], x[8], s = 0.0;
#pragma unroll
    for (int t = 0; t < 8; t++) {
        r[t] = L.gt_row[t * L.nel + e];
        v[t] = L.gt_val[t * L.nel + e];
    }
#pragma unroll
    for (int t = 0; t < 8; t++) x[t] = r[t] >= 0 ? load(r[t]) : 0.0;
#pragma unroll
    for (int t = 0; t < 8; t++)
        if (r[t] >= 0) s += v[t] * x[t];
    return s;
}

__device__ __forceinline__ double gt_elem(const LevelDev &L, int e, const double *__restrict__ x)
{
    return gt_elem_ld(L, e, [&](int r) { return x[r]; });
}

// Preconditioner data, Solver.c:54-64: BAB_e = sum_i G_ie^2 / Kdiag_i
__device__ __forceinline__ double bab_elem(const LevelDev &L, int e)
{
    double s = 0.0;
    for (int t = 0; t < 8; t++) {
        const int r = L.gt_row[t * L.nel + e];
        if (r < 0) break;
        const double g = L.gt_val[t * L.nel + e];
        s += g * g / L.Kdiag[r];
    }
    return s;
}

// ------------------------------------------------------------ persistent Uzawa

struct CgVecs {
    double *r, *s, *d, *q, *d2;   // d2: the other buffer of d
};

// Hanging-dof constraint, enforce_constrain_veq (Solver.c:1368-1437); the
// parents and the hanging values may belong to other workgroups.
static __device__ __forceinline__ void constrain_v(const LevelDev &L, double *__restrict__ x, int gtid, int gsize)
{
    if (L.nh == 0) return;
    if (L.h_serial) {
        if (gtid != 0) return;
        for (int k = 0; k < L.nh; k++) {
            for (int d = 0; d < 2; d++) {
                double t = 0.0;
                for (int c = 0; c < 2; c++) {
                    int kn = L.h_ci[c * L.nh + k];
                    int eqc = L.id[d * L.nno + kn];
                    t += eqc != -1 ? ald(x + eqc) : L.v_bc_val[d * L.nno + kn];
                }
                t *= 0.5;
                int eq = L.id[d * L.nno + L.h_ni[k]];
                if (eq >= 0) ast(x + eq, t);
            }
        }
        return;
    }
    for (int k = gtid; k < L.nh; k += gsize) {
        for (int d = 0; d < 2; d++) {
            double t = 0.0;
            for (int c = 0; c < 2; c++) {
                int kn = L.h_ci[c * L.nh + k];
                int eqc = L.id[d * L.nno + kn];
                t += eqc != -1 ? ald(x + eqc) : L.v_bc_val[d * L.nno + kn];
            }
            t *= 0.5;
            int eq = L.id[d * L.nno + L.h_ni[k]];
            if (eq >= 0) ast(x + eq, t);
        }
    }
}

static __device__ __forceinline__ void constrain_T(const LevelDev &L, double *__restrict__ x, int gtid, int gsize)
{
    if (L.nh == 0) return;
    int start = L.h_serial ? (gtid == 0 ? 0 : L.nh) : gtid;
    int step = L.h_serial ? 1 : gsize;
    for (int k = start; k < L.nh; k += step) {
        double t = 0.0;
        for (int c = 0; c < 2; c++) {
            int kn = L.h_ci[c * L.nh + k];
            int eqc = L.heat_id[kn];
            t += eqc != -1 ? ald(x + eqc) : L.T_bc_val[kn];
        }
        t *= 0.5;
        int eq = L.heat_id[L.h_ni[k]];
        if (eq >= 0) ast(x + eq, t);
    }
}

// An ELL matrix with its diagonal (explicit array or slot index per row).
struct EllMat {
    const int *col;
    const int *ncol;
    const double *val;
    const double *diag;      // diagonal values, or NULL to use diag_slot
    const int *diag_slot;
    int n;                   // rows
};

__device__ __forceinline__ double ell_diag(const EllMat &A, int i)
{
    return A.diag ? A.diag[i] : A.val[A.diag_slot[i] * A.n + i];
}

