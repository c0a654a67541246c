// FP64 kernels of libmcl_hip.so (gfx950).
//
// This translation unit is compiled with -ffp-contract=off: every operation
// on the parity path rounds like the reference's x86-64 build (no FMA), and
// every sum runs in the reference's order (element-ascending assembly, sorted
// row products), so assembly, sparse products and vector updates reproduce the
// reference bit for bit.  Only the dot products differ: they are compensated
// parallel reductions (the reference sums sequentially).
//
// Work decomposition (one HIP thread per item, grid-stride):
//   nodes     viscosity, buoyancy, nodal velocity, stress averaging
//   rows      velocity / heat equations: assembly of one matrix row from the
//             row's node-adjacent elements (atomic-free, element-ascending),
//             ELL products, G p, CG vector updates
//   elements  BAB, G^T d, pressure-space updates, SUPG tau, element stress
// The Uzawa solve and the heat step each run as one persistent kernel launched
// cooperatively; its phases are separated by grid-wide waits that carry their
// reductions (mcl_device.h).
#include "mcl_kernels.h"
#include "mcl_ops.h"

__constant__ ShapeTables c_shape;

extern "C" hipError_t mcl_upload_shape(const ShapeTables *s)
{
    return hipMemcpyToSymbol(HIP_SYMBOL(c_shape), s, sizeof(ShapeTables));
}

// ------------------------------------------------------------------ physics

// The level of a workgroup in a launch over all levels (lv[k].blk0: the first
// workgroup of level k).
template <typename T>
__device__ __forceinline__ const T &block_level(const T *__restrict__ lv, int nlev)
{
    int k = 0;
    while (k + 1 < nlev && (int)blockIdx.x >= lv[k + 1].blk0) k++;
    return lv[k];
}

// Viscosity.c:3-24: eta = exp(A (refT - T)), times lm_jump below z = 0.77; one
// thread a node of every level.  (A launch for each level cost 4.5 us, seven
// of them at 256x256; one 5 us.)
__global__ void __launch_bounds__(MCL_BLOCK) k_viscosity(const FieldLevel *__restrict__ lv, int nlev, double A,
                                                         double refT, double lm_jump)
{
    const FieldLevel &F = block_level(lv, nlev);
    const int i = ((int)blockIdx.x - F.blk0) * MCL_BLOCK + (int)threadIdx.x;
    if (i >= F.nno) return;
    double v = exp(A * (refT - F.T[i]));
    if (F.X[F.nno + i] < 0.77) v *= lm_jump;
    F.vis[i] = v;
}

// coarse_n = fine_{c2f(n)}: the finest temperature on the nodes of every
// coarser level
__global__ void __launch_bounds__(MCL_BLOCK) k_inject(const FieldLevel *__restrict__ lv, int nlev,
                                                      const double *__restrict__ fine)
{
    const FieldLevel &F = block_level(lv, nlev);
    const int i = ((int)blockIdx.x - F.blk0) * MCL_BLOCK + (int)threadIdx.x;
    if (i < F.nno) F.T[i] = fine[F.c2f[i]];
}

// Buoyancy.c:3-22 with get_node_horiz_avg (Parallel.c:354-437): a node row's
// average is the sum over its contribution list in the reference's order
// (elements ascending; within an element the interior points, then the top
// row or right column points, then the corner node).  Each entry adds
// N_a(xi, eta) * data[node_a] for a = 0..3 separately, as the reference does.
// A workgroup takes one row: its threads evaluate the terms of MCL_BUOY entries
// into LDS (the products are the reference's, independent of the running sum),
// then thread 0 adds them in list order, so the sum rounds exactly as the
// reference's sequential loop; what bounds it is that chain of additions.
// (One thread a row, reading the terms from memory, took 59 us for the 1028
// terms a row of 256x256; this 11 us.)  Entries with a negative element
// contribute one term (Ra T of the last node) and three +0.0 terms, which
// leave the sum unchanged.
__global__ void __launch_bounds__(MCL_BUOY) k_buoy_rows(int gnox, int nno, const int *__restrict__ ptr,
                                                        const int *__restrict__ ent_e,
                                                        const signed char *__restrict__ ent_xi,
                                                        const signed char *__restrict__ ent_eta,
                                                        const int *__restrict__ ienl, int nel,
                                                        const double *__restrict__ T, double Ra,
                                                        double *__restrict__ avg)
{
    __shared__ __attribute__((aligned(16))) double terms[4 * MCL_BUOY];
    const int t0 = ptr[blockIdx.x], t1 = ptr[blockIdx.x + 1];
    double s = 0.0;
    for (int b = t0; b < t1; b += MCL_BUOY) {
        const int t = b + (int)threadIdx.x;
        if (t < t1) {
            const int e = ent_e[t];
            double v0, v1 = 0.0, v2 = 0.0, v3 = 0.0;
            if (e < 0) {
                v0 = Ra * T[nno - 1];
            } else {
                double xi = (double)ent_xi[t], eta = (double)ent_eta[t];
                // Na values of Shape_function.c:180-197
                double n0 = 0.25 * (1.0 - xi) * (1.0 - eta);
                double n1 = 0.25 * (1.0 - xi) * (1.0 + eta);
                double n2 = 0.25 * (1.0 + xi) * (1.0 + eta);
                double n3 = 0.25 * (1.0 + xi) * (1.0 - eta);
                v0 = n0 * (Ra * T[ienl[e]]);
                v1 = n1 * (Ra * T[ienl[nel + e]]);
                v2 = n2 * (Ra * T[ienl[2 * nel + e]]);
                v3 = n3 * (Ra * T[ienl[3 * nel + e]]);
            }
            terms[4 * threadIdx.x] = v0;
            terms[4 * threadIdx.x + 1] = v1;
            terms[4 * threadIdx.x + 2] = v2;
            terms[4 * threadIdx.x + 3] = v3;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            const int n = 4 * min(MCL_BUOY, t1 - b);
            int u = 0;
            for (; u + 32 <= n; u += 32) {
                double v[32];
#pragma unroll
                for (int k = 0; k < 32; k++) v[k] = terms[u + k];
#pragma unroll
                for (int k = 0; k < 32; k++) s += v[k];
            }
            for (; u < n; u++) s += terms[u];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) avg[blockIdx.x] = s / gnox;
}

__global__ void k_buoy_apply(int nno, int gnoz, const int *__restrict__ node, const double *__restrict__ T,
                             double Ra, const double *__restrict__ avg, double *__restrict__ buoy)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < nno; i += gridDim.x * blockDim.x) {
        int nd = node[i];
        int ix = nd / gnoz, iz = nd - ix * gnoz;
        buoy[i] = Ra * T[i] - avg[iz];
    }
}

// ------------------------------------------------------------ Stokes assembly

// A row of the element stiffness matrix of get_element_K (Build_matrix.c:
// 192-271) after the reference's mirror step: entry (p, q) is the value of the
// upper entry (min(p, q), max(p, q)), a sum over the four Gauss points.  With u
// and w the upper entry's first dof's shape derivative along and across its
// direction, s and t the second's, and D = 2 eta for equal directions, else 0,
// the four cases of the reference are one expression, (u D) s + (w eta) t (its
// terms with a zero in the elasticity matrix add signed zeros, which leave the
// sum as it is).  Both orders are summed and one is taken: fewer instructions
// than choosing the operands.
struct KeRow {
    double u[4], w[4], we[4], eta[4];     // of the row's dof
    double D[2][4], uD[2][4];             // with column dofs along x, z
};

__device__ __forceinline__ double ke_entry(const KeRow &r, int p, int q, const double (&bx)[4], const double (&bz)[4],
                                           double jac)
{
    const bool jq = q & 1;
    double Kr = 0.0, Kq = 0.0;   // the row's dof first, the column's
#pragma unroll
    for (int g = 0; g < 4; g++) {
        const double s = jq ? bz[g] : bx[g], t = jq ? bx[g] : bz[g];
        Kr += r.uD[jq][g] * s + r.we[g] * t;
        Kq += (s * r.D[jq][g]) * r.u[g] + (t * r.eta[g]) * r.w[g];
    }
    return (q < p ? Kq : Kr) / jac;
}

// One thread per velocity row P: K row slots (element-ascending sums, the
// order of K_matrix, Build_matrix.c:42-115), F[P] (all boundary-value
// subtractions first, then the element loads of F_matrix, :117-140), Kdiag.
// The thread owns its row, so the slots accumulate without atomics: in the
// thread's own LDS column for rows of at most 18 slots (written to HBM once at
// the end), else in place in HBM; the additions to each slot come in the same
// order either way.  One launch assembles every level: each workgroup takes
// MCL_ASM_BLOCK rows of one level (lv[k].blk0 gives the first workgroup of level
// k), so the short levels run side by side instead of one launch each.  What
// bounds it is FP64 instruction issue (about 3000 a row): workgroups of 256
// threads spread the rows more evenly than 512.  At 256x256 about 50 us, 112 with
// the operands chosen per entry and every element's loads behind the last's.
#define MCL_ASM_LDS_SLOTS 18
__global__ void __launch_bounds__(MCL_ASM_BLOCK) k_assemble_K(const AsmLevel *__restrict__ lv, int nlev)
{
    __shared__ double kacc[MCL_ASM_LDS_SLOTS * MCL_ASM_BLOCK];
    __shared__ double sh[3][16];   // dN/dxi, dN/deta, N of (node, Gauss point)
    if (threadIdx.x < 16) {
        sh[0][threadIdx.x] = c_shape.dxi[threadIdx.x >> 2][threadIdx.x & 3];
        sh[1][threadIdx.x] = c_shape.deta[threadIdx.x >> 2][threadIdx.x & 3];
        sh[2][threadIdx.x] = c_shape.N[threadIdx.x >> 2][threadIdx.x & 3];
    }
    __syncthreads();
    double *acc = kacc + threadIdx.x;  // slot u at acc[u * MCL_ASM_BLOCK]
    const AsmLevel &lev = block_level(lv, nlev);
    const LevelDev &L = lev.L;
    const double *__restrict__ vis = lev.vis;
    const double *__restrict__ buoy = lev.buoy;
    const bool inl = L.WK <= MCL_ASM_LDS_SLOTS;
    {
        const int P = ((int)blockIdx.x - lev.blk0) * MCL_ASM_BLOCK + (int)threadIdx.x;
        if (P >= L.neq) return;
        const int n = L.veq_node[P], ip = L.veq_dof[P];
        const int nadj = L.p2n_cnt[n];
        if (inl)
            for (int u = 0; u < L.WK; u++) acc[u * MCL_ASM_BLOCK] = 0.0;
        else
            for (int s = 0; s < L.WK; s++) L.Kval[s * L.neq + P] = 0.0;
        // the elements at the row's node (a missing one reads the first's data)
        int el[4], a[4], idx[4][4];
        double dxdxi[4], dzdeta[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int kk = k < nadj ? k : 0;
            el[k] = L.p2n_el[kk * L.nno + n];
            a[k] = L.p2n_a[kk * L.nno + n];
        }
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int l = L.elev[el[k]];
            dxdxi[k] = 0.5 * L.lvl_dx[l];
            dzdeta[k] = 0.5 * L.lvl_dz[l];
#pragma unroll
            for (int d = 0; d < 4; d++) idx[k][d] = L.ienl[d * L.nel + el[k]];
        }
        double F = 0.0;
        int sd = -1;   // the diagonal's slot
#pragma unroll
        for (int k = 0; k < 4; k++) {
            if (k >= nadj) break;
            // keeps the next element's loads out of this one's registers
            asm volatile("" ::: "memory");
            const double jac = dxdxi[k] * dzdeta[k] - 0.0 * 0.0;
            int slot[8];
            char bc[8];
#pragma unroll
            for (int q = 0; q < 8; q++) {
                slot[q] = L.Kslot[(k * 8 + q) * L.neq + P];
                bc[q] = L.v_bc[(q & 1) * L.nno + idx[k][q >> 1]];
            }
            double vn[4];
            KeRow row;
#pragma unroll
            for (int d = 0; d < 4; d++) vn[d] = vis[idx[k][d]];
#pragma unroll
            for (int g = 0; g < 4; g++) {
                double s = 0.0;
#pragma unroll
                for (int d = 0; d < 4; d++) s += c_shape.N[d][g] * vn[d];
                const double ax = sh[0][4 * a[k] + g] * dzdeta[k], az = sh[1][4 * a[k] + g] * dxdxi[k];
                row.eta[g] = s;
                row.u[g] = ip ? az : ax;
                row.w[g] = ip ? ax : az;
                row.D[0][g] = ip ? 0.0 : 2.0 * s;
                row.D[1][g] = ip ? 2.0 * s : 0.0;
                row.uD[0][g] = row.u[g] * row.D[0][g];
                row.uD[1][g] = row.u[g] * row.D[1][g];
                row.we[g] = row.w[g] * s;
            }
            const int p = 2 * a[k] + ip;
            // column dofs in the reference's order: j outer, b inner
#pragma unroll
            for (int jb = 0; jb < 8; jb++) {
                const int j = jb >> 2, b = jb & 3, q = 2 * b + j;
                double bx[4], bz[4];
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    bx[g] = c_shape.dxi[b][g] * dzdeta[k];
                    bz[g] = c_shape.deta[b][g] * dxdxi[k];
                }
                const double kv = ke_entry(row, p, q, bx, bz, jac);
                if (q == p) sd = slot[q];
                if (slot[q] >= 0) {
                    if (inl) acc[slot[q] * MCL_ASM_BLOCK] += kv;
                    else L.Kval[slot[q] * L.neq + P] += kv;
                }
                if (bc[q] == 'V') F -= kv * L.v_bc_val[j * L.nno + idx[k][b]];
            }
        }
        // element loads, get_element_F (Build_matrix.c:273-344)
#pragma unroll
        for (int k = 0; k < 4; k++) {
            if (k >= nadj) break;
            asm volatile("" ::: "memory");
            const double jac = dxdxi[k] * dzdeta[k] - 0.0 * 0.0;
            double Fe = 0.0;
            if (ip == 1) {
                double fg[4], bn[4];
#pragma unroll
                for (int d = 0; d < 4; d++) bn[d] = buoy[idx[k][d]];
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    double s = 0.0;
#pragma unroll
                    for (int d = 0; d < 4; d++) s += c_shape.N[d][g] * bn[d];
                    fg[g] = s;
                }
#pragma unroll
                for (int g = 0; g < 4; g++) Fe += sh[2][4 * a[k] + g] * fg[g];
                Fe *= jac;
            }
            int nat = 0;
#pragma unroll
            for (int d = 0; d < 4; d++)
                if (L.v_bc[ip * L.nno + idx[k][d]] == 'S') nat += d;
            if (nat == 3) nat = 1;
            else if (nat == 1 || nat == 5) nat = 2;
            else if (nat == 0 || nat == 2) nat = 0;
            if (nat != 0) {
                double Lx = L.X[ip * L.nno + idx[k][2]] - L.X[ip * L.nno + idx[k][0]];
                Fe += 0.5 * Lx * L.v_bc_val[ip * L.nno + L.ienl[a[k] * L.nel + el[k]]];
            }
            F += Fe;
        }
        if (inl)
            for (int u = 0; u < L.WK; u++) L.Kval[u * L.neq + P] = acc[u * MCL_ASM_BLOCK];
        const double diag = sd < 0 ? 0.0 : inl ? acc[sd * MCL_ASM_BLOCK] : L.Kval[sd * L.neq + P];
        L.F[P] = F;
        L.Kdiag[P] = diag;
    }
}

// sum_i x_i y_i in index order, rounded after every product and every
// addition exactly as the reference's sequential loops (global_v_prod /
// global_p_prod, Array_work.c:287-341, at one rank).  Every workgroup computes
// it itself: the products in parallel into LDS, the additions in order by one
// thread, so all workgroups obtain the identical value without a barrier.
// The vectors must be complete (called after a grid wait) and written with
// agent-scope stores.
#define MCL_SEQ_CHUNK 2048
__device__ double seq_dot(const double *__restrict__ x, const double *__restrict__ y, int n)
{
    __shared__ double buf[MCL_SEQ_CHUNK];
    __shared__ double res;
    double s = 0.0;
    for (int base = 0; base < n; base += MCL_SEQ_CHUNK) {
        const int m = min(MCL_SEQ_CHUNK, n - base);
        __syncthreads();
        for (int t = threadIdx.x; t < m; t += blockDim.x) buf[t] = ald(x + base + t) * ald(y + base + t);
        __syncthreads();
        if (threadIdx.x == 0) {
            // loads batched sixteen at a time, additions strictly in order
            int t = 0;
            for (; t + 16 <= m; t += 16) {
                double v[16];
#pragma unroll
                for (int u = 0; u < 16; u++) v[u] = buf[t + u];
#pragma unroll
                for (int u = 0; u < 16; u++) s = s + v[u];
            }
            for (; t < m; t++) s = s + buf[t];
        }
    }
    if (threadIdx.x == 0) res = s;
    __syncthreads();
    return res;
}

// How a conjugate-gradient solve reads the vector of its product, one form for
// the whole grid (pcg_persistent):
//   CG_ROWS    one row a thread, the vector through the LDS window (row_window)
//   CG_GATHER  s + beta d gathered entry by entry with agent-scope loads
//   CG_CACHED  d stored by its row's thread, a fenced wait, then plain loads,
//              which the L1 and L2 serve to the rows that share an entry
enum CgForm { CG_ROWS, CG_GATHER, CG_CACHED };

// Conj_Grad (Solver.c:1589-1797) / Conj_Grad_heat (Update_temperature.c:
// 1140-1354) inside a persistent kernel.  All workgroups execute the same
// control flow: the scalars come from the grid waits, identical everywhere.
// kind 0: velocity (constraint on velocity dofs), 1: heat.
// Two grid waits an iteration:
//   (1) d = s + beta d and q = A d in one pass (the product gathers s + beta d,
//       the same rounding as the stored d), with d.q
//   (2) x += alpha d, r -= alpha q (every 50th iteration r = b - A x, after a
//       wait for x), s = r / diag, with r.s and max |alpha r|
// s, d and x cross workgroups with agent-scope accesses, so the waits need no
// cache maintenance and the matrix stays in the L2; r and q belong to the row's
// thread.  (CG_CACHED: one wait more, between d and the product; only d and x
// cross.)
// CG_ROWS: every thread owns at most one row (row_window): the row, r, q, d and x
// stay in registers and the gathered vector comes through the window; what is
// left of an iteration is the two waits and one round trip of loads.
// Measured per inner iteration (three fenced barriers, the matrix re-read after
// each, two rows a thread): 64x64 29 -> 7.7 us, 128x128 29 -> 8.2 us; of that
// the windows and registers are 2.7 us against gathers by agent-scope loads.
// The caller's phase may write b on this thread's rows (grid stride) right
// before the call; a non-zero x must be complete.  x is complete on return.
// Returns the iteration count; ok is cleared if a wait gave up.
template <int W, CgForm FORM>
__device__ __forceinline__ int pcg_rows(const LevelDev &L, const EllMat &A, const RowReg<W> &row, const Window &win,
                                        double diag, const double *__restrict__ b, double *x, bool x_zero, double accu,
                                        int max_cycle, int precond, int kind, CgVecs v, const GridSync &gs,
                                        WaitState &ws, bool &ok, long long &spmv, bool exact)
{
    const int gtid = blockIdx.x * blockDim.x + threadIdx.x, gsize = gridDim.x * blockDim.x;
    const int n = A.n;
    constexpr bool ROWS = FORM == CG_ROWS, cached = FORM == CG_CACHED;
    double rr = 0.0, rq = 0.0, rd = 0.0, rx = 0.0;
    if (ROWS && !x_zero && gtid < n) rx = ald(x + gtid);
    // row i times the vector value(j): the window's entries were filled before
    auto times = [&](int i, auto value) {
        if constexpr (ROWS) return row.dot(win.buf);
        else return ell_row_ld(A.col, A.val, A.ncol[i], n, i, value);
    };
    auto xat = [&](int j) { return ald(x + j); };
    // CG_CACHED: r, s and q are read by their row's thread alone (by all of
    // them in an exact dot product)
    auto put = [&](double *p, double y) {
        if (cached && !exact) *p = y;
        else ast(p, y);
    };
    auto get = [&](const double *p) { return cached && !exact ? *p : ald(p); };
    // r of row i and s = M r, with r.s
    auto residual = [&](int i, double r, dd &acc) {
        const double s = precond ? r / (ROWS ? diag : ell_diag(A, i)) : r;
        if (ROWS) rr = r;
        if (!ROWS || exact) put(v.r + i, r);
        put(v.s + i, s);
        acc = dd_add_prod(acc, r, s);
    };
    double delta_new;
    {
        dd acc[1] = {dd_zero()};
        if (ROWS && !x_zero) win.fill(xat);
        for (int i = gtid; i < n; i += gsize) residual(i, b[i] - (x_zero ? 0.0 : times(i, xat)), acc[0]);
        if (!x_zero) spmv++;
        double o[1] = {0.0};
        ok = ok && grid_sum<1>(gs, ws, acc, o);
        delta_new = exact ? seq_dot(v.r, v.s, n) : o[0];
    }
    const double delta0 = delta_new;
    double *dold = v.d, *dnew = v.d2, beta = 0.0;
    int cycle = 0;
    while (ok && cycle < max_cycle && delta_new > accu * delta0) {
        double t1;
        {
            auto dat = [&](int j) { return cycle == 0 ? ald(v.s + j) : ald(v.s + j) + beta * ald(dold + j); };
            dd acc[1] = {dd_zero()};
            if (ROWS) win.fill(dat);
            if constexpr (cached) {
                for (int i = gtid; i < n; i += gsize) {
                    const double s = get(v.s + i);
                    dnew[i] = cycle == 0 ? s : s + beta * dold[i];
                }
                ok = ok && grid_sync(gs, ws);
            }
            for (int i = gtid; i < n; i += gsize) {
                double d, q;
                if constexpr (cached) {
                    d = dnew[i];
                    q = ell_row(A.col, A.val, A.ncol[i], n, i, dnew);
                } else {
                    d = ROWS ? win.buf[i - win.w0] : dat(i);
                    q = times(i, dat);
                    ast(dnew + i, d);
                }
                if (ROWS) {
                    rd = d;
                    rq = q;
                }
                if (!ROWS || exact) put(v.q + i, q);
                acc[0] = dd_add_prod(acc[0], d, q);
            }
            spmv++;
            double o[1] = {0.0};
            ok = ok && grid_sum<1>(gs, ws, acc, o);
            t1 = exact ? seq_dot(dnew, v.q, n) : o[0];
        }
        const double alpha = delta_new / t1;
        for (int i = gtid; i < n; i += gsize) {
            rx = (ROWS ? rx : ald(x + i)) + alpha * (ROWS ? rd : cached ? dnew[i] : ald(dnew + i));
            ast(x + i, rx);
        }
        if (L.nh > 0) {
            ok = ok && grid_wait(gs, ws);
            if (kind == 0) constrain_v(L, x, gtid, gsize);
            else constrain_T(L, x, gtid, gsize);
        }
        const bool recompute = (cycle % 50) == 0;
        if (recompute || (ROWS && L.nh > 0)) {
            ok = ok && grid_wait(gs, ws);
            if (ROWS && gtid < n) rx = ald(x + gtid);   // a hanging value is written by another thread
            if (ROWS && recompute) win.fill(xat);
        }
        const double delta_old = delta_new;
        double res;
        {
            dd acc[1] = {dd_zero()};
            double mx[1] = {0.0}, o[2] = {0.0, 0.0};
            for (int i = gtid; i < n; i += gsize) {
                double r;
                if (recompute) r = b[i] - times(i, xat);
                else r = (ROWS ? rr : get(v.r + i)) - alpha * (ROWS ? rq : get(v.q + i));
                residual(i, r, acc[0]);
                mx[0] = fmax(mx[0], fabs(alpha * r));
            }
            if (recompute) spmv++;
            ok = ok && grid_reduce<1, 1>(gs, ws, acc, mx, o);
            delta_new = exact ? seq_dot(v.r, v.s, n) : o[0];
            res = o[1];
        }
        beta = delta_new / delta_old;
        double *t = dold;
        dold = dnew;
        dnew = t;
        cycle++;
        const bool brk = precond ? (res < accu) : (kind == 0 ? res < accu : (res < accu && cycle > 10));
        if (brk) break;
    }
    if (exact) ok = ok && grid_wait(gs, ws);   // every workgroup is done with seq_dot's vectors
    return cycle;
}

// The form of a solve that does not keep its rows (more rows than threads, or
// hanging nodes).  The fenced wait of CG_CACHED pays once a thread has more than
// one velocity row of 18 slots, or more than four temperature rows of 9.  us an
// inner iteration, CG_GATHER / CG_CACHED: 128x128 on 32 workgroups (two rows a
// thread) 22.8 / 18.1, on 8 74.9 / 46.5, on one 575 / 333; 512x512 on 256 (four
// rows) 51.0 / 46.0; an adapted mesh of 43 390 equations with one row a thread
// 20.7 / 21.5.  Temperature: 1024x512 on 256 workgroups (four rows a thread), a
// step 294 / 302 us; that adapted mesh on 5 (eight rows), an iteration 133 / 115.
template <int W>
__device__ __forceinline__ int pcg_persistent(const LevelDev &L, const EllMat &A, const RowReg<W> &row,
                                              const Window &win, double diag, const double *__restrict__ b, double *x,
                                              bool x_zero, double accu, int max_cycle, int precond, int kind, CgVecs v,
                                              const GridSync &gs, WaitState &ws, bool &ok, long long &spmv, bool exact)
{
    if (win.fits)
        return pcg_rows<W, CG_ROWS>(L, A, row, win, diag, b, x, x_zero, accu, max_cycle, precond, kind, v, gs, ws, ok,
                                    spmv, exact);
    if (A.n <= (kind == 0 ? 1 : 4) * (int)(gridDim.x * blockDim.x))
        return pcg_rows<W, CG_GATHER>(L, A, row, win, diag, b, x, x_zero, accu, max_cycle, precond, kind, v, gs, ws,
                                      ok, spmv, exact);
    return pcg_rows<W, CG_CACHED>(L, A, row, win, diag, b, x, x_zero, accu, max_cycle, precond, kind, v, gs, ws, ok,
                                  spmv, exact);
}

// ------------------------------------------------ stationary inner solvers
// The reference's solver="jc", "gs" and "mg" inner solves (Solver.c:82-89),
// with its arithmetic: every row sum in ascending-column order with the
// diagonal left out (prod += a_ij x_j, x_i = (b_i - prod) / a_ii), the stop on
// max |x - x_old| < accu, no hanging-node constraint.

// jacobi (Solver.c:1800-1864) over the whole grid: sweep k reads one buffer
// and writes the other (x_old needs no copy), both with agent-scope accesses;
// the wait that ends a sweep carries its maximum.  With one row a thread
// (row_window) the row stays in registers and x comes through the window: a
// sweep at 32x32 takes 2.4 us (14.5 us with a fenced barrier, its maxima
// collected in a second pass and every column's load waiting for the last);
// with more rows the loads of nine slots go together (128x128 on 4 workgroups, 16
// rows a thread: 68 us a sweep, 126 one column after the other).
// The caller's x must be complete; it is complete on return.
__device__ __forceinline__ int jacobi_grid(const EllMat &A, const RowReg<MCL_ROW_V> &row, const Window &win, double diag,
                                           const double *__restrict__ b, double *x, double *xt, double accu,
                                           int max_cycle, const GridSync &gs, WaitState &ws, bool &ok,
                                           long long &spmv)
{
    const int gtid = blockIdx.x * blockDim.x + threadIdx.x, gsize = gridDim.x * blockDim.x;
    const int n = A.n;
    const bool mine = gtid < n;
    int dslot = -1;
    double bi = 0.0;
    if (win.fits && mine) {
        bi = b[gtid];
#pragma unroll
        for (int u = 0; u < MCL_ROW_V; u++)
            if (u < row.n && row.off[u] == 8u * (unsigned)(gtid - win.w0)) dslot = u;
    }
    double *src = x, *dst = xt;
    int cycle = 0;
    // this thread's rows of a sweep, their loads issued nine slots at a time
    auto sweep = [&](double &mx) {
        for (int i = gtid; i < n; i += gsize) {
            double prod = 0.0, dg = 1.0;
            const int nc = A.ncol[i];
            for (int j = 0; j < nc; j += 9) {
                int c[9];
                double v[9], xv[9];
#pragma unroll
                for (int u = 0; u < 9; u++) {
                    c[u] = j + u < nc ? A.col[(j + u) * n + i] : -1;
                    v[u] = j + u < nc ? A.val[(j + u) * n + i] : 0.0;
                }
#pragma unroll
                for (int u = 0; u < 9; u++) xv[u] = c[u] >= 0 ? ald(src + c[u]) : 0.0;
#pragma unroll
                for (int u = 0; u < 9; u++) {
                    if (c[u] == i) dg = v[u];
                    else if (c[u] >= 0) prod += v[u] * xv[u];
                }
            }
            const double xn = (b[i] - prod) / dg;
            ast(dst + i, xn);
            mx = fmax(mx, fabs(xn - ald(src + i)));
        }
    };
    while (ok && cycle < max_cycle) {
        double mx[1] = {0.0}, o[1] = {0.0};
        if (win.fits) {
            win.fill([&](int j) { return ald(src + j); });
            if (mine) {
                const double xn = (bi - row.dot(win.buf, dslot)) / diag;
                ast(dst + gtid, xn);
                mx[0] = fabs(xn - win.buf[gtid - win.w0]);
            }
        } else {
            sweep(mx[0]);
        }
        spmv++;
        dd none[1] = {dd_zero()};
        ok = ok && grid_reduce<0, 1>(gs, ws, none, mx, o);
        double *t = src;
        src = dst;
        dst = t;
        cycle++;
        if (o[0] < accu) break;
    }
    if (src != x) {
        for (int i = gtid; i < n; i += gsize) ast(x + i, ald(src + i));
        ok = ok && grid_wait(gs, ws);
    }
    return cycle;
}

// gauss_seidel (Solver.c:1866-1928) in one workgroup: each sweep walks the
// level's wavefront groups in order, the rows of a group in parallel.
__device__ int gs_block(const GsLevelDev &A, const double *b, double *x, double *xt, double accu, int max_cycle,
                        double *ldsm, long long &spmv)
{
    const int t = threadIdx.x, n = A.n;
    int cycle = 0;
    while (cycle < max_cycle) {
        for (int i = t; i < n; i += blockDim.x) xt[i] = x[i];
        __syncthreads();
        for (int g = 0; g < A.nsched; g++) {
            const int k1 = A.sptr[g + 1];
            for (int k = A.sptr[g] + t; k < k1; k += blockDim.x) {
                const int i = A.srows[k];
                double prod = 0.0, diag = 1.0;
                const int nc = A.ncol[i];
                for (int j = 0; j < nc; j++) {
                    const int c = A.col[j * n + i];
                    const double v = A.val[j * n + i];
                    if (c != i) prod += v * x[c];
                    else diag = v;
                }
                x[i] = (b[i] - prod) / diag;
            }
            __syncthreads();
        }
        spmv++;
        cycle++;
        double mx = 0.0;
        for (int i = t; i < n; i += blockDim.x) mx = fmax(mx, fabs(x[i] - xt[i]));
        if (block_max(mx, ldsm) < accu) break;
    }
    return cycle;
}

// multigrid + MG (Solver.c:668-769) in one workgroup, levels coarsest first
// (lv[0] = min_level, lv[nl-1] = the finest).  Below the finest the iterate
// is the level's err vector itself, so the prolongation overwrites the
// smoothed iterate before it is added, as in the reference.  err keeps its
// values across V-cycles and is zeroed once per call (initial_error).
__device__ int mg_block(const GsLevelDev *lv, int nl, const double *b, double *x, double *xt_cycle, double *xt,
                        double accu, int mg_cycle, int fi, int ci, double *ldsm, long long &spmv)
{
    const int t = threadIdx.x, top = nl - 1;
    for (int l = 0; l < nl; l++)
        for (int i = t; i < lv[l].n; i += blockDim.x) lv[l].err[i] = 0.0;
    __syncthreads();
    const int n = lv[top].n;
    int cycle = 0;
    bool conv = false;
    while (!conv && cycle < mg_cycle) {
        for (int i = t; i < n; i += blockDim.x) xt_cycle[i] = x[i];
        __syncthreads();
        for (int l = top; l >= 1; l--) {
            const GsLevelDev &A = lv[l];
            const double *rhs = l == top ? b : A.rhs;
            double *xl = l == top ? x : A.err;
            gs_block(A, rhs, xl, xt, accu, fi, ldsm, spmv);
            // get_residual (Solver.c:1291-1316): res = b, then res -= a_ij x_j in column order
            for (int i = t; i < A.n; i += blockDim.x) {
                double r = rhs[i];
                const int nc = A.ncol[i];
                for (int j = 0; j < nc; j++) r -= A.val[j * A.n + i] * xl[A.col[j * A.n + i]];
                A.resu[i] = r;
            }
            __syncthreads();
            // project_res (Solver.c:770-832): injection
            for (int k = t; k < A.nproj; k += blockDim.x) lv[l - 1].rhs[A.proj_l[k]] = A.resu[A.proj_u[k]];
            __syncthreads();
        }
        gs_block(lv[0], lv[0].rhs, lv[0].err, xt, accu, 1000, ldsm, spmv);
        for (int l = 1; l <= top; l++) {
            const GsLevelDev &A = lv[l];
            const double *rhs = l == top ? b : A.rhs;
            double *xl = l == top ? x : A.err;
            const double *ec = lv[l - 1].err;
            // interp_error (Solver.c:1009-1143, local part)
            for (int u = t; u < A.n; u += blockDim.x) {
                const int m = A.pn[u];
                if (m > 0) {
                    double v = 0.0;
                    for (int a = 0; a < m; a++) {
                        const int c = A.pcol[a * A.n + u];
                        if (c != -1) v += ec[c];
                    }
                    A.err[u] = v / m;
                }
            }
            __syncthreads();
            for (int i = t; i < A.n; i += blockDim.x) xl[i] += A.err[i];
            __syncthreads();
            gs_block(A, rhs, xl, xt, accu, ci, ldsm, spmv);
        }
        double mx = 0.0;
        for (int i = t; i < n; i += blockDim.x) mx = fmax(mx, fabs(x[i] - xt_cycle[i]));
        conv = block_max(mx, ldsm) < accu;
        cycle++;
    }
    return cycle;
}

// The inner solve of citcom_solver (Solver.c:82-89) for the chosen solver, on
// a right-hand side that this thread's rows have just been written to and an x
// that is complete or, with x_zero, just zeroed; x is complete on return.
template <int SOLVER>
__device__ __forceinline__ int inner_solve(const UzawaParams &P, const LevelDev &L, const EllMat &K,
                                           const RowReg<MCL_ROW_V> &row, const Window &win, double diag, const double *b,
                                           double *x, bool x_zero, CgVecs cv, WaitState &ws, double *ldsm, bool &ok,
                                           long long &spmv)
{
    if constexpr (SOLVER == MCL_INNER_CG) {
        return pcg_persistent<MCL_ROW_V>(L, K, row, win, diag, b, x, x_zero, P.accuracy, P.max_cg_cycle, P.cg_precondition, 0,
                                  cv, P.gs, ws, ok, spmv, P.exact_dots != 0);
    } else if constexpr (SOLVER == MCL_INNER_JC) {
        if (x_zero) ok = ok && grid_wait(P.gs, ws);
        return jacobi_grid(K, row, win, diag, b, x, P.xt, P.accuracy, 1000, P.gs, ws, ok, spmv);
    } else {
        // one workgroup, plain accesses
        ok = ok && grid_sync(P.gs, ws);
        const int c = SOLVER == MCL_INNER_GS
                          ? gs_block(P.gsl[P.ngsl - 1], b, x, P.xt, P.accuracy, 1000, ldsm, spmv)
                          : mg_block(P.gsl, P.ngsl, b, x, P.xt2, P.xt, P.accuracy, P.mg_cycle, P.mg_finest_iteration,
                                     P.mg_coarse_iteration, ldsm, spmv);
        ok = ok && grid_sync(P.gs, ws);
        return c;
    }
}

// citcom_solver (Solver.c:14-249) as one persistent kernel.  Vectors that other
// workgroups read (u1, d and p at the start, z, s) are stored and loaded with
// agent-scope accesses; the rest belong to the thread of the row or element
// (grid stride).  An Uzawa iteration has three phases of its own: the search
// direction s2 = z1 + delta s1 with G s2 (gathered as z1 + delta s1, the same
// rounding), which the inner solve's start follows without a wait; G^T u1 with
// s2.G^T u1; the updates with their norms and the next z and r.z.  (r0.z0 is
// the previous iteration's r1.z1: the same vectors, the same sum.)
// One kernel per inner solver (each then has the registers to itself).
template <int SOLVER>
__global__ void __launch_bounds__(MCL_BLOCK) k_uzawa_fp64(UzawaParams P)
{
    __shared__ double ldsm[MCL_BLOCK / MCL_WAVE];
    const LevelDev &L = P.L;
    const int gtid = blockIdx.x * blockDim.x + threadIdx.x, gsize = gridDim.x * blockDim.x;
    const int neq = L.neq, nel = L.nel;
    if (blockIdx.x == 0 && threadIdx.x == 0) P.stats->t_begin = wall_clock64();
    WaitState ws;
    bool ok = sync_begin(P.gs, ws);
    long long spmv = 0, inner = 0;
    EllMat K{L.Kcol, L.Kncol, L.Kval, L.Kdiag, nullptr, neq};
    CgVecs cv{P.cg_r, P.cg_s, P.cg_d, P.cg_q, P.cg_d2};
    RowReg<MCL_ROW_V> row;
    Window win{nullptr, 0, 0, false};
    double diag = 1.0;
    if constexpr (SOLVER == MCL_INNER_CG || SOLVER == MCL_INNER_JC) {
        __shared__ double buf[MCL_WINDOW];
        win = row_window(row, K.col, K.ncol, K.val, neq, buf, P.rows_fit != 0);
        if (gtid < neq) diag = K.diag[gtid];
    }
    for (int e = gtid; e < nel; e += gsize) P.BAB[e] = bab_elem(L, e);
    double *r0 = P.r0, *r1 = P.r1, *r2 = P.r2, *z0 = P.z0, *z1 = P.z1, *s1 = P.s1, *s2 = P.s2;
    double dv = 1.0, dp = 1.0, r1z1 = 0.0, r0z0 = 0.0;
    int cycle = 0;
    bool first = true;   // the solve for the initial velocity's defect comes before the loop's
    auto zvec = [&](int e, double r) { return P.schur ? r / P.BAB[e] : P.BAB[e] * r; };
    while (true) {
        // the inner solve's right-hand side, then its one call site
        if (first) {
            // u1 = K d ; Ah = F - G p - u1   (:67-77)
            for (int i = gtid; i < neq; i += gsize) {
                double u = ell_row(L.Kcol, L.Kval, L.Kncol[i], neq, i, P.d);
                double gp = g_row(L, i, P.p);
                ast(P.u1 + i, u);
                P.Ahv[i] = L.F[i] - gp - u;
            }
            spmv++;
            ok = ok && grid_wait(P.gs, ws);   // the solve starts from u1
        } else {
            if (!(ok && (dv > P.citcom_accu || (dp > P.citcom_accu && P.check_v_only == 0)) &&
                  cycle < P.max_citcom_cycle))
                break;
            if (!(r1z1 == r1z1)) P.stats->nan_flag = 1;
            const double delta = cycle > 0 ? r1z1 / r0z0 : 0.0;
            auto s2at = [&](int e) { return cycle == 0 ? ald(z1 + e) : ald(z1 + e) + delta * ald(s1 + e); };
            for (int e = gtid; e < nel; e += gsize) ast(s2 + e, s2at(e));
            // Ah = G s2 ; u1 = 0 ; K u1 = Ah
            for (int i = gtid; i < neq; i += gsize) {
                P.Ahv[i] = g_row_ld(L, i, s2at);
                ast(P.u1 + i, 0.0);
            }
        }
        inner += inner_solve<SOLVER>(P, L, K, row, win, diag, P.Ahv, P.u1, !first, cv, ws, ldsm, ok, spmv);
        if (first) {
            first = false;
            for (int i = gtid; i < neq; i += gsize) ast(P.d + i, ald(P.d + i) + ald(P.u1 + i));
            ok = ok && grid_wait(P.gs, ws);
            // r1 = G^T d, z1 = BAB r1 (or r1 / BAB); r1.z1
            dd acc[1] = {dd_zero()};
            for (int e = gtid; e < nel; e += gsize) {
                const double r = gt_elem_ld(L, e, [&](int j) { return ald(P.d + j); }), z = zvec(e, r);
                ast(r1 + e, r);
                ast(z1 + e, z);
                acc[0] = dd_add_prod(acc[0], r, z);
            }
            double o[1] = {0.0};
            ok = ok && grid_sum<1>(P.gs, ws, acc, o);
            r1z1 = P.exact_dots ? seq_dot(r1, z1, nel) : o[0];
            continue;
        }
        // Ah = G^T u1 ; alpha = r1.z1 / s2.Ah
        double alpha;
        {
            dd acc[1] = {dd_zero()};
            for (int e = gtid; e < nel; e += gsize) {
                double a = gt_elem_ld(L, e, [&](int j) { return ald(P.u1 + j); });
                ast(P.Ahp + e, a);
                acc[0] = dd_add_prod(acc[0], ald(s2 + e), a);
            }
            double o[1] = {0.0};
            ok = ok && grid_sum<1>(P.gs, ws, acc, o);
            if (P.exact_dots) o[0] = seq_dot(s2, P.Ahp, nel);
            alpha = r1z1 / o[0];
        }
        {
            dd acc[5] = {dd_zero(), dd_zero(), dd_zero(), dd_zero(), dd_zero()};
            for (int e = gtid; e < nel; e += gsize) {
                const double r = ald(r1 + e) - alpha * ald(P.Ahp + e), se = ald(s2 + e), z = zvec(e, r);
                const double pe = ald(P.p + e) + alpha * se;
                ast(r2 + e, r);
                ast(P.p + e, pe);
                ast(z0 + e, z);   // z0's buffer becomes z1
                acc[0] = dd_add_prod(acc[0], se, se);
                acc[1] = dd_add_prod(acc[1], pe, pe);
                acc[4] = dd_add_prod(acc[4], r, z);
            }
            for (int i = gtid; i < neq; i += gsize) {
                const double u = ald(P.u1 + i), di = ald(P.d + i) - alpha * u;
                ast(P.d + i, di);
                acc[2] = dd_add_prod(acc[2], u, u);
                acc[3] = dd_add_prod(acc[3], di, di);
            }
            double o[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
            ok = ok && grid_sum<5>(P.gs, ws, acc, o);
            if (P.exact_dots) {
                o[0] = seq_dot(s2, s2, nel);
                o[1] = seq_dot(P.p, P.p, nel);
                o[2] = seq_dot(P.u1, P.u1, neq);
                o[3] = seq_dot(P.d, P.d, neq);
                o[4] = seq_dot(r2, z0, nel);
                ok = ok && grid_wait(P.gs, ws);   // the next phases write s2's and u1's successors
            }
            dp = alpha * sqrt(o[0] / (1.0e-32 + o[1]));
            dv = alpha * sqrt(o[2] / (1.0e-32 + o[3]));
            r0z0 = r1z1;
            r1z1 = o[4];
        }
        cycle++;
        double *sh;
        sh = s1; s1 = s2; s2 = sh;
        sh = r0; r0 = r1; r1 = r2; r2 = sh;
        sh = z0; z0 = z1; z1 = sh;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        P.stats->cycles = cycle;
        P.stats->dv = dv;
        P.stats->dp = dp;
        P.stats->inner = inner;
        P.stats->spmv = spmv;
        P.stats->aborted = ok ? 0 : 1;
        if (!(dv == dv) || !(dp == dp)) P.stats->nan_flag = 1;
        P.stats->t_end = wall_clock64();
    }
    sync_end(P.gs, ws);
}

const void *mcl_uzawa_fp64_kernel(int solver)
{
    switch (solver) {
    case MCL_INNER_JC: return (const void *)k_uzawa_fp64<MCL_INNER_JC>;
    case MCL_INNER_GS: return (const void *)k_uzawa_fp64<MCL_INNER_GS>;
    case MCL_INNER_MG: return (const void *)k_uzawa_fp64<MCL_INNER_MG>;
    default: return (const void *)k_uzawa_fp64<MCL_INNER_CG>;
    }
}

// Zero n 32-bit words (a kernel rather than hipMemsetAsync, so that a caller
// may capture it in a graph).
__global__ void k_zero_words(unsigned *p, long long n)
{
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        p[i] = 0u;
}

// v_to_nodes (Solver.c:1319-1343)
__global__ void k_v_to_nodes(LevelDev L, const double *__restrict__ d, double *__restrict__ V)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < L.nno; i += gridDim.x * blockDim.x)
        for (int k = 0; k < 2; k++) {
            int j = L.id[k * L.nno + i];
            V[k * L.nno + i] = j >= 0 ? d[j] : L.v_bc_val[k * L.nno + i];
        }
}

// compute_stress element part (Grain_size_evolution.c:154-209)
__global__ void k_stress_elem(LevelDev L, const double *__restrict__ vis,
                              const double *__restrict__ V, double *__restrict__ es, double *__restrict__ area)
{
    for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < L.nel; e += gridDim.x * blockDim.x) {
        int lev = L.elev[e];
        double dxdxi = 0.5 * L.lvl_dx[lev], dzdeta = 0.5 * L.lvl_dz[lev];
        double jac = dxdxi * dzdeta - 0.0 * 0.0;
        double eta = 0.0, u11 = 0.0, u22 = 0.0, u12 = 0.0;
        for (int a = 0; a < 4; a++) eta += 0.25 * vis[L.ienl[a * L.nel + e]];
        for (int a = 0; a < 4; a++) {
            int k = L.ienl[a * L.nel + e];
            double ax = c_shape.dxic[a] * dzdeta - c_shape.detac[a] * 0.0;
            double az = c_shape.detac[a] * dxdxi - c_shape.dxic[a] * 0.0;
            u11 += ax * V[k];
            u22 += az * V[L.nno + k];
            u12 += az * V[k];
        }
        u11 /= jac;
        u22 /= jac;
        u12 /= jac;
        double u21 = u12;
        double sr = u11 * u11 + u22 * u22 + u12 * u21 * 2.0;
        sr = sqrt(0.5 * sr);
        es[e] = 2.0 * eta * sr;
        int n0 = L.ienl[e], n2 = L.ienl[2 * L.nel + e];
        area[e] = (L.X[n2] - L.X[n0]) * (L.X[L.nno + n2] - L.X[L.nno + n0]);
    }
}

// p_to_nodes (Solver.c:1345-1366): area-weighted mean over the node's elements.
__global__ void k_stress_node(LevelDev L, const double *__restrict__ es, const double *__restrict__ area,
                              double *__restrict__ stress)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < L.nno; i += gridDim.x * blockDim.x) {
        double s = 0.0, t = 0.0;
        for (int k = 0; k < L.p2n_cnt[i]; k++) {
            int e = L.p2n_el[k * L.nno + i];
            s += area[e] * es[e];
            t += area[e];
        }
        stress[i] = s / t;
    }
}

// True residual norms after a solve: |F - K d - G p|^2, |G^T d|^2, |F|^2 as
// partial sums in reduction slots 12..14 (k_collect3 finishes them).
// Residual norms after a solve: |F - K d - G p|^2, |G^T d|^2 and |F|^2.
// galerkin != 0 (the mixed path on meshes with hanging nodes, which solves
// C^T K C u_f = C^T b): the momentum residual and F are measured in the
// constrained space, C^T (F - K d - G p) and C^T F, rows of hanging
// equations folded into their free parents.
__global__ void k_residuals(LevelDev L, RedBuf rb, const double *__restrict__ d, const double *__restrict__ p,
                            int galerkin)
{
    __shared__ dd lds[MCL_RED_ROWS][MCL_BLOCK / MCL_WAVE];
    const int gtid = blockIdx.x * blockDim.x + threadIdx.x, gsize = gridDim.x * blockDim.x;
    const bool gal = galerkin && L.nh > 0;
    dd acc[3] = {dd_zero(), dd_zero(), dd_zero()};
    for (int i = gtid; i < L.neq; i += gsize) {
        if (gal && L.hp_n[i] != 0) continue;
        double r = L.F[i] - ell_row(L.Kcol, L.Kval, L.Kncol[i], L.neq, i, d) - g_row(L, i, p);
        double f = L.F[i];
        if (gal) {
            for (int t = L.ch_ptr[i]; t < L.ch_ptr[i + 1]; t++) {
                const int h = L.ch_i[t];
                const double w = L.ch_w[t];
                r += w * (L.F[h] - ell_row(L.Kcol, L.Kval, L.Kncol[h], L.neq, h, d) - g_row(L, h, p));
                f += w * L.F[h];
            }
        }
        acc[0] = dd_add_prod(acc[0], r, r);
        acc[2] = dd_add_prod(acc[2], f, f);
    }
    for (int e = gtid; e < L.nel; e += gsize) {
        double c = gt_elem(L, e, d);
        acc[1] = dd_add_prod(acc[1], c, c);
    }
    reduce_publish<3>(rb, acc, lds);
}

__global__ void k_collect3(RedBuf rb, int nblocks, double *out)
{
    __shared__ dd lds[MCL_RED_ROWS][MCL_BLOCK / MCL_WAVE];
    double o[3];
    reduce_collect<3>(rb, nblocks, o, lds);
    if (threadIdx.x == 0)
        for (int r = 0; r < 3; r++) out[r] = o[r];
}

// ------------------------------------------------------------------ heat step

// SUPG tau, calculate_artificial_diffusivity (Update_temperature.c:241-291),
// and each element's advective time-step bound (advection_dt, :135-177, which
// uses the sizes L of the last element of the diffusive loop for every element).
__device__ __forceinline__ void elem_center_u(const LevelDev &L, int e, const double *__restrict__ V, double u[2])
{
    for (int d = 0; d < 2; d++) {
        double s = 0.0;
        for (int a = 0; a < 4; a++) s += 0.25 * V[d * L.nno + L.ienl[a * L.nel + e]];
        u[d] = s;
    }
}

// Heat row assembly (K_matrix_heat :293-423 with get_element_K_heat,
// F_matrix_heat :425-508, C_matrix_heat :510-594): one thread per heat row,
// element-ascending sums accumulated in the thread's own LDS column for rows of
// at most 9 slots (written to HBM once), else in place in the row's own slots;
// the additions to each slot come in the same order either way.
#define MCL_HEAT_LDS_SLOTS 9
__device__ __forceinline__ void heat_assemble_row(const LevelDev &L, const HeatParams &H, const ShapeTables &S, int P,
                                                  double *lk, double *lc)
{
    const int n = L.heq_node[P];
    const int nadj = L.p2n_cnt[n];
    const int nT = L.neqT;
    const bool inl = L.WT <= MCL_HEAT_LDS_SLOTS;
    for (int s = 0; s < L.WT; s++) {
        if (inl) {
            lk[s * MCL_BLOCK] = 0.0;
            lc[s * MCL_BLOCK] = 0.0;
        } else {
            H.hK[s * nT + P] = 0.0;
            H.hC[s * nT + P] = 0.0;
        }
    }
    double F = 0.0;
    for (int k = 0; k < nadj; k++) {
        int e = L.p2n_el[k * L.nno + n], a = L.p2n_a[k * L.nno + n];
        int lev = L.elev[e];
        double dxdxi = 0.5 * L.lvl_dx[lev], dzdeta = 0.5 * L.lvl_dz[lev];
        double jac = dxdxi * dzdeta - 0.0 * 0.0;
        double u1 = 0.0, u2 = 0.0;
        for (int c = 0; c < 4; c++) {
            int kn = L.ienl[c * L.nel + e];
            u1 += H.V[kn] * 0.25;
            u2 += H.V[L.nno + kn] * 0.25;
        }
        double t0 = ald(H.tau + e), t1 = ald(H.tau + L.nel + e);
        for (int b = 0; b < 4; b++) {
            double kv = 0.0, cv = 0.0;
            for (int g = 0; g < 4; g++) {
                double ax = S.dxi[a][g] * dzdeta - S.deta[a][g] * 0.0;
                double az = S.deta[a][g] * dxdxi - S.dxi[a][g] * 0.0;
                double bx = S.dxi[b][g] * dzdeta - S.deta[b][g] * 0.0;
                double bz = S.deta[b][g] * dxdxi - S.dxi[b][g] * 0.0;
                double nh = t0 * ax + t1 * az;
                double tt1 = u1 * S.N[a][g] * bx + u2 * S.N[a][g] * bz;
                double tt2 = u1 * nh * bx + u2 * nh * bz;
                double tt3 = ax * 1.0 * bx + ax * 0.0 * bz + az * 0.0 * bx + az * 1.0 * bz;
                kv += tt1 + (tt2 + tt3) / jac;
                cv += (S.N[a][g] + nh) * S.N[b][g];
            }
            cv *= jac;
            int slot = L.Tslot[(k * 4 + b) * nT + P];
            if (slot >= 0) {
                if (inl) {
                    lk[slot * MCL_BLOCK] += kv;
                    lc[slot * MCL_BLOCK] += cv;
                } else {
                    H.hK[slot * nT + P] += kv;
                    H.hC[slot * nT + P] += cv;
                }
            }
            int nb = L.ienl[b * L.nel + e];
            if (L.T_bc[nb] == 'T') F -= kv * L.T_bc_val[nb];
        }
    }
    for (int k = 0; k < nadj; k++) {
        int e = L.p2n_el[k * L.nno + n], a = L.p2n_a[k * L.nno + n];
        int lev = L.elev[e];
        double dxdxi = 0.5 * L.lvl_dx[lev], dzdeta = 0.5 * L.lvl_dz[lev];
        double jac = dxdxi * dzdeta - 0.0 * 0.0;
        double t0 = ald(H.tau + e), t1 = ald(H.tau + L.nel + e);
        int nat = 0;
        for (int c = 0; c < 4; c++)
            if (L.T_bc[L.ienl[c * L.nel + e]] == 'F') nat += c;
        if (nat == 3) nat = 1;
        else if (nat == 1 || nat == 5) nat = 2;
        else if (nat == 0 || nat == 2) nat = 0;
        double f = 0.0;
        for (int g = 0; g < 4; g++) {
            double ax = S.dxi[a][g] * dzdeta - S.deta[a][g] * 0.0;
            double az = S.deta[a][g] * dxdxi - S.dxi[a][g] * 0.0;
            double nh = t0 * ax + t1 * az;
            f += (S.N[a][g] + nh) * H.Q;
        }
        f *= jac;
        if (nat != 0) f -= 0.5 * L.lvl_dz[lev] * L.T_bc_val[L.ienl[a * L.nel + e]];
        F += f;
    }
    H.hF[P] = F;
    if (inl)
        for (int s = 0; s < L.WT; s++) {
            H.hK[s * nT + P] = lk[s * MCL_BLOCK];
            H.hC[s * nT + P] = lc[s * MCL_BLOCK];
        }
}

// update_temperature (Update_temperature.c:3-133) as one persistent kernel.
__global__ void __launch_bounds__(MCL_BLOCK) k_heat_fp64(HeatParams H)
{
    __shared__ double lds[2 * MCL_HEAT_LDS_SLOTS * MCL_BLOCK];
    __shared__ ShapeTables S;   // a thread's corner picks its entries: LDS serves 64 different ones at once
    const LevelDev &L = H.L;
    const int gtid = blockIdx.x * blockDim.x + threadIdx.x, gsize = gridDim.x * blockDim.x;
    const int n = L.neqT, nel = L.nel;
    for (int t = threadIdx.x; t < (int)(sizeof S / sizeof(double)); t += blockDim.x)
        ((double *)&S)[t] = ((const double *)&c_shape)[t];
    WaitState ws;
    bool ok = sync_begin(H.gs, ws);
    long long spmv = 0;
    // tau per element and the advective dt bound: the smallest 0.5 / uu is 0.5
    // over the largest uu (rounding is monotone)
    double umax[1] = {0.0};
    for (int e = gtid; e < nel; e += gsize) {
        int lev = L.elev[e];
        double Lx = L.lvl_dx[lev], Lz = L.lvl_dz[lev];
        double u[2];
        elem_center_u(L, e, H.V, u);
        double al[2], xi[2];
        double Ld[2] = {Lx, Lz};
        for (int d = 0; d < 2; d++) {
            al[d] = 0.5 * u[d] * Ld[d] / 1.0;
            xi[d] = fabs(al[d]) < H.accuracy ? 0.0 : cosh(al[d]) / sinh(al[d]) - 1.0 / al[d];
        }
        double us = (u[0] * u[0] + u[1] * u[1]);
        double kh = (xi[0] * u[0] * Ld[0] + xi[1] * u[1] * Ld[1]) * 0.5;
        ast(H.tau + e, kh * u[0] / us);
        ast(H.tau + nel + e, kh * u[1] / us);
        // advection_dt with the sizes of the last element (H.Llast)
        double uu = fabs(u[0]) / H.Llast0 + fabs(u[1]) / H.Llast1;
        umax[0] = fmax(umax[0], uu);
    }
    double dt;
    {
        dd none[1] = {dd_zero()};
        double o[1] = {0.0};
        ok = ok && grid_reduce<0, 1>(H.gs, ws, none, umax, o);
        const double step = 0.5 / o[0];
        dt = step < 1e10 ? step : 1e10;
        dt = dt < H.diff_dt ? dt : H.diff_dt;
        dt = dt * 0.75;
    }
    // rows, matrices and right-hand sides belong to their thread from here on;
    // the waits are those of the vectors that the products gather
    for (int P = gtid; P < n; P += gsize)
        heat_assemble_row(L, H, S, P, lds + threadIdx.x, lds + MCL_HEAT_LDS_SLOTS * MCL_BLOCK + threadIdx.x);
    EllMat Ch{L.Tcol, L.Tncol, H.hC, nullptr, L.Tdiag_slot, n};
    EllMat Ah{L.Tcol, L.Tncol, H.hA, nullptr, L.Tdiag_slot, n};
    CgVecs cv{H.cg_r, H.cg_s, H.cg_d, H.cg_q, H.cg_d2};
    auto hd = [&](int j) { return ald(H.hd + j); };
    // one of the two matrices at a time in registers; the LDS columns of the
    // assembly become the window
    static_assert(2 * MCL_HEAT_LDS_SLOTS * MCL_BLOCK >= MCL_WINDOW, "the window lies in the assembly's LDS");
    RowReg<MCL_ROW_T> row;
    auto cg = [&](const EllMat &A, double *x, bool x_zero, int max_cycle) __attribute__((always_inline)) {
        __syncthreads();
        const Window win = row_window(row, A.col, A.ncol, A.val, n, lds, H.rows_fit != 0);
        const double diag = gtid < n ? ell_diag(A, gtid) : 1.0;
        return pcg_persistent<MCL_ROW_T>(L, A, row, win, diag, H.B, x, x_zero, 1e-3, max_cycle, H.cg_precondition, 1, cv, H.gs,
                                 ws, ok, spmv, H.exact_dots != 0);
    };
    int init_cycles = 0;
    if (H.first_call) {
        // initial_T_dot (:179-239)
        for (int i = gtid; i < n; i += gsize) ast(H.hd + i, H.T[L.heq_node[i]]);
        ok = ok && grid_wait(H.gs, ws);
        for (int i = gtid; i < n; i += gsize) {
            H.B[i] = H.hF[i] - ell_row_ld(L.Tcol, H.hK, L.Tncol[i], n, i, hd);
            ast(H.hdd + i, 0.0);
        }
        init_cycles = cg(Ch, H.hdd, true, 400);
    }
    const double td = H.theta * dt;
    for (int i = gtid; i < n; i += gsize) {
        double ct = ell_row_ld(L.Tcol, H.hC, L.Tncol[i], n, i, hd);
        H.d0[i] = hd(i);
        H.B[i] = H.hF[i] + ct / td;
        for (int s = 0; s < L.Tncol[i]; s++) H.hA[s * n + i] = H.hC[s * n + i] / td + H.hK[s * n + i];
    }
    int cycles = cg(Ah, H.hd, false, 1000);
    for (int i = gtid; i < L.nno; i += gsize) {
        int k = L.heat_id[i];
        H.T[i] = k >= 0 ? hd(k) : L.T_bc_val[i];
    }
    for (int i = gtid; i < n; i += gsize)
        ast(H.hdd + i, 1.0 / (H.theta * dt) * (hd(i) - H.d0[i]) - (1.0 - H.theta) / H.theta * ald(H.hdd + i));
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        H.stats->cycles = cycles;
        H.stats->init_cycles = init_cycles;
        H.stats->dt = dt;
        H.stats->aborted = ok ? 0 : 1;
        *H.model_time += dt;
    }
    sync_end(H.gs, ws);
}
