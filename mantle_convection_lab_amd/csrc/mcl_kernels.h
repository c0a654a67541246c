// Device-side data layout of one quadtree level and the parameter blocks of
// the persistent kernels.  Shared by the kernel translation units and the
// host C-ABI implementation (mcl_api.cpp).
#pragma once
#include "mcl_device.h"

// One quadtree level resident in HBM.  Arrays indexed [k][i] are stored
// slot-major (k * n + i) so that consecutive threads (consecutive i) read
// consecutive addresses.
struct LevelDev {
    int L, lev;
    int nel, nno, neq, neqT, gnox, gnoz;
    // level tables: element sizes per quadtree level and the element gradient
    // vector g[level][p] of get_element_G (Build_matrix.c:346-381)
    const double *lvl_dx, *lvl_dz;   // [MCL_MAX_LEVELS]
    const double *gtab;              // [MCL_MAX_LEVELS][8]
    // elements
    const int *ienl;                 // [4][nel] local node index of corner a
    const int *elev;                 // [nel] element quadtree level
    const int *lm;                   // [8][nel] velocity eq of (dof d, corner a) at (d*4+a)
    const int *gt_row;               // [8][nel] free velocity rows of the element, ascending, -1 padded
    const double *gt_val;            // [8][nel] G of (gt_row, element)
    const int *g_el;                 // [4][neq] elements of the row's node, ascending, -1 padded
    const double *g_val;             // [4][neq] G of (row, g_el)
    // nodes
    const int *node;                 // [nno] global node id
    const int *p2n_cnt;              // [nno] number of elements at the node
    const int *p2n_el;               // [4][nno] those elements, ascending
    const int *p2n_a;                // [4][nno] corner index of the node in each
    const int *id;                   // [2][nno]
    const int *heat_id;              // [nno]
    const signed char *v_bc;         // [2][nno]
    const double *v_bc_val;          // [2][nno]
    const signed char *T_bc;         // [nno]
    const double *T_bc_val;          // [nno]
    const double *X;                 // [2][nno]
    // velocity rows (ELL, sorted columns)
    const int *veq_node;             // [neq] local node of the equation
    const int *veq_dof;              // [neq]
    int WK;
    const int *Kcol;                 // [WK][neq]
    const int *Kncol;                // [neq]
    const signed char *Kslot;        // [32][neq]: slot of (adjacent element k, element dof q)
    double *Kval;                    // [WK][neq]
    double *Kdiag, *F;               // [neq]
    // heat rows
    const int *heq_node;             // [neqT] local node of the heat equation
    int WT;
    const int *Tcol;                 // [WT][neqT]
    const int *Tncol;                // [neqT]
    const signed char *Tslot;        // [16][neqT]
    const int *Tdiag_slot;           // [neqT]
    // hanging nodes
    int nh, h_serial;
    const int *h_ni, *h_ci;          // [nh], [2][nh]
    // Galerkin constraint u = C u_free of the mixed path: hanging equation h
    // has hp_n[h] (1..4) free parents hp_i[k][h] with weights hp_w[k][h]
    // (hp_n = 0 for free equations; chains of hanging parents are expanded,
    // Dirichlet parents dropped); ch_* is the transpose (children of each
    // free equation, CSR)
    const int *hp_n, *hp_i;          // [neq], [4][neq]
    const double *hp_w;              // [4][neq]
    const int *ch_ptr, *ch_i;        // [neq + 1], [...]
    const double *ch_w;
};

#define MCL_PHASES 16
struct DevStats {
    int cycles, init_cycles, aborted, nan_flag;
    double dv, dp, dt;
    long long inner, spmv;
    long long phase[MCL_PHASES];   // 100 MHz ticks per solver phase (builds with MCL_PHASE_TIMERS)
    double probe_r1;               // |G^T d|^2 after the first inner solve (probe launches)
    long long t_begin, t_end;      // device wall clock (wall_clock64) at the FP64 Uzawa kernel's start and end
};

// One quadtree level for the reference's stationary inner solvers
// (Gauss-Seidel and the stand-alone multigrid, Solver.c:668-1316,1866-1928):
// the level's FP64 K in ELL form, the Gauss-Seidel wavefront schedule (rows
// grouped so that every row comes after each lower-numbered row it couples to
// and before each higher-numbered one: updating a group's rows in parallel
// reproduces the sequential sweep exactly), the transfer maps and the level's
// vectors.
struct GsLevelDev {
    int n, WK;
    const int *col, *ncol;   // [WK][n], [n]
    const double *val;       // [WK][n]
    int nsched;
    const int *sptr;         // [nsched + 1]
    const int *srows;        // [n] rows of group g: srows[sptr[g] .. sptr[g+1])
    // interp from the level below: row u <- mean of pn[u] entries pcol[a][u] (-1 skipped, still counted)
    const int *pn, *pcol;    // [n], [4][n]
    // injection into the level below: its row proj_l[k] <- this level's row proj_u[k]
    int nproj;
    const int *proj_l, *proj_u;
    double *err, *rhs, *resu;   // [n]: correction (G.err[lev]), right-hand side, residual
};

#define MCL_INNER_JC 0
#define MCL_INNER_GS 1
#define MCL_INNER_CG 2
#define MCL_INNER_MG 3

// One row a thread (mcl_ops.h): doubles of the LDS window, and the slots of a
// velocity and of a temperature row that registers hold.
#define MCL_WINDOW 6144
#define MCL_ROW_V 18
#define MCL_ROW_T 9

struct UzawaParams {
    LevelDev L;
    GridSync gs;
    DevStats *stats;
    double *d, *p, *u1, *Ahv, *Ahp, *BAB;
    double *r0, *r1, *r2, *z0, *z1, *s1, *s2;
    double *cg_r, *cg_s, *cg_d, *cg_q, *cg_d2;
    double accuracy, citcom_accu;
    int max_citcom_cycle, max_cg_cycle, cg_precondition, check_v_only, schur;
    int exact_dots;          // dot products in the reference's sequential order
    int rows_fit;            // one row a thread, its vector through the LDS window (all workgroups)
    // inner solver (MCL_INNER_*): Jacobi runs on the whole grid; Gauss-Seidel
    // and multigrid need a launch of one workgroup
    int solver, mg_cycle, mg_finest_iteration, mg_coarse_iteration;
    // [n_v] each, the context's also where the work space is not: previous
    // iterates (Jacobi ping-pong, sweep and V-cycle differences); with conjugate
    // gradients xt is cg_d2, and the mixed solve keeps K v of its constrained
    // product in xt2
    double *xt, *xt2;
    const GsLevelDev *gsl;   // [ngsl] levels, coarsest first (device memory)
    int ngsl;
};

struct HeatParams {
    LevelDev L;
    GridSync gs;
    DevStats *stats;
    const double *V;
    double *T, *tau, *hK, *hC, *hA, *hF, *hd, *hdd, *d0, *B;
    double *cg_r, *cg_s, *cg_d, *cg_q, *cg_d2;
    double *model_time;
    double accuracy, theta, Q, Llast0, Llast1, diff_dt;
    int first_call, cg_precondition;
    int rows_fit;            // as UzawaParams
    int exact_dots;
};

// One multigrid level of the FP32 inner solver (mixed precision).  Level 0 is
// the coarsest; the finest level shares its rows with the Stokes velocity
// equations.  Levels with block != 0 are small enough to be processed by one
// workgroup (LDS-speed barriers); the others are processed by the whole grid.
// Rows (summed over levels) of the coarse multigrid levels that every
// workgroup of the mixed solve keeps in LDS (three float vectors per row).
#ifndef MCL_MG_LDS_ROWS
#define MCL_MG_LDS_ROWS 1536
#endif
// Matrix entries (ELL slots summed over levels) of those levels, also kept in
// LDS (FP32 values and 16-bit columns, 6 bytes an entry).
#ifndef MCL_MG_LDS_NNZ
#define MCL_MG_LDS_NNZ 16384
#endif

// 32-bit words of the LDS pool of the coarse levels: vectors, matrices, and
// 8 KB more for the transfer maps and the coarsest inverse; smaller levels leave
// room for all of them (a solve at 32x32 3.64 ms, 3.70 with the maps in memory;
// 256x256 29.8, 30.4; hanging nodes at 32x16 54.1, 55.7).
#define MCL_MG_POOL (4 * MCL_MG_LDS_ROWS + MCL_MG_LDS_NNZ * 3 / 2 + 2048)

struct MgLevelDev {
    int n, WK;
    int block;               // coarse level run per workgroup from LDS
    // places in the LDS pool (32-bit words) of an LDS level: its vectors x, t, b,
    // 1/diag, matrix values and columns; its transfer maps and (level 0) the
    // coarsest inverse, -1: read from memory
    int v_off, d_off, a_off, c_off, p_off, r_off, i_off;
    const unsigned *pro;     // [n][2] prolongation packed: c0 | c1 << 12 | m << 24, c2 | c3 << 12, 0xfff: none
    const unsigned *res;     // [rw][n] restriction packed: fine row | m << 16, weight 1 / m, 0: none
    // The FP32 matrix and every column map hold two slots of a row together
    // (WK2 = (WK + 1) / 2 pairs, [pair][row]; an odd row length is padded with
    // the row itself and 0): half the loads of one slot each, and their address
    // registers (28 spilled registers before, 7 so; a solve at 32x32 3.81 ms
    // before, 3.72).  Maps into lists of at most 65 535 rows pack a pair into
    // one word.
    int WK2;
    const unsigned *col16;   // [WK2][n] (LDS levels)
    const int *col;          // [WK2][n][2]
    float *val;              // [WK2][n][2]
    float *dinv;             // [n] 1 / diag(K)
    // prolongation from level-1: fine row u <- mean of pn[u] coarse rows pcol[k][u] (-1 = fixed)
    const int *pn;           // [n]
    const int *pcol;         // [4][n]
    // restriction to level-1 (= P^T), stored on this level's coarse partner:
    // coarse row c <- sum_k rval[k][c] * r_fine[rcol[k][c]]
    int rw;
    const int *rcol;         // [rw][n_coarse]
    const float *rval;       // [rw][n_coarse]
    float *x, *b, *r, *t;    // level vectors
    // fused V-cycle phases of a grid level, with per-workgroup row lists for
    // the workgroup count of the mixed solve (a workgroup owns rows O of
    // own_rows; W = [O | H1] adds the K columns of O, V = [W | H2] those of W;
    // F = the fine rows its coarse rows restrict from, T = [O | Th] adds the
    // K columns of F, U = [T | Uh] those of T):
    //  fuse_up:   x' = x + P x_c on W, then sweep pre + 1 on O from x' in LDS;
    //  fuse_down: the residual on F into LDS, then the coarse right-hand side;
    //  deep_up (pre = 2): x' on V, sweep 3 on W, sweep 4 on O;
    //  deep_down (pre = 2): sweep 2 on T from x_1 on U, the residual on F,
    //      the coarse right-hand side (above the LDS levels: T = W, U = V and
    //      the residual on O).
    int fuse_up, fuse_down, deep_up, deep_down;
    const int *hu_ptr, *hu_row;        // [nb + 1], H1
    const unsigned *kl;                // [WK2][n] K columns of O as local indices (into W, V)
    const int *h2_ptr, *h2_row;        // [nb + 1], H2
    const unsigned *hm;                // H1 rows' K columns -> V, block hu_ptr[g] WK2, pair-major
    const int *hd_ptr, *hd_row;        // [nb + 1], F
    const short *rl;                   // [rw][n] (coarse level) restriction columns as indices into F
    const int *th_ptr, *th_row;        // [nb + 1], Th
    const int *uh_ptr, *uh_row;        // [nb + 1], Uh
    const unsigned *mt;                // T rows' K columns -> U, block (g R + th_ptr[g]) WK2, pair-major
    const unsigned *mf;                // F rows' K columns -> T, block hd_ptr[g] WK2, pair-major
};

// Rows of a workgroup's halo lists kept in LDS (16-bit row numbers).
#ifndef MCL_LDS_LIST
#define MCL_LDS_LIST 4608
#endif
// floats of the LDS buffer of the fused V-cycle phases (per workgroup).  The
// phases repeat their halo's row products, so more is not better: with 6144 the
// two-sweep form reaches the finest level of 256x256 and the one-sweep forms
// that of 512x512 (32.3 and 71.6 ms a solve; 30.4 and 67.5 so).
#ifndef MCL_HALO_LDS
#define MCL_HALO_LDS 4096
#endif

// Multigrid levels the mixed solve can hold (every workgroup keeps a copy of
// their descriptors in LDS).
#define MCL_MG_MAX_LEVELS 14

struct MixedParams {
    UzawaParams U;
    const MgLevelDev *mg;    // [nmg] (device memory)
    const float *lam;        // [nmg] Gershgorin bounds of D^-1 K per level
    int nmg;
    const double *cinv;      // dense inverse of the coarsest K [nc][nc]
    int nc;
    double *rr;              // FP64 residual of the inner CG
    double inner_rtol;       // relative residual tolerance of each inner solve
    double relax, relax_max; // relax > 0: Uzawa-loop inner solves to min(relax_max, max(inner_rtol, relax / dv)),
                             // then one correction solve of d for the final p
    int max_inner;
    int probe;               // 1: stop after the first inner solve and report |G^T d|^2
    // point-to-point waits in the V-cycle: neighbour workgroups of each
    // workgroup (CSR over workgroups, at most MCL_BLOCK each); use_nbr = 0
    // makes every wait a grid barrier
    const int *nbr_ptr, *nbr_idx;
    int use_nbr;
    int pre;                 // Jacobi sweeps per level on each leg of the V-cycle (>= 1)
    float omega;             // damped-Jacobi weight of the smoother
    // augmented Lagrangian (al_state != null): U.L's K is K + g G W G^T with
    // W = diag(al_w) and g = *al_state (0 or al_gamma), and the solve returns
    // p + g W G^T d; it then sets *al_state for the next solve: al_gamma if
    // its Uzawa count reached al_keep (g > 0) or al_start (g = 0), else 0
    double *al_state;
    const double *al_w;      // [nel] 1 / BAB of the plain K
    double al_gamma;
    int al_keep, al_start;
    // warm-start history (null: none): ws[0] solves since the history was
    // reset, ws[1], ws[2] the model time of the last two; the solve appends
    // itself after its last phase (model_time: the device's model time)
    double *ws;
    const double *model_time;
};

extern "C" hipError_t mcl_upload_shape(const ShapeTables *s);

// A level's nodal fields in a launch over all levels (blk0: its first workgroup).
struct FieldLevel {
    int nno, blk0;
    const int *c2f;      // [nno] the finest level's node of each node (coarser levels)
    const double *X;
    double *T, *vis;
};
__global__ void k_viscosity(const FieldLevel *lv, int nlev, double A, double refT, double lm_jump);
__global__ void k_inject(const FieldLevel *lv, int nlev, const double *fine);
#define MCL_BUOY 256   // threads of k_buoy_rows
__global__ void k_buoy_rows(int gnox, int nno, const int *ptr, const int *ent_e, const signed char *ent_xi,
                            const signed char *ent_eta, const int *ienl, int nel, const double *T, double Ra,
                            double *avg);
__global__ void k_buoy_apply(int nno, int gnoz, const int *node, const double *T, double Ra, const double *avg,
                             double *buoy);
// One level of the all-levels assembly launch: its rows occupy the
// workgroups [blk0, blk0 + ceil(neq / MCL_BLOCK)) of the grid.
struct AsmLevel {
    LevelDev L;
    const double *vis, *buoy;
    int blk0;
};
#define MCL_ASM_BLOCK 256   // threads of k_assemble_K
__global__ void k_assemble_K(const AsmLevel *lv, int nlev);
// k_uzawa_fp64 for an inner solver (MCL_INNER_*)
const void *mcl_uzawa_fp64_kernel(int solver);
__global__ void k_v_to_nodes(LevelDev L, const double *d, double *V);
__global__ void k_stress_elem(LevelDev L, const double *vis, const double *V, double *es, double *area);
__global__ void k_stress_node(LevelDev L, const double *es, const double *area, double *stress);
__global__ void k_residuals(LevelDev L, RedBuf rb, const double *d, const double *p, int galerkin);
__global__ void k_collect3(RedBuf rb, int nblocks, double *out);
__global__ void k_heat_fp64(HeatParams H);
__global__ void k_uzawa_mixed(MixedParams P);
__global__ void k_uzawa_probe(MixedParams P);
// One multigrid level of the all-levels FP32 preparation launch: its rows
// occupy the workgroups [blk0, blk0 + ceil(n / MCL_BLOCK)).
struct PrepLevel {
    int n, W;
    const double *val, *diag;
    float *val32, *dinv;         // val32: [(W + 1) / 2][n][2]
    unsigned *bound;
    int blk0;
};
// the coarsest level's K and where its dense inverse goes
struct CoarseInv {
    int n, blk;          // rows; the workgroup that computes it
    const int *col, *ncol;
    const double *val;
    double *inv;
};
__global__ void k_prepare_fp32(const PrepLevel *lv, int nlev, CoarseInv ci);
// One multigrid level of the augmented-Lagrangian launches: K_al = K +
// gamma G W G^T (W = diag(w), w_e = 1 / sum_i G_ie^2 / K_ii, the BAB of the
// plain K), same ELL pattern, gamma read from the device.  Elements occupy workgroups [eblk0, ...) of
// k_al_weights, rows [rblk0, ...) of k_al_rows.
struct AlLevel {
    LevelDev L;
    double *val, *diag, *w;
    const double *gamma;     // device scalar (0: K_al = K)
    int eblk0, rblk0;
};
__global__ void k_al_weights(const AlLevel *lv, int nlev);
// warm start from the last two solutions (MixedParams::ws): d, p extrapolated
// linearly in model time from themselves and the previous solution h ([nv +
// np]: d then p) once `after` solves (at least 2) have followed a reset of
// the history, step ratio at most rmax; then h = d, p
__global__ void k_extrapolate(int nv, int np, double *d, double *p, double *h, const double *ws,
                              const double *model_time, int after, double rmax);
__global__ void k_al_rows(const AlLevel *lv, int nlev);
__global__ void k_zero_words(unsigned *p, long long n);
