// Device utilities shared by the gfx950 kernels of libmcl_hip.so:
//  * a grid-wide barrier for persistent (cooperatively launched) kernels,
//  * compensated FP64 reductions (double-double accumulation, exact products),
//  * the bilinear-quad shape tables (Shape_function.c:17-121 values).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#ifndef MCL_BLOCK
#define MCL_BLOCK 512   // threads per workgroup of every kernel (8 waves: one CU each)
#endif
#define MCL_WAVE 64
#define MCL_MAX_LEVELS 20
#define MCL_MAX_WG 2048
#define MCL_RED_SLOTS 3     // sums a launch hands to the next (RedBuf)
// most workgroups of a persistent kernel (they are all resident at once)
#define MCL_SYNC_WG 512
// A line of the synchronisation block: 128 bytes, written by one workgroup
// only.  Flags of several workgroups in one line make their stores wait for
// each other (256 workgroups, neighbour wait: 2.66 us with flags 4 bytes
// apart, 0.94 us a line apart).
#define MCL_LINE 32
#define MCL_RED_GROUPS 16
#define MCL_RED_SETS 3
// synchronisation words: gen at 0, abort at 32, arrive[MCL_SYNC_WG] lines from
// 64, then MCL_RED_SETS sets of MCL_SYNC_WG + MCL_RED_GROUPS reduction lines
#define MCL_SYNC_WORDS (64 + MCL_LINE * (MCL_SYNC_WG + MCL_RED_SETS * (MCL_SYNC_WG + MCL_RED_GROUPS)))
#define MCL_SPIN_LIMIT (1u << 24)

// Shape tables, uploaded once from the host (computed there with the
// reference's expressions so the values are identical bit for bit).
struct ShapeTables {
    double N[4][4];      // N[a][g] at Gauss point g
    double dxi[4][4];    // dN_a/dxi at g
    double deta[4][4];   // dN_a/deta at g
    double dxic[4], detac[4];
};

// Per-level element sizes (G.dx, G.dz) passed by value to kernels.
struct LevelSizes {
    double dx[MCL_MAX_LEVELS];
    double dz[MCL_MAX_LEVELS];
};

// ---------------------------------------------------------------- grid waits
// Waits between the phases of a persistent kernel.  No atomic
// read-modify-write: every workgroup stores into lines of its own and polls
// lines of others with relaxed agent-scope loads.  Data that crosses
// workgroups between two phases is stored and loaded with agent-scope atomics
// (coherent at the device level: a store writes through the XCD's L2, a load
// never returns a stale line); before a workgroup announces itself, each of
// its waves waits for all its memory operations (s_waitcnt 0), and a waiter
// issues its next loads only after it has seen the announcement, so no L2
// write-back or invalidate is needed and the L2 keeps the read-only matrices.
// Plain stores and loads of shared data need the fenced grid_sync.
//
// Every spin is bounded: past MCL_SPIN_LIMIT polls it sets *abort and the wait
// returns false; every spinner checks *abort every 1024 polls, and every
// caller then leaves its loops, so all waves reach the end of the kernel.
// After an abort the host zeroes the block.
struct GridSync {
    unsigned *gen;      // generation the next launch starts from
    unsigned *abort;
    unsigned *arrive;   // [MCL_SYNC_WG] lines, then the reduction lines
    unsigned nblocks;
};

// A workgroup's place in the sequence of waits (every thread keeps it; every
// workgroup passes the same sequence): the generation of the flags and the
// set of reduction lines the next grid-wide wait uses.
struct WaitState {
    unsigned gen;
    int set;
};

// set once a spin of this workgroup has given up
__device__ __forceinline__ unsigned &abort_flag()
{
    __shared__ unsigned f;
    return f;
}

// the bounded part of a spin; false: given up
__device__ __forceinline__ bool spin_more(unsigned &spins, unsigned *abort)
{
    __builtin_amdgcn_s_sleep(1);
    if (++spins > MCL_SPIN_LIMIT) {
        __hip_atomic_store(abort, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        abort_flag() = 1;
        return false;
    }
    if ((spins & 1023u) == 0 && __hip_atomic_load(abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
        abort_flag() = 1;
        return false;
    }
    return true;
}

__device__ __forceinline__ void spin_until(const unsigned *flag, unsigned target, unsigned *abort)
{
    unsigned spins = 0;
    while ((int)(__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) - target) < 0)
        if (!spin_more(spins, abort)) break;
}

// A reduction line holds up to 16 doubles; a word that has not been written
// since its line was cleared holds this signalling NaN, which no arithmetic
// produces (results are quiet NaNs).
#define MCL_EMPTY 0x7ff4dead7ff4deadull

__device__ __forceinline__ unsigned long long *red_line(const GridSync &gs, int set, int line)
{
    return (unsigned long long *)(gs.arrive + MCL_LINE * (MCL_SYNC_WG + set * (MCL_SYNC_WG + MCL_RED_GROUPS) + line));
}

// Clear the lines this workgroup writes in a set (16 lanes of one wave).
__device__ __forceinline__ void red_clear(const GridSync &gs, int set, int lane)
{
    if (lane < 16) {
        __hip_atomic_store(red_line(gs, set, blockIdx.x) + lane, MCL_EMPTY, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
        if (blockIdx.x < MCL_RED_GROUPS)
            __hip_atomic_store(red_line(gs, set, MCL_SYNC_WG + blockIdx.x) + lane, MCL_EMPTY, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
    }
}

// Every wait starts here: all memory operations of the workgroup are complete.
__device__ __forceinline__ void wg_complete()
{
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
}

// Start of a persistent kernel: clears the workgroup's reduction lines and
// waits for the whole grid, so that no workgroup sees a line of an earlier
// launch.  sync_end() leaves the generation for the next launch.
__device__ __forceinline__ bool sync_begin(const GridSync &gs, WaitState &w)
{
    w.gen = __hip_atomic_load(gs.gen, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT) + 1;
    w.set = 0;
    if (threadIdx.x == 0) abort_flag() = 0;
    if (threadIdx.x < 16)
        for (int s = 0; s < MCL_RED_SETS; s++) red_clear(gs, s, threadIdx.x);
    wg_complete();
    if (threadIdx.x == 0)
        __hip_atomic_store(gs.arrive + MCL_LINE * blockIdx.x, w.gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (unsigned b = threadIdx.x; b < gs.nblocks; b += blockDim.x) spin_until(gs.arrive + MCL_LINE * b, w.gen, gs.abort);
    __syncthreads();
    return abort_flag() == 0;
}

__device__ __forceinline__ void sync_end(const GridSync &gs, const WaitState &w)
{
    if (blockIdx.x == 0 && threadIdx.x == 0)
        __hip_atomic_store(gs.gen, w.gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Wait for the workgroups of a neighbour list (thread t polls its neighbour
// nbr, nbr < 0: none), between phases whose data flow is confined to
// neighbours and uses agent-scope accesses.
__device__ __forceinline__ bool nbr_sync(const GridSync &gs, WaitState &w, int nbr)
{
    w.gen++;
    wg_complete();
    if (threadIdx.x == 0)
        __hip_atomic_store(gs.arrive + MCL_LINE * blockIdx.x, w.gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (nbr >= 0) spin_until(gs.arrive + MCL_LINE * nbr, w.gen, gs.abort);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __syncthreads();
    return abort_flag() == 0;
}

// ------------------------------------------------------- compensated reduction
// A double-double value (hi + lo).  Sums use TwoSum, products TwoProduct via
// fma, so a dot product is accumulated as if in ~106-bit precision and rounded
// once at the end (Ogita, Rump, Oishi 2005, "Accurate sum and dot product").
struct dd {
    double hi, lo;
};

__device__ __forceinline__ dd dd_zero() { return dd{0.0, 0.0}; }

__device__ __forceinline__ dd two_sum(double a, double b)
{
    double s = a + b;
    double bb = s - a;
    double e = (a - (s - bb)) + (b - bb);
    return dd{s, e};
}

__device__ __forceinline__ dd dd_add(dd a, dd b)
{
    dd s = two_sum(a.hi, b.hi);
    double lo = s.lo + (a.lo + b.lo);
    double hi = s.hi + lo;
    return dd{hi, lo - (hi - s.hi)};
}

__device__ __forceinline__ dd dd_add_prod(dd acc, double x, double y)
{
    double p = x * y;
    double pe = __builtin_fma(x, y, -p);
    dd s = two_sum(acc.hi, p);
    double lo = s.lo + (acc.lo + pe);
    double hi = s.hi + lo;
    return dd{hi, lo - (hi - s.hi)};
}

// a + b without the final renormalisation: the parts' sum and the running sum
// of the errors (Sum2 of the paper above: as accurate as if summed in twice
// the precision and rounded once, without dd_add's serial chain from one
// level of a tree to the next)
__device__ __forceinline__ dd dd_add2(dd a, dd b)
{
    const dd s = two_sum(a.hi, b.hi);
    return dd{s.hi, s.lo + (a.lo + b.lo)};
}

// Sums and maxima over the lanes of a wave by DPP moves, 16 lanes (the rows,
// result in each row's lane 15), 8 lanes (lane 7) or 64 lanes (lane 63).
// Lanes without a source lane add 0 (maxima: of values >= 0).
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_move(double x)
{
    const long long v = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(v >> 32), CTRL, ROWS, 0xf, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ void dpp_step(dd &v)
{
    v = dd_add2(v, dd{dpp_move<CTRL, ROWS>(v.hi), dpp_move<CTRL, ROWS>(v.lo)});
}

template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ void dpp_step(double &v)
{
    v = fmax(v, dpp_move<CTRL, ROWS>(v));
}

template <int LANES, typename T>
__device__ __forceinline__ void lane_reduce(T &v)
{
    dpp_step<0x111>(v);   // row_shr:1
    dpp_step<0x112>(v);   // row_shr:2
    dpp_step<0x114>(v);   // row_shr:4
    if (LANES > 8) dpp_step<0x118>(v);        // row_shr:8
    if (LANES > 16) {
        dpp_step<0x142, 0xa>(v);              // row_bcast:15 into rows 1 and 3
        dpp_step<0x143, 0xc>(v);              // row_bcast:31 into rows 2 and 3
    }
}

__device__ __forceinline__ dd dd_shfl_xor(dd v, int mask)
{
    return dd{__shfl_xor(v.hi, mask, MCL_WAVE), __shfl_xor(v.lo, mask, MCL_WAVE)};
}

__device__ __forceinline__ double dmax_shfl(double v)
{
    for (int m = MCL_WAVE / 2; m > 0; m >>= 1) v = fmax(v, __shfl_xor(v, m, MCL_WAVE));
    return v;
}

// Rows of a kernel's reduction scratch (__shared__ dd lds[MCL_RED_ROWS]
// [MCL_BLOCK / MCL_WAVE]): a reduction of NR values uses rows 0 .. NR - 1.
#define MCL_RED_ROWS 8

// Block reduction of NR double-double values (fixed order, deterministic).
template <int NR>
__device__ __forceinline__ void block_reduce_dd(dd (&v)[NR], dd (*lds)[MCL_BLOCK / MCL_WAVE])
{
    static_assert(NR <= MCL_RED_ROWS, "the reduction scratch has MCL_RED_ROWS rows");
    const int lane = threadIdx.x & (MCL_WAVE - 1), wave = threadIdx.x / MCL_WAVE;
#pragma unroll
    for (int r = 0; r < NR; r++)
        for (int m = MCL_WAVE / 2; m > 0; m >>= 1) v[r] = dd_add(v[r], dd_shfl_xor(v[r], m));
    __syncthreads();
    if (lane == 0)
#pragma unroll
        for (int r = 0; r < NR; r++) lds[r][wave] = v[r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < NR; r++) {
        dd t = lds[r][0];
        for (int w = 1; w < MCL_BLOCK / MCL_WAVE; w++) t = dd_add(t, lds[r][w]);
        v[r] = t;
    }
}

// Grid-wide wait that carries a reduction: NS sums (double-double partials)
// and NM maxima of values >= 0 over all threads of the grid; every workgroup
// gets the same values, reduced in the same order.  Each workgroup reduces its
// own values while its stores are in flight, then publishes them in its line:
// the line's words are the announcement, so arrival and data cross the fabric
// together.  Up to 64 workgroups every workgroup reads all lines; above that
// the workgroups of a group (those with equal number modulo 16) are summed by
// the group's first one, and every workgroup reads the 16 groups' lines.
// The three sets of lines rotate: the set after next is cleared once a wait is
// over (all workgroups have then left the wait that used it last), and is
// complete before this workgroup announces itself again.
// Measured (one sum, 512 threads a workgroup, us a wait) against partials,
// a barrier with a master workgroup and a second pass over the partials:
// 4 workgroups 1.6 / 4.0, 64: 2.4 / 4.7, 129: 2.9 / 4.9, 256: 3.0 / 5.0; one
// level of lines at 256: 4.2.
template <int NS, int NM>
__device__ __forceinline__ bool grid_reduce(const GridSync &gs, WaitState &w, dd (&v)[NS ? NS : 1],
                                            double (&mx)[NM ? NM : 1], double (&out)[NS + NM ? NS + NM : 1])
{
    constexpr int NW = NS || NM ? 2 * NS + NM : 1, WAVES = MCL_BLOCK / MCL_WAVE;
    static_assert(NW <= 16 && WAVES == 8, "a line holds 16 words; eight waves");
    __shared__ double part[NW][WAVES], res[NS + NM ? NS + NM : 1];
    const int lane = threadIdx.x & (MCL_WAVE - 1), wave = threadIdx.x / MCL_WAVE, nb = (int)gs.nblocks;
    const int set = w.set;
    w.set = set == MCL_RED_SETS - 1 ? 0 : set + 1;
#pragma unroll
    for (int r = 0; r < NS; r++) lane_reduce<64>(v[r]);
#pragma unroll
    for (int r = 0; r < NM; r++) lane_reduce<64>(mx[r]);
    if (lane == MCL_WAVE - 1) {
#pragma unroll
        for (int r = 0; r < NS; r++) {
            part[2 * r][wave] = v[r].hi;
            part[2 * r + 1][wave] = v[r].lo;
        }
#pragma unroll
        for (int r = 0; r < NM; r++) part[2 * NS + r][wave] = mx[r];
    }
    wg_complete();
    if (wave == 0) {
        // one line's words: published by lane r, read by the lane of the line
        double word[NW];
        auto publish = [&](int line, int from) {
            double mine = 0.0;
#pragma unroll
            for (int q = 0; q < NW; q++) {
                const double x = __shfl(word[q], from, MCL_WAVE);
                if (lane == q) mine = x;
            }
            if (lane < NW)
                __hip_atomic_store(red_line(gs, set, line) + lane, (unsigned long long)__double_as_longlong(mine),
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        };
        auto fold = [&](int lanes) {
#pragma unroll
            for (int r = 0; r < NS; r++) {
                dd t{word[2 * r], word[2 * r + 1]};
                if (lanes <= 8) lane_reduce<8>(t);
                else if (lanes <= 16) lane_reduce<16>(t);
                else lane_reduce<64>(t);
                word[2 * r] = t.hi;
                word[2 * r + 1] = t.lo;
            }
#pragma unroll
            for (int r = 0; r < NM; r++) {
                if (lanes <= 8) lane_reduce<8>(word[2 * NS + r]);
                else if (lanes <= 16) lane_reduce<16>(word[2 * NS + r]);
                else lane_reduce<64>(word[2 * NS + r]);
            }
        };
        auto collect = [&](int n, int line0, int stride) {
            if (lane < n) {
                const unsigned long long *p = red_line(gs, set, line0 + lane * stride);
                unsigned spins = 0;
                bool more = true;
                while (more) {
                    more = false;
#pragma unroll
                    for (int q = 0; q < NW; q++) {
                        const unsigned long long x =
                            __hip_atomic_load(p + q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        more = more || x == MCL_EMPTY;
                        word[q] = __longlong_as_double((long long)x);
                    }
                    if (more && !spin_more(spins, gs.abort)) break;
                }
            } else {
#pragma unroll
                for (int q = 0; q < NW; q++) word[q] = 0.0;
            }
        };
#pragma unroll
        for (int q = 0; q < NW; q++) word[q] = (NS || NM) && lane < WAVES ? part[q][lane] : 0.0;
        fold(8);
        int last = 7;
        if (nb > 1) publish(blockIdx.x, 7);
        if (nb == 1) {
            // nothing leaves the workgroup
        } else if (nb <= MCL_WAVE) {
            collect(nb, 0, 1);
            fold(nb);
            last = nb <= 8 ? 7 : nb <= 16 ? 15 : 63;
        } else {
            if (blockIdx.x < MCL_RED_GROUPS) {
                const int n = (nb - 1 - (int)blockIdx.x) / MCL_RED_GROUPS + 1;
                collect(n, blockIdx.x, MCL_RED_GROUPS);
                fold(n);
                publish(MCL_SYNC_WG + blockIdx.x, n <= 8 ? 7 : n <= 16 ? 15 : 63);
            }
            collect(MCL_RED_GROUPS, MCL_SYNC_WG, 1);
            fold(MCL_RED_GROUPS);
            last = 15;
        }
        if (lane == last) {
#pragma unroll
            for (int r = 0; r < NS; r++) res[r] = word[2 * r] + word[2 * r + 1];
#pragma unroll
            for (int r = 0; r < NM; r++) res[NS + r] = word[2 * NS + r];
        }
    }
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __syncthreads();
    if (wave == WAVES - 1) red_clear(gs, w.set == MCL_RED_SETS - 1 ? 0 : w.set + 1, lane);
#pragma unroll
    for (int r = 0; r < NS + NM; r++) out[r] = res[r];
    return abort_flag() == 0;
}

// sums only
template <int NS>
__device__ __forceinline__ bool grid_sum(const GridSync &gs, WaitState &w, dd (&v)[NS], double (&out)[NS])
{
    double none[1] = {0.0};
    return grid_reduce<NS, 0>(gs, w, v, none, out);
}

// a grid-wide wait alone
__device__ __forceinline__ bool grid_wait(const GridSync &gs, WaitState &w)
{
    dd v[1] = {dd_zero()};
    double none[1] = {0.0}, out[1];
    return grid_reduce<0, 0>(gs, w, v, none, out);
}

// Grid-wide wait for data written and read with plain accesses: an agent-scope
// release before (thread 0 writes back the L2 after all waves' stores), an
// acquire after (thread 0 invalidates the caches of its CU and XCD; every
// thread doing so costs 18 us at 256 workgroups).
__device__ __forceinline__ bool grid_sync(const GridSync &gs, WaitState &w)
{
    wg_complete();
    if (threadIdx.x == 0) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    const bool ok = grid_wait(gs, w);
    if (threadIdx.x == 0) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    __syncthreads();
    return ok;
}

// Partial sums between two launches: every workgroup of the first writes its
// partials, one workgroup of the second reduces them in a fixed order.
struct RedBuf {
    dd *part;      // [MCL_RED_SLOTS][MCL_MAX_WG]
};

template <int NR>
__device__ __forceinline__ void reduce_publish(const RedBuf &rb, dd (&v)[NR], dd (*lds)[MCL_BLOCK / MCL_WAVE])
{
    static_assert(NR <= MCL_RED_SLOTS, "the partials have MCL_RED_SLOTS slots");
    block_reduce_dd<NR>(v, lds);
    if (threadIdx.x == 0)
#pragma unroll
        for (int r = 0; r < NR; r++) {
            dd *p = rb.part + r * MCL_MAX_WG + blockIdx.x;
            __hip_atomic_store(&p->hi, v[r].hi, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&p->lo, v[r].lo, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
}

template <int NR>
__device__ __forceinline__ void reduce_collect(const RedBuf &rb, int nblocks, double (&out)[NR],
                                               dd (*lds)[MCL_BLOCK / MCL_WAVE])
{
    dd v[NR];
#pragma unroll
    for (int r = 0; r < NR; r++) v[r] = dd_zero();
    for (int b = threadIdx.x; b < nblocks; b += MCL_BLOCK)
#pragma unroll
        for (int r = 0; r < NR; r++) {
            const dd *p = rb.part + r * MCL_MAX_WG + b;
            const dd t{__hip_atomic_load(&p->hi, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT),
                       __hip_atomic_load(&p->lo, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)};
            v[r] = dd_add(v[r], t);
        }
    block_reduce_dd<NR>(v, lds);
#pragma unroll
    for (int r = 0; r < NR; r++) out[r] = v[r].hi + v[r].lo;
}

__device__ __forceinline__ double block_max(double v, double *lds)
{
    const int lane = threadIdx.x & (MCL_WAVE - 1), wave = threadIdx.x / MCL_WAVE;
    v = dmax_shfl(v);
    __syncthreads();
    if (lane == 0) lds[wave] = v;
    __syncthreads();
    double t = lds[0];
    for (int w = 1; w < MCL_BLOCK / MCL_WAVE; w++) t = fmax(t, lds[w]);
    return t;
}
