// Persistent batched solver: many small systems of uneven size in one launch.
//
// Small systems (a few thousand to a few tens of thousands of rows) are
// bound by launch and synchronisation latency on the stream path: every
// BiCGSTAB pass is ~16 kernels of a few microseconds of work each.  Here one
// workgroup of PBS threads runs a whole solve -- the reference loop
// (AFIIM/src/bicgstab.cpp:149-281, same constants, exit order and info
// codes; ACIFIM's non-finite alpha guard, ACIFIM/src/bicgstab.cpp:208-213) --
// with workgroup barriers in place of kernel boundaries, and a persistent
// grid pulls (system, right-hand side) items from a device work queue (one
// atomic counter) until it is empty.  Items are queued largest system first
// so the longest solves start early.  Every workgroup leaves the loop when
// the counter passes the item count, and every solve ends by NMAX, so the
// grid always drains.
//
// Systems of at most BT_ROWS rows and bt_mean entries per row run in
// k_batch_small, which keeps the vectors in LDS and registers and streams the
// matrices through LDS; the rest of this comment is k_batch_solve, for the
// others.
// Per workgroup: SpMV rows go to groups of LPR lanes (xor-shuffle sums inside
// the group); vector updates stride over the rows; dot products and norms
// are summed in a fixed order (per-thread, wave shuffles, then the waves in
// index order), so a result does not depend on which workgroup ran it or
// what else was in the batch.  The nine work vectors of a solve live in a
// per-workgroup slice of an arena; a system's matrices are read from its
// resident FP64 copies.
//
// restart_true = 1 adds a true-residual check: when the loop converges on
// the recursive residual, r = b - A x is recomputed and, if it is not below
// tol * ||r_0||, BiCGSTAB restarts from the current x (at most MAX_CYCLES
// cycles, NMAX passes in total).  restart_true = 0 is the reference loop
// unchanged.
#pragma once
#include "cm_resident.hpp"

namespace cm {

constexpr int PBS = 1024;       // threads per persistent workgroup
constexpr int LPR = 8;          // lanes per SpMV row
constexpr int MAX_CYCLES = 4;   // BiCGSTAB cycles with the true-residual check

struct BatchSys {
    int n, variant, maxmsteps, pad;
    // row pointers, columns and values of H (G^T on the symmetric PDFIIM
    // branch), G and A
    const int *p[3], *c[3];
    const double *v[3];
    const double *idv;
};

struct BatchItem {
    int sys, nmax;
    double tol;
    const double *b;  // device, n values
    double *x;        // device, n values: x0 in, solution out
    double resval;    // out
    int iter, info;   // out
    int cycles, pad;  // out: BiCGSTAB cycles run
};

// Sum of K values over the workgroup, returned to every thread.  Fixed
// order: wave shuffles, then the PBS/WAVE wave sums in wave order.
template <int K>
__device__ __forceinline__ void wg_allsum(double (&v)[K], double *lds /* K * PBS / WAVE */)
{
    const int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE;
#pragma unroll
    for (int k = 0; k < K; k++) v[k] = wave_sum(v[k]);
    __syncthreads();
    if (lane == 0)
#pragma unroll
        for (int k = 0; k < K; k++) lds[w * K + k] = v[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; k++) {
        double s = 0.0;
        for (int q = 0; q < PBS / WAVE; q++) s += lds[q * K + k];
        v[k] = s;
    }
    __syncthreads();  // lds is reused by the next reduction
}

// y = M x over the workgroup; f(row, sum) is called once per row by the
// row group's first lane.
template <class F>
__device__ __forceinline__ void wg_spmv(int n, const int *__restrict__ ptr, const int *__restrict__ col,
                                        const double *__restrict__ val, const double *__restrict__ x, F f)
{
    const int lane = threadIdx.x & (LPR - 1), g = threadIdx.x / LPR;
    for (int r = g; r < n; r += PBS / LPR) {
        double s = 0.0;
        const int e = ptr[r + 1];
        for (int k = ptr[r] + lane; k < e; k += LPR) s += val[k] * x[col[k]];
#pragma unroll
        for (int off = LPR / 2; off > 0; off >>= 1) s += __shfl_xor(s, off, WAVE);
        if (lane == 0) f(r, s);
    }
}

// out = G (D^-1 (H in)); tm is scratch.
__device__ __forceinline__ void wg_apply(const BatchSys &S, const double *in, double *tm, double *out)
{
    const double *idv = S.idv;
    wg_spmv(S.n, S.p[0], S.c[0], S.v[0], in, [&](int r, double s) { tm[r] = idv[r] * s; });
    __syncthreads();
    wg_spmv(S.n, S.p[1], S.c[1], S.v[1], tm, [&](int r, double s) { out[r] = s; });
    __syncthreads();
}

__device__ void wg_bicgstab(const BatchSys &S, BatchItem &it, double *w, double *lds, int restart_true)
{
    const int n = S.n;
    double *r0 = w, *r = w + n, *p = w + 2 * (size_t)n, *v = w + 3 * (size_t)n, *s = w + 4 * (size_t)n,
           *t = w + 5 * (size_t)n, *pc = w + 6 * (size_t)n, *sc = w + 7 * (size_t)n, *tm = w + 8 * (size_t)n;
    const double *b = it.b;
    double *x = it.x;
    const double eps = 1.11022302462516e-16;  // AFIIM/src/bicgstab.cpp:108
    int iter = 0, info = 3, cycles = 0;
    double ro0 = 0.0, resval = 0.0;
    const int ncyc = restart_true ? MAX_CYCLES : 1;
    for (int cyc = 0; cyc < ncyc; cyc++) {
        // r = b - A x; r0 = p = r; ro = ||r||   (AFIIM/src/bicgstab.cpp:149-165)
        double a1[1] = {0.0};
        wg_spmv(n, S.p[2], S.c[2], S.v[2], x, [&](int i, double q) {
            const double ri = b[i] + (-1.0) * q;
            r[i] = ri;
            r0[i] = ri;
            p[i] = ri;
            a1[0] += ri * ri;
        });
        wg_allsum<1>(a1, lds);
        const double ro = sqrt(a1[0]);
        cycles = cyc + 1;
        if (cyc == 0) {
            ro0 = ro;
            if (it.nmax <= 0) {  // NMAX < 0: the reference leaves info as the caller set it (-1 here)
                resval = ro / ro0;
                iter = 0;
                info = it.nmax == 0 ? 3 : -1;
                break;
            }
        } else if (ro < it.tol * ro0) {  // true residual below tol: done
            resval = ro / ro0;
            info = 0;
            break;
        }
        const double target = it.tol * ro0;
        double m1 = ro * ro, m2 = 0.0, rc = ro, prc = 0.0, alpha = 0.0, omega = 0.0, beta = 0.0;
        int stag = 0, msteps = 0;
        info = 3;
        bool conv = false;
        while (iter < it.nmax) {
            wg_apply(S, p, tm, pc);
            double a[1] = {0.0};
            wg_spmv(n, S.p[2], S.c[2], S.v[2], pc, [&](int i, double q) {
                v[i] = q;
                a[0] += r0[i] * q;
            });
            wg_allsum<1>(a, lds);
            alpha = m1 / a[0];
            if (S.variant == 2 && !isfinite(alpha)) {  // ACIFIM/src/bicgstab.cpp:208-213
                iter = it.nmax;
                info = 3;
                break;
            }
            for (int i = threadIdx.x; i < n; i += PBS) s[i] = r[i] + (-alpha) * v[i];
            __syncthreads();
            wg_apply(S, s, tm, sc);
            double o[2] = {0.0, 0.0};
            wg_spmv(n, S.p[2], S.c[2], S.v[2], sc, [&](int i, double q) {
                t[i] = q;
                o[0] += q * s[i];
                o[1] += q * q;
            });
            wg_allsum<2>(o, lds);
            omega = o[0] / o[1];
            double u[4] = {0.0, 0.0, 0.0, 0.0};
            for (int i = threadIdx.x; i < n; i += PBS) {
                const double pci = pc[i], xi = x[i], ri = r[i];
                u[0] += pci * pci;
                u[1] += xi * xi;
                u[2] += ri * ri;
                double xn = xi + alpha * pci;
                xn = xn + omega * sc[i];
                x[i] = xn;
                const double rn = s[i] + (-omega) * t[i];
                r[i] = rn;
                u[3] += r0[i] * rn;
            }
            wg_allsum<4>(u, lds);
            if (fabs(alpha) * sqrt(u[0]) < eps * sqrt(u[1])) stag++;
            else stag = 0;
            prc = rc;
            rc = sqrt(u[2]);
            if (prc < rc) msteps++;
            else msteps = 0;
            if (msteps >= S.maxmsteps) {
                info = 1;
                break;
            }
            if (stag >= 3) {
                info = 2;
                break;
            }
            if (rc < target) {
                info = 0;
                conv = true;
                break;
            }
            m2 = m1;
            m1 = u[3];
            beta = m1 * alpha / (omega * m2);
            const double c = -beta * omega;
            for (int i = threadIdx.x; i < n; i += PBS) {
                const double q = c * v[i] + beta * p[i];
                p[i] = q + r[i];
            }
            __syncthreads();
            iter++;
        }
        __syncthreads();
        resval = rc / ro0;
        if (!conv) break;  // divergence, stagnation, NMAX: as the reference reports it
    }
    if (threadIdx.x == 0) {
        it.resval = resval;
        it.iter = iter;
        it.info = info;
        it.cycles = cycles;
    }
}

// ---- systems of at most BT_ROWS rows (and bt_mean entries per row): vectors in
// LDS and registers
//
// A pass is bound by reading the matrices (12 bytes per entry): one CU holds
// some 60 reads in flight, which from the L2 and the MALL gives it about 20
// bytes per ns.  So each product streams its entries in tiles of BT_PER per
// thread, coalesced, every tile loaded while the tile before is summed (the
// next product's first tile while this one ends); the vectors that are
// gathered (p or s, H p, M p) sit in LDS, and each thread keeps its rows' x,
// r (then s), p, v and M p (then M s) in registers.  The products are staged
// in LDS and added by each row's thread in column order.  192 solves of 48
// systems of 300 to 3400 rows: 5260 us with 8 lanes per row gathering every
// entry's x from memory, 1890 us so (36 MB read for the longest solve, by one
// CU; 1024 threads, whose 128 registers spill, 2450 us).
constexpr int BT_BS = 512;    // threads: 8 waves, which leaves a thread 256 registers (1024 threads spilled)
constexpr int BT_PER = 16;
constexpr int BT_TILE = BT_PER * BT_BS;
constexpr int BT_ROWS = 4096;  // two vectors of them and a tile take 132 of the LDS's 160 KB
// entries per row of a matrix, on the mean, up to which this kernel is the faster one
constexpr int bt_mean(int n) { return n <= 2 * BT_BS ? 80 : 170; }

using BatchSysTable = RsConst<BatchSys>;  // the tables are written before the launch

// Entries [c0, c0 + BT_TILE) of matrix mi (0 H, 1 G, 2 A).
__device__ __forceinline__ void bt_load(BatchSysTable S, int mi, int c0, int (&j)[BT_PER], double (&ev)[BT_PER])
{
    const int *col = rs_glob(S->c[mi]);
    const double *val = rs_glob(S->v[mi]);
    const int k1 = rs_uni(rs_glob(S->p[mi])[S->n]);
    // the addresses are formed at each use: kept over the solve, they would
    // take the registers of the rows' vectors
    int tid = (int)threadIdx.x;
    asm volatile("" : "+v"(tid));
#pragma unroll
    for (int q = 0; q < BT_PER; q++) {
        const int k = c0 + q * BT_BS + tid;
        j[q] = -1;
        ev[q] = 0.0;
        if (k < k1) {
            j[q] = *rs_at(col, (unsigned)k);
            ev[q] = *rs_at(val, (unsigned)k);
        }
    }
}

// y = M src for the workgroup's rows q * BT_BS + thread, M matrix mi; src at
// lds[so].  (j, ev) hold M's first tile on entry and the next matrix's (A's
// successor is H) on return.
template <int R>
__device__ __forceinline__ void bt_rows(BatchSysTable S, int mi, double *lds, int so, int (&j)[BT_PER],
                                        double (&ev)[BT_PER], double (&y)[R])
{
#pragma clang fp contract(off)
    int tid = (int)threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int n = S->n;
    const int *ptr = rs_glob(S->p[mi]);
    const int nnz = rs_uni(ptr[n]);
    int a[R], e[R], first[R + 1];  // first: entries ahead of each row step, the same on every thread
#pragma unroll
    for (int q = 0; q <= R; q++) first[q] = rs_uni(ptr[min(q * BT_BS, n)]);
#pragma unroll
    for (int q = 0; q < R; q++) {
        const int i = q * BT_BS + tid;
        a[q] = *rs_at(ptr, (unsigned)min(i, n));
        e[q] = *rs_at(ptr, (unsigned)min(i + 1, n));
        y[q] = 0.0;
    }
#pragma unroll 1
    for (int c0 = 0;; c0 += BT_TILE) {  // uniform over the workgroup
#pragma unroll
        for (int q = 0; q < BT_PER; q++)
            if (j[q] >= 0) lds[q * BT_BS + tid] = ev[q] * lds[so + j[q]];
        const int c1 = c0 + BT_TILE;
        const bool last = c1 >= nnz;
        bt_load(S, last ? (mi == 2 ? 0 : mi + 1) : mi, last ? 0 : c1, j, ev);
        __syncthreads();
#pragma unroll
        for (int q = 0; q < R; q++)
            if (first[q] < c1 && first[q + 1] > c0) {
                const int k1 = min(e[q], c1);
                int k = max(a[q], c0);
                for (; k + 4 <= k1; k += 4) {
                    double t[4];
#pragma unroll
                    for (int u = 0; u < 4; u++) t[u] = lds[k - c0 + u];
#pragma unroll
                    for (int u = 0; u < 4; u++) y[q] += t[u];
                }
                for (; k < k1; k++) y[q] += lds[k - c0];
            }
        __syncthreads();  // the products are overwritten by the next tile, src by the next product
        if (last) break;
    }
}

// Sums of K values over the workgroup, the same on every thread, in a fixed
// order; red: K * BT_BS / WAVE doubles not used by the call before.
template <int K>
__device__ __forceinline__ void bt_allsum(double (&v)[K], double *red)
{
    constexpr int NW = BT_BS / WAVE;
    static_assert(NW == 8, "8 lanes per sum");
    const int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE;
#pragma unroll
    for (int k = 0; k < K; k++) v[k] = rs_wave_sum(v[k]);
    if (lane == 0)
#pragma unroll
        for (int k = 0; k < K; k++) red[k * NW + w] = v[k];
    __syncthreads();
    const double t = rs_group_sum<8>(lane < K * NW ? red[lane] : 0.0);
#pragma unroll
    for (int k = 0; k < K; k++) v[k] = rs_lane(t, k * NW);
}

// wg_bicgstab for n <= R * BT_BS rows.  w: n doubles of the arena (r0).
// lds: the tile's products, two vectors of R * BT_BS, and 3 x 32 doubles of sums.
// One loop iteration is one product with what follows it, so the product's
// code exists once: steps 0-2 are H, G, A on p, 3-5 on s, 6 the residual of x.
template <int R>
__device__ __forceinline__ void bt_bicgstab(BatchSysTable S, RsConst<BatchItem> in, BatchItem &it, double *w,
                                            double *lds, int restart_true)
{
    constexpr int VA = BT_TILE, VB = VA + R * BT_BS;  // the gathered vectors
    const int n = S->n;
    int tid = (int)threadIdx.x;
    double *red = lds + VB + R * BT_BS;  // three sets: a set comes again two reductions later
    double *r0 = w;
    const double eps = 1.11022302462516e-16;  // AFIIM/src/bicgstab.cpp:108
    double x[R], r[R], p[R], v[R], pc[R], y[R];
    int j[BT_PER];
    double ev[BT_PER];
    auto put = [&](int at, const double(&u)[R]) {
#pragma unroll
        for (int q = 0; q < R; q++) lds[at + q * BT_BS + tid] = u[q];  // the rows past n are 0
    };
    const double *b = rs_glob(in->b), *idv = rs_glob(S->idv);
    double *xg = rs_glob(in->x);
    const double tol = in->tol;
    const int nmax = in->nmax, variant = S->variant, maxmsteps = S->maxmsteps;
#pragma unroll
    for (int q = 0; q < R; q++) {
        const int i = q * BT_BS + tid;
        x[q] = i < n ? xg[i] : 0.0;
        r[q] = p[q] = v[q] = pc[q] = 0.0;
    }
    int iter = 0, info = 3, cycles = 0, stag = 0, msteps = 0, step = 6;
    double ro0 = 0.0, resval = 0.0, target = 0.0, m1 = 0.0, rc = 0.0, alpha = 0.0, pcn = 0.0, xn = 0.0, rn = 0.0;
    put(VA, x);
    bt_load(S, 2, 0, j, ev);
    __syncthreads();
#pragma unroll 1
    for (;;) {
        const int mi = step == 6 ? 2 : step % 3;
        asm volatile("" : "+v"(tid));
        bt_rows<R>(S, mi, lds, mi == 1 ? VB : VA, j, ev, y);
        if (mi == 0) {
#pragma unroll
            for (int q = 0; q < R; q++) {
                const int i = q * BT_BS + tid;
                lds[VB + i] = i < n ? idv[i] * y[q] : 0.0;
            }
        } else if (mi == 1) {
#pragma unroll
            for (int q = 0; q < R; q++) pc[q] = y[q];
            put(VA, pc);
        }
        if (mi != 2) {
            step++;
            __syncthreads();
            continue;
        }
        double sm[4] = {0.0, 0.0, 0.0, 0.0};
        if (step == 2) {
#pragma unroll
            for (int q = 0; q < R; q++) {
                const int i = q * BT_BS + tid;
                v[q] = y[q];
                sm[0] += i < n ? r0[i] * v[q] : 0.0;
                sm[1] += pc[q] * pc[q];
                sm[2] += x[q] * x[q];
                sm[3] += r[q] * r[q];
            }
        } else if (step == 5) {
#pragma unroll
            for (int q = 0; q < R; q++) {
                sm[0] += y[q] * r[q];
                sm[1] += y[q] * y[q];
            }
        } else {
            // r = b - A x; r0 = p = r; ro = ||r||   (AFIIM/src/bicgstab.cpp:149-165)
#pragma unroll
            for (int q = 0; q < R; q++) {
                const int i = q * BT_BS + tid;
                r[q] = 0.0;
                if (i < n) {
                    r[q] = b[i] + (-1.0) * y[q];
                    r0[i] = r[q];
                }
                p[q] = r[q];
                sm[0] += r[q] * r[q];
            }
        }
        bt_allsum<4>(sm, red + (step == 2 ? 32 : step == 5 ? 64 : 0));
        if (step == 2) {
            alpha = m1 / sm[0];
            if (variant == 2 && !isfinite(alpha)) {  // ACIFIM/src/bicgstab.cpp:208-213
                iter = nmax;
                info = 3;
                resval = rc / ro0;
                break;
            }
            pcn = sqrt(sm[1]);
            xn = sqrt(sm[2]);
            rn = sqrt(sm[3]);
#pragma unroll
            for (int q = 0; q < R; q++) {
                x[q] = x[q] + alpha * pc[q];
                r[q] = r[q] + (-alpha) * v[q];  // s
            }
            put(VA, r);
            step = 3;
            __syncthreads();
            continue;
        }
        if (step == 6) {
            const double ro = sqrt(sm[0]);
            cycles++;
            if (cycles == 1) {
                ro0 = ro;
                if (nmax <= 0) {  // NMAX < 0: the reference leaves info as the caller set it (-1 here)
                    resval = ro / ro0;
                    info = nmax == 0 ? 3 : -1;
                    break;
                }
            } else if (ro < tol * ro0) {  // true residual below tol: done
                resval = ro / ro0;
                info = 0;
                break;
            }
            target = tol * ro0;
            m1 = ro * ro;
            rc = ro;
            stag = msteps = 0;
            info = 3;
            if (iter >= nmax) {  // a cycle with no passes left
                resval = rc / ro0;
                break;
            }
        } else {
            const double omega = sm[0] / sm[1];
            double u[1] = {0.0};
#pragma unroll
            for (int q = 0; q < R; q++) {
                const int i = q * BT_BS + tid;
                x[q] = x[q] + omega * pc[q];
                r[q] = r[q] + (-omega) * y[q];
                u[0] += i < n ? r0[i] * r[q] : 0.0;
            }
            bt_allsum<1>(u, red);
            if (fabs(alpha) * pcn < eps * xn) stag++;
            else stag = 0;
            const double prc = rc;
            rc = rn;
            if (prc < rc) msteps++;
            else msteps = 0;
            resval = rc / ro0;
            if (msteps >= maxmsteps) {
                info = 1;
                break;
            }
            if (stag >= 3) {
                info = 2;
                break;
            }
            if (rc < target) {
                info = 0;
                if (cycles >= (restart_true ? MAX_CYCLES : 1)) break;
                // restart from x: its true residual next
                bt_load(S, 2, 0, j, ev);
                put(VA, x);
                step = 6;
                __syncthreads();
                continue;
            }
            const double m2 = m1;
            m1 = u[0];
            const double beta = m1 * alpha / (omega * m2), c = -beta * omega;
#pragma unroll
            for (int q = 0; q < R; q++) {
                const double t = c * v[q] + beta * p[q];
                p[q] = t + r[q];
            }
            if (++iter >= nmax) break;  // info 3
        }
        put(VA, p);
        step = 0;
        __syncthreads();
    }
#pragma unroll
    for (int q = 0; q < R; q++) {
        const int i = q * BT_BS + tid;
        if (i < n) xg[i] = x[q];
    }
    if (tid == 0) {
        it.resval = resval;
        it.iter = iter;
        it.info = info;
        it.cycles = cycles;
    }
}

// LDS of k_batch_small, in doubles: tile, two vectors, sums.
constexpr int BT_LDS = BT_TILE + 2 * BT_ROWS + 3 * 32;

// The queue of k_batch_solve for items whose systems have at most BT_ROWS rows
// (rows of any length).
__global__ __launch_bounds__(BT_BS) void k_batch_small(int nitems, const BatchSys *__restrict__ sys, BatchItem *items,
                                                       double *arena, size_t slot_stride, int *head, int restart_true)
{
    __shared__ double lds[BT_LDS];
    __shared__ int item_sh;
    double *w = arena + (size_t)blockIdx.x * slot_stride;
    for (;;) {
        if (threadIdx.x == 0) item_sh = atomicAdd(head, 1);
        __syncthreads();
        const int item = rs_uni(item_sh);
        __syncthreads();
        if (item >= nitems) break;
        const auto in = (RsConst<BatchItem>)items + item;
        const BatchSysTable S = (BatchSysTable)sys + in->sys;
        if (S->n <= 2 * BT_BS) bt_bicgstab<2>(S, in, items[item], w, lds, restart_true);
        else if (S->n <= 4 * BT_BS) bt_bicgstab<4>(S, in, items[item], w, lds, restart_true);
        else bt_bicgstab<8>(S, in, items[item], w, lds, restart_true);
        __syncthreads();
    }
}

__global__ __launch_bounds__(PBS) void k_batch_solve(int nitems, const BatchSys *__restrict__ sys,
                                                     BatchItem *items, double *arena, size_t slot_stride,
                                                     int *head, int restart_true)
{
    __shared__ double lds[4 * PBS / WAVE];
    __shared__ int item_sh;
    double *w = arena + (size_t)blockIdx.x * slot_stride;
    for (;;) {
        if (threadIdx.x == 0) item_sh = atomicAdd(head, 1);
        __syncthreads();
        const int item = item_sh;
        __syncthreads();
        if (item >= nitems) break;
        BatchItem &it = items[item];
        const BatchSys S = sys[it.sys];
        wg_bicgstab(S, it, w, lds, restart_true);
        __syncthreads();
    }
}

__global__ void k_zero_int(int *p) { p[threadIdx.x] = 0; }

}  // namespace cm
