// Sparse triangular solves (ACIFIM apply modes 'I' and 'J',
// ACIFIM/src/bicgstab.cpp:405-406,421-427: mkl_sparse_d_trsv on the unit
// triangular L and U with their stored diagonal): one launch per triangle, or
// one per level where levels are wide (k_trsv_level).
//
// The host orders the rows by dependency level once per factor (a row's level
// is one more than the deepest row it reads), stores the triangle's entries
// in that order and cuts every level into chunks of the rows one wave takes
// at a time.  Waves take chunks in that order from a ticket counter and solve
// a row as soon as the x entries it reads are there: x holds markers (one NaN
// bit pattern) until the owner stores the value, and a reader repeats its
// load until the marker is gone.  A chunk's rows share a level, so they read
// only rows of earlier chunks, never each other (the lanes of a wave wait
// together and could not), and tickets are handed out in chunk order to waves
// that are already running: the wave with the lowest unfinished chunk finds
// all it reads, and every wait ends, with any number of waves.  A wait that
// does not end within `spins` looks is given up all the same: fail is set,
// everybody leaves, and the host reports an error.
//
// What bounds the solve is the chain of levels (about 240 and 440 in the
// factors of a 64^3 system, a thousand rows each), so the workgroups that
// work are those of one XCD, whose waves meet in its L2: a plain store is
// written through to it and stays there, and an agent-scope load goes past
// the CU's L1 to it (a workgroup-scope load may be served from the L1).  That
// exchange takes 1.2 us with a barrier around it, against 2 us for agent-scope
// stores, which go on to memory, and 6.5 us for a kernel boundary per level.
// A level so takes 1.1 us up to 64^3 rows and 1.9 us at 128^3.
// The first workgroup to arrive fixes the XCD; the others leave.
//
// One XCD reads an eighth of what the device does, so a level of w rows takes
// about 1 + 0.4 w/1000 us here and 3.3 + 0.04 w/1000 us as a launch on all
// CUs (2^20 rows of four entries, L and U, us per apply, here / launches: 256
// levels 1430 / 1725, 128 levels 1070 / 890, 64 levels 1110 / 470, 16 levels
// 530 / 180, one level 465 / 57).  Summed over the levels the two are equal
// where the mean level has some 6000 rows: TRSV_LEVEL_ROWS.
#pragma once
#include "cm_resident.hpp"

namespace cm {

constexpr int TRSV_BS = 256;
constexpr int TRSV_LEVEL_ROWS = 6000;  // mean rows per level beyond which each level is a launch

struct TrsvCtl {  // cleared (xcd: -1) by k_trsv_prep
    int ticket;
    int pad0[31];
    int xcd;
    int pad1[31];
    int fail;
    int pad2[31];
};

// x and the control words of one or two triangular solves before their launch.
template <class T>
__global__ __launch_bounds__(BS) void k_trsv_prep(int n, T *__restrict__ x0, T *__restrict__ x1, TrsvCtl *c,
                                                  const SolveState *st)
{
    if (st && st->done) return;
    using U = typename RsBits<T>::U;
    const int t0 = blockIdx.x * BS + threadIdx.x;
    for (int i = t0; i < n; i += gridDim.x * BS) {
        reinterpret_cast<U *>(x0)[i] = RsBits<T>::MARK;
        reinterpret_cast<U *>(x1)[i] = RsBits<T>::MARK;
    }
    if (t0 < 2) {
        c[t0].ticket = 0;
        c[t0].xcd = -1;
        c[t0].fail = 0;
    }
}

// One level of a triangular solve, the rows rows[0 .. cnt) with the entries
// tptr[q] .. tptr[q + 1] of row q: x[i] = (b[i] - sum_{j != i} T[i,j] x[j]) /
// T[i,i], as k_trsv_flow below, the rows it reads being there from the
// launches before.  LPR lanes per row, lane l takes its entries l, l + LPR, ...
// Bound by memory: a level of 2^20 rows of one entry takes 14 us, 44 MB.
template <class T, class V, int LPR>
__global__ __launch_bounds__(BS) void k_trsv_level(int cnt, const int *__restrict__ rows, const int *__restrict__ tptr,
                                                   const int *__restrict__ tcol, const V *__restrict__ tval,
                                                   const float *__restrict__ rowscale, const T *__restrict__ b,
                                                   const T *__restrict__ dscale, T *x, const SolveState *st)
{
    if (st && st->done) return;
    const int q = (int)((blockIdx.x * (unsigned)BS + threadIdx.x) / LPR), l = (int)(threadIdx.x % LPR);
    if (q >= cnt) return;  // the row's LPR lanes leave together
    const int i = rows[q], e = tptr[q + 1];
    const double sc = rowscale ? (double)rowscale[i] : 1.0;
    double s = 0.0, d = 0.0, hasd = 0.0;
    for (int k = tptr[q] + l; k < e; k += LPR) {
        const int j = tcol[k];
        const double a = load_val<V, double>(tval, k) * sc;
        if (j == i) {
            d = a;
            hasd = 1.0;
        } else {
            s += a * (double)x[j];
        }
    }
#pragma unroll
    for (int o = LPR / 2; o > 0; o >>= 1) {
        s += __shfl_xor(s, o, LPR);
        d += __shfl_xor(d, o, LPR);
        hasd += __shfl_xor(hasd, o, LPR);
    }
    if (l == 0) x[i] = (T)(((dscale ? (double)(b[i] * dscale[i]) : (double)b[i]) - s) / (hasd > 0.0 ? d : 1.0));
}

// One chunk's row as a lane sees it: LPR lanes per row, lane l holds the
// row's entries l, l + LPR, ...
struct TrsvRow {
    int4 at;  // row (-1: none), its entries [y, z)
    int col[TRSV_P];
    double val[TRSV_P];
    double b, sc;
};

// x = T^{-1} b for the triangle whose entries are tcol / tval, row by row in
// chunk order: x[i] = (b[i] - sum_{j != i} T[i,j] x[j]) / T[i,i], T[i,i] = 1
// when the row stores no diagonal.  Only the declared triangle's entries are
// stored there, as the TRIANGULAR descriptor makes mkl_sparse_d_trsv read
// (ACIFIM/src/bicgstab.cpp:170-176).  Chunk c's rows are crow[c * rpc ..],
// rpc <= WAVE / LPR, all of one level.  dscale (or null): b is taken as b .* dscale,
// rounded to T (the D^-1 between the two solves of mode I).  Three chunks are
// under way in a wave: the rows of the third are being read, the entries and
// right-hand sides of the second, and the first waits for x, so no load but
// x's is waited for when its turn comes (with one chunk ahead a wave took 8
// us per chunk, mostly on the three dependent loads).  rep: told when a wait
// is given up.
template <class T, class V, int LPR>
__global__ __launch_bounds__(TRSV_BS) void k_trsv_flow(int chunks, int rpc, const int4 *__restrict__ crow,
                                                       const int *__restrict__ tcol, const V *__restrict__ tval,
                                                       const float *__restrict__ rowscale, const T *__restrict__ b,
                                                       const T *__restrict__ dscale, T *x, TrsvCtl *c, int spins,
                                                       const SolveState *st, SolveState *rep)
{
    static_assert(LPR >= 1 && LPR <= WAVE && (LPR & (LPR - 1)) == 0, "lanes per row: a power of two");
    if (st && st->done) return;
    constexpr int P = TRSV_P;
    using B = RsBits<T>;
    using U = typename B::U;
    __shared__ int sh_mine;
    if (threadIdx.x == 0) {
        const int xcd = __builtin_amdgcn_s_getreg(20 | (3 << 11));  // HW_REG_XCC_ID, 4 bits
        int want = -1;
        __hip_atomic_compare_exchange_strong(&c->xcd, &want, xcd, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT);
        sh_mine = want < 0 || want == xcd;
    }
    __syncthreads();
    if (!sh_mine) return;
    const int lane = (int)threadIdx.x & (WAVE - 1), g = lane / LPR, l = lane % LPR;
    auto take = [&]() {
        int t = 0;
        if (lane == 0) t = __hip_atomic_fetch_add(&c->ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return t;
    };
    auto rows = [&](int chunk) {  // chunk past the last: no rows
        return chunk < chunks && g < rpc ? crow[(size_t)chunk * rpc + g] : make_int4(-1, 0, 0, 0);
    };
    auto fetch = [&](TrsvRow &rw) {
        const int i = rw.at.x;
        rw.b = 0.0;
        rw.sc = 1.0;
#pragma unroll
        for (int e = 0; e < P; e++) {
            const int k = rw.at.y + l + e * LPR;
            rw.col[e] = -1;
            rw.val[e] = 0.0;
            if (k < rw.at.z) {
                rw.col[e] = tcol[k];
                rw.val[e] = load_val<V, double>(tval, k);
            }
        }
        if (i >= 0) {
            rw.b = dscale ? (double)(b[i] * dscale[i]) : (double)b[i];
            if (rowscale) rw.sc = (double)rowscale[i];
        }
    };
    bool gone = false;  // this lane saw a wait given up
    // x entries j[e] (-1: none), waiting for those not there yet
    auto gather = [&](const int(&j)[P], T(&v)[P]) {
        U w[P];
#pragma unroll
        for (int e = 0; e < P; e++) w[e] = j[e] >= 0 ? rs_peek(x, j[e]) : 0;
        for (int spin = 1;; spin++) {
            bool miss = false;
#pragma unroll
            for (int e = 0; e < P; e++) miss |= w[e] == B::MARK;
            if (!miss) break;
            if (spin % 1024 == 0 || spin >= spins) {
                if (spin >= spins) __hip_atomic_store(&c->fail, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (__hip_atomic_load(&c->fail, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) gone = true;
            }
            if (gone) break;
            __builtin_amdgcn_s_sleep(1);
#pragma unroll
            for (int e = 0; e < P; e++)
                if (w[e] == B::MARK) w[e] = rs_peek(x, j[e]);
        }
#pragma unroll
        for (int e = 0; e < P; e++) v[e] = rs_val<T>(w[e]);
    };
    TrsvRow cur, nxt;
    int t0 = rs_uni(take());
    if (t0 >= chunks) return;
    int t1 = take(), t2 = take();
    cur.at = rows(t0);
    t1 = rs_uni(t1);
    nxt.at = rows(t1);
    fetch(cur);
    for (;;) {
        const int t3 = take();
        t2 = rs_uni(t2);
        const int4 third = rows(t2);
        fetch(nxt);
        if (cur.at.x >= 0) {  // a row's LPR lanes together
            const int i = cur.at.x;
            double s = 0.0, d = 0.0, hasd = 0.0;
            int j[P];
            T xv[P];
#pragma unroll
            for (int e = 0; e < P; e++) j[e] = cur.col[e] == i ? -1 : cur.col[e];
            gather(j, xv);
#pragma unroll
            for (int e = 0; e < P; e++) {
                if (cur.col[e] < 0) continue;
                const double a = cur.val[e] * cur.sc;
                if (cur.col[e] == i) {
                    d = a;
                    hasd = 1.0;
                } else {
                    s += a * (double)xv[e];
                }
            }
            for (int k = cur.at.y + l + P * LPR; k < cur.at.z; k += P * LPR) {
                int jc[P];
                double a[P];
#pragma unroll
                for (int e = 0; e < P; e++) {
                    jc[e] = j[e] = -1;
                    a[e] = 0.0;
                    if (k + e * LPR < cur.at.z) {
                        jc[e] = tcol[k + e * LPR];
                        a[e] = load_val<V, double>(tval, k + e * LPR) * cur.sc;
                        j[e] = jc[e] == i ? -1 : jc[e];
                    }
                }
                gather(j, xv);
#pragma unroll
                for (int e = 0; e < P; e++) {
                    if (jc[e] < 0) continue;
                    if (jc[e] == i) {
                        d = a[e];
                        hasd = 1.0;
                    } else {
                        s += a[e] * (double)xv[e];
                    }
                }
            }
#pragma unroll
            for (int o = LPR / 2; o > 0; o >>= 1) {
                s += __shfl_xor(s, o, LPR);
                d += __shfl_xor(d, o, LPR);
                hasd += __shfl_xor(hasd, o, LPR);
            }
            if (l == 0 && !gone) {
                const T xi = (T)((cur.b - s) / (hasd > 0.0 ? d : 1.0));
                U w;
                __builtin_memcpy(&w, &xi, sizeof w);
                __hip_atomic_store(reinterpret_cast<U *>(x) + i, w == B::MARK ? B::QNAN : w, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
            }
        }
        if (__any(gone)) {
            if (lane == 0 && rep) {
                rep->stalled = 1;
                rep->done = 1;
            }
            break;
        }
        if (t1 >= chunks) break;
        t1 = t2;
        t2 = t3;
        cur = nxt;
        nxt.at = third;
    }
}

}  // namespace cm
