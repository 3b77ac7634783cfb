// Whole BiCGSTAB solves in one launch: a grid that stays resident on the
// device and passes vectors between its workgroups while it runs.
//
// A pass of the launch-per-operation path is 12 kernels of a few microseconds
// (45-55 us on systems of 10^4 to 10^5 rows), whatever the system's size: it
// is bound by launches, kernel boundaries and dependent loads, not by memory.
// Here every workgroup owns a fixed range of rows, and each thread keeps its
// R rows' x, r (then s), r0, p, v and M p (then M s), and their values on the
// matrices' diagonals, in registers for the whole solve.  FP64, per pass: 18
// us at 100^2 rows (45 launched), 26 us at 45^3 (54), 42 us at 58^3 (75), 68
// us at 64^3 (75), 84 us at 73^3 (93); FP32 32 us at 58^3 (62), 46 us at 73^3
// (75).  What bounds it is the chain of eight exchanges: of the
// pass at 100^2 rows the gathers of its six products are 6.5 us, the two
// reductions 5.5, the sums over the diagonals 2, the rest LDS writes, barriers
// and stores.  With three and four rows per thread (FP64) the values held
// spill or are read again.
//
// Exchange.  Only the vectors that other rows gather go through memory (p,
// H p, M p and s, H s, M s).  Each entry is its own arrival flag: the buffers
// hold a marker (one NaN bit pattern) until the owner stores the value, and a
// reader repeats its load until the marker is gone.  Stores and loads are
// relaxed agent-scope atomics, which go past the per-XCD L2s; a value is
// published once and never changed while anybody may read it, so no fence,
// no cache invalidation and no separate flag is needed.  One exchange costs
// 2.0-2.4 us from 32 to 256 workgroups (10^4 to 9*10^4 rows), a device-wide
// barrier with cache invalidation 2.5-6 us and a kernel boundary 3.5 us.
// A result that equals the marker bit for bit is published as another NaN.
//
// Columns.  The right-hand sides of a block are columns of the grid (gridDim
// y): each has its own workgroups, exchanged vectors, reduction slots,
// scalars and exits, and they meet only on arrival.
//
// The two reductions of a pass (alpha; omega) are all-to-all exchanges of the
// workgroups' partial sums, added in workgroup order by every workgroup, so
// all of them compute the same scalars and take the same exits.  They also
// order the reuse of the buffers: an owner restores the markers of a buffer
// after the reduction that every reader's last read precedes, and its stores
// are complete before it takes part in the next reduction, which precedes
// the next read of that buffer.
//
// Progress.  Waiting needs every workgroup running at once.  The grid is at
// most one workgroup per CU (on some CUs less, rs_room), and a workgroup starts working only when all
// have arrived: each counts itself in, the first closes the count when the
// grid is complete or after RS_JOIN_TICKS, and if anyone is missing then all
// leave; the caller launches the grid again and at last takes the
// launch-per-operation path.  All other waits
// end after RS_SPINS loads.  A workgroup whose wait ended so leaves without
// writing its rows of x, and a column counts as solved only when all its
// workgroups have written theirs: others may still get through the reduction
// that one gave up on, if its own sums were out by then.  The host gives the
// columns that do not count their starting x back (k_rs_restore) and takes
// the launch-per-operation path for them.
#pragma once
#include "cm_kernels.hpp"

namespace cm {

constexpr int RS_WGS = 256;                // workgroups at most (one per CU)
constexpr int RS_MAX_ROWS = RS_WGS / 4 * 3 * 512 * 4;
constexpr int RS_PER = 8;                  // staged entries per thread and step
constexpr int RS_STEPS = 16;               // window steps at most (half of them with 1024 threads)
constexpr int RS_SPINS = 1 << 20;          // loads of one entry before a wait gives up (about a second)
constexpr int RS_GROUP = 256;              // rows over which the spread of CSR entries is taken
constexpr double RS_CSR_STEPS = 4.0;       // gather steps of the three products' CSR entries
constexpr int RS_CSR_TWICE = 1 << 19;      // rows on which twice those
constexpr double RS_CSR_ROW = 256.0;       // entries of the three products' longest CSR rows
constexpr int RS_TRIES = 16;               // launches of a grid that does not arrive
constexpr int RS_SKIP = 16;                // launched solves after that
constexpr long long RS_JOIN_TICKS = 1000000;  // 100 MHz ticks the grid may take to arrive (10 ms)
constexpr int RS_K = 4;                    // sums per reduction
constexpr int RS_SETS = 5;                 // reduction slots: setup, alpha and omega of even and odd passes

// CUs that resident grids of this shape may take, so that kernels of other
// streams go on.  These start on what registers a CU has left, and where a
// shader engine has room on none of its 8 CUs they wait for the solve to end
// (dispatch waits for the engine whose turn it is).
// * FP64 on 512 threads (254 to 256 registers) and FP32 with 4 rows take a CU
//   whole.  A launched solve of 100^2 rows (2.3 ms alone) beside a loop of such
//   solves took 3.0 ms next to 216 workgroups, 120 to 340 next to 233 to 256;
//   one of 110^3 rows (21.5 ms alone) 42, 62 and 115 ms next to 140, 191 and
//   215, 530 to 1400 next to 233 to 256.  They get three quarters.
// * FP32 with 2 and 3 rows (218 to 225 registers) leaves room for small
//   kernels on each CU: 3.3 and 42 to 57 ms next to 245 workgroups, but 22 to
//   27 and 92 to 115 next to 256.  A CU of each XCD is left.
// * 256 threads and FP32 with one row (174) leave a third of every CU or
//   more: 3.2 and 32 ms next to 250 workgroups.
// grid: workgroups of one grid; whole: they take their CUs whole, and all such
// grids together get no more; all: grids of any shape together.
struct RsRoom {
    int grid, all;
    bool whole;
};
template <class T>
constexpr RsRoom rs_room(int bsz, int rows, int cus)
{
    const bool f64 = sizeof(T) == 8;
    const int most = cus - cus / 32;
    if (bsz == 256 || (!f64 && rows == 1)) return {cus, cus, false};
    return f64 || rows == 4 ? RsRoom{cus - cus / 4, most, true} : RsRoom{most, most, false};
}

constexpr int rs_steps(int bsz) { return bsz < 1024 ? RS_STEPS : RS_STEPS / 2; }

template <class T>
struct RsBits;
template <>
struct RsBits<double> {
    using U = unsigned long long;
    static constexpr U MARK = 0xfff5c0de5ea15eedull, QNAN = 0x7ff8000000000000ull;
};
template <>
struct RsBits<float> {
    using U = unsigned;
    static constexpr U MARK = 0xffe5ea1du, QNAN = 0x7fc00000u;
};

template <class T>
__device__ __forceinline__ void rs_put_bits(T *p, typename RsBits<T>::U b)
{
    __hip_atomic_store(reinterpret_cast<typename RsBits<T>::U *>(p), b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ __forceinline__ void rs_put(T *p, T v)
{
    typename RsBits<T>::U b;
    __builtin_memcpy(&b, &v, sizeof b);
    rs_put_bits(p, b == RsBits<T>::MARK ? RsBits<T>::QNAN : b);
}
// p[i], i >= 0, through a 32-bit byte offset (the vectors and the diagonals
// of RS_MAX_ROWS rows stay below 4 GB), so a wave needs one address register
// per load
template <class T>
__device__ __forceinline__ const T *rs_at(const T *p, unsigned i)
{
    return reinterpret_cast<const T *>(reinterpret_cast<const char *>(p) + i * (unsigned)sizeof(T));
}
template <class T>
__device__ __forceinline__ typename RsBits<T>::U rs_peek(const T *p, int i)
{
    return __hip_atomic_load(reinterpret_cast<const typename RsBits<T>::U *>(rs_at(p, (unsigned)i)), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ __forceinline__ T rs_val(typename RsBits<T>::U b)
{
    T v;
    __builtin_memcpy(&v, &b, sizeof v);
    return v;
}

// A value that is the same on every lane, held in scalar registers.
__device__ __forceinline__ int rs_uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ double rs_uni(double v)
{
    int w[2];
    __builtin_memcpy(w, &v, sizeof w);
    w[0] = rs_uni(w[0]);
    w[1] = rs_uni(w[1]);
    __builtin_memcpy(&v, w, sizeof w);
    return v;
}

// A pointer read from a table, known to point to device memory: its loads are
// global ones, not flat ones (which also wait for LDS).
template <class X>
__device__ __forceinline__ X *rs_glob(X *p)
{
    return (X *)(__attribute__((address_space(1))) X *)p;
}

constexpr int RS_COLS = 16;  // columns of a launch at most

// Control words of one launch, cleared by k_rs_prep.
struct RsCtl {
    unsigned join;  // arrivals; top bit: closed
    unsigned pad0[31];
    unsigned verdict;  // 1: all arrived, 2: leave
    unsigned pad1[31];
    unsigned fin[RS_COLS];  // workgroups of a column that wrote their x
};

// One matrix of the solve: diagonals with a CSR remainder (nd diagonals), or
// CSR alone (nd = 0, the remainder is the matrix).
template <class V>
struct RsMat {
    int nd, ldn;
    const V *dval;
    const int *ptr, *col;  // remainder or CSR; ptr null: no remainder
    const V *val;
    const float *rowscale;
    // the x windows, cut into steps of one entry per thread: step s holds x
    // entries (first row of the workgroup) + gs[s] + thread, thread < gc[s],
    // at LDS position s * BSZ + thread; diagonal d of the workgroup's row k
    // reads position wpos[d] + k
    int ns;
    int gs[RS_STEPS], gc[RS_STEPS], wpos[DIA_MAX];
};

// The windows of the diagonals `off` (ascending) for workgroups of `rows`
// rows in steps of bsz; false when they need more than RS_STEPS steps.
// Offsets at most `rows` apart share a window: the gap between them then
// costs no more entries than a second window.
template <class V>
static bool rs_windows(const std::vector<int> &off, int bsz, int rows, RsMat<V> &m)
{
    m.ns = 0;
    for (size_t d = 0; d < off.size();) {
        size_t e = d + 1;
        while (e < off.size() && off[e] - off[e - 1] <= rows) e++;
        const int lo = off[d], len = off[e - 1] - lo + rows;
        for (size_t k = d; k < e; k++) m.wpos[k] = m.ns * bsz + (off[k] - lo);
        for (int c = 0; c < len; c += bsz) {
            if (m.ns == rs_steps(bsz)) return false;
            m.gs[m.ns] = lo + c;
            m.gc[m.ns++] = len - c < bsz ? len - c : bsz;
        }
        d = e;
    }
    return true;
}

// Column k of the launch (blockIdx.y) is column col[k] of b and x, which hold
// `stride` columns interleaved, and solves to tol[k].
template <class T, class VA, class VF>
struct RsArgs {
    int n, nmax, variant, maxmsteps, info_in, zero_start, trace_cap, stride, ncols, spins;
    long long join_ticks;
    int col[RS_COLS];
    double tol[RS_COLS], eps;
    double *trace;  // device; first column
    RsMat<VF> H, G;
    RsMat<VA> A;
    const T *idv, *b;
    T *x, *save;      // save: the starting x (n x stride), not used on a zero start
    T *ex[6];         // exchanged vectors of ncols x n: p, H p, M p, s, H s, M s
    double *slots;    // ncols x RS_SETS x RS_K x RS_WGS
    RsCtl *ctl;
    SolveState *out;  // pinned host memory, one per column of the launch
};

// What differs between the columns of a launch.
template <class T>
struct RsCol {
    double tol, *slots, *trace;
    T *ex[6], *x;
    const T *b;
    SolveState *out;
};
template <class T, class VA, class VF>
struct RsTable {
    RsArgs<T, VA, VF> a;
    RsCol<T> c[RS_COLS];
};

// The arguments lie in device memory and are read through the scalar cache
// (the constant address space), whatever index a step picks a matrix by.
template <class X>
using RsConst = const __attribute__((address_space(4))) X *;

// The longest row and the most entries in RS_GROUP consecutive rows, out[0]
// and out[1] (0 before); a workgroup per group.
__global__ __launch_bounds__(RS_GROUP) void k_row_spread(int n, const int *ptr, int *out)
{
    const int r0 = blockIdx.x * RS_GROUP, i = r0 + threadIdx.x;
    int len = i < n ? ptr[i + 1] - ptr[i] : 0;
    for (int d = WAVE / 2; d > 0; d /= 2) len = max(len, __shfl_xor(len, d, WAVE));
    if (threadIdx.x % WAVE == 0) atomicMax(out, len);
    if (threadIdx.x == 0) atomicMax(out + 1, ptr[min(r0 + RS_GROUP, n)] - ptr[r0]);
}

// Markers into the exchanged vectors and reduction slots, control words 0, the
// starting x kept, and the arguments to where the solve reads them (every column's pointers
// ready: computed in the solve they made a pass 1.5% slower).
template <class T, class VA, class VF>
__global__ __launch_bounds__(BS) void k_rs_prep(RsArgs<T, VA, VF> a, RsTable<T, VA, VF> *to)
{
    const int t0 = blockIdx.x * BS + threadIdx.x, st = gridDim.x * BS;
    using U = typename RsBits<T>::U;
    for (int i = t0; i < a.n * a.ncols; i += st) {
#pragma unroll
        for (int e = 0; e < 6; e++) reinterpret_cast<U *>(a.ex[e])[i] = RsBits<T>::MARK;
    }
    for (int i = t0; i < a.ncols * RS_SETS * RS_K * RS_WGS; i += st)
        reinterpret_cast<unsigned long long *>(a.slots)[i] = RsBits<double>::MARK;
    if (!a.zero_start)
        for (int i = t0; i < a.n * a.stride; i += st) a.save[i] = a.x[i];
    if (t0 == 0) {
        a.ctl->join = 0;
        a.ctl->verdict = 0;
        to->a = a;
    }
    if (t0 < RS_COLS) a.ctl->fin[t0] = 0;
    if (t0 < a.ncols) {
        RsCol<T> c;
        int col = 0;
#pragma unroll
        for (int k = 0; k < RS_COLS; k++)
            if (k == t0) {
                c.tol = a.tol[k];
                col = a.col[k];
            }
        c.slots = a.slots + (size_t)t0 * RS_SETS * RS_K * RS_WGS;
        c.trace = t0 == 0 ? a.trace : nullptr;
#pragma unroll
        for (int e = 0; e < 6; e++) c.ex[e] = a.ex[e] + (size_t)t0 * a.n;
        c.x = a.x + col;
        c.b = a.b + col;
        c.out = a.out + t0;
        to->c[t0] = c;
    }
}

// Column col of x as it was before the launch.
template <class T>
__global__ __launch_bounds__(BS) void k_rs_restore(int n, int stride, int col, const T *__restrict__ save,
                                                   T *__restrict__ x)
{
    for (int i = blockIdx.x * BS + threadIdx.x; i < n; i += gridDim.x * BS)
        x[(size_t)i * stride + col] = save[(size_t)i * stride + col];
}

// x[j[q]] for the q with j[q] >= 0 (0 otherwise), waiting for entries that
// are not there yet; dead[0] is set (and honoured) when a wait gives up, after
// dead[1] loads.
template <class T, int R>
__device__ __forceinline__ void rs_gather(const T *x, const int (&j)[R], T (&v)[R], volatile int *dead)
{
    using B = RsBits<T>;
    typename B::U b[R];
#pragma unroll
    for (int q = 0; q < R; q++) b[q] = j[q] >= 0 ? rs_peek(x, j[q]) : 0;
    for (int spin = 0;;) {
        bool miss = false;
#pragma unroll
        for (int q = 0; q < R; q++) miss |= b[q] == B::MARK;
        if (!miss) break;
        if (++spin >= dead[1]) *dead = 1;
        if (*dead) break;
#pragma unroll
        for (int q = 0; q < R; q++)
            if (b[q] == B::MARK) b[q] = rs_peek(x, j[q]);
    }
#pragma unroll
    for (int q = 0; q < R; q++) v[q] = rs_val<T>(b[q]);
}

// A product's part that does not depend on x, fetched one product ahead: the
// thread's first remainder entries (positions in x, -1: none, and values) and
// its rows' remainder bounds.
constexpr int RS_NW = 8;  // window steps gathered together
constexpr int RS_DC = 6;  // diagonals per step of those not held
// remainder entries gathered with them: fewer where the rows' values take
// most of the registers (spilling them made a pass 10-30% slower)
template <class Acc, int R>
constexpr int rs_nr() { return R * sizeof(Acc) <= 8 ? 4 : 2; }
template <class Acc, int R>
struct RsTile {
    int j[rs_nr<Acc, R>()], a[R], e[R];
    Acc ev[rs_nr<Acc, R>()];
};

// x entry of window step s for this thread, -1 for none.
template <class V>
__device__ __forceinline__ int rs_window(RsConst<RsMat<V>> m, int s, int n, int row0)
{
    const int c = row0 + m->gs[s] + (int)threadIdx.x;
    return (int)threadIdx.x < m->gc[s] && (unsigned)c < (unsigned)n ? c : -1;
}

// N remainder entries per thread from c0 on: positions in x and values.
template <class V, class Acc, int BSZ, int N>
__device__ __forceinline__ void rs_tile(RsConst<RsMat<V>> m, int c0, int re, int *j, Acc *ev)
{
#pragma unroll
    for (int q = 0; q < N; q++) {
        const int k = c0 + q * BSZ + (int)threadIdx.x;
        j[q] = -1;
        ev[q] = 0;
        if (k < re) {
            j[q] = rs_glob(m->col)[k];
            ev[q] = load_val<V, Acc>(rs_glob(m->val), k);
        }
    }
}

template <class V, class Acc, int BSZ, int R>
__device__ __forceinline__ void rs_ahead(RsConst<RsMat<V>> m, int rs, int re, int n, int row0, RsTile<Acc, R> &f)
{
    constexpr int NR = rs_nr<Acc, R>();
#pragma unroll
    for (int q = 0; q < NR; q++) f.j[q] = -1;
    if (re > rs) {
        rs_tile<V, Acc, BSZ, NR>(m, rs, re, f.j, f.ev);
#pragma unroll
        for (int q = 0; q < R; q++) {
            const int i = row0 + q * BSZ + (int)threadIdx.x;
            f.a[q] = rs_glob(m->ptr)[min(i, n)];
            f.e[q] = rs_glob(m->ptr)[min(i + 1, n)];
        }
    }
}

// A thread's values on the first ND diagonals of m, held for the whole solve.
template <class V, int BSZ, int R, int ND>
__device__ __forceinline__ void rs_hold(RsConst<RsMat<V>> m, int n, int row0, V (&dv)[R][ND])
{
#pragma unroll
    for (int q = 0; q < R; q++) {
        const int i = row0 + q * BSZ + (int)threadIdx.x;
#pragma unroll
        for (int d = 0; d < ND; d++)
            dv[q][d] = d < m->nd && i < n ? *rs_at(rs_glob(m->dval), (unsigned)(d * m->ldn + i)) : (V)0.0f;
    }
}

// The first NW window steps and the entries fetched ahead, gathered together.
template <class T, class V, class Acc, int BSZ, int R, int NW>
__device__ __forceinline__ void rs_first(RsConst<RsMat<V>> m, const RsTile<Acc, R> &f, bool rest, int n, int row0,
                                         const T *x, T *win, Acc *prod, volatile int *dead)
{
    constexpr int NR = rs_nr<Acc, R>();
    const int tid = (int)threadIdx.x, ns = m->ns;
    int j[NW + NR];
    T xv[NW + NR];
#pragma unroll
    for (int q = 0; q < NW; q++) j[q] = rs_window(m, q, n, row0);
#pragma unroll
    for (int q = 0; q < NR; q++) j[NW + q] = f.j[q];
    rs_gather<T, NW + NR>(x, j, xv, dead);
#pragma unroll
    for (int q = 0; q < NW; q++)
        if (q < ns) win[q * BSZ + tid] = xv[q];
    if (rest)
#pragma unroll
        for (int q = 0; q < NR; q++) prod[q * BSZ + tid] = f.ev[q] * (Acc)xv[NW + q];
}

// Row sums y of m x for the workgroup's R * BSZ rows from row0 on (row q *
// BSZ + thread of them in y[q]).  The part of x that the diagonals touch is a
// few windows (diagonals whose offsets lie closer than the workgroup's rows
// share one: the 17 diagonals of a 3D factor are 3), which the workgroup
// gathers once into LDS, so an entry is loaded past the L2s once or twice per
// workgroup instead of once per diagonal.  The remainder (or the whole
// matrix, in CSR) is one contiguous range of entries [rs, re), gathered by
// the whole workgroup and added by each row's thread in column order.  Every
// thread of the workgroup takes part.
template <class T, class V, class Acc, int BSZ, int R, int ND>
__device__ __forceinline__ void rs_rows(RsConst<RsMat<V>> m, const V (&dv)[R][ND], const RsTile<Acc, R> &f, int rs,
                                        int re, int n, int row0, const T *x, T *win, Acc *prod, volatile int *dead,
                                        Acc (&y)[R])
{
#pragma clang fp contract(off)
    constexpr int NR = rs_nr<Acc, R>();
    const int tid = (int)threadIdx.x, nd = m->nd, ns = m->ns;
    // fewer loads in the chain where few windows are read (no second copy with 4 rows per thread: spills)
    if (R < 4 && ns <= RS_NW / 2) rs_first<T, V, Acc, BSZ, R, RS_NW / 2>(m, f, re > rs, n, row0, x, win, prod, dead);
    else rs_first<T, V, Acc, BSZ, R, RS_NW>(m, f, re > rs, n, row0, x, win, prod, dead);
    for (int s0 = RS_NW; s0 < ns; s0 += RS_NW) {
        int j2[RS_NW];
        T x2[RS_NW];
#pragma unroll
        for (int q = 0; q < RS_NW; q++) j2[q] = rs_window(m, s0 + q, n, row0);
        rs_gather<T, RS_NW>(x, j2, x2, dead);
#pragma unroll
        for (int q = 0; q < RS_NW; q++) win[(s0 + q) * BSZ + tid] = x2[q];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < R; q++) y[q] = 0;
    if constexpr (R >= 4) {  // no registers left for more than one at a time
#pragma unroll
        for (int d = 0; d < ND; d++)
            if (d < nd) {
                const int w = m->wpos[d] + tid;
#pragma unroll
                for (int q = 0; q < R; q++) y[q] += dia_val<V, Acc>(dv[q][d]) * (Acc)win[w + q * BSZ];
            }
    } else {
        // DH diagonals at a time: their positions, their x, then the sums in
        // order.  One by one each waited for its position and its x, 60 cycles
        // a diagonal; with this and the shorter gather of few windows a pass
        // took 18.3 us instead of 19.2 at 100^2 rows, 25.9 (27.5) at 45^3,
        // 40.3 (43.5) at 64^3 and in FP32 24.8 (27.9) and 32.1 (34.7).
        constexpr int DH = R * sizeof(Acc) <= 8 ? 6 : 4;
#pragma unroll
        for (int d0 = 0; d0 < ND; d0 += DH)
            if (d0 < nd) {
                T xd[R][DH];
#pragma unroll
                for (int d = 0; d < DH; d++)
#pragma unroll
                    for (int q = 0; q < R; q++)
                        if (d0 + d < ND) xd[q][d] = win[m->wpos[d0 + d] + tid + q * BSZ];
#pragma unroll
                for (int d = 0; d < DH; d++)
                    if (d0 + d < ND)
#pragma unroll
                        for (int q = 0; q < R; q++) {
                            const Acc t = dia_val<V, Acc>(dv[q][d0 + d]) * (Acc)xd[q][d];
                            y[q] += d0 + d < nd ? t : (Acc)0;  // y, a sum begun at 0, is never -0
                        }
            }
    }
    for (int d0 = ND; d0 < nd; d0 += RS_DC) {  // diagonals not held
        V v[R][RS_DC];
#pragma unroll
        for (int d = 0; d < RS_DC; d++)
#pragma unroll
            for (int q = 0; q < R; q++)
                v[q][d] = *rs_at(rs_glob(m->dval), (unsigned)(min(d0 + d, nd - 1) * m->ldn + min(row0 + q * BSZ + tid, n - 1)));
#pragma unroll
        for (int d = 0; d < RS_DC; d++)
            if (d0 + d < nd) {
                const int w = m->wpos[d0 + d] + tid;
#pragma unroll
                for (int q = 0; q < R; q++) y[q] += dia_val<V, Acc>(v[q][d]) * (Acc)win[w + q * BSZ];
            }
    }
    if (re > rs) {
        int c1 = rs + NR * BSZ;
#pragma unroll
        for (int q = 0; q < R; q++) {
            const int k1 = min(f.e[q], c1);
            for (int k = f.a[q]; k < k1; k++) y[q] += prod[k - rs];
        }
        for (int c0 = c1; c0 < re; c0 = c1) {  // uniform over the workgroup
            int jt[RS_PER];
            Acc ev[RS_PER];
            T xt[RS_PER];
            rs_tile<V, Acc, BSZ, RS_PER>(m, c0, re, jt, ev);
            rs_gather<T, RS_PER>(x, jt, xt, dead);
            __syncthreads();  // prod of the tile before has been read
#pragma unroll
            for (int q = 0; q < RS_PER; q++) prod[q * BSZ + tid] = ev[q] * (Acc)xt[q];
            __syncthreads();
            c1 = c0 + RS_PER * BSZ;
#pragma unroll
            for (int q = 0; q < R; q++) {
                const int k1 = min(f.e[q], c1);
                for (int k = max(f.a[q], c0); k < k1; k++) y[q] += prod[k - c0];
            }
        }
    }
    __syncthreads();  // the LDS is overwritten by the next product
#pragma unroll
    for (int q = 0; q < R; q++) {
        const int i = row0 + q * BSZ + tid;
        if (m->rowscale && i < n) y[q] *= (Acc)rs_glob(m->rowscale)[i];
        if (i >= n) y[q] = 0;  // rows past n took other rows' values
    }
}

// v moved across the lanes of a row of 16 by one DPP step.
template <int CTRL>
__device__ __forceinline__ double rs_dpp(double v)
{
    int w[2];
    __builtin_memcpy(w, &v, sizeof w);
    w[0] = __builtin_amdgcn_update_dpp(0, w[0], CTRL, 0xf, 0xf, true);
    w[1] = __builtin_amdgcn_update_dpp(0, w[1], CTRL, 0xf, 0xf, true);
    __builtin_memcpy(&v, w, sizeof w);
    return v;
}
// Sum over each aligned group of N = 4, 8 or 16 lanes, on all of them.
template <int N>
__device__ __forceinline__ double rs_group_sum(double v)
{
    v += rs_dpp<0xb1>(v);  // lane ^ 1
    v += rs_dpp<0x4e>(v);  // lane ^ 2
    if constexpr (N >= 8) v += rs_dpp<0x141>(v);   // mirrored halves of a row
    if constexpr (N >= 16) v += rs_dpp<0x140>(v);  // mirrored row
    return v;
}
__device__ __forceinline__ double rs_lane(double v, int lane)
{
    int w[2];
    __builtin_memcpy(w, &v, sizeof w);
    w[0] = __builtin_amdgcn_readlane(w[0], lane);
    w[1] = __builtin_amdgcn_readlane(w[1], lane);
    __builtin_memcpy(&v, w, sizeof w);
    return v;
}
// Sum over the wave, on every lane.  In registers (DPP and lane reads): the
// six LDS-crossbar shuffles of wave_sum are about 0.3 us in a chain.
__device__ __forceinline__ double rs_wave_sum(double v)
{
    v = rs_group_sum<16>(v);
    return (rs_lane(v, 0) + rs_lane(v, 16)) + (rs_lane(v, 32) + rs_lane(v, 48));
}

// Sums of RS_K values over the grid, the same on every thread: the workgroups'
// sums are exchanged through set `set` of the slots and added in workgroup
// order.  Every store the workgroup made before is complete when its sums
// are published.  red: LDS of this set's own (a set comes again only after
// other reductions' barriers).
template <int BSZ>
__device__ __forceinline__ void rs_allsum(double (&v)[RS_K], double *slots, int set, double *red, volatile int *dead)
{
    constexpr int K = RS_K, NW = BSZ / WAVE, C = RS_WGS / WAVE;
    static_assert((NW == 4 || NW == 8 || NW == 16) && C == 4 && C <= NW, "waves per workgroup");
    const int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE;
#pragma unroll
    for (int k = 0; k < K; k++) v[k] = rs_wave_sum(v[k]);
    if (lane == 0)
#pragma unroll
        for (int k = 0; k < K; k++) red[k * NW + w] = v[k];
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    double *base = slots + (size_t)set * K * RS_WGS;
    if (w == 0) {
        const double q = rs_group_sum<NW>(lane < K * NW ? red[lane] : 0.0);
        // a workgroup that gave up withholds its sums, so nobody goes on without it
        if (lane < K * NW && lane % NW == 0 && !*dead) rs_put(base + (lane / NW) * RS_WGS + blockIdx.x, q);
    }
    if (w < C) {  // wave w adds workgroups [w * WAVE, (w + 1) * WAVE)
        const int b = w * WAVE + lane;
        int j[K];
        double t[K];
#pragma unroll
        for (int k = 0; k < K; k++) j[k] = b < (int)gridDim.x ? k * RS_WGS + b : -1;
        rs_gather<double, K>(base, j, t, dead);
#pragma unroll
        for (int k = 0; k < K; k++) t[k] = rs_wave_sum(t[k]);
        if (lane == 0)
#pragma unroll
            for (int k = 0; k < K; k++) red[K * NW + k * C + w] = t[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; k++) {
        const double *t = red + K * NW + k * C;
        v[k] = rs_uni((t[0] + t[1]) + (t[2] + t[3]));
    }
}

// Arrival of the grid; true when every workgroup is running.
__device__ __forceinline__ bool rs_join(RsCtl *c, long long ticks, int *sh)
{
    const unsigned all = gridDim.x * gridDim.y;
    if (threadIdx.x == 0) {
        constexpr unsigned CLOSED = 0x80000000u;
        unsigned verdict = 2;
        const unsigned q = __hip_atomic_fetch_add(&c->join, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (!(q & CLOSED)) {
            if (q == 0) {
                const long long t0 = wall_clock64();
                while (__hip_atomic_load(&c->join, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < all &&
                       wall_clock64() - t0 < ticks) {
                }
                const unsigned f = __hip_atomic_fetch_or(&c->join, CLOSED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                verdict = f == all && ticks > 0 ? 1u : 2u;  // no time at all: never (tests)
                __hip_atomic_store(&c->verdict, verdict, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            } else {
                for (int spin = 0; spin < RS_SPINS; spin++) {
                    verdict = __hip_atomic_load(&c->verdict, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    if (verdict) break;
                }
                if (!verdict) verdict = 2;
            }
        }
        *sh = (int)verdict;
    }
    __syncthreads();
    return rs_uni(*sh) == 1;
}

// The reference loop (AFIIM/src/bicgstab.cpp:149-281, ACIFIM's non-finite
// alpha guard, ACIFIM/src/bicgstab.cpp:208-213) on R rows per thread: row
// (blockIdx * R + q) * BSZ + thread.  out->done is set when all workgroups of
// the column wrote their x; when the grid did not arrive x is as it was, when
// a wait gave up some rows may be written.  One loop iteration is half a pass:
// step 2 applies M and A to p and ends in alpha, step 5 to s and ends in
// omega; step 6 is the initial residual.  The new r0 . r is formed from the
// sums the omega reduction carries anyway, r0 . s - omega (r0 . t), where
// r0 . s is what rounding leaves of 0; this saves an exchange of 2 us per pass.
template <class T, class VA, class VF, int BSZ, int R>
__global__ __launch_bounds__(BSZ) void k_rs_solve(const RsTable<T, VA, VF> *args)
{
    auto g = (RsConst<RsArgs<T, VA, VF>>)&args->a;
    auto c = (RsConst<RsCol<T>>)&args->c[blockIdx.y];
    using Acc = typename std::conditional<std::is_same<T, double>::value, double, float>::type;
    __shared__ Acc prod[RS_PER * BSZ];
    __shared__ T win[rs_steps(BSZ) * BSZ];
    __shared__ double red[RS_SETS][RS_K * (BSZ / WAVE + RS_WGS / WAVE)];
    __shared__ int sh_join, sh_dead[2];  // a wait gave up; loads until one does
    if (threadIdx.x == 0) {
        sh_dead[0] = 0;
        sh_dead[1] = g->spins;
    }
    if (!rs_join(g->ctl, g->join_ticks, &sh_join)) return;
    volatile int *dead = sh_dead;
    const int n = g->n, tid = threadIdx.x;
    int row0 = (int)blockIdx.x * R * BSZ;
    T x[R], r[R], r0[R], p[R], v[R], w[R], dv[R];  // w: M p, then M s
#pragma unroll
    for (int q = 0; q < R; q++) {
        const int i = row0 + q * BSZ + tid;
        x[q] = r[q] = dv[q] = r0[q] = p[q] = v[q] = w[q] = (T)0;
        if (i < n) {
            dv[q] = rs_glob(g->idv)[i];
            r[q] = rs_glob(c->b)[(size_t)i * g->stride];
            if (!g->zero_start) {  // the initial residual gathers x
                x[q] = rs_glob(c->x)[(size_t)i * g->stride];
                rs_put(rs_glob(c->ex[5]) + i, x[q]);
            }
        }
    }
    // diagonals held in registers: a 7-point matrix's and its PDFIIM factors'
    // 17 and 4, A's only while they fit
    constexpr int HA = R * sizeof(Acc) <= 8 ? 7 : 1;
    VF dh[R][17], dg[R][4];
    VA da[R][HA];
    rs_hold<VF, BSZ, R, 17>(&g->H, n, row0, dh);
    rs_hold<VF, BSZ, R, 4>(&g->G, n, row0, dg);
    rs_hold<VA, BSZ, R, HA>(&g->A, n, row0, da);
    // the workgroup's remainder (CSR) entries of H, G and A
    int lo[3], hi[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const int *ptr = k == 0 ? g->H.ptr : k == 1 ? g->G.ptr : g->A.ptr;
        lo[k] = ptr ? rs_uni(ptr[min(row0, n)]) : 0;
        hi[k] = ptr ? rs_uni(ptr[min(row0 + R * BSZ, n)]) : 0;
    }
    RsTile<Acc, R> tile;
    rs_ahead<VA, Acc, BSZ, R>(&g->A, lo[2], hi[2], n, row0, tile);
    double ro = 0.0, m1 = 0.0, rc = 0.0, alpha = 0.0, pcn = 0.0, xn = 0.0, rn = 0.0;
    int iter = 0, stag = 0, msteps = 0, ntrace = 0, info = g->info_in, par = 0, step = 6;
    for (;;) {
        // the matrices' tables are read again in every step: kept across
        // steps they would take the registers that hold the values
        asm volatile("" : "+s"(g), "+s"(c));
        if constexpr (R == 2 && sizeof(T) == 8) asm volatile("" : "+s"(row0));  // and the rows' addresses
        Acc y[R];
        const T *src = rs_glob(c->ex[5]);
        if (step != 6) {
            T *const ex[3] = {rs_glob(step == 2 ? c->ex[0] : c->ex[3]),
                              rs_glob(step == 2 ? c->ex[1] : c->ex[4]),
                              rs_glob(step == 2 ? c->ex[2] : c->ex[5])};
            rs_rows<T, VF, Acc, BSZ, R, 17>(&g->H, dh, tile, lo[0], hi[0], n, row0, ex[0], win, prod, dead, y);
            rs_ahead<VF, Acc, BSZ, R>(&g->G, lo[1], hi[1], n, row0, tile);
#pragma unroll
            for (int q = 0; q < R; q++) {
                const int i = row0 + q * BSZ + tid;
                if (i < n) rs_put(ex[1] + i, dv[q] * (T)y[q]);
            }
            rs_rows<T, VF, Acc, BSZ, R, 4>(&g->G, dg, tile, lo[1], hi[1], n, row0, ex[1], win, prod, dead, y);
            rs_ahead<VA, Acc, BSZ, R>(&g->A, lo[2], hi[2], n, row0, tile);
#pragma unroll
            for (int q = 0; q < R; q++) {
                const int i = row0 + q * BSZ + tid;
                w[q] = (T)y[q];
                if (i < n) rs_put(ex[2] + i, w[q]);
            }
            src = ex[2];
        }
        if (step == 6 && g->zero_start) {
#pragma unroll
            for (int q = 0; q < R; q++) y[q] = 0;
        } else {
            rs_rows<T, VA, Acc, BSZ, R, HA>(&g->A, da, tile, lo[2], hi[2], n, row0, src, win, prod, dead, y);
        }
        rs_ahead<VF, Acc, BSZ, R>(&g->H, lo[0], hi[0], n, row0, tile);
        // the sums the step's reduction carries
        double sm[4] = {0.0, 0.0, 0.0, 0.0};
        int set;
        if (step == 2) {
            set = 1 + par;
#pragma unroll
            for (int q = 0; q < R; q++) {
                v[q] = (T)y[q];
                sm[0] += (double)r0[q] * (double)v[q];
                sm[1] += (double)w[q] * (double)w[q];
                sm[2] += (double)x[q] * (double)x[q];
                sm[3] += (double)r[q] * (double)r[q];
            }
        } else if (step == 5) {
            set = 3 + par;
#pragma unroll
            for (int q = 0; q < R; q++) {
                const T t = (T)y[q];
                sm[0] += (double)t * (double)r[q];
                sm[1] += (double)t * (double)t;
                sm[2] += (double)r0[q] * (double)r[q];
                sm[3] += (double)r0[q] * (double)t;
            }
        } else {
            set = 0;
#pragma unroll
            for (int q = 0; q < R; q++) {
                r[q] = r[q] + (T)(-1.0) * (T)y[q];
                r0[q] = p[q] = r[q];
                sm[0] += (double)r[q] * (double)r[q];
            }
        }
        rs_allsum<BSZ>(sm, rs_glob(c->slots), set, red[set], dead);
        if (rs_uni(*dead)) return;
        if (step == 2) {
            alpha = m1 / sm[0];
            if (g->variant == 2 && !isfinite(alpha)) {
                iter = g->nmax;
                info = 3;
                break;
            }
            pcn = sqrt(sm[1]);
            xn = sqrt(sm[2]);
            rn = sqrt(sm[3]);
            // every reader is done with p, H p and M p, and with the last omega sums
            const T al = (T)alpha, na = (T)(-alpha);
#pragma unroll
            for (int q = 0; q < R; q++) {
                const int i = row0 + q * BSZ + tid;
                x[q] = x[q] + al * w[q];
                r[q] = r[q] + na * v[q];  // s
                if (i < n) {
                    rs_put(rs_glob(c->ex[3]) + i, r[q]);
#pragma unroll
                    for (int e = 0; e < 3; e++) rs_put_bits(rs_glob(c->ex[e]) + i, RsBits<T>::MARK);
                }
            }
            if (tid < RS_K)
                rs_put_bits(rs_glob(c->slots) + ((size_t)(3 + (par ^ 1)) * RS_K + tid) * RS_WGS + blockIdx.x,
                            RsBits<double>::MARK);
            step = 5;
            continue;
        }
        double beta = 0.0, omega = 0.0;
        if (step == 5) {
            omega = sm[0] / sm[1];
            const T om = (T)omega, nom = (T)(-omega);
#pragma unroll
            for (int q = 0; q < R; q++) {
                x[q] = x[q] + om * w[q];
                r[q] = r[q] + nom * (T)y[q];
            }
            // the exits on the lagged ||r||, in FinPass's order
            if (fabs(alpha) * pcn < g->eps * xn) stag++;
            else stag = 0;
            const double prc = rc;
            rc = rn;
            if (c->trace && ntrace < g->trace_cap && blockIdx.x == 0 && tid == 0) c->trace[ntrace] = rc;
            ntrace++;
            if (prc < rc) msteps++;
            else msteps = 0;
            if (msteps >= g->maxmsteps) {
                info = 1;
                break;
            }
            if (stag >= 3) {
                info = 2;
                break;
            }
            if (rc < c->tol * ro) {
                info = 0;
                break;
            }
            const double m2 = m1;
            m1 = sm[2] - omega * sm[3];
            beta = m1 * alpha / (omega * m2);
            if (++iter >= g->nmax) {
                info = 3;
                break;
            }
            const T be = (T)beta, c = (T)(-beta * omega);
#pragma unroll
            for (int q = 0; q < R; q++) {
                const T u = c * v[q] + be * p[q];
                p[q] = u + r[q];
            }
        } else {
            ro = rc = sqrt(sm[0]);
            m1 = ro * ro;
            if (g->nmax <= 0) {
                if (g->nmax == 0) info = 3;
                break;
            }
        }
        // every reader is done with s, H s and M s, and with the pass's alpha sums
#pragma unroll
        for (int q = 0; q < R; q++) {
            const int i = row0 + q * BSZ + tid;
            if (i < n) {
                rs_put(rs_glob(c->ex[0]) + i, p[q]);
                if (step == 5 || !g->zero_start)
#pragma unroll
                    for (int e = 3; e < 6; e++) rs_put_bits(rs_glob(c->ex[e]) + i, RsBits<T>::MARK);
            }
        }
        if (step == 5) {
            if (tid < RS_K)
                rs_put_bits(rs_glob(c->slots) + ((size_t)(1 + par) * RS_K + tid) * RS_WGS + blockIdx.x, RsBits<double>::MARK);
            par ^= 1;
        }
        step = 2;
    }
#pragma unroll
    for (int q = 0; q < R; q++) {
        const int i = row0 + q * BSZ + tid;
        if (i < n && (g->nmax > 0 || g->zero_start)) rs_glob(c->x)[(size_t)i * g->stride] = x[q];
    }
    if (tid == 0) {
        SolveState *o = c->out;
        if (blockIdx.x == 0) {
            o->ro = ro;
            o->rc = rc;
            o->iter = iter;
            o->info = info;
            o->ntrace = ntrace;
        }
        // after the last reduction a workgroup's waves all come here or none
        // does; what they wrote is in place when the launch has ended
        const unsigned q = __hip_atomic_fetch_add(&g->ctl->fin[blockIdx.y], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (q + 1 == gridDim.x) o->done = 1;
    }
}

}  // namespace cm
