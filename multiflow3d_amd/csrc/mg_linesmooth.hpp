// mg_linesmooth.hpp -- the two other smoothers of mgrelax
// (mgsolver.for:403-545): lexicographic Gauss-Seidel (mg_itrsch = 1) and
// ADI line relaxation with the Thomas algorithm (mg_itrsch = 2).
//
// Both update the level's potential in place, in an order whose every
// read sees what the reference's sequential loop would see, so the FP64
// results are the reference's bitwise:
//
// * Lexicographic GS runs its loops k, j, i (i innermost), so cell (i,j,k)
//   reads this sweep's W, S and B neighbours and the previous E, N and T.
//   All cells with i + j + k = s depend only on cells of s - 1 and s + 1:
//   one launch per hyperplane s, in increasing s, every cell of the
//   hyperplane (of every block) one thread.
// * ADI solves j lines in the order (k, i), then i lines in the order
//   (k, j), then k lines in the order (i, j).  A line reads the cross
//   neighbours of the lines before it in its pass (new) and after it
//   (old): with lines indexed (u, v) in loop order, line (u, v) needs
//   (u-1, v) and (u, v-1) finished and (u+1, v), (u, v+1) untouched --
//   the diagonals u + v in increasing order, the lines of a diagonal in
//   parallel.  Blocks are independent within a sweep (a block reads only
//   its own ghosts), so one workgroup per block walks the diagonals of a
//   pass with a barrier between them.  Where the level's blocks fit in
//   LDS, one launch runs the whole sweep there, the RHS staged in LDS too
//   when it fits.  The forward recurrence keeps c(m) in the line's own
//   potential entries (no other line reads them before the diagonal ends)
//   and a(m) in a scratch; the backward pass overwrites c with phi.
//
// The per-cell arithmetic is the reference's: GS as the red-black sweep
// (accumulated aw*W + ae*E + as*S + an*N + ab*B + at*T, then
// (rhs - s)/ap, or times 1/ap in the FP32 inner cycle); TDMA as
// apr = 1/(ap - a_lo*a(m-1)), a(m) = a_hi*apr,
// c(m) = (rhs - x1 - x2 - x3 - x4 - a_lo*c(m-1))*apr with the cross terms
// in the reference's order per pass, phi(m) = c(m) - a(m)*phi(m+1).
#pragma once

#include <hip/hip_runtime.h>

#include "mg_common.hpp"

namespace mf3d {

// One hyperplane i + j + k = s of every block (grid: x over j, y over k in
// 16 x 16 tiles, z = block).
template <typename T, bool VAR, bool RCP>
__global__ __launch_bounds__(256) void k_lex(T *__restrict__ p, const T *__restrict__ rhs,
                                             const T *__restrict__ cx, const T *__restrict__ cy,
                                             const T *__restrict__ cz, const BlockLevel *__restrict__ bls, int s,
                                             const int *__restrict__ done) {
    if (done && *done) return;
    const BlockLevel g = bls[blockIdx.z];
    const int j = blockIdx.x * 16 + (int)(threadIdx.x & 15) + 1;
    const int k = blockIdx.y * 16 + (int)(threadIdx.x >> 4) + 1;
    const int i = s - j - k;
    if (j > g.n1 || k > g.n2 || i < 1 || i > g.n0) return;
    const long long q = gidx(g, i, j, k);
    T aw, ae, as, an, ab, at, ap;
    coefs<T, VAR>(g, cx, cy, cz, q, i, j, k, aw, ae, as, an, ab, at, ap);
    T t = aw * p[q - 1];
    t = t + ae * p[q + 1];
    t = t + as * p[q - g.sy];
    t = t + an * p[q + g.sy];
    t = t + ab * p[q - g.sz];
    t = t + at * p[q + g.sz];
    const T r = rhs[q];
    p[q] = RCP ? (r - t) * (T(1) / ap) : (r - t) / ap;
}

// The cross terms and coefficients of cell (i,j,k) of a line along axis AX:
// t = rhs - the four cross terms in the reference's order for that pass
// (mgsolver.for:450-458, 484-492, 520-528), lo / hi the coefficients
// towards the previous / next cell of the line, ap the diagonal.  The
// potential is read through P at offset lp and the RHS through R at
// offset lr (global memory or LDS); the operator at arena offset q.
template <typename T, bool VAR, int AX>
__device__ __forceinline__ void adi_terms(const BlockLevel &g, const T *P, long long lp, long long sy, long long sz,
                                          const T *R, long long lr, const T *__restrict__ cx,
                                          const T *__restrict__ cy, const T *__restrict__ cz, long long q, int i,
                                          int j, int k, T &t, T &lo, T &hi, T &ap) {
    T aw, ae, as, an, ab, at;
    coefs<T, VAR>(g, cx, cy, cz, q, i, j, k, aw, ae, as, an, ab, at, ap);
    if (AX == 1) {
        lo = as;
        hi = an;
        t = R[lr] - ae * P[lp + 1];
        t = t - aw * P[lp - 1];
        t = t - at * P[lp + sz];
        t = t - ab * P[lp - sz];
    } else if (AX == 0) {
        lo = aw;
        hi = ae;
        t = R[lr] - an * P[lp + sy];
        t = t - as * P[lp - sy];
        t = t - at * P[lp + sz];
        t = t - ab * P[lp - sz];
    } else {
        lo = ab;
        hi = at;
        t = R[lr] - an * P[lp + sy];
        t = t - as * P[lp - sy];
        t = t - ae * P[lp + 1];
        t = t - aw * P[lp - 1];
    }
}

// The lines of one diagonal u + v = d of a pass (lines along AX) over
// block g.  LDS: P is the block's ghosted potential in LDS and A a
// per-thread LDS scratch for a(m) (entry m*blockDim + thread); otherwise P
// is the level arena and A a level-sized scratch at the cells' offsets.
// RLDS: R is the block's RHS in LDS, else the arena.  Each line runs in
// chunks of U cells whose loads are all issued before that part of the
// recurrence.
template <typename T, bool VAR, int AX, bool LDS, bool RLDS>
__device__ __forceinline__ void adi_diagonal(const BlockLevel &g, T *P, const T *R, T *A, const T *__restrict__ cx,
                                             const T *__restrict__ cy, const T *__restrict__ cz, int d) {
    constexpr int U = VAR ? 4 : 8;
    const int nm = AX == 0 ? g.n0 : (AX == 1 ? g.n1 : g.n2);
    const int nu = AX == 1 ? g.n0 : g.n1;
    const int nv = AX == 2 ? g.n0 : g.n2;
    const long long sy = g.sy, sz = g.sz;
    const long long st = AX == 0 ? 1 : (AX == 1 ? sy : sz);  // stride along the line
    const long long pb = LDS ? 0 : g.off, rb = RLDS ? 0 : g.off;
    const int nt = (int)blockDim.x, tid = (int)threadIdx.x;
    const int ulo = max(1, d - nv), uhi = min(nu, d - 1);
    for (int u = ulo + tid; u <= uhi; u += nt) {
        const int v = d - u;
        const int i0 = AX == 1 ? u : (AX == 0 ? 0 : v);
        const int j0 = AX == 1 ? 0 : u;
        const int k0 = AX == 2 ? 0 : v;
        const long long l0 = i0 + sy * j0 + sz * k0;  // the ghost before the line, block-local
        auto aix = [&](int m) -> long long { return LDS ? (long long)m * nt + tid : g.off + l0 + st * m; };
        T a_prev = T(0), c_prev = P[pb + l0];
        for (int m0 = 1; m0 <= nm; m0 += U) {  // forward: a(m) into A, c(m) into the line's own cells
            T tt[U], lo[U], hi[U], ap[U];
#pragma unroll
            for (int e = 0; e < U; ++e) {
                const int m = min(m0 + e, nm);  // past the end: a repeat of the last cell, not used
                const int i = AX == 0 ? m : i0, j = AX == 1 ? m : j0, k = AX == 2 ? m : k0;
                const long long l = l0 + st * m;
                adi_terms<T, VAR, AX>(g, P, pb + l, sy, sz, R, rb + l, cx, cy, cz, g.off + l, i, j, k, tt[e], lo[e],
                                      hi[e], ap[e]);
            }
#pragma unroll
            for (int e = 0; e < U; ++e) {
                if (m0 + e > nm) break;
                const T apr = T(1) / (ap[e] - lo[e] * a_prev);
                a_prev = hi[e] * apr;
                c_prev = (tt[e] - lo[e] * c_prev) * apr;
                A[aix(m0 + e)] = a_prev;
                P[pb + l0 + st * (m0 + e)] = c_prev;
            }
        }
        T nxt = P[pb + l0 + st * (nm + 1)];  // the ghost after the line
        for (int m1 = nm; m1 >= 1; m1 -= U) {  // backward: phi(m) = c(m) - a(m)*phi(m+1)
            T cc[U], aa[U];
#pragma unroll
            for (int e = 0; e < U; ++e) {
                const int m = max(m1 - e, 1);
                cc[e] = P[pb + l0 + st * m];
                aa[e] = A[aix(m)];
            }
#pragma unroll
            for (int e = 0; e < U; ++e) {
                if (m1 - e < 1) break;
                nxt = cc[e] - aa[e] * nxt;
                P[pb + l0 + st * (m1 - e)] = nxt;
            }
        }
    }
}

// One pass of ADI (lines along AX) on a level in global memory, one
// workgroup per block walking the diagonals with a barrier between them;
// sa is a level-sized scratch for a(m).
template <typename T, bool VAR, int AX>
__global__ __launch_bounds__(256) void k_adi(T *__restrict__ p, T *__restrict__ sa, const T *__restrict__ rhs,
                                             const T *__restrict__ cx, const T *__restrict__ cy,
                                             const T *__restrict__ cz, const BlockLevel *__restrict__ bls,
                                             const int *__restrict__ done) {
    if (done && *done) return;
    const BlockLevel g = bls[blockIdx.x];
    const int nu = AX == 1 ? g.n0 : g.n1;
    const int nv = AX == 2 ? g.n0 : g.n2;
    for (int d = 2; d <= nu + nv; ++d) {
        adi_diagonal<T, VAR, AX, false, false>(g, p, rhs, sa, cx, cy, cz, d);
        __syncthreads();
    }
}

// The Thomas coefficients of every line along AX: apr(m) =
// 1/(ap - lo*a(m-1)), a(m) = hi*apr(m), a(0) = 0 -- the reference's
// operations (mgsolver.for:447-449, 481-483, 517-519).  They depend on the
// operator only, so they are built once per coefficient build and the
// sweeps' recurrence keeps no division.  Grid: x over the block's lines in
// 256s, y = block.
template <typename T, bool VAR, int AX>
__global__ __launch_bounds__(256) void k_adi_coef(T *__restrict__ apr_out, T *__restrict__ a_out,
                                                  const T *__restrict__ cx, const T *__restrict__ cy,
                                                  const T *__restrict__ cz, const BlockLevel *__restrict__ bls) {
    const BlockLevel g = bls[blockIdx.y];
    const int nm = AX == 0 ? g.n0 : (AX == 1 ? g.n1 : g.n2);
    const int nu = AX == 1 ? g.n0 : g.n1;
    const int nv = AX == 2 ? g.n0 : g.n2;
    const int t = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (t >= nu * nv) return;
    const int u = t % nu + 1, v = t / nu + 1;
    const int i0 = AX == 1 ? u : (AX == 0 ? 0 : v), j0 = AX == 1 ? 0 : u, k0 = AX == 2 ? 0 : v;
    const long long st = AX == 0 ? 1 : (AX == 1 ? g.sy : g.sz);
    const long long q0 = gidx(g, i0, j0, k0);
    T a_prev = T(0);
    for (int m = 1; m <= nm; ++m) {
        const long long q = q0 + st * m;
        const int i = AX == 0 ? m : i0, j = AX == 1 ? m : j0, k = AX == 2 ? m : k0;
        T aw, ae, as, an, ab, at, ap;
        coefs<T, VAR>(g, cx, cy, cz, q, i, j, k, aw, ae, as, an, ab, at, ap);
        const T lo = AX == 0 ? aw : (AX == 1 ? as : ab), hi = AX == 0 ? ae : (AX == 1 ? an : at);
        const T apr = T(1) / (ap - lo * a_prev);
        a_prev = hi * apr;
        apr_out[q] = apr;
        a_out[q] = a_prev;
    }
}

// Pointers to a level's ADI line coefficients, apr and a per line axis.
template <typename T>
struct AdiCoef {
    const T *apr[3];
    const T *a[3];
};

// Geometry of one diagonal u + v = d of a pass over block g.
template <int AX>
struct AdiDiag {
    int nm, ulo, nl;
    long long st;
    __device__ AdiDiag(const BlockLevel &g, int d) {
        nm = AX == 0 ? g.n0 : (AX == 1 ? g.n1 : g.n2);
        const int nu = AX == 1 ? g.n0 : g.n1, nv = AX == 2 ? g.n0 : g.n2;
        ulo = max(1, d - nv);
        nl = max(0, min(nu, d - 1) - ulo + 1);
        st = AX == 0 ? 1 : (AX == 1 ? g.sy : g.sz);
    }
    // block-local offset of cell m of the diagonal's line ln (m = 0: the
    // ghost before the line), and its (i, j, k)
    __device__ long long cell(const BlockLevel &g, int d, int ln, int m, int &i, int &j, int &k) const {
        const int u = ulo + ln, v = d - u;
        const int i0 = AX == 1 ? u : (AX == 0 ? 0 : v), j0 = AX == 1 ? 0 : u, k0 = AX == 2 ? 0 : v;
        i = AX == 0 ? m : i0;
        j = AX == 1 ? m : j0;
        k = AX == 2 ? m : k0;
        return i + g.sy * j + g.sz * k;
    }
    // entry e = (m-1)*nl + ln of the diagonal's cell list -> (ln, m), without
    // an integer division: a float estimate (e < 2^20, nl <= 1024) corrected
    // by one step either way
    __device__ void split(int e, float rnl, int &ln, int &m) const {
        int q = (int)((float)e * rnl);
        q -= q * nl > e ? 1 : 0;
        q += (q + 1) * nl <= e ? 1 : 0;
        ln = e - q * nl;
        m = q + 1;
    }
};

// The apr and a of diagonal d's cells (entry e = (m-1)*nl + line), up to
// two per thread of a 256-thread workgroup: loaded into registers now,
// stored into LDS later, so the loads fly while the previous diagonal runs.
template <typename T, int AX>
struct AdiPrefetch {
    static constexpr int K = 4;  // entries per thread (the scratch holds at most 256*K)
    T ap[K], aa[K];
    __device__ void load(const BlockLevel &g, const AdiCoef<T> &ac, int d, int dmax) {
        if (d > dmax) return;
        const AdiDiag<AX> D(g, d);
        const float rnl = 1.0f / (float)max(D.nl, 1);
        const T *apr = ac.apr[AX] + g.off, *a = ac.a[AX] + g.off;
#pragma unroll
        for (int q = 0; q < K; ++q) {
            const int e = (int)threadIdx.x + q * 256;
            if (e < D.nl * D.nm) {
                int i, j, k, ln, m;
                D.split(e, rnl, ln, m);
                const int l = (int)D.cell(g, d, ln, m, i, j, k);
                ap[q] = apr[l];
                aa[q] = a[l];
            }
        }
    }
    __device__ void store(const BlockLevel &g, int d, int dmax, T *APR, T *A) const {
        if (d > dmax) return;
        const AdiDiag<AX> D(g, d);
#pragma unroll
        for (int q = 0; q < K; ++q) {
            const int e = (int)threadIdx.x + q * 256;
            if (e < D.nl * D.nm) {
                APR[e] = ap[q];
                A[e] = aa[q];
            }
        }
    }
};

// One pass (lines along AX) of a block in LDS.  Per diagonal:
//   1. every thread: the cross terms t of the diagonal's cells (into the
//      cells themselves in P -- no other line reads them before the
//      diagonal ends) and lo (into LO); and the loads of the next
//      diagonal's apr and a;
//   2. one lane per line: c(m) = (t - lo*c(m-1))*apr(m) into P;
//   3. the same lane: phi(m) = c(m) - a(m)*phi(m+1), backwards;
//   then the next diagonal's apr and a go to the other LDS buffer.
template <typename T, bool VAR, int AX, bool RLDS>
__device__ __forceinline__ void adi_pass_lds(const BlockLevel &g, T *P, const T *R, T *LO, T *APR0, T *A0,
                                             T *APR1, T *A1, const AdiCoef<T> &ac, const T *__restrict__ cx,
                                             const T *__restrict__ cy, const T *__restrict__ cz) {
    const int nu = AX == 1 ? g.n0 : g.n1, nv = AX == 2 ? g.n0 : g.n2;
    const int dmax = nu + nv;
    const long long rb = RLDS ? 0 : g.off;
    const int tid = (int)threadIdx.x;
    AdiPrefetch<T, AX> pf;
    pf.load(g, ac, 2, dmax);
    pf.store(g, 2, dmax, APR0, A0);
    __syncthreads();
    for (int d = 2; d <= dmax; ++d) {
        T *APR = (d & 1) ? APR1 : APR0, *A = (d & 1) ? A1 : A0;
        const AdiDiag<AX> D(g, d);
        const float rnl = 1.0f / (float)max(D.nl, 1);
        for (int e = tid; e < D.nl * D.nm; e += 256) {  // phase 1
            int i, j, k, ln, m;
            D.split(e, rnl, ln, m);
            const int l = (int)D.cell(g, d, ln, m, i, j, k);
            T t, lo, hi, ap;
            adi_terms<T, VAR, AX>(g, P, l, g.sy, g.sz, R, rb + l, cx, cy, cz, g.off + l, i, j, k, t, lo, hi, ap);
            P[l] = t;
            LO[e] = lo;
        }
        pf.load(g, ac, d + 1, dmax);
        __syncthreads();
        constexpr int U = 8;  // full chunks run without branches, the remainder one cell at a time
        for (int ln = tid; ln < D.nl; ln += 256) {  // phases 2 and 3
            int i, j, k;
            const int l0 = (int)D.cell(g, d, ln, 0, i, j, k);  // LDS offsets fit in 32 bits
            const int st = (int)D.st, nm = D.nm, nl = D.nl;
            T c_prev = P[l0];
            int m = 1;
            for (; m + U - 1 <= nm; m += U) {
                const int l = l0 + st * m, e = (m - 1) * nl + ln;
                T lo[U], ap[U], tt[U];
#pragma unroll
                for (int q = 0; q < U; ++q) {
                    lo[q] = LO[e + q * nl];
                    ap[q] = APR[e + q * nl];
                    tt[q] = P[l + q * st];
                }
#pragma unroll
                for (int q = 0; q < U; ++q) {
                    c_prev = (tt[q] - lo[q] * c_prev) * ap[q];
                    P[l + q * st] = c_prev;
                }
            }
            for (; m <= nm; ++m) {
                const int e = (m - 1) * nl + ln;
                c_prev = (P[l0 + st * m] - LO[e] * c_prev) * APR[e];
                P[l0 + st * m] = c_prev;
            }
            T nxt = P[l0 + st * (nm + 1)];
            m = nm;
            for (; m - U + 1 >= 1; m -= U) {
                const int l = l0 + st * m, e = (m - 1) * nl + ln;
                T cc[U], aa[U];
#pragma unroll
                for (int q = 0; q < U; ++q) {
                    cc[q] = P[l - q * st];
                    aa[q] = A[e - q * nl];
                }
#pragma unroll
                for (int q = 0; q < U; ++q) {
                    nxt = cc[q] - aa[q] * nxt;
                    P[l - q * st] = nxt;
                }
            }
            for (; m >= 1; --m) {
                nxt = P[l0 + st * m] - A[(m - 1) * nl + ln] * nxt;
                P[l0 + st * m] = nxt;
            }
        }
        pf.store(g, d + 1, dmax, (d & 1) ? APR0 : APR1, (d & 1) ? A0 : A1);
        __syncthreads();
    }
}

// A whole ADI sweep (j, i, then k lines) of one block per 256-thread
// workgroup with the block in LDS: its ghosted potential, with RLDS its
// RHS, and per-diagonal scratch of 5 arrays of sstride entries (lo, and
// two buffers of apr and a); loaded once, written back once.  Dynamic
// LDS: (cells + (RLDS ? cells : 0) + 5*sstride) entries, cells = the
// largest block's ghosted box; sstride <= 1024 (the prefetch holds 4
// entries per thread).
template <typename T, bool VAR, bool RLDS>
__global__ __launch_bounds__(256) void k_adi_lds(T *__restrict__ p, const T *__restrict__ rhs,
                                                 const T *__restrict__ cx, const T *__restrict__ cy,
                                                 const T *__restrict__ cz, AdiCoef<T> ac,
                                                 const BlockLevel *__restrict__ bls, int cells_max, int sstride,
                                                 const int *__restrict__ done) {
    if (done && *done) return;
    extern __shared__ __align__(16) unsigned char adi_smem[];
    T *P = reinterpret_cast<T *>(adi_smem);
    T *R = P + cells_max;
    T *LO = RLDS ? R + cells_max : R;
    T *APR0 = LO + sstride, *A0 = APR0 + sstride, *APR1 = A0 + sstride, *A1 = APR1 + sstride;
    const BlockLevel g = bls[blockIdx.x];
    const int cells = (int)(g.sz * (g.n2 + 2));
    for (int c = (int)threadIdx.x; c < cells; c += (int)blockDim.x) {
        P[c] = p[g.off + c];
        if (RLDS) R[c] = rhs[g.off + c];
    }
    __syncthreads();
    const T *Rs = RLDS ? (const T *)R : rhs;
    adi_pass_lds<T, VAR, 1, RLDS>(g, P, Rs, LO, APR0, A0, APR1, A1, ac, cx, cy, cz);
    adi_pass_lds<T, VAR, 0, RLDS>(g, P, Rs, LO, APR0, A0, APR1, A1, ac, cx, cy, cz);
    adi_pass_lds<T, VAR, 2, RLDS>(g, P, Rs, LO, APR0, A0, APR1, A1, ac, cx, cy, cz);
    for (int c = (int)threadIdx.x; c < cells; c += (int)blockDim.x) p[g.off + c] = P[c];
}

// ---------------------------------------------------------------------------
// Constant coefficients: the same sweep with little but the recurrences left
// between two diagonals.
//
// What bounds it: the chain of line recurrences, 3 dependent operations a
// cell forward and 2 back on one lane a line (22 and 15 clocks in FP64),
// diagonal after diagonal, and the LDS accesses of the one wave that runs
// it: a wave issues one about every 10 to 20 clocks, however few lanes it
// has.  HBM, LDS bandwidth and the other waves are idle beside it.  So
//   - the lines of a diagonal pass through LDS with a line's cells side by
//     side, two (FP64) or four (FP32) a 16-byte access, and c(m) stays in
//     registers: 2 accesses for 2 cells and direction where k_adi_lds has 6;
//   - the Thomas sequences depend on the line only through the walls it
//     touches: at most 16 classes a pass (low / high end of each cross axis),
//     a table in LDS (k_adi_classes builds it once), not a stream per cell;
//   - every thread keeps its cells' (lane coordinate, place on the line) for
//     the whole pass and moves to the next diagonal by adding one stride; it
//     stores the finished diagonal's phi and forms the next one's cross terms
//     in one phase;
//   - the loop over the diagonals stays rolled, so that its code fits in the
//     instruction cache.
// The reference's 80 blocks of 40 x 10 x 25: 413 -> 173 us a sweep in FP64,
// 370 -> 147 us in FP32.
//
// Lanes run along k in the j pass (whose lines are the shortest) and along j
// in the others; diagonals and every operand are those of the sweep above.
constexpr int ADC_NT = 512, ADC_LINE = 48, ADC_CLS = 16;
static_assert(3 * ADC_CLS <= 64 && ADC_LINE * ADC_LINE <= 5 * ADC_NT, "a wave builds a block's classes; 5 cells a thread reach");

// Entries between two lines of a diagonal in LDS: whole groups of 8 cells, as
// adc_line reads them, and 4 more to spread the banks.
__host__ __device__ inline int adc_stride(int nm) { return (nm + 7) / 8 * 8 + 4; }

// apr(m) and a(m) of every class of lines: tab[block][axis][apr, a][class][m],
// ADC_LINE entries a line.  Class bits: 1 low / 2 high end of the lane axis, 4
// low / 8 high end of the other (adc_axes).  One thread a class and axis.
template <typename T>
__global__ __launch_bounds__(64) void k_adi_classes(T *__restrict__ tab, const BlockLevel *__restrict__ bls) {
    const BlockLevel g = bls[blockIdx.x];
    const int ax = (int)threadIdx.x / ADC_CLS, cls = (int)threadIdx.x % ADC_CLS;
    if (ax >= 3) return;
    const int n[3] = {g.n0, g.n1, g.n2};
    const int ua = ax == 1 ? 2 : 1, va = ax == 2 ? 0 : (ax == 1 ? 0 : 2);  // lane axis, other axis
    T lo[3], hi[3];  // the coefficient below and above along each axis
    for (int d = 0; d < 3; ++d) lo[d] = hi[d] = cconst<T>(g, d);
    if ((cls & 1) && (g.neu & (1 << (2 * ua)))) lo[ua] = T(0);
    if ((cls & 2) && (g.neu & (2 << (2 * ua)))) hi[ua] = T(0);
    if ((cls & 4) && (g.neu & (1 << (2 * va)))) lo[va] = T(0);
    if ((cls & 8) && (g.neu & (2 << (2 * va)))) hi[va] = T(0);
    T *apr_out = tab + ((long long)blockIdx.x * 3 + ax) * 2 * ADC_CLS * ADC_LINE + cls * ADC_LINE;
    T *a_out = apr_out + ADC_CLS * ADC_LINE;
    T a_prev = T(0);
    for (int m = 1; m <= n[ax]; ++m) {
        T l[3] = {lo[0], lo[1], lo[2]}, h[3] = {hi[0], hi[1], hi[2]};
        if (m == 1 && (g.neu & (1 << (2 * ax)))) l[ax] = T(0);
        if (m == n[ax] && (g.neu & (2 << (2 * ax)))) h[ax] = T(0);
        T s = l[0] + h[0];
        s = s + l[1];
        s = s + h[1];
        s = s + l[2];
        s = s + h[2];
        const T ap = -s;
        const T apr = T(1) / (ap - l[ax] * a_prev);
        a_prev = h[ax] * apr;
        apr_out[m - 1] = apr;
        a_out[m - 1] = a_prev;
    }
}

// One line's recurrences on one lane, at most 8 * NCH cells: t(m) from tl, apr
// and a from ta and tb, phi(m) to tl (each 16-byte aligned, 8 * NCH entries;
// past the line's end they are read and written but feed nothing).  cur, nxt:
// the ghosts before and after the line; lo1, lo: the coefficient towards the
// previous cell of the first cell and of the others.
template <typename T, int NCH>
__device__ __forceinline__ void adc_line(T *tl, int nm, const T *ta, const T *tb, T cur, T nxt, T lo1, T lo) {
    constexpr int V = 16 / (int)sizeof(T), N = 8 * NCH, G = 4;  // G cells' operands are read together
    constexpr int NG = N / G;                                    // the last group may lie past the end: left out
    using TV = T __attribute__((ext_vector_type(16 / sizeof(T))));
    const TV *t4 = reinterpret_cast<const TV *>(tl), *p4 = reinterpret_cast<const TV *>(ta),
             *a4 = reinterpret_cast<const TV *>(tb);
    T c[N];
    TV t[3][G / V], x[3][G / V];
    auto ld = [&](const TV *q, int g, TV *r) {
#pragma unroll
        for (int e = 0; e < G / V; ++e) r[e] = q[g * (G / V) + e];
    };
#pragma unroll
    for (int g = 0; g < 2; ++g) {
        ld(t4, g, t[g]);
        ld(p4, g, x[g]);
    }
#pragma unroll
    for (int g = 0; g < NG; ++g) {
        if (g + 2 < NG) {
            ld(t4, g + 2, t[(g + 2) % 3]);
            ld(p4, g + 2, x[(g + 2) % 3]);
        }
        if (g == NG - 1 && g * G >= nm) continue;
#pragma unroll
        for (int e = 0; e < G; ++e) {
            cur = (t[g % 3][e / V][e % V] - (g == 0 && e == 0 ? lo1 : lo) * cur) * x[g % 3][e / V][e % V];
            c[g * G + e] = cur;
        }
    }
    ld(a4, NG - 1, x[(NG - 1) % 3]);
    ld(a4, NG - 2, x[(NG - 2) % 3]);
#pragma unroll
    for (int g = NG - 1; g >= 0; --g) {
        if (g > 1) ld(a4, g - 2, x[(g - 2) % 3]);
        if (g == NG - 1 && g * G >= nm) continue;
        TV o[G / V];
#pragma unroll
        for (int e = G - 1; e >= 0; --e) {
            const T f = c[g * G + e] - x[g % 3][e / V][e % V] * nxt;
            nxt = g < NG - 2 || g * G + e < nm ? f : nxt;  // only cells of the last two groups may lie past the end
            o[e / V][e % V] = nxt;
        }
#pragma unroll
        for (int e = 0; e < G / V; ++e) reinterpret_cast<TV *>(tl)[g * (G / V) + e] = o[e];
    }
}

// One pass (lines along AX) of a block in LDS, K cells a thread.  L: the
// dynamic LDS; at tt the lines of the current diagonal and those of the one
// before, ttn entries each and in turn, S entries a line, lane coordinate u =
// 1 .. at u - 1: t before the recurrences, phi after them; at po the block.
template <typename T, int AX, int K>
__device__ __forceinline__ void adc_pass(const BlockLevel &g, T *L, int tt, int ttn, int po,
                                         const T *__restrict__ rhs, const T *__restrict__ tab) {
    constexpr int NT = ADC_NT;
    const int sy = (int)g.sy, sz = (int)g.sz, tid = (int)threadIdx.x;
    const int nm = AX == 0 ? g.n0 : (AX == 1 ? g.n1 : g.n2), st = AX == 0 ? 1 : (AX == 1 ? sy : sz);
    // the cross terms' first and second axis, in the reference's order
    // (j pass: E, W, T, B; i pass: N, S, T, B; k pass: N, S, E, W)
    const int np = AX == 1 ? g.n0 : g.n1, nq = AX == 2 ? g.n0 : g.n2;
    const int sp = AX == 1 ? 1 : sy, sq = AX == 2 ? 1 : sz;
    const T cp = cconst<T>(g, AX == 1 ? 0 : 1), cq = cconst<T>(g, AX == 2 ? 0 : 2);
    const bool plo = g.neu & (AX == 1 ? kNeuW : kNeuS), phi = g.neu & (AX == 1 ? kNeuE : kNeuN);
    const bool qlo = g.neu & (AX == 2 ? kNeuW : kNeuB), qhi = g.neu & (AX == 2 ? kNeuE : kNeuT);
    // lanes along u, the other cross axis v = d - u
    constexpr bool SEC = AX == 1;
    const int nu = SEC ? nq : np, nv = SEC ? np : nq, su = SEC ? sq : sp, sv = SEC ? sp : sq, dmax = nu + nv;
    const int S = adc_stride(nm);
    T *TA = L, *TB = L + ADC_CLS * ADC_LINE;
    for (int e = tid; e < ADC_CLS * ADC_LINE; e += NT) {
        TA[e] = tab[e];
        TB[e] = tab[ADC_CLS * ADC_LINE + e];
    }
    int uu[K], base[K], tix[K];
    T ulo[K], uhi[K];  // the coefficients below and above along the lane axis
    const T cu = SEC ? cq : cp, cv = SEC ? cp : cq;
    const bool uwl = SEC ? qlo : plo, uwh = SEC ? qhi : phi, vwl = SEC ? plo : qlo, vwh = SEC ? phi : qhi;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int c = tid + k * NT, m = c / nu, u = c - m * nu + 1;
        uu[k] = c < nu * nm ? u : 1 << 20;  // no cell: never on a diagonal
        base[k] = po + u * (su - sv) + (m + 1) * st;
        tix[k] = tt + (u - 1) * S + m;
        ulo[k] = uwl && u == 1 ? T(0) : cu;
        uhi[k] = uwh && u == nu ? T(0) : cu;
    }
    T r[K];
    auto load = [&](int d) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int v = d - uu[k];
            r[k] = v >= 1 && v <= nv ? rhs[base[k] - po + d * sv] : T(0);
        }
    };
    load(2);
    const int lane = tid & 63;
    const T lo = cconst<T>(g, AX), lo1 = (g.neu & (1 << (2 * AX))) ? T(0) : lo;
    __syncthreads();  // the class table, and the pass before
#pragma unroll 1
    for (int d = 2; d <= dmax + 1; ++d) {
        // phi of diagonal d - 1 into the block, the cross terms of diagonal d.
        // All four reads are made together, at entry 0 where there is none.
        const int now = d & 1 ? ttn : 0, then = ttn - now;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int u = uu[k], v = d - u, at = base[k] + d * sv;
            const bool on = v >= 1 && v <= nv, was = v >= 2 && v <= nv + 1;
            const T before = L[was ? tix[k] + then : (on ? at - sv : 0)];  // (u, v-1): just solved, or the ghost
            const T below = L[on ? (u == 1 ? at - su : tix[k] + then - S) : 0];  // (u-1, v)
            const T above = L[on ? at + su : 0], next = L[on ? at + sv : 0];
            const T vlo = vwl && v == 1 ? T(0) : cv, vhi = vwh && v == nv ? T(0) : cv;
            T s;
            if (SEC) {
                s = r[k] - vhi * next;
                s = s - vlo * before;
                s = s - uhi[k] * above;
                s = s - ulo[k] * below;
            } else {
                s = r[k] - uhi[k] * above;
                s = s - ulo[k] * below;
                s = s - vhi * next;
                s = s - vlo * before;
            }
            if (on) L[tix[k] + now] = s;
            if (was) L[at - sv] = before;
        }
        if (d > dmax) break;  // uniform: the last diagonal is stored
        load(d + 1);
        const int u = lane + 1, v = d - u;
        const bool solve = tid < 64 && u <= nu && v >= 1 && v <= nv;
        const int q0 = po + (solve ? u * su + v * sv : 0);
        const T g0 = L[q0], g1 = L[q0 + st * (nm + 1)];  // the line's ghosts, which no pass changes
        __syncthreads();
        if (solve) {
            const int cls = (u == 1 ? 1 : 0) | (u == nu ? 2 : 0) | (v == 1 ? 4 : 0) | (v == nv ? 8 : 0);
            const T *ta = TA + cls * ADC_LINE, *tb = TB + cls * ADC_LINE;
            T *tl = L + tt + now + lane * S;
            switch ((nm + 7) / 8) {
                case 1: adc_line<T, 1>(tl, nm, ta, tb, g0, g1, lo1, lo); break;
                case 2: adc_line<T, 2>(tl, nm, ta, tb, g0, g1, lo1, lo); break;
                case 3: adc_line<T, 3>(tl, nm, ta, tb, g0, g1, lo1, lo); break;
                case 4: adc_line<T, 4>(tl, nm, ta, tb, g0, g1, lo1, lo); break;
                case 5: adc_line<T, 5>(tl, nm, ta, tb, g0, g1, lo1, lo); break;
                default: adc_line<T, 6>(tl, nm, ta, tb, g0, g1, lo1, lo); break;
            }
        }
        __syncthreads();
    }
    __syncthreads();
}

// A whole ADI sweep (j, i, then k lines) of one block per workgroup, constant
// coefficients, every extent at most ADC_LINE and K * ADC_NT cells at most on
// each plane of lane axis x line.  Dynamic LDS: the class tables (2 * ADC_CLS *
// ADC_LINE entries), two diagonals' lines (tt entries each), the block's ghosted potential.
template <typename T, int K>
__global__ __launch_bounds__(ADC_NT) void k_adi_cls(T *__restrict__ p, const T *__restrict__ rhs,
                                                    const T *__restrict__ tab, int tt,
                                                    const BlockLevel *__restrict__ bls,
                                                    const int *__restrict__ done) {
    if (done && *done) return;
    extern __shared__ __align__(16) unsigned char adc_smem[];
    constexpr int t0 = 2 * ADC_CLS * ADC_LINE;
    T *L = reinterpret_cast<T *>(adc_smem), *P = L + t0 + 2 * tt;
    const BlockLevel g = bls[blockIdx.x];
    const int cells = (int)(g.sz * (g.n2 + 2));
    T *pg = p + g.off;
    constexpr int U = 8;
    for (int c0 = (int)threadIdx.x; c0 < cells; c0 += U * ADC_NT) {
        T v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = pg[min(c0 + u * ADC_NT, cells - 1)];
#pragma unroll
        for (int u = 0; u < U; ++u) P[min(c0 + u * ADC_NT, cells - 1)] = v[u];
    }
    const T *tb = tab + (long long)blockIdx.x * 3 * 2 * ADC_CLS * ADC_LINE;
    adc_pass<T, 1, K>(g, L, t0, tt, t0 + 2 * tt, rhs + g.off, tb + 2 * ADC_CLS * ADC_LINE);
    adc_pass<T, 0, K>(g, L, t0, tt, t0 + 2 * tt, rhs + g.off, tb);
    adc_pass<T, 2, K>(g, L, t0, tt, t0 + 2 * tt, rhs + g.off, tb + 4 * ADC_CLS * ADC_LINE);
    for (int c = (int)threadIdx.x; c < cells; c += ADC_NT) pg[c] = P[c];
}

}  // namespace mf3d
