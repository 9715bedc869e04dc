// mg_tail.hpp -- the coarse-level tail of the V-cycle in LDS.
//
// One workgroup per block runs everything from level lt down to the
// coarsest and back up to the post-smoothing of level lt -- sweeps, ghost
// exchange, restriction, prolongation + Neumann copy -- on level arrays held
// in LDS, then writes level lt's potential (with ghosts) to global memory.
// Only for blocks without neighbours or periodic partners (a lone block
// wraps onto itself), where the exchange is local to the workgroup.  Same
// operations, same order and same rounding as the per-level kernels.
//
// What bounds it: one CU runs ~40 dependent phases of a few thousand cells
// each, so a phase costs its LDS accesses (128 bytes a clock for the whole
// workgroup), its instructions (16 waves on 4 SIMDs) and one pass of their
// latency; HBM and the matrix cores play no part.  So the host lists each
// level's cells and ghosts (tail_tables), a visit loads this thread's
// entries into registers while the transfer before it runs -- which leaves a
// sweep no index arithmetic: the addresses and coefficients of the thread's
// cells do not change over the sweeps --, the updates of a thread's cells are
// issued together, and restriction and prolongation share the loads of a
// 2 x 2 x 2 block of cells.  16^3 .. 4^3, V(2,2): 37.0 -> 22.9 us in FP32,
// 43.1 -> 26.3 us in FP64 (a sweep of 16^3: 2.8 -> 1.25 and 3.6 -> 1.5 us).
// Storing the potential by colour (unit-stride accesses) measured no faster
// in FP32 and slower in FP64, 512- and 256-thread workgroups 1.3 and 2 times
// slower.
#pragma once
#include <vector>

#include "mg_coarse.hpp"
#include "mg_common.hpp"

namespace mf3d {

constexpr int TAIL_MAXL = 16;
constexpr int TAIL_NT = 1024;

template <typename T>
struct TailArgs {
    const T *cx[TAIL_MAXL];
    const T *cy[TAIL_MAXL];
    const T *cz[TAIL_MAXL];
};

// c / d for 0 <= c, c * d < 2^32, by the high word of one product with
// m = floor((2^32 - 1) / d) + 1: exactly 2^32/d for a power of two, else
// above 2^32/d by less than 1, so that c*m/2^32 exceeds c/d by less than
// c/2^32 < 1/d and the floors agree.  d = 1 (m would be 2^32) has m = 0.
__host__ __device__ inline unsigned tail_magic(int d) { return d == 1 ? 0u : 0xffffffffu / (unsigned)d + 1u; }
__device__ __forceinline__ int tail_div(int c, unsigned m) { return m ? (int)__umulhi((unsigned)c, m) : c; }

// Products of small non-negative numbers: the 24-bit multiply runs at full
// rate, the 32-bit one at a quarter of it.
__device__ __forceinline__ int mul24(int a, int b) { return __mul24(a, b); }

// One level of one block inside the tail: extents, strides and the LDS
// entries of its potential and RHS (both in the ghosted shape), the length
// of its lists and where they start (tail_tables); m0, m1, mh0, mh1: tail_magic
// of n0, n1, n0/2+1, n1/2+1.
struct TLv {
    int n0, n1, n2, neu, sy, sz, po, ro, cells, ghosts, tab;
    unsigned m0, m1, mh0, mh1;
};

inline TLv tlv_of(int n0, int n1, int n2, int neu) {
    TLv v{};
    v.n0 = n0; v.n1 = n1; v.n2 = n2; v.neu = neu;
    v.sy = n0 + 2;
    v.sz = v.sy * (n1 + 2);
    v.cells = (n0 + 1) / 2 * n1 * n2;
    v.m0 = tail_magic(n0);
    v.m1 = tail_magic(n1);
    v.mh0 = tail_magic(n0 / 2 + 1);
    v.mh1 = tail_magic(n1 / 2 + 1);
    return v;
}

// A list entry no cell or ghost stands behind has bit 31 clear: its loads are
// in bounds, its store is left out.
constexpr unsigned TAIL_VALID = 0x80000000u;

// The lists of one level (host): colour 0, then colour 1, `cells` items each:
// a row (j,k) holds the cells i = i0, i0+2, ... with i0 = 1 + ((1 + j + k +
// colour) & 1) in (n0+1)/2 items: the cell's place in the ghosted array,
// above 16 bits the Neumann faces it touches, TAIL_VALID (not past a row's
// end); then the ghosts: the ghost's place (below 2^16), above 16 bits that of
// the interior cell it stands for (below 2^15) -- wrap on a periodic axis,
// reflect on a Neumann one --, TAIL_VALID.
inline void tail_tables(TLv &v, std::vector<unsigned> &tab) {
    v.tab = (int)tab.size();
    for (int colour = 0; colour < 2; ++colour)
        for (int k = 1; k <= v.n2; ++k)
            for (int j = 1; j <= v.n1; ++j)
                for (int m = 0; m < (v.n0 + 1) / 2; ++m) {
                    const int i = 1 + ((1 + j + k + colour) & 1) + 2 * m;
                    unsigned f = 0;
                    if (i == 1) f |= kNeuW;
                    if (i == v.n0) f |= kNeuE;
                    if (j == 1) f |= kNeuS;
                    if (j == v.n1) f |= kNeuN;
                    if (k == 1) f |= kNeuB;
                    if (k == v.n2) f |= kNeuT;
                    tab.push_back(i > v.n0 ? (unsigned)(1 + v.sy + v.sz)
                                           : (unsigned)(i + v.sy * j + v.sz * k) | ((f & (unsigned)v.neu) << 16) |
                                                 TAIL_VALID);
                }
    const size_t g0 = tab.size();
    auto image = [](int c, int n, bool lo, bool hi) { return c == 0 ? (lo ? 1 : n) : (c == n + 1 ? (hi ? n : 1) : c); };
    for (int k = 0; k <= v.n2 + 1; ++k)
        for (int j = 0; j <= v.n1 + 1; ++j)
            for (int i = 0; i <= v.n0 + 1; ++i) {
                const int si = image(i, v.n0, v.neu & kNeuW, v.neu & kNeuE);
                const int sj = image(j, v.n1, v.neu & kNeuS, v.neu & kNeuN);
                const int sk = image(k, v.n2, v.neu & kNeuB, v.neu & kNeuT);
                if (si != i || sj != j || sk != k)
                    tab.push_back((unsigned)(i + v.sy * j + v.sz * k) |
                                  ((unsigned)(si + v.sy * sj + v.sz * sk) << 16) | TAIL_VALID);
            }
    v.ghosts = (int)(tab.size() - g0);
}

// A thread's share of one level's sweeps: its first KC cells of each colour
// and KG ghosts, read from the table once per visit.  A level with more than
// KC * 1024 items reads the later ones again in every phase.
struct TailLevel {
    static constexpr int KC = 2, KG = 2;
    TLv v;
    const unsigned *tab;
    unsigned cell[2][KC], gh[KG];
    __device__ __forceinline__ TailLevel(const TLv &lv, const unsigned *__restrict__ t) : v(lv), tab(t + lv.tab) {
#pragma unroll
        for (int m = 0; m < KC; ++m) {
            cell[0][m] = item(m, 0, v.cells, (unsigned)(1 + v.sy + v.sz));
            cell[1][m] = item(m, v.cells, v.cells, (unsigned)(1 + v.sy + v.sz));
        }
#pragma unroll
        for (int m = 0; m < KG; ++m) gh[m] = item(m, 2 * v.cells, v.ghosts, 0u);
    }
    // this thread's m-th entry of the list of n entries at `first`
    __device__ __forceinline__ unsigned item(int m, int first, int n, unsigned none) const {
        const int c = (int)threadIdx.x + m * TAIL_NT;
        const unsigned e = tab[first + min(c, n - 1)];
        return c < n ? e : none;
    }
};

// The neighbour coefficients of a cell: constants with the Neumann zeros of
// its face flags, or the level's face arrays.
template <typename T, bool VAR>
__device__ __forceinline__ void tail_coefs(T c0, T c1, T c2, unsigned f, const T *__restrict__ cx,
                                           const T *__restrict__ cy, const T *__restrict__ cz, long long q,
                                           long long sy, long long sz, T *a) {
    if (VAR) {
        a[0] = cx[q];
        a[1] = cx[q + 1];
        a[2] = cy[q];
        a[3] = cy[q + sy];
        a[4] = cz[q];
        a[5] = cz[q + sz];
    } else {
        a[0] = (f & kNeuW) ? T(0) : c0;
        a[1] = (f & kNeuE) ? T(0) : c0;
        a[2] = (f & kNeuS) ? T(0) : c1;
        a[3] = (f & kNeuN) ? T(0) : c1;
        a[4] = (f & kNeuB) ? T(0) : c2;
        a[5] = (f & kNeuT) ? T(0) : c2;
    }
}

template <typename T>
__device__ __forceinline__ T tail_ap(const T *a) {
    T s = a[0] + a[1];
    s = s + a[2];
    s = s + a[3];
    s = s + a[4];
    s = s + a[5];
    return -s;
}

// One colour: U cells of this thread at a time, all their loads before the
// first store (cells of one colour do not read each other) and none of
// them behind a branch, so that they are in flight together.
template <typename T, bool VAR, int U>
__device__ __forceinline__ void tail_update(T *P, const T *R, const TLv &v, const BlockLevel &g, T c0, T c1, T c2,
                                            const unsigned *e, const T *cx, const T *cy, const T *cz) {
    T out[U], w[U][6], r[U];
#pragma unroll
    for (int m = 0; m < U; ++m) {
        const int q = (int)(e[m] & 0xffffu);
        w[m][0] = P[q - 1];
        w[m][1] = P[q + 1];
        w[m][2] = P[q - v.sy];
        w[m][3] = P[q + v.sy];
        w[m][4] = P[q - v.sz];
        w[m][5] = P[q + v.sz];
        r[m] = R[q];
    }
#pragma unroll
    for (int m = 0; m < U; ++m) {
        T a[6];
        tail_coefs<T, VAR>(c0, c1, c2, e[m] >> 16, cx, cy, cz, g.off + (e[m] & 0xffffu), v.sy, v.sz, a);
        const T ap = tail_ap<T>(a);
        T s = a[0] * w[m][0];
        s = madd(s, a[1], w[m][1]);
        s = madd(s, a[2], w[m][2]);
        s = madd(s, a[3], w[m][3]);
        s = madd(s, a[4], w[m][4]);
        s = madd(s, a[5], w[m][5]);
        // FP64 divides as the reference does; the FP32 inner cycle multiplies by 1/ap
        out[m] = sizeof(T) == 8 ? (r[m] - s) / ap : (r[m] - s) * (T(1) / ap);
    }
#pragma unroll
    for (int m = 0; m < U; ++m)
        if (e[m] & TAIL_VALID) P[e[m] & 0xffffu] = out[m];
}

template <typename T, bool VAR>
__device__ __forceinline__ void tail_colour(T *sm, const TailLevel &L, const BlockLevel &g, T c0, T c1, T c2,
                                            const T *cx, const T *cy, const T *cz, int colour) {
    constexpr int KC = TailLevel::KC;
    T *P = sm + L.v.po;
    const T *R = sm + L.v.ro;
    const int w0 = __builtin_amdgcn_readfirstlane((int)threadIdx.x);  // uniform: this wave's items in the list
    if (w0 + TAIL_NT < L.v.cells) tail_update<T, VAR, KC>(P, R, L.v, g, c0, c1, c2, L.cell[colour], cx, cy, cz);
    else if (w0 < L.v.cells) tail_update<T, VAR, 1>(P, R, L.v, g, c0, c1, c2, L.cell[colour], cx, cy, cz);
    for (int c = KC; w0 + c * TAIL_NT < L.v.cells; ++c) {
        const unsigned x = L.item(c, colour * L.v.cells, L.v.cells, (unsigned)(1 + L.v.sy + L.v.sz));
        tail_update<T, VAR, 1>(P, R, L.v, g, c0, c1, c2, &x, cx, cy, cz);
    }
}

// Every ghost takes the interior cell it stands for.  Sources are interior
// cells, so the order is free.
template <typename T>
__device__ __forceinline__ void tail_exchange(T *sm, const TailLevel &L) {
    constexpr int KG = TailLevel::KG;
    T *P = sm + L.v.po;
    const int w0 = __builtin_amdgcn_readfirstlane((int)threadIdx.x);
    if (w0 >= L.v.ghosts) return;
    T g[KG];
#pragma unroll
    for (int m = 0; m < KG; ++m) g[m] = P[(L.gh[m] >> 16) & 0x7fffu];
#pragma unroll
    for (int m = 0; m < KG; ++m)
        if (L.gh[m] & TAIL_VALID) P[L.gh[m] & 0xffffu] = g[m];
    for (int t = (int)threadIdx.x + KG * TAIL_NT; t < L.v.ghosts; t += TAIL_NT) {
        const unsigned x = L.tab[2 * L.v.cells + t];
        P[x & 0xffffu] = P[(x >> 16) & 0x7fffu];
    }
}

// Residual of the fine level restricted into the coarse RHS (:688-751); the
// coarse potential is zeroed including its ghosts (:650-657).  A thread
// takes a coarse cell: its eight children and the 24 cells around them are
// loaded once, two planes of children at a time.
template <typename T, bool VAR>
__device__ __forceinline__ void tail_restrict(T *sm, const TLv &vf, const BlockLevel &gf, const TLv &vc,
                                              const T *cx, const T *cy, const T *cz) {
    const T *P = sm + vf.po;
    const T *R = sm + vf.ro;
    T *RC = sm + vc.ro;
    T *PC = sm + vc.po;
    const int MC = vc.sz * (vc.n2 + 2);
    for (int c = threadIdx.x; c < MC; c += TAIL_NT) PC[c] = T(0);
    const int N = mul24(vc.n0, mul24(vc.n1, vc.n2));
    const T c0 = cconst<T>(gf, 0), c1 = cconst<T>(gf, 1), c2 = cconst<T>(gf, 2);
    for (int c = threadIdx.x; c < N; c += TAIL_NT) {
        const int r = tail_div(c, vc.m0), kk = tail_div(r, vc.m1);
        const int i = c - mul24(r, vc.n0) + 1, j = r - mul24(kk, vc.n1) + 1, k = kk + 1;
        unsigned fl[2][3];  // Neumann faces of the children's positions along each axis
        fl[0][0] = i == 1 ? kNeuW : 0;
        fl[1][0] = i == vc.n0 ? kNeuE : 0;
        fl[0][1] = j == 1 ? kNeuS : 0;
        fl[1][1] = j == vc.n1 ? kNeuN : 0;
        fl[0][2] = k == 1 ? kNeuB : 0;
        fl[1][2] = k == vc.n2 ? kNeuT : 0;
        const int q0 = (2 * i - 1) + mul24(vf.sy, 2 * j - 1) + mul24(vf.sz, 2 * k - 1);
        T acc = T(0);
        // children in the order (0,0,0) (1,0,0) (0,1,0) (1,1,0) (0,0,1) (1,0,1) (0,1,1) (1,1,1)
#pragma unroll
        for (int dz = 0; dz < 2; ++dz) {
            const int qz = q0 + dz * vf.sz;
            T w[4][4], lo[2][2], hi[2][2];  // this plane with its x and y neighbours; the planes below and above
#pragma unroll
            for (int y = 0; y < 4; ++y)
#pragma unroll
                for (int x = 0; x < 4; ++x)
                    if ((y == 1 || y == 2) || (x == 1 || x == 2)) w[y][x] = P[qz + (x - 1) + vf.sy * (y - 1)];
#pragma unroll
            for (int y = 0; y < 2; ++y)
#pragma unroll
                for (int x = 0; x < 2; ++x) {
                    lo[y][x] = P[qz + x + vf.sy * y - vf.sz];
                    hi[y][x] = P[qz + x + vf.sy * y + vf.sz];
                }
#pragma unroll
            for (int y = 0; y < 2; ++y)
#pragma unroll
                for (int x = 0; x < 2; ++x) {
                    const int q = qz + x + vf.sy * y;
                    T a[6];
                    tail_coefs<T, VAR>(c0, c1, c2, (fl[x][0] | fl[y][1] | fl[dz][2]) & (unsigned)vf.neu, cx, cy,
                                       cz, gf.off + q, vf.sy, vf.sz, a);
                    const T ap = tail_ap<T>(a);
                    T s = a[0] * w[y + 1][x];
                    s = s + a[1] * w[y + 1][x + 2];
                    s = s + a[2] * w[y][x + 1];
                    s = s + a[3] * w[y + 2][x + 1];
                    s = s + a[4] * lo[y][x];
                    s = s + a[5] * hi[y][x];
                    s = s + ap * w[y + 1][x + 1];
                    const T res = R[q] - s;
                    acc = (dz == 0 && y == 0 && x == 0) ? res : acc + res;
                }
        }
        RC[i + mul24(vc.sy, j) + mul24(vc.sz, k)] = T(0.125) * acc;
    }
}

// Prolongation + correction of every fine cell including ghosts, then the
// Neumann copy (mgsolver.for:823-902).  A thread takes an octet of fine cells
// (2m, 2m+1) on each axis, which read the same eight coarse values; a ghost
// on a Neumann face and the cell it reflects lie in one octet (a level with
// a coarser one has even extents), so the copy is made in registers.
template <typename T>
__device__ __forceinline__ void tail_prolong(T *sm, const TLv &vf, const TLv &vc) {
    T *PF = sm + vf.po;
    const T *PC = sm + vc.po;
    const int a = (vf.n0 >> 1) + 1, b = (vf.n1 >> 1) + 1, d = (vf.n2 >> 1) + 1, M = a * b * d;
    for (int c = threadIdx.x; c < M; c += TAIL_NT) {
        const int r = tail_div(c, vf.mh0), mz = tail_div(r, vf.mh1), mx = c - mul24(r, a), my = r - mul24(mz, b);
        T *F = PF + 2 * (mx + mul24(vf.sy, my) + mul24(vf.sz, mz));
        const T *E = PC + mx + mul24(vc.sy, my) + mul24(vc.sz, mz);
        T e[2][2][2], v[2][2][2];
#pragma unroll
        for (int z = 0; z < 2; ++z)
#pragma unroll
            for (int y = 0; y < 2; ++y)
#pragma unroll
                for (int x = 0; x < 2; ++x) {
                    e[z][y][x] = E[x + vc.sy * y + vc.sz * z];
                    v[z][y][x] = F[x + vf.sy * y + vf.sz * z];
                }
#pragma unroll
        for (int z = 0; z < 2; ++z)
#pragma unroll
            for (int y = 0; y < 2; ++y)
#pragma unroll
                for (int x = 0; x < 2; ++x) {
                    const T wi0 = x ? T(1) : T(3), wi1 = x ? T(3) : T(1);
                    const T wj0 = y ? T(1) : T(3), wj1 = y ? T(3) : T(1);
                    const T wk0 = z ? T(1) : T(3), wk1 = z ? T(3) : T(1);
                    T s = (wi0 * wj0 * wk0) * e[0][0][0];
                    s = s + (wi0 * wj1 * wk0) * e[0][1][0];
                    s = s + (wi0 * wj0 * wk1) * e[1][0][0];
                    s = s + (wi0 * wj1 * wk1) * e[1][1][0];
                    s = s + (wi1 * wj0 * wk0) * e[0][0][1];
                    s = s + (wi1 * wj1 * wk0) * e[0][1][1];
                    s = s + (wi1 * wj0 * wk1) * e[1][0][1];
                    s = s + (wi1 * wj1 * wk1) * e[1][1][1];
                    v[z][y][x] = v[z][y][x] + s / T(64);
                }
        // a Neumann ghost takes the value of the cell it reflects, axis by axis
        const bool w = mx == 0 && (vf.neu & kNeuW), ea = mx == a - 1 && (vf.neu & kNeuE);
        const bool s = my == 0 && (vf.neu & kNeuS), n = my == b - 1 && (vf.neu & kNeuN);
        const bool bo = mz == 0 && (vf.neu & kNeuB), t = mz == d - 1 && (vf.neu & kNeuT);
#pragma unroll
        for (int z = 0; z < 2; ++z)
#pragma unroll
            for (int y = 0; y < 2; ++y) {
                v[z][y][0] = w ? v[z][y][1] : v[z][y][0];
                v[z][y][1] = ea ? v[z][y][0] : v[z][y][1];
            }
#pragma unroll
        for (int z = 0; z < 2; ++z)
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                v[z][0][x] = s ? v[z][1][x] : v[z][0][x];
                v[z][1][x] = n ? v[z][0][x] : v[z][1][x];
            }
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                v[0][y][x] = bo ? v[1][y][x] : v[0][y][x];
                v[1][y][x] = t ? v[0][y][x] : v[1][y][x];
            }
#pragma unroll
        for (int z = 0; z < 2; ++z)
#pragma unroll
            for (int y = 0; y < 2; ++y)
#pragma unroll
                for (int x = 0; x < 2; ++x) F[x + vf.sy * y + vf.sz * z] = v[z][y][x];
    }
}

template <typename T, bool VAR>
__device__ __forceinline__ void tail_sweeps(T *sm, const TailLevel &L, const BlockLevel &g, const T *cx, const T *cy,
                                            const T *cz, int n) {
    const T c0 = cconst<T>(g, 0), c1 = cconst<T>(g, 1), c2 = cconst<T>(g, 2);
    for (int s = 0; s < n; ++s) {
        tail_colour<T, VAR>(sm, L, g, c0, c1, c2, cx, cy, cz, 1);
        __syncthreads();
        tail_colour<T, VAR>(sm, L, g, c0, c1, c2, cx, cy, cz, 0);
        __syncthreads();
        tail_exchange<T>(sm, L);
        __syncthreads();
    }
}

// FP64 direct solve of the coarsest level inside the tail (one block): the
// level's RHS in cell order (i fastest) widened into sb, phi = Minv * rhs
// by one wave per row (coarse_row, as k_coarse_solve computes it), then the
// ghost fill.
template <typename T>
__device__ __forceinline__ void tail_direct(T *sm, const TailLevel &L, const double *__restrict__ cinv, int nc,
                                            double *sb) {
    const TLv &v = L.v;
    for (int c = threadIdx.x; c < nc; c += TAIL_NT) {
        const int r = tail_div(c, v.m0), kk = tail_div(r, v.m1);
        sb[c] = (double)sm[v.ro + (c - r * v.n0 + 1) + v.sy * (r - kk * v.n1 + 1) + v.sz * (kk + 1)];
    }
    __syncthreads();
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int c = wave; c < nc; c += TAIL_NT / 64) {
        const double s = coarse_row(cinv + (long long)c * nc, sb, nc, lane);
        if (lane == 0) {
            const int r = tail_div(c, v.m0), kk = tail_div(r, v.m1);
            sm[v.po + (c - r * v.n0 + 1) + v.sy * (r - kk * v.n1 + 1) + v.sz * (kk + 1)] = (T)s;
        }
    }
    __syncthreads();
    tail_exchange<T>(sm, L);
    __syncthreads();
}

// The reference's sweeps of the coarsest level computed in FP64 inside an
// FP32 tail: the level's RHS widened into sd (after the potential), the potential from zero, n sweeps with FP64 coefficients
// (cx..cz: the level's FP64 face coefficients under VAR), then every
// entry, ghosts included, narrowed back.
template <typename T, bool VAR>
__device__ __forceinline__ void tail_sweeps_fp64(T *sm, const TailLevel &L, const BlockLevel &g, const double *cx,
                                                 const double *cy, const double *cz, int n, double *sd) {
    const TLv &v = L.v;
    TailLevel D = L;
    D.v.po = 0;
    const int M = v.sz * (v.n2 + 2);
    D.v.ro = M;
    for (int c = threadIdx.x; c < M; c += TAIL_NT) {
        sd[c] = 0.0;
        sd[M + c] = (double)sm[v.ro + c];
    }
    __syncthreads();
    tail_sweeps<double, VAR>(sd, D, g, cx, cy, cz, n);
    for (int c = threadIdx.x; c < M; c += TAIL_NT) sm[v.po + c] = (T)sd[c];
    __syncthreads();
}

// cinv (nullptr: sweeps): the coarsest level's inverse operator, nc cells;
// c64: the coarsest level's sweeps in FP64, with its FP64 coefficients
// c64c[0..2] under VAR.  Their FP64 staging goes after the level arrays in
// LDS.
template <typename T>
struct TailC64 {
    int on;
    const double *cx, *cy, *cz;
};

template <typename T, bool VAR>
__global__ __launch_bounds__(TAIL_NT) void k_tail(const BlockLevel *__restrict__ tl, const TLv *__restrict__ lv,
                                                  const unsigned *__restrict__ tab, int nb, int nlev,
                                                  const T *__restrict__ rhs_in,
                                                  const T *__restrict__ phi_in, T *__restrict__ phi_out,
                                                  TailArgs<T> co, int nu_pre, int nu_post,
                                                  const double *__restrict__ cinv, int nc, TailC64<T> c64,
                                                  const int *__restrict__ done) {
    if (done && *done) return;
    extern __shared__ unsigned char smem_raw[];
    T *sm = reinterpret_cast<T *>(smem_raw);
    const int b = blockIdx.x;
    const long long goff = tl[b].off;
    {
        const int M = lv[b].sz * (lv[b].n2 + 2), po = lv[b].po, ro = lv[b].ro;
        constexpr int KL = 6;
        for (int c0 = (int)threadIdx.x; c0 < M; c0 += KL * TAIL_NT) {
            T r[KL], p[KL];
#pragma unroll
            for (int m = 0; m < KL; ++m) {  // the last entry again past the end
                r[m] = rhs_in[goff + min(c0 + m * TAIL_NT, M - 1)];
                p[m] = phi_in ? phi_in[goff + min(c0 + m * TAIL_NT, M - 1)] : T(0);
            }
#pragma unroll
            for (int m = 0; m < KL; ++m) {
                sm[ro + min(c0 + m * TAIL_NT, M - 1)] = r[m];
                sm[po + min(c0 + m * TAIL_NT, M - 1)] = p[m];
            }
        }
    }
    for (int li = 0; li < nlev; ++li) {
        const TailLevel L(lv[li * nb + b], tab);
        if (li > 0)
            tail_restrict<T, VAR>(sm, lv[(li - 1) * nb + b], tl[(li - 1) * nb + b], L.v, co.cx[li - 1], co.cy[li - 1],
                                  co.cz[li - 1]);
        __syncthreads();
        if ((cinv || c64.on) && li == nlev - 1) {
            const int end = L.v.ro + L.v.sz * (L.v.n2 + 2);  // the last level's RHS ends the T arrays
            double *sb = reinterpret_cast<double *>(smem_raw + ((size_t)end * sizeof(T) + 7) / 8 * 8);
            if (cinv) tail_direct<T>(sm, L, cinv, nc, sb);
            else tail_sweeps_fp64<T, VAR>(sm, L, tl[li * nb + b], c64.cx, c64.cy, c64.cz, nu_pre + nu_post, sb);
        } else {
            tail_sweeps<T, VAR>(sm, L, tl[li * nb + b], co.cx[li], co.cy[li], co.cz[li],
                                nu_pre + (li == nlev - 1 ? nu_post : 0));
        }
    }
    for (int li = nlev - 2; li >= 0; --li) {
        const TailLevel L(lv[li * nb + b], tab);
        tail_prolong<T>(sm, L.v, lv[(li + 1) * nb + b]);
        __syncthreads();
        tail_sweeps<T, VAR>(sm, L, tl[li * nb + b], co.cx[li], co.cy[li], co.cz[li], nu_post);
    }
    const int M = lv[b].sz * (lv[b].n2 + 2), po = lv[b].po;
    for (int c = threadIdx.x; c < M; c += TAIL_NT) phi_out[goff + c] = sm[po + c];
}

}  // namespace mf3d
