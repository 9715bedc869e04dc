// mg_leg.hpp -- one leg of the V-cycle on a level of a lone block or of a
// conforming grid of blocks in one pass over memory: down (two red-black sweeps from zero, the residual and its
// restriction) and up (prolongation and two red-black sweeps).
//
// What the sweeps, restriction and prolongation of a leg cost apart is their
// passes over memory (5 and 6 fields in, 3 out and a quarter of one more) and,
// on small levels, their launches.  Here a leg reads the RHS (and the
// potential and the coarse potential) once and writes the potential (and
// the coarse RHS) once.
//
// A workgroup owns a tile of columns and marches over planes.  A thread owns
// two neighbouring columns of one row, the cells (i, i+1) with i odd, and
// keeps their potential and RHS of the last planes in registers.  At step c
// it updates, of the column whose turn it is, red plane c of the first
// sweep, black plane c-1, red plane c-2 of the second sweep and black plane
// c-3: four updates of one column, because the colour of a column's cells
// alternates with the plane.  Labelling the columns by their parity instead
// of their place -- A: i + j even, B: i + j odd -- makes that column the same
// label in every thread, A on odd planes c and B on even ones, so with the
// march unrolled nothing selects at run time.  An update's z neighbours and one
// x neighbour are the thread's own registers, the other x neighbour is a
// neighbouring lane's (a DPP move), the two y neighbours come through LDS, where
// each update leaves its value.  An update reads there only what the step
// before wrote, so every buffer has two halves used in turn and a step
// has one barrier.
//
// Tiles overlap: cells in a ring around the stored ones are computed by the
// neighbouring workgroups too, from the same inputs, one cell less on
// every half sweep.  Beyond a periodic face the ring holds the cells it wraps
// to, beyond a face to another block (MB) that block's cells.  The reference refreshes a block's ghosts only after a whole
// sweep (mgsolver.for:610-611), so across such a face a black update reads
// the red value from before the sweep: updates keep the value they replace
// (o1, o2), and a neighbour across the face takes that one.  Beyond a wall
// the coefficient is zero and the ring's values, finite, do not matter.
// Same operands, same order as k_rbs, k_restrict and k_prolong: bitwise
// their results.
//
// A grid of blocks needs the ghosts of its potential only after the up leg, by the
// exchange; apart, each sweep was followed by one.  Eight blocks of 96 to 192
// cells a side (26.2 million cells), FP32: down 201 us and two exchanges of 13.5
// against 107, up 216 and two against 116 and one.
//
// Measured on the level of 256^3 cells, sweeps and transfers apart against the
// leg: FP32 down 125 us (47 + 50 + 28) against 69, up 127 (27 + 2 x 50) against 82;
// FP64 down 264 against 140, up 310 against 180.  HBM traffic is 1.12 to 1.32
// times what a leg has to move and takes half the time; the bound is a step's
// serial chain, 2700 clocks in FP32 for about 120 vector and 80 scalar
// instructions a wavefront between two barriers, the four updates
// depending on each other.  Small levels: a fixed 3 us and 1 us a step, and the
// instruction cache, cold in every launch, so rare cases (the planes
// beside the z faces) take a divisor from LDS instead of code of their own: 64^3
// FP32 13.0 a leg against 16.3 in two or three launches.
//
// Variable coefficients (FP32): a cell's faces and 1 / ap are loaded and formed
// once, two planes ahead, and stay in registers for its two or three uses;
// apart, each sweep and the restriction read the three face arrays again.  On
// 384^3 cells: down 1221 us (420 + 494 + 307) against 396, up 1096 (108 + 2 x
// 494) against 457, of which the bytes a leg moves, 20.5 and 24.5 a cell, take
// 235 and 281 at 4.93 TB/s.
#pragma once
#include "mg_common.hpp"
#include "mg_sweep.hpp"

namespace mf3d {

// Rows and pairs of columns (32) of a workgroup; the ring is 4 rows, and 6
// columns: the outermost pair has no lane beside it to take coarse values from.
// FP64 has 24 rows, 168 registers a thread; at 32 rows, 128, it spills.  Levels
// too small to fill the card take LEG_NY_SMALL rows.
constexpr int LEG_TX = 52, LEG_NY_SMALL = 16;
template <typename T>
constexpr int leg_ny(bool var) { return var ? 24 : (sizeof(T) == 4 ? 32 : 24); }
// Variable coefficients are marched in FP32 only: in FP64 a thread's
// coefficients of the four planes would not fit in registers.
template <typename T, bool VAR>
constexpr bool leg_march() { return sizeof(T) == 4 || !VAR; }

template <int CTRL>
__device__ __forceinline__ int dpp_i(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true);
}
// The value of lane - 1 (from_left) and lane + 1 (from_right); 0 past the wavefront's ends.
template <int CTRL>
__device__ __forceinline__ float dpp(float v) { return __builtin_bit_cast(float, dpp_i<CTRL>(__builtin_bit_cast(int, v))); }
template <int CTRL>
__device__ __forceinline__ double dpp(double v) {
    const uint2 b = __builtin_bit_cast(uint2, v);
    return __builtin_bit_cast(double, uint2{(unsigned)dpp_i<CTRL>((int)b.x), (unsigned)dpp_i<CTRL>((int)b.y)});
}
template <typename T> __device__ __forceinline__ T from_left(T v) { return dpp<0x138>(v); }
template <typename T> __device__ __forceinline__ T from_right(T v) { return dpp<0x130>(v); }

// Planes in flight: what the registers leave room for.
template <typename T, bool UP>
constexpr int leg_depth(bool var) { return var ? 2 : (sizeof(T) == 8 && UP ? 1 : 3); }

// Two neighbouring entries of a field, at a byte offset of any alignment of
// one entry.
template <typename T> struct Pair { T l, r; };
template <typename T> __device__ __forceinline__ Pair<T> bload2(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff);
template <> __device__ __forceinline__ Pair<float> bload2<float>(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    return __builtin_bit_cast(Pair<float>, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
}
template <> __device__ __forceinline__ Pair<double> bload2<double>(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    return __builtin_bit_cast(Pair<double>, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}
template <typename T> __device__ __forceinline__ void bstore2(__amdgpu_buffer_rsrc_t r, Pair<T> v, uint32_t voff, uint32_t soff);
template <> __device__ __forceinline__ void bstore2<float>(__amdgpu_buffer_rsrc_t r, Pair<float> v, uint32_t voff, uint32_t soff) {
    using V = decltype(__builtin_amdgcn_raw_buffer_load_b64(r, 0, 0, 0));
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(V, v), r, voff, soff, 0);
}
template <> __device__ __forceinline__ void bstore2<double>(__amdgpu_buffer_rsrc_t r, Pair<double> v, uint32_t voff, uint32_t soff) {
    using V = decltype(__builtin_amdgcn_raw_buffer_load_b128(r, 0, 0, 0));
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(V, v), r, voff, soff, 0);
}

// The cell 1..n that coordinate v stands for: around a periodic axis, or
// the nearest one beyond walls.
__device__ __forceinline__ int leg_map(int v, int n, bool per) {
    if (!per) return v < 1 ? 1 : (v > n ? n : v);
    while (v < 1) v += n;
    while (v > n) v -= n;
    return v;
}

// The blocks that hold the cells around a block, by offset (ox, oy, oz) at
// (oz + 1) * 9 + (oy + 1) * 3 + ox + 1; an offset beyond a wall counts as 0.
struct LegBlocks {
    int nb[27];
};

// The face coefficients of a variable-coefficient level (FP32).
template <typename T> struct LegFaces {
    const T *__restrict__ x, *__restrict__ y, *__restrict__ z;
};

// LDS: a thread's divisors on the planes beside the z faces (four), then
// halves of 32 * (rows + 2) entries: up: the old black, red 1, black 1, red 2
// planes (two each) and, where y is periodic, the reds they replace; down: red
// 1, black 1 (two each), red 2 (three), black 2 (two), then the replaced reds.
template <typename T>
constexpr int leg_lds(bool up, bool yper, int ny, bool var) {
    return 32 * (int)sizeof(T) *
           ((var ? 0 : 4) * ny + (ny + 2) * (up ? 8 + (yper ? 4 : 0) : 9 + (yper ? 2 : 0)));
}

template <typename T, bool UP, int NY, bool VAR = false, bool MB = false>
__global__ __launch_bounds__(32 * NY) void k_leg(const T *__restrict__ pin, T *__restrict__ pout,
                                                const T *__restrict__ rhs, LegFaces<T> faces, uint32_t bytes,
                                                const BlockLevel *__restrict__ bls, const Tile *__restrict__ tiles,
                                                const int *__restrict__ done, const T *__restrict__ phic,
                                                T *__restrict__ rhsc, uint32_t cbytes,
                                                const BlockLevel *__restrict__ blc,
                                                const LegBlocks *__restrict__ around) {
    const int stop = done ? *done : 0;  // awaited with the tile
    extern __shared__ __align__(16) unsigned char leg_smem[];
    T *face = reinterpret_cast<T *>(leg_smem), *sm = face + (VAR ? 0 : 4) * 32 * NY;
    constexpr uint32_t W = sizeof(T);
    constexpr int LEG_NT = 32 * NY, LEG_TY = NY - 8, LEG_ROW = 32 * (NY + 2);
    constexpr int NS = 6;  // planes in the registers' rings, the unroll
    const Tile t = tiles[blockIdx.x];
    const BlockLevel g = bls[t.b], gc = blc[t.b];
    if (stop) return;
    const auto rs_in = make_rsrc(pin, bytes), rs_f = make_rsrc(rhs, bytes), rs_out = make_rsrc(pout, bytes);
    const auto rs_c = make_rsrc(UP ? phic : rhsc, cbytes);
    // A wavefront takes two rows: down, whose restriction adds them, an odd row
    // and the even one after it; up two rows of one parity, whose prolongation
    // weights are then scalars.
    const int tid = (int)threadIdx.x;
    const int row = UP ? (tid >> 7) * 4 + ((tid >> 6) & 1) + ((tid >> 5) & 1) * 2 : tid >> 5;
    const int pair = (row & 1) ? 31 - (tid & 31) : (tid & 31);
    const int i = t.x0 - 6 + 2 * pair, j = t.y0 - 4 + row;  // i odd: the pair (i, i+1)
    const bool wallW = g.neu & kNeuW, wallE = g.neu & kNeuE, wallS = g.neu & kNeuS, wallN = g.neu & kNeuN;
    const bool wallBot = g.neu & kNeuB, wallTop = g.neu & kNeuT;
    // The block, pair and row this thread's cells are in: the tile's own or,
    // in the ring beyond a face that is no wall, those there (a lone block's
    // own again).  Beyond a wall the nearest ones, whose values do not matter.
    int ip, jm, n0 = g.n0, n1 = g.n1;  // extents of that block
    uint32_t vo, vc, pb = (uint32_t)g.sz * W, cpb = (uint32_t)gc.sz * W, csy = (uint32_t)gc.sy * W;
    uint32_t vo_b = 0, vo_t = 0, vc_b = 0, vc_t = 0;  // MB: columns of the blocks below and above
    int n2b = g.n2;                                   // planes of the block below
    bool inx = true, iny = true;
    if constexpr (MB) {
        const int *nb = around[t.b].nb;
        const int xk = i < 1 && !wallW ? -1 : (i > g.n0 && !wallE ? 1 : 0);
        const int yk = j < 1 && !wallS ? -1 : (j > g.n1 && !wallN ? 1 : 0);
        const int col = 13 + 3 * yk + xk;
        const BlockLevel &q = bls[nb[col]], &qc = blc[nb[col]];
        n0 = q.n0;
        n1 = q.n1;
        inx = xk == 0;
        iny = yk == 0;
        ip = xk < 0 ? n0 + i : (xk > 0 ? i - g.n0 : (i < 1 ? 1 : i));
        ip = ip > n0 - 1 ? n0 - 1 : ip;  // past what the stored cells need
        jm = yk < 0 ? n1 + j : (yk > 0 ? j - g.n1 : (j < 1 ? 1 : j));
        jm = jm > n1 ? n1 : jm;
        n2b = bls[nb[4]].n2;
        pb = (uint32_t)q.sz * W;
        cpb = (uint32_t)qc.sz * W;
        csy = (uint32_t)qc.sy * W;
        const int at = ip + (int)q.sy * jm, ac = ((ip + 1) >> 1) + (int)qc.sy * (jm >> 1);
        vo = ((uint32_t)q.off + (uint32_t)at) * W;
        vc = ((uint32_t)qc.off + (uint32_t)ac) * W;
        vo_b = ((uint32_t)bls[nb[col - 9]].off + (uint32_t)at) * W;
        vo_t = ((uint32_t)bls[nb[col + 9]].off + (uint32_t)at) * W;
        vc_b = ((uint32_t)blc[nb[col - 9]].off + (uint32_t)ac) * W;
        vc_t = ((uint32_t)blc[nb[col + 9]].off + (uint32_t)ac) * W;
    } else {
        const int im = leg_map(i, g.n0, !wallW) | 1;  // | 1: beyond a wall, the last pair's left
        ip = im > g.n0 ? g.n0 - 1 : im;
        jm = leg_map(j, g.n1, !wallS);
        vo = ((uint32_t)g.off + (uint32_t)(ip + (int)g.sy * jm)) * W;
        vc = ((uint32_t)gc.off + (uint32_t)(((ip + 1) >> 1) + (int)gc.sy * (jm >> 1))) * W;
    }
    // where plane k (of the own block's count, up to 9 beyond it) is
    struct At {
        uint32_t v, s;  // byte offsets, a thread's and a scalar
    };
    auto plane_at = [&](int k) {
        if (k < 1 && !wallBot) return MB ? At{vo_b + (uint32_t)(k + n2b) * pb, 0u} : At{vo, (uint32_t)(k + g.n2) * pb};
        if (k > g.n2 && !wallTop) return MB ? At{vo_t + (uint32_t)(k - g.n2) * pb, 0u} : At{vo, (uint32_t)(k - g.n2) * pb};
        const uint32_t m = (uint32_t)(k < 1 ? 1 : (k > g.n2 ? g.n2 : k));
        return MB ? At{vo + m * pb, 0u} : At{vo, m * pb};
    };
    // the same from the plane before's, for the loads of the march of a lone
    // block: from k alone the compiler moves them up, 40 registers in VAR
    int kl = 0, kf = 0;
    auto next_at = [&](int k, int &before) {
        if constexpr (MB) {
            return plane_at(k);
        } else {
            before = wallBot ? (k < 1 ? 1 : (k > g.n2 ? g.n2 : k)) : (before == g.n2 ? 1 : before + 1);
            return At{vo, (uint32_t)before * pb};
        }
    };
    auto mapped = [&](int k) { return wallBot ? (k < 1 ? 1 : (k > g.n2 ? g.n2 : k)) : (k < 1 ? k + g.n2 : (k > g.n2 ? k - g.n2 : k)); };
    auto coarse_at = [&](int m) {  // coarse planes 0 and nc + 1 are ghosts
        const int nc = g.n2 >> 1;
        if (m < 0 && !wallBot) return MB ? At{vc_b + (uint32_t)(m + (n2b >> 1)) * cpb, 0u} : At{vc, (uint32_t)(m + nc) * cpb};
        if (m > nc + 1 && !wallTop) return MB ? At{vc_t + (uint32_t)(m - nc) * cpb, 0u} : At{vc, (uint32_t)(m - nc) * cpb};
        const uint32_t q = (uint32_t)(m < 0 ? 0 : (m > nc + 1 ? nc + 1 : m));
        return MB ? At{vc + q * cpb, 0u} : At{vc, q * cpb};
    };
    const bool py = !(wallS && wallN);
    // Column A (i + j even) is the left one of an odd row's pairs and the right
    // one of an even row's.  Even rows run from right to left, so that A's outer
    // x neighbour is the lane before in both, and B's the one after.
    const bool la = UP ? (__builtin_amdgcn_readfirstlane(j) & 1) != 0 : (j & 1) != 0;
    // coefficients: towards the pair's other column always c0; towards the
    // outer side zero at a wall (FP64 keeps c0 and takes a zero neighbour);
    // S and N are c1, a wall row's neighbour read as zero from a pad row
    const T c0 = cconst<T>(g, 0), c1 = cconst<T>(g, 1), c2 = cconst<T>(g, 2);
    const bool wL = i == 1 && (g.neu & kNeuW), wR = i + 1 == g.n0 && (g.neu & kNeuE);
    const T oL = wL ? T(0) : c0, oR = wR ? T(0) : c0;
    const T oA = la ? oL : oR, oB = la ? oR : oL;
    const T wA = la ? oL : c0, eAc = la ? c0 : oR, wB = la ? c0 : oL, eBc = la ? oR : c0;  // aw and ae
    const bool wS = j == 1 && (g.neu & kNeuS), wN = j == g.n1 && (g.neu & kNeuN);
    constexpr bool RCP = sizeof(T) == 4;  // the FP32 inner cycle multiplies by 1/ap
    auto part = [&](T o) {  // a column's diagonal without the z faces
        T s = o + c0;  // aw + ae: one of them is c0, the sum does not depend on the order
        s = s + (wS ? T(0) : c1);
        return s + (wN ? T(0) : c1);
    };
    auto diag = [](T s, T ab, T at) { return -((s + ab) + at); };
    auto divisor = [&](T s, T ab, T at) { return RCP ? T(1) / diag(s, ab, at) : diag(s, ab, at); };
    const T sA = part(oA), sB = part(oB);
    const T dA = divisor(sA, c2, c2), dB = divisor(sB, c2, c2);
    // divisors of planes 1 and n2 of the two columns
    auto at_face = [&](int m, bool isA) -> T & { return face[((m == 1 ? 0 : 2) + (isA ? 0 : 1)) * LEG_NT + tid]; };
    const T wallB = g.neu & kNeuB ? T(0) : c2, wallT = g.neu & kNeuT ? T(0) : c2;
    if constexpr (!VAR) {
        at_face(1, true) = divisor(sA, wallB, c2);
        at_face(1, false) = divisor(sB, wallB, c2);
        at_face(g.n2, true) = divisor(sA, c2, wallT);
        at_face(g.n2, false) = divisor(sB, c2, wallT);
    }
    // the red value of this column that goes to the lane across a periodic
    // face is the one from before the sweep
    const bool eL = ip == 1 && !(inx && wallW), eR = ip + 1 == n0 && !(inx && wallE);
    const bool eA = la ? eL : eR, eB = la ? eR : eL;
    // this thread's entry of an LDS half (after a pad row), its y neighbours'
    // (a pad row's zero beyond a wall), and whether one lies across a periodic face
    const int at0 = 32 * (row + 1) + pair, atS = !VAR && wS ? pair : at0 - 32, atN = !VAR && wN ? pair : at0 + 32;
    const bool ySo = jm == 1 && !(iny && wallS), yNo = jm == n1 && !(iny && wallN);

    auto buf = [&](int b, int slot) { return sm + (2 * b + slot) * LEG_ROW; };
    // buffers: up 0 old black, 1 red 1, 2 black 1, 3 red 2, 4 / 5 the reds that
    // sweep 1 / 2 replaced; down 1 -> 0 red 1, 2 -> 1 black 1, 2 black 2, (red 2:
    // three planes after those), 4 the reds that sweep 2 replaced
    constexpr int R1 = UP ? 1 : 0, B1 = UP ? 2 : 1, B2 = 2, O1 = 4, O2 = UP ? 5 : 4;
    auto red2 = [&](int slot2, int slot3) { return UP ? buf(3, slot2) : sm + (6 + slot3) * LEG_ROW; };
    auto old2 = [&](int slot2) { return UP ? buf(O2, slot2) : sm + (9 + slot2) * LEG_ROW; };
    T A[NS], B[NS], fA[NS], fB[NS], o1[NS], o2[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) A[s] = B[s] = fA[s] = fB[s] = o1[s] = o2[s] = T(0);

    // Loads run D planes ahead, so a step's wait finds them done.  Planes 2m and
    // 2m + 1 take the coarse planes m and m + 1 (rows jm/2 and jm/2 + 1 of each,
    // e0 and e1; around a periodic axis a ghost plane holds the same values as
    // the plane it wraps to); en: plane m + 2, on its way.
    constexpr int D = leg_depth<T, UP>(VAR);
    struct In {
        Pair<T> f, p;
    } L[D];
    T e0[2], e1[2], en[2];
    auto load = [&](In &q, const At &a) {
        q.f = bload2<T>(rs_f, a.v, a.s);
        if constexpr (UP) q.p = bload2<T>(rs_in, a.v, a.s);
    };
    // Variable coefficients: per plane and column the west, east, south, north and
    // top faces and 1 / ap; the bottom face is the top one of the plane below, but
    // for plane 1, whose own bottom face a block's edge makes one-sided (zb).
    const auto rs_x = make_rsrc(faces.x, bytes), rs_y = make_rsrc(faces.y, bytes), rs_z = make_rsrc(faces.z, bytes);
    constexpr int NV = VAR ? NS : 1, DV = 2;  // DV planes in flight
    T wwA[NV], eeA[NV], ssA[NV], nnA[NV], ttA[NV], vvA[NV], wwB[NV], eeB[NV], ssB[NV], nnB[NV], ttB[NV], vvB[NV];
    T zbA = T(0), zbB = T(0);
    struct Faces {
        Pair<T> x, s, n, t;
        T xr;
    } F[VAR ? DV : 1];
    auto load_f = [&](Faces &q, const At &a) {
        const uint32_t o = a.s;
        q.x = bload2<T>(rs_x, vo, o);
        q.xr = bload<T>(rs_x, vo + 2 * W, o);
        q.s = bload2<T>(rs_y, vo, o);
        q.n = bload2<T>(rs_y, vo, o + (uint32_t)g.sy * W);
        q.t = bload2<T>(rs_z, vo, o + pb);
    };
    auto take_f = [&](const Faces &q, int k, auto slot, auto below) {  // plane k into the rings
        constexpr int S = VAR ? decltype(slot)::value : 0, L = VAR ? decltype(below)::value : 0;
        wwA[S] = la ? q.x.l : q.x.r;
        eeA[S] = la ? q.x.r : q.xr;
        wwB[S] = la ? q.x.r : q.x.l;
        eeB[S] = la ? q.xr : q.x.r;
        ssA[S] = la ? q.s.l : q.s.r;
        ssB[S] = la ? q.s.r : q.s.l;
        nnA[S] = la ? q.n.l : q.n.r;
        nnB[S] = la ? q.n.r : q.n.l;
        const bool first = k == 1 || k == g.n2 + 1;
        const T bA = first ? zbA : ttA[L], bB = first ? zbB : ttB[L];
        ttA[S] = la ? q.t.l : q.t.r;
        ttB[S] = la ? q.t.r : q.t.l;
        vvA[S] = T(1) / -(((((wwA[S] + eeA[S]) + ssA[S]) + nnA[S]) + bA) + ttA[S]);
        vvB[S] = T(1) / -(((((wwB[S] + eeB[S]) + ssB[S]) + nnB[S]) + bB) + ttB[S]);
        // here and now: moved to where they are used, the divisions would keep
        // their operands in registers (UP 215 of them instead of 159)
        asm volatile("" : "+v"(vvA[S]), "+v"(vvB[S]));
    };
    auto load_c = [&](T *e, int m) {  // coarse plane m of the unwrapped planes 2m - 2 .. 2m + 1
        const At a = coarse_at(m);
        e[0] = bload<T>(rs_c, a.v, a.s);
        e[1] = MB ? bload<T>(rs_c, a.v + csy, a.s) : bload<T>(rs_c, a.v, a.s + csy);
    };
    // a plane's values, the potential corrected as k_prolong does it
    auto take = [&](const In &q, bool odd, T &a, T &b, T &ra, T &rb) {
        ra = la ? q.f.l : q.f.r;
        rb = la ? q.f.r : q.f.l;
        if constexpr (UP) {
            const T m[4] = {e0[0], e0[1], e1[0], e1[1]};
            // weights of the coarse rows and planes, literals: every call has
            // its plane's parity and its branch the row's
            auto weight = [&](int n, bool odd_row) {
                return T((((n & 1) != 0) == odd_row ? 3 : 1) * (((n & 2) != 0) == odd ? 3 : 1));
            };
            // the pair's own coarse column (weight 3) and the outer one (weight
            // 1): the left column's terms begin with the outer one's
            auto outer_first = [&](auto shift, bool odd_row) {
                T v = weight(0, odd_row) * shift(m[0]);
#pragma unroll
                for (int n = 1; n < 4; ++n) v = v + weight(n, odd_row) * shift(m[n]);
#pragma unroll
                for (int n = 0; n < 4; ++n) v = v + (T(3) * weight(n, odd_row)) * m[n];
                return v;
            };
            auto own_first = [&](auto shift, bool odd_row) {
                T v = (T(3) * weight(0, odd_row)) * m[0];
#pragma unroll
                for (int n = 1; n < 4; ++n) v = v + (T(3) * weight(n, odd_row)) * m[n];
#pragma unroll
                for (int n = 0; n < 4; ++n) v = v + weight(n, odd_row) * shift(m[n]);
                return v;
            };
            auto before = [](T v) { return from_left(v); };
            auto after = [](T v) { return from_right(v); };
            if (la) {  // uniform: an odd row
                a = q.p.l + outer_first(before, true) / T(64);
                b = q.p.r + own_first(after, true) / T(64);
            } else {
                a = q.p.r + own_first(before, false) / T(64);
                b = q.p.l + outer_first(after, false) / T(64);
            }
            asm volatile("" : "+v"(a), "+v"(b));  // here and now, as in take_f
        }
    };
    // One update of column A (X_A) or B on plane k.  The outer x
    // neighbour and the own one are ordered W, E in FP32, whose sum contracts;
    // in FP64 the two products are rounded before they are added and the
    // order is free.  zB, zT: the neighbours below and above; qB, qT: those a
    // black update takes across a periodic face.
    auto sum = [&](auto slot, bool isA, T outer, T own, T yS, T yN, T ab, T zB, T at, T zT) -> T {
        T s;
        if constexpr (VAR) {
            constexpr int S = decltype(slot)::value;
            const bool left = isA ? la : !la;
            s = (isA ? wwA : wwB)[S] * (left ? outer : own);
            s = madd(s, (isA ? eeA : eeB)[S], left ? own : outer);
            s = madd(s, (isA ? ssA : ssB)[S], yS);
            s = madd(s, (isA ? nnA : nnB)[S], yN);
            s = madd(s, ab, zB);
            return madd(s, at, zT);
        }
        if constexpr (RCP) {
            const bool left = isA ? la : !la;
            s = (isA ? wA : wB) * (left ? outer : own);
            s = madd(s, isA ? eAc : eBc, left ? own : outer);
        } else {
            s = c0 * outer;
            s = s + c0 * own;
        }
        s = madd(s, c1, yS);
        s = madd(s, c1, yN);
        s = madd(s, ab, zB);
        s = madd(s, at, zT);
        return s;
    };
    auto relax = [&](auto slot, auto below, bool isA, T r, T outer, T own, T yS, T yN, int k, T zB, T zT, T qB, T qT) -> T {
        T d = isA ? dA : dB, ab = c2, at = c2;
        if constexpr (VAR) {
            d = (isA ? vvA : vvB)[decltype(slot)::value];
            ab = (isA ? ttA : ttB)[decltype(below)::value];
            at = (isA ? ttA : ttB)[decltype(slot)::value];
        }
        if ((unsigned)k <= 1u || (unsigned)(k - g.n2) <= 1u) {  // beside a z face of a block; uniform, rare
            if (k == 1 || k == g.n2 + 1) {
                if constexpr (VAR) ab = isA ? zbA : zbB;
                if (k == 1 && wallBot) {
                    if constexpr (!VAR) {
                        ab = T(0);
                        d = at_face(1, isA);
                    }
                } else {
                    zB = qB;
                }
            } else if (k == g.n2 && wallTop) {
                if constexpr (!VAR) {
                    at = T(0);
                    d = at_face(k, isA);
                }
            } else {
                zT = qT;
            }
        }
        const T s = sum(slot, isA, outer, own, yS, yN, ab, zB, at, zT);
        return RCP ? (r - s) * d : (r - s) / d;
    };
    const bool xw = sizeof(T) == 8 && (wallW || wallE), xA = xw && (la ? wL : wR), xB = xw && (la ? wR : wL);  // A, B beside a wall
    auto outer_of = [&](bool isA, T v) {
        T o = isA ? from_left(v) : from_right(v);
        if (xw) o = (isA ? xA : xB) ? T(0) : o;  // uniform
        return o;
    };

    const int cm = UP ? t.z0 - 3 : t.z0 - 4, ce = UP ? t.z1 + 3 : t.z1 + 4;  // first and last step
    constexpr int P0 = UP ? 0 : 1;                                           // parity of cm (z0 is odd)
    // plane cm + d sits in slot d mod NS
    kl = mapped(cm + 1 + D);
    kf = mapped(cm + DV);
    {
        Pair<T> zb, top;
        Faces f0;
        if constexpr (VAR) {
            zb = bload2<T>(rs_z, vo, pb);
            top = bload2<T>(rs_z, vo, plane_at(cm - 1).s + pb);
            load_f(f0, plane_at(cm));
#pragma unroll
            for (int d = 0; d < DV; ++d) load_f(F[d], plane_at(cm + 1 + d));
        }
        In q[3];
        if constexpr (UP) {  // planes cm - 1 (odd), cm, cm + 1
            load(q[0], plane_at(cm - 1));
            load_c(e0, (cm - 2) / 2);
            load_c(e1, cm / 2);
            load_c(en, cm / 2 + 1);
        }
        load(q[1], plane_at(cm));
        load(q[2], plane_at(cm + 1));
#pragma unroll
        for (int d = 0; d < D; ++d) load(L[d], plane_at(cm + 2 + d));
        // while they travel; the pad rows stay zero, the first steps read the rest before it is written
        for (int e = tid; e < LEG_ROW * (UP ? 8 + (py ? 4 : 0) : 9 + (py ? 2 : 0)); e += LEG_NT) sm[e] = T(0);
        __syncthreads();
        if constexpr (VAR) {
            zbA = la ? zb.l : zb.r;
            zbB = la ? zb.r : zb.l;
            ttA[NS - 1] = la ? top.l : top.r;
            ttB[NS - 1] = la ? top.r : top.l;
            take_f(f0, cm, Step<0>{}, Step<NS - 1>{});
        }
        if constexpr (UP) {
            take(q[0], true, A[NS - 1], B[NS - 1], fA[NS - 1], fB[NS - 1]);
            e0[0] = e1[0];
            e0[1] = e1[1];
            e1[0] = en[0];
            e1[1] = en[1];
            load_c(en, cm / 2 + 2);
        }
        take(q[1], P0, A[0], B[0], fA[0], fB[0]);
        take(q[2], !P0, A[1], B[1], fA[1], fB[1]);
        if constexpr (UP) buf(0, P0)[at0] = P0 ? B[0] : A[0];  // black: A on even planes
    }
    __syncthreads();

    const bool stored = pair >= 3 && pair < 3 + LEG_TX / 2 && i <= g.n0 && row >= 4 && row < 4 + LEG_TY && j <= g.n1;
    const bool img = __any(stored && (ghost_image(i, g.n0, g.neu & kNeuW, g.neu & kNeuE) >= 0 ||
                                      ghost_image(i + 1, g.n0, g.neu & kNeuW, g.neu & kNeuE) >= 0 ||
                                      ghost_image(j, g.n1, g.neu & kNeuS, g.neu & kNeuN) >= 0));  // in the wavefront
    const int sy = (int)g.sy;
    const uint32_t ob = (uint32_t)g.off * W, ob_z = (uint32_t)g.sz * W;
    auto roff = [&](int x, int y) { return ob + (uint32_t)(x + sy * y) * W; };
    const uint32_t vs = roff(i, j);
    auto store = [&](int z, T a, T b) {  // plane z of this thread's stored cells and their ghost images
        if (z < t.z0 || z > t.z1) return;  // uniform
        if (!stored) return;
        const Pair<T> v{la ? a : b, la ? b : a};
        bstore2<T>(rs_out, v, vs, (uint32_t)z * ob_z);
        if (!UP || MB || !(img || z == 1 || z == g.n2)) return;  // uniform; the up leg reads no ghosts of its level
        const int iz = ghost_image(z, g.n2, g.neu & kNeuB, g.neu & kNeuT);
        int x = i, y = j;  // opaque, or the addresses of every image stay in registers
        asm volatile("" : "+v"(x), "+v"(y));
        const int xl = ghost_image(x, g.n0, g.neu & kNeuW, g.neu & kNeuE);
        const int xr = ghost_image(x + 1, g.n0, g.neu & kNeuW, g.neu & kNeuE);
        const int yg = ghost_image(y, g.n1, g.neu & kNeuS, g.neu & kNeuN);
        auto plane = [&](int zz) {
            const uint32_t s = (uint32_t)zz * ob_z;
            if (zz != z) bstore2<T>(rs_out, v, roff(x, y), s);
            if (yg >= 0) bstore2<T>(rs_out, v, roff(x, yg), s);
            if (xl >= 0) {
                bstore<T>(rs_out, v.l, roff(xl, y), s);
                if (yg >= 0) bstore<T>(rs_out, v.l, roff(xl, yg), s);
            }
            if (xr >= 0) {
                bstore<T>(rs_out, v.r, roff(xr, y), s);
                if (yg >= 0) bstore<T>(rs_out, v.r, roff(xr, yg), s);
            }
        };
        plane(z);
        if (iz >= 0) plane(iz);
    };

    const uint32_t vcs = ((uint32_t)gc.off + (uint32_t)(((i + 1) >> 1) + (int)gc.sy * ((j + 1) >> 1))) * W;
    T acc = T(0);  // down: the restricted residual's sum so far
    // Step J of a turn, plane c = cm + NS m + J: X is the column updated in
    // it (red on planes c and c-2, black on c-1 and c-3), Y the other.
    auto step = [&](int c, auto jc) {
        constexpr int J = decltype(jc)::value, PC = (J + P0) & 1, J3 = J % 3;
        constexpr auto sl = [](int d) { return ((J + d) % NS + NS) % NS; };
        constexpr bool XA = PC != 0;  // X is column A
        T *X = XA ? A : B, *Y = XA ? B : A;
        const T *fX = XA ? fA : fB, *fY = XA ? fB : fA;
        const bool edge = XA ? eB : eA;  // of the sending column, Y
        // the y neighbours of the four updates, written in the step before
        T y1S = T(0), y1N = T(0);
        if constexpr (UP) {
            const T *b0 = buf(0, PC);
            y1S = b0[atS];
            y1N = b0[atN];
        }
        const T *b1 = buf(R1, 1 - PC), *b2 = buf(B1, PC), *b3 = red2(1 - PC, (J3 + 1) % 3);
        T y2S = b1[atS], y2N = b1[atN];
        const T y3S = b2[atS], y3N = b2[atN];
        T y4S = b3[atS], y4N = b3[atN];
        if (py) {  // uniform
            if constexpr (UP) {
                const T *q = buf(O1, 1 - PC);
                const T a = q[atS], b = q[atN];
                y2S = ySo ? a : y2S;
                y2N = yNo ? b : y2N;
            } else {
                y2S = ySo ? T(0) : y2S;
                y2N = yNo ? T(0) : y2N;
            }
            const T *q = old2(1 - PC);
            const T a = q[atS], b = q[atN];
            y4S = ySo ? a : y4S;
            y4N = yNo ? b : y4N;
        }
        if constexpr (UP) buf(0, 1 - PC)[at0] = X[sl(1)];  // plane c+1: its black column is X

        // red, sweep 1, plane c
        if constexpr (UP) {
            const T v = X[sl(0)];
            o1[sl(0)] = v;
            if (py) buf(O1, PC)[at0] = v;
            X[sl(0)] = relax(Step<VAR ? sl(0) : 0>{}, Step<VAR ? sl(-1) : 0>{}, XA, fX[sl(0)], outer_of(XA, Y[sl(0)]), Y[sl(0)], y1S, y1N, c, X[sl(-1)], X[sl(1)],
                             X[sl(-1)], X[sl(1)]);
        } else {
            T d = XA ? dA : dB;
            if constexpr (VAR) d = (XA ? vvA : vvB)[VAR ? sl(0) : 0];
            else if ((c == 1 && wallBot) || (c == g.n2 && wallTop)) d = at_face(c, XA);
            X[sl(0)] = RCP ? (fX[sl(0)] - T(0)) * d : (fX[sl(0)] - T(0)) / d;
        }
        buf(R1, PC)[at0] = X[sl(0)];

        // black, sweep 1, plane c-1; across a periodic face the old reds
        {
            const T yv = edge ? o1[sl(-1)] : Y[sl(-1)];
            X[sl(-1)] = relax(Step<VAR ? sl(-1) : 0>{}, Step<VAR ? sl(-2) : 0>{}, XA, fX[sl(-1)], outer_of(XA, yv), Y[sl(-1)], y2S, y2N, c - 1, X[sl(-2)], X[sl(0)],
                              o1[sl(-2)], o1[sl(0)]);
            buf(B1, 1 - PC)[at0] = X[sl(-1)];
        }
        // red, sweep 2, plane c-2
        {
            const T v = X[sl(-2)];
            o2[sl(-2)] = v;
            if (py) old2(PC)[at0] = v;
            X[sl(-2)] = relax(Step<VAR ? sl(-2) : 0>{}, Step<VAR ? sl(-3) : 0>{}, XA, fX[sl(-2)], outer_of(XA, Y[sl(-2)]), Y[sl(-2)], y3S, y3N, c - 2, X[sl(-3)],
                              X[sl(-1)], X[sl(-3)], X[sl(-1)]);
            red2(PC, (J3 + 2) % 3)[at0] = X[sl(-2)];
        }
        // black, sweep 2, plane c-3
        {
            const T yv = edge ? o2[sl(-3)] : Y[sl(-3)];
            X[sl(-3)] = relax(Step<VAR ? sl(-3) : 0>{}, Step<VAR ? sl(-4) : 0>{}, XA, fX[sl(-3)], outer_of(XA, yv), Y[sl(-3)], y4S, y4N, c - 3, X[sl(-4)], X[sl(-2)],
                              o2[sl(-4)], o2[sl(-2)]);
            if constexpr (!UP) buf(B2, 1 - PC)[at0] = X[sl(-3)];
        }
        store(c - 3, A[sl(-3)], B[sl(-3)]);

        if constexpr (!UP) {  // the residual of plane c-4, its ghosts refreshed, into the coarse RHS
            const int z = c - 4;  // only planes of the chunk matter, which map to themselves
            const T ab = z == 1 ? wallB : c2, at = z == g.n2 ? wallT : c2;
            const T *bb = buf(B2, PC), *br = red2(0, J3);
            auto res = [&](bool isA, T o, T f, T own, T outer, T yS, T yN, T zB, T zT, T self) {
                // without contraction, as k_restrict: aw*W + ae*E is free of order
                if constexpr (VAR) {
                    constexpr int S = VAR ? sl(-4) : 0, L = VAR ? sl(-5) : 0;
                    const bool left = isA ? la : !la;
                    const T w = (isA ? wwA : wwB)[S], e = (isA ? eeA : eeB)[S], so = (isA ? ssA : ssB)[S],
                            no = (isA ? nnA : nnB)[S], b = z == 1 ? (isA ? zbA : zbB) : (isA ? ttA : ttB)[L],
                            t = (isA ? ttA : ttB)[S];
                    T v = w * (left ? outer : own);
                    v = v + e * (left ? own : outer);
                    v = v + so * yS;
                    v = v + no * yN;
                    v = v + b * zB;
                    v = v + t * zT;
                    v = v + -(((((w + e) + so) + no) + b) + t) * self;
                    return f - v;
                }
                T s = (RCP ? o : c0) * outer;
                s = s + c0 * own;
                s = s + c1 * yS;
                s = s + c1 * yN;
                s = s + ab * zB;
                s = s + at * zT;
                s = s + diag(isA ? sA : sB, ab, at) * self;
                return f - s;
            };
            // X on plane c-4 is red (its y neighbours black 2), Y black (red 2)
            const T rx = res(XA, XA ? oA : oB, fX[sl(-4)], Y[sl(-4)], outer_of(XA, Y[sl(-4)]), bb[atS], bb[atN],
                             X[sl(-5)], X[sl(-3)], X[sl(-4)]);
            const T ry = res(!XA, XA ? oB : oA, fY[sl(-4)], X[sl(-4)], outer_of(!XA, X[sl(-4)]), br[atS], br[atN],
                             Y[sl(-5)], Y[sl(-3)], Y[sl(-4)]);
            const T ra = XA ? rx : ry, rb = XA ? ry : rx;
            // the even row's (A is its right column): the same pair, in the
            // wavefront's upper half from the other end
            const T ul = __shfl_xor(rb, 63, 64), ur = __shfl_xor(ra, 63, 64);
            // children in the order (0,0,0) (1,0,0) (0,1,0) (1,1,0) (0,0,1) (1,0,1) (0,1,1) (1,1,1)
            acc = PC ? ra : acc + ra;  // plane c-4 odd: the lower one
            acc = acc + rb;
            acc = acc + ul;
            acc = acc + ur;
            if (!PC && z >= t.z0 && z <= t.z1 && stored && !(row & 1)) bstore<T>(rs_c, T(0.125) * acc, vcs, (uint32_t)(z >> 1) * (uint32_t)(gc.sz * W));
        }
        if constexpr (UP && PC == 0) {  // plane c+2 is even: the next two coarse planes
            e0[0] = e1[0];
            e0[1] = e1[1];
            e1[0] = en[0];
            e1[1] = en[1];
            load_c(en, (c + 2) / 2 + 2);
        }
        take(L[J % D], PC != 0, A[sl(2)], B[sl(2)], fA[sl(2)], fB[sl(2)]);
        load(L[J % D], next_at(c + 2 + D, kl));
        if constexpr (VAR) {  // the faces of plane c+1
            take_f(F[J % DV], c + 1, Step<sl(1)>{}, Step<sl(0)>{});
            load_f(F[J % DV], next_at(c + 1 + DV, kf));
        }
        __syncthreads();
    };
    for (int c = cm; c <= ce; c += NS) {
        step(c, Step<0>{});
        if (c + 1 > ce) break;
        step(c + 1, Step<1>{});
        if (c + 2 > ce) break;
        step(c + 2, Step<2>{});
        if (c + 3 > ce) break;
        step(c + 3, Step<3>{});
        if (c + 4 > ce) break;
        step(c + 4, Step<4>{});
        if (c + 5 > ce) break;
        step(c + 5, Step<5>{});
    }
}

// The same leg on a small level, a box at a time: a workgroup takes
// 8 x 8 x 8 cells with a ring of 4 (16^3 cells) into LDS and does the four half
// sweeps there, one barrier each, where the march above takes a step of about
// 1 us for each of at least ten planes.  The ring makes it eight times the
// cells of the box, so it pays only while the level does not fill the card
// (32^3 FP64: 6.7 us down and 9.3 up where the march takes 13.0 and 13.4; both
// sides by size stand at the rule in leg_level).  One workgroup of 1024 threads has a
// compute unit's registers in FP64 (82 a thread) and with variable
// coefficients; held to 64, for two, it spills and takes 11.3 and 13.0.
//
// A thread owns two pairs of cells (odd i and i + 1), eight planes apart: one red
// and one black cell each, their RHS (and coefficients) in registers.  In P every
// cell's potential; in Q the values that the red updates replace, which a
// black update takes across a periodic face.  Each half sweep updates the
// cells one further in from the box's surface.
constexpr int L3_N = 16, L3_TILE = 8, L3_SY = 18, L3_SZ = L3_SY * L3_N, L3_CELLS = L3_SZ * L3_N, L3_NT = 1024;
template <typename T>
constexpr int leg3_lds() { return 2 * L3_CELLS * (int)sizeof(T); }

template <typename T, bool UP, bool VAR, bool MB = false>
__global__ __launch_bounds__(L3_NT) void k_leg3(const T *__restrict__ pin, T *__restrict__ pout,
                                                const T *__restrict__ rhs, LegFaces<T> faces, uint32_t bytes,
                                                const BlockLevel *__restrict__ bls, const Tile *__restrict__ tiles,
                                                const int *__restrict__ done, const T *__restrict__ phic,
                                                T *__restrict__ rhsc, uint32_t cbytes,
                                                const BlockLevel *__restrict__ blc,
                                                const LegBlocks *__restrict__ around) {
    const int stop = done ? *done : 0;  // awaited with the tile
    extern __shared__ __align__(16) unsigned char leg_smem[];
    T *P = reinterpret_cast<T *>(leg_smem), *Q = P + L3_CELLS;
    constexpr uint32_t W = sizeof(T);
    constexpr bool RCP = sizeof(T) == 4;  // the FP32 inner cycle multiplies by 1/ap
    const Tile t = tiles[blockIdx.x];
    const BlockLevel g = bls[t.b], gc = blc[t.b];
    if (stop) return;
    const auto rs_in = make_rsrc(pin, bytes), rs_f = make_rsrc(rhs, bytes), rs_out = make_rsrc(pout, bytes);
    const auto rs_c = make_rsrc(UP ? phic : rhsc, cbytes);
    const auto rs_x = make_rsrc(faces.x, bytes), rs_y = make_rsrc(faces.y, bytes), rs_z = make_rsrc(faces.z, bytes);
    const bool wallW = g.neu & kNeuW, wallE = g.neu & kNeuE, wallS = g.neu & kNeuS, wallN = g.neu & kNeuN;
    const bool wallBot = g.neu & kNeuB, wallTop = g.neu & kNeuT;
    const T c0 = cconst<T>(g, 0), c1 = cconst<T>(g, 1), c2 = cconst<T>(g, 2);
    const int tid = (int)threadIdx.x, i = tid & 7, y = (tid >> 3) & 15, zh = tid >> 7;
    const uint32_t rb = (uint32_t)g.sy * W;
    const int X = t.x0 - 4 + 2 * i, Y = t.y0 - 4 + y;
    // the side of the block that coordinate v is on (0: the block, or beyond a wall),
    // and the cell 1..m there (n, m: extents of the block and of the one there)
    auto side = [](int v, int n, bool lo, bool hi) { return v < 1 && !lo ? -1 : (v > n && !hi ? 1 : 0); };
    auto cell = [](int v, int n, int m, int k) {
        const int c = k < 0 ? v + m : (k > 0 ? v - n : v);
        return c < 1 ? 1 : (c > m ? m : c);
    };
    const int xk = side(X, g.n0, wallW, wallE), yk = side(Y, g.n1, wallS, wallN);
    const int *nb = MB ? around[t.b].nb : nullptr;
    const BlockLevel &own = MB ? bls[nb[13 + 3 * yk + xk]] : bls[t.b];  // the column's block, beside this one
    const int n0 = own.n0, n1 = own.n1;
    const int im = cell(X, g.n0, n0, xk) | 1, ip = im > n0 ? n0 - 1 : im, jm = cell(Y, g.n1, n1, yk);
    const uint32_t pb = (uint32_t)own.sz * W;
    // this thread's cells: r red (i + j + k odd), b black
    T fr[2], fb[2], pr[2], pbk[2];
    int qr[2], qb[2], dr[2], db[2];
    unsigned er[2], eb[2];  // faces of its block beside the cell, W E S N B T: to other cells, then (<< 6) walls
    struct Coef {
        T w, e, s, n, b, t;
    } kr[VAR ? 2 : 1], kb[VAR ? 2 : 1];
    T vr[VAR ? 2 : 1], vb[VAR ? 2 : 1];
    struct In {
        Pair<T> f, p, xl, s, n, b, t;
        T xr;
    } in[2];
    bool left[2];  // the left cell is the red one
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int z = zh + 8 * u, Z = t.z0 - 4 + z, zk = side(Z, g.n2, wallBot, wallTop);
        const BlockLevel &there = MB ? bls[nb[13 + 9 * zk + 3 * yk + xk]] : bls[t.b];
        const int n2 = there.n2, km = cell(Z, g.n2, n2, zk);
        const uint32_t o = ((uint32_t)there.off + (uint32_t)(ip + (int)own.sy * jm)) * W, s = (uint32_t)km * pb;
        in[u].f = bload2<T>(rs_f, o + s, 0);
        if constexpr (UP) in[u].p = bload2<T>(rs_in, o + s, 0);
        if constexpr (VAR) {
            in[u].xl = bload2<T>(rs_x, o + s, 0);
            in[u].xr = bload<T>(rs_x, o + s + 2 * W, 0);
            in[u].s = bload2<T>(rs_y, o + s, 0);
            in[u].n = bload2<T>(rs_y, o + s + rb, 0);
            in[u].b = bload2<T>(rs_z, o + s, 0);
            in[u].t = bload2<T>(rs_z, o + s + pb, 0);
        }
        left[u] = !((Y + t.z0 + z) & 1);
        const int q = 2 * i + L3_SY * y + L3_SZ * z;
        const int d = min(min(y, 15 - y), min(z, 15 - z));
        const int dl = min(d, min(2 * i, 15 - 2 * i)), dd = min(d, min(2 * i + 1, 14 - 2 * i));
        auto face = [](bool at, bool wall, unsigned bit) { return at ? (wall ? bit << 6 : bit) : 0u; };
        const unsigned e = face(jm == 1, yk == 0 && wallS, 4) | face(jm == n1, yk == 0 && wallN, 8) |
                           face(km == 1, zk == 0 && wallBot, 16) | face(km == n2, zk == 0 && wallTop, 32);
        const unsigned el = e | face(ip == 1, xk == 0 && wallW, 1), ed = e | face(ip + 1 == n0, xk == 0 && wallE, 2);
        qr[u] = left[u] ? q : q + 1;
        qb[u] = left[u] ? q + 1 : q;
        dr[u] = left[u] ? dl : dd;
        db[u] = left[u] ? dd : dl;
        er[u] = left[u] ? el : ed;
        eb[u] = left[u] ? ed : el;
    }
    if constexpr (UP) {  // the coarse potential around the box, 10^3, waits in Q
        if (tid < 1000) {
            const int a = tid % 10, b = tid / 10 % 10, c = tid / 100;
            auto cside = [](int v, int n, bool lo, bool hi) { return v < 0 && !lo ? -1 : (v > n + 1 && !hi ? 1 : 0); };
            auto ccell = [](int v, int n, int m, int k) {  // 0 and m + 1 are ghosts
                const int q = k < 0 ? v + m : (k > 0 ? v - n : v);
                return q < 0 ? 0 : (q > m + 1 ? m + 1 : q);
            };
            const int cx = (t.x0 - 5) / 2 + a, cy = (t.y0 - 5) / 2 + b, cz = (t.z0 - 5) / 2 + c;
            const int ka = cside(cx, gc.n0, wallW, wallE), kb2 = cside(cy, gc.n1, wallS, wallN),
                      kc = cside(cz, gc.n2, wallBot, wallTop);
            const BlockLevel &q = MB ? blc[nb[13 + 9 * kc + 3 * kb2 + ka]] : blc[t.b];
            const int ci = ccell(cx, gc.n0, q.n0, ka), cj = ccell(cy, gc.n1, q.n1, kb2), ck = ccell(cz, gc.n2, q.n2, kc);
            Q[tid] = bload<T>(rs_c, ((uint32_t)q.off + (uint32_t)(ci + (int)q.sy * cj + (int)q.sz * ck)) * W, 0);
        }
        __syncthreads();
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int z = zh + 8 * u;
        Pair<T> p{T(0), T(0)};
        if constexpr (UP) {  // corrected as k_prolong does it
            const T *e = Q + i + 10 * ((y + 1) >> 1) + 100 * ((z + 1) >> 1);
            const T wj0 = (y & 1) ? T(3) : T(1), wj1 = (y & 1) ? T(1) : T(3);
            const T wk0 = (z & 1) ? T(3) : T(1), wk1 = (z & 1) ? T(1) : T(3);
            auto child = [&](int a, T wi0, T wi1) {
                T s = (wi0 * wj0 * wk0) * e[a];
                s = s + (wi0 * wj1 * wk0) * e[a + 10];
                s = s + (wi0 * wj0 * wk1) * e[a + 100];
                s = s + (wi0 * wj1 * wk1) * e[a + 110];
                s = s + (wi1 * wj0 * wk0) * e[a + 1];
                s = s + (wi1 * wj1 * wk0) * e[a + 11];
                s = s + (wi1 * wj0 * wk1) * e[a + 101];
                s = s + (wi1 * wj1 * wk1) * e[a + 111];
                return s / T(64);
            };
            p.l = in[u].p.l + child(0, T(1), T(3));
            p.r = in[u].p.r + child(1, T(3), T(1));
        }
        fr[u] = left[u] ? in[u].f.l : in[u].f.r;
        fb[u] = left[u] ? in[u].f.r : in[u].f.l;
        pr[u] = left[u] ? p.l : p.r;
        pbk[u] = left[u] ? p.r : p.l;
        if constexpr (VAR) {
            const In &v = in[u];
            const Coef l{v.xl.l, v.xl.r, v.s.l, v.n.l, v.b.l, v.t.l}, r{v.xl.r, v.xr, v.s.r, v.n.r, v.b.r, v.t.r};
            kr[u] = left[u] ? l : r;
            kb[u] = left[u] ? r : l;
            auto divisor = [](const Coef &k) {
                const T ap = -(((((k.w + k.e) + k.s) + k.n) + k.b) + k.t);
                return RCP ? T(1) / ap : ap;
            };
            vr[u] = divisor(kr[u]);
            vb[u] = divisor(kb[u]);
        }
    }
    if constexpr (UP) __syncthreads();  // Q is free

    auto coef = [&](int u, bool red, unsigned e) {  // walls have no coefficient
        if constexpr (VAR) return red ? kr[u] : kb[u];
        else
            return Coef{(e & 64) ? T(0) : c0, (e & 128) ? T(0) : c0, (e & 256) ? T(0) : c1,
                        (e & 512) ? T(0) : c1, (e & 1024) ? T(0) : c2, (e & 2048) ? T(0) : c2};
    };
    auto diag = [](const Coef &k) { return -(((((k.w + k.e) + k.s) + k.n) + k.b) + k.t); };
    auto divide = [&](int u, bool red, const Coef &k, T r) {
        if constexpr (VAR) return RCP ? r * (red ? vr[u] : vb[u]) : r / (red ? vr[u] : vb[u]);
        else if constexpr (RCP) return r * (T(1) / diag(k));
        else return r / diag(k);
    };
    auto update = [&](int u, bool red) {
        const int q = red ? qr[u] : qb[u];
        const unsigned e = red ? er[u] : eb[u];
        T w = P[q - 1], ea = P[q + 1], s = P[q - L3_SY], n = P[q + L3_SY], b = P[q - L3_SZ], tp = P[q + L3_SZ];
        if (!red && (e & 63)) {  // across a face of its block, the red value from before the sweep
            if (e & 1) w = Q[q - 1];
            if (e & 2) ea = Q[q + 1];
            if (e & 4) s = Q[q - L3_SY];
            if (e & 8) n = Q[q + L3_SY];
            if (e & 16) b = Q[q - L3_SZ];
            if (e & 32) tp = Q[q + L3_SZ];
        }
        const Coef k = coef(u, red, e);
        T a = k.w * w;
        a = madd(a, k.e, ea);
        a = madd(a, k.s, s);
        a = madd(a, k.n, n);
        a = madd(a, k.b, b);
        a = madd(a, k.t, tp);
        return divide(u, red, k, (red ? fr[u] : fb[u]) - a);
    };
    constexpr int D0 = UP ? 1 : 0;  // distance from the box's surface of the first half sweep
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        if constexpr (UP) {
            P[qr[u]] = pr[u];
        } else {
            pr[u] = divide(u, true, coef(u, true, er[u]), fr[u] - T(0));
            P[qr[u]] = pr[u];
            Q[qr[u]] = T(0);
        }
        P[qb[u]] = pbk[u];
    }
    __syncthreads();
    auto reds = [&](int dmin) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
            if (dr[u] >= dmin) {
                const T v = update(u, true);
                Q[qr[u]] = pr[u];
                P[qr[u]] = pr[u] = v;
            }
        __syncthreads();
    };
    auto blacks = [&](int dmin) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
            if (db[u] >= dmin) P[qb[u]] = pbk[u] = update(u, false);
        __syncthreads();
    };
    if constexpr (UP) reds(D0);
    blacks(D0 + 1);
    reds(D0 + 2);
    blacks(D0 + 3);

#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int z = zh + 8 * u, Z = t.z0 - 4 + z;
        const uint32_t pl = (uint32_t)g.sz * W;
        if (i < 2 || i > 5 || y < 4 || y > 11 || z < 4 || z > 11) continue;  // the ring
        if (X > g.n0 || Y > g.n1 || Z > g.n2) continue;
        const Pair<T> v{left[u] ? pr[u] : pbk[u], left[u] ? pbk[u] : pr[u]};
        auto at = [&](int x, int yy, int zz) { return ((uint32_t)g.off + (uint32_t)(x + (int)g.sy * yy)) * W + (uint32_t)zz * pl; };
        bstore2<T>(rs_out, v, at(X, Y, Z), 0);
        if constexpr (UP && !MB) {  // the ghost images; the up leg reads no ghosts of its level, so down writes none
            const int xl = ghost_image(X, g.n0, g.neu & kNeuW, g.neu & kNeuE);
            const int xr = ghost_image(X + 1, g.n0, g.neu & kNeuW, g.neu & kNeuE);
            const int yg = ghost_image(Y, g.n1, g.neu & kNeuS, g.neu & kNeuN);
            const int zg = ghost_image(Z, g.n2, g.neu & kNeuB, g.neu & kNeuT);
#pragma unroll 1
            for (int m = 0; m < 4; ++m) {
                const int yy = m & 1 ? yg : Y, zz = m & 2 ? zg : Z;
                if (yy < 0 || zz < 0) continue;
                if (m) bstore2<T>(rs_out, v, at(X, yy, zz), 0);
                if (xl >= 0) bstore<T>(rs_out, v.l, at(xl, yy, zz), 0);
                if (xr >= 0) bstore<T>(rs_out, v.r, at(xr, yy, zz), 0);
            }
        }
        if constexpr (!UP) {  // the residual, its ghosts refreshed, without contraction as k_restrict
            auto residual = [&](bool red) {
                const int q = red ? qr[u] : qb[u];
                const Coef k = coef(u, red, red ? er[u] : eb[u]);
                T s = k.w * P[q - 1];
                s = s + k.e * P[q + 1];
                s = s + k.s * P[q - L3_SY];
                s = s + k.n * P[q + L3_SY];
                s = s + k.b * P[q - L3_SZ];
                s = s + k.t * P[q + L3_SZ];
                s = s + diag(k) * P[q];
                return (red ? fr[u] : fb[u]) - s;
            };
            Q[qr[u]] = residual(true);
            Q[qb[u]] = residual(false);
        }
    }
    if constexpr (!UP) {
        __syncthreads();
        if (tid < 64) {
            const int a = tid & 3, b = (tid >> 2) & 3, c = tid >> 4;
            const int ci = (t.x0 + 1) / 2 + a, cj = (t.y0 + 1) / 2 + b, ck = (t.z0 + 1) / 2 + c;
            if (ci <= gc.n0 && cj <= gc.n1 && ck <= gc.n2) {
                const T *r = Q + (4 + 2 * a) + L3_SY * (4 + 2 * b) + L3_SZ * (4 + 2 * c);
                T s = r[0];
                s = s + r[1];
                s = s + r[L3_SY];
                s = s + r[L3_SY + 1];
                s = s + r[L3_SZ];
                s = s + r[L3_SZ + 1];
                s = s + r[L3_SZ + L3_SY];
                s = s + r[L3_SZ + L3_SY + 1];
                bstore<T>(rs_c, T(0.125) * s, ((uint32_t)gc.off + (uint32_t)(ci + (int)gc.sy * cj + (int)gc.sz * ck)) * W, 0);
            }
        }
    }
}

}  // namespace mf3d
