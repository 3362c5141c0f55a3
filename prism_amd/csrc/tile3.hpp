// tile3.hpp -- one 16^3 tile (plus its +1 halo) of a 3-D field on one
// workgroup of 256 lanes: the tile in LDS, the stages of the four levels, and
// the codes between the level-major array (or the bit-planes) and the tile.
//
// Reference: InterpolationPredictor.cu -- 1-D rule 1229-1352,
// multi-dimensional rule 1414-1750, level loop 1823-2026, tile staging
// 997-1170, compaction 2028-2088.
#pragma once

#include <type_traits>

#include "common.hpp"
#include "spline_rules.hpp"

namespace pa {
namespace {

// ------------------------------------------------------------ LDS layout --
// Value (x, y, z) of the tile lies at z * 297 + Y(y) * 17 + x, where Y lists
// the even y before the odd ones.  A stage's lanes enumerate every other
// coordinate, which in the plain [17][17][17] order hit few of the banks:
// the multi-dimensional stages of a float32 tile took 7.2 LDS cycles per
// instruction, 5.1 of them conflicts.  The order, the plane pitch and the
// stages' lane enumerations were chosen together by counting the conflicts
// of every access of a level-0 pass (cycles of float32 / float64, forward
// + reverse + multi-dimensional: 5019 / 5519 plain, 3196 / 4724 here; all
// eight subsets of axes and pitches 289..301 were counted).  The strides
// along an axis stay compile-time constants, and 5041 values still let 4
// float64 or 8 float32 workgroups share the 160 KB.
constexpr int kYP = 17, kYO = 9 * 17, kZP = 297;
constexpr int kTileLds = 16 * kZP + 17 * 17;  // 5041

__host__ __device__ constexpr int tslot(int x, int y, int z) { return z * kZP + (y >> 1) * kYP + (y & 1) * kYO + x; }

// Along axis A (0 = x, 1 = y, 2 = z) at unit U: slots between even multiples
// of U (2U apart), and from an even multiple to the odd one after it.
template <int U, int A>
constexpr int slot_step() {
    return A == 0 ? 2 * U : (A == 1 ? U * kYP : 2 * U * kZP);
}
template <int U, int A>
constexpr int slot_half() {
    return A == 0 ? U : (A == 1 ? (U == 1 ? kYO : U / 2 * kYP) : U * kZP);
}

// A decompressing workgroup holds kGroup tiles adjacent along x, 256 lanes each.  A
// float32 tile's rows are 64 bytes, half a cache line: a copy of a 512^3 float32
// field in the tiles' access pattern (halo included) takes 322 us, 248 us in pairs
// (258 us in fours).  Decompression, which is bound by its accesses, takes
// pairs (round 4 of that field 287 us against 319 us one by one); compression,
// which is bound by its stages, is faster with 256-lane workgroups (342
// against 372 us: half as many waves meet at each of its 13 barriers).
template <typename T>
constexpr int kGroup = sizeof(T) == 4 ? 2 : 1;

// A field of one tile along x has no tiles to pair, and its tiles are taken one by
// one.  (With the second half of every workgroup idle instead, decompressing
// 4 x 4096 x 4096 float32 values took 1122 us, 16 x 2048 x 2048 448; 671 and 338
// one by one.)
template <typename T>
inline bool lone_tiles(int64_t nx, int64_t nz) {
    return kGroup<T> > 1 && nx <= 16 && nz > 1;
}

// IN: not the last tile along any axis, all 17^3 points inside the field
// (every stencil then is decided at compile time), and rows short enough for
// 32-bit offsets.  rx, ry, rz: points of the
// tile inside the field along each axis, halo included (17: not the last).
template <typename T, bool IN>
struct Tile {
    T* s;
    int ox, oy, oz;
    int rx, ry, rz;
    Geom g;
    T eb_r, ebx2;  // of the current level
    int32_t* qc_out;

    template <int A>
    __device__ __forceinline__ bool in(int c) const {
        return IN || c < (A == 0 ? rx : (A == 1 ? ry : rz));
    }
    __device__ __forceinline__ bool in3(int x, int y, int z) const { return IN || (x < rx && y < ry && z < rz); }
};

// every tile of group px is such a tile
template <int P>
__device__ __forceinline__ bool interior_group(const Geom& g, int px, int by, int bz) {
    return (px + 1) * (16 * P) < g.nx && by * 16 + 16 < g.ny && bz * 16 + 16 < g.nz && g.nx < (1 << 24);
}

// groups along x
template <int P>
__host__ __device__ inline int groups_x(const Geom& g) {
    return (g.gx + P - 1) / P;
}

// width: points along x the tile (or a group of tiles, taken as one) may
// have.  A group's second tile may lie outside the field (rx <= 0): its
// lanes then find no point inside.
template <typename T, bool IN>
__device__ __forceinline__ Tile<T, IN> make_tile(const Geom& g, T* s, int bx, int by, int bz, int32_t* qc_out,
                                                 int width = kTS) {
    Tile<T, IN> t;
    t.s = s;
    t.ox = bx * 16;
    t.oy = by * 16;
    t.oz = bz * 16;
    t.rx = min(g.nx - t.ox, width);
    t.ry = min(g.ny - t.oy, kTS);
    t.rz = min(g.nz - t.oz, kTS);
    t.g = g;
    t.qc_out = qc_out;
    return t;
}

// Lane of the phases that move rows between memory and the group's tiles:
// column X = 0 .. 16 P - 1 of the group of P, row y.
template <int P>
struct RowLane {
    int X, y;
    __device__ __forceinline__ RowLane() {
        const int v = thread_id();
        X = v & (16 * P - 1);
        y = (int)((unsigned)v / (16 * P));
    }
    // slot of point (x, y', z') of the lane's column in the group's LDS
    __device__ __forceinline__ int slot(int yy, int zz) const {
        return (X >> 4) * kTileLds + tslot(X & 15, yy, zz);
    }
};

// ---------------------------------------------------------------- stencils --
// Point j of a line of N = 8 / U points lies between the known values j and
// j + 1 of N + 1 (0 .. last inside the field, last = N away from the far
// face).  Which neighbours exist decides its formula
// (InterpolationPredictor.cu:1269-1326, 1538-1545), in the order of
// preference of the multi-dimensional rules:
enum Rank { R_NONE, R_LIN, R_QUAD, R_CUBIC };

template <int N, bool IN>
__device__ __forceinline__ Rank rank_of(int j, int last) {
    const bool has2 = IN || last >= j + 1, has3 = j + 2 <= N && (IN || last >= j + 2);
    if (!has2) return R_NONE;
    return j == 0 ? (has3 ? R_QUAD : R_LIN) : (has3 ? R_CUBIC : R_QUAD);
}

// The value of the formula of point j's rank; v0..v3 are the known values
// j - 1 .. j + 2 (anything where there is none).  R_NONE keeps v1.
template <typename T, int N, bool IN>
__device__ __forceinline__ T pred_line(int j, int last, T v0, T v1, T v2, T v3) {
    if constexpr (IN) {
        if (N == 1) return lin(v1, v2);  // (j is a constant)
        return j == 0 ? quad_r(v1, v2, v3) : (j == N - 1 ? quad_l(v0, v1, v2) : cubic(v0, v1, v2, v3));
    } else {
        T p = v1;
        if (last >= j + 1) p = j == 0 ? lin(v1, v2) : quad_l(v0, v1, v2);
        if (j + 2 <= N && last >= j + 2) p = j == 0 ? quad_r(v1, v2, v3) : cubic(v0, v1, v2, v3);
        return p;
    }
}

// ------------------------------------------------------------------ stages --
// Codes of a compressing tile stay in registers with their points' slots
// until the last stage (whose own codes go straight into its points' slots) is
// done: no stage reads values after that, every code then joins its slot, and
// all levels leave the tile as rows.  (Codes of levels 1-3 stored from their
// stages instead are scattered 4-byte writes, five times the requests, and
// their index arithmetic lengthens the chain of short stages.)
template <int N>
struct RegCodes {
    int32_t code[N];
    int slot, step;  // slot of code 0 (-1: none), distance of the slots
    __device__ __forceinline__ RegCodes() : slot(-1), step(0) {}
};

template <int N, typename T>
__device__ __forceinline__ void join_slots(T* s, const RegCodes<N>& r) {
    if (r.slot >= 0) {
#pragma unroll
        for (int k = 0; k < N; ++k) s[r.slot + k * r.step] = code_slot(r.code[k], T());
    }
}

template <int L, typename T, bool IN>
__device__ __forceinline__ uint32_t lm_at(const Tile<T, IN>& t, int x, int y, int z) {
    return lm_index<L>(t.g, t.ox + x, t.oy + y, t.oz + z);
}

// Levels 1-3 have few points, and the chain of their nine stages is bound by
// its length in instructions: there a lane takes a part of a line, kPart points
// (of the 4, 2 or 1 of its level), instead of all of it.
template <int U>
constexpr int kPart = U == 1 ? 8 : (U == 2 ? 2 : 1);
template <int U>
constexpr int kParts = 8 / U / kPart<U>;  // 1, 2, 2, 1 per line

// The wave that takes a stage's first 64 lanes.  The coarse levels' stages
// keep one to three of the four waves busy: they are dealt so that no lane
// would have to hold codes of two stages in one of its level's registers (see
// level3), and the waves' work evens out.
template <int U, int STAGE, bool MD>
constexpr int stage_wave() {
    if (U == 1) return 0;
    if (U == 2) return MD ? (STAGE == 1 ? 2 : 0) : (STAGE == 0 ? 0 : (STAGE == 1 ? 2 : 1));
    return STAGE;
}

// One point: its slot's value (or code) against pred.
template <typename T, int M, bool LAST, bool IN>
__device__ __forceinline__ void put_point(Tile<T, IN>& t, int slot, T v, T pred, int32_t& code) {
    if constexpr (M == COMPRESS) {
        code = quantize_val(v, pred, t.eb_r, t.ebx2);
        t.s[slot] = LAST ? code_slot(code, T()) : v;
    } else {
        t.s[slot] = pred + (T)slot_code(v) * t.ebx2;
    }
}

// Part h of a line per lane (all of it at level 0): known values at slots base
// + j * step, points at base + half + j * step (step and half: compile-time
// constants, or per-lane values where the lanes' lines differ in direction).
// A part of level 1 is one end of its line: the point at the end and the one
// next to it, which has four known values around it (w0 .. w3, from known
// value h on).
template <typename T, int U, int M, bool LAST, bool IN, class Step, class Half>
__device__ __forceinline__ void line_points(Tile<T, IN>& t, int base, Step step, Half half, int r, int h,
                                            RegCodes<kPart<U>>& rc) {
    constexpr int N = 8 / U;
    const int last = (int)((unsigned)(r - 1) / (2 * U));
    if constexpr (U == 1) {
        T k[N + 1], v[N];
#pragma unroll
        for (int j = 0; j <= N; ++j) k[j] = t.s[base + j * step];
#pragma unroll
        for (int j = 0; j < N; ++j) v[j] = t.s[base + half + j * step];
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const T pred = pred_line<T, N, IN>(j, last, k[j > 0 ? j - 1 : 0], k[j], k[j + 1], k[j + 2 <= N ? j + 2 : N]);
            int32_t code = 0;
            put_point<T, M, LAST>(t, base + half + j * step, v[j], pred, code);
            if constexpr (M == COMPRESS && !LAST) rc.code[j] = code;
        }
        if constexpr (!LAST) {  // (the last stage leaves the first one's codes alone)
            rc.slot = base + half;
            rc.step = step;
        }
    } else if constexpr (U == 2) {
        const int w = base + h * step, inner = base + half + (1 + h) * step, end = base + half + 3 * h * step;
        const T w0 = t.s[w], w1 = t.s[w + step], w2 = t.s[w + 2 * step], w3 = t.s[w + 3 * step];
        const T vi = t.s[inner], ve = t.s[end];
        T pi, pe;
        if constexpr (IN) {
            const T qr = quad_r(w0, w1, w2), ql = quad_l(w1, w2, w3);
            pi = cubic(w0, w1, w2, w3);
            pe = h == 0 ? qr : ql;
        } else {
            pi = pred_line<T, N, false>(1 + h, last, w0, w1, w2, w3);
            pe = pred_line<T, N, false>(3 * h, last, w1, h == 0 ? w0 : w2, h == 0 ? w1 : w3, w2);
        }
        int32_t ci = 0, ce = 0;
        put_point<T, M, LAST>(t, inner, vi, pi, ci);
        put_point<T, M, LAST>(t, end, ve, pe, ce);
        if constexpr (M == COMPRESS) {
            rc.code[0] = ci;
            rc.code[1] = ce;
        }
        rc.slot = inner;
        rc.step = end - inner;
    } else {
        const T w0 = t.s[base], w1 = t.s[base + step], w2 = t.s[base + (N == 2 ? 2 : 1) * step];
        const int slot = base + half + h * step;
        const T v = t.s[slot];
        T pred;
        if constexpr (N == 1) {
            pred = pred_line<T, 1, IN>(0, last, w0, w0, w1, w1);
        } else if constexpr (IN) {
            const T qr = quad_r(w0, w1, w2), ql = quad_l(w0, w1, w2);
            pred = h == 0 ? qr : ql;
        } else {
            pred = pred_line<T, 2, false>(h, last, w0, h == 0 ? w0 : w1, h == 0 ? w1 : w2, w2);
        }
        put_point<T, M, LAST>(t, slot, v, pred, rc.code[0]);
        rc.slot = slot;
    }
}

// A 1-D stage: lines along A over the other two axes, P (the lower) fastest;
// ALLP / ALLQ: at every multiple of U, or at the even ones.  LAST: the last
// stage of level 0, own points only (x, y, z < 16).
template <typename T, int U, int STAGE, int A, bool ALLP, bool ALLQ, int M, bool IN>
__device__ __forceinline__ void line_stage(Tile<T, IN>& t, RegCodes<kPart<U>>& rc) {
    constexpr int N = 8 / U;
    constexpr bool LAST = U == 1 && STAGE == 2;
    constexpr int CP = LAST ? 16 : (ALLP ? 2 * N + 1 : N + 1), CQ = LAST ? 16 : (ALLQ ? 2 * N + 1 : N + 1);
    static_assert(kParts<U> * CP * CQ <= kThreads, "one part of a line per lane");
    const int l = lane_id(stage_wave<U, STAGE, false>());
    if (l < kParts<U> * CP * CQ) {
        const int h = kParts<U> == 1 ? 0 : l / (CP * CQ), m = l - h * (CP * CQ);
        const int p = (m % CP) * (ALLP ? U : 2 * U), q = (m / CP) * (ALLQ ? U : 2 * U);
        const int x = A == 0 ? 0 : p, y = A == 1 ? 0 : (A == 0 ? p : q), z = A == 2 ? 0 : q;
        if (t.template in<A == 0 ? 1 : 0>(p) && t.template in<A == 2 ? 1 : 2>(q))
            line_points<T, U, M, LAST>(t, tslot(x, y, z), std::integral_constant<int, slot_step<U, A>()>{},
                                       std::integral_constant<int, slot_half<U, A>()>{},
                                       A == 0 ? t.rx : (A == 1 ? t.ry : t.rz), h, rc);
    }
    lds_barrier();
}

// LINE points (one odd coordinate): the lines along x, y and z through the
// points with both other coordinates even, in one sweep.
template <typename T, int U, int M, bool IN>
__device__ __forceinline__ void lines3_stage(Tile<T, IN>& t, RegCodes<kPart<U>>& rc) {
    constexpr int N = 8 / U, C = N + 1, LINES = 3 * C * C;
    static_assert(kParts<U> * LINES <= kThreads, "one part of a line per lane");
    const int l = lane_id(stage_wave<U, 0, true>());
    if (l < kParts<U> * LINES) {
        const int h = kParts<U> == 1 ? 0 : (l >= LINES ? 1 : 0), ln = l - h * LINES;
        const int grp = ln / (C * C), m = ln % (C * C), i = 2 * U * (m % C), j = 2 * U * (m / C);
        const int x = grp == 0 ? 0 : i, y = grp == 0 ? i : (grp == 1 ? 0 : j), z = grp == 2 ? 0 : j;
        if (t.in3(x, y, z)) {
            const int step = grp == 0 ? slot_step<U, 0>() : (grp == 1 ? slot_step<U, 1>() : slot_step<U, 2>());
            const int half = grp == 0 ? slot_half<U, 0>() : (grp == 1 ? slot_half<U, 1>() : slot_half<U, 2>());
            line_points<T, U, M, false>(t, tslot(x, y, z), step, half, grp == 0 ? t.rx : (grp == 1 ? t.ry : t.rz), h, rc);
        }
    }
    lds_barrier();
}

// The prediction of a point from its two directions: the formulas compete by
// rank (InterpolationPredictor.cu:1546-1669): equal ranks are averaged, the
// higher one wins, and where neither has a far neighbour the point continues
// the plane through its three known neighbours.  Point ja of a line along
// one axis with known values a0..a3 around it (last known index lasta), jb
// and b0..b3 along the other; corner: slot of the known value below both.
// IN: fa, the rank along A, is a constant.
template <typename T, int N, bool IN>
__device__ __forceinline__ T pred_face2(const T* corner, Rank fa, int ja, int lasta, T a0, T a1, T a2, T a3, int jb,
                                        int lastb, T b0, T b1, T b2, T b3) {
    const Rank fb = rank_of<N, IN>(jb, lastb);
    if constexpr (IN) {
        // every value first, then selections: a branch per lane costs more
        if (N == 1) return (lin(a1, a2) + lin(b1, b2)) / (T)2;
        const T ar = quad_r(a1, a2, a3), al = quad_l(a0, a1, a2), br = quad_r(b1, b2, b3), bl = quad_l(b0, b1, b2);
        const T edge = ((ja == 0 ? ar : al) + (jb == 0 ? br : bl)) / (T)2;
        if (N == 2) return edge;
        const T cb = cubic(b0, b1, b2, b3);
        if (fa != R_CUBIC) return fb == R_CUBIC ? cb : edge;
        const T ca = cubic(a0, a1, a2, a3), two = (ca + cb) / (T)2;
        return fb == R_CUBIC ? two : ca;
    } else {
        const T pa = pred_line<T, N, false>(ja, lasta, a0, a1, a2, a3);
        const T pb = pred_line<T, N, false>(jb, lastb, b0, b1, b2, b3);
        T pred = fa > fb ? pa : pb;
        if (fa == fb) pred = fa == R_NONE ? (a1 + b1) - *corner : (pa + pb) / (T)2;
        return pred;
    }
}

// FACE points (two odd coordinates): a lane takes a line (or part h of one)
// along A (z, or y for the points with even z) at one odd position jb of the
// other odd axis B: the known values of the line are read once, four taps along
// B per point.
template <typename T, int U, int M, bool IN>
__device__ __forceinline__ void faces_stage(Tile<T, IN>& t, RegCodes<kPart<U>>& rc) {
    constexpr int N = 8 / U, C = N + 1, LINES = 3 * N * C;
    static_assert(kParts<U> * LINES <= kThreads, "one part of a line per lane");
    const int l = lane_id(stage_wave<U, 1, true>());
    if (l < kParts<U> * LINES) {
        // groups: (y, z) odd at even x, x fastest; (x, z) odd at even y, x
        // fastest; (x, y) odd at even z, z fastest
        const int h = kParts<U> == 1 ? 0 : (l >= LINES ? 1 : 0), ln = l - h * LINES;
        const int grp = ln / (N * C), m = ln - grp * (N * C);
        const int q = grp == 1 ? m / N : m / C, p = grp == 1 ? m - q * N : m - q * C;
        const int jb = grp == 1 ? p : q, c = 2 * U * (grp == 1 ? q : p), b = 2 * U * jb;
        const int x = grp == 0 ? c : b, y = grp == 0 ? b : (grp == 1 ? c : 0), z = grp == 2 ? c : 0;
        if (t.in3(grp == 0 ? x : x + U, grp == 1 ? y : y + U, grp == 2 ? z : z + U)) {
            const int sa = grp == 2 ? slot_step<U, 1>() : slot_step<U, 2>();
            const int ha = grp == 2 ? slot_half<U, 1>() : slot_half<U, 2>();
            const int sb = grp == 0 ? slot_step<U, 1>() : slot_step<U, 0>();
            const int hb = grp == 0 ? slot_half<U, 1>() : slot_half<U, 0>();
            const T* left = t.s + tslot(x, y, z);  // A and B even
            const T* ka = left + hb;               // A even, B odd: known values along A
            const int own = tslot(x, y, z) + hb + ha;  // the points
            const T *p1 = left + ha, *p0 = p1 - (jb > 0 ? sb : 0), *p2 = p1 + sb, *p3 = p2 + (jb < N - 1 ? sb : 0);
            const int ra = grp == 2 ? t.ry : t.rz, rb = grp == 0 ? t.ry : t.rx;
            const int lasta = (int)((unsigned)(ra - 1) / (2 * U)), lastb = (int)((unsigned)(rb - 1) / (2 * U));
            if constexpr (U == 1) {
                T k[N + 1], v[N];
#pragma unroll
                for (int j = 0; j <= N; ++j) k[j] = ka[j * sa];
#pragma unroll
                for (int j = 0; j < N; ++j) v[j] = t.s[own + j * sa];
                // taps of G points are read together, ahead of the writes of
                // the points before them
                constexpr int G = sizeof(T) == 8 ? 2 : 4;
#pragma unroll
                for (int j0 = 0; j0 < N; j0 += G) {
                    T w[4][G];
#pragma unroll
                    for (int d = 0; d < G; ++d) {
                        const int o = (j0 + d) * sa;
                        w[0][d] = p0[o];
                        w[1][d] = p1[o];
                        w[2][d] = p2[o];
                        w[3][d] = p3[o];
                    }
#pragma unroll
                    for (int d = 0; d < G; ++d) {
                        const int j = j0 + d;
                        const T pred = pred_face2<T, N, IN>(left + j * sa, rank_of<N, IN>(j, lasta), j, lasta,
                                                            k[j > 0 ? j - 1 : 0], k[j], k[j + 1], k[j + 2 <= N ? j + 2 : N],
                                                            jb, lastb, w[0][d], w[1][d], w[2][d], w[3][d]);
                        int32_t code = 0;
                        put_point<T, M, false>(t, own + j * sa, v[j], pred, code);
                        if constexpr (M == COMPRESS) rc.code[j] = code;
                    }
                }
                rc.slot = own;
                rc.step = sa;
            } else if constexpr (U == 2) {
                const int ji = 1 + h, je = 3 * h, oi = ji * sa, oe = je * sa;
                const T *w = ka + h * sa, w0 = w[0], w1 = w[sa], w2 = w[2 * sa], w3 = w[3 * sa];
                const T i0 = p0[oi], i1 = p1[oi], i2 = p2[oi], i3 = p3[oi];
                const T e0 = p0[oe], e1 = p1[oe], e2 = p2[oe], e3 = p3[oe];
                const T vi = t.s[own + oi], ve = t.s[own + oe];
                const T pi = pred_face2<T, N, IN>(left + oi, IN ? R_CUBIC : rank_of<N, IN>(ji, lasta), ji, lasta, w0, w1, w2,
                                                  w3, jb, lastb, i0, i1, i2, i3);
                const T pe = pred_face2<T, N, IN>(left + oe, IN ? R_QUAD : rank_of<N, IN>(je, lasta), je, lasta, w1,
                                                  h == 0 ? w0 : w2, h == 0 ? w1 : w3, w2, jb, lastb, e0, e1, e2, e3);
                int32_t ci = 0, ce = 0;
                put_point<T, M, false>(t, own + oi, vi, pi, ci);
                put_point<T, M, false>(t, own + oe, ve, pe, ce);
                if constexpr (M == COMPRESS) {
                    rc.code[0] = ci;
                    rc.code[1] = ce;
                }
                rc.slot = own + oi;
                rc.step = oe - oi;
            } else {
                const int o = h * sa;
                const T w0 = ka[0], w1 = ka[sa], w2 = ka[(N == 2 ? 2 : 1) * sa];
                const T b0 = p0[o], b1 = p1[o], b2 = p2[o], b3 = p3[o], v = t.s[own + o];
                const T pred = pred_face2<T, N, IN>(left + o, IN ? R_QUAD : rank_of<N, IN>(h, lasta), h, lasta, w0,
                                                    h == 0 ? w0 : w1, h == 0 ? w1 : w2, w2, jb, lastb, b0, b1, b2, b3);
                put_point<T, M, false>(t, own + o, v, pred, rc.code[0]);
                rc.slot = own + o;
            }
        }
    }
    lds_barrier();
}

// CUBE points (three odd coordinates, InterpolationPredictor.cu:1671-1723):
// the mean of the directions whose formula is the cubic; without one, x's
// formula.
template <typename T, int U, int M, bool IN>
__device__ __forceinline__ void cubes_stage(Tile<T, IN>& t, RegCodes<kPart<U>>& rc) {
    constexpr int N = 8 / U, TOTAL = N * N * N;
    constexpr bool LAST = U == 1;
    constexpr int SX = slot_step<U, 0>(), SY = slot_step<U, 1>(), SZ = slot_step<U, 2>();
    constexpr int HX = slot_half<U, 0>(), HY = slot_half<U, 1>(), HZ = slot_half<U, 2>();
    const int l = lane_id(stage_wave<U, 2, true>());
#pragma unroll
    for (int it = 0; it < (TOTAL + kThreads - 1) / kThreads; ++it) {
        const int p = l + it * kThreads;
        if (TOTAL % kThreads == 0 || p < TOTAL) {
            const int i = p % N, j = (p / N) % N, k = p / (N * N);
            const int x = (2 * i + 1) * U, y = (2 * j + 1) * U, z = (2 * k + 1) * U;
            if (t.in3(x, y, z)) {
                const int lastx = (int)((unsigned)(t.rx - 1) / (2 * U)), lasty = (int)((unsigned)(t.ry - 1) / (2 * U)),
                          lastz = (int)((unsigned)(t.rz - 1) / (2 * U));
                const int corner = i * SX + j * SY + k * SZ, own_slot = corner + HX + HY + HZ;
                // x's taps: y and z odd, from the left neighbour
                const T* bx = t.s + corner + (HY + HZ);
                const T own = t.s[own_slot];
                const T x0 = bx[i > 0 ? -SX : 0], x1 = bx[0], x2 = bx[SX], x3 = bx[i < N - 1 ? 2 * SX : SX];
                const Rank fx = rank_of<N, IN>(i, lastx);
                T pred = x1;
                if constexpr (N == 1) {
                    if (IN || fx == R_LIN) pred = lin(x1, x2);
                } else {
                    const T qr = quad_r(x1, x2, x3), ql = quad_l(x0, x1, x2);
                    if constexpr (!IN) {
                        if (fx == R_LIN) pred = lin(x1, x2);
                    }
                    pred = IN || fx == R_QUAD ? (i == 0 ? qr : ql) : pred;
                }
                if constexpr (N > 2) {
                    const T *by = t.s + corner + (HX + HZ), *bz = t.s + corner + (HX + HY);
                    const T y0 = by[j > 0 ? -SY : 0], y1 = by[0], y2 = by[SY], y3 = by[j < N - 1 ? 2 * SY : SY];
                    const T z0 = bz[k > 0 ? -SZ : 0], z1 = bz[0], z2 = bz[SZ], z3 = bz[k < N - 1 ? 2 * SZ : SZ];
                    const bool cx = fx == R_CUBIC, cy = rank_of<N, IN>(j, lasty) == R_CUBIC,
                               cz = rank_of<N, IN>(k, lastz) == R_CUBIC;
                    // an absent direction adds 0 (a zero's sign cannot reach a
                    // value or code: each adds code * ebx2 to the prediction)
                    const T px = cx ? cubic(x0, x1, x2, x3) : (T)0;
                    const T py = cy ? cubic(y0, y1, y2, y3) : (T)0;
                    const T pz = cz ? cubic(z0, z1, z2, z3) : (T)0;
                    const T sum = (px + py) + pz;
                    const T half = sum / (T)2, third = third_of(sum);
                    const bool all = cx && cy && cz, two = (cx && cy) || (cz && (cx || cy)), any = cx || cy || cz;
                    pred = any ? sum : pred;
                    pred = two ? half : pred;
                    pred = all ? third : pred;
                }
                int32_t code = 0;
                put_point<T, M, LAST>(t, own_slot, own, pred, code);
                if constexpr (M == COMPRESS && !LAST) {  // one point: every code its, step 0
#pragma unroll
                    for (int d = 0; d < kPart<U>; ++d) rc.code[d] = code;
                    rc.slot = own_slot;
                    rc.step = 0;
                }
            }
        }
    }
    lds_barrier();
}

// Level 0's codes of a tile in the level-major array, by column (x, y): at odd
// z a row holds every x, at even z every x of an odd y and the odd x of an
// even y; from z to z + 2 the index advances by 2 lxy0 - lxy1.  The tile's
// part of an index is uniform (a scalar base that steps along z), the lane's
// a 32-bit offset (nx is below 2^24 in an IN tile; elsewhere the lane's part
// is added in 64 bits).
template <typename E, bool IN>
struct Columns0 {
    using Off = std::conditional_t<IN, uint32_t, int64_t>;
    E *even, *odd;  // z = 0 and z = 1
    int64_t step;
    Off off_even, off_odd;

    template <typename T>
    __device__ __forceinline__ Columns0(const Tile<T, IN>& t, E* q, int x, int y) {
        const int64_t lx0 = t.g.lx[0], lx1 = t.g.lx[1], lxy0 = t.g.lxy[0], lxy1 = t.g.lxy[1];
        step = 2 * lxy0 - lxy1;
        const int64_t base = t.g.prefix[0] + t.oy * lx0 + (t.oz >> 1) * step;
        even = q + (base - (t.oy >> 1) * lx1);
        odd = q + (base + t.ox + lxy0 - lxy1);
        const Off row = (Off)y * (Off)lx0;
        off_odd = row + (Off)x;
        off_even = row - (Off)((y + 1) >> 1) * (Off)lx1 + (Off)((y & 1) ? t.ox + x : (t.ox + x) >> 1);
    }
    __device__ __forceinline__ E& at_even() const { return *(E*)((char*)even + off_even * (Off)sizeof(E)); }
    __device__ __forceinline__ E& at_odd() const { return *(E*)((char*)odd + off_odd * (Off)sizeof(E)); }
    __device__ __forceinline__ void next() {
        even += step;
        odd += step;
    }
};

// The codes of the tile, all in their slots, written out row by row.
// Level 0: a row lane takes its column's z = 0..15 (rows of 16 or 8 adjacent
// codes).  Level 1: the points with even coordinates, in two passes of 8 adjacent
// codes per row; levels 2 and 3 in one.
// Returns the magnitudes of the lane's codes (live_words).
template <typename T, bool IN>
__device__ __forceinline__ Mags codes_out(const Tile<T, IN>& t) {
    Mags g;
    {
        const RowLane<1> r;
        if (t.template in<0>(r.X) && t.template in<1>(r.y)) {
            const T* src = t.s + r.slot(r.y, 0);
            Columns0<int32_t, IN> c(t, t.qc_out, r.X, r.y);
            const bool on_even = (r.X | r.y) & 1;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                if (t.template in<2>(2 * k + 1)) c.at_odd() = g.fine(slot_code(src[(2 * k + 1) * kZP]));
                if (on_even && t.template in<2>(2 * k)) c.at_even() = g.fine(slot_code(src[2 * k * kZP]));
                c.next();
            }
        }
    }
    const int v = thread_id();
#pragma unroll
    for (int it = 0; it < 2; ++it) {
        const int x = 2 * (v & 7), y = 2 * ((v / 8) & 7), z = 2 * (v / 64 + 4 * it);
        if (((x | y | z) & 2) && t.in3(x, y, z)) t.qc_out[lm_at<1>(t, x, y, z)] = g.coarse(slot_code(t.s[tslot(x, y, z)]));
    }
    if (v < 64) {
        const int x = 4 * (v & 3), y = 4 * ((v / 4) & 3), z = 4 * (v / 16);
        if (((x | y | z) & 4) && t.in3(x, y, z)) t.qc_out[lm_at<2>(t, x, y, z)] = g.coarse(slot_code(t.s[tslot(x, y, z)]));
    } else if (v < 72) {
        const int w = v - 64, x = 8 * (w & 1), y = 8 * ((w / 2) & 1), z = 8 * (w / 4);
        if (((x | y | z) & 8) && t.in3(x, y, z)) t.qc_out[lm_at<3>(t, x, y, z)] = g.coarse(slot_code(t.s[tslot(x, y, z)]));
    }
    return g;
}

// The three stages of one level (InterpolationPredictor.cu:1940-2025); a, b:
// the codes' registers.  At level 0 they hold the first two stages' codes.  At
// levels 2 and 3 each stage has a wave of its own, and a holds them all; at
// level 1 a and b hold the codes of disjoint lanes: stages 0 and 2 (a: wave 0;
// waves 1-3), 1 (b: waves 2, 3), or in the multi-dimensional form 0 (a: waves
// 0-2), 1 and 2 (b: waves 2, 3; wave 0).
template <typename T, int U, int M, bool IN>
__device__ __forceinline__ void level3(Tile<T, IN>& t, bool md, bool rev, RegCodes<kPart<U>>& a, RegCodes<kPart<U>>& b) {
    if (md) {
        lines3_stage<T, U, M>(t, a);
        faces_stage<T, U, M>(t, U > 2 ? a : b);
        cubes_stage<T, U, M>(t, U > 2 ? a : b);
    } else if (rev) {
        line_stage<T, U, 0, 0, false, false, M>(t, a);
        line_stage<T, U, 1, 1, true, false, M>(t, U > 2 ? a : b);
        line_stage<T, U, 2, 2, true, true, M>(t, a);
    } else {
        line_stage<T, U, 0, 2, false, false, M>(t, a);
        line_stage<T, U, 1, 1, false, true, M>(t, U > 2 ? a : b);
        line_stage<T, U, 2, 0, true, true, M>(t, a);
    }
}

// The flags in two steps: every lane loads one byte before the tile's loads
// are issued, and once those are in their slots the bytes become a scalar mask
// (bit i: flags8[i] is set).  Flags kept in registers as loaded instead made
// the compiler wait for every outstanding access (the codes already stored,
// the previous values still on their way) at each level.
__device__ __forceinline__ uint32_t flags_load(const uint8_t* flags8) { return flags8[threadIdx.x & 7]; }
__device__ __forceinline__ uint32_t flags_mask(uint32_t byte) {
    asm volatile("" : "+v"(byte));  // (the comparison stays here)
    return (uint32_t)__ballot(byte != 0u) & 0xFFu;
}

// The four levels of a tile, coarsest first; compressing, every code ends up
// in its point's slot.
template <typename T, int M, bool IN>
__device__ __forceinline__ void tile_levels(Tile<T, IN>& t, const LevelEb<T>& le, uint32_t flags, int maxlevel) {
    RegCodes<1> c3, c2;
    RegCodes<2> c1a, c1b;
    RegCodes<8> a, b;
    if (3 <= maxlevel) { t.eb_r = le.eb_r[3]; t.ebx2 = le.ebx2[3]; level3<T, 8, M>(t, flags & 8, flags & 128, c3, c3); }
    if (2 <= maxlevel) { t.eb_r = le.eb_r[2]; t.ebx2 = le.ebx2[2]; level3<T, 4, M>(t, flags & 4, flags & 64, c2, c2); }
    if (1 <= maxlevel) { t.eb_r = le.eb_r[1]; t.ebx2 = le.ebx2[1]; level3<T, 2, M>(t, flags & 2, flags & 32, c1a, c1b); }
    if (0 <= maxlevel) { t.eb_r = le.eb_r[0]; t.ebx2 = le.ebx2[0]; level3<T, 1, M>(t, flags & 1, flags & 16, a, b); }
    if constexpr (M == COMPRESS) {
        join_slots(t.s, c3);
        join_slots(t.s, c2);
        join_slots(t.s, c1a);
        join_slots(t.s, c1b);
        join_slots(t.s, a);
        join_slots(t.s, b);
        lds_barrier();
    }
}

// ------------------------------------------------------- tile and memory --
// The 17^3 points of a tile are taken as 20 sets of at most one point per
// lane: the rows y < 16 at z = 0..16, the rows y = 16 at z < 16 (both by the
// group's row lanes), then by the tile's own lanes the face x = 16 (lane
// (y, z) = (l mod 16, l / 16)) and the last rows (x, 16, 16), (16, 16, z) and
// (16, y, 16).  Addresses of the first advance by a plane from point to point.
// false: the lane has no point.
__device__ __forceinline__ bool edge_point(int l, int& x, int& y, int& z) {
    x = l < 16 ? l : 16;
    y = l < 33 ? 16 : l - 33;
    z = l >= 16 && l < 33 ? l - 16 : 16;
    return l < 49;
}

// Column (x, y) of a tile of a field (base: the tile's first value), plane by
// plane: a uniform base that steps by a plane and the lane's 32-bit offset
// (nx is below 2^24 in an IN tile; elsewhere 64-bit).
template <typename T, bool IN>
struct Column {
    using Off = std::conditional_t<IN, uint32_t, uint64_t>;
    T* base;
    uint32_t plane;
    Off off;

    __device__ __forceinline__ Column(T* b, uint32_t nx, uint32_t nxy, int x, int y)
        : base(b), plane(nxy), off((Off)y * nx + (Off)x) {}
    __device__ __forceinline__ T& at() const { return *(T*)((char*)base + off * (Off)sizeof(T)); }
    __device__ __forceinline__ void next() { base += plane; }
};

// Tile plus halo into LDS: all global loads of a lane are issued before the
// first LDS write so the tile costs one memory latency.  Points outside the
// field are not read (no formula uses their slots).
template <typename T, bool IN>
__device__ __forceinline__ void tile_load(const Tile<T, IN>& t, const T* __restrict__ data) {
    const uint32_t nx = (uint32_t)t.g.nx, nxy = nx * (uint32_t)t.g.ny;  // (fields have fewer than 2^31 values)
    const T* base = data + ((uint64_t)t.oz * nxy + (uint64_t)t.oy * nx + t.ox);
    T v[17], fy = (T)0, fx = (T)0, e = (T)0;
    const RowLane<1> r;
    const bool on = t.template in<0>(r.X) && t.template in<1>(r.y);
    Column<const T, IN> p(base, nx, nxy, r.X, r.y);
#pragma unroll
    for (int z = 0; z < 17; ++z) {
        v[z] = (T)0;
        if (on && t.template in<2>(z)) v[z] = p.at();
        p.next();
    }
    if (t.in3(r.X, 16, r.y)) fy = base[(uint64_t)r.y * nxy + (16 * (uint64_t)nx + r.X)];
    const int l = lane_id(), y = l & 15, z = l >> 4;
    int ex, ey, ez;
    const bool edge = edge_point(l, ex, ey, ez);
    if (t.in3(16, y, z)) fx = base[(uint64_t)z * nxy + ((uint64_t)y * nx + 16)];
    if (edge && t.in3(ex, ey, ez)) e = base[(uint64_t)ez * nxy + ((uint64_t)ey * nx + ex)];
    T* d = t.s + r.slot(r.y, 0);
#pragma unroll
    for (int k = 0; k < 17; ++k) d[k * kZP] = v[k];
    t.s[r.slot(16, r.y)] = fy;
    t.s[tslot(16, y, z)] = fx;
    if (edge) t.s[tslot(ex, ey, ez)] = e;
}

// Decompression first fills the slot of every point with the bit pattern of
// its own code (corners: the anchors; points of skipped levels: 0); a stage
// then reads the slot of the point it reconstructs and overwrites it.  E:
// int32_t or int16_t codes.
template <typename T>
struct TileCodes {
    int32_t v0[17], fy, fx, e;  // level 0, the point sets above
    int32_t v1[3], v23;         // levels 1 (9^3 points), 2 (5^3, lanes 0..) and 3 (3^3, lanes 128..)
    T anc;
};

// the tile's eight corner anchors (x_reset_scratch_data 1051-1061)
template <typename T, bool IN>
__device__ __forceinline__ T anchor_load(const Tile<T, IN>& t, const T* __restrict__ anchors, int bx, int by, int bz) {
    const int l = lane_id();
    T a = (T)0;
    if (l < 8) {
        const int ax = bx + (l & 1), ay = by + ((l >> 1) & 1), az = bz + (l >> 2);
        if (anchors && ax < t.g.gx && ay < t.g.gy && az < t.g.gz)
            a = anchors[ax + (int64_t)ay * t.g.gx + (int64_t)az * t.g.gx * t.g.gy];
    }
    return a;
}

template <typename T, bool IN>
__device__ __forceinline__ void anchor_store(const Tile<T, IN>& t, T anc) {
    const int l = lane_id();
    if (l < 8) t.s[tslot(16 * (l & 1), 16 * ((l >> 1) & 1), 16 * (l >> 2))] = anc;
}

// lane's point of levels 2 and 3 in lattice units
__device__ __forceinline__ bool coarse_point(int l, int& unit, int& i, int& j, int& k) {
    const bool l3 = l >= 128;
    const int m = l3 ? l - 128 : l;
    unit = l3 ? 8 : 4;
    i = l3 ? m % 3 : m % 5;
    j = l3 ? (m / 3) % 3 : (m / 5) % 5;
    k = l3 ? m / 9 : m / 25;
    return m < (l3 ? 27 : 125);
}

template <int P, typename T, bool IN, typename E>
__device__ __forceinline__ void codes_load(const Tile<T, IN>& t, const Tile<T, IN>& m, const E* __restrict__ q, int maxlevel,
                                           const T* __restrict__ anchors, int bx, int by, int bz, TileCodes<T>& c) {
    const int l = lane_id();
    const bool l0 = maxlevel >= 0;
    c.v23 = 0;
    {
        int u, i, j, k;
        if (coarse_point(l, u, i, j, k) && ((i | j | k) & 1) && t.in3(u * i, u * j, u * k)) {
            if (u == 4) {
                if (maxlevel >= 2) c.v23 = q[lm_at<2>(t, 4 * i, 4 * j, 4 * k)];
            } else if (maxlevel >= 3) {
                c.v23 = q[lm_at<3>(t, 8 * i, 8 * j, 8 * k)];
            }
        }
    }
#pragma unroll
    for (int it = 0; it < 3; ++it) {
        const int p = l + it * kThreads, i = p % 9, j = (p / 9) % 9, k = p / 81;
        c.v1[it] = 0;
        if (maxlevel >= 1 && p < 729 && ((i | j | k) & 1) && t.in3(2 * i, 2 * j, 2 * k))
            c.v1[it] = q[lm_at<1>(t, 2 * i, 2 * j, 2 * k)];
    }
    const RowLane<P> r;
    const bool on = l0 && m.template in<0>(r.X) && m.template in<1>(r.y), on_even = on && ((r.X | r.y) & 1);
    Columns0<const E, IN> col(m, q, r.X, r.y);
#pragma unroll
    for (int k = 0; k <= 8; ++k) {
        c.v0[2 * k] = 0;
        if (on_even && m.template in<2>(2 * k)) c.v0[2 * k] = col.at_even();
        if (k < 8) {
            c.v0[2 * k + 1] = 0;
            if (on && m.template in<2>(2 * k + 1)) c.v0[2 * k + 1] = col.at_odd();
        }
        col.next();
    }
    c.fy = c.fx = c.e = 0;
    if (l0 && ((r.X | r.y) & 1) && m.in3(r.X, 16, r.y)) c.fy = q[lm_at<0>(m, r.X, 16, r.y)];
    const int y = l & 15, z = l >> 4;
    if (l0 && ((y | z) & 1) && t.in3(16, y, z)) c.fx = q[lm_at<0>(t, 16, y, z)];
    int ex, ey, ez;
    if (edge_point(l, ex, ey, ez) && l0 && ((ex | ey | ez) & 1) && t.in3(ex, ey, ez)) c.e = q[lm_at<0>(t, ex, ey, ez)];
    c.anc = anchor_load(t, anchors, bx, by, bz);
}

template <int P, typename T, bool IN>
__device__ __forceinline__ void codes_store(const Tile<T, IN>& t, const Tile<T, IN>& m, const TileCodes<T>& c) {
    const int l = lane_id();
    {
        int u, i, j, k;
        if (coarse_point(l, u, i, j, k) && ((i | j | k) & 1)) t.s[tslot(u * i, u * j, u * k)] = code_slot(c.v23, T());
    }
#pragma unroll
    for (int it = 0; it < 3; ++it) {
        const int p = l + it * kThreads, i = p % 9, j = (p / 9) % 9, k = p / 81;
        if (p < 729 && ((i | j | k) & 1)) t.s[tslot(2 * i, 2 * j, 2 * k)] = code_slot(c.v1[it], T());
    }
    const RowLane<P> r;
    T* d = m.s + r.slot(r.y, 0);
#pragma unroll
    for (int k = 0; k < 8; ++k) d[(2 * k + 1) * kZP] = code_slot(c.v0[2 * k + 1], T());
    if ((r.X | r.y) & 1) {
#pragma unroll
        for (int k = 0; k <= 8; ++k) d[2 * k * kZP] = code_slot(c.v0[2 * k], T());
        m.s[r.slot(16, r.y)] = code_slot(c.fy, T());
    }
    const int y = l & 15, z = l >> 4;
    if ((y | z) & 1) t.s[tslot(16, y, z)] = code_slot(c.fx, T());
    int ex, ey, ez;
    if (edge_point(l, ex, ey, ez) && ((ex | ey | ez) & 1)) t.s[tslot(ex, ey, ez)] = code_slot(c.e, T());
    anchor_store(t, c.anc);
}

}  // namespace
}  // namespace pa
